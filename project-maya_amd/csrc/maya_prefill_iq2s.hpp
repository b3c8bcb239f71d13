// maya_prefill_iq2s.hpp - the prompt chunk's grouped GEMM on IQ2_S rows in the stream packing (included by
// maya_prefill.hip inside namespace maya; the skeleton - tiles, the activations' copies, the barriers - is pf_tile's).
// out[row][n] = 1/8 sum over blocks b of (d_w[n][b] d_x[row][b]) * sum over the block's 16-value groups j of (2 ls_j +
// 1) (w_j . c_j), w = the grid magnitudes with their signs: the integer sums of the CPU path's IQ2_S x Q8_K row dot
// (src/kernels/cpu/iq_avx2.cpp:160-176, 225-250).
//
// A weight is one of six values of its group, +-(2 ls + 1) x {8, 25, 43} (at most 1333), so it is taken as two int8
// digits, u = 256 hi + lo, and each digit as a byte looked up by v_perm_b32 in the group's six: a 16-entry table in LDS
// gives a lane its group's eight bytes of either digit, the grid (its magnitudes as 0 / 1 / 2) joined with a sign table (4 in
// the bytes of set bits) gives the selectors, and one v_perm_b32 a digit makes four weights, signed and scaled.  The two
// digits' products with the codes then run through the 32x32x32 matrix instructions over the whole 256-value block, as
// Q4_K's two planes do (pf_tile): no scaled sums outside the matrix cores, one convert and two multiplies an output a block.
// The form before this one gave a matrix instruction the magnitudes of ONE 16-value group (the operand's other half zero) and
// added (2 ls + 1) x its sums on the vector ALU: 41 vector instructions to decode 512 weights and two multiply-adds an
// output every 32 values, 79 % of the cycles in vector issue.  A 75-token chunk on
// 160 experts of 6144 x 1536 735 -> 535 us; gate/up IQ2_S with Q4_K down, 1187 tokens on 256 of 7168 x 2048, 2830 -> 2190 us.
// LDS of one buffer of activations: the codes [kPfRows][256], d [kPfRows]
constexpr int kPfPlane = kPfRows * 256;
constexpr int kPfDOffNoS = kPfPlane, kPfBufBytesNoS = kPfDOffNoS + kPfRows * 4;
// The tile's activations go from global memory to LDS without passing registers (each lane's 16 bytes land at the
// wave's base + 16 lane): buffer loads whose per-lane offsets are fixed for the tile - the super-block rides in the
// scalar offset - so a copy costs no vector arithmetic.  Rows past the tile's end repeat its last row (their results
// are never stored).
template <int NMT>
struct PfDma {
    __amdgpu_buffer_rsrc_t rq, rd;
    uint32_t oq[NMT], od;
    int wave;
    __device__ __forceinline__ void init(const PfGemm& a, int row0, int nrows, int wave_, int lane) {
        wave = wave_;
        const int last = nrows - 1;
        rq = __builtin_amdgcn_make_buffer_rsrc((void*) (a.x.q + (size_t) row0 * a.k), 0, (int) (nrows * a.k), 0x00020000);
        rd = __builtin_amdgcn_make_buffer_rsrc((void*) (a.x.d + (size_t) row0 * (a.k >> 8)), 0, (int) (nrows * (a.k >> 8) * 4), 0x00020000);
#pragma unroll
        for (int n = 0; n < NMT; ++n) {
            const int r = 4 * (wave + 4 * n) + (lane >> 4), cp = lane & 15;   // rows 4 i .. 4 i + 3, i = wave + 4 n
            oq[n] = (uint32_t) (min(r, last) * (int) a.k + ((cp ^ (r & 15)) * 16));
        }
        od = (uint32_t) (min(lane, last) * (int) (a.k >> 8) * 4);
    }
    // super-block sb into the buffer at `buf`
    __device__ __forceinline__ void copy(uint8_t* buf, int sb) const {
#pragma unroll
        for (int n = 0; n < NMT; ++n)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rq, (pf_lptr) (buf + (wave + 4 * n) * 1024), 16, oq[n], sb * 256, 0, 0);
        if (wave == 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(rd, (pf_lptr) (buf + kPfDOffNoS), 4, od, sb * 4, 0, 0);
    }
};

constexpr int kIqMags = 0, kIqSigns = 8192, kIqScales = kIqSigns + 2048, kIqTables = kIqScales + 256;   // byte offsets in LDS
constexpr int kIqLdsBytes = kIqTables + 3 * kPfBufBytesNoS;

struct IqLook {   // the LDS look-ups of one sub-block: selectors and signs of the lane's two grid entries, its group's digits
    pf_i2 m0, m1, s0, s1;
    v4i sc;       // the low digits of +{8, 25, 43}, of -{8, 25, 43}, then the high ones
};
template <int BUT, int NM> __device__ __forceinline__ void iq_wait(IqLook& l, v4i (&x)[NM]) {
    static_assert(NM == 1 || NM == 2, "1 or 2 row groups");
    if constexpr (NM == 1)
        asm volatile("s_waitcnt lgkmcnt(%6)" : "+v"(l.m0), "+v"(l.m1), "+v"(l.s0), "+v"(l.s1), "+v"(l.sc), "+v"(x[0]) : "n"(BUT));
    else
        asm volatile("s_waitcnt lgkmcnt(%7)" : "+v"(l.m0), "+v"(l.m1), "+v"(l.s0), "+v"(l.s1), "+v"(l.sc), "+v"(x[0]), "+v"(x[1]) : "n"(BUT));
}
template <int BUT> __device__ __forceinline__ void iq_wait_tail(v4f (&d)[4]) {
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3]) : "n"(BUT));
}

template <bool GU, int NM>
__device__ __forceinline__ void pf_tile_iq2s(const PfGemm& a, uint8_t* b0, uint8_t* b1, uint8_t* b2, int ex, int row0, int nrows) {
    typedef const __attribute__((address_space(1))) uint8_t* wptr;
    typedef uint32_t w2 __attribute__((ext_vector_type(2)));
    constexpr int NMT = 2 * NM;
    wptr blob = (wptr) a.table[ex];
    const int tid = threadIdx.x, lane = tid & 63, ln = lane & 31, kh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nsb = (int) (a.k >> 8);
    const size_t qb = 4u * (size_t) nsb * 82u;   // bytes of a quad of rows

    wptr quad;
    int64_t n0;   // the wave's first feature (gate/up) or output row (down)
    if constexpr (GU) {
        n0 = (int64_t) blockIdx.x * 64 + wave * 16;
        quad = blob + a.off[ln >> 4] + (size_t) ((n0 + (ln & 15)) >> 2) * qb;
    } else {
        n0 = (int64_t) blockIdx.x * 128 + wave * 32;
        quad = blob + a.off[0] + (size_t) ((n0 + ln) >> 2) * qb;
    }
    const bool wave_on = n0 < a.n;   // (a.n is a multiple of the wave's rows: checked on the host)

    pf_v16f acc[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;

    PfDma<NMT> dma;
    dma.init(a, row0, nrows, wave, lane);
    dma.copy(b0, 0);
    if (nsb > 1) dma.copy(b1, 1);

    // The weights of a super-block, one ahead in registers: lane (ln, kh) of row ln loads the (index, sign) words and the
    // (high bits, scales) pairs of sub-blocks 4 kh .. 4 kh + 3, and one half-wave swap a pair of words then leaves every lane
    // with its own half - the entries 2 kh and 2 kh + 1, the group kh - of all eight.
    wptr pi = quad + 128 * kh + 8 * (ln & 3), ph = quad + 256 * (size_t) nsb + 32 * kh + 2 * (ln & 3),
         pd = quad + 320 * (size_t) nsb + 2 * (ln & 3);
    w2 is[4];
    uint32_t hs[4], dn;
    auto load_block = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i) is[i] = *(const __attribute__((address_space(1))) w2*) (pi + 32 * i);
#pragma unroll
        for (int i = 0; i < 4; ++i) hs[i] = *(const __attribute__((address_space(1))) uint16_t*) (ph + 8 * i);
        dn = *(const __attribute__((address_space(1))) uint16_t*) pd;
        pi += 256, ph += 64, pd += 8;
    };
    uint32_t v[8], g[8];   // a sub-block: the two index bytes, then the two sign bytes; the high bits << 11 and ls << 19
    float d = 0.0f;
    auto unpack = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const auto r = __builtin_amdgcn_permlane32_swap(__builtin_amdgcn_perm(is[i].y, is[i].x, 0x05040100u),
                                                            __builtin_amdgcn_perm(is[i].y, is[i].x, 0x07060302u), false, false);
            v[i] = r[0], v[4 + i] = r[1];
            const auto q = __builtin_amdgcn_permlane32_swap((hs[i] << 11) & 0x787800u, (hs[i] << 7) & 0x787800u, false, false);
            g[i] = q[0], g[4 + i] = q[1];
        }
        d = f16_bits_to_f32((uint16_t) dn);
    };
    if (wave_on) load_block();
    const int a_base = ln * 256, a_swz = ((ln & 15) ^ kh) << 4;   // (a lane's 16 codes of sub-block j: chunk 2 j + kh of the row)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (wave_on) unpack();

    auto step = [&](int sb, const uint8_t* buf, uint8_t* buf2) {   // super-block sb from buf; sb + 2 is copied into buf2
        if (wave_on && sb + 1 < nsb) load_block();
        // (after the weights' loads, so that waiting for everything but these copies covers the weights too)
        if (sb + 2 < nsb) dma.copy(buf2, sb + 2);
        if (wave_on) {
            const uint32_t lbuf = pf_lds_addr(buf);
            pf_v16i dot[NM][2];
            v4i xr[2][NM];
            IqLook lk[2];
            auto read_x = [&](int j, v4i (&dst)[NM]) {
                const uint32_t at = lbuf + a_base + (a_swz ^ ((2 * j) << 4));
                pf_for_m<0, NM>([&](auto mc) {
                    constexpr int m = decltype(mc)::value;
                    dst[m] = pf_lds_i32x4<m * 8192>(at);
                });
            };
            auto look = [&](int j, IqLook& o) {
                const uint32_t x = v[j], h = g[j];
                o.m0 = pf_lds_b64<kIqMags>(((x << 3) & 0x7f8u) | (h & 0x1800u));
                o.m1 = pf_lds_b64<kIqMags>(((x >> 5) & 0x7f8u) | ((h >> 2) & 0x1800u));
                o.s0 = pf_lds_b64<kIqSigns>((x >> 13) & 0x7f8u);
                o.s1 = pf_lds_b64<kIqSigns>((x >> 21) & 0x7f8u);
                o.sc = pf_lds_i32x4<kIqScales>((h >> 15) & 0xf0u);
            };
            v4f dxr[NM][4];
            look(0, lk[0]);
            read_x(0, xr[0]);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                IqLook& l = lk[j & 1];
                if (j < 7) {   // the next sub-block's look-ups go out under this one's arithmetic
                    look(j + 1, lk[(j + 1) & 1]);
                    read_x(j + 1, xr[(j + 1) & 1]);
                    iq_wait<5 + NM>(l, xr[j & 1]);
                } else {       // and the closing stage's block scales before the last one's
                    pf_for_m<0, NM>([&](auto mc) {
                        constexpr int m = decltype(mc)::value;
                        const uint32_t at = lbuf + 16 * kh;
                        dxr[m][0] = pf_lds_f32x4<kPfDOffNoS + m * 128>(at);
                        dxr[m][1] = pf_lds_f32x4<kPfDOffNoS + m * 128 + 32>(at);
                        dxr[m][2] = pf_lds_f32x4<kPfDOffNoS + m * 128 + 64>(at);
                        dxr[m][3] = pf_lds_f32x4<kPfDOffNoS + m * 128 + 96>(at);
                    });
                    iq_wait<4 * NM>(l, xr[j & 1]);
                }
                const uint32_t q[4] = {(uint32_t) (l.m0.x | l.s0.x), (uint32_t) (l.m0.y | l.s0.y), (uint32_t) (l.m1.x | l.s1.x), (uint32_t) (l.m1.y | l.s1.y)};
                v4i wl, wh;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    wl[i] = (int) __builtin_amdgcn_perm((uint32_t) l.sc[1], (uint32_t) l.sc[0], q[i]);
                    wh[i] = (int) __builtin_amdgcn_perm((uint32_t) l.sc[3], (uint32_t) l.sc[2], q[i]);
                }
#pragma unroll
                for (int m = 0; m < NM; ++m) {
                    const pf_v16i z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
                    dot[m][0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xr[j & 1][m], wl, j ? dot[m][0] : z, 0, 0, 0);
                    dot[m][1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xr[j & 1][m], wh, j ? dot[m][1] : z, 0, 0, 0);
                }
            }
            // once a block: lo + 256 hi = the block's integer sum, times the two block scales (blocks of 8 rows past the tile's
            // last row are skipped)
            pf_for_m<0, NM>([&](auto mc) {
                constexpr int m = decltype(mc)::value;
                iq_wait_tail<4 * (NM - 1 - m)>(dxr[m]);
                const int nb = (nrows - 32 * m + 7) >> 3;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    if (b < nb) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int i = 4 * b + r;
                            acc[m][i] = fmaf(__fmul_rn(dxr[m][b][r], d), (float) (dot[m][0][i] + 256 * dot[m][1][i]), acc[m][i]);
                        }
                    }
                }
            });
            if (sb + 1 < nsb) unpack();
        }
        // super-block sb + 1 has landed once only the wave's youngest NMT operations - this iteration's copies (of sb + 2), in the
        // last steps some of the nine weight loads, which `unpack` has waited for - may still be in flight; a wave that
        // holds no weight rows has nothing younger than its last copies then and waits for all
        if (sb + 2 < nsb || wave_on) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(NMT) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    for (int sb = 0; sb < nsb; sb += 3) {
        step(sb, b0, b2);
        if (sb + 1 < nsb) step(sb + 1, b1, b0);
        if (sb + 2 < nsb) step(sb + 2, b2, b1);
    }
    if (!wave_on) return;

    // outputs: lane (ln, kh) holds weight row ln for the tile's rows 32 m + 8 b + 4 kh + r (i = 4 b + r)
#pragma unroll
    for (int m = 0; m < NM; ++m) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int r = 32 * m + 8 * (i >> 2) + 4 * kh + (i & 3);
            const float val = __fmul_rn(acc[m][i], 0.125f);
            if constexpr (GU) {
                const float up = __shfl(val, (lane + 16) & 63, kWave);   // the up row of a feature sits 16 lanes above its gate row
                if (ln < 16 && r < nrows) a.out[(size_t) (row0 + r) * a.n + n0 + ln] = pf_swiglu(val, up, a.limit);
            } else {
                if (r < nrows) a.out[(size_t) (row0 + r) * a.n + n0 + ln] = val;
            }
        }
    }
}

// grid (bands of weight rows, tiles at most)
template <bool GU>
__global__ __launch_bounds__(256, 2) void prefill_iq2s_kernel(PfGemm a, Codebooks cb) {
    // ONE array, so that it starts at LDS address 0 and the tables' addresses need no base added (five additions a sub-block):
    // prefill_iq2s_lds_ok holds the built kernel against that before a launch
    __shared__ __attribute__((aligned(256))) uint8_t lds[kIqLdsBytes];
    uint8_t *tables = lds, *b0 = lds + kIqTables, *b1 = b0 + kPfBufBytesNoS, *b2 = b1 + kPfBufBytesNoS;
    const int tile = blockIdx.y;
    if (tile >= *a.plan.n_tiles) return;
    const int tid = threadIdx.x;
    // the magnitudes 8, 25, 43 as 0, 1, 2 (their bits 4 and 5)
#pragma unroll
    for (int i = 0; i < 4; ++i) ((uint64_t*) (tables + kIqMags))[tid + 256 * i] = (cb.iq2s[tid + 256 * i] >> 4) & 0x0303030303030303ull;
    {
        uint64_t m = 0ull;
#pragma unroll
        for (int b = 0; b < 8; ++b)
            if (tid & (1 << b)) m |= 4ull << (8 * b);
        ((uint64_t*) (tables + kIqSigns))[tid] = m;
    }
    if (tid < 16) {
        v4i e = {0, 0, 0, 0};
        const int mag[3] = {8, 25, 43};
#pragma unroll
        for (int i = 0; i < 6; ++i) {
            const int u = (2 * tid + 1) * (i < 3 ? mag[i] : -mag[i - 3]), lo = (int) (int8_t) (u & 255), hi = (u - lo) >> 8;
            const int at = 8 * (i % 3);
            e[i / 3] |= (lo & 255) << at;
            e[2 + i / 3] |= (hi & 255) << at;
        }
        ((v4i*) (tables + kIqScales))[tid] = e;
    }
    const int ex = a.plan.tile_expert[tile], row0 = a.plan.tile_row0[tile];
    const int nrows = min(kPfRows, a.plan.bounds[ex + 1] - row0);
    if (nrows <= 32) pf_tile_iq2s<GU, 1>(a, b0, b1, b2, ex, row0, nrows);
    else pf_tile_iq2s<GU, 2>(a, b0, b1, b2, ex, row0, nrows);
}
// Refuses a built kernel that has other LDS than its array (a second __shared__ object may be placed in front of it, and the
// tables would be read from the wrong addresses).  Asked of the runtime once a kernel.
template <bool GU>
static int prefill_iq2s_lds_ok(const char* what) {
    static std::atomic<size_t> bytes{0};
    if (bytes.load(std::memory_order_relaxed) == 0) {
        hipFuncAttributes at{};
        MAYA_HIP(hipFuncGetAttributes(&at, (const void*) prefill_iq2s_kernel<GU>));
        bytes.store(at.sharedSizeBytes, std::memory_order_relaxed);
    }
    const size_t got = bytes.load(std::memory_order_relaxed);
    if (got != (size_t) kIqLdsBytes) return fail(MAYA_E_UNSUPPORTED, "%s: the IQ2_S kernel was built with %zu bytes of LDS, its array has %d", what, got, kIqLdsBytes);
    return MAYA_OK;
}
