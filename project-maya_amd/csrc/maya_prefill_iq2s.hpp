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
// Tiles of up to 128 rows keep a super-block's planes for their row groups, as Q4_K's do: the look-ups and the 200 vector
// instructions of a decode are paid once.  1187 tokens top-8 of 256 experts of 7168 x 2048 under a skewed routing, gate/up 1388 -> 1232
// us; 75 tokens of 160 experts of 6144 x 1536, where every tile has one group, 340 and 335.
// Chunks of few rows an expert run on a form of one group of 32 rows, of which a compute unit holds three workgroups instead of two
// (prefill_iq2s_few_kernel).  What bounds that one is LDS, busy 76 to 80 % of the cycles, 46 % of that with bank conflicts of the sign and digit
// look-ups, which come at random.  What bounds the form of up to 128 rows: vector instructions (46 to 56 % of the cycles) and the matrix
// instructions (27 to 35 %), which a SIMD's two waves overlap little.
constexpr int kIqMags = 0, kIqSigns = 8192, kIqScales = kIqSigns + 2048, kIqTables = kIqScales + 256;   // byte offsets in LDS

// A quad of rows (the stream packing's unit) holds, a super-block, 256 bytes of (index, sign) words [sub-block][row], 64 of (high
// bits, scales) pairs [sub-block][row] and 8 of block scales [row]: three copies of a wave's eight quads.  The words' 16-byte
// pieces sit in LDS at their index ^ twice the quad, so that a sub-block's words of 32 rows meet every bank once.
template <bool GU, int RING = 4> struct PfIq2s {
    static constexpr bool kSums = false;
    static constexpr int kLdsAt = kIqTables, kStep = 2048 + 512 + 64 + 192, kWave = 2 * kStep;   // (multiples of 256: addresses below are xor-ed)
    static constexpr int kMats = GU ? 2 : 1, kQuads = 8 / kMats, kCopies = GU ? 6 : 5, kOneGroupBut = 2 + kCopies, kRing = RING;
    static constexpr int kHiFactor = 256, kLook = 5;
    static constexpr float kOutFactor = 0.125f;
    __amdgpu_buffer_rsrc_t r[kMats];
    uint32_t wat[2], pat[kMats == 2 ? 1 : 2], sat, ix_at, pair_sel, word_sel;
    int lane, nsb;
    __device__ __forceinline__ void init(const PfGemm& a, const uint8_t* blob, int64_t n0, int lane_) {
        lane = lane_;
        nsb = (int) (a.k >> 8);
        const int qb = 4 * nsb * 82;   // bytes of a quad
#pragma unroll
        for (int m = 0; m < kMats; ++m)
            r[m] = __builtin_amdgcn_make_buffer_rsrc((void*) (blob + a.off[m] + (size_t) (n0 >> 2) * (size_t) qb), 0, kQuads * qb, 0x00020000);
#pragma unroll
        for (int i = 0; i < 2; ++i)   // the words of quads 4 i .. 4 i + 3 (gate/up: of either matrix its four)
            wat[i] = (uint32_t) (((GU ? 0 : 4 * i) + (lane >> 4)) * qb + (((lane & 15) ^ (2 * (4 * i + (lane >> 4)))) * 16));
#pragma unroll
        for (int i = 0; i < 2 / kMats; ++i)   // the pairs of quads 4 i ..., two rows a word, as [rows][sub-block]
            pat[i] = (uint32_t) ((4 * i + (lane >> 4)) * qb + 256 * nsb + (lane & 7) * 8 + ((lane >> 3) & 1) * 4);
        sat = (uint32_t) ((lane >> 1) * qb + 320 * nsb + (lane & 1) * 4);
        const int ln = lane & 31, kh = lane >> 5, quad = ln >> 2, row = ln & 3;
        ix_at = quad * 256 + (row & 1) * 8 + (((row >> 1) ^ (2 * quad)) * 16);
        pair_sel = row & 1 ? 0x07030602u : 0x05010400u;   // of two sub-blocks' words: the row's high bits, its scales
        word_sel = kh ? 0x07060302u : 0x05040100u;     // the half of the index word, the half of the sign word
    }
    __device__ __forceinline__ void copy(pf_lds8 to, int sb) const {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r[GU ? i : 0], (pf_lptr) (to + i * 1024), 16, wat[i], sb * 256, 0, 0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(r[GU ? i : 0], (pf_lptr) (to + 2048 + i * 256), 4, pat[GU ? 0 : i], sb * 64, 0, 0);
        // (the lane number is hidden from the compiler: it would follow one `if` into the next, merge copies of different places and
        // pick their LDS address by lane, which has to be the same for the wave)
        int l = lane;
        asm volatile("" : "+v"(l));
        if (l < 2 * kQuads) {
#pragma unroll
            for (int m = 0; m < kMats; ++m)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r[m], (pf_lptr) (to + 2560 + m * 32), 4, sat, sb * 8, 0, 0);
        }
    }
    __device__ __forceinline__ void first(pf_lds8 to) const {
        copy(to, 0);
        if (nsb > 1) copy(to + kStep, 1);
    }
    // super-block sb is in registers: its LDS takes the super-block after the next one's
    __device__ __forceinline__ void next(pf_lds8 to, int sb) const {
        if (sb + 2 < nsb) copy(to + (sb & 1) * kStep, sb + 2);
    }
    struct Look {   // the LDS look-ups of one sub-block: selectors and signs of the lane's two grid entries, its group's digits
        pf_i2 m0, m1, s0, s1;
        v4i sc;     // the low digits of +{8, 25, 43}, of -{8, 25, 43}, then the high ones
    };
    struct Row {
        pf_i2 is[8];
        v4i hs[2];
        uint32_t dw;
        float d;
        uint32_t v[8];             // a sub-block: the lane's two index bytes, then its two sign bytes
        uint32_t e0[2], e1[2], sc[2];   // a byte a sub-block: the two entries' high bits, 16 ls
        Look lk[2];
    };
    __device__ __forceinline__ void read(Row& w, uint32_t base, int sb) const {
        base += (sb & 1) * kStep;
        const uint32_t at = base + ix_at;
#pragma unroll
        for (int j = 0; j < 8; ++j) w.is[j] = pf_lds_b64<0>(at ^ (32 * j));
        const uint32_t pt = base + ((lane & 31) >> 1) * 32;
        w.hs[0] = pf_lds_i32x4<2048>(pt);
        w.hs[1] = pf_lds_i32x4<2048 + 16>(pt);
        asm volatile("ds_read_u16 %0, %1 offset:2560" : "=v"(w.dw) : "v"(base + 2 * (lane & 31)) : "memory");
    }
    template <int BUT> __device__ __forceinline__ void wait(Row& w) const {
        asm volatile("s_waitcnt lgkmcnt(%11)"
                     : "+v"(w.is[0]), "+v"(w.is[1]), "+v"(w.is[2]), "+v"(w.is[3]), "+v"(w.is[4]), "+v"(w.is[5]), "+v"(w.is[6]), "+v"(w.is[7]),
                       "+v"(w.hs[0]), "+v"(w.hs[1]), "+v"(w.dw)
                     : "n"(BUT));
    }
    __device__ __forceinline__ void open(Row& w) const {
        const int kh = lane >> 5;
#pragma unroll
        for (int j = 0; j < 8; ++j) w.v[j] = __builtin_amdgcn_perm((uint32_t) w.is[j].y, (uint32_t) w.is[j].x, word_sel);
#pragma unroll
        for (int i = 0; i < 2; ++i) {   // (four sub-blocks' high bits, two an entry, and scales, four bits a group, as bytes of a word each)
            const uint32_t a = __builtin_amdgcn_perm((uint32_t) w.hs[i].y, (uint32_t) w.hs[i].x, pair_sel);
            const uint32_t b = __builtin_amdgcn_perm((uint32_t) w.hs[i].w, (uint32_t) w.hs[i].z, pair_sel);
            const uint32_t h = __builtin_amdgcn_perm(b, a, 0x05040100u) >> (4 * kh), l = __builtin_amdgcn_perm(b, a, 0x07060302u);
            w.e0[i] = h & 0x03030303u;
            w.e1[i] = (h >> 2) & 0x03030303u;
            w.sc[i] = (l << (4 - 4 * kh)) & 0xf0f0f0f0u;
        }
        w.d = f16_bits_to_f32((uint16_t) w.dw);
    }
    template <int J> __device__ __forceinline__ void look(Row& w) const {
        constexpr int b = J & 3;   // (an entry's 10-bit index: its byte, and the high bits' byte behind it)
        const uint32_t x = w.v[J];
        Look& o = w.lk[J & 1];
        o.m0 = pf_lds_b64<kIqMags>(__builtin_amdgcn_perm(w.e0[J >> 2], x, 0x0c0c0400u + 0x100u * b) << 3);
        o.m1 = pf_lds_b64<kIqMags>(__builtin_amdgcn_perm(w.e1[J >> 2], x, 0x0c0c0401u + 0x100u * b) << 3);
        o.s0 = pf_lds_b64<kIqSigns>((x >> 13) & 0x7f8u);
        o.s1 = pf_lds_b64<kIqSigns>((x >> 21) & 0x7f8u);
        o.sc = pf_lds_i32x4<kIqScales>((w.sc[J >> 2] >> (8 * b)) & 0xf0u);
    }
    template <int BUT> __device__ __forceinline__ void wait_look(int j, Row& w, v4i& x) const {
        Look& l = w.lk[j & 1];
        asm volatile("s_waitcnt lgkmcnt(%6)" : "+v"(l.m0), "+v"(l.m1), "+v"(l.s0), "+v"(l.s1), "+v"(l.sc), "+v"(x) : "n"(BUT));
    }
    __device__ __forceinline__ void planes(const Row& w, int j, v4i& wl, v4i& wh) const {
        const Look& l = w.lk[j & 1];
        const uint32_t q[4] = {(uint32_t) (l.m0.x | l.s0.x), (uint32_t) (l.m0.y | l.s0.y), (uint32_t) (l.m1.x | l.s1.x), (uint32_t) (l.m1.y | l.s1.y)};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            wl[i] = (int) __builtin_amdgcn_perm((uint32_t) l.sc[1], (uint32_t) l.sc[0], q[i]);
            wh[i] = (int) __builtin_amdgcn_perm((uint32_t) l.sc[3], (uint32_t) l.sc[2], q[i]);
        }
    }
};
// tables, the activations' ring (the sums' place in a slot stays empty, as the weights have no minimums), the weights [4 waves][2]
constexpr int kIqLdsBytes = 70912;
static_assert(kIqLdsBytes == PfLds<PfIq2s<true>>::bytes && kIqLdsBytes == PfLds<PfIq2s<false>>::bytes);
static_assert(kIqLdsBytes <= 80 * 1024, "two workgroups a compute unit");

__device__ __forceinline__ void pf_iq2s_tables(uint8_t* tables, const Codebooks& cb, int tid) {
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
}

// The kernels' LDS is ONE array, so that it starts at LDS address 0 and the tables' addresses need no base added (five additions a
// sub-block): prefill_iq2s_lds_ok holds the built kernels against that before a launch.
// grid (bands of weight rows, items or tiles at most)
template <bool GU>
__global__ __launch_bounds__(256, 2) void prefill_iq2s_kernel(PfGemm a, Codebooks cb) {
    __shared__ __attribute__((aligned(256))) uint8_t lds[kIqLdsBytes];
    PfTile t;
    if (!pf_my_rows(a, t)) return;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));   // (nothing made of it for the tables stays in a register)
    pf_iq2s_tables(lds, cb, tid);   // (the tile's first barrier is in front of the first look-up)
    typedef PfIq2s<GU> W;
    if (t.nrows <= 32) pf_tile<W, GU, 1>(a, (pf_lds8) lds, t);
    else if (t.nrows <= 64) pf_tile<W, GU, 2>(a, (pf_lds8) lds, t);
    else if (t.nrows <= 96) pf_tile<W, GU, 3>(a, (pf_lds8) lds, t);
    else pf_tile<W, GU, 4>(a, (pf_lds8) lds, t);
}
// Chunks of few rows an expert: one group of 32 rows at a time, in registers and LDS that leave room for three workgroups a
// compute unit, as the look-ups, the vector instructions and the matrix instructions take turns with two (LDS busy 57 % of the cycles, vector issue
// 44 %, matrix cores 23 %).  75 tokens of 160 experts of 6144 x 1536 530 -> 483 us, 17 tokens 321 -> 293, with 10.3 waves a compute unit
// where there were 7.1.  An item of more than 32 rows decodes its weights once a group.
constexpr int kIqFewRing = 2, kIqFewLdsBytes = PfLds<PfIq2s<true, kIqFewRing>>::bytes;
static_assert(kIqFewLdsBytes == PfLds<PfIq2s<false, kIqFewRing>>::bytes && kIqFewLdsBytes <= 160 * 1024 / 3, "three workgroups a compute unit");
template <bool GU>
__global__ __launch_bounds__(256, 3) void prefill_iq2s_few_kernel(PfGemm a, Codebooks cb) {
    __shared__ __attribute__((aligned(256))) uint8_t lds[kIqFewLdsBytes];
    PfTile t;
    if (!pf_my_rows<false>(a, t)) return;
    pf_iq2s_tables(lds, cb, threadIdx.x);
    typedef PfIq2s<GU, kIqFewRing> W;
    for (int r = 0; r < t.nrows; r += 32) {
        if (r) __syncthreads();   // (the copies of these rows go where the others may still be read)
        pf_tile<W, GU, 1>(a, (pf_lds8) lds, {t.blob, t.row0 + r, min(32, t.nrows - r)});
    }
}
// Refuses a built kernel that has other LDS than its array (a second __shared__ object may be placed in front of it, and the
// tables would be read from the wrong addresses).  Asked of the runtime once a kernel.
template <void (*KERNEL)(PfGemm, Codebooks), int BYTES>
static int prefill_iq2s_kernel_lds_ok(const char* what) {
    static std::atomic<size_t> bytes{0};
    if (bytes.load(std::memory_order_relaxed) == 0) {
        hipFuncAttributes at{};
        MAYA_HIP(hipFuncGetAttributes(&at, (const void*) KERNEL));
        bytes.store(at.sharedSizeBytes, std::memory_order_relaxed);
    }
    const size_t got = bytes.load(std::memory_order_relaxed);
    if (got != (size_t) BYTES) return fail(MAYA_E_UNSUPPORTED, "%s: an IQ2_S kernel was built with %zu bytes of LDS, its array has %d", what, got, BYTES);
    return MAYA_OK;
}
static int prefill_iq2s_lds_ok(const char* what) {
    int rc = prefill_iq2s_kernel_lds_ok<prefill_iq2s_kernel<true>, kIqLdsBytes>(what);
    if (!rc) rc = prefill_iq2s_kernel_lds_ok<prefill_iq2s_kernel<false>, kIqLdsBytes>(what);
    if (!rc) rc = prefill_iq2s_kernel_lds_ok<prefill_iq2s_few_kernel<true>, kIqFewLdsBytes>(what);
    if (!rc) rc = prefill_iq2s_kernel_lds_ok<prefill_iq2s_few_kernel<false>, kIqFewLdsBytes>(what);
    return rc;
}
// Whether a chunk's IQ2_S products run on the kernel for few rows an expert.  The host does not know the routing: an expert has 8 rows at most on
// average, and the tokens are few enough that one which nearly all of them take, which this kernel decodes once a 32 of them, costs no more
// than the others save.  Microseconds a layer call, kernel of 128 rows / this one, routing even, skewed by 0.6 and by 1.1:
//   160 experts of 6144 x 1536 top-8, 75 tokens 520 / 485, 391 / 375, 233 / 224;  90 tokens 538 / 496, 423 / 402, 251 / 254;  110 tokens 537 / 497,
//   465 / 440, 272 / 271;  top-4, 128 tokens by 0.6 342 / 330, by 1.1 168 / 164;  top-1, 250 tokens 195 / 183, 120 / 116;
//   256 of 7168 x 2048 top-8, 80 tokens by 0.6 702 / 656, by 1.1 347 / 348;  80 of 7168 x 2048, 80 tokens 415 / 395, 317 / 320;
//   256 of 4096 x 2048 top-8, 110 tokens 470 / 447, 244 / 247;  top-2, 250 tokens 281 / 271, 117 / 112;
//   288 of 4096 x 1024 top-10, 88 tokens 275 / 264, 158 / 152;  64 of 3072 x 1536 top-6, 64 tokens 131 / 123, 131 / 121, 97 / 92
// With more tokens even routing gains as much, but a skewed one loses: 160 experts of 6144 x 1536 top-8, 120 tokens by 1.1 276 / 288, 160 tokens
// 554 / 510, 513 / 497, 320 / 332;  top-4, 220 tokens by 1.1 208 / 215;  top-1, 512 tokens 132 / 138;  256 of 4096 x 2048 top-8, 256 tokens
// 774 / 712, 680 / 653, 355 / 376.
static bool prefill_iq2s_few(int n_tokens, int n_entries, int n_expert) {
    return n_entries <= 8 * n_expert && n_tokens <= (n_entries <= 512 ? 256 : 112);
}
template <bool GU>
static void prefill_iq2s_launch(const PfGemm& a, const Codebooks& cb, dim3 grid, hipStream_t s) {
    if (a.work.few) hipLaunchKernelGGL(prefill_iq2s_few_kernel<GU>, grid, dim3(256), 0, s, a, cb);
    else hipLaunchKernelGGL(prefill_iq2s_kernel<GU>, grid, dim3(256), 0, s, a, cb);
}
