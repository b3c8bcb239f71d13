// maya_fastx.hpp - the position-mapped gate/up kernel for IQ2_XXS rows, in their GGUF order (the type has no stream packing: a block
// of 256 values is a scale and 8 bytes a sub-block, so eight lanes' words are 64 bytes in a row and a wave's load one run of bytes).
#pragma once

namespace maya {

typedef u32x2 __attribute__((aligned(2))) u32x2_a2;
typedef const __attribute__((address_space(1))) u32x2_a2* gptr64_a2;

// LDS: [0, 512) words the codebook, [512, 768) the v_perm_b32 selectors of the 128 sign indices (store_iq2s_selectors; bit 7 is the
// parity of the seven)
constexpr int kFastXLdsWords = 512 + 256;
template <int NT>
__device__ __forceinline__ void stage_iq2xxs_tables(int* lds, const Codebooks& cb) {
    TablePieces<512, NT> t;
    table_request(cb.iq2xxs, t);
    for (int j = threadIdx.x; j < 128; j += NT) {
        const uint32_t i = Fmt<kIQ2_XXS>::signs8((uint32_t) j);
        uint32_t lo = 0x03020100u, hi = 0x03020100u;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            if (i & (1u << b)) lo |= 4u << (8 * b);
            if (i & (16u << b)) hi |= 4u << (8 * b);
        }
        lds[512 + 2 * j] = (int) lo;
        lds[512 + 2 * j + 1] = (int) hi;
    }
    table_store(lds, t);
}
// one lane's sub-block of four rows: index word and sign word, FP16 scale
struct RowsIQ2XXS {
    u32x2 w[4];
    uint32_t d[4];
};
// (the row's address stays in scalar registers and the lane's offset a 32-bit one: left to itself the compiler keeps a 64-bit address a
// lane for each of the eight loads)
__device__ __forceinline__ RowsIQ2XXS load_xxs(uint64_t mat, uint32_t row0, uint32_t rb, uint32_t ow, uint32_t od) {
    RowsIQ2XXS q;
    asm volatile("" : "+v"(ow), "+v"(od));
    uint64_t p = mat + (uint64_t) row0 * rb;
#pragma unroll
    for (int i = 0; i < 4; ++i, p += rb) {
        asm("" : "+s"(p));
        const gptr8 row = (gptr8) p;
        q.w[i] = *(gptr64_a2) (row + ow);
        q.d[i] = gld16(row + od);
    }
    return q;
}
// one sub-block against the lane's codes y and their negation yn (unit_value's way with the signs); dy8 = activation scale / 8
__device__ __forceinline__ float xxs_value(const u32x2 w, uint32_t d, const char* lds, const int (&y)[8], const int (&yn)[8], float dy8) {
    int s = 0;
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const uint2 g = *(const uint2*) (lds + ((l ? w.x >> (8 * l - 3) : w.x << 3) & 0x7f8u));
        const uint2 sl = *(const uint2*) (lds + 2048 + ((l ? w.y >> (7 * l - 3) : w.y << 3) & 0x3f8u));
        s = dot4((int) g.x, (int) __builtin_amdgcn_perm((uint32_t) yn[2 * l], (uint32_t) y[2 * l], sl.x), s);
        s = dot4((int) g.y, (int) __builtin_amdgcn_perm((uint32_t) yn[2 * l + 1], (uint32_t) y[2 * l + 1], sl.y), s);
    }
    const int isum = __mul24(2 * (int) (w.y >> 28) + 1, s);
    return __fmul_rn(__fmul_rn(f16_bits_to_f32((uint16_t) d), dy8), (float) isum);
}
template <int B>
__device__ __forceinline__ void xxs_values(const RowsIQ2XXS& q, const int* lds, const int (&y)[8], const int (&yn)[8], float dy8, float (&acc)[8]) {
#define MAYA_ROW(R)                                                              \
    acc[B + R] = xxs_value(q.w[R], q.d[R], (const char*) lds, y, yn, dy8);       \
    asm volatile("" : "+v"(acc[B + R]));                                         \
    __builtin_amdgcn_sched_barrier(0);
    MAYA_ROW(0) MAYA_ROW(1) MAYA_ROW(2) MAYA_ROW(3)
#undef MAYA_ROW
}

// ---- gate/up: gate_up_iq2s_pos_kernel's split - a workgroup of NW waves = 2 * 32 NW lanes for the sub-block positions of a (gate
// row, up row) pair, ROWS pairs, four rows ahead; grid (n_ff / ROWS, entries).  A lane past the row's last position reads the last
// one's words and has zero codes and scales.
// Bound by the LDS look-ups (8 of 8 bytes a sub-block of 8 bytes).  The general kernel gave 8 waves a row pair at a time with the
// activations read back from LDS for every row, and took 241 us where this one takes 51 (four tokens of 160 experts top-8, 6144 x 2048,
// 188 MB); the layer with IQ2_S down 268 -> 77.6, one token 37.5 -> 27.7, 16 tokens 683 -> 275, 2816 x 1280 four tokens 107.7 -> 34.6.
template <int NW, int ROWS, int MINW, bool FIT>
__global__ __launch_bounds__(64 * NW, MINW) void gate_up_iq2xxs_pos_kernel(maya_moe_args a, Codebooks cb) {
    static_assert(ROWS % 8 == 0, "a batch is eight rows");
    constexpr int NU = 32 * NW;
    __shared__ __align__(16) int lds[kFastXLdsWords];
    __shared__ float part[2][2 * NW][8];
    if (a.skip && *a.skip) return;
    const int e = (a.grp_ent && !a.grp_ptr) ? a.grp_ent[blockIdx.y] : (int) blockIdx.y;   // (the order of grp_ent: gate_up_iq2s_pos_kernel)
    if (e < 0) return;
    const uint64_t blob = a.plan_ptr[e];
    if (blob == 0ull) return;
    const int t = threadIdx.x, lane = t & 63, hw = t >> 5;
    const bool is_up = t >= NU;
    const int nu = FIT ? NU : a.layout.n_embd >> 5, lu = is_up ? t - NU : t;   // sub-blocks a row; the lane's position among 32 NW
    const bool on = FIT || lu < nu;
    const int u = on ? lu : nu - 1;
    const int n_ff = a.layout.n_ff, r0 = blockIdx.x * ROWS;
    const uint32_t rb = (uint32_t) (nu >> 3) * 66u;   // bytes of a row
    const uint64_t mat = blob + a.layout.gate_off;
    const uint32_t od = (is_up ? (uint32_t) (a.layout.up_off - a.layout.gate_off) : 0u) + (uint32_t) (u >> 3) * 66u;
    const uint32_t ow = od + 2u + 8u * (uint32_t) (u & 7);
    RowsIQ2XXS nxt = load_xxs(mat, (uint32_t) r0, rb, ow, od);
    stage_iq2xxs_tables<64 * NW>(lds, cb);
    const int tok = e / a.k;
    int y[8];
    {
        const int4* q = (const int4*) (a.x.q + (size_t) tok * (32 * nu));
        const int4 ya = q[2 * u], yb = q[2 * u + 1];
        y[0] = ya.x, y[1] = ya.y, y[2] = ya.z, y[3] = ya.w, y[4] = yb.x, y[5] = yb.y, y[6] = yb.z, y[7] = yb.w;
    }
    float dy8 = a.x.d[(size_t) tok * nu + u] * 0.125f;
    idle_lane_zero(on, y, dy8);
    int yn[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) yn[i] = neg4(y[i]);
    __syncthreads();
    float acc[8];
#pragma unroll 1
    for (int r = 0; r < ROWS; r += 8) {
        {
            const RowsIQ2XXS cur = nxt;
            nxt = load_xxs(mat, (uint32_t) (r0 + r + 4), rb, ow, od);
            xxs_values<0>(cur, lds, y, yn, dy8, acc);
        }
        {
            const RowsIQ2XXS cur = nxt;
            if (r + 8 < ROWS) nxt = load_xxs(mat, (uint32_t) (r0 + r + 8), rb, ow, od);
            xxs_values<4>(cur, lds, y, yn, dy8, acc);
        }
        if constexpr (!FIT) {   // (an idle lane's weights are another's: a scale that is not a number stays out)
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] = on ? acc[i] : 0.0f;
        }
        const float v = reduce8_half(acc, lane);
        const int buf = (r >> 3) & 1;
        if ((lane & 3) == 0) part[buf][hw][(lane >> 2) & 7] = v;
        __syncthreads();
        if (t < 8) {
            float g = part[buf][0][t], up = part[buf][NW][t];
#pragma unroll
            for (int w = 1; w < NW; ++w) {
                g += part[buf][w][t];
                up += part[buf][NW + w][t];
            }
            if (r0 + r + t < n_ff) a.h[(size_t) e * n_ff + r0 + r + t] = swiglu(g, up, a.limit);
        }
    }
}

}  // namespace maya
