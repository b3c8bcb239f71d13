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
// one sub-block against the lane's codes y and their negation yn (unit_value's way with the signs), added to the lane's chain as
// row_dot adds it: d = activation scale
__device__ __forceinline__ float xxs_add(const u32x2 w, uint32_t db, const char* lds, const int (&y)[8], const int (&yn)[8], float d, float acc) {
    int s = 0;
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const uint2 g = *(const uint2*) (lds + ((l ? w.x >> (8 * l - 3) : w.x << 3) & 0x7f8u));
        const uint2 sl = *(const uint2*) (lds + 2048 + ((l ? w.y >> (7 * l - 3) : w.y << 3) & 0x3f8u));
        s = dot4((int) g.x, (int) __builtin_amdgcn_perm((uint32_t) yn[2 * l], (uint32_t) y[2 * l], sl.x), s);
        s = dot4((int) g.y, (int) __builtin_amdgcn_perm((uint32_t) yn[2 * l + 1], (uint32_t) y[2 * l + 1], sl.y), s);
    }
    const int isum = __mul24(2 * (int) (w.y >> 28) + 1, s);
    return fmaf(__fmul_rn(__fmul_rn(f16_bits_to_f32((uint16_t) db), 0.125f), d), (float) isum, acc);
}
// four rows' sub-blocks onto acc[B] ... acc[B + 3]; a lane past the row's last position (`on` false) adds nothing
template <int B, int ROWS>
__device__ __forceinline__ void xxs_rows(const RowsIQ2XXS& q, const int* lds, const int (&y)[8], const int (&yn)[8], float d, bool on, float (&acc)[ROWS]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float t = xxs_add(q.w[r], q.d[r], (const char*) lds, y, yn, d, acc[B + r]);
        acc[B + r] = on ? t : acc[B + r];
        asm volatile("" : "+v"(acc[B + r]));
        __builtin_amdgcn_sched_barrier(0);
    }
}

// ---- gate/up: a wave takes ROWS (gate row, up row) pairs, the gate rows on its lanes 0 .. 31, the up rows on 32 .. 63: lane l adds the
// sub-blocks l, l + 32, ... of a row up one behind the other, and 32 lanes meet at the end - gate_up_kernel's order, so that h is
// its h bit for bit.  Four waves a workgroup; grid (n_ff / (4 ROWS), entries).  The walk is 32 sub-blocks at a time over all ROWS
// pairs, so that a lane's activations of these are read and negated once, four rows' weights ahead.
// Bound by the LDS look-ups (8 of 8 bytes a sub-block of 8 bytes) and the vector instructions between them.  The general kernel gives
// 8 waves a row pair at a time with the activations read back from LDS for every row.  Layers with IQ2_S down, general / this: 6144 x
// 2048 top-8 of 160, one token 38.7 / 29.5 us, four 298 / 79.6, 16 875 / 278; 2816 x 1280 top-4, four tokens 61.9 / 25.6.  A form
// that gave a workgroup one row pair's positions side by side took 28.7, 86.0, 308 and 25.0, and summed in another order.
template <int ROWS, int MINW>
__global__ __launch_bounds__(256, MINW) void gate_up_iq2xxs_pos_kernel(maya_moe_args a, Codebooks cb) {
    static_assert(ROWS == 4 || ROWS == 8, "batches of four rows");
    __shared__ __align__(16) int lds[kFastXLdsWords];
    if (a.skip && *a.skip) return;
    const int e = (a.grp_ent && !a.grp_ptr) ? a.grp_ent[blockIdx.y] : (int) blockIdx.y;   // (the order of grp_ent: gate_up_iq2s_pos_kernel)
    if (e < 0) return;
    const uint64_t blob = a.plan_ptr[e];
    if (blob == 0ull) return;
    const int lane = threadIdx.x & 63, l = lane & 31, wave = __builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
    const bool is_up = lane >= 32;
    const int nu = a.layout.n_embd >> 5, nc = (nu + 31) >> 5;   // sub-blocks a row, steps of 32
    const int n_ff = a.layout.n_ff;
    const uint32_t r0 = (uint32_t) ((int) blockIdx.x * 4 + wave) * ROWS;
    const uint32_t rb = (uint32_t) (nu >> 3) * 66u;   // bytes of a row
    const uint64_t mat = blob + a.layout.gate_off;
    const uint32_t om = is_up ? (uint32_t) (a.layout.up_off - a.layout.gate_off) : 0u;
    // (a lane past the row's last position reads the last one's words)
    auto load = [&](int c, int b) {
        const uint32_t u = (uint32_t) min(32 * c + l, nu - 1), od = om + (u >> 3) * 66u;
        return load_xxs(mat, r0 + 4 * b, rb, od + 2u + 8u * (u & 7u), od);
    };
    const int tok = e / a.k;
    const int4* xq = (const int4*) (a.x.q + (size_t) tok * (32 * nu));
    const float* xd = a.x.d + (size_t) tok * nu;
    RowsIQ2XXS nxt = load(0, 0);
    int4 ya = xq[2 * min(l, nu - 1)], yb = xq[2 * min(l, nu - 1) + 1];
    float dn = xd[min(l, nu - 1)];
    stage_iq2xxs_tables<256>(lds, cb);
    __syncthreads();
    float acc[ROWS];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) acc[i] = 0.0f;
#pragma unroll 1
    for (int c = 0; c < nc; ++c) {
        const bool on = 32 * c + l < nu, more = c + 1 < nc;
        const int y[8] = {ya.x, ya.y, ya.z, ya.w, yb.x, yb.y, yb.z, yb.w};
        const float d = dn;
        if (more) {
            const int u = min(32 * (c + 1) + l, nu - 1);
            ya = xq[2 * u], yb = xq[2 * u + 1];
            dn = xd[u];
        }
        int yn[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) yn[i] = neg4(y[i]);
        if constexpr (ROWS == 8) {
            const RowsIQ2XXS cur = nxt;
            nxt = load(c, 1);
            xxs_rows<0>(cur, lds, y, yn, d, on, acc);
        }
        const RowsIQ2XXS cur = nxt;
        if (more) nxt = load(c + 1, 0);
        xxs_rows<ROWS - 4>(cur, lds, y, yn, d, on, acc);
    }
    float g;
    if constexpr (ROWS == 8) g = reduce8_half(acc, lane);
    else g = reduce4_half(acc, lane);
    const float up = xor_lane<32>(g);
    constexpr int each = 32 / ROWS;   // lanes that hold a row's sum
    if (lane < 32 && lane % each == 0) a.h[(size_t) e * n_ff + r0 + lane / each] = swiglu(g, up, a.limit);
}

}  // namespace maya
