// maya_exl3.hip - EXL3 (exllamav3 trellis) routed experts on gfx950: decode mat-vec kernels and their C ABI.
//
// A workgroup owns 128 output columns (one block of the output Hadamard transform): its 8 waves take one 16-column
// tile each and walk down the k / 16 row tiles.  For a tile a lane decodes 4 consecutive trellis steps - by the tile's
// element order (include/strata/kernels/exl3.hpp:15-16) those are 4 rows of ONE column - and multiplies them with the
// rotated, FP16-rounded activation held in LDS; the rotation H(x * suh) is done by the workgroup itself before the walk
// and the output rotation, the svh scaling, the SwiGLU and the FP32 stores after it.  Several activations (a verify
// window's tokens routed to one expert) share one decode of the weights.
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <math.h>
#include <stdint.h>

#include <type_traits>

#include "maya_host.h"
#include "maya_dev.hpp"
#include "maya_groups.hpp"
#include "maya_route.hpp"

namespace maya {

constexpr int kExThreads = 512;

// ---- codebooks: the value of a 16-bit state, as the FP16 bits the format defines (src/kernels/cpu/exl3_ref.cpp:11-27)
template <int CB>
__device__ __forceinline__ __half exl3_value(uint32_t state) {
    if constexpr (CB == 2) {
        // fp16(1024 + bytesum(state * 0x83DCD12D)) * fp16(0x1eee) + fp16(0xc931) in one FP16 FMA
        const uint32_t x = state * 0x83DCD12Du;
        const uint32_t bs = __builtin_amdgcn_sad_u8(x, 0u, 1024u);   // 1024 + the sum of the four bytes
        const __half h = __ushort2half_rn((unsigned short) bs);      // exact: an integer below 2048
        return __hfma(h, __ushort_as_half(0x1eee), __ushort_as_half(0xc931));
    } else {
        uint32_t x = CB == 1 ? state * 0xCBAC1FEDu : state * 89226354u + 64248484u;
        x = (x & 0x8fff8fffu) ^ 0x3b603b60u;
        return __hadd(__ushort_as_half((unsigned short) (x & 0xffffu)), __ushort_as_half((unsigned short) (x >> 16)));
    }
}

// step p's state of a tile whose 4 * k2 words are in t[] (LDS or registers): the 16-bit window that ends at bit
// floor((p + 1) k2 / 2) of the words read MSB-first, around the ring (src/kernels/cpu/exl3_ref.cpp:33-43)
__device__ __forceinline__ uint32_t exl3_state(const uint32_t* t, int k2, int p) {
    const int W = 4 * k2;
    const int e = ((p + 1) * k2) >> 1;            // the window's end bit, 1 .. 128 k2
    const int i1 = (e - 1) >> 5;                  // the word of its last bit
    const int i0 = e < 16 ? W - 1 : (e - 16) >> 5;  // ... of its first bit (before bit 0: the ring's last word)
    const int sh = ((i1 + 1) << 5) - e;
    const uint64_t m = ((uint64_t) t[i0] << 32) | (uint64_t) t[i1];
    return (uint32_t) (m >> sh) & 0xffffu;
}

// tile step p -> (row, column) inside the 16 x 16 tile (src/kernels/cpu/exl3_ref.cpp:52-55)
__device__ __forceinline__ void exl3_rc(int p, int& r, int& c) {
    const int lane = p >> 3, j = p & 7;
    r = (lane & 3) * 2 + (j & 1) + 8 * ((j >> 1) & 1);
    c = (lane >> 2) + 8 * (j >> 2);
}

template <int CB>
__global__ __launch_bounds__(256) void exl3_inner_kernel(const uint32_t* __restrict__ trellis, int64_t k, int64_t n, int k2,
                                                         uint16_t* __restrict__ dst) {
    __shared__ uint32_t t[64];
    const int64_t tiles_n = n >> 4;
    const int64_t tile = blockIdx.x;
    const int W = 4 * k2;
    if ((int) threadIdx.x < W) t[threadIdx.x] = trellis[tile * W + threadIdx.x];
    __syncthreads();
    const int p = threadIdx.x;
    int r, c;
    exl3_rc(p, r, c);
    const __half v = exl3_value<CB>(exl3_state(t, k2, p));
    const int64_t ks = tile / tiles_n, tc = tile % tiles_n;
    dst[(ks * 16 + r) * n + tc * 16 + c] = __half_as_ushort(v);
}

// ---- the blockwise Hadamard transform H / sqrt(128) of one 128-value block inside a wave: lane L holds values L and L + 64.
// Stage h < 64 pairs lane L with lane L ^ h (the lower index adds, the upper takes lower - upper), stage 64 pairs the
// lane's own two values: the butterflies, their order and every rounding are the reference's
// (src/kernels/cpu/exl3_ref.cpp:61-75), so the same bits.
// The partner's value comes through a DPP operand, a swizzle or the half-wave swap (xor_lane), not through __shfl_xor's
// LDS-routed permute: six exchanges a value, each of which was an LDS round trip.
template <int H>
__device__ __forceinline__ void had128_stage(float& v0, float& v1, int lane) {
    const float p0 = xor_lane<H>(v0), p1 = xor_lane<H>(v1);
    const bool upper = (lane & H) != 0;
    v0 = upper ? __fsub_rn(p0, v0) : __fadd_rn(v0, p0);
    v1 = upper ? __fsub_rn(p1, v1) : __fadd_rn(v1, p1);
}
__device__ __forceinline__ void had128_wave(float& v0, float& v1, int lane) {
    had128_stage<1>(v0, v1, lane);
    had128_stage<2>(v0, v1, lane);
    had128_stage<4>(v0, v1, lane);
    had128_stage<8>(v0, v1, lane);
    had128_stage<16>(v0, v1, lane);
    had128_stage<32>(v0, v1, lane);
    const float a = v0, c = v1;
    v0 = __fadd_rn(a, c);
    v1 = __fsub_rn(a, c);
    const float s = 1.0f / sqrtf(128.0f);
    v0 = __fmul_rn(v0, s);
    v1 = __fmul_rn(v1, s);
}

// xr = FP16(H(x * suh)) of one activation into LDS; every wave of the workgroup takes blocks of 128 values, transformed in registers
// PAIRED (the compile-time walk): inside every 16 rows the word of rows 2q, 2q + 1 and the word of rows 2q + 8, 2q + 9 -
// a lane's four rows - sit side by side (words 2q, 2q + 1), so the walk reads them in one 8-byte LDS read
__device__ __forceinline__ int paired_pos(int i) {
    const int w = (i >> 1) & 7;
    return (i & ~15) | ((w < 4 ? 2 * w : 2 * (w - 4) + 1) << 1) | (i & 1);
}
template <bool PAIRED>
__device__ __forceinline__ void rotate_in(const float* __restrict__ x, const uint16_t* __restrict__ suh, int k, __half* xr) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int nb = k >> 7;
    // a wave's blocks three at a time: their loads go out together (one block a pass of the loop is one trip to memory a
    // pass: the compiler waits for a pass's loads before it issues the next pass's)
    constexpr int kAtOnce = 3, kWaves = kExThreads / 64;
    for (int b0 = wave; b0 < nb; b0 += kAtOnce * kWaves) {
        float xa[kAtOnce], xb[kAtOnce];
        uint16_t sa[kAtOnce], sb[kAtOnce];
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            const int b = b0 + u * kWaves;
            const int i0 = (b < nb ? b : b0) * 128 + lane;   // (past the end: the first block again, its result dropped)
            xa[u] = x[i0], xb[u] = x[i0 + 64];
            sa[u] = suh[i0], sb[u] = suh[i0 + 64];
        }
#pragma unroll
        for (int u = 0; u < kAtOnce; ++u) {
            const int b = b0 + u * kWaves;
            if (b < nb) {
                const int i0 = b * 128 + lane;
                float v0 = __fmul_rn(xa[u], f16_bits_to_f32(sa[u])), v1 = __fmul_rn(xb[u], f16_bits_to_f32(sb[u]));
                had128_wave(v0, v1, lane);
                xr[PAIRED ? paired_pos(i0) : i0] = __float2half_rn(v0);
                xr[PAIRED ? paired_pos(i0 + 64) : i0 + 64] = __float2half_rn(v1);
            }
        }
    }
    __syncthreads();
}
// the output rotation of nb blocks of 128 values in LDS, block b by wave b (nb <= 8), in place
__device__ __forceinline__ void had128_out(float* v, int nb) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    if (wave < nb) {
        float v0 = v[wave * 128 + lane], v1 = v[wave * 128 + lane + 64];
        had128_wave(v0, v1, lane);
        v[wave * 128 + lane] = v0;
        v[wave * 128 + lane + 64] = v1;
    }
    __syncthreads();
}

// One matrix's 16-column tile over all its row tiles for NT activations: returns this lane's partial sums for its column
// (the lane's 4 steps are rows 2q, 2q+1, 2q+8, 2q+9 of column (L >> 3) + 8 (L & 1), q = (L >> 1) & 3)
template <int CB, int NT>
__device__ __forceinline__ void walk_tiles(const uint32_t* __restrict__ trellis, int k, int ld, int tc, int k2, int lane,
                                           uint32_t* wt, const __half* xr, int xr_stride, float (&acc)[NT]) {
    const int W = 4 * k2, q = (lane >> 1) & 3;
    for (int ks = 0; ks < (k >> 4); ++ks) {
        const uint32_t* tile = trellis + ((size_t) ks * ld + tc) * W;
        if (lane < W) wt[lane] = tile[lane];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_s_waitcnt(0);  // the wave's own LDS writes have landed before any lane reads them
        float w[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i] = __half2float(exl3_value<CB>(exl3_state(wt, k2, 4 * lane + i)));
        __builtin_amdgcn_wave_barrier();
        const int rb = ks * 16 + 2 * q;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const __half* xv = xr + t * xr_stride + rb;
            float s = acc[t];
            s = fmaf(w[0], __half2float(xv[0]), s);
            s = fmaf(w[1], __half2float(xv[1]), s);
            s = fmaf(w[2], __half2float(xv[8]), s);
            s = fmaf(w[3], __half2float(xv[9]), s);
            acc[t] = s;
        }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {  // the 4 lanes of a column: q = bits 1, 2 of the lane
        acc[t] += __shfl_xor(acc[t], 2, 64);
        acc[t] += __shfl_xor(acc[t], 4, 64);
    }
}

// ---- the same walk with the bit rate a compile-time constant (K2 <= 10): no LDS staging of the tile.  (The layer's kernels take it
// for every codebook: mcg, 6144 x 1536 at 3 bits, one token, 429 us through the general walk, 61 like this.)
// A lane's 4 windows span 16 + 3 K2 / 2 <= 31 bits, so they sit in the two words around the last window's end - two
// dword buffer loads at lane-constant offsets, the tile's address in the scalar offset - and one 64-bit shift puts all
// four into one register, where they are bit-field extracts at compile-time positions.  1024 + the byte sum is an FP16
// whose bit pattern is 0x6400 + the byte sum (one v_sad_u8); values are made two at a time (v_pk_fma_f16) and meet the
// FP16 activation pairs (rows 2q, 2q+1 and 2q+8, 2q+9 are adjacent) in v_dot2_f32_f16.
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
template <int K2> struct Taps {
    static constexpr int end(int i) { return ((i + 1) * K2) / 2; }       // end bit of step i above the lane's 2 L K2
    static constexpr int below(int i) { return end(3) - end(i); }        // how far window i ends before the last one
};
__device__ __forceinline__ h2 as_h2(uint32_t v) {
    union { uint32_t u; h2 h; } c;
    c.u = v;
    return c.h;
}
template <int CB, int K2>
__device__ __forceinline__ void tile_values(uint32_t c, h2& w01, h2& w23) {   // c: the lane's windows
    uint32_t prod[4];
    if constexpr (CB != 2) {
        // 3inst / mcg: the sum of the two halves of (state * a [+ b]) & 0x8fff8fff ^ 0x3b603b60; a pair's low halves and its high
        // halves are gathered into a register each and added two at a time
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t s = __builtin_amdgcn_ubfe(c, Taps<K2>::below(i), 16);
            prod[i] = ((CB == 1 ? s * 0xCBAC1FEDu : s * 89226354u + 64248484u) & 0x8fff8fffu) ^ 0x3b603b60u;
        }
        w01 = as_h2(__builtin_amdgcn_perm(prod[1], prod[0], 0x05040100u)) + as_h2(__builtin_amdgcn_perm(prod[1], prod[0], 0x07060302u));
        w23 = as_h2(__builtin_amdgcn_perm(prod[3], prod[2], 0x05040100u)) + as_h2(__builtin_amdgcn_perm(prod[3], prod[2], 0x07060302u));
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) prod[i] = __builtin_amdgcn_ubfe(c, Taps<K2>::below(i), 16) * 0x83DCD12Du;
    // 0x6400 + the byte sum (at most 1020: no carry out of the half) = the bits of FP16(1024 + byte sum); the pair's second
    // sum lands in the upper half directly (v_sad_hi_u8: (sum << 16) + the third operand), so the pair needs no packing
    const uint32_t p01 = __builtin_amdgcn_sad_hi_u8(prod[1], 0u, __builtin_amdgcn_sad_u8(prod[0], 0u, 0x64006400u));
    const uint32_t p23 = __builtin_amdgcn_sad_hi_u8(prod[3], 0u, __builtin_amdgcn_sad_u8(prod[2], 0u, 0x64006400u));
    const h2 kinv = as_h2(0x1eee1eeeu), kbias = as_h2(0xc931c931u);
    w01 = __builtin_elementwise_fma(as_h2(p01), kinv, kbias);
    w23 = __builtin_elementwise_fma(as_h2(p23), kinv, kbias);
}
// A wave's row tiles are ld * W * 4 bytes apart (a 96-byte read every 9 KB at 3 bits a weight): only many reads in flight keep the
// memory busy, so the walk runs kAhead tiles ahead in a ring of registers - requested as early as the caller can, before
// the input is rotated.
constexpr int kAhead = 8;   // (k is a multiple of 128: the row tiles come in eights)
template <int K2> struct TileRing {
    __amdgpu_buffer_rsrc_t rs;
    uint32_t oa, ob, step, t_off;
    int sh;
    uint32_t ra[kAhead], rb[kAhead];
    // k rows of the matrix at `trellis`, whose tiles are `ld` a row; this wave's column tile tc
    __device__ __forceinline__ void request(const uint32_t* __restrict__ trellis, int k, int ld, int tc, int lane) {
        static_assert(K2 >= 2 && K2 <= 10, "the four windows of a lane must fit 32 bits");
        constexpr int W = 4 * K2;
        const int E = 2 * lane * K2 + Taps<K2>::end(3);   // the end bit of the lane's last window: 1 .. 128 K2
        const int ib = (E - 1) >> 5, ia = ib == 0 ? W - 1 : ib - 1;
        sh = 32 * (ib + 1) - E;
        const uint64_t base = (uint64_t) trellis;
        const uint32_t b_lo = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) base);
        const uint32_t b_hi = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) (base >> 32));
        rs = __builtin_amdgcn_make_buffer_rsrc((void*) (((uint64_t) b_hi << 32) | b_lo), 0, (int) ((uint32_t) (k >> 4) * ld * W * 4), 0x00020000);
        oa = 4u * ia, ob = 4u * ib, step = (uint32_t) ld * W * 4;
        // (tc comes from the wave's index: uniform, but only readfirstlane tells the compiler so - a divergent scalar offset
        // would turn every load into a loop over the lanes)
        t_off = (uint32_t) __builtin_amdgcn_readfirstlane(tc) * W * 4;
#pragma unroll
        for (int i = 0; i < kAhead; ++i) {
            load(i, i);
            __builtin_amdgcn_sched_barrier(0);   // (in this order, the loop's own: its waits count on it)
        }
    }
    __device__ __forceinline__ void load(int i, int tile) {   // (past the matrix: the buffer returns 0)
        ra[i] = __builtin_amdgcn_raw_buffer_load_b32(rs, oa, t_off + (uint32_t) tile * step, 0);
        rb[i] = __builtin_amdgcn_raw_buffer_load_b32(rs, ob, t_off + (uint32_t) tile * step, 0);
    }
};
// after_block(b, acc): called with every lane's sums after each 128 rows (8 tiles), b = 0, 1, ...
template <int CB, int K2, int NT, typename F>
__device__ __forceinline__ void walk_tiles_fast(TileRing<K2>& ring, int k, int lane, const __half* xr, int xr_stride, float (&acc)[NT],
                                                F&& after_block) {
    const int q = (lane >> 1) & 3, nks = k >> 4;
    const uint2* xw = (const uint2*) xr;   // the lane's two pairs of FP16 activations of a row tile (rotate_in<true>'s order)
    const int xs = xr_stride >> 2;
    // Two tiles a step.  A tile's two words become one register of windows BEFORE they are requested again (asked for first, the
    // compiler keeps copies of them: two moves of a tile's 19 vector instructions, 115 registers instead of 71), and the
    // activations come from LDS one step ahead; the order is pinned, since left to itself the compiler gathers the requests
    // behind all eight decodes.  4 tokens on 160 experts of 6144 x 1536 at 3 bits 174.4 -> 159.4 us, one token at 4 bits 69.4 -> 67.1.
    uint2 xn[2][NT];
    auto read_x = [&](int ks) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int t = 0; t < NT; ++t) xn[i][t] = xw[t * xs + (ks + i) * 4 + q];
    };
    read_x(0);
#pragma unroll 1
    for (int ks = 0; ks < nks; ks += kAhead) {
#pragma unroll
        for (int i = 0; i < kAhead; i += 2) {
            uint32_t c[2];
            uint2 xv[2][NT];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                c[j] = __builtin_amdgcn_alignbit(ring.ra[i + j], ring.rb[i + j], (uint32_t) ring.sh);   // (a : b) >> sh, 0 <= sh < 32
                asm volatile("" : "+v"(c[j]));
#pragma unroll
                for (int t = 0; t < NT; ++t) xv[j][t] = xn[j][t];
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) ring.load(i + j, ks + i + j + kAhead);
            read_x(ks + i + 2);   // (past the last tile: what lies behind in LDS - the next activation, the raw outputs - and is dropped)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                h2 w01, w23;
                tile_values<CB, K2>(c[j], w01, w23);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    acc[t] = __builtin_amdgcn_fdot2(w01, as_h2(xv[j][t].x), acc[t], false);
                    acc[t] = __builtin_amdgcn_fdot2(w23, as_h2(xv[j][t].y), acc[t], false);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        after_block(ks >> 3, acc);
    }
}
// the sums of a column: its 4 lanes are q = bits 1, 2 of the lane
template <int NT> __device__ __forceinline__ void column_sums(float (&acc)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        acc[t] += xor_lane<2>(acc[t]);
        acc[t] += xor_lane<4>(acc[t]);
    }
}
// K2 > 0: the compile-time walk; 0: the general one
template <int CB, int NT, int K2>
__device__ __forceinline__ void walk(const uint32_t* __restrict__ trellis, int k, int ld, int tc, int k2, int lane,
                                     uint32_t* wt, const __half* xr, int xr_stride, float (&acc)[NT]) {
    if constexpr (K2 > 0) {
        TileRing<K2> ring;
        ring.request(trellis, k, ld, tc, lane);
        walk_tiles_fast<CB, K2, NT>(ring, k, lane, xr, xr_stride, acc, [](int, float (&)[NT]) {});
        column_sums(acc);
    } else walk_tiles<CB, NT>(trellis, k, ld, tc, k2, lane, wt, xr, xr_stride, acc);
}

__device__ __forceinline__ float ex_swiglu(float g, float u, float limit) {
    if (limit > 0.0f && limit < INFINITY) {
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit);
    }
    return __fmul_rn(__fdiv_rn(g, __fadd_rn(1.0f, expf(-g))), u);
}

// dynamic LDS: [8 waves x 64 words of tile][NT x 2 x k halves of rotated inputs][NT*2*128 floats of raw outputs]
// grid (n_ff / 128, groups)
template <int CB, int NT, int K2>
__global__ __launch_bounds__(kExThreads) void exl3_gate_up_kernel(maya_exl3_args a) {
    extern __shared__ uint32_t lds[];
    GroupRef gr;
    if (!group_of<false>(a, blockIdx.y, gr)) return;
    const int k = a.layout.n_embd, n = a.layout.n_ff;
    uint32_t* wt = lds + (threadIdx.x >> 6) * 64;
    __half* xr = (__half*) (lds + 8 * 64);                       // [NT][2][k]
    float* tmp = (float*) (xr + (size_t) NT * 2 * k);            // the raw outputs [NT][2][128]
    const uint8_t* blob = (const uint8_t*) gr.blob;
    const int64_t xs = a.x_stride ? a.x_stride : k;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int tc = blockIdx.x * 8 + wave;
    // the group's entries two at a time while two are left (one decode of the weights serves both), else one
    auto chunk = [&](auto ntc, int c0) {
        constexpr int NTC = decltype(ntc)::value;
        int ents[NTC];
#pragma unroll
        for (int t = 0; t < NTC; ++t) ents[t] = entry_of(a, gr, c0 + t);
        __syncthreads();
        for (int t = 0; t < NTC; ++t) {
            const float* x = a.x + (size_t) (ents[t] / a.k) * xs;
            for (int role = 0; role < 2; ++role)
                rotate_in<(K2 > 0)>(x, (const uint16_t*) (blob + a.layout.suh[role]), k, xr + ((size_t) t * 2 + role) * k);
        }
        float raw[2][NTC];
#pragma unroll
        for (int role = 0; role < 2; ++role) {
            float acc[NTC];
#pragma unroll
            for (int t = 0; t < NTC; ++t) acc[t] = 0.0f;
            walk<CB, NTC, K2>((const uint32_t*) (blob + a.layout.trellis[role]), k, n >> 4, tc, a.layout.k2[role], lane, wt,
                              xr + (size_t) role * k, 2 * k, acc);
#pragma unroll
            for (int t = 0; t < NTC; ++t) raw[role][t] = acc[t];
        }
        __syncthreads();
        // the lane with q = 0 of each column holds the sums: column (L >> 3) + 8 (L & 1) of the wave's tile
        if (((lane >> 1) & 3) == 0) {
            const int col = wave * 16 + (lane >> 3) + 8 * (lane & 1);
#pragma unroll
            for (int t = 0; t < NTC; ++t) {
                tmp[(t * 2 + 0) * 128 + col] = raw[0][t];
                tmp[(t * 2 + 1) * 128 + col] = raw[1][t];
            }
        }
        __syncthreads();
        had128_out(tmp, NTC * 2);
        const uint16_t* svg = (const uint16_t*) (blob + a.layout.svh[0]) + blockIdx.x * 128;
        const uint16_t* svu = (const uint16_t*) (blob + a.layout.svh[1]) + blockIdx.x * 128;
        for (int i = threadIdx.x; i < NTC * 128; i += kExThreads) {
            const int t = i >> 7, c = i & 127;
            const float g = __fmul_rn(tmp[(t * 2 + 0) * 128 + c], f16_bits_to_f32(svg[c]));
            const float u = __fmul_rn(tmp[(t * 2 + 1) * 128 + c], f16_bits_to_f32(svu[c]));
            a.h[(size_t) ents[t] * n + blockIdx.x * 128 + c] = ex_swiglu(g, u, a.limit);
        }
    };
    for (int c0 = 0; c0 < gr.ne;) {
        if (NT >= 2 && gr.ne - c0 >= 2) {
            chunk(std::integral_constant<int, 2>{}, c0);
            c0 += 2;
        } else {
            chunk(std::integral_constant<int, 1>{}, c0);
            c0 += 1;
        }
    }
}

// The clamped SwiGLU of an entry's gate/up sums in S slices (slice 0 first) on one wave: the lane's two values of the 128-value block
// whose first value this lane takes is c (values c and c + 64), P as exl3_slices_kernel left it.
__device__ __forceinline__ void swiglu_block(const float* __restrict__ P, int S, size_t n, int e, int c, float limit, float& h0, float& h1) {
    float g[2], u[2];
    const float* pg = P + ((size_t) e * 2 + 0) * S * n + c;
    const float* pu = P + ((size_t) e * 2 + 1) * S * n + c;
    if (S == 4) {   // (the layer's usual form: sixteen loads side by side)
        float a[4][4];
#pragma unroll
        for (int q = 0; q < 4; ++q) a[0][q] = pg[q * n], a[1][q] = pg[q * n + 64], a[2][q] = pu[q * n], a[3][q] = pu[q * n + 64];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            g[i] = __fadd_rn(__fadd_rn(__fadd_rn(a[i][0], a[i][1]), a[i][2]), a[i][3]);
            u[i] = __fadd_rn(__fadd_rn(__fadd_rn(a[2 + i][0], a[2 + i][1]), a[2 + i][2]), a[2 + i][3]);
        }
    } else {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            g[i] = pg[64 * i], u[i] = pu[64 * i];
            for (int q = 1; q < S; ++q) {
                g[i] = __fadd_rn(g[i], pg[q * n + 64 * i]);
                u[i] = __fadd_rn(u[i], pu[q * n + 64 * i]);
            }
        }
    }
    h0 = ex_swiglu(g[0], u[0], limit), h1 = ex_swiglu(g[1], u[1], limit);
}

// ---- the combine at the end of the down launch.  The workgroups of a 128-column block (all groups, all slices) count themselves in
// done[block], which the gate/up launch before them cleared; the one that comes last adds the block's partial outputs up for
// every token.  Nobody waits for anybody.  The partial outputs go past the XCD's L2 both ways (agent scope), a workgroup
// counts itself when its own have arrived; the order of the sums is fixed, so the bits do not depend on who is last.
// (counters 256 bytes apart: side by side in two cache lines, the 768 workgroups' counts took turns at one memory channel)
constexpr int kDoneStride = 64;
__device__ __forceinline__ void store_part(float* p, float v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ float load_part(const float* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void combine_by_last(const maya_exl3_args& a, const float* part, int S, uint32_t* done, uint32_t* lds) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the wave's own partial outputs are where every XCD sees them
    __syncthreads();
    if (threadIdx.x == 0) lds[0] = __hip_atomic_fetch_add(done + kDoneStride * blockIdx.x, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (lds[0] != gridDim.y * gridDim.z - 1u || (a.skip && *a.skip)) return;
    const int n = a.layout.n_embd;
    for (int i = threadIdx.x; i < a.n_tokens * 128; i += kExThreads) {
        const int t = __builtin_amdgcn_readfirstlane(i >> 7), c = blockIdx.x * 128 + (i & 127), e0 = t * a.k;   // (a wave: half a token's columns)
        float sum = 0.0f;
        bool first = true;
        for (int j0 = 0; j0 < a.k; j0 += 8) {
            float v[8][2], w[8];
            uint64_t b[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {   // eight slots' loads side by side (past the last slot: its own again, dropped)
                const int e = e0 + min(j0 + j, a.k - 1);
                v[j][0] = load_part(part + (size_t) e * S * n + (uint32_t) c);
                v[j][1] = load_part(part + ((size_t) e * S + (S - 1)) * n + (uint32_t) c);
                w[j] = a.plan_w[e];
                b[j] = a.plan_ptr[e];
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (j0 + j >= a.k || b[j] == 0ull) continue;
                const float p = __fmul_rn(S > 1 ? __fadd_rn(v[j][0], v[j][1]) : v[j][0], w[j]);
                sum = first ? p : __fadd_rn(sum, p);
                first = false;
            }
        }
        if (a.add && (!a.add_flag || *a.add_flag)) sum = __fadd_rn(sum, a.add[(size_t) t * n + c]);
        if (a.add2) sum = __fadd_rn(sum, a.add2[(size_t) t * n + c]);
        a.out[(size_t) t * n + c] = sum;
    }
}

// ---- the products in row slices (the compile-time walk only).  A matrix's rows are cut into S slices of whole 128-row blocks; a
// workgroup takes 128 columns and SP neighbouring slices of one matrix: it rotates its part of the input (gate/up) or copies the
// rotated h (down), walks down its rows, and at each slice's end leaves its 128 sums in LDS; these are rotated and scaled at the
// end - both linear, so the slices' outputs simply add - and stored to P[entry][matrix][slice][columns].  What a slice
// holds and the order in which the next kernel adds the slices depend on the expert's shape alone, so a window's tokens get
// the bits they get alone; how many slices a workgroup walks is chosen by how many workgroups the call then has.
// grid (columns / 128, groups, matrices * S / SP); dynamic LDS: [NT][rows] halves of rotated input, [SP][NT][128] sums.
// done: the down launch's counters of column blocks (combine_by_last), cleared by the gate/up launch; NULL: nobody counts.
// hr NULL (down): the workgroup makes its rows of h itself from the gate/up sums Pgu in Sgu slices.  One token's down launch
// does - the sums are one trip to memory where the rotated h would be one, against a launch of 4.8 us of its own - windows do
// not: there every one of a group's 48 workgroups would make them again for each token (4 tokens: 168.5 -> 173.2 us).
__device__ __forceinline__ int slice_block(int s, int nb, int S) { return (s * nb) >> (S >> 1); }   // slice s's first block of nb (S = 1, 2 or 4)
// COMB (down): the launch adds up as well, over the counters `done`.
// whole_groups: the group arrays are a layer's workspace, a word for every entry (group_of); 0: a stage call's, which may end sooner.
// HEAD (gate/up, one token, NT = 1): the router rides in the launch.  Every workgroup finds the experts for itself on its last wave by
// the order of the logits (the exact router there where two are too close to call); the first one routes the token exactly on the
// wave before and writes ids, weights and plan.  (A workgroup of its own for that took the place of one that walks: 768 fill the
// chip, and one token of 6144 x 1536 at 4 bits took 52.2 us like that, 50.2 with the router in a launch before.)
struct Exl3Head {
    const float* logits;
    const uint64_t* table;
    int n_expert;
    int32_t* ids;
    float* weights;
    uint64_t* plan;
};
// every thread of a workgroup calls it; lds: kHeadLdsWords.  The blob of slot `slot` (0: none)
constexpr int kHeadLdsWords = 64 + 256 + 512;
__device__ __forceinline__ uint64_t exl3_head(const Exl3Head& hd, int k, int slot, bool first, uint32_t* lds) {
    uint64_t* s_blob = (uint64_t*) lds;
    float* s_lv = (float*) (lds + 64);
    uint64_t* s_tab = (uint64_t*) (lds + 64 + 256);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ne = hd.n_expert;
    const bool picker = wave == kExThreads / 64 - 1;
    if (picker || (first && wave == kExThreads / 64 - 2)) {
        float lv[4];
        uint64_t tab[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int e = 64 * r + lane;
            lv[r] = e < ne ? hd.logits[e] : -INFINITY;
            tab[r] = e < ne ? hd.table[e] : 0ull;
        }
        int id;
        float w;
        uint64_t ptr;
        bool exact = true;
        if (picker) {
            __builtin_amdgcn_s_setprio(3);   // the workgroup waits for this wave: it goes first on its SIMD
#pragma unroll
            for (int r = 0; r < 4; ++r) s_tab[64 * r + lane] = tab[r];
            exact = !route_wave_order_only(lv, true, ne, k, s_lv, 1e-6f, 60.0f, id);
            if (!exact) ptr = s_tab[lane < k ? id : 0];
        }
        if (exact) route_wave_softmax(lv, tab, ne, k, id, w, ptr);
        if (lane < k) {
            if (picker) s_blob[lane] = ptr;
            else hd.ids[lane] = id, hd.weights[lane] = w, hd.plan[lane] = ptr;
        }
        __builtin_amdgcn_s_setprio(0);
    }
    __syncthreads();
    const uint64_t b = s_blob[slot];
    const uint32_t lo = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) b), hi = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) (b >> 32));
    __syncthreads();   // (the rotated input takes this LDS next)
    return ((uint64_t) hi << 32) | lo;
}
template <int CB, int NT, int K2, bool DOWN, bool COMB, bool HEAD = false>
__global__ __launch_bounds__(kExThreads) void exl3_slices_kernel(maya_exl3_args a, int S, int SP, const __half* __restrict__ hr,
                                                                 const float* __restrict__ Pgu, int Sgu, float* P, uint32_t* done, Exl3Head hd, int whole_groups) {
    extern __shared__ uint32_t lds[];
    if (!DOWN && done && blockIdx.y == 0 && blockIdx.z == 0)
        for (int i = blockIdx.x * kExThreads + threadIdx.x; i < a.layout.n_embd >> 7; i += gridDim.x * kExThreads) done[kDoneStride * i] = 0u;
    GroupRef gr;
    if constexpr (HEAD) {
        static_assert(NT == 1 && !DOWN, "one token's gate/up launch");
        gr.e0 = blockIdx.y, gr.ne = 1;
        gr.blob = exl3_head(hd, a.k, (int) blockIdx.y, blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0, lds);
        if (gr.blob == 0ull) return;
    } else if (!(whole_groups ? group_of<true>(a, blockIdx.y, gr) : group_of<false>(a, blockIdx.y, gr))) {
        if constexpr (COMB) combine_by_last(a, P, S, done, lds);
        return;
    }
    const int per = S / SP, role = DOWN ? 2 : (int) blockIdx.z / per, s0 = ((int) blockIdx.z % per) * SP;
    const int k = DOWN ? a.layout.n_ff : a.layout.n_embd, n = DOWN ? a.layout.n_embd : a.layout.n_ff, nb = k >> 7;
    const int b0 = slice_block(s0, nb, S), kb = (slice_block(s0 + SP, nb, S) - b0) * 128;   // the workgroup's rows
    __half* xr = (__half*) lds;                         // [NT][kb]
    float* tmp = (float*) (xr + (size_t) NT * kb);      // [SP][NT][128]
    const uint8_t* blob = (const uint8_t*) gr.blob;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int tc = blockIdx.x * 8 + wave, ld = n >> 4;
    const uint32_t* trellis = (const uint32_t*) (blob + a.layout.trellis[role]) + (size_t) b0 * 8 * ld * (4 * K2);
    const uint16_t* sv = (const uint16_t*) (blob + a.layout.svh[role]) + blockIdx.x * 128;
    auto chunk = [&](auto ntc, int c0) {
        constexpr int NTC = decltype(ntc)::value;
        int ents[NTC];
#pragma unroll
        for (int t = 0; t < NTC; ++t) ents[t] = entry_of(a, gr, c0 + t);
        TileRing<K2> ring;
        ring.request(trellis, kb, ld, tc, lane);
        __syncthreads();
        if (DOWN && NT == 1 && hr == nullptr) {
            const uint16_t* suh = (const uint16_t*) (blob + a.layout.suh[2]) + (size_t) b0 * 128;
            for (int b = wave; b < kb >> 7; b += kExThreads / 64) {
                const int i0 = b * 128 + lane;
                const uint16_t sa = suh[i0], sb = suh[i0 + 64];
                float h0, h1;
                swiglu_block(Pgu, Sgu, k, ents[0], b0 * 128 + i0, a.limit, h0, h1);
                float v0 = __fmul_rn(h0, f16_bits_to_f32(sa)), v1 = __fmul_rn(h1, f16_bits_to_f32(sb));
                had128_wave(v0, v1, lane);
                xr[paired_pos(i0)] = __float2half_rn(v0);
                xr[paired_pos(i0 + 64)] = __float2half_rn(v1);
            }
            __syncthreads();
        } else if constexpr (DOWN) {
#pragma unroll
            for (int t = 0; t < NTC; ++t)
                for (int i = threadIdx.x; i < kb >> 3; i += kExThreads)
                    ((uint4*) (xr + (size_t) t * kb))[i] = ((const uint4*) (hr + (size_t) ents[t] * k + (size_t) b0 * 128))[i];
            __syncthreads();
        } else {
            const int64_t xs = a.x_stride ? a.x_stride : k;
            const uint16_t* suh = (const uint16_t*) (blob + a.layout.suh[role]) + (size_t) b0 * 128;
            for (int t = 0; t < NTC; ++t)
                rotate_in<true>(a.x + (size_t) (ents[t] / a.k) * xs + (size_t) b0 * 128, suh, kb, xr + (size_t) t * kb);
        }
        float acc[NTC];
#pragma unroll
        for (int t = 0; t < NTC; ++t) acc[t] = 0.0f;
        int s = 0, end = slice_block(s0 + 1, nb, S) - b0;
        walk_tiles_fast<CB, K2, NTC>(ring, kb, lane, xr, kb, acc, [&](int b, float (&v)[NTC]) {
            if (b + 1 == end) {
                column_sums(v);
                if (((lane >> 1) & 3) == 0) {
                    const int col = wave * 16 + (lane >> 3) + 8 * (lane & 1);
#pragma unroll
                    for (int t = 0; t < NTC; ++t) tmp[(s * NTC + t) * 128 + col] = v[t];
                }
#pragma unroll
                for (int t = 0; t < NTC; ++t) v[t] = 0.0f;
                ++s;
                end = slice_block(s0 + s + 1, nb, S) - b0;
            }
        });
        __syncthreads();
        had128_out(tmp, SP * NTC);
        for (int i = threadIdx.x; i < SP * NTC * 128; i += kExThreads) {
            const int c = i & 127, j = i >> 7, t = j % NTC, sl = s0 + j / NTC;
            const size_t at = DOWN ? (size_t) ents[t] * S + sl : ((size_t) ents[t] * 2 + role) * S + sl;
            const float v = __fmul_rn(tmp[i], f16_bits_to_f32(sv[c]));
            if constexpr (COMB) store_part(P + at * n + blockIdx.x * 128 + c, v);
            else P[at * n + blockIdx.x * 128 + c] = v;
        }
    };
    for (int c0 = 0; c0 < gr.ne;) {
        if (NT >= 4 && gr.ne - c0 >= 4) {
            chunk(std::integral_constant<int, NT >= 4 ? 4 : 1>{}, c0);
            c0 += 4;
        } else if (NT >= 2 && gr.ne - c0 >= 2) {
            chunk(std::integral_constant<int, NT >= 2 ? 2 : 1>{}, c0);
            c0 += 2;
        } else {
            chunk(std::integral_constant<int, 1>{}, c0);
            c0 += 1;
        }
    }
    if constexpr (COMB) combine_by_last(a, P, S, done, lds);
}
// grid (n_ff / 512 rounded up, entries): the clamped SwiGLU of the slices' sums (slice 0 first), a 128-value block a wave: written
// to h, or - hr given - as the down product's rotated input FP16(H(h * suh)) in the walk's order, once an entry instead
// of once a workgroup of the down launch
__global__ __launch_bounds__(256) void exl3_swiglu_kernel(maya_exl3_args a, int S, const float* __restrict__ P, __half* __restrict__ hr) {
    if (a.skip && *a.skip) return;
    const int e = blockIdx.y, lane = threadIdx.x & 63, b = blockIdx.x * 4 + (threadIdx.x >> 6), n = a.layout.n_ff, c = b * 128 + lane;
    if (b * 128 >= n) return;
    const uint64_t blob = a.plan_ptr[e];
    if (blob == 0ull) return;
    float h0, h1;
    swiglu_block(P, S, n, e, c, a.limit, h0, h1);
    if (hr == nullptr) {
        a.h[(size_t) e * n + c] = h0;
        a.h[(size_t) e * n + c + 64] = h1;
        return;
    }
    const uint16_t* suh = (const uint16_t*) ((const uint8_t*) blob + a.layout.suh[2]);
    float v0 = __fmul_rn(h0, f16_bits_to_f32(suh[c])), v1 = __fmul_rn(h1, f16_bits_to_f32(suh[c + 64]));
    had128_wave(v0, v1, lane);
    hr[(size_t) e * n + paired_pos(c)] = __float2half_rn(v0);
    hr[(size_t) e * n + paired_pos(c + 64)] = __float2half_rn(v1);
}

// grid (n_embd / 128, groups): part[e][columns] = the down product of h[e]
template <int CB, int NT, int K2>
__global__ __launch_bounds__(kExThreads) void exl3_down_kernel(maya_exl3_args a) {
    extern __shared__ uint32_t lds[];
    GroupRef gr;
    if (!group_of<false>(a, blockIdx.y, gr)) return;
    const int k = a.layout.n_ff, n = a.layout.n_embd;
    uint32_t* wt = lds + (threadIdx.x >> 6) * 64;
    __half* xr = (__half*) (lds + 8 * 64);             // [NT][k]
    float* tmp = (float*) (xr + (size_t) NT * k);      // the raw outputs [NT][128]
    const uint8_t* blob = (const uint8_t*) gr.blob;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int tc = blockIdx.x * 8 + wave;
    auto chunk = [&](auto ntc, int c0) {
        constexpr int NTC = decltype(ntc)::value;
        int ents[NTC];
#pragma unroll
        for (int t = 0; t < NTC; ++t) ents[t] = entry_of(a, gr, c0 + t);
        __syncthreads();
        for (int t = 0; t < NTC; ++t)
            rotate_in<(K2 > 0)>(a.h + (size_t) ents[t] * k, (const uint16_t*) (blob + a.layout.suh[2]), k, xr + (size_t) t * k);
        float acc[NTC];
#pragma unroll
        for (int t = 0; t < NTC; ++t) acc[t] = 0.0f;
        walk<CB, NTC, K2>((const uint32_t*) (blob + a.layout.trellis[2]), k, n >> 4, tc, a.layout.k2[2], lane, wt, xr, k, acc);
        __syncthreads();
        if (((lane >> 1) & 3) == 0) {
            const int col = wave * 16 + (lane >> 3) + 8 * (lane & 1);
#pragma unroll
            for (int t = 0; t < NTC; ++t) tmp[t * 128 + col] = acc[t];
        }
        __syncthreads();
        had128_out(tmp, NTC);
        const uint16_t* sv = (const uint16_t*) (blob + a.layout.svh[2]) + blockIdx.x * 128;
        for (int i = threadIdx.x; i < NTC * 128; i += kExThreads) {
            const int t = i >> 7, c = i & 127;
            a.part[(size_t) ents[t] * n + blockIdx.x * 128 + c] = __fmul_rn(tmp[t * 128 + c], f16_bits_to_f32(sv[c]));
        }
    };
    for (int c0 = 0; c0 < gr.ne;) {
        if (NT >= 2 && gr.ne - c0 >= 2) {
            chunk(std::integral_constant<int, 2>{}, c0);
            c0 += 2;
        } else {
            chunk(std::integral_constant<int, 1>{}, c0);
            c0 += 1;
        }
    }
}

// (part: the down outputs in S slices an entry, added slice 0 first)
__global__ __launch_bounds__(256) void exl3_combine_kernel(maya_exl3_args a, const float* __restrict__ part, int S) {
    if (a.skip && *a.skip) return;
    const int t = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x, n = a.layout.n_embd;
    if (c >= n) return;
    float sum = 0.0f;
    bool first = true;
    for (int i = 0; i < a.k; ++i) {
        const int e = t * a.k + i;
        if (a.plan_ptr[e] == 0ull) continue;
        float v = part[(size_t) e * S * n + c];
        for (int s = 1; s < S; ++s) v = __fadd_rn(v, part[((size_t) e * S + s) * n + c]);
        const float p = __fmul_rn(v, a.plan_w[e]);
        sum = first ? p : __fadd_rn(sum, p);
        first = false;
    }
    if (a.add && (!a.add_flag || *a.add_flag)) sum = __fadd_rn(sum, a.add[(size_t) t * n + c]);
    if (a.add2) sum = __fadd_rn(sum, a.add2[(size_t) t * n + c]);
    a.out[(size_t) t * n + c] = sum;
}

bool exl3_k2_ok(int k2, int cb) {
    return (k2 >= 2 && k2 <= 16 && (k2 & 1) == 0 && cb >= 0 && cb <= 2) || ((k2 == 3 || k2 == 5 || k2 == 7) && cb == 2);
}
int exl3_check(const maya_exl3_args* a) {
    if (!a) return fail(MAYA_E_ARG, "exl3: null args");
    const maya_exl3_layout& l = a->layout;
    for (int r = 0; r < 3; ++r)
        if (!exl3_k2_ok(l.k2[r], l.cb)) return fail(MAYA_E_UNSUPPORTED, "exl3: k2 %d with codebook %d", l.k2[r], l.cb);
    if (l.n_embd <= 0 || l.n_ff <= 0 || l.n_embd % 128 || l.n_ff % 128 || l.n_embd > 16384 || l.n_ff > 16384)
        return fail(MAYA_E_SHAPE, "exl3: n_embd %d / n_ff %d: multiples of 128 up to 16384 wanted", l.n_embd, l.n_ff);
    for (int r = 0; r < 3; ++r)
        if (l.trellis[r] % 4 || l.suh[r] % 2 || l.svh[r] % 2) return fail(MAYA_E_ARG, "exl3: misaligned part offsets");
    if (a->n_tokens < 1 || a->n_tokens > MAYA_MAX_TOKENS || a->k < 1 || a->k > MAYA_MAX_K)
        return fail(MAYA_E_SHAPE, "exl3: n_tokens %d / k %d", a->n_tokens, a->k);
    if (!a->plan_ptr || !a->plan_w) return fail(MAYA_E_ARG, "exl3: null plan");
    if (a->grp_ptr && (!a->grp_start || !a->grp_ent || !a->n_groups)) return fail(MAYA_E_ARG, "exl3: incomplete groups");
    return MAYA_OK;
}

template <int NT>
int launch_exl3_gate_up(const maya_exl3_args& a, const DeviceState& st, hipStream_t s) {
    const int k = a.layout.n_embd;
    const size_t scratch = (size_t) NT * 256 * 4;
    const size_t lds = 8 * 64 * 4 + (size_t) NT * 2 * k * 2 + scratch;
    if (lds > (size_t) st.lds_limit) return fail(MAYA_E_SHAPE, "exl3 gate/up needs %zu bytes of LDS, the device gives %d", lds, st.lds_limit);
    const dim3 grid((unsigned) (a.layout.n_ff / 128), (unsigned) (a.n_tokens * a.k));
#define MAYA_EX(CBV, K2V)                                                                                         \
    {                                                                                                             \
        auto kern = exl3_gate_up_kernel<CBV, NT, K2V>;                                                            \
        if (lds > 65536) MAYA_HIP(hipFuncSetAttribute((const void*) kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds)); \
        hipLaunchKernelGGL(kern, grid, dim3(kExThreads), lds, s, a);                                              \
    }
    // the compile-time walk: mul1, gate and up at one bit rate of at most 5 bits a weight
    const int k2f = a.layout.cb == 2 && a.layout.k2[0] == a.layout.k2[1] && a.layout.k2[0] <= 10 ? a.layout.k2[0] : 0;
    switch (k2f) {
        case 2: MAYA_EX(2, 2) break;
        case 3: MAYA_EX(2, 3) break;
        case 4: MAYA_EX(2, 4) break;
        case 5: MAYA_EX(2, 5) break;
        case 6: MAYA_EX(2, 6) break;
        case 7: MAYA_EX(2, 7) break;
        case 8: MAYA_EX(2, 8) break;
        case 10: MAYA_EX(2, 10) break;
        default:
            if (a.layout.cb == 2) MAYA_EX(2, 0) else if (a.layout.cb == 1) MAYA_EX(1, 0) else MAYA_EX(0, 0)
    }
#undef MAYA_EX
    MAYA_LAUNCHED("exl3_gate_up_kernel");
    return MAYA_OK;
}
// Slices a workgroup walks: as many as leave the call three workgroups a compute unit, at least one.  Three is what the registers of
// the two-token kernels (70) let a compute unit hold at once; one token's hold four (58) or three (70, the down launch that makes h),
// the four-token ones two (96 to 100): a call of theirs that is cut for three runs its last third as a second round.
// And half as many slices where the call then still has less than twice that and a workgroup 16 blocks of rows: a compute unit's three
// end one after the other (the wave that came first issues first), with nothing to take their place, or a second round of workgroups is a part
// of one.  Six a compute unit, three before: 4 tokens top-8 of 6144 x 1536 at 3 bits 145.5 -> 142.2 us, 5 tokens 204 -> 188, 8 tokens
// top-6 of 4096 x 1536 148.5 -> 141.5, 4 tokens top-8 of 7168 x 2048 at 5 bits 235 -> 229.  Shorter workgroups do not pay: 2 tokens of 6144 x 1536
// (12 blocks) 78.3 -> 79.2, 3 of 4096 x 1024 (8 blocks) 61.7 -> 64.2.
static int slices_per_wg(long long wgs, int S, int blocks, const DeviceState& st) {
    int sp = S;
    while (sp > 1 && (S % sp != 0 || wgs * (S / sp) < 3ll * st.n_cu)) --sp;
    if (sp % 2 == 0 && wgs * (S / sp) < 6ll * st.n_cu && blocks / S * (sp / 2) >= 16) sp /= 2;
    return sp;
}
template <int NT, bool DOWN, bool COMB, bool HEAD = false>
int launch_exl3_slices(const maya_exl3_args& a, int S, const __half* hr, const float* Pgu, int Sgu, float* P, uint32_t* done, bool whole_groups,
                       const DeviceState& st, hipStream_t s, const Exl3Head& hd = Exl3Head{}) {
    const maya_exl3_layout& l = a.layout;
    const int k = DOWN ? l.n_ff : l.n_embd, n = DOWN ? l.n_embd : l.n_ff, mats = DOWN ? 1 : 2;
    int SP = slices_per_wg((long long) (n / 128) * a.n_tokens * a.k * mats, S, k / 128, st);
    while (SP * NT > 8) SP >>= 1;   // (the closing rotation takes a block of 128 sums a wave)
    const int rows = ((k / 128 + S - 1) / S) * SP * 128;   // the longest workgroup's
    size_t lds = (size_t) NT * rows * 2 + (size_t) SP * NT * 128 * 4;
    if (HEAD && lds < 4 * kHeadLdsWords) lds = 4 * kHeadLdsWords;   // (exl3_head's)
    if (lds > (size_t) st.lds_limit) return fail(MAYA_E_SHAPE, "exl3 slices need %zu bytes of LDS, the device gives %d", lds, st.lds_limit);
    const dim3 grid((unsigned) (n / 128), (unsigned) (a.n_tokens * a.k), (unsigned) (mats * (S / SP)));
#define MAYA_EX(CBV, K2V)                                                                                         \
    case 16 * CBV + K2V: {                                                                                        \
        auto kern = exl3_slices_kernel<CBV, NT, K2V, DOWN, COMB, HEAD>;                                                       \
        if (lds > 65536) MAYA_HIP(hipFuncSetAttribute((const void*) kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds)); \
        hipLaunchKernelGGL(kern, grid, dim3(kExThreads), lds, s, a, S, SP, hr, Pgu, Sgu, P, done, hd, whole_groups ? 1 : 0);              \
        break;                                                                                                    \
    }
    switch (16 * l.cb + l.k2[DOWN ? 2 : 0]) {
        MAYA_EX(2, 2) MAYA_EX(2, 3) MAYA_EX(2, 4) MAYA_EX(2, 5) MAYA_EX(2, 6) MAYA_EX(2, 7) MAYA_EX(2, 8) MAYA_EX(2, 10)
        MAYA_EX(1, 2) MAYA_EX(1, 4) MAYA_EX(1, 6) MAYA_EX(1, 8) MAYA_EX(1, 10)
        MAYA_EX(0, 2) MAYA_EX(0, 4) MAYA_EX(0, 6) MAYA_EX(0, 8) MAYA_EX(0, 10)
        default: return fail(MAYA_E_UNSUPPORTED, "exl3 slices: k2 %d, codebook %d", l.k2[DOWN ? 2 : 0], l.cb);
    }
#undef MAYA_EX
    MAYA_LAUNCHED("exl3_slices_kernel");
    return MAYA_OK;
}
int launch_exl3_swiglu(const maya_exl3_args& a, int S, const float* P, __half* hr, hipStream_t s) {
    hipLaunchKernelGGL(exl3_swiglu_kernel, dim3((unsigned) ((a.layout.n_ff + 511) / 512), (unsigned) (a.n_tokens * a.k)), dim3(256), 0, s, a, S, P, hr);
    MAYA_LAUNCHED("exl3_swiglu_kernel");
    return MAYA_OK;
}
// the gate/up product in slices when the stage call's `part` holds its partial outputs (one bit rate <= 5 bits for gate and up):
// 1 launched, 0 not applicable
static bool walk_is_fast(const maya_exl3_layout& l, int r) { return l.k2[r] <= 10; }
template <int NT>
int try_exl3_gu_split(const maya_exl3_args& a, const DeviceState& st, hipStream_t s, int* rc) {
    const maya_exl3_layout& l = a.layout;
    if (!walk_is_fast(l, 0) || l.k2[0] != l.k2[1] || !a.part) return 0;
    const int S = (l.n_embd % 256 == 0 && l.n_embd >= 4 * l.n_ff) ? 2 : (l.n_embd >= 2 * l.n_ff ? 1 : 0);
    if (S == 0) return 0;
    *rc = launch_exl3_slices<NT, false, false>(a, S, nullptr, nullptr, 0, a.part, nullptr, false, st, s);
    if (!*rc) *rc = launch_exl3_swiglu(a, S, a.part, nullptr, s);
    return 1;
}

template <int NT>
int launch_exl3_down(const maya_exl3_args& a, const DeviceState& st, hipStream_t s) {
    const int k = a.layout.n_ff;
    const size_t scratch = (size_t) NT * 128 * 4;
    const size_t lds = 8 * 64 * 4 + (size_t) NT * k * 2 + scratch;
    if (lds > (size_t) st.lds_limit) return fail(MAYA_E_SHAPE, "exl3 down needs %zu bytes of LDS, the device gives %d", lds, st.lds_limit);
    const dim3 grid((unsigned) (a.layout.n_embd / 128), (unsigned) (a.n_tokens * a.k));
#define MAYA_EX(CBV, K2V)                                                                                         \
    {                                                                                                             \
        auto kern = exl3_down_kernel<CBV, NT, K2V>;                                                               \
        if (lds > 65536) MAYA_HIP(hipFuncSetAttribute((const void*) kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds)); \
        hipLaunchKernelGGL(kern, grid, dim3(kExThreads), lds, s, a);                                              \
    }
    const int k2f = a.layout.cb == 2 && a.layout.k2[2] <= 10 ? a.layout.k2[2] : 0;
    switch (k2f) {
        case 2: MAYA_EX(2, 2) break;
        case 3: MAYA_EX(2, 3) break;
        case 4: MAYA_EX(2, 4) break;
        case 5: MAYA_EX(2, 5) break;
        case 6: MAYA_EX(2, 6) break;
        case 7: MAYA_EX(2, 7) break;
        case 8: MAYA_EX(2, 8) break;
        case 10: MAYA_EX(2, 10) break;
        default:
            if (a.layout.cb == 2) MAYA_EX(2, 0) else if (a.layout.cb == 1) MAYA_EX(1, 0) else MAYA_EX(0, 0)
    }
#undef MAYA_EX
    MAYA_LAUNCHED("exl3_down_kernel");
    return MAYA_OK;
}

}  // namespace maya

using namespace maya;

extern "C" {

int maya_exl3_supported(int k2, int cb) { return exl3_k2_ok(k2, cb) ? 1 : 0; }

size_t maya_exl3_layout_init(maya_exl3_layout* l, int n_embd, int n_ff, const int32_t* k2, int cb, int order) {
    if (!l || !k2 || n_embd <= 0 || n_ff <= 0 || n_embd % 128 || n_ff % 128 || (order != MAYA_EXL3_ORDER_SCALES_FIRST && order != MAYA_EXL3_ORDER_TRELLIS_FIRST))
        return 0;
    for (int r = 0; r < 3; ++r)
        if (!exl3_k2_ok(k2[r], cb)) return 0;
    *l = maya_exl3_layout{};
    l->cb = cb;
    l->n_embd = n_embd;
    l->n_ff = n_ff;
    // every piece starts on a multiple of `al` bytes: 16 for the compact order, 256 for the engine's assembled blobs
    const size_t al = order == MAYA_EXL3_ORDER_TRELLIS_FIRST ? 256 : 16;
    auto up = [al](size_t n) { return (n + al - 1) / al * al; };
    size_t off = 0;
    for (int r = 0; r < 3; ++r) {
        const int64_t k = r == 2 ? n_ff : n_embd, n = r == 2 ? n_embd : n_ff;
        const size_t tb = maya_exl3_trellis_bytes(k, n, k2[r]);
        l->k2[r] = k2[r];
        if (order == MAYA_EXL3_ORDER_TRELLIS_FIRST) {
            l->trellis[r] = off, off += up(tb);
            l->suh[r] = off, off += up(2 * (size_t) k);
            l->svh[r] = off, off += up(2 * (size_t) n);
        } else {
            l->suh[r] = off, off += up(2 * (size_t) k);
            l->svh[r] = off, off += up(2 * (size_t) n);
            l->trellis[r] = off, off += up(tb);
        }
    }
    return off;
}
size_t maya_exl3_trellis_bytes(int64_t k, int64_t n, int k2) { return (size_t) (k / 16) * (size_t) (n / 16) * 16u * (size_t) k2; }

// nine pieces an expert (the trellis, suh and svh of gate, up and down) copied to their places in the expert's blob:
// grid (blocks, 9, n_expert).  16 bytes a thread where source and destination allow it, else byte by byte.
__global__ __launch_bounds__(256) void exl3_pack_kernel(const uint64_t* __restrict__ pieces, maya_exl3_layout l, uint8_t* __restrict__ dst,
                                                        size_t dst_stride) {
    const int piece = blockIdx.y, r = piece / 3, what = piece % 3, e = blockIdx.z;
    const int64_t k = r == 2 ? l.n_ff : l.n_embd, n = r == 2 ? l.n_embd : l.n_ff;
    const size_t bytes = what == 0 ? (size_t) (k / 16) * (size_t) (n / 16) * 16u * (size_t) l.k2[r] : what == 1 ? 2 * (size_t) k : 2 * (size_t) n;
    const size_t off = what == 0 ? l.trellis[r] : what == 1 ? l.suh[r] : l.svh[r];
    const uint8_t* src = (const uint8_t*) pieces[(size_t) e * 9 + piece];
    uint8_t* d = dst + (size_t) e * dst_stride + off;
    if (src == nullptr) return;
    const size_t stride = (size_t) gridDim.x * 256;
    if ((((uintptr_t) src | (uintptr_t) d) & 15) == 0) {
        const size_t n16 = bytes >> 4;
        for (size_t i = (size_t) blockIdx.x * 256 + threadIdx.x; i < n16; i += stride) ((uint4*) d)[i] = ((const uint4*) src)[i];
        for (size_t i = (n16 << 4) + (size_t) blockIdx.x * 256 + threadIdx.x; i < bytes; i += stride) d[i] = src[i];
    } else {
        for (size_t i = (size_t) blockIdx.x * 256 + threadIdx.x; i < bytes; i += stride) d[i] = src[i];
    }
}

int maya_exl3_pack_experts(const maya_exl3_layout* l, const uint64_t* pieces, int n_expert, void* dst, size_t dst_stride, void* stream) {
    DeviceState* st;
    if (const int rc = current_state(&st)) return rc;
    if (!l || !pieces || !dst) return fail(MAYA_E_ARG, "exl3_pack_experts: null pointer");
    if (n_expert <= 0 || n_expert > 65535) return fail(MAYA_E_SHAPE, "exl3_pack_experts: %d experts", n_expert);
    if (l->n_embd <= 0 || l->n_ff <= 0 || l->n_embd % 128 || l->n_ff % 128) return fail(MAYA_E_SHAPE, "exl3_pack_experts: %d x %d", l->n_embd, l->n_ff);
    size_t end = 0;
    for (int r = 0; r < 3; ++r) {
        if (!exl3_k2_ok(l->k2[r], l->cb)) return fail(MAYA_E_UNSUPPORTED, "exl3_pack_experts: k2 %d with codebook %d", l->k2[r], l->cb);
        const int64_t k = r == 2 ? l->n_ff : l->n_embd, n = r == 2 ? l->n_embd : l->n_ff;
        if ((l->trellis[r] & 3) || (l->suh[r] & 1) || (l->svh[r] & 1)) return fail(MAYA_E_ARG, "exl3_pack_experts: a trellis needs 4-byte, suh / svh 2-byte alignment");
        end = end > l->trellis[r] + maya_exl3_trellis_bytes(k, n, l->k2[r]) ? end : l->trellis[r] + maya_exl3_trellis_bytes(k, n, l->k2[r]);
        end = end > l->suh[r] + 2 * (size_t) k ? end : l->suh[r] + 2 * (size_t) k;
        end = end > l->svh[r] + 2 * (size_t) n ? end : l->svh[r] + 2 * (size_t) n;
    }
    if (dst_stride < end) return fail(MAYA_E_ARG, "exl3_pack_experts: blobs of %zu bytes do not fit a stride of %zu", end, dst_stride);
    hipLaunchKernelGGL(exl3_pack_kernel, dim3(64, 9, (unsigned) n_expert), dim3(256), 0, as_stream(stream), pieces, *l, (uint8_t*) dst, dst_stride);
    MAYA_LAUNCHED("exl3_pack_kernel");
    return MAYA_OK;
}

int maya_exl3_reconstruct_inner(const uint32_t* trellis, int64_t k, int64_t n, int k2, int cb, uint16_t* dst, void* stream) {
    DeviceState* st;
    if (const int rc = current_state(&st)) return rc;
    if (!exl3_k2_ok(k2, cb)) return fail(MAYA_E_UNSUPPORTED, "exl3: k2 %d with codebook %d", k2, cb);
    if (!trellis || !dst) return fail(MAYA_E_ARG, "exl3 reconstruct: null pointer");
    if (k <= 0 || n <= 0 || k % 16 || n % 16) return fail(MAYA_E_SHAPE, "exl3 reconstruct: k %lld n %lld", (long long) k, (long long) n);
    const dim3 grid((unsigned) ((k / 16) * (n / 16)));
    hipStream_t s = as_stream(stream);
    if (cb == 2) hipLaunchKernelGGL(exl3_inner_kernel<2>, grid, dim3(256), 0, s, trellis, k, n, k2, dst);
    else if (cb == 1) hipLaunchKernelGGL(exl3_inner_kernel<1>, grid, dim3(256), 0, s, trellis, k, n, k2, dst);
    else hipLaunchKernelGGL(exl3_inner_kernel<0>, grid, dim3(256), 0, s, trellis, k, n, k2, dst);
    MAYA_LAUNCHED("exl3_inner_kernel");
    return MAYA_OK;
}

int maya_exl3_gate_up(const maya_exl3_args* a, void* stream) {
    DeviceState* st;
    if (const int rc = current_state(&st)) return rc;
    if (const int rc = exl3_check(a)) return rc;
    if (!a->x || !a->h) return fail(MAYA_E_ARG, "exl3 gate_up: null x or h");
    const int nt = a->grp_ptr && a->n_tokens >= 2 ? 2 : 1;
    int rc = 0;
    if (nt == 2 ? try_exl3_gu_split<2>(*a, *st, as_stream(stream), &rc) : try_exl3_gu_split<1>(*a, *st, as_stream(stream), &rc)) return rc;
    return nt == 2 ? launch_exl3_gate_up<2>(*a, *st, as_stream(stream)) : launch_exl3_gate_up<1>(*a, *st, as_stream(stream));
}

int maya_exl3_down(const maya_exl3_args* a, void* stream) {
    DeviceState* st;
    if (const int rc = current_state(&st)) return rc;
    if (const int rc = exl3_check(a)) return rc;
    if (!a->h || !a->part || !a->out) return fail(MAYA_E_ARG, "exl3 down: null h, part or out");
    const int nt = a->grp_ptr && a->n_tokens >= 2 ? 2 : 1;
    const int rc = nt == 2 ? launch_exl3_down<2>(*a, *st, as_stream(stream)) : launch_exl3_down<1>(*a, *st, as_stream(stream));
    if (rc) return rc;
    const dim3 grid((unsigned) ((a->layout.n_embd + 255) / 256), (unsigned) a->n_tokens);
    hipLaunchKernelGGL(exl3_combine_kernel, grid, dim3(256), 0, as_stream(stream), *a, (const float*) a->part, 1);
    MAYA_LAUNCHED("exl3_combine_kernel");
    return MAYA_OK;
}

// A layer call's slices (exl3_slices_kernel): gate/up rows in four, down rows in two - one token's eight experts of 6144 x 1536
// are then 768 workgroups a launch, three a compute unit, instead of 384 that leave half of them with one workgroup and half
// with two, and the rotation of h is done once an entry - where every walk is a compile-time one; else none (0) and the stage
// calls' kernels.  One token at 4 bits 67.1 -> 58.9 us, 4 tokens at 3 bits 159.4 -> 156.9.
struct Exl3Slices {
    int gu, dn;
};
static Exl3Slices exl3_slices(const maya_exl3_layout& l) {
    if (!walk_is_fast(l, 0) || !walk_is_fast(l, 2) || l.k2[0] != l.k2[1]) return Exl3Slices{0, 0};
    const int be = l.n_embd / 128, bf = l.n_ff / 128;
    return Exl3Slices{be >= 4 ? 4 : 1, bf >= 2 ? 2 : 1};
}
struct Exl3Ws {
    uint64_t *plan_ptr, *grp_ptr;
    int32_t *grp_start, *grp_ent, *n_groups;
    float *h, *part;   // (slices: h holds the rotated FP16 input of down, part the gate/up slices' sums)
    float* dn;         // (slices: the down slices' partial outputs - one token's down launch still reads the gate/up sums)
    uint32_t* done;    // (slices: a counter a 128-column block of the output)
    size_t bytes;
};
static Exl3Ws exl3_carve(const maya_exl3_layout& l, int n_tokens, int k, uint8_t* base) {
    Exl3Ws w{};
    size_t off = 0;
    const int ne = n_tokens * k;
    auto take = [&](size_t n) {
        uint8_t* p = base ? base + off : nullptr;
        off += (n + 255) & ~(size_t) 255;
        return p;
    };
    w.plan_ptr = (uint64_t*) take(sizeof(uint64_t) * ne);
    w.grp_ptr = (uint64_t*) take(sizeof(uint64_t) * ne);
    w.grp_start = (int32_t*) take(sizeof(int32_t) * (ne + 1));
    w.grp_ent = (int32_t*) take(sizeof(int32_t) * ne);
    w.n_groups = (int32_t*) take(sizeof(int32_t));
    w.h = (float*) take(sizeof(float) * (size_t) ne * l.n_ff);
    const Exl3Slices sl = exl3_slices(l);
    w.part = (float*) take(sizeof(float) * (size_t) ne * (sl.gu ? (size_t) 2 * sl.gu * l.n_ff : (size_t) l.n_embd));
    w.dn = (float*) take(sizeof(float) * (size_t) ne * sl.dn * l.n_embd);
    w.done = (uint32_t*) take(sl.dn ? sizeof(uint32_t) * kDoneStride * (size_t) (l.n_embd / 128) : 0);
    w.bytes = off;
    return w;
}
size_t maya_exl3_workspace_bytes(const maya_exl3_layout* l, int n_tokens, int k) {
    if (!l || n_tokens < 1 || n_tokens > MAYA_MAX_TOKENS || k < 1 || k > MAYA_MAX_K || l->n_embd <= 0 || l->n_ff <= 0) return 0;
    return exl3_carve(*l, n_tokens, k, nullptr).bytes;
}

int maya_exl3_layer_decode(const maya_exl3_layout* l, const uint64_t* expert_table, int n_expert, int k, const float* logits,
                           const float* x, int n_tokens, float limit, const float* add, int32_t* ids, float* weights,
                           float* out, void* workspace, size_t workspace_bytes, void* stream) {
    if (!l || !expert_table || !x || !ids || !weights || !out || !workspace) return fail(MAYA_E_ARG, "exl3 layer: null pointer");
    if (n_tokens < 1 || n_tokens > MAYA_MAX_TOKENS || k < 1 || k > MAYA_MAX_K) return fail(MAYA_E_SHAPE, "exl3 layer: n_tokens %d / k %d", n_tokens, k);
    if (((uintptr_t) workspace & 255) != 0) return fail(MAYA_E_ARG, "exl3 layer: workspace not 256-byte aligned");
    const Exl3Ws w = exl3_carve(*l, n_tokens, k, (uint8_t*) workspace);
    if (workspace_bytes < w.bytes) return fail(MAYA_E_ARG, "exl3 layer: workspace %zu < %zu bytes", workspace_bytes, w.bytes);
    int rc;
    bool grouped = false;
    const Exl3Slices sl = exl3_slices(*l);
    // one token on the sliced kernels: the router rides in the gate/up launch (a launch less before it:
    // 6144 x 1536 at 4 bits 50.2 -> 46.3 us, 4096 x 1280 34.8 -> 31.8, 2048 x 768 23.0 -> 19.1)
    const bool head = logits && n_tokens == 1 && sl.gu != 0 && n_expert <= 256 && k < n_expert;
    if (head) {
    } else if (logits && n_tokens > 1 && maya_moe_route_window_ok(nullptr, n_tokens, n_expert, k)) {   // route, plan and group in one launch
        if ((rc = maya_moe_route_window(nullptr, logits, n_tokens, n_expert, k, expert_table, ids, weights, w.plan_ptr, w.grp_ptr, w.grp_start,
                                        w.grp_ent, w.n_groups, stream)))
            return rc;
        grouped = true;
    } else if (logits) {   // route and plan in one launch; null: ids / weights are given
        if ((rc = maya_moe_route_plan(nullptr, logits, n_tokens, n_expert, k, expert_table, ids, weights, w.plan_ptr, stream))) return rc;
    } else if ((rc = maya_moe_plan(ids, n_tokens * k, expert_table, n_expert, w.plan_ptr, stream))) return rc;
    maya_exl3_args a{};
    a.layout = *l;
    a.n_tokens = n_tokens;
    a.k = k;
    a.plan_ptr = w.plan_ptr;
    a.plan_w = weights;
    if (n_tokens > 1) {
        if (!grouped && (rc = maya_moe_group(w.plan_ptr, n_tokens * k, w.grp_ptr, w.grp_start, w.grp_ent, w.n_groups, stream))) return rc;
        a.grp_ptr = w.grp_ptr;
        a.grp_start = w.grp_start;
        a.grp_ent = w.grp_ent;
        a.n_groups = w.n_groups;
    }
    a.limit = limit;
    a.x = x;
    a.h = w.h;
    a.part = w.part;
    a.add = add;
    a.out = out;
    if (sl.gu == 0) {
        if ((rc = maya_exl3_gate_up(&a, stream))) return rc;
        return maya_exl3_down(&a, stream);
    }
    DeviceState* st;
    if ((rc = current_state(&st))) return rc;
    if ((rc = exl3_check(&a))) return rc;
    hipStream_t s = as_stream(stream);
    __half* hr = (__half*) w.h;
    // tokens that share one decode of the weights: four where an expert has an entry or more on the average
    // (16 tokens top-8 of 48 experts: 244 us with two before, 186; of 160, 0.8 entries an expert: 451 with two, 468 with four), else two
    const int nt = n_tokens == 1 ? 1 : n_tokens >= 4 && n_tokens * k >= n_expert ? 4 : 2;
    const __half* in = n_tokens == 1 ? nullptr : hr;
    // The combine rides in the down launch up to four tokens: 6144 x 1536 at 3 bits, two tokens 90.3 -> 85.5 us, four 155.5 -> 152;
    // 4096 x 1280 at 4 bits, one token (with h made there too) 41.5 -> 34.8, four 108.2 -> 103.6.  From eight on nothing was
    // gained (256.6 -> 259.9): one workgroup a column block then adds up eight tokens, and the launch saved is one in sixty.
    uint32_t* done = n_tokens <= 4 && nt <= 2 ? w.done : nullptr;
    auto slices = [&](auto ntc, auto down, auto comb, int S, float* P) {
        return launch_exl3_slices<decltype(ntc)::value, decltype(down)::value, decltype(comb)::value>(a, S, in, w.part, sl.gu, P, done, true, *st, s);
    };
    using std::false_type, std::true_type;
    const std::integral_constant<int, 1> one;
    const std::integral_constant<int, 2> two;
    const std::integral_constant<int, 4> four;
    if ((rc = nt == 4   ? slices(four, false_type{}, false_type{}, sl.gu, w.part)
              : nt == 2 ? slices(two, false_type{}, false_type{}, sl.gu, w.part)
              : head    ? launch_exl3_slices<1, false, false, true>(a, sl.gu, in, w.part, sl.gu, w.part, done, true, *st, s,
                                                                    Exl3Head{logits, expert_table, n_expert, ids, weights, w.plan_ptr})
                        : slices(one, false_type{}, false_type{}, sl.gu, w.part)))
        return rc;
    if (in && (rc = launch_exl3_swiglu(a, sl.gu, w.part, hr, s))) return rc;
    rc = nt == 4   ? slices(four, true_type{}, false_type{}, sl.dn, w.dn)
         : nt == 1 ? slices(one, true_type{}, true_type{}, sl.dn, w.dn)
         : done    ? slices(two, true_type{}, true_type{}, sl.dn, w.dn)
                   : slices(two, true_type{}, false_type{}, sl.dn, w.dn);
    if (rc || done) return rc;
    hipLaunchKernelGGL(exl3_combine_kernel, dim3((unsigned) ((l->n_embd + 255) / 256), (unsigned) n_tokens), dim3(256), 0, s, a, (const float*) w.dn, sl.dn);
    MAYA_LAUNCHED("exl3_combine_kernel");
    return MAYA_OK;
}

}  // extern "C"
