// maya_prefill.hip - a prompt chunk's routed experts on gfx950: the device-side plan (count, scan, stable scatter, tile
// list), the Q8_K activation quantizers over the plan's rows, and the grouped GEMM of Q4_K weights with those
// activations on the int8 matrix cores (IQ2_S weights: maya_prefill_iq2s.hpp).
//
// The GEMM: a workgroup takes up to 128 rows of one expert (two tiles of the plan) and a band of weight rows; each of its 4 waves
// takes 32 weight rows (gate/up: the gate rows of 16 features and their up rows, so the SwiGLU stays inside the wave).  A Q4_K
// weight is two int8 planes (its code times the low and the high 3 bits of its sub-block's scale), and v_mfma_i32_32x32x32_i8 sums
// a whole 256-value super-block of either exactly; the two F32 scales and the minimums' term are applied once an output a
// super-block.  Weights and activations go from HBM to LDS without registers, about two super-blocks and two or three row groups ahead.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <math.h>
#include <stdint.h>

#include "maya_host.h"

namespace maya {

constexpr int kPfRows = 64;        // rows of a tile
constexpr int kPlanThreads = 1024;
constexpr int kPlanWaves = kPlanThreads / 64;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------------------------------- the plan
// An expert's rows keep the entries' order: entry e sits behind every entry of a lower expert and behind the earlier entries of
// its own.  Each workgroup scatters one share of the entries, its waves a contiguous run of them each, and counts ALL entries
// for itself - those in front of its share, its waves' own, those behind - so nothing passes between workgroups and the plan
// stays one launch with no scratch: an entry costs a load and an LDS add a workgroup, the scatter (a chain of LDS steps a
// 64-entry chunk) runs on as many workgroups as there are runs of 1024 entries.  32768 entries over 288 experts: 193 us with
// one workgroup scattering all 32 chunks a wave, 11.9 us like this; 4096 entries over 256: 12 us, 7.5 us.
// dynamic LDS: [kPlanWaves][n_expert] 64-bit lane masks (with_masks), seg[kPlanWaves][n_expert] counts -> bases,
// before[n_expert], total[n_expert], base[n_expert + 1], tbase[n_expert + 1], with a work list wbase[n_expert + 1]

// What a layer call's GEMMs are to do, a row of their grids an item (a stage call has the plan's tiles only).  Every row of the grid
// but the last ones has work.  With a workgroup for each tile of 64 rows, the second tile of every pair was a workgroup that
// returned at once; workgroups go to an XCD's shader engines in turn whatever they do and in order, so with few bands of weight rows an
// XCD some engines got the work and the others the returns.  Microseconds a layer call, tiles and items: 128 experts
// of 4096 x 512 (8 bands), 94 rows each, Q4_K 393 -> 327, IQ2_S 379 -> 305; 288 of 3072 x 1536 (24 bands) 1445 -> 1314; 512 tokens,
// skewed, of 256 experts of 7168 x 2048 (32 and 56) 836 -> 808; 4096 tokens of 288 of 4096 x 2048 (32) 2490 -> 2462.
// Workgroups that stay and take item after item from a counter were slower than one an item: 4096 tokens 2470, the skewed 512
// 832 (an item's stores have to land before the next one's copies can be told apart from them; a new workgroup does not wait).
// So was finding the leading tiles in the GEMM from the plan's list: 2595.
struct PfItem {
    uint64_t blob;   // an expert's bytes
    int32_t row0, nrows;   // of its rows
};
struct PfWork {
    PfItem* list;
    int32_t* n;      // [1] items
    int rows;        // of an item at most: a power of two
    bool few;        // IQ2_S products: on the kernel for few rows an expert
};
constexpr int kPlanMaxGroups = 64;   // (at 1 << 20 entries the counting would outweigh the scatter)
__global__ __launch_bounds__(kPlanThreads) void prefill_plan_kernel(const int32_t* __restrict__ ids, int n_entries,
                                                                    const uint64_t* __restrict__ table, int n_expert,
                                                                    maya_prefill_plan p, int max_tiles, int with_masks, PfWork work) {
    extern __shared__ __attribute__((aligned(16))) int32_t sm[];
    unsigned long long* mask = with_masks ? (unsigned long long*) sm : nullptr;
    int32_t* seg = sm + (with_masks ? 2 * kPlanWaves * n_expert : 0);
    int32_t* before = seg + kPlanWaves * n_expert;
    int32_t* total = before + n_expert;              // (first the count of the entries behind the share)
    int32_t* base = total + n_expert;
    int32_t* tbase = base + n_expert + 1;
    int32_t* wbase = tbase + n_expert + 1;
    __shared__ unsigned long long resident[MAYA_MAX_EXPERTS / 64];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    uint64_t blob;   // (of expert tid)
    {
        blob = tid < n_expert ? table[tid] : 0ull;
        const unsigned long long r = __ballot(blob != 0ull);   // (n_expert <= kPlanThreads: checked on the host)
        if (lane == 0) resident[wave] = r;
    }
    for (int i = tid; i < (kPlanWaves + 2) * n_expert; i += kPlanThreads) seg[i] = 0;
    if (mask != nullptr)
        for (int i = tid; i < kPlanWaves * n_expert; i += kPlanThreads) mask[i] = 0ull;
    __syncthreads();
    const int per = (((n_entries + kPlanWaves * (int) gridDim.x - 1) / (kPlanWaves * (int) gridDim.x)) + 63) & ~63;   // whole chunks of 64
    const int lo = ((int) blockIdx.x * kPlanWaves + wave) * per, hi = min(n_entries, lo + per);
    auto expert_of = [&](int e) {
        const int x = ids[e];
        return (x >= 0 && x < n_expert && ((resident[x >> 6] >> (x & 63)) & 1ull)) ? x : -1;
    };
    auto count = [&](int from, int to, int step, int32_t* into) {   // (several loads in flight: the adds wait for none of their own)
        for (int e0 = from; e0 < to; e0 += 8 * step) {
            int x[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = e0 + i * step < to ? ids[e0 + i * step] : -1;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (x[i] >= 0 && x[i] < n_expert && ((resident[x[i] >> 6] >> (x[i] & 63)) & 1ull)) atomicAdd(&into[x[i]], 1);
        }
    };
    const int first = min(n_entries, (int) blockIdx.x * kPlanWaves * per), last = min(n_entries, first + kPlanWaves * per);
    count(tid, first, kPlanThreads, before);
    count(lo + lane, hi, 64, seg + wave * n_expert);
    count(last + tid, n_entries, kPlanThreads, total);
    __syncthreads();
    // per expert: the waves' counts -> offsets from the expert's first row, and the total
    for (int x = tid; x < n_expert; x += kPlanThreads) {
        int run = before[x];
        for (int w = 0; w < kPlanWaves; ++w) {
            const int c = seg[w * n_expert + x];
            seg[w * n_expert + x] = run;
            run += c;
        }
        total[x] += run;
    }
    __syncthreads();
    // the experts' first rows (wave 0), tiles (wave 1) and items (wave 2): a lane a run of experts, a scan over the lanes between two passes
    auto first_of = [&](auto size, int32_t* o) {
        const int per_lane = (n_expert + 63) >> 6, x0 = lane * per_lane;
        int local = 0;
        for (int i = 0; i < per_lane; ++i)
            if (x0 + i < n_expert) local += size(x0 + i);
        int incl = local;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int up = __shfl_up(incl, d, 64);
            if (lane >= d) incl += up;
        }
        int run = incl - local;
        for (int i = 0; i < per_lane; ++i)
            if (x0 + i < n_expert) {
                o[x0 + i] = run;
                run += size(x0 + i);
                if (x0 + i == n_expert - 1) o[n_expert] = run;
            }
    };
    if (wave == 0) first_of([&](int x) { return total[x]; }, base);
    if (wave == 1) first_of([&](int x) { return (total[x] + kPfRows - 1) / kPfRows; }, tbase);
    if (wave == 2 && work.list != nullptr) {
        const int log2_rows = __ffs(work.rows) - 1;   // (a division would make this wave the one that the others wait for)
        first_of([&](int x) { return (total[x] + work.rows - 1) >> log2_rows; }, wbase);
    }
    __syncthreads();
    if (blockIdx.x == 0) {
        for (int x = tid; x <= n_expert; x += kPlanThreads) p.bounds[x] = base[x];
        // tiles: expert x's rows in runs of kPfRows
        for (int x = tid; x < n_expert; x += kPlanThreads)
            for (int t = tbase[x]; t < min(tbase[x + 1], max_tiles); ++t) {
                p.tile_expert[t] = x;
                p.tile_row0[t] = base[x] + (t - tbase[x]) * kPfRows;
            }
        if (tid == 0) *p.n_tiles = min(tbase[n_expert], max_tiles);
    }
    if (work.list != nullptr && blockIdx.x == min(1u, gridDim.x - 1)) {   // the GEMMs' work list: every expert's rows in runs of work.rows
        if (tid == 0) *work.n = wbase[n_expert];
        if (tid < n_expert)
            for (int r = 0, t = wbase[tid]; r < total[tid]; r += work.rows, ++t) work.list[t] = {blob, base[tid] + r, min(work.rows, total[tid] - r)};
    }
    // the stable scatter: 64 entries a step, a lane's rank = the earlier lanes of the step with its expert
    for (int c0 = lo; c0 < hi; c0 += 64) {
        const int e = c0 + lane;
        const int x = e < hi ? expert_of(e) : -1;
        int rank = 0, cnt = 0;
        if (mask != nullptr) {
            // every lane sets its bit in its expert's word; the word then tells each lane how many earlier lanes share its
            // expert (LDS operations of one wave complete in order); the expert's last lane clears the word again
            unsigned long long* mk = mask + (size_t) wave * n_expert;
            if (x >= 0) atomicOr(&mk[x], 1ull << lane);
            __builtin_amdgcn_wave_barrier();
            if (x >= 0) {
                const unsigned long long m = mk[x];
                rank = __popcll(m & ((1ull << lane) - 1ull));
                cnt = __popcll(m);
            }
            __builtin_amdgcn_wave_barrier();
            if (x >= 0 && rank == cnt - 1) mk[x] = 0ull;
        }
        unsigned long long todo = mask != nullptr ? 0ull : __ballot(x >= 0);
        while (todo) {
            const int leader = __ffsll((long long) todo) - 1;
            const int lx = __shfl(x, leader, 64);
            const unsigned long long same = __ballot(x == lx);
            if (x == lx) {
                rank = __popcll(same & ((1ull << lane) - 1ull));
                cnt = __popcll(same);
            }
            todo &= ~same;
        }
        if (x >= 0) {
            const int row = base[x] + seg[wave * n_expert + x] + rank;
            p.row_entry[row] = e;
            p.entry_row[e] = row;
        } else if (e < hi) {
            p.entry_row[e] = -1;
        }
        __builtin_amdgcn_wave_barrier();
        if (x >= 0 && rank == cnt - 1) seg[wave * n_expert + x] += cnt;   // one lane an expert: no two write one word
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_s_waitcnt(0);
    }
}

// ------------------------------------------------------------------------------------------ activation quantizer

// Q8_K rows - the activation format of the reference's CPU expert path for the K-quants
// (src/kernels/cuda/quantize_act.cu:161-207) - rounded 32 values a lane, 8 lanes a 256-value block (q8k_round_lane32: no
// LDS, no barrier): the block's signed maximum is the value at the FIRST largest magnitude, iscale = -127 / max,
// c = min(127, nearest_int(iscale x)), d = 1 / iscale; s = the sum of each 32 codes - what the minimums of a Q4_K
// sub-block multiply - as two FP16 digits, sum = lo + 64 hi with lo in 0..63: both are exact in FP16, and so is every
// product with a 6-bit minimum (times 64 for the high digit), which lets an FP16 matrix instruction form the integer
// sum over a block's 8 sub-blocks exactly.
struct PfLane {
    int y[8];      // 32 codes
    float d;
    int sum;
};
__device__ __forceinline__ PfLane pf_round_lane(const float (&v)[32], int lane) {
    PfLane o;
    q8k_round_lane32(v, [&](int i) { return 32 * (lane & 7) + i; }, o.y, o.d);
    int sum = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) sum = dot4(0x01010101, o.y[i], sum);
    o.sum = sum;
    return o;
}
__device__ __forceinline__ void pf_store_lane(const maya_prefill_act& o, size_t row, int64_t k, int64_t v0, int lane, const PfLane& c) {
    const size_t at = row * (size_t) k + (size_t) v0;
    int4* q = (int4*) (o.q + at);
    q[0] = make_int4(c.y[0], c.y[1], c.y[2], c.y[3]);
    q[1] = make_int4(c.y[4], c.y[5], c.y[6], c.y[7]);
    // (a block's 16 halves: the low digits of its 8 sub-blocks, then the high digits)
    _Float16* sp = (_Float16*) o.s + (at >> 8) * 16 + (lane & 7);
    sp[0] = (_Float16) (float) (c.sum & 63);
    sp[8] = (_Float16) (float) (c.sum >> 6);
    if ((lane & 7) == 0) o.d[at >> 8] = c.d;
}

// grid (k / 8192 rounded up, tokens): a token's values are rounded once and written to the rows of all its entries in the plan
template <int DT>
__global__ __launch_bounds__(256) void prefill_quant_kernel(const void* __restrict__ x, int64_t x_stride, maya_prefill_plan p,
                                                            int top_k, int64_t k, maya_prefill_act o) {
    const int t = blockIdx.y, lane = threadIdx.x & 63;
    const int64_t v0 = ((int64_t) blockIdx.x * 256 + threadIdx.x) * 32;
    const bool on = v0 < k;   // (k is a multiple of 256: the 8 lanes of a block are on or off together)
    float v[32];
    act_load32<DT>(x, (int64_t) t * x_stride + v0, on, v);
    const PfLane c = pf_round_lane(v, lane);
    if (!on) return;
    for (int j = 0; j < top_k; ++j) {
        const int row = p.entry_row[t * top_k + j];
        if (row < 0) continue;   // an entry of an expert that is not resident
        pf_store_lane(o, (size_t) row, k, v0, lane, c);
    }
}
// grid (k / 8192 rounded up, rows at most): the plan's row blockIdx.y of an F32 matrix (the SwiGLU outputs)
__global__ __launch_bounds__(256) void prefill_quant_rows_kernel(const float* __restrict__ x, maya_prefill_plan p, int n_expert,
                                                                 int64_t k, maya_prefill_act o) {
    const int row = blockIdx.y, lane = threadIdx.x & 63;
    if (row >= p.bounds[n_expert]) return;
    const int64_t v0 = ((int64_t) blockIdx.x * 256 + threadIdx.x) * 32;
    const bool on = v0 < k;
    float v[32];
    act_load32<MAYA_DT_F32>(x, (int64_t) row * k + v0, on, v);
    const PfLane c = pf_round_lane(v, lane);
    if (on) pf_store_lane(o, (size_t) row, k, v0, lane, c);
}

// ---------------------------------------------------------------------------------------------------- the GEMM
// out[row][n] = sum over 256-value blocks b of (d_w[n][b] d_x[row][b]) * sum_j sc[n][j] (q[n] . c[row])_j  -  the
// minimums' term: ggml_vec_dot_q4_K_q8_K's integer sums, exactly.  The 6-bit sub-block scale is split sc = 8 hi + lo, so
// q sc = 8 (q hi) + (q lo) with both products <= 105: two int8 planes of the weights.  Their products with the codes run
// on the int8 matrix cores and are accumulated in int32 over the whole 256-value block - the sub-block scales never leave
// the integer domain, and the vector ALU converts and scales once per 256 values.
struct PfGemm {
    const uint64_t* table;
    maya_prefill_plan plan;
    uint64_t off[2];       // gate and up (gate/up), down and unused (down): byte offsets of the matrices in a blob
    int64_t k, n;          // inner length, weight rows of one matrix
    int64_t row_bytes;
    maya_prefill_act x;    // the tile rows' activations [rows][k]
    float* out;            // gate/up: the SwiGLU outputs [rows][n] F32; down: part [rows][n]
    float limit;
    PfWork work;           // (list null: the plan's tiles, a workgroup each)
};

// The codes of a group of rows in LDS: 256 bytes a row, 16-byte chunk c of row r at position c ^ (r & 15): the 16 rows x 4
// k-groups of a matrix-core operand read then hit distinct banks.
typedef __attribute__((address_space(3))) void* pf_lptr;
typedef __attribute__((address_space(3))) uint8_t* pf_lds8;
// the 8 six-bit scales and 8 six-bit minimums of a Q4_K block's 12 bytes, as bytes of two words each
// (get_scale_min_k4, include/strata/artifact/dequant.hpp:162-172)
__device__ __forceinline__ void q4k_unpack_scales(uint32_t s0, uint32_t s1, uint32_t s2, uint32_t (&sc)[2], uint32_t (&mn)[2]) {
    sc[0] = s0 & 0x3f3f3f3fu;
    mn[0] = s1 & 0x3f3f3f3fu;
    sc[1] = (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u);
    mn[1] = ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u);
}

__device__ __forceinline__ float pf_swiglu(float g, float u, float limit) {
    if (limit > 0.0f && limit < INFINITY) {
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit);
    }
    return __fmul_rn(__fdiv_rn(g, __fadd_rn(1.0f, expf(-g))), u);
}

typedef unsigned short pf_u16x2 __attribute__((ext_vector_type(2)));

// LDS reads of the GEMM loop are written out by hand.  The compiler cannot tell which LDS buffer a direct-to-LDS copy
// fills, so before any LDS read of its own it waits for every copy in flight - here that would be the copy of the
// super-block two ahead, issued moments earlier.  These reads it does not see; each group is followed by a wait
// on the registers it filled (the values pass through the wait, so nothing that uses them can move above it).
__device__ __forceinline__ uint32_t pf_lds_addr(pf_lds8 p) { return (uint32_t) (uintptr_t) p; }
typedef int pf_i2 __attribute__((ext_vector_type(2)));
template <int OFF> __device__ __forceinline__ pf_i2 pf_lds_b64(uint32_t addr) {
    pf_i2 v;
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF) : "memory");
    return v;
}
template <int OFF> __device__ __forceinline__ v4f pf_lds_f32x4(uint32_t addr) {
    v4f v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF) : "memory");
    return v;
}
template <int OFF> __device__ __forceinline__ v4i pf_lds_i32x4(uint32_t addr) {
    v4i v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF) : "memory");
    return v;
}
// (... have landed once at most BUT later LDS reads are outstanding: LDS operations complete in order)
template <int BUT> __device__ __forceinline__ void pf_lds_wait_tail(v4f (&d)[4]) {
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3]) : "n"(BUT));
}
template <int BUT> __device__ __forceinline__ void pf_lds_wait_tail(v4i& a, v4f (&d)[4]) {
    asm volatile("s_waitcnt lgkmcnt(%5)" : "+v"(a), "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3]) : "n"(BUT));
}
// (compile-time loops over the row groups of a tile)
template <int M, int NMT, typename F> __device__ __forceinline__ void pf_for_m(F&& f) {
    if constexpr (M < NMT) {
        f(std::integral_constant<int, M>{});
        pf_for_m<M + 1, NMT>(f);
    }
}

typedef int pf_v16i __attribute__((ext_vector_type(16)));
typedef float pf_v16f __attribute__((ext_vector_type(16)));
typedef _Float16 pf_v8h __attribute__((ext_vector_type(8)));
typedef _Float16 pf_v2h __attribute__((ext_vector_type(2)));

// A tile of up to 4 x 32 rows against the wave's 32 weight rows (gate/up: the gate rows of 16 features, then their up rows;
// down: 32 output rows), on the 32x32 matrix instructions: lane (ln = lane & 31, kh = lane >> 5) holds 16 of a
// sub-block's 32 values of activation row ln (A operand, from LDS) and of weight row ln (B operand, decoded in
// registers), and 16 outputs: weight row ln against the rows 8 b + 4 kh + r (b, r = 0..3) of the 32.  The 32-cycle
// instructions leave the vector ALU about six slots each; the 16-cycle 16x16 forms leave it none.
//
// The work goes by passes: a pass is one group of 32 rows against one super-block.  A super-block's weights are decoded in its
// first pass and stay in 64 registers for the others, so a tile of 128 rows pays a quarter of the decode a row group:
// 12 vector instructions a matrix instruction at 64 rows with a decode each, 7 now.
//
// Weights and activations both go to LDS without registers, and a lane reads its pieces from there.  A lane that loads its
// own weight row from memory makes each lane of the instruction a cache access of its own: 64 clocks a compute unit for
// 1 KB out of L2, five such loads a wave a super-block, and the data path of the cache busy 85 % of the kernel; a copy takes it by
// eight lanes in a run (16 clocks).  Q4_K rows come in pieces of 128 bytes, not in blocks of 144: a block lies in two or three
// cache lines, two of which its neighbours ask for again, and a compute unit has about 400 line requests in flight (32 copies of
// 144-byte runs, 48 of 128-byte ones, before the next one waits).  The copies of a super-block wait 320 clocks to be issued
// where they waited 1265, and chunks of few rows an expert take 6 to 10 % less: 64 tokens top-8 of 256 experts of 7168 x 2048 1047 ->
// 945 us, 256 of 288 of 4096 x 2048 848 -> 765, 512 under a skewed routing 835 -> 814; where every expert fills its tiles
// nothing changes (4096 tokens 2435).
//
// Tiles of up to 24 rows (NB blocks of 8) take the codes themselves to the matrix cores, one instruction a sub-block instead of
// two planes': the sub-block sums of their few rows times the scales cost less on the vector ALU (4 multiply-adds a lane for 8
// rows) than the planes' 64 multiplies and 8 matrix instructions, up to 24 rows; at 32 the two forms take the same.
//
// Measured, one box: 4096 tokens top-8 of 288 experts of 4096 x 2048, gate/up 1817 -> 1420 us, down 891 -> 745; 512 tokens
// top-8 of 256 experts of 7168 x 2048 under a skewed routing (70 of its 93 experts with 24 rows or fewer), 627 -> 520 and 336 ->
// 291.  What bounds it: on full tiles vector issue (59 % of the cycles) and matrix time (50 %), at the 1.75 GHz that this
// load leaves of 2.4; few rows an expert stream their weights at 3.2 TB/s, of 5.2 without arithmetic.
constexpr int kPfPlane = 32 * 256;                   // codes of a pass
constexpr int kPfSlotS = kPfPlane, kPfSlotD = kPfSlotS + 1024, kPfSlot = kPfSlotD + 256;   // codes [32][256], sums [32][16], scales [32]

// The tile's activations, a row group of a super-block at a time.  Every group but the last is whole: its copies are the first
// one's at another scalar offset.  Rows past the tile's end repeat its last row (their results are never stored).
template <bool SUMS> struct PfRowsDma {   // SUMS: with the code sums that a type with minimums wants
    __amdgpu_buffer_rsrc_t rq, rs, rd;
    uint32_t oq[2], os, od, lq[2], ls, ld;   // the first group's offsets, the last one's
    int wave, k;
    __device__ __forceinline__ void init(const PfGemm& a, int row0, int nrows, int groups, int wave_, int lane) {
        wave = wave_;
        k = (int) a.k;
        const int last = nrows - 1;
        rq = __builtin_amdgcn_make_buffer_rsrc((void*) (a.x.q + (size_t) row0 * a.k), 0, (int) (nrows * a.k), 0x00020000);
        rs = __builtin_amdgcn_make_buffer_rsrc((void*) (a.x.s + (size_t) row0 * (a.k >> 4)), 0, (int) (nrows * (a.k >> 5) * 4), 0x00020000);
        rd = __builtin_amdgcn_make_buffer_rsrc((void*) (a.x.d + (size_t) row0 * (a.k >> 8)), 0, (int) (nrows * (a.k >> 8) * 4), 0x00020000);
        const int l0 = 32 * (groups - 1);
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const int r = 4 * (wave + 4 * n) + (lane >> 4), c = ((lane & 15) ^ (r & 15)) * 16;   // rows 4 i .. 4 i + 3, i = wave + 4 n
            oq[n] = (uint32_t) (r * k + c);
            lq[n] = (uint32_t) (min(l0 + r, last) * k + c);
        }
        os = (uint32_t) ((lane >> 1) * (k >> 5) * 4 + (lane & 1) * 16);
        ls = (uint32_t) (min(l0 + (lane >> 1), last) * (k >> 5) * 4 + (lane & 1) * 16);
        od = (uint32_t) ((lane & 31) * (k >> 8) * 4);
        ld = (uint32_t) (min(l0 + (lane & 31), last) * (k >> 8) * 4);
    }
    template <bool LAST> __device__ __forceinline__ void copy(pf_lds8 buf, int sb, int m) const {
        const int at = LAST ? 0 : 32 * m;
#pragma unroll
        for (int n = 0; n < 2; ++n)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rq, (pf_lptr) (buf + (wave + 4 * n) * 1024), 16, LAST ? lq[n] : oq[n], sb * 256 + at * k, 0, 0);
        if (SUMS && wave == 0) __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (pf_lptr) (buf + kPfSlotS), 16, LAST ? ls : os, sb * 32 + at * (k >> 3), 0, 0);
        if (wave == 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(rd, (pf_lptr) (buf + kPfSlotD), 4, LAST ? ld : od, sb * 4 + at * (k >> 6), 0, 0);
    }
};

template <int BUT> __device__ __forceinline__ void pf_lds_wait1(v4i& r) { asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(r) : "n"(BUT)); }
// FP16 1024 + c of two bytes c of w, as a pair
__device__ __forceinline__ pf_v2h pf_bytes_1024(uint32_t w, uint32_t sel) {
    return __builtin_bit_cast(pf_v2h, __builtin_amdgcn_perm(0x64646464u, w, sel));
}

// What the tile wants of a weight type: the copies of a wave's 32 rows of a super-block into LDS (kCopies instructions, kWave
// bytes), a lane's reads of its row's part of them, and the two planes of a sub-block out of the registers these filled.
template <bool GU> struct PfQ4K {
    static constexpr bool kSums = true;
    // A piece is 128 bytes of each of the 32 rows, 16-byte granule g of row r at g ^ (r / 2 & 7): the 16-byte reads of 16 rows meet
    // every bank once.  A super-block's nine granules lie in two pieces, a ring of three holds the one behind them as well.  (A fourth,
    // in the place of the activations' fourth slot or not, does not fit two workgroups' LDS; the fourth slot gave nothing.)
    static constexpr int kPiece = 32 * 128, kLdsAt = 0, kWave = 3 * kPiece;
    static constexpr int kCopies = 4, kRing = 3;   // (kRing: passes of activations in LDS, all but one of them ahead)
    static constexpr int kOneGroupBut = kCopies;   // (the piece that every eighth super-block ends in was asked for one super-block ago)
    static constexpr int kHiFactor = 8, kLook = 0;   // (a sum is lo + 8 hi; LDS look-ups of a sub-block's planes)
    __amdgpu_buffer_rsrc_t r[2];   // 16 rows each
    uint32_t at[2], row_at, swizzle, m_shift;   // at: a lane's offsets in the piece to ask for next
    int lane, left, cur;           // left: the pieces not asked for yet; cur: where the ring's first one sits
    pf_v2h m_mul, m_add;
    __device__ __forceinline__ void init(const PfGemm& a, const uint8_t* blob, int64_t n0, int lane_) {
        const int row_bytes = (int) a.row_bytes;
        lane = lane_, left = (row_bytes + 127) >> 7, cur = 0;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            r[i] = __builtin_amdgcn_make_buffer_rsrc((void*) (blob + a.off[GU ? i : 0] + (size_t) (n0 + (GU ? 0 : 16 * i)) * a.row_bytes), 0, 16 * row_bytes, 0x00020000);
            at[i] = (uint32_t) ((8 * i + (lane >> 3)) * row_bytes + ((lane & 7) ^ (4 * i + (lane >> 4))) * 16);   // 8 rows a copy, 8 lanes a row
        }
        const int kh = lane >> 5;
        row_at = (lane & 31) * 128;
        swizzle = 16 * ((lane >> 1) & 7);
        m_shift = 2 * kh;
        m_mul = kh ? pf_v2h{(_Float16) 16.0f, (_Float16) 16.0f} : pf_v2h{(_Float16) 1.0f, (_Float16) 1.0f};
        m_add = kh ? pf_v2h{(_Float16) -16384.0f, (_Float16) -16384.0f} : pf_v2h{(_Float16) -1024.0f, (_Float16) -1024.0f};
    }
    __device__ __forceinline__ int behind(int slot) const { return slot == 2 * kPiece ? 0 : slot + kPiece; }
    // The next piece, to `to`.  (The piece is in the lanes' offsets, not in the scalar one, which need not take part in the buffer's range
    // check: a row's last piece goes on into the row behind it, and behind the matrix there may be nothing.)
    __device__ __forceinline__ void copy(pf_lds8 to) {
        if (left <= 0) return;
#pragma unroll
        for (int i = 0; i < 4; ++i) __builtin_amdgcn_raw_ptr_buffer_load_lds(r[i >> 1], (pf_lptr) (to + i * 1024), 16, at[i & 1], 0, 0, 0);
        at[0] += 128, at[1] += 128, --left;
    }
    __device__ __forceinline__ void first(pf_lds8 to) {
#pragma unroll
        for (int i = 0; i < 3; ++i) copy(to + i * kPiece);
    }
    // super-block sb is in registers: the one or two pieces that it was the last to want make room
    __device__ __forceinline__ void next(pf_lds8 to, int sb) {
        copy(to + cur);
        cur = behind(cur);
        if ((sb & 7) == 7) {
            copy(to + cur);
            cur = behind(cur);
        }
    }
    struct Row {   // a lane's part of its row: the header, four 16-byte pieces of the codes (bytes 32 c + 16 kh of their 128: the low
                   // nibbles are 16 values of sub-block 2 c, the high ones of 2 c + 1), and what `open` makes of them
        v4i hdr, q[4];
        float d, ndmin;
        uint32_t sc[2];
        pf_u16x2 flo[2][2], fhi[2][2];
        pf_v8h mb;
    };
    __device__ __forceinline__ void read(Row& w, uint32_t base, int sb) const {
        const uint32_t here = base + row_at + cur, behind_it = base + row_at + behind(cur);
        const uint32_t g = 16 * (sb & 7);   // (granule 9 sb, in its piece)
        w.hdr = pf_lds_i32x4<0>(here + (g ^ swizzle));
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const uint32_t at = (16 * (lane >> 5) + g + 16 + 32 * c) ^ swizzle;   // (bit 7: in the piece behind)
            w.q[c] = pf_lds_i32x4<0>((at & 128 ? behind_it : here) + (at & 0x70));
        }
    }
    template <int BUT> __device__ __forceinline__ void wait(Row& w) const {
        asm volatile("s_waitcnt lgkmcnt(%5)" : "+v"(w.hdr), "+v"(w.q[0]), "+v"(w.q[1]), "+v"(w.q[2]), "+v"(w.q[3]) : "n"(BUT));
    }
    __device__ __forceinline__ void open(Row& w) const {
        uint32_t mn[2];
        w.d = f16_bits_to_f32((uint16_t) (w.hdr[0] & 0xffff));
        w.ndmin = -f16_bits_to_f32((uint16_t) ((uint32_t) w.hdr[0] >> 16));
        q4k_unpack_scales((uint32_t) w.hdr[1], (uint32_t) w.hdr[2], (uint32_t) w.hdr[3], w.sc, mn);
        // the scales' low and high digits as 16-bit pairs: [i][p] those of sub-blocks 4 i + p and 4 i + 2 + p
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                w.flo[i][p] = __builtin_bit_cast(pf_u16x2, (w.sc[i] >> (8 * p)) & 0x00070007u);
                w.fhi[i][p] = __builtin_bit_cast(pf_u16x2, (w.sc[i] >> (8 * p + 3)) & 0x00070007u);
            }
        // The minimums' operand: k = 0..7 pairs m_j with the sums' low digits, k = 8..15 pairs 64 m_j with their high digits.
        // A byte b behind 0x64 is FP16 1024 + b: m, or 4 m and 16 times that.
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t mw = mn[i] << m_shift;
            const pf_v2h t0 = __builtin_elementwise_fma(pf_bytes_1024(mw, 0x04010400u), m_mul, m_add);
            const pf_v2h t1 = __builtin_elementwise_fma(pf_bytes_1024(mw, 0x04030402u), m_mul, m_add);
            w.mb[4 * i] = t0[0], w.mb[4 * i + 1] = t0[1], w.mb[4 * i + 2] = t1[0], w.mb[4 * i + 3] = t1[1];
        }
    }
    template <int J> __device__ __forceinline__ void look(Row&) const {}
    template <int BUT> __device__ __forceinline__ void wait_look(int, Row&, v4i& x) const { pf_lds_wait1<BUT>(x); }
    __device__ __forceinline__ void planes(const Row& w, int j, v4i& wl, v4i& wh) const {
        const pf_u16x2 lo = w.flo[j >> 2][j & 1], hi = w.fhi[j >> 2][j & 1];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            // four 4-bit codes (one a byte) times a factor <= 7: no byte overflows, so one packed 16-bit multiply does it
            const pf_u16x2 c = __builtin_bit_cast(pf_u16x2, ((uint32_t) w.q[j >> 1][i] >> (4 * (j & 1))) & 0x0f0f0f0fu);
            wl[i] = __builtin_bit_cast(int, j & 2 ? c * lo.yy : c * lo.xx);
            wh[i] = __builtin_bit_cast(int, j & 2 ? c * hi.yy : c * hi.xx);
        }
    }
    __device__ __forceinline__ v4i codes(const Row& w, int j) const {
        v4i c;
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i] = (int) (((uint32_t) w.q[j >> 1][i] >> (4 * (j & 1))) & 0x0f0f0f0fu);
        return c;
    }
};

template <typename W> struct PfLds {   // the weight type's tables, the activations' ring, the weights of the 4 waves
    static constexpr int ring = W::kLdsAt, w = ring + W::kRing * kPfSlot, bytes = w + 4 * W::kWave;
};

// the rows that a workgroup computes, of the expert whose bytes are at blob
struct PfTile {
    const uint8_t* blob;
    int row0, nrows;
};

// NB: 0, or the blocks of 8 rows of a tile that takes the codes themselves to the matrix cores
template <typename W, bool GU, int NM, int NB = 0>
__device__ __forceinline__ void pf_tile(const PfGemm& a, pf_lds8 lds, const PfTile& t) {
    const int row0 = t.row0, nrows = t.nrows;
    typedef PfLds<W> S;
    const int tid = threadIdx.x, lane = tid & 63, ln = lane & 31, kh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // the wave's first feature (gate/up) or output row (down): n is a multiple of 256, every workgroup has all its rows
    const int64_t n0 = GU ? (int64_t) blockIdx.x * 64 + wave * 16 : (int64_t) blockIdx.x * 128 + wave * 32;
    pf_v16f acc[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;

    const int nsb = (int) (a.k >> 8);
    PfRowsDma<W::kSums> dma;
    dma.init(a, row0, nrows, NM, wave, lane);
    W wts;
    const pf_lds8 wlds = lds + S::w + wave * W::kWave;
    // the copies of pass (sb, m) + kAhead go into the slot of the pass before (sb, m); in the prologue, of the first kAhead passes
    constexpr int kAhead = W::kRing - 1;
    auto copy_pass = [&](auto mc, int sb, int slot) {   // (M in 0 .. NM - 1 + kAhead: pass M of super-block sb on)
        constexpr int M = decltype(mc)::value, m = M % NM;
        const int b = sb + M / NM;
        if (b < nsb) dma.template copy<m == NM - 1>(lds + S::ring + slot * kPfSlot, b, m);
    };
    pf_for_m<0, kAhead>([&](auto mc) { copy_pass(mc, 0, decltype(mc)::value); });
    int slot = 0;
    wts.init(a, t.blob, n0, lane);
    wts.first(wlds);
    // a lane's 16 codes of sub-block j: the row's 16-byte chunk 2 j + kh, which sits at that index ^ (the row & 15)
    const uint32_t a_base = ln * 256 + (((ln & 15) ^ kh) << 4);
    const uint32_t lbase = pf_lds_addr(lds) + S::ring, wbase = pf_lds_addr(wlds);
    for (int sb = 0; sb < nsb; ++sb) {
        const bool steady = sb + 2 < nsb;
        v4i P[8][2];   // the block's planes: sub-block, low and high digit
        typename W::Row w;
        pf_for_m<0, NM>([&](auto mc) {
            constexpr int m = decltype(mc)::value;
            // What this pass reads has landed once only what was issued after it is in flight: the activations of the passes behind it
            // (at least two copies a wave each) and the weights issued in the passes since its own activations were; with one group a
            // super-block its weights decide.
            constexpr int kIssued = [] {
                int n = 0;
                for (int i = 1; i <= kAhead; ++i) n += (m + 4 * NM - i) % NM == 0;
                return n;
            }();
            constexpr int kActs = 2 * (kAhead - 1) + W::kCopies * kIssued, kBut = NM == 1 && W::kOneGroupBut < kActs ? W::kOneGroupBut : kActs;
            if (!steady || (m == 0 && sb == 0)) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kBut) : "memory");
            const uint32_t lbuf = lbase + slot * kPfSlot;
            if constexpr (m == 0) wts.read(w, wbase, sb);
            copy_pass(std::integral_constant<int, m + kAhead>{}, sb, slot ? slot - 1 : kAhead);
            slot = slot == kAhead ? 0 : slot + 1;
            // The two plane products of the block, int32, a matrix instruction a sub-block and plane, accumulated over the 8
            // sub-blocks.  The activation operand is requested from LDS two sub-blocks ahead.
            pf_v16i dot[2];
            v4i xr[3];
            const uint32_t xa = lbuf + a_base;
            xr[0] = pf_lds_i32x4<0>(xa);
            xr[1] = pf_lds_i32x4<0>(xa ^ 32);
            int sum[NB ? 4 * NB : 1];
            pf_v16i part[NB ? 3 : 1];   // (sub-block sums, worked off two sub-blocks on: a matrix instruction's results take a while)
            auto add_part = [&](int jj) {
                if constexpr (NB != 0) {
                    const int scale = (int) ((w.sc[jj >> 2] >> (8 * (jj & 3))) & 0x3fu);
#pragma unroll
                    for (int i = 0; i < 4 * NB; ++i) {
                        sum[i] = __mul24(part[jj % 3][i], scale) + (jj ? sum[i] : 0);
                        asm("" : "+v"(sum[i]));   // (keeps multiply and add one instruction)
                    }
                    // (the registers of rows that are not there stay taken until now: given away behind the matrix instruction, they
                    // made the next instruction wait until it had written them)
                    asm volatile("" ::"v"(part[jj % 3]));
                }
            };
            if constexpr (m == 0) {
                wts.template wait<2>(w);
                wts.next(wlds, sb);
                wts.open(w);
                wts.template look<0>(w);
            }
            v4i sa;
            v4f dxr[4];
            pf_for_m<0, 8>([&](auto jc) {
                constexpr int jj = decltype(jc)::value;
                if constexpr (m == 0 && jj < 7) wts.template look<jj + 1>(w);
                if constexpr (jj < 6) xr[(jj + 2) % 3] = pf_lds_i32x4<0>(xa ^ (32 * (jj + 2)));
                if constexpr (jj == 6) {   // the closing stage's operands: the code sums, the block scales
                    if constexpr (W::kSums) sa = pf_lds_i32x4<kPfSlotS>(lbuf + ln * 32 + kh * 16);
                    const uint32_t at = lbuf + 16 * kh;
                    dxr[0] = pf_lds_f32x4<kPfSlotD>(at);
                    dxr[1] = pf_lds_f32x4<kPfSlotD + 32>(at);
                    dxr[2] = pf_lds_f32x4<kPfSlotD + 64>(at);
                    dxr[3] = pf_lds_f32x4<kPfSlotD + 96>(at);
                }
                // this sub-block's operands have landed once only the reads issued after them are outstanding (LDS answers in
                // order): the activations of the two sub-blocks behind it, the next one's look-ups, the closing stage's
                constexpr int kTail = 4 + (W::kSums ? 1 : 0), kNext = m == 0 && jj < 7 ? W::kLook : 0;
                constexpr int kAfter = (jj < 6 ? 2 : jj == 6 ? 1 + kTail : kTail) + kNext - (kNext && jj == 0 ? 1 : 0);
                if constexpr (m == 0) wts.template wait_look<kAfter>(jj, w, xr[jj % 3]);
                else pf_lds_wait1<kAfter>(xr[jj % 3]);
                const pf_v16i z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
                if constexpr (NB != 0) {
                    part[jj % 3] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xr[jj % 3], wts.codes(w, jj), z, 0, 0, 0);
                    if (jj > 1) add_part(jj - 2);
                } else {
                    if constexpr (m == 0) wts.planes(w, jj, P[jj][0], P[jj][1]);
                    dot[0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xr[jj % 3], P[jj][0], jj ? dot[0] : z, 0, 0, 0);
                    dot[1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(xr[jj % 3], P[jj][1], jj ? dot[1] : z, 0, 0, 0);
                }
            });
            // Once a block lo + 8 hi = the block's integer sum (< 2^25) and d_x (d_w sum - dmin_w minimums); the minimums' integer term
            // sum_j m_j (sum of sub-block j's codes) comes, exactly, from one FP16 matrix instruction (every operand and every
            // partial sum an integer below 2^24).
            // (a lane's outputs 4 b .. 4 b + 3 are the tile's rows 32 m + 8 b + 4 kh + 0..3: blocks of 8 rows past the
            // tile's last row are skipped - most tiles of a skewed routing hold 8 rows or fewer)
            const int nb = m == NM - 1 ? (nrows - 32 * m + 7) >> 3 : 4;
            if constexpr (W::kSums) {
                pf_lds_wait_tail<0>(sa, dxr);
                const pf_v16f z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
                const pf_v16f mins = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(pf_v8h, sa), w.mb, z, 0, 0, 0);
                if constexpr (NB != 0) add_part(6), add_part(7);
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    if (NB ? b < NB : m < NM - 1 || b < nb) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int i = 4 * b + r;
                            const float t = fmaf(w.ndmin, mins[i], __fmul_rn(w.d, (float) (NB ? sum[NB ? i : 0] : dot[0][i] + W::kHiFactor * dot[1][i])));
                            acc[m][i] = fmaf(dxr[b][r], t, acc[m][i]);
                        }
                    }
                }
            } else {
                pf_lds_wait_tail<0>(dxr);
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    if (m < NM - 1 || b < nb) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int i = 4 * b + r;
                            acc[m][i] = fmaf(__fmul_rn(dxr[b][r], w.d), (float) (dot[0][i] + W::kHiFactor * dot[1][i]), acc[m][i]);
                        }
                    }
                }
            }
            asm volatile("" : "+v"(acc[m]));   // (here, not when the block's other passes are done: that would keep every pass's sums)
        });
    }
    if constexpr (!W::kSums) {
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[m][i] = __fmul_rn(acc[m][i], W::kOutFactor);
    }
    // outputs: lane (ln, kh) holds weight row ln for the tile's rows 32 m + 8 b + 4 kh + r (i = 4 b + r)
    pf_for_m<0, NM>([&](auto mc) {
        constexpr int m = decltype(mc)::value;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int r0 = 32 * m + 8 * b;
            if (NB ? b >= NB : m == NM - 1 && r0 >= nrows) continue;
            if constexpr (GU) {
                // The up row of a feature sits 16 lanes above its gate row.  One swap of every second 16 lanes between two rows'
                // values leaves the lanes of the gate rows with gate and up of the first, the others with those of the second.
                float* o = a.out + (size_t) (row0 + r0 + 4 * kh) * a.n + n0 + (ln & 15) + (ln < 16 ? 0 : a.n);
#pragma unroll
                for (int r = 0; r < 4; r += 2) {
                    const auto gu = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[m][4 * b + r]), __float_as_uint(acc[m][4 * b + r + 1]), false, false);
                    const float h = pf_swiglu(__uint_as_float(gu[0]), __uint_as_float(gu[1]), a.limit);
                    if (m < NM - 1 || r0 + 4 * kh + r + (ln >> 4) < nrows) o[(size_t) r * a.n] = h;
                }
            } else {
                float* o = a.out + (size_t) (row0 + r0 + 4 * kh) * a.n + n0 + ln;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (m < NM - 1 || r0 + 4 * kh + r < nrows) o[(size_t) r * a.n] = acc[m][4 * b + r];
            }
        }
    });
}

// The workgroup's rows: a listed tile, and with it the next one on the list where that goes on with the expert's rows and starts in
// the middle of 128 of them.  False where there are none: past the last tile, or the workgroup of the tile before takes them.
// (Both sides read the list itself, so a caller's part of it is what is computed.)  Every tile alone for a kernel that decodes its weights
// once a group of 32 rows whatever it is given (PAIRS false).
static_assert(2 * kPfRows == 4 * 32, "four row groups of a workgroup at most");
template <bool PAIRS>
__device__ __forceinline__ bool pf_my_tile(const PfGemm& a, PfTile& t) {
    const int tile = blockIdx.y, n = *a.plan.n_tiles;
    if (tile >= n) return false;
    const int ex = a.plan.tile_expert[tile];
    t.row0 = a.plan.tile_row0[tile];
    t.blob = (const uint8_t*) a.table[ex];
    if (!PAIRS) {
        t.nrows = min(kPfRows, a.plan.bounds[ex + 1] - t.row0);
        return true;
    }
    const int before = max(tile - 1, 0), behind = min(tile + 1, n - 1);
    const int bx = a.plan.tile_expert[before], b0 = a.plan.tile_row0[before], nx = a.plan.tile_expert[behind], n0 = a.plan.tile_row0[behind];
    const int first = a.plan.bounds[ex], at = (t.row0 - first) % (2 * kPfRows);
    if (at == kPfRows && bx == ex && b0 == t.row0 - kPfRows) return false;
    const bool two = at == 0 && nx == ex && n0 == t.row0 + kPfRows;
    t.nrows = min(two ? 2 * kPfRows : kPfRows, a.plan.bounds[ex + 1] - t.row0);
    return true;
}

// the same from the work list where there is one
template <bool PAIRS = true>
__device__ __forceinline__ bool pf_my_rows(const PfGemm& a, PfTile& t) {
    if (a.work.list == nullptr) return pf_my_tile<PAIRS>(a, t);
    if ((int) blockIdx.y >= *a.work.n) return false;
    const PfItem i = a.work.list[blockIdx.y];
    t.blob = (const uint8_t*) i.blob, t.row0 = i.row0, t.nrows = i.nrows;
    return true;
}

#include "maya_prefill_iq2s.hpp"

// grid (bands of weight rows, items or tiles at most)
template <bool GU>
__global__ __launch_bounds__(256, 2) void prefill_q4k_kernel(PfGemm a) {
    typedef PfQ4K<GU> W;
    __shared__ __attribute__((aligned(256))) uint8_t lds[PfLds<W>::bytes];
    PfTile t;
    if (!pf_my_rows(a, t)) return;
    if (t.nrows <= 8) pf_tile<W, GU, 1, 1>(a, (pf_lds8) lds, t);
    else if (t.nrows <= 16) pf_tile<W, GU, 1, 2>(a, (pf_lds8) lds, t);
    else if (t.nrows <= 24) pf_tile<W, GU, 1, 3>(a, (pf_lds8) lds, t);
    else if (t.nrows <= 32) pf_tile<W, GU, 1>(a, (pf_lds8) lds, t);
    else if (t.nrows <= 64) pf_tile<W, GU, 2>(a, (pf_lds8) lds, t);
    else if (t.nrows <= 96) pf_tile<W, GU, 3>(a, (pf_lds8) lds, t);
    else pf_tile<W, GU, 4>(a, (pf_lds8) lds, t);
}

template <int ODT>
__global__ __launch_bounds__(256) void prefill_combine_kernel(const int32_t* __restrict__ entry_row, const float* __restrict__ w,
                                                              const float* __restrict__ part, int k, int64_t n,
                                                              const float* __restrict__ add, void* __restrict__ out) {
    const int t = blockIdx.y;
    const int64_t c = (int64_t) blockIdx.x * 256 + threadIdx.x;
    if (c >= n) return;
    float sum = 0.0f;
    bool first = true;
    for (int j = 0; j < k; ++j) {
        const int row = entry_row[t * k + j];
        if (row < 0) continue;
        const float v = __fmul_rn(part[(size_t) row * n + c], w[t * k + j]);
        sum = first ? v : __fadd_rn(sum, v);
        first = false;
    }
    if (add) sum = __fadd_rn(sum, add[(size_t) t * n + c]);
    if constexpr (ODT == MAYA_DT_F32) ((float*) out)[(size_t) t * n + c] = sum;
    else if constexpr (ODT == MAYA_DT_BF16) {
        uint32_t u = __float_as_uint(sum);
        if ((u & 0x7fffffffu) > 0x7f800000u) u |= 0x00400000u;          // NaN stays NaN
        else u += 0x7fffu + ((u >> 16) & 1u);                            // round to nearest even
        ((uint16_t*) out)[(size_t) t * n + c] = (uint16_t) (u >> 16);
    } else ((__half*) out)[(size_t) t * n + c] = __float2half_rn(sum);
}

// the same, four columns a thread (n a multiple of 4, 16-byte aligned rows): the k rows' loads are issued together, the
// sum keeps the slot order
template <int ODT>
__global__ __launch_bounds__(256) void prefill_combine4_kernel(const int32_t* __restrict__ entry_row, const float* __restrict__ w,
                                                               const float* __restrict__ part, int k, int64_t n,
                                                               const float* __restrict__ add, void* __restrict__ out) {
    const int t = blockIdx.y;
    const int64_t c = ((int64_t) blockIdx.x * 256 + threadIdx.x) * 4;
    if (c >= n) return;
    float4 v[MAYA_MAX_K];
    float wj[MAYA_MAX_K];
    bool on[MAYA_MAX_K];
#pragma unroll
    for (int j = 0; j < MAYA_MAX_K; ++j) {
        const int row = j < k ? entry_row[t * k + j] : -1;
        on[j] = row >= 0;
        if (on[j]) {
            v[j] = *(const float4*) (part + (size_t) row * n + c);
            wj[j] = w[t * k + j];
        }
    }
    float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    bool first = true;
#pragma unroll
    for (int j = 0; j < MAYA_MAX_K; ++j) {
        if (!on[j]) continue;
        const float p[4] = {__fmul_rn(v[j].x, wj[j]), __fmul_rn(v[j].y, wj[j]), __fmul_rn(v[j].z, wj[j]), __fmul_rn(v[j].w, wj[j])};
#pragma unroll
        for (int i = 0; i < 4; ++i) sum[i] = first ? p[i] : __fadd_rn(sum[i], p[i]);
        first = false;
    }
    if (add) {
        const float4 a = *(const float4*) (add + (size_t) t * n + c);
        sum[0] = __fadd_rn(sum[0], a.x), sum[1] = __fadd_rn(sum[1], a.y), sum[2] = __fadd_rn(sum[2], a.z), sum[3] = __fadd_rn(sum[3], a.w);
    }
    if constexpr (ODT == MAYA_DT_F32) {
        *(float4*) ((float*) out + (size_t) t * n + c) = make_float4(sum[0], sum[1], sum[2], sum[3]);
    } else {
        uint16_t h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (ODT == MAYA_DT_BF16) {
                uint32_t u = __float_as_uint(sum[i]);
                if ((u & 0x7fffffffu) > 0x7f800000u) u |= 0x00400000u;          // NaN stays NaN
                else u += 0x7fffu + ((u >> 16) & 1u);                            // round to nearest even
                h[i] = (uint16_t) (u >> 16);
            } else {
                h[i] = __half_as_ushort(__float2half_rn(sum[i]));
            }
        }
        *(uint2*) ((uint16_t*) out + (size_t) t * n + c) = make_uint2(h[0] | ((uint32_t) h[1] << 16), h[2] | ((uint32_t) h[3] << 16));
    }
}

static bool plan_ok(const maya_prefill_plan* p) {
    return p && p->bounds && p->row_entry && p->entry_row && p->tile_expert && p->tile_row0 && p->n_tiles;
}
static bool act_ok(const maya_prefill_act& a) {
    return a.q && a.d && a.s && (((uintptr_t) a.q | (uintptr_t) a.s) & 15) == 0 && ((uintptr_t) a.d & 3) == 0;
}
// The rows of a GEMM's grid: every tile of a plan, or the items that a list can hold.
static unsigned pf_grid_rows(const PfWork& work, int n_entries, int n_expert) {
    return work.list ? (unsigned) (n_entries / work.rows + std::min(n_entries, n_expert)) : (unsigned) maya_moe_prefill_max_tiles(n_entries, n_expert);
}
// A stage call's: no list; the slots of a token, which it is not told, taken as 8.
static PfWork pf_stage_work(int n_entries, int n_expert) {
    PfWork w{};
    w.few = prefill_iq2s_few(n_entries / 8, n_entries, n_expert);
    return w;
}
template <bool GU>
static void pf_launch(const PfGemm& a, dim3 grid, hipStream_t s) {
    hipLaunchKernelGGL(prefill_q4k_kernel<GU>, grid, dim3(256), 0, s, a);
}

}  // namespace maya

using namespace maya;

static int pf_plan(const int32_t* ids, int n_entries, const uint64_t* expert_table, int n_expert, const maya_prefill_plan* plan,
                   const PfWork& work, void* stream) {
    DeviceState* st;
    if (const int rc = current_state(&st)) return rc;
    if (!ids || !expert_table || !plan_ok(plan)) return fail(MAYA_E_ARG, "prefill_plan: null pointer");
    if (n_entries <= 0 || n_entries > (1 << 20) || n_expert <= 0 || n_expert > MAYA_MAX_EXPERTS)
        return fail(MAYA_E_SHAPE, "prefill_plan: entries %d experts %d", n_entries, n_expert);
    // (a wave's 64-bit lane masks an expert ride along while LDS holds them beside the kernel's own 128 bytes: up to 771 experts with a
    // work list, 786 without; ballots beyond)
    size_t lds = sizeof(int32_t) * ((size_t) (kPlanWaves + 4) * n_expert + 2);
    if (work.list != nullptr) lds += sizeof(int32_t) * ((size_t) n_expert + 1);
    const size_t masks = sizeof(unsigned long long) * (size_t) kPlanWaves * n_expert;
    const int with_masks = lds + masks + 256 <= (size_t) st->lds_limit;
    if (with_masks) lds += masks;
    if (lds > 65536) MAYA_HIP(hipFuncSetAttribute((const void*) prefill_plan_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int) lds));
    const int groups = (n_entries + kPlanThreads - 1) / kPlanThreads;
    hipLaunchKernelGGL(prefill_plan_kernel, dim3(groups < kPlanMaxGroups ? groups : kPlanMaxGroups), dim3(kPlanThreads), lds, as_stream(stream),
                       ids, n_entries, expert_table, n_expert, *plan, maya_moe_prefill_max_tiles(n_entries, n_expert), with_masks, work);
    MAYA_LAUNCHED("prefill_plan_kernel");
    return MAYA_OK;
}

static int prefill_check(const char* what, const maya_moe_layout* l, const uint64_t* table, int n_expert, const maya_prefill_plan* plan,
                         int n_entries, int type_a, int type_b, int64_t k) {
    if (!l || !table || !plan_ok(plan)) return fail(MAYA_E_ARG, "%s: null pointer", what);
    if (type_a != type_b || (type_a != kQ4_K && type_a != kIQ2_S))
        return fail(MAYA_E_UNSUPPORTED, "%s: weight types %d / %d (Q4_K or IQ2_S, gate and up alike)", what, type_a, type_b);
    if (l->packing != MAYA_PACK_GGUF && l->packing != MAYA_PACK_STREAM) return fail(MAYA_E_UNSUPPORTED, "%s: packing %d", what, l->packing);
    if (type_a == kIQ2_S && l->packing != MAYA_PACK_STREAM)
        return fail(MAYA_E_UNSUPPORTED, "%s: IQ2_S rows are taken in the stream packing (maya_moe_repack)", what);
    if (l->n_embd <= 0 || l->n_ff <= 0 || l->n_embd % 256 || l->n_ff % 256)
        return fail(MAYA_E_SHAPE, "%s: n_embd %d / n_ff %d: multiples of 256 wanted", what, l->n_embd, l->n_ff);
    // (IQ2_S: the kernel's 16-byte copies into LDS want quads - 328 bytes a block - of a multiple of 16 bytes: an even number of blocks)
    if (type_a == kIQ2_S && k % 512) return fail(MAYA_E_SHAPE, "%s: IQ2_S rows of %lld values: a multiple of 512 wanted", what, (long long) k);
    if (type_a == kIQ2_S)
        if (const int rc = prefill_iq2s_lds_ok(what)) return rc;
    if ((l->gate_off | l->up_off | l->down_off) & 15) return fail(MAYA_E_ARG, "%s: matrix offsets not 16-byte aligned", what);
    // (an entry is a row of the second grid dimension in the quantizers' launches)
    if (n_entries <= 0 || n_entries > 65535 || n_expert <= 0) return fail(MAYA_E_SHAPE, "%s: entries %d (1..65535) experts %d", what, n_entries, n_expert);
    return MAYA_OK;
}

static int pf_gate_up(const maya_moe_layout* l, const uint64_t* expert_table, int n_expert, const maya_prefill_plan* plan, int n_entries,
                      maya_prefill_act xq, float limit, float* h, maya_prefill_act hq, const PfWork& work, void* stream) {
    DeviceState* st;
    if (const int rc = current_state(&st)) return rc;
    if (const int rc = prefill_check("prefill_gate_up", l, expert_table, n_expert, plan, n_entries, l ? l->gate_type : 0, l ? l->up_type : 0, l ? l->n_embd : 0)) return rc;
    if (!act_ok(xq) || !act_ok(hq) || !h) return fail(MAYA_E_ARG, "prefill_gate_up: null or misaligned activations");
    PfGemm a{};
    a.table = expert_table;
    a.plan = *plan;
    a.off[0] = l->gate_off;
    a.off[1] = l->up_off;
    a.k = l->n_embd;
    a.n = l->n_ff;
    a.row_bytes = (int64_t) (l->n_embd / 256) * 144;
    a.x = xq;
    a.out = h;
    a.limit = limit;
    a.work = work;
    const dim3 grid((unsigned) (l->n_ff / 64), pf_grid_rows(work, n_entries, n_expert));
    if (l->gate_type == kIQ2_S) {
        prefill_iq2s_launch<true>(a, st->cb, grid, as_stream(stream));
        MAYA_LAUNCHED("prefill_iq2s_kernel<gate_up>");
    } else {
        pf_launch<true>(a, grid, as_stream(stream));
        MAYA_LAUNCHED("prefill_q4k_kernel<gate_up>");
    }
    const dim3 qgrid((unsigned) ((l->n_ff + 8191) / 8192), (unsigned) n_entries);
    hipLaunchKernelGGL(prefill_quant_rows_kernel, qgrid, dim3(256), 0, as_stream(stream), (const float*) h, *plan, n_expert, (int64_t) l->n_ff, hq);
    MAYA_LAUNCHED("prefill_quant_rows_kernel");
    return MAYA_OK;
}

static int pf_down(const maya_moe_layout* l, const uint64_t* expert_table, int n_expert, const maya_prefill_plan* plan, int n_entries,
                   maya_prefill_act hq, float* part, const PfWork& work, void* stream) {
    DeviceState* st;
    if (const int rc = current_state(&st)) return rc;
    if (const int rc = prefill_check("prefill_down", l, expert_table, n_expert, plan, n_entries, l ? l->down_type : 0, l ? l->down_type : 0, l ? l->n_ff : 0)) return rc;
    if (!act_ok(hq) || !part) return fail(MAYA_E_ARG, "prefill_down: null or misaligned pointer");
    if (l->n_embd % 32) return fail(MAYA_E_SHAPE, "prefill_down: n_embd %d", l->n_embd);
    PfGemm a{};
    a.table = expert_table;
    a.plan = *plan;
    a.off[0] = l->down_off;
    a.k = l->n_ff;
    a.n = l->n_embd;
    a.row_bytes = (int64_t) (l->n_ff / 256) * 144;
    a.x = hq;
    a.out = part;
    a.work = work;
    const dim3 grid((unsigned) ((l->n_embd + 127) / 128), pf_grid_rows(work, n_entries, n_expert));
    if (l->down_type == kIQ2_S) {
        prefill_iq2s_launch<false>(a, st->cb, grid, as_stream(stream));
        MAYA_LAUNCHED("prefill_iq2s_kernel<down>");
    } else {
        pf_launch<false>(a, grid, as_stream(stream));
        MAYA_LAUNCHED("prefill_q4k_kernel<down>");
    }
    return MAYA_OK;
}

extern "C" {

int maya_moe_prefill_tile_rows(void) { return kPfRows; }
int maya_moe_prefill_max_tiles(int n_entries, int n_expert) {
    if (n_entries <= 0 || n_expert <= 0) return 0;
    return (n_entries + kPfRows - 1) / kPfRows + n_expert;
}
int maya_moe_prefill_supported(int type) { return type == kQ4_K || type == kIQ2_S ? 1 : 0; }

int maya_moe_prefill_plan(const int32_t* ids, int n_entries, const uint64_t* expert_table, int n_expert,
                          const maya_prefill_plan* plan, void* stream) {
    return pf_plan(ids, n_entries, expert_table, n_expert, plan, PfWork{}, stream);
}

int maya_moe_prefill_quant(const void* x, int x_dtype, int64_t x_stride, const maya_prefill_plan* plan, int n_entries,
                           int n_expert, int k, int64_t n_embd, maya_prefill_act xq, void* stream) {
    DeviceState* st;
    if (const int rc = current_state(&st)) return rc;
    if (x_dtype < 0 || x_dtype > 2) return fail(MAYA_E_UNSUPPORTED, "prefill_quant: dtype %d", x_dtype);
    if (!x || !plan_ok(plan) || !act_ok(xq)) return fail(MAYA_E_ARG, "prefill_quant: null or misaligned pointer");
    if (n_entries <= 0 || n_entries > 65535 || k <= 0 || n_embd <= 0 || n_embd % 256 || n_expert <= 0)
        return fail(MAYA_E_SHAPE, "prefill_quant: entries %d k %d n_embd %lld", n_entries, k, (long long) n_embd);
    if (x_stride == 0) x_stride = n_embd;
    if (n_entries % k) return fail(MAYA_E_SHAPE, "prefill_quant: %d entries are not whole tokens of %d", n_entries, k);
    const dim3 grid((unsigned) ((n_embd + 8191) / 8192), (unsigned) (n_entries / k));
    hipStream_t s = as_stream(stream);
    switch (x_dtype) {
        case MAYA_DT_F32: hipLaunchKernelGGL(prefill_quant_kernel<MAYA_DT_F32>, grid, dim3(256), 0, s, x, x_stride, *plan, k, n_embd, xq); break;
        case MAYA_DT_BF16: hipLaunchKernelGGL(prefill_quant_kernel<MAYA_DT_BF16>, grid, dim3(256), 0, s, x, x_stride, *plan, k, n_embd, xq); break;
        default: hipLaunchKernelGGL(prefill_quant_kernel<MAYA_DT_F16>, grid, dim3(256), 0, s, x, x_stride, *plan, k, n_embd, xq); break;
    }
    MAYA_LAUNCHED("prefill_quant_kernel");
    return MAYA_OK;
}

int maya_moe_prefill_gate_up(const maya_moe_layout* l, const uint64_t* expert_table, int n_expert, const maya_prefill_plan* plan,
                             int n_entries, maya_prefill_act xq, float limit, float* h, maya_prefill_act hq, void* stream) {
    return pf_gate_up(l, expert_table, n_expert, plan, n_entries, xq, limit, h, hq, pf_stage_work(n_entries, n_expert), stream);
}

int maya_moe_prefill_down(const maya_moe_layout* l, const uint64_t* expert_table, int n_expert, const maya_prefill_plan* plan,
                          int n_entries, maya_prefill_act hq, float* part, void* stream) {
    return pf_down(l, expert_table, n_expert, plan, n_entries, hq, part, pf_stage_work(n_entries, n_expert), stream);
}

int maya_moe_prefill_combine(const maya_prefill_plan* plan, const float* weights, const float* part, int n_tokens, int k,
                             int64_t n_embd, const float* add, void* out, int out_dtype, void* stream) {
    DeviceState* st;
    if (const int rc = current_state(&st)) return rc;
    if (!plan_ok(plan) || !weights || !part || !out) return fail(MAYA_E_ARG, "prefill_combine: null pointer");
    if (out_dtype < 0 || out_dtype > 2) return fail(MAYA_E_UNSUPPORTED, "prefill_combine: dtype %d", out_dtype);
    if (n_tokens <= 0 || n_tokens > 65535 || k <= 0 || n_embd <= 0) return fail(MAYA_E_SHAPE, "prefill_combine: tokens %d k %d", n_tokens, k);
    hipStream_t s = as_stream(stream);
    if (n_embd % 4 == 0 && k <= MAYA_MAX_K && (((uintptr_t) part | (uintptr_t) add | (uintptr_t) out) & 15) == 0) {
        const dim3 grid4((unsigned) ((n_embd / 4 + 255) / 256), (unsigned) n_tokens);
        switch (out_dtype) {
            case MAYA_DT_F32: hipLaunchKernelGGL(prefill_combine4_kernel<MAYA_DT_F32>, grid4, dim3(256), 0, s, plan->entry_row, weights, part, k, n_embd, add, out); break;
            case MAYA_DT_BF16: hipLaunchKernelGGL(prefill_combine4_kernel<MAYA_DT_BF16>, grid4, dim3(256), 0, s, plan->entry_row, weights, part, k, n_embd, add, out); break;
            default: hipLaunchKernelGGL(prefill_combine4_kernel<MAYA_DT_F16>, grid4, dim3(256), 0, s, plan->entry_row, weights, part, k, n_embd, add, out); break;
        }
        MAYA_LAUNCHED("prefill_combine4_kernel");
        return MAYA_OK;
    }
    const dim3 grid((unsigned) ((n_embd + 255) / 256), (unsigned) n_tokens);
    switch (out_dtype) {
        case MAYA_DT_F32: hipLaunchKernelGGL(prefill_combine_kernel<MAYA_DT_F32>, grid, dim3(256), 0, s, plan->entry_row, weights, part, k, n_embd, add, out); break;
        case MAYA_DT_BF16: hipLaunchKernelGGL(prefill_combine_kernel<MAYA_DT_BF16>, grid, dim3(256), 0, s, plan->entry_row, weights, part, k, n_embd, add, out); break;
        default: hipLaunchKernelGGL(prefill_combine_kernel<MAYA_DT_F16>, grid, dim3(256), 0, s, plan->entry_row, weights, part, k, n_embd, add, out); break;
    }
    MAYA_LAUNCHED("prefill_combine_kernel");
    return MAYA_OK;
}

struct PrefillWs {
    maya_prefill_plan plan;
    PfWork work;
    maya_prefill_act x, h;
    float *hf, *part;
    size_t bytes;
};
static PrefillWs prefill_carve(const maya_moe_layout& l, int n_tokens, int k, int n_expert, uint8_t* base) {
    PrefillWs w{};
    size_t off = 0;
    const size_t ne = (size_t) n_tokens * k;
    auto take = [&](size_t n) {
        uint8_t* p = base ? base + off : nullptr;
        off += (n + 255) & ~(size_t) 255;
        return p;
    };
    const size_t mt = (size_t) maya_moe_prefill_max_tiles((int) ne, n_expert);
    w.plan.bounds = (int32_t*) take(4 * ((size_t) n_expert + 1));
    w.plan.row_entry = (int32_t*) take(4 * ne);
    w.plan.entry_row = (int32_t*) take(4 * ne);
    w.plan.tile_expert = (int32_t*) take(4 * mt);
    w.plan.tile_row0 = (int32_t*) take(4 * mt);
    w.plan.n_tiles = (int32_t*) take(4);
    // Items of 128 rows, a workgroup's most; of 64 where the IQ2_S kernel of few rows takes them.
    w.work.few = prefill_iq2s_few(n_tokens, (int) ne, n_expert);
    w.work.rows = l.gate_type == kIQ2_S && w.work.few ? kPfRows : 2 * kPfRows;
    w.work.list = (PfItem*) take(sizeof(PfItem) * mt);   // (fewer than the tiles)
    w.work.n = (int32_t*) take(4);
    auto take_act = [&](maya_prefill_act& a, size_t k) {
        a.q = (int8_t*) take(ne * k);
        a.d = (float*) take(ne * (k / 256) * 4);
        a.s = (uint16_t*) take(ne * (k / 32) * 4);
    };
    take_act(w.x, (size_t) l.n_embd);
    take_act(w.h, (size_t) l.n_ff);
    w.hf = (float*) take(ne * l.n_ff * 4);
    w.part = (float*) take(ne * l.n_embd * 4);
    w.bytes = off;
    return w;
}
size_t maya_moe_prefill_workspace_bytes(const maya_moe_layout* l, int n_tokens, int k, int n_expert) {
    if (!l || n_tokens <= 0 || k <= 0 || n_expert <= 0 || l->n_embd <= 0 || l->n_ff <= 0) return 0;
    return prefill_carve(*l, n_tokens, k, n_expert, nullptr).bytes;
}

int maya_moe_prefill_layer(const maya_moe_layout* l, const uint64_t* expert_table, int n_expert, int k, const float* logits,
                           const void* x, int x_dtype, int n_tokens, float limit, const float* add, int32_t* ids,
                           float* weights, void* out, int out_dtype, void* workspace, size_t workspace_bytes, void* stream) {
    if (!l || !expert_table || !x || !ids || !weights || !out || !workspace) return fail(MAYA_E_ARG, "prefill_layer: null pointer");
    if (n_tokens <= 0 || n_tokens > 8192 || k <= 0 || k > MAYA_MAX_K || (int64_t) n_tokens * k > 65535)
        return fail(MAYA_E_SHAPE, "prefill_layer: tokens %d k %d (at most 65535 entries a call)", n_tokens, k);
    if (((uintptr_t) workspace & 255) != 0) return fail(MAYA_E_ARG, "prefill_layer: workspace not 256-byte aligned");
    // everything a stage would refuse is refused here, before the first launch ("> 0: not covered, nothing launched")
    {
        DeviceState* st;
        if (const int rc0 = current_state(&st)) return rc0;
        if (n_expert <= 0 || n_expert > MAYA_MAX_EXPERTS || k > n_expert)
            return fail(MAYA_E_SHAPE, "prefill_layer: experts %d (1..%d) k %d", n_expert, MAYA_MAX_EXPERTS, k);
        if (x_dtype < 0 || x_dtype > 2 || out_dtype < 0 || out_dtype > 2) return fail(MAYA_E_UNSUPPORTED, "prefill_layer: dtypes %d / %d", x_dtype, out_dtype);
        maya_prefill_plan probe{};   // (the plan's pointers come from the workspace: only the layout's side is checked here)
        int32_t dummy = 0;
        probe.bounds = probe.row_entry = probe.entry_row = probe.tile_expert = probe.tile_row0 = probe.n_tiles = &dummy;
        if (const int rc0 = prefill_check("prefill_layer", l, expert_table, n_expert, &probe, n_tokens * k, l->gate_type, l->up_type, l->n_embd)) return rc0;
        if (const int rc0 = prefill_check("prefill_layer", l, expert_table, n_expert, &probe, n_tokens * k, l->down_type, l->down_type, l->n_ff)) return rc0;
        if (l->n_embd % 32) return fail(MAYA_E_SHAPE, "prefill_layer: n_embd %d", l->n_embd);
    }
    const PrefillWs w = prefill_carve(*l, n_tokens, k, n_expert, (uint8_t*) workspace);
    if (workspace_bytes < w.bytes) return fail(MAYA_E_ARG, "prefill_layer: workspace %zu < %zu bytes", workspace_bytes, w.bytes);
    const int ne = n_tokens * k;
    int rc;
    if (logits && (rc = maya_moe_route_topk(logits, n_tokens, n_expert, k, ids, weights, stream))) return rc;   // (null: ids / weights are given)
    if ((rc = pf_plan(ids, ne, expert_table, n_expert, &w.plan, w.work, stream))) return rc;
    if ((rc = maya_moe_prefill_quant(x, x_dtype, 0, &w.plan, ne, n_expert, k, l->n_embd, w.x, stream))) return rc;
    if ((rc = pf_gate_up(l, expert_table, n_expert, &w.plan, ne, w.x, limit, w.hf, w.h, w.work, stream))) return rc;
    if ((rc = pf_down(l, expert_table, n_expert, &w.plan, ne, w.h, w.part, w.work, stream))) return rc;
    return maya_moe_prefill_combine(&w.plan, weights, w.part, n_tokens, k, l->n_embd, add, out, out_dtype, stream);
}

}  // extern "C"
