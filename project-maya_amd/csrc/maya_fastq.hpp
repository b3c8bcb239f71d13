// maya_fastq.hpp - position-mapped kernels for Q8_0 rows in the stream packing (a row = its k codes, then its k / 32 FP16
// scales: aligned 16-byte loads; the GGUF order interleaves a 2-byte scale with every 32 codes).  Made for the expert
// every token takes (a shared expert, a dense FFN): the tokens of a group share one read of the weights.  A lane owns
// one 32-value block position; the batch of a step is 8 (row, token) values - 8 / NT rows of NT tokens - so one
// transposing butterfly reduces a step whatever NT is.
#pragma once

namespace maya {

// the group's entries c0 .. c0 + NT - 1 (-1 past its end) and their tokens' codes / scales at block position u
template <int NT>
__device__ __forceinline__ void q80_chunk(const maya_moe_args& a, const GroupRef& gr, int c0, const maya_act& x, bool by_token,
                                          int k, int u, int (&ents)[NT], int (&y)[NT][8], float (&dx)[NT]) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        ents[t] = c0 + t < gr.ne ? entry_of(a, gr, c0 + t) : -1;
        if (ents[t] >= 0) {
            const int row = by_token ? ents[t] / a.k : ents[t];
            const int4* q = (const int4*) (x.q + (size_t) row * k);
            const int4 ya = q[2 * u], yb = q[2 * u + 1];
            y[t][0] = ya.x, y[t][1] = ya.y, y[t][2] = ya.z, y[t][3] = ya.w;
            y[t][4] = yb.x, y[t][5] = yb.y, y[t][6] = yb.z, y[t][7] = yb.w;
            dx[t] = x.d[(size_t) row * (k >> 5) + u];
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) y[t][i] = 0;
            dx[t] = 0.0f;
        }
    }
}
// one row's block at this position against NT tokens: acc[base + t] = d_w d_x[t] * (codes . y[t])
template <int NT>
__device__ __forceinline__ void q80_values(const u32x4 qa, const u32x4 qb, uint32_t dbits, const int (&y)[NT][8],
                                           const float (&dx)[NT], float (&acc)[8], int base) {
    const float dw = f16_bits_to_f32((uint16_t) dbits);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        int s = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s = dot4((int) qa[i], y[t][i], s);
            s = dot4((int) qb[i], y[t][4 + i], s);
        }
        acc[base + t] = __fmul_rn(__fmul_rn(dw, dx[t]), (float) s);
    }
}

// a row's block at one position
struct Q80Row {
    u32x4 a, b;
    uint32_t d;
};
__device__ __forceinline__ Q80Row q80_load(const __amdgpu_buffer_rsrc_t rs, uint32_t oq, uint32_t od, uint32_t ro) {
    return Q80Row{__builtin_amdgcn_raw_buffer_load_b128(rs, oq, ro, 0), __builtin_amdgcn_raw_buffer_load_b128(rs, oq + 16u, ro, 0),
                  (uint32_t) __builtin_amdgcn_raw_buffer_load_b16(rs, od, ro, 0)};
}

// ---- gate/up: a workgroup of NW waves = 2 * 32 NW lanes for the block positions of a (gate row, up row) pair (lanes past the
// row's last position idle, as in the IQ2_S kernels); grid (n_ff / ROWS, groups).  A step takes 8 / NT row pairs for NT tokens.
// Bound by the latency of a workgroup's loads (of one expert there is one workgroup a CU): the next step's rows are on their way
// while one is multiplied, and the sums of all steps wait in LDS for one closing by ROWS * NT lanes - no barrier between steps.
// 7168 x 2048, one expert: 4 tokens 14.5 -> 9.7 us, 8 tokens 17.8 -> 13.4 (31 MB); a layer of 64 experts, 8 tokens, 398 -> 338.
// SELF: the call has one token, and the workgroup rounds its activations itself, a block a lane, from `xf` (no a.x, and no launch
// to fill it): for one expert only - 8 experts' workgroups all rounding the token took 88.7 us a layer instead of 78.5.
template <int NW, int NT, int ROWS, bool FIT, bool SELF>
__global__ __launch_bounds__(64 * NW) void gate_up_q80_pos_kernel(maya_moe_args a, const void* __restrict__ xf, int x_dtype) {
    constexpr int NU = 32 * NW, R = 8 / NT;
    static_assert(ROWS % R == 0, "whole steps");
    static_assert(!SELF || NT == 1, "one token");
    __shared__ float part[ROWS / R][2 * NW][8];
    GroupRef gr;
    if (!group_of<false>(a, blockIdx.y, gr)) return;
    const int t = threadIdx.x, lane = t & 63, hw = t >> 5;
    const bool is_up = t >= NU;
    const int nu = FIT ? NU : a.layout.n_embd >> 5, lu = is_up ? t - NU : t;   // blocks a row; the lane's position among 32 NW
    const bool on = FIT || lu < nu;
    const int u = on ? lu : nu - 1;
    const int k = 32 * nu, n_ff = a.layout.n_ff, r0 = blockIdx.x * ROWS;
    const uint32_t rb = (uint32_t) nu * 34u;   // bytes of a row
    const uint32_t gu_bytes = (uint32_t) (a.layout.down_off - a.layout.gate_off);
    const __amdgpu_buffer_rsrc_t rs = weight_rsrc(gr.blob + a.layout.gate_off, gu_bytes);
    const uint32_t mat = is_up ? (uint32_t) (a.layout.up_off - a.layout.gate_off) : 0u;
    const uint32_t oq = mat + 32u * u, od = on ? mat + 32u * nu + 2u * u : gu_bytes;   // (an idle lane's scale: as in quad_offs)
    for (int c0 = 0; c0 < gr.ne; c0 += NT) {
        Q80Row w[2][R];
#pragma unroll
        for (int rr = 0; rr < R; ++rr) w[0][rr] = q80_load(rs, oq, od, (uint32_t) (r0 + rr) * rb);
        int ents[NT], y[NT][8];
        float dx[NT];
        if constexpr (SELF) {
            ents[0] = entry_of(a, gr, c0);
            const int64_t v0 = (int64_t) (ents[0] / a.k) * k + 32 * u;
            float v[32];
            if (x_dtype == MAYA_DT_BF16) act_load32<MAYA_DT_BF16>(xf, v0, true, v);
            else if (x_dtype == MAYA_DT_F16) act_load32<MAYA_DT_F16>(xf, v0, true, v);
            else act_load32<MAYA_DT_F32>(xf, v0, true, v);
            q80_round_lane32(v, y[0], dx[0]);
        } else {
            q80_chunk<NT>(a, gr, c0, a.x, true, k, u, ents, y, dx);
        }
#pragma unroll
        for (int i = 0; i < NT; ++i) idle_lane_zero(on, y[i], dx[i]);
        if (c0) __syncthreads();   // (the chunk before is read)
#pragma unroll
        for (int r = 0; r < ROWS; r += R) {
            const int cur = (r / R) & 1;
            if (r + R < ROWS) {
#pragma unroll
                for (int rr = 0; rr < R; ++rr) w[cur ^ 1][rr] = q80_load(rs, oq, od, (uint32_t) (r0 + r + R + rr) * rb);
            }
            float acc[8];
#pragma unroll
            for (int rr = 0; rr < R; ++rr) q80_values<NT>(w[cur][rr].a, w[cur][rr].b, w[cur][rr].d, y, dx, acc, rr * NT);
            const float v = reduce8_half(acc, lane);
            if ((lane & 3) == 0) part[r / R][hw][(lane >> 2) & 7] = v;
        }
        __syncthreads();
        if (t < ROWS * NT) {   // the closing of every step at once: 8 values a step
            const int st = t >> 3, i = t & 7, row = r0 + st * R + i / NT;
            const int ent = c0 + i % NT < gr.ne ? entry_of(a, gr, c0 + i % NT) : -1;
            float g = part[st][0][i], up = part[st][NW][i];
#pragma unroll
            for (int w2 = 1; w2 < NW; ++w2) {
                g += part[st][w2][i];
                up += part[st][NW + w2][i];
            }
            if (ent >= 0 && row < n_ff) a.h[(size_t) ent * n_ff + row] = swiglu(g, up, a.limit);
        }
    }
}

// out[t][c] of a call with one slot a token: combine_kernel's arithmetic
__device__ __forceinline__ float combine_one(const maya_moe_args& a, float p, float add, float add2) {
    if (a.add && (!a.add_flag || *a.add_flag)) p = __fadd_rn(p, add);
    return a.add2 ? __fadd_rn(p, add2) : p;
}
// ---- down, n_ff = 32 nu <= 2048 (nu block positions a row on the first nu lanes of one wave, the lanes past them idle):
// every wave takes its own rows (wg_rows / 8 of them), a step 8 / NT rows for NT entries of the group, the next step's rows on
// their way; grid (n_embd / wg_rows, groups).  Writes part[entry][row] - or, of a call with one slot a token, the weighted row
// with the residuals on it into out[token][row] (combine_kernel's arithmetic, no launch for it).
// hq.q NULL: the workgroup rounds h itself, a wave an entry, a block a lane, into LDS, in quant_q80_kernel's rounding - the launch
// for it and the combining one took 8.5 us of a shared expert's 35 (7168 x 2048, 8 tokens) beside the 8 of this one, which is 11.8 with both.
template <int NT, int NU>
__global__ __launch_bounds__(512) void down_q80_pos_kernel(maya_moe_args a, int wg_rows) {
    constexpr int R = 8 / NT;
    constexpr bool AHEAD = NT >= 4;   // (of fewer entries a step has enough rows in flight)
    __shared__ int4 s_y[NT][2][64];
    __shared__ float s_d[NT][64];
    const int n_embd = a.layout.n_embd;
    const bool one = a.k == 1;
    if (one) {
        if (a.skip && *a.skip) return;
        if (a.plan_ptr[blockIdx.y] == 0ull) {   // (a slot left out: the residuals alone)
            const size_t row = (size_t) blockIdx.y * n_embd;
            for (int c = blockIdx.x * wg_rows + (int) threadIdx.x; c < min(n_embd, (int) (blockIdx.x + 1) * wg_rows); c += 512)
                a.out[row + c] = combine_one(a, 0.0f, a.add ? a.add[row + c] : 0.0f, a.add2 ? a.add2[row + c] : 0.0f);
        }
    }
    GroupRef gr;
    if (!group_of<false>(a, blockIdx.y, gr)) return;
    const int wave = threadIdx.x >> 6, lane0 = threadIdx.x & 63;
    // (an idle lane reads the last position's codes again and meets them with zero activations; its scale reads as zero)
    const int nu = NU ? NU : a.layout.n_ff >> 5;
    const bool on = NU == 64 || lane0 < nu;
    const int lane = on ? lane0 : nu - 1;
    const int k = 32 * nu;
    // (the wave's row offset is uniform, but only readfirstlane tells the compiler so)
    const int per_wave = wg_rows >> 3, r0 = __builtin_amdgcn_readfirstlane(blockIdx.x * wg_rows + wave * per_wave);
    const uint32_t rb = (uint32_t) nu * 34u;
    const uint64_t mat = gr.blob + a.layout.down_off;
    const __amdgpu_buffer_rsrc_t rs = weight_rsrc(mat, (uint32_t) n_embd * rb);
    const uint32_t oq = 32u * lane, od = on ? 32u * nu + 2u * lane : (uint32_t) n_embd * rb;
    const int li = (lane0 >> 2) & 7, lr = li / NT, tk = li % NT;   // the value of a step that the lane ends up with
    for (int c0 = 0; c0 < gr.ne; c0 += NT) {
        Q80Row w[R];
        if constexpr (AHEAD) {
#pragma unroll
            for (int rr = 0; rr < R; ++rr) w[rr] = q80_load(rs, oq, od, (uint32_t) (r0 + rr) * rb);
        }
        int ents[NT], y[NT][8];
        float dx[NT];
        if (a.hq.q) {
            q80_chunk<NT>(a, gr, c0, a.hq, false, k, lane, ents, y, dx);
        } else {
#pragma unroll
            for (int t = 0; t < NT; ++t) ents[t] = c0 + t < gr.ne ? entry_of(a, gr, c0 + t) : -1;
            if (c0) __syncthreads();   // (the entries before are read)
            if (wave < NT) {
                int q[8] = {0, 0, 0, 0, 0, 0, 0, 0};
                float d = 0.0f;
                if (c0 + wave < gr.ne) {
                    float v[32];
                    act_load32<MAYA_DT_F32>(a.h, (int64_t) entry_of(a, gr, c0 + wave) * k + 32 * lane, true, v);
                    q80_round_lane32(v, q, d);
                }
                s_y[wave][0][lane0] = make_int4(q[0], q[1], q[2], q[3]);
                s_y[wave][1][lane0] = make_int4(q[4], q[5], q[6], q[7]);
                s_d[wave][lane0] = d;
            }
            __syncthreads();
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int4 ya = s_y[t][0][lane0], yb = s_y[t][1][lane0];
                y[t][0] = ya.x, y[t][1] = ya.y, y[t][2] = ya.z, y[t][3] = ya.w;
                y[t][4] = yb.x, y[t][5] = yb.y, y[t][6] = yb.z, y[t][7] = yb.w;
                dx[t] = s_d[t][lane0];
            }
        }
#pragma unroll
        for (int i = 0; i < NT; ++i) idle_lane_zero(on, y[i], dx[i]);
        const int ent = c0 + tk < gr.ne ? entry_of(a, gr, c0 + tk) : -1;
        const bool mine = (lane0 & 35) == 0 && ent >= 0;
        const float pw = one && mine ? a.plan_w[ent] : 0.0f;
        for (int r = 0; r < per_wave; r += R) {
            Q80Row nx[R];
            if (!AHEAD) {
#pragma unroll
                for (int rr = 0; rr < R; ++rr) w[rr] = q80_load(rs, oq, od, (uint32_t) (r0 + r + rr) * rb);
            } else if (r + R < per_wave) {
#pragma unroll
                for (int rr = 0; rr < R; ++rr) nx[rr] = q80_load(rs, oq, od, (uint32_t) (r0 + r + R + rr) * rb);
            }
            const bool put = mine && r0 + r + lr < n_embd;
            const size_t at = (size_t) (put ? ent : 0) * n_embd + r0 + r + lr;
            const float add = one && put && a.add ? a.add[at] : 0.0f, add2 = one && put && a.add2 ? a.add2[at] : 0.0f;
            float acc[8];
#pragma unroll
            for (int rr = 0; rr < R; ++rr) q80_values<NT>(w[rr].a, w[rr].b, w[rr].d, y, dx, acc, rr * NT);
            float v = reduce8_half(acc, lane0);
            v = add_other_half(v);
            if (put) {
                if (a.part) a.part[at] = v;
                if (one) a.out[at] = combine_one(a, __fmul_rn(v, pw), add, add2);
            }
            if constexpr (AHEAD) {
#pragma unroll
                for (int rr = 0; rr < R; ++rr) w[rr] = nx[rr];
            }
        }
    }
}

}  // namespace maya
