// maya_fastk.hpp - position-mapped decode kernels for Q4_K rows in their own GGUF order (blobs 16-byte aligned): the same
// skeleton as the IQ2_S ones.  A lane owns one 16-byte piece of every block's codes - the low nibbles are 16 values of
// sub-block 2j, the high nibbles 16 values of sub-block 2j + 1 - so its 32 activation codes, their two sums and the
// block's activation scale stay in registers while it walks down the rows; 8 lanes read a block's 128 code bytes as one
// contiguous run and all 8 the block's 16-byte header.  The format is cheap to decode (about 45 vector operations for 18
// bytes), so these kernels are bound by the weight stream.
#pragma once

namespace maya {

// the lane's fixed part: activation codes (low-nibble values, then high-nibble values), their sums, the scale
struct PosQ4K {
    int ylo[4], yhi[4];
    int slo, shi;
    float dx;
    uint32_t o_hdr, o_q;   // byte offsets of the block header and of the lane's piece inside a row
    int sh;                // bit offset of the lane's two sub-blocks' scale bytes in their packed word
    int wsel;              // which packed word (sub-blocks 0-3 or 4-7)
};
// position u of a row: block u >> 3, piece u & 7 (sub-block pair j = piece >> 1, half = piece & 1); an idle lane (`on` false)
// asks behind the resource's `past` bytes, as in quad_offs
__device__ __forceinline__ void pos_q4k_init(PosQ4K& p, int u, uint32_t mat_off, bool on = true, uint32_t past = 0u) {
    const int b = u >> 3, piece = u & 7, j = piece >> 1;
    p.o_hdr = on ? mat_off + 144u * b : past;
    p.o_q = on ? mat_off + 144u * b + 16u + 16u * piece : past;
    p.wsel = j >> 1;
    p.sh = 16 * (j & 1);
}
__device__ __forceinline__ void pos_q4k_codes(PosQ4K& p, int u, const int8_t* q, const float* d, const int16_t* bsums) {
    const int b = u >> 3, piece = u & 7, j = piece >> 1, half = piece & 1;
    const int v0 = 256 * b + 64 * j + 16 * half;
    const int4 lo = *(const int4*) (q + v0), hi = *(const int4*) (q + v0 + 32);
    p.ylo[0] = lo.x, p.ylo[1] = lo.y, p.ylo[2] = lo.z, p.ylo[3] = lo.w;
    p.yhi[0] = hi.x, p.yhi[1] = hi.y, p.yhi[2] = hi.z, p.yhi[3] = hi.w;
    p.dx = d[v0 >> 5];
    if (bsums) {
        p.slo = bsums[v0 >> 4];
        p.shi = bsums[(v0 + 32) >> 4];
    } else {
        p.slo = dot4(0x01010101, p.ylo[0], dot4(0x01010101, p.ylo[1], dot4(0x01010101, p.ylo[2], dot4(0x01010101, p.ylo[3], 0))));
        p.shi = dot4(0x01010101, p.yhi[0], dot4(0x01010101, p.yhi[1], dot4(0x01010101, p.yhi[2], dot4(0x01010101, p.yhi[3], 0))));
    }
}
// a lane past the row's last position: no codes, no scale
__device__ __forceinline__ void pos_q4k_idle(PosQ4K& p, bool on) {
#pragma unroll
    for (int i = 0; i < 4; ++i) p.ylo[i] = on ? p.ylo[i] : 0, p.yhi[i] = on ? p.yhi[i] : 0;
    p.slo = on ? p.slo : 0, p.shi = on ? p.shi : 0;
    p.dx = on ? p.dx : 0.0f;
}
// one row's value at this position: dx (d (sc0 t0 + sc1 t1) - dmin (m0 s0 + m1 s1))
__device__ __forceinline__ float pos_q4k_value(const PosQ4K& p, const u32x4 hdr, const u32x4 q) {
    // the 6-bit scales / minimums of the lane's two sub-blocks (get_scale_min_k4: include/strata/artifact/dequant.hpp:162-172)
    const uint32_t s0 = hdr.y, s1 = hdr.z, s2 = hdr.w;
    const uint32_t scw = p.wsel ? ((s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u)) : (s0 & 0x3f3f3f3fu);
    const uint32_t mnw = p.wsel ? (((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u)) : (s1 & 0x3f3f3f3fu);
    const uint32_t sc2 = scw >> p.sh, mn2 = mnw >> p.sh;
    int t0 = 0, t1 = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        t0 = dot4((int) (q[i] & 0x0f0f0f0fu), p.ylo[i], t0);
        t1 = dot4((int) ((q[i] >> 4) & 0x0f0f0f0fu), p.yhi[i], t1);
    }
    const int is = __mul24((int) (sc2 & 0xffu), t0) + __mul24((int) ((sc2 >> 8) & 0xffu), t1);
    const int ms = __mul24((int) (mn2 & 0xffu), p.slo) + __mul24((int) ((mn2 >> 8) & 0xffu), p.shi);
    const float d = f16_bits_to_f32((uint16_t) (hdr.x & 0xffffu)), dmin = f16_bits_to_f32((uint16_t) (hdr.x >> 16));
    return __fmul_rn(p.dx, __fsub_rn(__fmul_rn(d, (float) is), __fmul_rn(dmin, (float) ms)));
}

// ---- gate/up: a workgroup of NW waves = 2 * 32 NW lanes for the positions of a (gate row, up row) pair (lanes past the row's
// last position idle, as in the IQ2_S kernels); grid (n_ff / ROWS, entries); entry e = token e / k, slot e % k.  Rows in batches of 8, one row ahead in registers.
// AHEAD (8 rows): all of a lane's rows are requested up front - the launches of a few entries, whose workgroups do not fill
// the chip and would otherwise run at the memory's latency a row.
// HEAD (4 or 8: a token's experts a lane): the layer's head rides in this launch (head_in_gate_up) - grid (n_ff / ROWS + 1, k), of
// several tokens (MANY) (n_ff / ROWS, tokens k + 1), with the tokens in bits 8 to 15 of n_ent and 2^16 / tokens, rounded up, above.
// The leading arguments (MAYA_HEAD_ARGS) are what it asks of memory first, in scalar registers with the dispatch.
template <int NW, int ROWS, int MINW, bool FIT, bool AHEAD = false, int HEAD = 0, bool MANY = false>
__global__ __launch_bounds__(64 * NW, MINW) void gate_up_q4k_pos_kernel(MAYA_HEAD_PARAMS, maya_moe_args a, LayerHead out) {
    static_assert(ROWS % 8 == 0, "rows come in batches of 8");
    static_assert(!AHEAD || ROWS == 8, "every row up front: one batch");
    constexpr int NU = 32 * NW;
    __shared__ float part[2][2 * NW][8];
    const int t = threadIdx.x, lane = t & 63, hw = t >> 5;
    const bool is_up = t >= NU;
    const int nu = FIT ? NU : mode >> 16, lu = is_up ? t - NU : t;   // positions a row; the lane's among 32 NW
    const bool on = FIT || lu < nu;
    const int u = on ? lu : nu - 1;
    PosQ4K p;
    const uint32_t gu_bytes = (uint32_t) (a.layout.down_off - a.layout.gate_off);
    pos_q4k_init(p, u, is_up ? (uint32_t) (a.layout.up_off - a.layout.gate_off) : 0u, on, gu_bytes);
    int e;
    uint64_t blob;
    if constexpr (HEAD) {
        // position u holds the block's values v0 .. v0 + 15 (against the low nibbles) and v0 + 32 .. v0 + 47 (the high ones)
        const int v0 = 256 * (u >> 3) + 64 * ((u & 7) >> 1) + 16 * (u & 1);
        int y[8];
        float d;
        int slot, tok = 0, rank = 0;
        if constexpr (MANY) {
            const int n_tok = (n_ent >> 8) & 0xff, i = (int) blockIdx.y - 1;
            rank = (int) ((uint32_t) max(i, 0) * ((uint32_t) n_ent >> 16) >> 16);   // (i / n_tok: i < 256, 2 <= n_tok <= 16)
            tok = i - rank * n_tok;
            if (i < 0) {
                if ((int) blockIdx.x >= n_tok) return;
                tok = blockIdx.x, rank = -1;
            }
            n_ent &= 0xff;
        }
        const LayerHeadIn hd = {logits, table, x, bias, n_expert, mode & 255, (mode >> 8) & 1, out, mode >> 16 << 5};
        if (!head_in_gate_up<NW, HEAD, MANY ? kExpertOrder : kOneToken>(hd, n_ent, skip, is_up, on, lu, v0, v0 + 32, y, d, blob, slot, tok, rank)) return;
        e = MANY ? tok * n_ent + slot : slot;
#pragma unroll
        for (int i = 0; i < 4; ++i) p.ylo[i] = y[i], p.yhi[i] = y[4 + i];
        p.dx = d;
        p.slo = dot4(0x01010101, p.ylo[0], dot4(0x01010101, p.ylo[1], dot4(0x01010101, p.ylo[2], dot4(0x01010101, p.ylo[3], 0))));
        p.shi = dot4(0x01010101, p.yhi[0], dot4(0x01010101, p.yhi[1], dot4(0x01010101, p.yhi[2], dot4(0x01010101, p.yhi[3], 0))));
    } else {
        if (skip && *skip) return;
        // (a window's entries in the order of grp_ent where one is given: the entries of an expert side by side; -1 ends it)
        e = (a.grp_ent && !a.grp_ptr) ? a.grp_ent[blockIdx.y] : (int) blockIdx.y;
        if (e < 0) return;
        blob = a.plan_ptr[e];
        if (blob == 0ull) return;
        const int tok = e / a.k;
        pos_q4k_codes(p, u, a.x.q + (size_t) tok * (32 * nu), a.x.d + (size_t) tok * nu, a.x.bsums + (size_t) tok * (2 * nu));
        pos_q4k_idle(p, on);
    }
    const uint32_t rb = (uint32_t) nu * 18u;   // bytes of a row: 144 a block
    const int n_ff = a.layout.n_ff, r0 = blockIdx.x * ROWS;
    const __amdgpu_buffer_rsrc_t rs = weight_rsrc(blob + a.layout.gate_off, gu_bytes);
    u32x4 hn = __builtin_amdgcn_raw_buffer_load_b128(rs, p.o_hdr, (uint32_t) r0 * rb, 0);
    u32x4 qn = __builtin_amdgcn_raw_buffer_load_b128(rs, p.o_q, (uint32_t) r0 * rb, 0);
    u32x4 ha[AHEAD ? ROWS : 1], qa[AHEAD ? ROWS : 1];
    if constexpr (AHEAD) {
        ha[0] = hn, qa[0] = qn;
#pragma unroll
        for (int i = 1; i < ROWS; ++i) {
            ha[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, p.o_hdr, (uint32_t) (r0 + i) * rb, 0);
            qa[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, p.o_q, (uint32_t) (r0 + i) * rb, 0);
        }
    }
    float acc[8];
#pragma unroll 1
    for (int r = 0; r < ROWS; r += 8) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if constexpr (AHEAD) {
                acc[i] = pos_q4k_value(p, ha[i], qa[i]);
            } else {
                const u32x4 hc = hn, qc = qn;
                if (r + i + 1 < ROWS) {
                    hn = __builtin_amdgcn_raw_buffer_load_b128(rs, p.o_hdr, (uint32_t) (r0 + r + i + 1) * rb, 0);
                    qn = __builtin_amdgcn_raw_buffer_load_b128(rs, p.o_q, (uint32_t) (r0 + r + i + 1) * rb, 0);
                }
                acc[i] = pos_q4k_value(p, hc, qc);
            }
            asm volatile("" : "+v"(acc[i]));
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

// ---- down + combine, n_ff = 32 nu <= 2048 (nu positions a row, lanes past them idle): wave w = slot w of token blockIdx.y, of at
// most SLOTS, rows in batches of 8; grid (n_embd / ROWS, tokens).  Without a rounded h (hq.q == NULL) a wave rounds its slot's h
// to Q8_K itself.
// PAIR (nu <= 32): a wave takes two rows at a time, one on either half of its lanes - rows r .. r + 3 of a batch below, r + 4 ..
// r + 7 above - instead of leaving half of them without a position.
// AHEAD: all ROWS rows of the wave are requested before anything else is done (one or two slots on one token: a few
// hundred waves on the whole chip, each with one row in flight, run at the memory's latency a row).
// The leading arguments repeat fields of `a`: they arrive in scalar registers with the dispatch (down_iq2s_pos_kernel).  What
// the kernel asks of memory first - the plan, the combine's weights, h - goes out side by side; it used to wait for the plan
// before h, and the combine read plan and weights slot by slot at the end.
// Measured: 2048 x 768 top-8, one token, 8.1 -> 5.2 us a launch (sixteen layers in a graph 249 -> 196 us); 7168 x 2048 top-1 5.5 -> 5.0.
template <int ROWS, int MINW, int SLOTS, int NU, bool AHEAD = false, bool PAIR = false>
__global__ __launch_bounds__(64 * SLOTS, MINW) void down_q4k_pos_kernel(const uint64_t* __restrict__ plan_ptr, const float* __restrict__ plan_w,
                                                                  const float* __restrict__ h, const int32_t* __restrict__ skip,
                                                                  const int8_t* __restrict__ hq_q, int k, int n_embd, int n_pos, maya_moe_args a) {
    static_assert(ROWS % 8 == 0, "rows come in batches of 8");
    static_assert(!AHEAD || ROWS == 8, "every row up front: one batch");
    static_assert(!PAIR || NU == 0, "two rows a wave: at most 32 positions");
    constexpr int NB = PAIR ? 4 : 8;   // row steps of a batch
    __shared__ float part[SLOTS][ROWS];
    __shared__ float s_w[SLOTS];
    __shared__ int s_on[SLOTS];
    const int nu = NU ? NU : n_pos;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    int bx, by;
    down_block_of_grid(bx, by);
    const int r0 = bx * ROWS;
    const int e0 = by * k, ent = e0 + wave;   // (64 k threads: every wave has a slot)
    const int skipv = skip ? *skip : 0;
    const uint64_t blob = plan_ptr[ent];      // (asked for first: the weights' request waits for this one)
    const int ci = e0 + min((int) threadIdx.x & (SLOTS - 1), k - 1);
    const uint64_t c_ptr = plan_ptr[ci];
    const float c_w = plan_w[ci];
    // (an idle lane's weights read as zero, and so do its activations)
    const int at = PAIR ? lane & 31 : lane;
    const bool on = NU == 64 || at < nu;
    const int pos = on ? at : nu - 1;
    PosQ4K p;
    // Q8_K of h in registers (quant_q8k_block's arithmetic): the lane's 32 values are two runs of 16, a block is 8 lanes; the
    // block's signed maximum is the value at the FIRST largest magnitude, so candidates carry their index
    const int piece = pos & 7, j = piece >> 1, half = piece & 1;
    const bool rounded = hq_q != nullptr;
    float v[32];
    if (rounded) {
        pos_q4k_codes(p, pos, hq_q + (size_t) ent * (32 * nu), a.hq.d + (size_t) ent * nu, a.hq.bsums + (size_t) ent * (2 * nu));
    } else {
        const float* hrow = h + (size_t) ent * (32 * nu) + 256 * (pos >> 3) + 64 * j + 16 * half;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 lo = *(const float4*) (hrow + 4 * i), hi = *(const float4*) (hrow + 32 + 4 * i);
            v[4 * i] = lo.x, v[4 * i + 1] = lo.y, v[4 * i + 2] = lo.z, v[4 * i + 3] = lo.w;
            v[16 + 4 * i] = hi.x, v[16 + 4 * i + 1] = hi.y, v[16 + 4 * i + 2] = hi.z, v[16 + 4 * i + 3] = hi.w;
        }
    }
    if (skipv) return;
    const uint32_t rb = (uint32_t) nu * 18u, past = (uint32_t) n_embd * rb;   // bytes of a row: 144 a block
    pos_q4k_init(p, pos, PAIR ? (uint32_t) (lane >> 5) * 4u * rb : 0u, on, past);
    // the first rows' weights are requested before h is rounded: their latency hides behind that arithmetic
    // (no blob: an empty resource, whose loads read as zero and touch nothing)
    const uint64_t mat = blob ? blob + a.layout.down_off : 0ull;
    const uint32_t mat_lo = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) mat);
    const uint32_t mat_hi = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) (mat >> 32));
    const __amdgpu_buffer_rsrc_t rs = weight_rsrc(((uint64_t) mat_hi << 32) | (uint64_t) mat_lo, (mat_lo | mat_hi) != 0u ? past : 0u);
    constexpr int DEPTH = AHEAD ? NB : 1;
    u32x4 hd[DEPTH], qd[DEPTH];
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
        hd[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, p.o_hdr, (uint32_t) (r0 + i) * rb, 0);
        qd[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, p.o_q, (uint32_t) (r0 + i) * rb, 0);
    }
    if (threadIdx.x < SLOTS) {
        s_on[threadIdx.x] = (int) threadIdx.x < k && c_ptr != 0ull;
        s_w[threadIdx.x] = c_w;
    }
    if (blob != 0ull) {
        if (!rounded) {
            if (!on) {
#pragma unroll
                for (int i = 0; i < 32; ++i) v[i] = 0.0f;
            }
            int y[8];
            float d;
            q8k_round_lane32(v, [&](int i) { return 64 * j + 16 * half + (i < 16 ? i : i + 16); }, y, d);
#pragma unroll
            for (int i = 0; i < 4; ++i) p.ylo[i] = y[i], p.yhi[i] = y[4 + i];
            p.dx = d;
            p.slo = dot4(0x01010101, p.ylo[0], dot4(0x01010101, p.ylo[1], dot4(0x01010101, p.ylo[2], dot4(0x01010101, p.ylo[3], 0))));
            p.shi = dot4(0x01010101, p.yhi[0], dot4(0x01010101, p.yhi[1], dot4(0x01010101, p.yhi[2], dot4(0x01010101, p.yhi[3], 0))));
        }
        pos_q4k_idle(p, on);
#pragma unroll 1
        for (int r = 0; r < ROWS; r += 8) {
            float acc[NB];
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const u32x4 hc = hd[i % DEPTH], qc = qd[i % DEPTH];
                if (!AHEAD && (i + 1 < NB || r + 8 < ROWS)) {   // (the next step's rows, or the next batch's first)
                    const uint32_t next = (uint32_t) (r0 + r + (i + 1 < NB ? i + 1 : 8)) * rb;
                    hd[0] = __builtin_amdgcn_raw_buffer_load_b128(rs, p.o_hdr, next, 0);
                    qd[0] = __builtin_amdgcn_raw_buffer_load_b128(rs, p.o_q, next, 0);
                }
                acc[i] = pos_q4k_value(p, hc, qc);
                asm volatile("" : "+v"(acc[i]));
            }
            if constexpr (PAIR) {
                const float s = reduce4_half(acc, lane);
                if ((lane & 7) == 0) part[wave][r + 4 * (lane >> 5) + ((lane >> 3) & 3)] = s;
            } else {
                const float s = add_other_half(reduce8_half(acc, lane));
                if ((lane & 35) == 0) part[wave][r + ((lane >> 2) & 7)] = s;
            }
        }
    }
    __syncthreads();
    if (threadIdx.x < ROWS) {
        const int c = threadIdx.x;
        float sum = 0.0f;
        bool first = true;
#pragma unroll
        for (int i = 0; i < SLOTS; ++i) {   // the present slots in slot order; the first product starts the sum
            const bool have = s_on[i] != 0;
            const float pv = __fmul_rn(part[i][c], s_w[i]);
            const float t = first ? pv : __fadd_rn(sum, pv);
            sum = have ? t : sum;
            first = first && !have;
        }
        const size_t o = (size_t) by * n_embd + r0 + c;
        if (a.add && (!a.add_flag || *a.add_flag)) sum = __fadd_rn(sum, a.add[o]);
        if (a.add2) sum = __fadd_rn(sum, a.add2[o]);
        a.out[o] = sum;
        if (a.part)
            for (int i = 0; i < k; ++i)
                if (s_on[i]) a.part[(size_t) (e0 + i) * n_embd + r0 + c] = part[i][c];
    }
}

}  // namespace maya
