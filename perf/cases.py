"""The calls a user of this framework makes, as cases that can be timed: decode layers (one token, verify windows, batches of
sequences), prompt chunks, and EXL3 layers, each through MoeLayer / DenseExpert / PrefillLayer / Exl3Layer as a serving
program holds them: the experts of one layer (or of several, where `layers` says so) resident in HBM in the packing the
kernels take, the layer objects made once, and a pass = one forward call a layer on inputs that are on the device."""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.abspath("project-maya_amd"))
from maya_amd import exl3, lib, prefill  # noqa: E402

Q8_0, Q4_K, IQ2_XXS, IQ1_S, IQ2_S, IQ1_M = lib.Q8_0, lib.Q4_K, lib.IQ2_XXS, lib.IQ1_S, lib.IQ2_S, lib.IQ1_M
DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
# a weight type's block: bytes, values, and where its FP16 scale sits and the range it is drawn from (IQ1_M spreads its
# scale over four words: made whole in `blocks`)
BLOCK = {Q8_0: (34, 32), Q4_K: (144, 256), IQ2_XXS: (66, 256), IQ1_S: (50, 256), IQ2_S: (82, 256), IQ1_M: (56, 256)}
SCALE = {Q8_0: (1e-4, 4e-4), IQ2_XXS: (2e-3, 6e-3), IQ1_S: (3e-3, 9e-3), IQ2_S: (2e-3, 6e-3)}


def decode(name, gate, down, n_embd, n_ff, experts, k, tokens, **more):
    c = {"kind": "decode", "gate": gate, "down": down, "n_embd": n_embd, "n_ff": n_ff, "experts": experts, "k": k, "tokens": tokens,
         "dtype": "bf16", "router": "softmax", "shared": 0, "layers": 1, "graph": False}
    c.update(more)
    return dict(c, name=name) if name else c


def prompt(name, gate, down, n_embd, n_ff, experts, k, tokens, **more):
    c = {"kind": "prompt", "gate": gate, "down": down, "n_embd": n_embd, "n_ff": n_ff, "experts": experts, "k": k, "tokens": tokens,
         "dtype": "bf16", "skew": 0.0}
    c.update(more)
    return dict(c, name=name) if name else c


def trellis(name, n_embd, n_ff, experts, k, tokens, k2, cb=exl3.CB_MUL1):
    c = {"kind": "exl3", "n_embd": n_embd, "n_ff": n_ff, "experts": experts, "k": k, "tokens": tokens, "k2": k2, "cb": cb}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one expert's GLU on one token, Q4_K: the smallest call there is (a dense FFN's row, a top-1 router)
        decode("expert_q4k_1tok", Q4_K, Q4_K, 7168, 2048, 16, 1, 1, dtype="f32"),
        # chat with one user: the routed layer of a large model on one token, two-bit experts
        decode("decode_iq2s_1tok", IQ2_S, IQ2_S, 7168, 2048, 256, 8, 1),
        # the same on a small model of many narrow experts: sixteen layers of a token, replayed from a graph as a serving
        # loop whose launches count does
        decode("decode_narrow_q4k_graph", Q4_K, Q4_K, 2048, 768, 128, 8, 1, layers=16, graph=True),
        # speculative decoding: a 4-token verify window over one-bit gate/up and two-bit down experts, the sigmoid router
        decode("window_iq1s_4tok", IQ1_S, IQ2_S, 6144, 2048, 160, 8, 4, router="sigmoid"),
        # eight users: mixed quantization (two-bit gate/up, four-bit down) and the shared expert every token takes
        decode("batch_mixed_shared_8tok", IQ2_S, Q4_K, 7168, 2048, 256, 8, 8, dtype="f32", shared=Q8_0),
        # the largest decode batch, four-bit experts of a middle-sized model
        decode("batch_q4k_16tok", Q4_K, Q4_K, 5120, 1536, 160, 8, 16),
        # a prompt's chunk under skewed routing, four-bit experts
        prompt("prompt_q4k_512tok", Q4_K, Q4_K, 7168, 2048, 256, 8, 512, dtype="f32", skew=1.1),
        # a long prompt taken in one chunk
        prompt("prompt_q4k_4096tok", Q4_K, Q4_K, 4096, 2048, 288, 8, 4096),
        # an odd-sized chunk over the mixed experts
        prompt("prompt_mixed_1187tok", IQ2_S, Q4_K, 7168, 2048, 256, 8, 1187, skew=0.6),
        # the tail of a prompt, or a short question: fewer tokens than experts
        prompt("prompt_iq2s_75tok", IQ2_S, IQ2_S, 6144, 1536, 160, 8, 75),
        # EXL3: a verify window at 3 bits a weight, and one token at 4
        trellis("exl3_3bit_4tok", 6144, 1536, 160, 8, 4, 6),
        trellis("exl3_4bit_1tok", 6144, 1536, 160, 8, 1, 8),
    ]


MOST_BYTES = 6.5e9       # a layer's resident experts
MOST_OPS = 1.6e12        # operations of a drawn prompt chunk


def log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    """One more case: widths of any multiple the formats allow, any number of experts, of slots and of tokens."""
    kind = rng.choice(("decode", "decode", "decode", "prompt", "prompt", "exl3"))
    if kind == "exl3":
        k2, cb = rng.choice(((4, 2), (5, 2), (6, 2), (7, 2), (8, 2), (10, 2), (6, 1), (8, 1)))
        return trellis(None, 128 * rng.randint(16, 56), 128 * rng.randint(6, 16), rng.randint(24, 200), rng.randint(2, 10),
                       log_int(rng, 1, 16), k2, cb)
    experts, k = rng.randint(16, 288), rng.randint(1, 10)
    n_embd, n_ff = 256 * rng.randint(8, 28), 256 * rng.randint(2, 8)
    if kind == "prompt":
        gate, down = rng.choice(((Q4_K, Q4_K), (Q4_K, Q4_K), (IQ2_S, Q4_K), (IQ2_S, IQ2_S)))
        n_embd, n_ff = 512 * -(-n_embd // 512), 512 * -(-n_ff // 512)   # (IQ2_S rows of a chunk: whole pairs of blocks)
        tokens = min(log_int(rng, 17, 4096), int(MOST_OPS / (6 * n_embd * n_ff * k)))
        experts = min(experts, int(MOST_BYTES / blob_bytes(gate, down, n_embd, n_ff)))
        return prompt(None, gate, down, n_embd, n_ff, experts, k, tokens, dtype=rng.choice(("bf16", "bf16", "f16", "f32")),
                      skew=rng.choice((0.0, 0.6, 1.1)))
    gate, down = rng.choice(((Q4_K, Q4_K), (Q4_K, Q4_K), (IQ2_S, IQ2_S), (IQ2_S, Q4_K), (IQ1_S, IQ2_S), (IQ1_S, IQ1_S),
                             (IQ1_M, IQ1_M), (IQ2_XXS, IQ2_S), (Q8_0, Q8_0)))
    experts = min(experts, int(MOST_BYTES / blob_bytes(gate, down, n_embd, n_ff)))
    return decode(None, gate, down, n_embd, n_ff, experts, k, log_int(rng, 1, 16), dtype=rng.choice(("bf16", "bf16", "f16", "f32")),
                  router=rng.choice(("softmax", "sigmoid")), shared=rng.choice((0, 0, 0, Q8_0)))


# ---- the algorithm's own bytes and operations

def blob_bytes(gate, down, n_embd, n_ff):
    row = lambda t, n: n // BLOCK[t][1] * BLOCK[t][0]  # noqa: E731
    return 2 * n_ff * row(gate, n_embd) + n_embd * row(down, n_ff)


def distinct(case):
    """Experts with at least one token, by the routing's distribution."""
    g = np.random.default_rng(1)
    ne, k = case["experts"], case["k"]
    got = []
    for _ in range(8 if case["tokens"] <= 16 else 1):
        s = g.standard_normal((case["tokens"], ne)) - case.get("skew", 0.0) * np.log(np.arange(1, ne + 1))
        got.append(np.unique(np.argpartition(-s, k - 1, axis=1)[:, :k]).size)
    return float(np.mean(got))


def exl3_bytes(case):
    return exl3.make_layout(case["n_embd"], case["n_ff"], case["k2"], case["cb"])[1]


def work(case):
    e, f, t, k = case["n_embd"], case["n_ff"], case["tokens"], case["k"]
    blob = exl3_bytes(case) if case["kind"] == "exl3" else blob_bytes(case["gate"], case["down"], e, f)
    x_size = 4 if case["kind"] == "exl3" else DTYPES[case["dtype"]].itemsize
    out_size = 2 if case["kind"] == "prompt" else 4
    n_bytes = distinct(case) * blob + t * (e * (x_size + out_size) + case["experts"] * 4)
    flops = 6 * e * f * t * k
    if case.get("shared"):
        n_bytes += blob_bytes(case["shared"], case["shared"], e, f)
        flops += 6 * e * f * t
    layers = case.get("layers", 1)
    return {"bytes": layers * n_bytes, "flops": layers * flops}


def tolerance(case):
    # The integer sums are exact and the F32 ones differ by order alone: the stream-packed kernels against the general ones on
    # the same experts in GGUF order, 3e-7.  What shows beyond that is a value of h next to a rounding boundary of its int8
    # code that moves by one code: 1 / (30 sqrt(n_ff)) of one expert's output, up to 1.5e-3 on one slot and 2.5e-4 over eight.
    # EXL3 rounds its rotated inputs to FP16, the same case at 2^-11.  bf16 outputs: 1.66e-3 from the F32 ones, and two of
    # them differ where a value sits next to a rounding boundary.
    if case["kind"] == "prompt":
        return {"rel": 2e-3, "max": 2e-2}
    return {"rel": 1e-3, "max": 1e-2}


# ---- inputs

def generator(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 1000003 + salt)
    return g


def q4k_blocks(n, g):
    """n Q4_K blocks of N(0, 0.02) weights: a sub-block's 32 values between its least and its greatest in 15 steps, the
    sub-blocks' steps and minimums in 63 steps of the block's two FP16 scales."""
    x = (torch.randn((n, 8, 32), device="cuda", generator=g) * 0.02)
    lo = x.amin(2)
    step = (x.amax(2) - lo) / 15
    d, dmin = ((v.amax(1) / 63).to(torch.float16) for v in (step, -lo))
    sc = (step / d.float()[:, None]).round().clamp(1, 63).int()
    m = (-lo / dmin.float()[:, None]).round().clamp(0, 63).int()
    q = ((x + (dmin.float()[:, None] * m)[:, :, None]) / (d.float()[:, None] * sc)[:, :, None]).round().clamp(0, 15).int()
    b = torch.empty((n, 144), dtype=torch.uint8, device="cuda")
    b[:, 0:2], b[:, 2:4] = d.view(torch.uint8).view(n, 2), dmin.view(torch.uint8).view(n, 2)
    b[:, 4:8] = (sc[:, :4] | (sc[:, 4:] >> 4 << 6)).to(torch.uint8)
    b[:, 8:12] = (m[:, :4] | (m[:, 4:] >> 4 << 6)).to(torch.uint8)
    b[:, 12:16] = ((sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)).to(torch.uint8)
    q = q.view(n, 4, 2, 32)
    b[:, 16:] = (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(n, 128).to(torch.uint8)
    return b


def blocks(t, n, g):
    """n blocks of type t: Q4_K encoded from Gaussian weights, Q8_0 codes of the same, the codebook formats' indices and signs at
    random (every pattern is a codebook entry) under block scales of a usual size."""
    if t == Q4_K:
        return q4k_blocks(n, g)
    size = BLOCK[t][0]
    b = torch.randint(0, 256, (n, size), dtype=torch.uint8, device="cuda", generator=g)
    if t == IQ1_M:   # the FP16 scale's four nibbles are the top ones of the last four words
        d = (torch.rand(n, device="cuda", generator=g) * 6e-3 + 3e-3).to(torch.float16).view(torch.int16).int() & 0xffff
        for i in range(4):
            b[:, 49 + 2 * i] = ((b[:, 49 + 2 * i].int() & 15) | (((d >> (4 * i)) & 15) << 4)).to(torch.uint8)
        return b
    lo, hi = SCALE[t]
    d = (torch.rand(n, device="cuda", generator=g) * (hi - lo) + lo).to(torch.float16)
    b[:, 0:2] = d.view(torch.uint8).view(n, 2)
    if t == Q8_0:
        codes = (torch.randn((n, 32), device="cuda", generator=g) * 50).round().clamp(-127, 127).to(torch.int8)
        b[:, 2:] = codes.view(torch.uint8)
    return b


def rows(t, n_bytes, g):
    """n_bytes of blocks in random order out of 2^15 different ones."""
    size = BLOCK[t][0]
    base = blocks(t, 1 << 15, g)
    return base[torch.randint(0, 1 << 15, (n_bytes // size,), device="cuda", generator=g)].view(-1)


def expert_pool(gate, down, n_embd, n_ff, experts, g):
    """The layer's experts as its loader puts them into HBM (stream packing), and the table of their addresses."""
    gguf, size = lib.layout(gate, down, n_embd, n_ff)
    mats = [rows(t, experts * n, g) for t, n in ((gate, gguf.up_off), (gate, gguf.down_off - gguf.up_off), (down, size - gguf.down_off))]
    stride = -(-size // 256) * 256
    pool = torch.empty(experts * stride, dtype=torch.uint8, device="cuda")
    lib.pack_experts(gguf, mats[0], mats[1], mats[2], experts, lib.PACK_STREAM, pool, stride)
    table = torch.arange(experts, dtype=torch.int64, device="cuda") * stride + pool.data_ptr()
    return pool, table


def trellis_pool(case, g):
    l, size = exl3.make_layout(case["n_embd"], case["n_ff"], case["k2"], case["cb"])
    stride, ne = -(-size // 256) * 256, case["experts"]
    pool = torch.randint(-2 ** 63, 2 ** 63 - 1, (ne, stride // 8), dtype=torch.int64, device="cuda", generator=g).view(torch.uint8).view(ne, stride)
    for r in range(3):
        k, n = exl3.matrix_of(l, r)
        suh = (torch.randint(0, 2, (ne, k), device="cuda", generator=g) * 2 - 1).to(torch.float16)
        svh = ((torch.randint(0, 2, (ne, n), device="cuda", generator=g) * 2 - 1) *
               (torch.rand((ne, n), device="cuda", generator=g) + 0.5) / k ** 0.5).to(torch.float16)
        pool[:, l.suh[r]:l.suh[r] + 2 * k] = suh.view(torch.uint8)
        pool[:, l.svh[r]:l.svh[r] + 2 * n] = svh.view(torch.uint8)
    return l, pool, torch.arange(ne, dtype=torch.int64, device="cuda") * stride + pool.data_ptr()


def prepare(case, seed):
    lib.check(lib.load().maya_init())
    ne, t, e, f = case["experts"], case["tokens"], case["n_embd"], case["n_ff"]
    calls, keep = [], []
    for i in range(case.get("layers", 1)):
        g = generator(seed, i)
        logits = torch.randn((t, ne), device="cuda", generator=g)
        x = torch.randn((t, e), device="cuda", generator=g)
        if case["kind"] == "exl3":
            l, pool, table = trellis_pool(case, g)
            layer, more = exl3.Exl3Layer(l, ne, case["k"], max_tokens=t), {}
            x = x.half().float()
        elif case["kind"] == "prompt":
            pool, table = expert_pool(case["gate"], case["down"], e, f, ne, g)
            logits -= case["skew"] * torch.log(torch.arange(1, ne + 1, device="cuda"))
            l = lib.copy_layout(lib.layout(case["gate"], case["down"], e, f)[0], lib.PACK_STREAM)
            layer, more = prefill.PrefillLayer(l, ne, case["k"], t), {}
            x = x.to(DTYPES[case["dtype"]])
        else:
            pool, table = expert_pool(case["gate"], case["down"], e, f, ne, g)
            layer, more = lib.MoeLayer(case["gate"], case["down"], e, f, ne, case["k"], max_tokens=t, packing=lib.PACK_STREAM), {}
            x = x.to(DTYPES[case["dtype"]])
            if case["router"] == "sigmoid":
                bias = torch.randn(ne, device="cuda", generator=g) * 0.1
                more["router"] = lib.Router(lib.ROUTER_SIGMOID, lib.NORM_CLAMP, bias.data_ptr(), 2.5)
                keep.append(bias)
            if case["shared"]:
                shared_pool, at = expert_pool(case["shared"], case["shared"], e, f, 1, g)
                more["shared"] = lib.DenseExpert(case["shared"], case["shared"], e, f, t, int(at.item()), packing=lib.PACK_STREAM)
                keep.append(shared_pool)
        keep.append(pool)
        calls.append((layer, table, logits, x, more))
    state = {"calls": calls, "keep": keep, "tokens": t, "graph": None}
    if case.get("graph"):
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(side):
            forward(calls)
        side.synchronize()
        with torch.cuda.graph(graph, stream=side):
            forward(calls)
        state["graph"] = graph
    return state


def forward(calls):
    return [layer.forward(table, logits, x, **more) for layer, table, logits, x, more in calls]


def run(state):
    """One pass: the layers' outputs, the experts chosen and their weights."""
    t = state["tokens"]
    if state["graph"] is not None:
        state["graph"].replay()
        outs = [c[0].out[:t] for c in state["calls"]]
    else:
        outs = forward(state["calls"])
    return {"out": outs, "ids": [c[0].ids[:t] for c in state["calls"]], "weights": [c[0].weights[:t] for c in state["calls"]]}
