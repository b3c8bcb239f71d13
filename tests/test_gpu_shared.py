"""The routed layer with the shared expert beside it (maya_moe_layer_decode_shared): the shared expert's launches run on
the library's second stream while the routed experts' head and gate/up run on the caller's.  The result must be the bits
of the two calls it replaces - the shared expert through the stage calls, then the routed layer with add = its output -
eagerly, call after call on changing inputs, and replayed from a HIP graph."""
import numpy as np
import pytest
import torch

from gpu_util import oracle_layer, rel_l2
import bench_workloads as workloads

pytestmark = pytest.mark.gpu
IQ2_S, Q4_K, Q8_0 = 22, 12, 8
FIELDS = {IQ2_S: (82, {0: (2e-3, 6e-3)}), Q4_K: (144, {0: (2e-4, 6e-4), 2: (2e-4, 6e-4)}), Q8_0: (34, {0: (1e-4, 4e-4)})}


@pytest.fixture(scope="module")
def lib():
    from maya_amd import lib as L
    L.load()
    return L


def build(lib, gt, dt, st, E, FF, NE, TK, T, seed):
    gguf, bb = lib.layout(gt, dt, E, FF)
    pool = torch.empty(NE * bb, dtype=torch.uint8, device="cuda")
    view = pool.view(NE, bb)
    view[:, :gguf.down_off] = workloads.random_blocks(NE * gguf.down_off, *FIELDS[gt], seed).view(NE, -1)
    view[:, gguf.down_off:] = workloads.random_blocks(NE * (bb - gguf.down_off), *FIELDS[dt], seed + 1).view(NE, -1)
    packed = torch.empty_like(pool)
    for e in range(NE):
        lib.repack(gguf, view[e], packed[e * bb:(e + 1) * bb])
    table = torch.tensor([packed.data_ptr() + e * bb for e in range(NE)], dtype=torch.int64, device="cuda")
    sg, sbb = lib.layout(st, st, E, FF)
    sh = workloads.random_blocks(sbb, *FIELDS[st], seed + 2)
    sh_packed = torch.empty_like(sh)
    lib.repack(sg, sh, sh_packed)
    torch.cuda.synchronize()
    layer = lib.MoeLayer(gt, dt, E, FF, NE, TK, max_tokens=T, packing=lib.PACK_STREAM)
    dense = lib.DenseExpert(st, st, E, FF, T, sh_packed.data_ptr(), packing=lib.PACK_STREAM)
    return dict(gguf=gguf, view=view, packed=packed, table=table, sg=sg, sh=sh, sh_packed=sh_packed, layer=layer, dense=dense)


def inputs(E, NE, T, seed):
    rng = np.random.default_rng(seed)
    return (torch.from_numpy(rng.standard_normal((T, NE)).astype(np.float32)).cuda(),
            torch.from_numpy(rng.standard_normal((T, E)).astype(np.float32)).cuda(),
            torch.from_numpy(rng.standard_normal((T, E)).astype(np.float32)).cuda())


def two_calls(w, logits, x, add, limit):
    """The shared expert through the stage calls (the residual in its down launch), then the routed layer on top of it."""
    a = w["dense"].args
    a.add = add.data_ptr() if add is not None else None
    sh = w["dense"].forward(x, limit=limit)
    a.add = None
    return w["layer"].forward(w["table"], logits, x, add=sh).clone()


@pytest.mark.parametrize("gt,dt,st,E,FF,NE,TK,T", [
    (IQ2_S, Q4_K, Q8_0, 7168, 2048, 32, 8, 8),    # configs[2]'s types and shape (fewer experts resident)
    (IQ2_S, IQ2_S, Q8_0, 7168, 2048, 16, 8, 1),   # one token: the down kernel that rounds h itself waits for the join
    (Q4_K, Q4_K, Q4_K, 4096, 1024, 8, 2, 3),
    (IQ2_S, Q4_K, Q8_0, 2816, 1280, 16, 4, 3),    # rows that end inside a wave
    (Q4_K, Q4_K, IQ2_S, 1792, 768, 12, 10, 2),    # and more than 8 slots
])
def test_layer_with_shared_expert_is_the_two_calls(lib, gt, dt, st, E, FF, NE, TK, T):
    w = build(lib, gt, dt, st, E, FF, NE, TK, T, 500 + T)
    for rep in range(3):   # call after call: the second stream's buffers are reused without a host synchronisation
        logits, x, add = inputs(E, NE, T, 510 + rep)
        use_add = add if rep != 1 else None
        got = w["layer"].forward(w["table"], logits, x, add=use_add, shared=w["dense"], shared_limit=7.0).clone()
        ids = w["layer"].ids[:T].clone()
        want = two_calls(w, logits, x, use_add, 7.0)
        torch.cuda.synchronize()
        assert torch.equal(ids, w["layer"].ids[:T])
        assert torch.equal(got, want), rep
        assert float(got.abs().max()) > 0


def test_against_the_cpu_path(lib, oracle):
    gt, dt, st, E, FF, NE, TK, T = IQ2_S, Q4_K, Q8_0, 7168, 2048, 32, 8, 4
    w = build(lib, gt, dt, st, E, FF, NE, TK, T, 530)
    logits, x, _ = inputs(E, NE, T, 531)
    out = w["layer"].forward(w["table"], logits, x, shared=w["dense"]).cpu().numpy()

    class Blobs:
        def __getitem__(self, e):
            return w["view"][e].cpu().numpy()
    ids, _, want = oracle_layer(oracle, gt, dt, Blobs(), TK, E, FF, logits.cpu().numpy(), x.cpu().numpy())
    assert np.array_equal(w["layer"].ids[:T].cpu().numpy(), ids)
    shb, sg = w["sh"].cpu().numpy(), w["sg"]
    for t in range(T):
        s = oracle.expert(st, st, shb, shb[sg.up_off:], shb[sg.down_off:], E, FF, x[t:t + 1].cpu().numpy())[0]
        assert rel_l2(out[t], want[t] + s) <= 1e-3, (t, rel_l2(out[t], want[t] + s))


def test_replayed_from_a_graph(lib):
    """Captured once, replayed with eager work and synchronisations in between, on inputs that change between replays."""
    gt, dt, st, E, FF, NE, TK, T = IQ2_S, Q4_K, Q8_0, 7168, 2048, 32, 8, 8
    w = build(lib, gt, dt, st, E, FF, NE, TK, T, 540)
    logits, x, _ = inputs(E, NE, T, 541)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        w["layer"].forward(w["table"], logits, x, shared=w["dense"], stream=s)   # (warm: nothing is set up under capture)
    s.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        w["layer"].forward(w["table"], logits, x, shared=w["dense"], stream=torch.cuda.current_stream())
    for rep in range(4):
        l2, x2, _ = inputs(E, NE, T, 550 + rep)
        logits.copy_(l2)
        x.copy_(x2)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        got = w["layer"].out[:T].clone()
        want = two_calls(w, logits, x, None, float("inf"))
        torch.cuda.synchronize()
        assert torch.equal(got, want), rep


def test_refusals_leave_the_stream_usable(lib):
    gt, dt, st, E, FF, NE, TK, T = Q4_K, Q4_K, Q4_K, 4096, 1024, 8, 2, 3
    w = build(lib, gt, dt, st, E, FF, NE, TK, T, 560)
    logits, x, _ = inputs(E, NE, T, 561)
    other = lib.DenseExpert(st, st, E, FF, T + 1, w["sh_packed"].data_ptr(), packing=lib.PACK_STREAM)
    with pytest.raises(AssertionError):
        w["layer"].forward(w["table"], logits, x, shared=other)
    a = other.args
    import ctypes as C
    L = lib.load()
    rc = L.maya_moe_layer_decode_shared(C.byref(w["layer"].layout), w["table"].data_ptr(), NE, TK, None, logits.data_ptr(), x.data_ptr(), 0, T,
                                        float("inf"), C.byref(a), w["layer"].ids.data_ptr(), w["layer"].weights.data_ptr(),
                                        w["layer"].out.data_ptr(), w["layer"].ws.data_ptr(), w["layer"].ws_bytes, None)
    assert rc != 0 and b"tokens" in L.maya_last_error()
    # a routed layer that is refused (k above the number of experts): asked before the fork, so the status is > 0, nothing
    # was launched on either stream, and the next call works
    rc = L.maya_moe_layer_decode_shared(C.byref(w["layer"].layout), w["table"].data_ptr(), 1, TK, None, logits.data_ptr(), x.data_ptr(), 0, T,
                                        float("inf"), C.byref(w["dense"].args), w["layer"].ids.data_ptr(), w["layer"].weights.data_ptr(),
                                        w["layer"].out.data_ptr(), w["layer"].ws.data_ptr(), w["layer"].ws_bytes, None)
    assert rc > 0 and b"n_expert" in L.maya_last_error()
    torch.cuda.synchronize()
    got = w["layer"].forward(w["table"], logits, x, shared=w["dense"]).clone()
    want = two_calls(w, logits, x, None, float("inf"))
    torch.cuda.synchronize()
    assert torch.equal(got, want)


def test_another_stream_is_refused_while_the_side_stream_is_inside_a_capture(lib):
    """The device's one side stream belongs to an open capture until that capture ends: a call from another stream in between
    gets MAYA_E_BUSY and launches nothing, the capture stays valid (the same capture may call again), and its graph replays
    with the right bits."""
    import ctypes as C
    gt, dt, st, E, FF, NE, TK, T = IQ2_S, Q4_K, Q8_0, 4096, 2048, 16, 4, 2
    w = build(lib, gt, dt, st, E, FF, NE, TK, T, 570)
    logits, x, _ = inputs(E, NE, T, 571)
    L = lib.load()
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    with torch.cuda.stream(s1):
        w["layer"].forward(w["table"], logits, x, shared=w["dense"], stream=s1)
    s1.synchronize()
    out2 = torch.zeros_like(w["layer"].out)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s1):
        w["layer"].forward(w["table"], logits, x, shared=w["dense"], stream=torch.cuda.current_stream())
        rc = L.maya_moe_layer_decode_shared(C.byref(w["layer"].layout), w["table"].data_ptr(), NE, TK, None, logits.data_ptr(), x.data_ptr(),
                                            0, T, float("inf"), C.byref(w["dense"].args), w["layer"].ids.data_ptr(),
                                            w["layer"].weights.data_ptr(), out2.data_ptr(), w["layer"].ws.data_ptr(), w["layer"].ws_bytes,
                                            C.c_void_p(s2.cuda_stream))
        busy_msg = L.maya_last_error()
        w["layer"].forward(w["table"], logits, x, shared=w["dense"], stream=torch.cuda.current_stream())   # the same capture again
    assert rc == 5 and b"capture" in busy_msg
    s2.synchronize()
    assert not out2.any()   # nothing ran for the refused call
    l2, x2, _ = inputs(E, NE, T, 572)
    logits.copy_(l2)
    x.copy_(x2)
    torch.cuda.synchronize()
    g.replay()
    torch.cuda.synchronize()
    got = w["layer"].out[:T].clone()
    want = two_calls(w, logits, x, None, float("inf"))
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    # after the capture has ended the other stream is served
    with torch.cuda.stream(s2):
        got2 = w["layer"].forward(w["table"], logits, x, shared=w["dense"], stream=s2).clone()
    s2.synchronize()
    assert torch.equal(got2, want)


@pytest.mark.parametrize("gt,E,FF,NE,TK,T,dtype", [
    (IQ2_S, 7168, 2048, 24, 8, 1, torch.bfloat16),    # one token: the shared expert's gate/up rounds x itself
    (Q4_K, 2304, 768, 40, 3, 1, torch.float16),       # rows that end inside a wave
    (Q4_K, 2048, 512, 300, 2, 5, torch.float32),      # more experts than the head of several tokens takes: x rounded by its own launch
    (Q8_0, 2816, 1280, 20, 4, 9, torch.bfloat16),     # the head rounds x once for both; two chunks of tokens
    (Q4_K, 4096, 2048, 32, 1, 16, torch.float32),     # one slot a token
])
def test_shared_q8_0_in_one_stream(lib, gt, E, FF, NE, TK, T, dtype):
    """A Q8_0 shared expert's two launches round x and h and combine themselves: the bits of its stage calls with their own
    launches for that, then the routed layer on top; x also from an address that is not 16-byte aligned."""
    w = build(lib, gt, gt, Q8_0, E, FF, NE, TK, T, 600 + T)
    for rep in range(2):
        logits, x, add = inputs(E, NE, T, 610 + rep)
        x = x.to(dtype)
        x[0, 32:64] = 0.0
        buf = torch.zeros(T * E + 2, dtype=dtype, device="cuda")
        xs = buf[2:].view(T, E).copy_(x) if rep else x
        use_add = None if rep else add
        got = w["layer"].forward(w["table"], logits, xs, add=use_add, shared=w["dense"], shared_limit=5.0).clone()
        shared = w["dense"].out.clone()
        want = two_calls(w, logits, x, use_add, 5.0)
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(shared, w["dense"].out), rep


def test_down_of_one_slot_combines_as_of_two(lib):
    """down_q80_pos_kernel writes a one-slot call's combined rows itself: the bits of the two-slot call whose second slot is left
    out (which combines in a launch), with a token whose only slot is left out, weights, both residuals, a flagged one and skip."""
    import ctypes as C
    E, FF, T = 2304, 768, 3
    gguf, bb = lib.layout(Q8_0, Q8_0, E, FF)
    raw = workloads.random_blocks(bb, *FIELDS[Q8_0], 77)
    blob = torch.empty_like(raw)
    lib.repack(gguf, raw, blob)
    rng = np.random.default_rng(78)
    t = lambda *s: torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda()  # noqa: E731
    h, add, add2, wts = t(T, FF), t(T, E), t(T, E), t(T)
    ptr1 = torch.tensor([blob.data_ptr(), 0, blob.data_ptr()], dtype=torch.int64, device="cuda")
    ptr2 = torch.stack([ptr1, torch.zeros_like(ptr1)], 1).reshape(-1).contiguous()
    h2 = torch.stack([h, h], 1).reshape(2 * T, FF).contiguous()
    w2 = torch.stack([wts, wts], 1).reshape(-1).contiguous()
    flag, skip = torch.zeros(1, dtype=torch.int32, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")

    def down(k, ptr, wt, hh):
        grp = lib.group(ptr)
        hq = lib.quant_act(Q8_0, hh)
        out, part = torch.full((T, E), 3.0, device="cuda"), torch.zeros((T * k, E), device="cuda")
        a = lib.Args()
        a.layout = lib.copy_layout(gguf, lib.PACK_STREAM)
        a.n_tokens, a.k = T, k
        a.plan_ptr, a.plan_w = ptr.data_ptr(), wt.data_ptr()
        a.grp_ptr, a.grp_start, a.grp_ent, a.n_groups = (g.data_ptr() for g in grp)
        a.x, a.h, a.hq, a.part, a.out = hq.c(), hh.data_ptr(), hq.c(), part.data_ptr(), out.data_ptr()
        a.add, a.add2, a.add_flag, a.skip = add.data_ptr(), add2.data_ptr(), flag.data_ptr(), skip.data_ptr()
        lib.check(lib.load().maya_moe_down(C.byref(a), lib._stream(None)))
        torch.cuda.synchronize()
        return out, part
    for f, s in ((0, 0), (1, 0), (1, 1)):
        flag.fill_(f)
        skip.fill_(s)
        (one, p1), (two, p2) = down(1, ptr1, wts, h), down(2, ptr2, w2, h2)
        assert torch.equal(one, two), (f, s)
        assert s or torch.equal(p1[::2], p2.view(T, 2, E)[::2, 0])


def kernels_of(call):
    """The kernel launches of a call, counted in a captured graph."""
    import ctypes as C
    hip, g = C.CDLL("libamdhip64.so"), torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(g, stream=torch.cuda.Stream()):
        call()
    graph, n = C.c_void_p(g.raw_cuda_graph()), C.c_size_t(0)
    assert hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0
    nodes, kind, count = (C.c_void_p * n.value)(), C.c_int(0), 0
    assert hip.hipGraphGetNodes(graph, nodes, C.byref(n)) == 0
    for node in nodes:
        assert hip.hipGraphNodeGetType(C.c_void_p(node), C.byref(kind)) == 0
        count += kind.value == 0   # hipGraphNodeTypeKernel
    return count


@pytest.mark.parametrize("sigmoid", (False, True))
def test_short_windows_beside_the_second_stream_take_the_one_launch_head(lib, sigmoid):
    """Two to four tokens beside a shared expert of a type that has launches of its own: one launch less than more tokens have
    (the head groups its plan itself), counted in captured graphs; the bits of the two calls either way."""
    gt, st, E, FF, NE, TK = Q4_K, Q4_K, 2048, 768, 24, 8
    w = build(lib, gt, gt, st, E, FF, NE, TK, 8, 620)
    bias = torch.zeros(NE, device="cuda")
    router = lib.Router(lib.ROUTER_SIGMOID, 1, bias.data_ptr(), 2.5) if sigmoid else None
    dense = {T: lib.DenseExpert(st, st, E, FF, T, w["sh_packed"].data_ptr(), packing=lib.PACK_STREAM) for T in (2, 4, 5)}
    kernels = {}
    for T in dense:
        logits, x, _ = inputs(E, NE, T, 621 + T)
        sh = dense[T].forward(x)
        want = w["layer"].forward(w["table"], logits, x, add=sh, router=router).clone()
        got = w["layer"].forward(w["table"], logits, x, shared=dense[T], router=router).clone()
        torch.cuda.synchronize()
        assert torch.equal(got, want), T
        kernels[T] = kernels_of(lambda: w["layer"].forward(w["table"], logits, x, shared=dense[T], router=router, stream=torch.cuda.current_stream()))
    assert kernels[2] == kernels[4] == kernels[5] - 1, kernels


def test_a_shared_q8_0_experts_sums_at_any_two_byte_address(lib):
    """The head of several tokens stores two code sums at a time: where the caller's buffer is not aligned for that, x is rounded by a
    launch of its own, as maya_quant_act takes any buffer - the same codes, sums and outputs."""
    gt, E, FF, NE, TK, T = Q4_K, 2304, 768, 20, 4, 3
    w = build(lib, gt, gt, Q8_0, E, FF, NE, TK, T, 640)
    logits, x, _ = inputs(E, NE, T, 641)
    call = lambda: w["layer"].forward(w["table"], logits, x, shared=w["dense"], stream=torch.cuda.current_stream())  # noqa: E731
    want = call().clone()
    torch.cuda.synchronize()
    plain, sums = kernels_of(call), w["dense"].xq.bsums.clone()
    off = torch.zeros(T * (E // 16) + 1, dtype=torch.int16, device="cuda")[1:]
    assert off.data_ptr() % 4 == 2
    w["dense"].args.x.bsums = off.data_ptr()
    got = call().clone()
    torch.cuda.synchronize()
    assert torch.equal(got, want) and torch.equal(off.view(T, -1), sums)
    assert kernels_of(call) == plain + 1
