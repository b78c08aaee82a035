"""HIP graph capture of a decode step (marked ``gpu``).

Two layers of a decode step are captured once with ``torch.cuda.graph`` and replayed
several times, with other GPU work and host synchronisation between the replays:
  - RMSNorm and the INT4 QKV projection (a norm pass, then a GEMM whose K splits are added
    inside its launch, six of them at 8 rows and three at 64);
  - the fused RoPE + pool write at per-row positions;
  - paged attention over per-row lengths;
  - the INT4 O projection.

Each replay must equal the eager step bit for bit: the same kernels on the same inputs,
rewriting the same pool slots. None of these entry points records a memset or allocates
inside the library. The decode workspace is the caller's; the INT4 workspaces are part of the
graph (one per captured call).

A captured ``PagedKVCache.append`` advances the device allocator once per replay, exactly
as the same number of eager appends on a twin cache does.
"""

import numpy as np
import pytest
import torch

from conftest import banner

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
HQ, HKV, D, BS, L = 24, 8, 128, 64, 2


def _setup(B, seed):
    from fast_infer_amd import precompute_freqs, quantize_int4_groupwise

    g = torch.Generator(device=DEV).manual_seed(seed)
    rng = np.random.default_rng(seed)
    lens = torch.from_numpy(rng.integers(200, 1000, B).astype(np.int32)).to(DEV)
    width = 16
    N = B * width + 4
    table = torch.from_numpy(rng.permutation(N)[:B * width].astype(np.int32)).view(B, width).to(DEV)
    pools = [(torch.randn(N, BS, HKV, D, device=DEV, generator=g).half(),
              torch.randn(N, BS, HKV, D, device=DEV, generator=g).half()) for _ in range(L)]
    weights = []
    for _ in range(L):
        wqkv = (torch.randn(5120, 3072, device=DEV, generator=g) * 0.02).half()
        wo = (torch.randn(3072, 3072, device=DEV, generator=g) * 0.02).half()
        weights.append((quantize_int4_groupwise(wqkv), quantize_int4_groupwise(wo)))
    cos, sin = precompute_freqs(D, 4096)
    x = torch.randn(B, 3072, device=DEV, generator=g).half()
    norm_w = (1.0 + 0.1 * torch.randn(3072, device=DEV, generator=g)).half()
    return dict(lens=lens, pos=(lens - 1).contiguous(), table=table, pools=pools, weights=weights,
                cos=cos.half().to(DEV), sin=sin.half().to(DEV), x=x, norm_w=norm_w)


def _step(st, x, ws):
    from fast_infer_amd import int4_matmul, paged_attention, rms_norm_int4_matmul, rope_store_kv

    B = x.shape[0]
    for layer in range(L):
        wqkv, wo = st["weights"][layer]
        kc, vc = st["pools"][layer]
        qkv = rms_norm_int4_matmul(x, st["norm_w"], wqkv)
        q = qkv[:, :HQ * D].view(B, 1, HQ, D)
        k = qkv[:, HQ * D:(HQ + HKV) * D].view(B, 1, HKV, D)
        v = qkv[:, (HQ + HKV) * D:].view(B, 1, HKV, D)
        q_rot, _ = rope_store_kv(q, k, v, st["cos"], st["sin"], 0, kc, vc, st["table"],
                                 start_positions=st["pos"], return_k=False)
        attn = paged_attention(q_rot.view(B, HQ, D), kc, vc, st["table"], BS, 1024,
                               context_lens=st["lens"], workspace=ws)
        x = int4_matmul(attn.view(B, HQ * D), wo)
    return x


@pytest.mark.parametrize("B", [8, 64])
def test_decode_step_graph_replay(hip, B):
    banner(f"graph capture of a 2-layer decode step, batch {B}")
    from fast_infer_amd import paged_attention, paged_attention_workspace

    st = _setup(B, 50 + B)
    ws = paged_attention_workspace(B, HQ, HKV, 1024, D, DEV)
    # eager reference; the step rewrites the same
    # pool slots each time, so running it again leaves the pools unchanged
    ref = _step(st, st["x"], ws).clone()
    ref_pools = [(k.clone(), v.clone()) for k, v in st["pools"]]
    torch.cuda.synchronize()

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _step(st, st["x"], ws)  # warm-up on the capture stream's side, as torch advises
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()

    graph = torch.cuda.CUDAGraph()
    static_x = st["x"].clone()
    with torch.cuda.graph(graph):
        out = _step(st, static_x, ws)
    torch.cuda.synchronize()

    for rep in range(3):
        # unrelated eager work between replays, including a different decode call
        noise = torch.randn(1 << 20, device=DEV).sum()
        paged_attention(torch.randn(B, HQ, D, device=DEV).half(), st["pools"][0][0],
                        st["pools"][0][1], st["table"], BS, 1024, context_lens=st["lens"],
                        workspace=ws)
        torch.cuda.synchronize()
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ref), (rep, float((out.float() - ref.float()).abs().max()))
        for (k, v), (rk, rv) in zip(st["pools"], ref_pools):
            assert torch.equal(k, rk) and torch.equal(v, rv), rep
        assert torch.isfinite(noise)


@pytest.mark.parametrize("M,N,K,norm", [(8, 5120, 3072, False), (4, 3072, 8192, False),
                                        (12, 5120, 3072, True), (300, 3072, 8192, False)])
def test_default_captures_replayed_at_once(hip, M, N, K, norm):
    """Two graphs of split-K calls, captured the ordinary way (both on torch's shared capture
    stream, no workspace given), replayed at the same time on two streams beside eager calls on
    that capture stream: no call shares its workspace with another, so all keep their bits."""
    banner(f"two default captures replayed at once, {M} x {N} x {K}, norm {norm}")
    from fast_infer_amd import int4_matmul, quantize_int4_groupwise, rms_norm_int4_matmul

    g = torch.Generator(device=DEV).manual_seed(M + N)
    w = quantize_int4_groupwise((torch.randn(N, K, device=DEV, generator=g) * 0.02).half())
    nw = (1.0 + 0.1 * torch.randn(K, device=DEV, generator=g)).half()
    xs = [torch.randn(M, K, device=DEV, generator=g).half() for _ in range(3)]

    def call(x):
        return rms_norm_int4_matmul(x, nw, w) if norm else int4_matmul(x, w)

    refs = [call(x) for x in xs]
    capture = torch.cuda.graph.default_capture_stream or torch.cuda.Stream()
    torch.cuda.graph.default_capture_stream = capture
    with torch.cuda.stream(capture):
        call(xs[2])
    torch.cuda.synchronize()
    graphs, outs = [], []
    for x in xs[:2]:
        graphs.append(torch.cuda.CUDAGraph())
        with torch.cuda.graph(graphs[-1]):
            outs.append([call(x) for _ in range(20)])
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    for rep in range(6):
        for o in outs[0] + outs[1]:
            o.zero_()
        torch.cuda.synchronize()
        for graph, st in zip(graphs, streams):
            with torch.cuda.stream(st):
                graph.replay()
        with torch.cuda.stream(capture):
            eager = [call(xs[2]) for _ in range(20)]
        torch.cuda.synchronize()
        for got, ref in ((outs[0], refs[0]), (outs[1], refs[1]), (eager, refs[2])):
            assert all(torch.equal(o, ref) for o in got), rep


def test_captured_branches_of_split_calls(hip):
    """One capture on two streams, 20 split-K calls on each side of a fork: the branches may run
    at once, so each keeps counters of its own; calls of one branch and calls that need more
    counters than the first (a wide weight after a narrow one) share or replace theirs."""
    banner("two branches of split-K calls in one graph")
    from fast_infer_amd import int4_matmul, quantize_int4_groupwise

    g = torch.Generator(device=DEV).manual_seed(3)
    ws = [quantize_int4_groupwise((torch.randn(n, 3072, device=DEV, generator=g) * 0.02).half())
          for n in (640, 36864)]
    xs = [torch.randn(8, 3072, device=DEV, generator=g).half() for _ in range(2)]
    refs = [[int4_matmul(x, w) for w in ws] for x in xs]
    main, side = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    outs = [[], []]
    with torch.cuda.graph(graph, stream=main):
        side.wait_stream(main)
        with torch.cuda.stream(side):
            outs[1] = [int4_matmul(xs[1], ws[i % 3 // 2]) for i in range(20)]
        outs[0] = [int4_matmul(xs[0], ws[i % 3 // 2]) for i in range(20)]
        main.wait_stream(side)
    for rep in range(4):
        for o in outs[0] + outs[1]:
            o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        for got, ref in zip(outs, refs):
            assert all(torch.equal(o, ref[i % 3 // 2]) for i, o in enumerate(got)), rep


def test_many_captures_keep_the_in_launch_sum(hip):
    """A server that captures its step again and again: after 9000 captured split-K calls in 150
    graphs, a call is still one node (its K splits are added inside the launch).  The counters
    are told apart by the runtime's capture ids: no two captures may share one."""
    banner("150 captures of 60 split-K calls")
    import ctypes

    from fast_infer_amd import _lib, quantize_int4_groupwise

    maps = open("/proc/self/maps").read().split("\n")
    hiprt = ctypes.CDLL(next(m.split()[-1] for m in maps if "libamdhip64" in m))
    lib = _lib.load()
    M, N, K = 8, 5120, 3072
    w, sc = quantize_int4_groupwise((torch.randn(N, K, device=DEV) * 0.02).half())
    x, out = torch.randn(M, K, device=DEV).half(), torch.empty(M, N, dtype=torch.float16, device=DEV)
    need = lib.fi_int4_matmul_workspace_size(M, N, K)
    assert need > 0
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    side = torch.cuda.Stream()

    def call():
        _lib.check(lib.fi_int4_matmul(x.data_ptr(), K, M, K, w.data_ptr(), K // 2, sc.data_ptr(), K // 128,
                                      N, 128, out.data_ptr(), N, ws.data_ptr(), need, side.cuda_stream),
                   "fi_int4_matmul")

    call()  # the placement check runs at a device's first eager call
    torch.cuda.synchronize()
    st = ctypes.c_void_p(side.cuda_stream)
    ids = set()
    for i in range(150):
        graph, nodes = ctypes.c_void_p(), ctypes.c_size_t()
        status, capture = ctypes.c_int(), ctypes.c_ulonglong()
        assert hiprt.hipStreamBeginCapture(st, 1) == 0  # thread-local mode
        assert hiprt.hipStreamGetCaptureInfo(st, ctypes.byref(status), ctypes.byref(capture)) == 0
        ids.add(capture.value)
        for _ in range(60):
            call()
        assert hiprt.hipStreamEndCapture(st, ctypes.byref(graph)) == 0
        assert hiprt.hipGraphGetNodes(graph, None, ctypes.byref(nodes)) == 0
        assert hiprt.hipGraphDestroy(graph) == 0
        assert nodes.value == 60, i
    assert len(ids) == 150


def test_int4_workspace_two_captures_shared_pool(hip):
    """Graphs captured back to back on a shared memory pool, the last needing a larger split-K
    workspace than the first: the first graph's workspace must stay allocated, so replaying
    all (in either order, repeatedly) equals the eager results bit for bit."""
    banner("int4 split-K workspace across captures (8, 17, then 64 rows)")
    from fast_infer_amd import _lib, int4_matmul, quantize_int4_groupwise

    rows = (8, 17, 64)
    sizes = [_lib.load().fi_int4_matmul_workspace_size(m, 5120, 3072) for m in rows]
    assert 0 < sizes[0] < sizes[-1]

    g = torch.Generator(device=DEV).manual_seed(77)
    w = quantize_int4_groupwise((torch.randn(5120, 3072, device=DEV, generator=g) * 0.02).half())
    xs = {m: torch.randn(m, 3072, device=DEV, generator=g).half() for m in rows}
    refs = {m: int4_matmul(x, w).clone() for m, x in xs.items()}
    torch.cuda.synchronize()
    pool = torch.cuda.graph_pool_handle()
    graphs, outs = {}, {}
    for m in rows:
        graphs[m] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graphs[m], pool=pool):
            outs[m] = int4_matmul(xs[m], w)
        torch.cuda.synchronize()
    for rep in range(3):
        for m in (rows if rep % 2 == 0 else rows[::-1]):
            outs[m].zero_()
            graphs[m].replay()
        torch.cuda.synchronize()
        for m in rows:
            assert torch.equal(outs[m], refs[m]), (rep, m)


def test_block_manager_append_graph_replay(hip):
    banner("graph capture of PagedKVCache.append")
    from fast_infer_amd import PagedKVCache

    B = 16
    a = PagedKVCache(1, 8, 128, 2048, 64, DEV, max_batch=B, num_blocks=400)
    b = PagedKVCache(1, 8, 128, 2048, 64, DEV, max_batch=B, num_blocks=400)
    lens0 = torch.randint(0, 700, (B,), generator=torch.Generator().manual_seed(3)).int()
    a.append(lens0.to(DEV))
    b.append(lens0.to(DEV))
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        starts_g, lens_g = a.append(1)  # recorded, not run
    torch.cuda.synchronize()
    assert torch.equal(a.seq_lens, b.seq_lens)
    for rep in range(5):
        graph.replay()
        sb, lb = b.append(1)
        torch.cuda.synchronize()
        assert torch.equal(starts_g, sb) and torch.equal(lens_g, lb), rep
        assert torch.equal(a.block_table, b.block_table), rep
        assert torch.equal(a.seq_lens, b.seq_lens) and torch.equal(a.num_alloc, b.num_alloc), rep
        assert torch.equal(a.free_queue, b.free_queue) and torch.equal(a.state, b.state), rep
    a.check()
