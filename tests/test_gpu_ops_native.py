"""The native form of the torch-facing calls (csrc/ops_binding.cpp) against their Python form, and the workspace that it
takes: other streams, threads on one stream, graphs."""
import ctypes
import threading

import pytest
import torch

from amdgpu_rustdsl_amd import lib, ops

pytestmark = pytest.mark.gpu
D = 128


class _Declines:
    """In place of the native module: every call goes to the Python form."""

    @staticmethod
    def _none(*a):
        return None

    attend = quantize_rows = quantize_v = quantize_qkv = _none


def _case(gpu, B, H, HK, S, SK, seed=0):
    g = torch.Generator(device=gpu)
    g.manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=g, device=gpu, dtype=torch.bfloat16)   # noqa: E731
    qs = torch.zeros(B * S * H * 4 + 2048 * H, dtype=torch.uint8, device=gpu)[: B * S * H * 4].view(B, S, H, 4)
    ks = torch.zeros(B * SK * HK * 4 + 2560 * H, dtype=torch.uint8, device=gpu)[: B * SK * HK * 4].view(B, SK, HK, 4)
    q, k = ops.quantize_mxfp8(r(B, S, H, D), qs, mul=ops.LOG2E_OVER_SQRT_D), ops.quantize_mxfp8(r(B, SK, HK, D), ks)
    v, vs = ops.quantize_v(r(B, SK, HK, D))
    return q, k, v, qs, ks, vs


def _out(t):
    return torch.full(t[0].shape, float("nan"), dtype=torch.bfloat16, device=t[0].device)


SHAPES = [(1, 1, 1, 256, 256), (1, 8, 8, 256, 2048), (2, 8, 2, 3, 1500), (8, 32, 8, 1, 2048), (1, 4, 4, 300, 129)]


@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
@pytest.mark.parametrize("kw", [{}, {"lse": True, "causal": True}, {"softmax_scale": 0.1, "partials": "fp32", "kv_fill": False}],
                         ids=["default", "lse_causal", "scaled_f32_nofill"])
def test_native_call_equals_python_call(gpu, monkeypatch, shape, kw):
    t = _case(gpu, *shape)
    kw = dict(kw)
    want_lse = kw.pop("lse", False)
    got = []
    for native in (True, False):
        if native:
            assert ops._native.attend.__name__ == "attend"
        else:
            monkeypatch.setattr(ops, "_native", _Declines)
        out, lse = _out(t), torch.zeros(t[0].shape[0], t[0].shape[2], t[0].shape[1], device=gpu) if want_lse else None
        ran = ops.fmha_fwd_mxfp8(*t, out, lse=lse, **kw)
        torch.cuda.synchronize()
        got.append((tuple(ran), ran.partials, out, lse))
    a, b = got
    assert a[:2] == b[:2]
    assert torch.equal(a[2].view(torch.int16), b[2].view(torch.int16))
    assert not want_lse or torch.equal(a[3], b[3])


def test_native_declines_what_python_reports(gpu):
    t = _case(gpu, 1, 4, 4, 64, 300)
    out = _out(t)
    bad = [(0, t[0].transpose(1, 2)), (0, t[0].cpu()), (1, t[1][:, :, :3]), (6, out.float()), (3, t[3][:, :-1])]
    for i, x in bad:
        args = list(t) + [out]
        args[i] = x
        assert ops._native.attend(*args, None, -1, 0, 0, 0, 0.0, 0, 0, 0, None) is None
        with pytest.raises(ValueError):
            ops.fmha_fwd_mxfp8(*args)
    short = torch.zeros(64 * 16, dtype=torch.uint8, device=gpu).view(1, 64, 4, 4)   # no slack behind the scales
    with pytest.raises(lib.FmhaError, match="GV-HOST-EXTENT") as e:
        ops.fmha_fwd_mxfp8(t[0], t[1], t[2], short, *t[4:], out)
    assert e.value.code == lib.FMHA_ERR_EXTENT
    with pytest.raises(RuntimeError):   # a batched tensor has no memory of its own: refused, not a crash
        torch.vmap(lambda q: (ops.fmha_fwd_mxfp8(q, *t[1:], out), q)[1])(t[0].unsqueeze(0))


def test_threads_and_streams_share_nothing_they_should_not(gpu):
    """Calls that use the workspace from four threads, two on one stream: every output is the single-threaded one."""
    cases = [_case(gpu, 2, 8, 2, 4, 3000, seed=i) for i in range(4)]
    want = []
    for t in cases:
        o = _out(t)
        ops.fmha_fwd_mxfp8(*t, o)
        want.append(o)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(gpu), torch.cuda.Stream(gpu)]
    outs = [[_out(t) for _ in range(12)] for t in cases]
    torch.cuda.synchronize()
    errors = []

    def work(i):
        try:
            with torch.cuda.stream(streams[i % 2]):
                for o in outs[i]:
                    ops.fmha_fwd_mxfp8(*cases[i], o)
        except Exception as e:   # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [x.start() for x in threads]
    [x.join() for x in threads]
    torch.cuda.synchronize()
    assert not errors, errors
    for i in range(4):
        for o in outs[i]:
            assert torch.equal(o.view(torch.int16), want[i].view(torch.int16)), i


def test_graph_survives_workspace_growth(gpu):
    """A captured call's workspace stays its own when a later, larger call grows the stream's workspace."""
    small, large = _case(gpu, 2, 8, 2, 4, 3000, seed=1), _case(gpu, 8, 32, 8, 4, 4096, seed=2)
    eager = _out(small)
    ops.fmha_fwd_mxfp8(*small, eager)
    torch.cuda.synchronize()
    s = torch.cuda.Stream(gpu)
    out = _out(small)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(s):
        ops.fmha_fwd_mxfp8(*small, out)   # the stream's workspace and the code objects, before the capture
        s.synchronize()
        with torch.cuda.graph(graph, stream=s):
            ops.fmha_fwd_mxfp8(*small, out)
        big = _out(large)
        ops.fmha_fwd_mxfp8(*large, big)
        s.synchronize()
        trash = [torch.full((1 << 22,), 0xff, dtype=torch.uint8, device=gpu) for _ in range(8)]   # would take a freed workspace
    torch.cuda.synchronize()
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), eager.view(torch.int16))
        trash[0].add_(1)
    del trash


def _eager(cases):
    want = []
    for t in cases:
        o = _out(t)
        ops.fmha_fwd_mxfp8(*t, o)
        want.append(o)
    torch.cuda.synchronize()
    return want


def test_calls_keep_no_memory(gpu):
    """A call gives its workspace back: on streams that were never used, eager, and around a capture."""
    t = _case(gpu, 2, 8, 2, 4, 3000, seed=1)
    out = _out(t)
    ops.fmha_fwd_mxfp8(*t, out)
    torch.cuda.synchronize()
    s, graph = torch.cuda.Stream(gpu), torch.cuda.CUDAGraph()
    before = torch.cuda.memory_allocated(gpu)
    with torch.cuda.stream(s):
        ops.fmha_fwd_mxfp8(*t, out)
    ops.fmha_fwd_mxfp8(*t, out, stream=torch.cuda.Stream(gpu).cuda_stream)
    with torch.cuda.graph(graph):
        ops.fmha_fwd_mxfp8(*t, out)
    torch.cuda.synchronize()
    # (torch keeps 1 KiB of random state for a graph; one partial of this call's 64 rows takes 33 KB)
    assert torch.cuda.memory_allocated(gpu) - before < 4096


def test_graphs_of_one_capture_stream_replay_together(gpu):
    """Two graphs captured one after the other, each of more calls than the workspace has slots, replayed on two streams at
    once, with eager calls on the capture stream between: the memory of each is its own."""
    cases = [_case(gpu, 8, 32, 8, 1, 2048, seed=i) for i in range(12)]
    want = _eager(cases)
    s = torch.cuda.Stream(gpu)
    graphs, outs = [], [_out(t) for t in cases]
    for half in (0, 6):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=s):
            for i in range(half, half + 6):
                ops.fmha_fwd_mxfp8(*cases[i], outs[i])
        graphs.append(graph)
    streams = [torch.cuda.Stream(gpu), torch.cuda.Stream(gpu)]
    extra = _out(cases[0])
    for _ in range(10):
        for o in outs:
            o.fill_(float("nan"))
        torch.cuda.synchronize()
        for st, graph in zip(streams, graphs):
            with torch.cuda.stream(st):
                graph.replay()
        with torch.cuda.stream(s):
            ops.fmha_fwd_mxfp8(*cases[0], extra)
        torch.cuda.synchronize()
        for i in range(12):
            assert torch.equal(outs[i].view(torch.int16), want[i].view(torch.int16)), i
        assert torch.equal(extra.view(torch.int16), want[0].view(torch.int16))


def test_stream_argument_takes_no_memory_in_use(gpu):
    """A call on another stream than torch's current one: memory that pending work of the current stream still writes is not
    its workspace."""
    t = _case(gpu, 2, 8, 2, 4, 3000, seed=3)
    (want,) = _eager([t])
    s, out = torch.cuda.Stream(gpu), _out(t)
    torch.cuda.synchronize()
    for size in (1 << 22, 1 << 24, 1 << 26):
        torch.cuda.empty_cache()
        blocks = [torch.empty(size, dtype=torch.uint8, device=gpu) for _ in range(4)]
        torch.cuda._sleep(20_000_000)   # (a spin of about 10 ms)
        for x in blocks:
            x.fill_(0xff)
        del blocks, x
        ops.fmha_fwd_mxfp8(*t, out, stream=s.cuda_stream)
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), want.view(torch.int16)), size


def _hip():
    """The HIP runtime that this process runs on."""
    with open("/proc/self/maps") as f:
        path = next(x.split()[-1] for x in f if "libamdhip64" in x)
    return ctypes.CDLL(path)


def test_capture_that_torch_does_not_know(gpu):
    """A graph captured through HIP itself: its workspace is nobody else's when it is replayed."""
    t, other = _case(gpu, 2, 8, 2, 4, 3000, seed=4), _case(gpu, 2, 8, 2, 4, 3000, seed=5)
    want, want_other = _eager([t, other])
    hip, s = _hip(), torch.cuda.Stream(gpu)
    handle, graph, ex = ctypes.c_void_p(s.cuda_stream), ctypes.c_void_p(), ctypes.c_void_p()
    out, o2 = _out(t), _out(other)
    torch.cuda.synchronize()
    assert hip.hipStreamBeginCapture(handle, 1) == 0   # thread-local mode
    for _ in range(5):
        ops.fmha_fwd_mxfp8(*t, out, stream=s.cuda_stream)
    assert hip.hipStreamEndCapture(handle, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    torch.cuda.empty_cache()
    trash = [torch.full((1 << 22,), 0xff, dtype=torch.uint8, device=gpu) for _ in range(8)]
    for _ in range(3):
        out.fill_(float("nan"))
        o2.fill_(float("nan"))
        torch.cuda.synchronize()
        assert hip.hipGraphLaunch(ex, handle) == 0
        with torch.cuda.stream(s):
            ops.fmha_fwd_mxfp8(*other, o2)
        ops.fmha_fwd_mxfp8(*other, o2)
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), want.view(torch.int16))
        assert torch.equal(o2.view(torch.int16), want_other.view(torch.int16))
        assert all(bool((x == 0xff).all()) for x in trash)
    assert hip.hipGraphExecDestroy(ex) == 0 and hip.hipGraphDestroy(graph) == 0


def test_without_memory_for_a_workspace(gpu):
    """A full-sequence call takes a workspace where it can have one; where it can't, its own kernel runs without, as it does for
    callers that pass none. The KV split needs its partials and says so."""
    B, H, S = 3, 8, 3001
    t, kv = _case(gpu, B, H, H, S, S), _case(gpu, 1, 8, 8, 2048, 2048)
    out, own, kv_out = _out(t), _out(t), _out(kv)
    p = lib.Params()
    p.o, p.q, p.k, p.v = (x.data_ptr() for x in (own, *t[:3]))
    p.q_descale, p.k_descale, p.v_descale = (x.data_ptr() for x in t[3:])
    p.B, p.H, p.HK, p.S, p.SK, p.path, p.no_check = B, H, H, S, S, -1, 1
    need = lib.auto_workspace_bytes(p)
    if not need:
        pytest.skip("this device's CU count splits no blocks of the shape")
    lib.run_auto(p, None, 0, torch.cuda.current_stream(gpu).cuda_stream)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(gpu).total_memory
    spare = []
    try:
        torch.cuda.set_per_process_memory_fraction(torch.cuda.memory_reserved(gpu) / total, gpu)
        for size in (32 << 20, 4 << 20):   # what the live tensors' segments have left, down to less than the workspaces
            with pytest.raises(torch.OutOfMemoryError):
                while True:
                    spare.append(torch.empty(size, dtype=torch.uint8, device=gpu))
        ops.fmha_fwd_mxfp8(*t, out)
        torch.cuda.synchronize()
        with pytest.raises(torch.OutOfMemoryError):
            ops.fmha_fwd_mxfp8(*kv, kv_out)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, gpu)
    assert torch.equal(out.view(torch.int16), own.view(torch.int16))
    del spare
    ops.fmha_fwd_mxfp8(*kv, kv_out)
    torch.cuda.synchronize()
    assert torch.isfinite(kv_out.float()).all()


def test_per_thread_streams(gpu):
    """hipStreamPerThread (handle 2) is one handle for as many streams as there are threads: their calls, at once."""
    cases = [_case(gpu, 8, 32, 8, 1, 2048, seed=i) for i in range(4)]
    want = _eager(cases)
    outs = [[_out(t) for _ in range(10)] for t in cases]
    torch.cuda.synchronize()
    errors = []

    def work(i):
        try:
            for o in outs[i]:
                ops.fmha_fwd_mxfp8(*cases[i], o, stream=2)
        except Exception as e:   # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [x.start() for x in threads]
    [x.join() for x in threads]
    torch.cuda.synchronize()
    assert not errors, errors
    for i in range(4):
        for o in outs[i]:
            assert torch.equal(o.view(torch.int16), want[i].view(torch.int16)), i
