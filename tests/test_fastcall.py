"""The native call path of the ops against their Python steps: the same
results, and the same errors for what neither takes."""

import math

import pytest

torch = pytest.importorskip("torch")

from decodebench_amd import ops  # noqa: E402
from decodebench_amd.quant import quantize_e4m3_rows  # noqa: E402


class _Sub(torch.Tensor):
    pass


@pytest.fixture
def steps(monkeypatch):
    """A function that runs a call through the Python steps only."""
    def run(fn):
        with monkeypatch.context() as m:
            m.setattr(ops, "_fast", None)
            return fn()
    return run


def _outcome(fn):
    try:
        return fn()
    except Exception as exc:
        return type(exc), str(exc)


def _load():
    if not ops.LIB_PATH.exists():
        pytest.skip("the HIP library is not built")
    ops.load_library()
    assert ops._fast is not None, "lib/_fastcall.so did not load"


def test_refusals_are_the_python_steps_own(steps):
    """CPU tensors, wrong ranks, types and objects: refused with the same
    exception, before anything is launched."""
    _load()
    h = torch.zeros(2, 64, dtype=torch.float16)
    W = torch.zeros(8, 64, dtype=torch.float16)
    g = torch.zeros(64, dtype=torch.float16)
    q, K = torch.zeros(1, 8, 128).half(), torch.zeros(1, 2, 16, 128).half()
    calls = [
        lambda: ops.gemv(h, W), lambda: ops.gemv(h.float(), W), lambda: ops.gemv(h[None], W),
        lambda: ops.gemv(h, W[:, :32]), lambda: ops.gemv(h, W, w_scale=g),
        lambda: ops.gemv(h, W.to(torch.float8_e4m3fn)), lambda: ops.gemv([1.0], W),
        lambda: ops.gemv(None, W), lambda: ops.f1_rmsnorm_gemv(h, g, W),
        lambda: ops.f1_rmsnorm_gemv(h, g[:8], W), lambda: ops.f1_rmsnorm_gemv(h, g, W, "x"),
        lambda: ops.f2_gateup_swiglu(h, W, W[:4]), lambda: ops.f2_gateup_swiglu(h, W, W.float()),
        lambda: ops.f2_rmsnorm_gateup_swiglu(h, g, W, W), lambda: ops.f4_flashdecode(q, K, K),
        lambda: ops.f4_flashdecode(q, K, K[:, :, :8]), lambda: ops.f4_flashdecode(q[0], K, K),
    ]
    for fn in calls:
        fast, slow = _outcome(fn), _outcome(lambda fn=fn: steps(fn))
        assert isinstance(fast, tuple) and fast == slow


def test_a_module_built_for_another_torch_is_not_used(monkeypatch):
    """Its symbols may resolve all the same; its object layouts need not fit."""
    _load()
    from decodebench_amd import build

    assert not build._fast_stale()
    monkeypatch.setattr(ops, "_fast", None)
    monkeypatch.setattr(torch, "__version__", "0.0")
    ops._load_fast(ops.load_library())
    assert ops._fast is None and build._fast_stale()


def test_the_library_is_built_where_the_call_path_is_not(monkeypatch, tmp_path):
    """No g++, headers or torch: a warning, the library, and no stale module."""
    from decodebench_amd import build

    lib, old = tmp_path / "lib.so", tmp_path / "_fastcall.so"
    lib.write_bytes(b"linked")
    old.write_bytes(b"stale")

    def no_compiler(cmd, **kw):
        raise FileNotFoundError(cmd[0])

    monkeypatch.setattr(build, "_sources", list)
    monkeypatch.setattr(build, "LIB", lib)
    monkeypatch.setattr(build, "FAST_LIB", old)
    monkeypatch.setattr(build.subprocess, "run", no_compiler)
    with pytest.warns(UserWarning, match="native call path"):
        assert build.build(verbose=False) == lib
    assert not old.exists()


def _inputs():
    gen = torch.Generator(device="cuda").manual_seed(3)

    def rn(*s, std=1.0):
        return (torch.randn(*s, generator=gen, device="cuda") * std).half()

    x, g = rn(3, 256), rn(256)
    W, W2 = rn(96, 256, std=0.1), rn(96, 256, std=0.1)
    (Q, s), (Q2, s2) = quantize_e4m3_rows(W), quantize_e4m3_rows(W2)
    q, K, V = rn(2, 8, 128), rn(2, 2, 700, 128), rn(2, 2, 700, 128)
    return x, g, W, W2, Q, s, Q2, s2, q, K, V


@pytest.mark.gpu
def test_results_and_refusals_match_on_the_gpu(steps):
    _load()
    x, g, W, W2, Q, s, Q2, s2, q, K, V = _inputs()
    B8 = Q.view(torch.uint8)
    xg = x.clone().requires_grad_()
    wide = torch.zeros(3, 512, dtype=torch.float16, device="cuda")
    accepted = [
        lambda: ops.gemv(x, W), lambda: ops.gemv(x[0], W), lambda: ops.gemv(x, Q, w_scale=s),
        lambda: ops.gemv(x, B8, w_scale=s), lambda: ops.gemv(xg, W),
        lambda: ops.gemv(torch.nn.Parameter(x), W), lambda: ops.gemv(x.as_subclass(_Sub), W),
        lambda: ops.gemv(x, W, out=torch.empty(3, 96, dtype=torch.float16, device="cuda")),
        lambda: ops.f1_rmsnorm_gemv(x, g, W), lambda: ops.f1_rmsnorm_gemv(x, g, W, 0),
        lambda: ops.f1_rmsnorm_gemv(x[0], g, Q, 1e-5, w_scale=s),
        lambda: ops.f2_gateup_swiglu(x, W, W2), lambda: ops.f2_gateup_swiglu(x, Q, Q2, s, s2),
        lambda: ops.f2_rmsnorm_gateup_swiglu(x, g, W, W2),
        lambda: ops.f2_rmsnorm_gateup_swiglu(x[0], g, Q, Q2, sg=s, su=s2),
        lambda: ops.f4_flashdecode(q, K, V), lambda: ops.f4_flashdecode(q, K, V, scale=1),
        lambda: ops.f4_flashdecode(q, K, V, scale=0.05, n_splits=1),
        lambda: ops.f4_flashdecode(q, K, V, n_splits=3), lambda: ops.f4_flashdecode(q, K, V),
    ]
    for i, fn in enumerate(accepted):
        print(f"[fastcall] accepted {i}", flush=True)
        a, b = fn(), steps(fn)
        assert type(a) is type(b) and a.shape == b.shape and a.dtype == b.dtype
        assert a.requires_grad == b.requires_grad and torch.equal(a, b)
    refused = [
        lambda: ops.gemv(wide[:, ::2], W), lambda: ops.gemv(x, W.t()),
        lambda: ops.gemv(x, W, w_scale=s), lambda: ops.gemv(x, Q, w_scale=s[:5]),
        lambda: ops.gemv(x, Q, w_scale=s.double()), lambda: ops.gemv(x, Q, w_scale=s.cpu()),
        lambda: ops.gemv(x.cpu(), W), lambda: ops.gemv(x, W.cpu()),
        lambda: ops.gemv(x[:0], W), lambda: ops.gemv(x[:, :250].contiguous(), W[:, :250].contiguous()),
        lambda: ops.gemv(wide.view(-1)[1:769].view(3, 256), W),
        lambda: ops.f1_rmsnorm_gemv(x, g, W, -1.0), lambda: ops.f1_rmsnorm_gemv(x, g, W, math.nan),
        lambda: ops.f1_rmsnorm_gemv(x, g.cpu(), W), lambda: ops.f2_gateup_swiglu(x, W, Q2, None, s2),
        lambda: ops.f4_flashdecode(q, K, V, n_splits=0),
        lambda: ops.f4_flashdecode(q, K, V, n_splits=257),
        lambda: ops.f4_flashdecode(q, K, V, scale=math.inf),
        lambda: ops.f4_flashdecode(q[:, :6].contiguous(), K, V),
        lambda: ops.f4_flashdecode(q[..., :64].contiguous(), K[..., :64].contiguous(),
                                   V[..., :64].contiguous()),
    ]
    for i, fn in enumerate(refused):
        print(f"[fastcall] refused {i}", flush=True)
        a, b = _outcome(fn), _outcome(lambda fn=fn: steps(fn))
        assert isinstance(a, tuple) and a == b, (i, a, b)


@pytest.mark.gpu
def test_streams_threads_and_capture():
    """Calls on several streams and threads at once, and a captured call (its
    own workspace, not the stream's cached one), give the plain result."""
    import threading

    _load()
    x, g, W, W2, Q, s, Q2, s2, q, K, V = _inputs()
    ref, att = ops.gemv(x, W), ops.f4_flashdecode(q, K, V, n_splits=5)
    torch.cuda.synchronize()
    bad = []

    def work():
        st = torch.cuda.Stream()
        with torch.cuda.stream(st):
            for _ in range(50):
                y, o = ops.gemv(x, W), ops.f4_flashdecode(q, K, V, n_splits=5)
            st.synchronize()
        if not (torch.equal(y, ref) and torch.equal(o, att)):
            bad.append(1)

    ts = [threading.Thread(target=work) for _ in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not bad
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        ops.f4_flashdecode(q, K, V, n_splits=5)
    before = len(ops._captured_ws)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        o = ops.f4_flashdecode(q, K, V, n_splits=5)
        y = ops.f1_rmsnorm_gemv(x, g, W)
    assert len(ops._captured_ws) == before + 1
    for _ in range(4):
        eager = ops.f1_rmsnorm_gemv(x, g, W)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, att) and torch.equal(y, eager)
    del graph
    ops.release_captured_workspaces()
