"""The streamed tile GEMV (gemv_tile) at the edges of its tiles.

Every case forces the kernel and compares with fp64 products of the same
fp16 inputs.  The bound is derived per output, from the fp16 roundings
(2^-11 each) and the fp32 sums:

* one matrix: 2^-11 |y| for the output, (2^-11 + K 2^-23) sum_k |w p| for the
  rounded operands (norm modes) and the sums;
* gate/up: that error on gate and up, their own fp16 rounding, carried through
  silu(g) u (|silu'| <= 1.1), and the roundings of silu and of the product.
"""

import pytest

torch = pytest.importorskip("torch")

from decodebench_amd import ops  # noqa: E402
from decodebench_amd.quant import dequantize_e4m3_rows, quantize_e4m3_rows  # noqa: E402

pytestmark = pytest.mark.gpu

U = 2.0 ** -11   # fp16 rounding
TINY = 2.0 ** -24


@pytest.fixture(autouse=True)
def _force_tile():
    ops.tune("gemv_tile", 1)
    yield
    ops.tune("gemv_tile", 0)


def _randn(gen, *shape, std=1.0, mean=0.0):
    t = torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)
    return (t * std + mean).half()


def _call(mode, x, g, W, s):
    if mode == "gemv":
        return ops.gemv(x, W[0], w_scale=s[0])
    if mode == "f1":
        return ops.f1_rmsnorm_gemv(x, g, W[0], w_scale=s[0])
    if mode == "f2":
        return ops.f2_gateup_swiglu(x, W[0], W[1], s[0], s[1])
    return ops.f2_rmsnorm_gateup_swiglu(x, g, W[0], W[1], sg=s[0], su=s[1])


def _check(mode, x, g, W, s, W64):
    norm = mode in ("f1", "f2n")
    K = x.shape[1]
    p = x.double()
    if norm:
        p = p * torch.rsqrt(p.square().mean(-1, keepdim=True) + 1e-6) * g.double()

    def linear(w):
        wt = w.t().contiguous()
        return p @ wt, ((U if norm else 0.0) + K * 2.0 ** -23) * (p.abs() @ wt.abs())

    y = _call(mode, x, g, W, s).double()
    a, da = linear(W64[0])
    if mode in ("gemv", "f1"):
        ref, bound = a, da + U * a.abs()
    else:
        u, du = linear(W64[1])
        da, du = da + U * a.abs(), du + U * u.abs()
        sil = a * torch.sigmoid(a)
        ref = sil * u
        bound = 1.1 * da * (u.abs() + du) + sil.abs() * du + 3 * U * ref.abs()
    # 1.01: the bound's own second-order terms
    bad = (y - ref).abs() > 1.01 * bound + 2 * TINY
    assert torch.isfinite(y).all()
    assert not bad.any(), f"{int(bad.sum())} outputs outside the bound, worst " \
                          f"{((y - ref).abs() / (bound + TINY)).max().item():.2f} of it"


def _weights(gen, n, N, K, dtype):
    W, s, W64 = [], [], []
    for _ in range(n):
        w = _randn(gen, N, K, std=K ** -0.5)
        if dtype == "fp8":
            w, sc = quantize_e4m3_rows(w)
            W64.append(dequantize_e4m3_rows(w, sc).double())
        else:
            sc = None
            W64.append(w.double())
        W.append(w)
        s.append(sc)
    return W, s, W64


# Batch rows at the edges of the 8-row groups and the 64-row pass; K below one
# block, at its edges and with 1 to 9 blocks per wave; N at the edges of the
# 4-row shares and of every tile count (256 workgroups x 16 rows, 8 outputs for
# the pair), and above what 8 tiles hold.
CASES = [
    ("gemv", "f16", 2, 8, 1), ("f1", "f16", 3, 16, 3), ("f2", "f16", 9, 64, 5),
    ("f2n", "f16", 16, 72, 1023), ("gemv", "fp8", 7, 16, 1), ("f1", "fp8", 8, 128, 1025),
    ("f2", "fp8", 17, 144, 4), ("f2n", "fp8", 24, 112, 1030),
    ("gemv", "f16", 25, 3000, 2052), ("f1", "f16", 32, 2568, 4097), ("f1", "fp8", 33, 2576, 4095),
    ("gemv", "fp8", 48, 4608, 1500), ("f2", "f16", 49, 1000, 2049), ("f2n", "fp8", 64, 1040, 2047),
    ("f1", "f16", 65, 520, 515), ("gemv", "fp8", 130, 528, 4100),
    ("gemv", "f16", 5, 200, 28673), ("gemv", "f16", 64, 136, 20481), ("f1", "fp8", 41, 272, 24577),
    ("gemv", "f16", 12, 64, 33000), ("f2", "f16", 6, 328, 14337), ("f2", "fp8", 64, 192, 12289),
    ("f2n", "f16", 40, 264, 10241), ("f2n", "fp8", 4, 272, 8193), ("f2", "f16", 20, 64, 16500),
]


@pytest.mark.parametrize("mode,dtype,B,K,N", CASES)
def test_tile_edges(mode, dtype, B, K, N):
    print(f"[tile] {mode} {dtype} B={B} K={K} N={N}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(B * 7919 + K + N)
    x = _randn(gen, B, K)
    g = _randn(gen, K, std=0.1, mean=1.0)
    _check(mode, x, g, *_weights(gen, 2 if mode in ("f2", "f2n") else 1, N, K, dtype))


@pytest.mark.parametrize("dtype", ["f16", "fp8"])
@pytest.mark.parametrize("rows", ["tiny", "large", "mixed", "late", "early", "zero"])
def test_tile_norm_keeps_precision_over_the_fp16_range(rows, dtype):
    """x whose products with gamma leave fp16 (tiny, large, a row of each), or
    whose first columns do not say so (late: 3e4 after columns of 1e-3; early:
    the other way round), and rows of zeros."""
    print(f"[tile-norm] {rows} {dtype}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(5)
    B, K, N = 12, 1536, 300
    # a few ulps wide, so that tiny values keep their relative precision
    x = (_randn(gen, B, K).sign().float() * (1 + 0.5 * torch.rand(B, K, generator=gen,
                                                                  device="cuda")))
    scale = torch.ones(B, K, device="cuda")
    if rows == "tiny":
        scale *= 2.0 ** -13
    elif rows == "large":
        scale *= 2.0 ** 14
    elif rows == "mixed":
        scale[::2] *= 2.0 ** -12
        scale[1::2] *= 2.0 ** 14
    elif rows == "late":
        scale *= 2.0 ** -10
        scale[:, K // 2:] = 2.0 ** 14
    elif rows == "early":
        scale *= 2.0 ** 14
        scale[:, K // 2:] = 2.0 ** -3
    x = (x * scale).half()
    if rows == "zero":
        x[3:9] = 0
    g = _randn(gen, K, std=1.0, mean=16.0)
    _check("f1", x, g, *_weights(gen, 1, N, K, dtype))


# Rows at both numbers of 8-row groups per 16-row tile; outputs for 8 waves of
# one tile and 4 of more.
NORM_CASES = [("f1", "f16", 4, 5120, 300), ("f1", "f16", 20, 3072, 4500),
              ("f1", "fp8", 4, 3072, 300), ("f1", "fp8", 8, 8192, 4500),
              ("f1", "fp8", 12, 3072, 300), ("f1", "fp8", 24, 3072, 4500),
              ("f2n", "f16", 24, 4096, 300), ("f2n", "fp8", 8, 3072, 2500),
              ("f2n", "fp8", 20, 4096, 2500)]


@pytest.mark.parametrize("mode,dtype,B,K,N", NORM_CASES)
def test_tile_norm_where_a_wave_scales_its_rows(mode, dtype, B, K, N):
    """x around the mean squares at which a wave scales its rows, where its
    first block says one thing and its columns another."""
    gen = torch.Generator(device="cuda").manual_seed(B + K)
    g = _randn(gen, K, std=0.1, mean=1.0)
    weights = _weights(gen, 2 if mode == "f2n" else 1, N, K, dtype)
    for std in (0.1, 0.12, 0.13, 0.14, 0.25, 100.0, 128.0, 200.0):
        print(f"[tile-scale] {mode} {dtype} B={B} K={K} N={N} std={std}", flush=True)
        _check(mode, _randn(gen, B, K, std=std), g, *weights)


@pytest.mark.parametrize("mode,dtype,B,K,N", NORM_CASES)
def test_tile_norm_where_one_block_is_unlike_the_others(mode, dtype, B, K, N):
    """One block of columns far below or above the rest, at the first place, in
    the middle and at the last: the block that some workgroup's wave starts at."""
    gen = torch.Generator(device="cuda").manual_seed(B + K)
    g = _randn(gen, K, std=0.1, mean=1.0)
    weights = _weights(gen, 2 if mode == "f2n" else 1, N, K, dtype)
    kb = 64 if dtype == "f16" else 128
    for block in (0, K // kb // 2, K // kb - 1):
        for e in (-12, -9, 9):
            print(f"[tile-block] {mode} {dtype} B={B} K={K} N={N} block={block} e={e}", flush=True)
            x = _randn(gen, B, K).float()
            x[:, block * kb:(block + 1) * kb] *= 2.0 ** e
            _check(mode, x.half(), g, *weights)


@pytest.mark.parametrize("dtype", ["f16", "fp8"])
@pytest.mark.parametrize("B", [4, 12])
def test_tile_norm_where_one_product_leaves_fp16(B, dtype):
    """Rows of ordinary mean square with one value whose product with gamma
    overflows fp16, at the first columns, in the middle and at the last."""
    gen = torch.Generator(device="cuda").manual_seed(B)
    K, N = 5120, 4500
    g = _randn(gen, K, std=1.0, mean=24.0)
    weights = _weights(gen, 1, N, K, dtype)
    for col in (3, K // 2 + 9, K - 1):
        print(f"[tile-product] {dtype} B={B} col={col}", flush=True)
        x = _randn(gen, B, K, std=60.0)
        x[:, col] = 3000.0
        _check("f1", x, g, *weights)


@pytest.mark.parametrize("dtype", ["f16", "fp8"])
@pytest.mark.parametrize("std", [0.126, 0.25, 1.0])
def test_tile_norm_keeps_precision_under_a_small_gamma(std, dtype):
    """gamma of 2^-13: its product with a normalised row, of which fp16 keeps 11
    bits, less what the subnormals below 2^-14 lose.  Relative error, of the
    2-norms: 2^-11 x 0.41 for each of two roundings (the mean over a binade),
    2^-24 / sqrt(12) of 2^-13 for the subnormals: 3.2e-4; 4.5e-4 allows for the
    stage's third rounding.  Without a scale x of 0.25 gives 5.9e-4."""
    print(f"[tile-gamma] std={std} {dtype}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(6)
    B, K, N = 12, 3072, 1000
    x = _randn(gen, B, K, std=std)
    g = ((torch.randn(K, generator=gen, device="cuda") * 0.1 + 1) * 2.0 ** -13).half()
    w = _randn(gen, N, K, std=8 * K ** -0.5)
    w, s = quantize_e4m3_rows(w) if dtype == "fp8" else (w, None)
    w64 = (dequantize_e4m3_rows(w, s) if dtype == "fp8" else w).double()
    p = x.double()
    p = p * torch.rsqrt(p.square().mean(-1, keepdim=True) + 1e-6) * g.double()
    ref = p @ w64.t().contiguous()
    err = (ops.f1_rmsnorm_gemv(x, g, w, w_scale=s).double() - ref).norm() / ref.norm()
    assert err <= 4.5e-4, f"{err.item():.2e}"


@pytest.mark.parametrize("dtype,B,K,N", [("f16", 17, 2048, 700), ("fp8", 24, 4096, 333),
                                         ("f16", 49, 4096, 500), ("fp8", 64, 2048, 512)])
def test_pair_passes_keep_precision_over_the_fp16_range(dtype, B, K, N):
    """RMSNorm -> gate/up of few outputs above 16 rows, which the 16-row passes
    take: x at every scale, one block unlike the others, one product of gamma
    that leaves fp16, rows of zeros, and gamma of 2^-13."""
    gen = torch.Generator(device="cuda").manual_seed(B + K)
    ops.tune("gemv_tile", 0)
    weights = _weights(gen, 2, N, K, dtype)
    g = _randn(gen, K, std=0.1, mean=1.0)
    for std in (2.0 ** -13, 1e-3, 0.12, 0.24, 0.26, 1.0, 3.9, 4.1, 200.0, 1.2e4):
        print(f"[pass-range] {dtype} B={B} K={K} N={N} std={std}", flush=True)
        x = _randn(gen, B, K).sign() * (1 + 0.5 * torch.rand(B, K, generator=gen, device="cuda"))
        _check("f2n", (x * std).half(), g, *weights)
    for e in (-12, 9):
        x = _randn(gen, B, K).float()
        x[:, K // 2:K // 2 + 256] *= 2.0 ** e
        x[3] = 0
        _check("f2n", x.half(), g, *weights)
    x = _randn(gen, B, K, std=60.0)
    x[:, 9] = 3000.0
    _check("f2n", x, _randn(gen, K, std=1.0, mean=24.0), *weights)
    _check("f2n", _randn(gen, B, K, std=0.3), (g.float() * 2.0 ** -13).half(), *weights)


# K split over workgroups: counts that divide the blocks and that do not, a
# last split of one block, outputs that no quad or tile divides, more rows
# than a pass, every mode and weight type.
SPLIT_CASES = [
    ("gemv", "f16", 9, 520, 1000, 2), ("gemv", "fp8", 17, 2064, 1023, 4),
    ("f1", "f16", 24, 1336, 517, 3), ("f1", "fp8", 64, 4112, 2050, 8),
    ("f2", "f16", 41, 1000, 700, 3), ("f2", "fp8", 12, 3088, 333, 4),
    ("f2n", "f16", 16, 2600, 1021, 2), ("f2n", "fp8", 33, 4624, 512, 5),
    ("gemv", "f16", 70, 3000, 4097, 4), ("f1", "f16", 130, 520, 260, 2),
]


@pytest.mark.parametrize("mode,dtype,B,K,N,S", SPLIT_CASES)
def test_tile_splits(mode, dtype, B, K, N, S):
    print(f"[tile-split] {mode} {dtype} B={B} K={K} N={N} S={S}", flush=True)
    lib = ops.load_library()
    gen = torch.Generator(device="cuda").manual_seed(B * 7919 + K + N)
    x = _randn(gen, B, K)
    g = _randn(gen, K, std=0.1, mean=1.0)
    weights = _weights(gen, 2 if mode in ("f2", "f2n") else 1, N, K, dtype)
    ops.tune("gemv_splits", S)
    try:
        assert lib.db_gemv_workspace_bytes(mode in ("f1", "f2n"), mode in ("f2", "f2n"), B, K, N,
                                           dtype == "fp8") > 0
        _check(mode, x, g, *weights)
        # a call that brings its output takes one launch and allocates nothing
        if mode == "gemv":
            out = torch.empty(B, N, dtype=torch.float16, device="cuda")
            held = torch.cuda.memory_stats()["allocation.all.allocated"]
            ops.gemv(x, weights[0][0], w_scale=weights[1][0], out=out)
            assert torch.cuda.memory_stats()["allocation.all.allocated"] == held
            y = ops.gemv(x, weights[0][0], w_scale=weights[1][0])
            assert (y.double() - out.double()).norm() <= 1e-3 * out.double().norm()
    finally:
        ops.tune("gemv_splits", 0)


def test_tile_splits_capture_and_streams():
    """Split calls captured into a graph (their workspaces come from its pool)
    and on two streams at once."""
    gen = torch.Generator(device="cuda").manual_seed(9)
    x = _randn(gen, 20, 4096)
    W = [_randn(gen, 1000, 4096, std=1 / 64) for _ in range(3)]
    ops.tune("gemv_splits", 4)
    try:
        ref = [ops.gemv(x, w) for w in W]
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            ys = [ops.gemv(x, w) for w in W]
        streams = [torch.cuda.Stream() for _ in range(2)]
        for _ in range(4):
            for st in streams:
                st.wait_stream(torch.cuda.current_stream())
            graph.replay()
            side = []
            for st in streams:
                with torch.cuda.stream(st):
                    side.append([ops.gemv(x, w) for w in W])
            torch.cuda.synchronize()
            for got in (ys, *side):
                assert all(torch.equal(a, b) for a, b in zip(got, ref))
    finally:
        ops.tune("gemv_splits", 0)


@pytest.mark.parametrize("dtype,B,K,N", [("fp8", 49, 8192, 4096), ("fp8", 64, 6144, 2057),
                                         ("f16", 65, 8192, 260), ("fp8", 129, 10240, 1000)])
def test_long_rows_of_many_batch_rows_take_the_tile_kernel(dtype, B, K, N):
    """Into a given output (one launch): the bits of the forced tile kernel."""
    print(f"[tile-long] {dtype} B={B} K={K} N={N}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(B * 7919 + K + N)
    x = _randn(gen, B, K)
    W, s, W64 = _weights(gen, 1, N, K, dtype)
    out = [torch.empty(B, N, dtype=torch.float16, device="cuda") for _ in range(2)]
    ops.gemv(x, W[0], w_scale=s[0], out=out[0])
    ops.tune("gemv_tile", 0)
    ops.gemv(x, W[0], w_scale=s[0], out=out[1])
    assert torch.equal(*out)
    _check("gemv", x, None, W, s, W64)


@pytest.mark.parametrize("knob,value", [("gemv_tile", 2), ("gemv_long_kc", 2),
                                        ("gemv_long_gpw", 1), ("gemv_long_stage", 2)])
@pytest.mark.parametrize("dtype", ["f16", "fp8"])
def test_knobs_that_bar_the_tile_kernel_bar_its_splits(knob, value, dtype):
    """Long plain rows that would split K: with the knob they get no workspace
    and run the launch that a call with its own output runs."""
    print(f"[tile-knob] {knob}={value} {dtype}", flush=True)
    lib = ops.load_library()
    gen = torch.Generator(device="cuda").manual_seed(11)
    B, K, N = 32, 14336, 1000
    x = _randn(gen, B, K)
    W, s, W64 = _weights(gen, 1, N, K, dtype)
    ops.tune("gemv_tile", 0)
    assert lib.db_gemv_workspace_bytes(0, 0, B, K, N, dtype == "fp8") > 0
    try:
        ops.tune(knob, value)
        assert lib.db_gemv_workspace_bytes(0, 0, B, K, N, dtype == "fp8") == 0
        out = torch.empty(B, N, dtype=torch.float16, device="cuda")
        ops.gemv(x, W[0], w_scale=s[0], out=out)
        assert torch.equal(ops.gemv(x, W[0], w_scale=s[0]), out)
        _check("gemv", x, None, W, s, W64)
    finally:
        ops.tune(knob, 0)


def test_split_workspace_is_bounded_at_any_batch():
    """One round of workgroups: 256 of up to 8 tiles of 16 outputs, 64 batch
    rows and 4 bytes, 8 MB, and the sums of x^2 (8 splits x 4 bytes a row)."""
    lib = ops.load_library()
    ops.tune("gemv_tile", 0)
    split = 0
    for B in (9, 40, 64, 65, 128, 129, 256, 600, 8192, 65536):
        for K in (3072, 4096, 5120, 8192, 14336):
            for N in (512, 1024, 3000, 4096, 5120, 14336):
                for norm, pair in ((0, 0), (1, 0), (0, 1), (1, 1)):
                    for dt in (0, 1):
                        n = lib.db_gemv_workspace_bytes(norm, pair, B, K, N, dt)
                        assert n <= (8 << 20) + 32 * B, (B, K, N, norm, pair, dt)
                        split += n > 0
    assert split > 0


# More rows than a pass: splits of one round of workgroups, shapes that would
# take two rounds (no splits), and long rows that no longer split.  Up to one:
# two passes side by side that read as little of x (no splits).
@pytest.mark.parametrize("mode,dtype,B,K,N,split", [
    ("gemv", "fp8", 49, 3072, 2432, False), ("f1", "f16", 51, 3072, 1280, False),
    ("gemv", "f16", 41, 11008, 4096, True), ("gemv", "fp8", 28, 6144, 1408, True),
    ("gemv", "f16", 65, 11008, 2050, True), ("gemv", "fp8", 129, 14336, 1024, True),
    ("f1", "f16", 100, 8192, 2047, True), ("f2n", "f16", 130, 8192, 1021, True),
    ("gemv", "f16", 65, 4096, 4096, False), ("gemv", "fp8", 200, 8192, 4095, False),
    ("f2", "f16", 129, 8192, 2048, False), ("gemv", "f16", 257, 6144, 2040, False),
])
def test_automatic_splits(mode, dtype, B, K, N, split):
    print(f"[tile-rows] {mode} {dtype} B={B} K={K} N={N}", flush=True)
    lib = ops.load_library()
    ops.tune("gemv_tile", 0)
    assert (lib.db_gemv_workspace_bytes(mode in ("f1", "f2n"), mode in ("f2", "f2n"), B, K, N,
                                        dtype == "fp8") > 0) == split
    gen = torch.Generator(device="cuda").manual_seed(B * 7919 + K + N)
    x = _randn(gen, B, K)
    g = _randn(gen, K, std=0.1, mean=1.0)
    _check(mode, x, g, *_weights(gen, 2 if mode in ("f2", "f2n") else 1, N, K, dtype))


def test_split_call_without_room_for_its_workspace_takes_one_launch(monkeypatch):
    """Memory for the output but not for the partial sums: the call still
    answers, through either call path."""
    ops.tune("gemv_tile", 0)
    B, K, N = 40, 11008, 4096
    gen = torch.Generator(device="cuda").manual_seed(2)
    x, W = _randn(gen, B, K), _randn(gen, N, K, std=K ** -0.5)
    nbytes = ops.load_library().db_gemv_workspace_bytes(0, 0, B, K, N, 0)
    assert nbytes > 1 << 20
    ref = ops.gemv(x, W, out=torch.empty(B, N, dtype=torch.float16, device="cuda"))
    assert not torch.equal(ops.gemv(x, W), ref)  # split, with memory
    total = torch.cuda.get_device_properties(0).total_memory
    for fast in (ops._fast, None):
        monkeypatch.setattr(ops, "_fast", fast)
        y = torch.empty(B, N, dtype=torch.float16, device="cuda")
        torch.cuda.empty_cache()
        torch.cuda.set_per_process_memory_fraction(
            (torch.cuda.memory_reserved() + (1 << 20)) / total)
        full = []
        try:
            with pytest.raises(torch.cuda.OutOfMemoryError):
                while True:  # every block that the workspace would fit in
                    full.append(torch.empty(nbytes, dtype=torch.uint8, device="cuda"))
            del y  # room for the output
            y = ops.gemv(x, W)
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        assert torch.equal(y, ref)


# Widths of no other MFMA kernel: both sides of the lines at which fp16 without
# the norm stays on the VALU kernel, by row alignment (2 rows) and by outputs,
# length and batch.
@pytest.mark.parametrize("mode,dtype,B,K,N,tile", [
    ("gemv", "f16", 2, 5136, 8001, False), ("gemv", "f16", 2, 5184, 8001, True),
    ("gemv", "fp8", 2, 5136, 8001, True), ("f2n", "f16", 2, 3088, 8001, True),
    ("gemv", "f16", 8, 11008, 1023, False), ("gemv", "f16", 8, 11008, 1024, True),
    ("f2", "f16", 7, 6160, 512, False), ("f2", "f16", 7, 6160, 513, True),
    ("gemv", "f16", 9, 6208, 1000, True), ("gemv", "f16", 16, 10112, 256, False),
    ("gemv", "f16", 17, 10112, 256, True), ("f1", "f16", 8, 11008, 512, True),
])
def test_fp16_calls_that_stay_on_the_valu_kernel(mode, dtype, B, K, N, tile):
    print(f"[tile-valu] {mode} {dtype} B={B} K={K} N={N}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(B * 7919 + K + N)
    x = _randn(gen, B, K)
    g = _randn(gen, K, std=0.1, mean=1.0)
    W, s, W64 = _weights(gen, 2 if mode in ("f2", "f2n") else 1, N, K, dtype)
    ops.tune("gemv_splits", 1)
    try:
        got = {}
        for knob in (0, 1, 2):
            ops.tune("gemv_tile", knob)
            got[knob] = _call(mode, x, g, W, s)
        assert torch.equal(got[0], got[1 if tile else 2])
        assert not torch.equal(got[1], got[2])
        ops.tune("gemv_tile", 0)
        _check(mode, x, g, W, s, W64)
    finally:
        ops.tune("gemv_splits", 0)


# Both sides of the lines at which the gate/up pair leaves the 16-row passes:
# 256 workgroups of 8 outputs and 16 rows, and the batch.
@pytest.mark.parametrize("mode,dtype,B,K,N,tile", [
    ("f2n", "fp8", 17, 4096, 1024, False), ("f2n", "fp8", 17, 4096, 1025, True),
    ("f2n", "f16", 49, 2048, 512, False), ("f2n", "f16", 49, 2048, 513, True),
    ("f2", "f16", 49, 2048, 512, False), ("f2", "f16", 49, 2048, 513, True),
    ("f2", "fp8", 32, 2048, 680, True), ("f2", "fp8", 33, 2048, 680, False),
    ("f2", "f16", 48, 4096, 512, True), ("f2", "f16", 49, 4096, 512, False),
])
def test_pair_of_few_outputs_keeps_its_passes(mode, dtype, B, K, N, tile):
    print(f"[tile-few] {mode} {dtype} B={B} K={K} N={N}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(B * 7919 + K + N)
    x = _randn(gen, B, K)
    g = _randn(gen, K, std=0.1, mean=1.0)
    W, s, W64 = _weights(gen, 2, N, K, dtype)
    ops.tune("gemv_splits", 1)  # one launch, as with a given output
    try:
        got = {}
        for knob in (0, 1, 2):
            ops.tune("gemv_tile", knob)
            got[knob] = _call(mode, x, g, W, s)
        assert torch.equal(got[0], got[1 if tile else 2])
        assert not torch.equal(got[1], got[2])
        ops.tune("gemv_tile", 0)
        _check(mode, x, g, W, s, W64)
    finally:
        ops.tune("gemv_splits", 0)
