"""Parity of the HIP kernels (through the C ABI) with the CPU oracle.

Bar (the benchmark's parity target): outputs within rtol 1e-2 / atol 1e-2 of the
reference's PyTorch stage definitions (oracle/stages.py, run on CPU with the
same seeded fp16 inputs).  Because atol 1e-2 is weak where outputs are small
(F4 at long context), every case also checks the relative L2 error against
the exact fp64 oracle (oracle/cref.c):
    F1, F2   rel-L2 <= 2e-3   (fp16 output rounding is ~3e-4)
    F4       rel-L2 <= 5e-3
Full-size cases whose CPU oracle would be slow use size-independent
properties instead: split count invariance and agreement of batch rows with
single-row launches.
"""

import functools
import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from decodebench_amd import ops  # noqa: E402
from oracle import cref, stages  # noqa: E402

pytestmark = pytest.mark.gpu

RTOL = ATOL = 1e-2
CHAIN_TOL = 2e-2     # the decode-layer chain (see test_decode_layer_chain_parity)
F12_REL_L2 = 2e-3
F4_REL_L2 = 5e-3


def rel_l2(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def randn(gen, shape, std=1.0, mean=0.0):
    t = torch.randn(*shape, generator=gen, dtype=torch.float32)
    return (t * std + mean).half()


def assert_parity(got, stage_ref, exact, rel_bound, what, tol=RTOL):
    got = got.detach().float().cpu().numpy().astype(np.float64)
    ref = stage_ref.float().numpy().astype(np.float64)
    assert np.isfinite(got).all(), f"{what}: non-finite output"
    bad = ~np.isclose(got, ref, rtol=tol, atol=tol)
    assert not bad.any(), (f"{what}: {bad.sum()} elements outside rtol/atol {tol}; "
                           f"max abs err {np.abs(got - ref).max():.3e}")
    err = rel_l2(got, exact)
    assert err <= rel_bound, f"{what}: rel-L2 {err:.3e} > {rel_bound}"


@pytest.fixture(scope="module", autouse=True)
def _lib():
    ops.load_library()
    cref.load()
    torch.manual_seed(0)


# ------------------------------------------------------------------- F1
F1_CASES = [
    (1, 256, 64, 0.05), (2, 512, 100, 0.05), (3, 1024, 33, 0.05), (1, 4104, 17, 0.02),
    (1, 4096, 4096, 1 / 64), (1, 4096, 6144, 0.02), (4, 4096, 6144, 0.02),
    (8, 4096, 6144, 0.02), (5, 4096, 512, 0.02), (16, 4096, 1024, 0.02),
    (1, 14336, 4096, 0.01),
    # config 3 (fused QKV, W [6144, 4096]) at the batch sizes of its sweep that take the MFMA
    # kernel's 16-row and 32-row passes
    (16, 4096, 6144, 0.02), (32, 4096, 6144, 0.02),
    # one batch row: 2 rows per wave where (N + 15) / 16 fills every CU with whole 8-wave
    # workgroups (K = 2048, and N = 4095 with a half-empty last group), else 1
    (1, 2048, 8192, 0.02), (1, 4096, 4095, 1 / 64),
]


@pytest.mark.parametrize("B,K,N,w_std", F1_CASES)
def test_f1_rmsnorm_gemv_parity(B, K, N, w_std):
    print(f"[f1] B={B} K={K} N={N}", flush=True)
    gen = torch.Generator().manual_seed(1000 + B + K + N)
    x = randn(gen, (B, K))
    g = randn(gen, (K,), std=0.1, mean=1.0)
    W = randn(gen, (N, K), std=w_std)
    y = ops.f1_rmsnorm_gemv(x.cuda(), g.cuda(), W.cuda(), eps=1e-6)
    torch.cuda.synchronize()
    assert y.shape == (B, N) and y.dtype == torch.float16
    ref = stages.f1(x, g, W, 1e-6)
    exact = cref.f1_exact(x.numpy(), g.numpy(), W.numpy(), 1e-6)
    assert_parity(y, ref, exact, F12_REL_L2, f"f1 B={B} K={K} N={N}")


def test_f1_one_dimensional_input_and_determinism():
    gen = torch.Generator().manual_seed(7)
    x = randn(gen, (4096,)).cuda()
    g = randn(gen, (4096,), std=0.1, mean=1.0).cuda()
    W = randn(gen, (4096, 4096), std=1 / 64).cuda()
    a = ops.f1_rmsnorm_gemv(x, g, W)
    b = ops.f1_rmsnorm_gemv(x.unsqueeze(0), g, W)[0]
    assert a.shape == (4096,)
    assert torch.equal(a, b)


# ------------------------------------------------------------------- F2
F2_CASES = [(1, 256, 96), (2, 1024, 300), (1, 4096, 14336), (4, 4096, 14336),
            (16, 4096, 2048), (3, 4096, 1000),
            # batch 1 with rows numbered by XCD in 32-row slices: a grid of a multiple
            # of 8 workgroups with N not a multiple of 256 (padded row groups), and a
            # grid that is not a multiple of 8 (launch order)
            (1, 4096, 2000), (1, 512, 16000), (1, 4096, 1004),
            # config 2 at B = 16: two batch tiles and alternating register sets on the
            # MFMA kernel at the full gate/up shape
            (16, 4096, 14336)]


@pytest.mark.parametrize("B,K,N", F2_CASES)
def test_f2_gateup_swiglu_parity(B, K, N):
    print(f"[f2] B={B} K={K} N={N}", flush=True)
    gen = torch.Generator().manual_seed(2000 + B + K + N)
    x = randn(gen, (B, K))
    Wg = randn(gen, (N, K), std=0.02)
    Wu = randn(gen, (N, K), std=0.02)
    y = ops.f2_gateup_swiglu(x.cuda(), Wg.cuda(), Wu.cuda())
    torch.cuda.synchronize()
    ref = stages.f2(x, Wg, Wu)
    exact = cref.f2_exact(x.numpy(), Wg.numpy(), Wu.numpy())
    assert_parity(y, ref, exact, 5e-3, f"f2 B={B} K={K} N={N}")


def test_plain_gemv_parity():
    gen = torch.Generator().manual_seed(3)
    x = randn(gen, (2, 14336), std=0.5)
    W = randn(gen, (4096, 14336), std=0.01)
    y = ops.gemv(x.cuda(), W.cuda())
    ref = stages.gemv(x, W)
    exact = cref.gemv_exact(x.numpy(), W.numpy())
    assert_parity(y, ref, exact, F12_REL_L2, "gemv 2x14336x4096")


# --------------------------------------------------- batched GEMV (MFMA)
# Batches from 3 rows (2 for the e4m3 gate/up pair) with K in
# {2048, 4096} take the MFMA kernel: ragged batches (one and two 16-row
# passes), N not a multiple of the 8-row group.
MFMA_CASES = [
    ("f1", 3, 4096, 1000), ("f1", 17, 4096, 6144), ("f1", 32, 2048, 1032),
    ("f2", 4, 4096, 14336), ("f2", 32, 4096, 1792), ("f2", 9, 2048, 777),
    ("plain", 16, 4096, 4100), ("plain", 3, 2048, 8), ("f2", 3, 4096, 1000),
    ("f2", 3, 2048, 515),
    # one matrix above 16 rows (16-row passes sharing the weights through an
    # XCD's L2): the QKV shape at B=32, ragged batches, three passes (B=40),
    # K=2048 with more groups
    ("f1", 32, 4096, 6144), ("plain", 24, 4096, 4096), ("f1", 21, 2048, 1000),
    ("plain", 40, 2048, 3000), ("plain", 32, 4096, 2040),
    # the norm at one batch tile with x staged through LDS: K=2048 (two rows
    # per load), a partial tile
    ("f1", 5, 2048, 520), ("f1", 8, 4096, 6144),
]


@pytest.mark.parametrize("mode,B,K,N", MFMA_CASES)
def test_batched_gemv_mfma_parity(mode, B, K, N):
    print(f"[mfma] {mode} B={B} K={K} N={N}", flush=True)
    gen = torch.Generator().manual_seed(4000 + B + K + N)
    x = randn(gen, (B, K))
    if mode == "f1":
        g = randn(gen, (K,), std=0.1, mean=1.0)
        W = randn(gen, (N, K), std=0.02)
        y = ops.f1_rmsnorm_gemv(x.cuda(), g.cuda(), W.cuda())
        ref, exact, bound = stages.f1(x, g, W), cref.f1_exact(x.numpy(), g.numpy(), W.numpy()), \
            F12_REL_L2
    elif mode == "f2":
        Wg = randn(gen, (N, K), std=0.02)
        Wu = randn(gen, (N, K), std=0.02)
        y = ops.f2_gateup_swiglu(x.cuda(), Wg.cuda(), Wu.cuda())
        ref, exact, bound = stages.f2(x, Wg, Wu), \
            cref.f2_exact(x.numpy(), Wg.numpy(), Wu.numpy()), 5e-3
    else:
        W = randn(gen, (N, K), std=0.02)
        y = ops.gemv(x.cuda(), W.cuda())
        ref, exact, bound = stages.gemv(x, W), cref.gemv_exact(x.numpy(), W.numpy()), F12_REL_L2
    torch.cuda.synchronize()
    assert y.shape == (B, N)
    assert_parity(y, ref, exact, bound, f"{mode} B={B} K={K} N={N}")


def test_mfma_and_valu_gemv_paths_agree():
    """The same batch through both kernels (the MFMA threshold raised to force
    the VALU path) differs only by fp32 summation order."""
    gen = torch.Generator().manual_seed(77)
    x = randn(gen, (8, 4096)).cuda()
    g = randn(gen, (4096,), std=0.1, mean=1.0).cuda()
    W = randn(gen, (6144, 4096), std=0.02).cuda()
    Wu = randn(gen, (6144, 4096), std=0.02).cuda()
    lib = ops.load_library()
    try:
        outs = []
        for thr in (2, 1 << 20):
            assert lib.db_tune(b"gemv_mfma_min_batch", thr) == 0
            outs.append((ops.f1_rmsnorm_gemv(x, g, W), ops.f2_gateup_swiglu(x, W, Wu),
                         ops.gemv(x, W)))
    finally:
        lib.db_tune(b"gemv_mfma_min_batch", 0)
    for a, b in zip(*outs):
        assert rel_l2(a.float().cpu().numpy(), b.float().cpu().numpy()) < 1e-3


def test_one_matrix_pass_shapes_agree():
    """One weight matrix above 16 rows: 16-row passes on the default split
    grid, on 8 to 256 workgroups per pass, and 32-row passes with rows 16..31
    of x in LDS (gemv_xb) agree to fp32 summation order, fp16 and e4m3, with
    and without the RMSNorm."""
    from decodebench_amd.quant import quantize_e4m3_rows

    gen = torch.Generator().manual_seed(81)
    lib = ops.load_library()
    try:
        for B, K, N in ((17, 4096, 6144), (32, 4096, 4096), (40, 2048, 1000), (64, 4096, 520)):
            print(f"[passes] B={B} K={K} N={N}", flush=True)
            x = randn(gen, (B, K)).cuda()
            g = randn(gen, (K,), std=0.1, mean=1.0).cuda()
            W = randn(gen, (N, K), std=0.02)
            Wq, s = (t.cuda() for t in quantize_e4m3_rows(W))
            W = W.cuda()

            def run():
                return (ops.f1_rmsnorm_gemv(x, g, W), ops.gemv(x, W),
                        ops.f1_rmsnorm_gemv(x, g, Wq, w_scale=s), ops.gemv(x, Wq, w_scale=s))

            base = run()
            for xb, grid in ((1, 0), (0, 8), (0, 64), (0, 256)):
                assert lib.db_tune(b"gemv_xb", xb) == 0
                assert lib.db_tune(b"gemv_pass_grid", grid) == 0
                for a, b in zip(run(), base):
                    err = rel_l2(a.float().cpu().numpy(), b.float().cpu().numpy())
                    assert err < 1e-3, f"B={B} K={K} N={N} xb={xb} grid={grid}: rel-L2 {err:.2e}"
    finally:
        lib.db_tune(b"gemv_xb", 0)
        lib.db_tune(b"gemv_pass_grid", 0)


# --------------------------------------------------- long rows (MFMA, streamed x)
# Plain GEMV with K a multiple of 2048 above 4096 -- the decode chain's down
# projection, K = 14336: the launch the library chooses, and the long-row
# kernel, which streams both operands in K chunks: batch tiles of
# 8, 16 and 32 rows in one pass, two passes above 32, N not a multiple of
# the 8-row group, fewer groups than CUs, fp16 and e4m3 weights.
LONG_CASES = [
    ("f16", 3, 14336, 4096), ("f16", 16, 14336, 4096), ("f16", 32, 14336, 1000),
    ("f16", 9, 8192, 4100), ("f16", 40, 6144, 520), ("f16", 12, 14336, 7),
    ("fp8", 8, 14336, 4096), ("fp8", 32, 14336, 2048), ("fp8", 17, 28672, 300),
    ("fp8", 5, 6144, 9), ("fp8", 33, 10240, 264),
    # two rows, which take this kernel too
    ("f16", 2, 14336, 4096), ("fp8", 2, 14336, 1000),
]


@pytest.mark.parametrize("dtype,B,K,N", LONG_CASES)
def test_long_row_gemv_mfma_parity(dtype, B, K, N):
    from decodebench_amd.quant import quantize_e4m3_rows

    print(f"[long] {dtype} B={B} K={K} N={N}", flush=True)
    gen = torch.Generator().manual_seed(8000 + B + K + N)
    x = randn(gen, (B, K))
    W = randn(gen, (N, K), std=1.0 / math.sqrt(K))
    if dtype == "fp8":
        Wq, s = quantize_e4m3_rows(W)
        call = functools.partial(ops.gemv, x.cuda(), Wq.cuda(), w_scale=s.cuda())
        ref = stages.gemv_fp8(x, Wq, s)
        exact = cref.gemv_fp8_exact(x.numpy(), Wq.view(torch.uint8).numpy(), s.numpy())
    else:
        call = functools.partial(ops.gemv, x.cuda(), W.cuda())
        ref, exact = stages.gemv(x, W), cref.gemv_exact(x.numpy(), W.numpy())
    lib = ops.load_library()
    for stage in (0, 2):  # 2: the long-row kernel as it runs by itself
        assert lib.db_tune(b"gemv_long_stage", stage) == 0
        try:
            y = call()
        finally:
            lib.db_tune(b"gemv_long_stage", 0)
        torch.cuda.synchronize()
        assert y.shape == (B, N)
        assert_parity(y, ref, exact, F12_REL_L2, f"long {dtype} B={B} K={K} N={N} stage={stage}")


def test_long_row_gemv_launch_shapes_agree():
    """The down-projection shape at 2, 16 and 32 rows through both activation
    paths (direct and LDS-staged), every chunk size and row-group count of the
    long-row kernel, and through the VALU kernel, agrees to fp32 summation
    order."""
    from decodebench_amd.quant import quantize_e4m3_rows

    gen = torch.Generator().manual_seed(79)
    lib = ops.load_library()
    W = randn(gen, (4096, 14336), std=1.0 / math.sqrt(14336))
    Wq, s = (t.cuda() for t in quantize_e4m3_rows(W))
    W = W.cuda()
    try:
        for B in (2, 16, 32):
            x = randn(gen, (B, 14336)).cuda()
            assert lib.db_tune(b"gemv_mfma_min_batch", 1 << 20) == 0
            base = (ops.gemv(x, W), ops.gemv(x, Wq, w_scale=s))
            assert lib.db_tune(b"gemv_mfma_min_batch", 2) == 0
            for stage in (1, 2):
                for kc in (2, 4):
                    for gpw in (1, 2, 4):
                        assert lib.db_tune(b"gemv_long_stage", stage) == 0
                        assert lib.db_tune(b"gemv_long_kc", kc) == 0
                        assert lib.db_tune(b"gemv_long_gpw", gpw) == 0
                        got = (ops.gemv(x, W), ops.gemv(x, Wq, w_scale=s))
                        for a, b in zip(got, base):
                            err = rel_l2(a.float().cpu().numpy(), b.float().cpu().numpy())
                            assert err < 1e-3, \
                                f"B={B} stage={stage} kc={kc} gpw={gpw}: rel-L2 {err:.2e}"
    finally:
        for key in (b"gemv_mfma_min_batch", b"gemv_long_kc", b"gemv_long_gpw",
                    b"gemv_long_stage"):
            lib.db_tune(key, 0)


# --------------------------------------------------- gate/up pair, streamed x
# The gate/up pair + SwiGLU, and RMSNorm -> gate/up + SwiGLU, from 17 rows: the
# full config-2 shape at B=32, more and fewer outputs than the CUs' shares, N
# that no tile divides, fp16 and e4m3; the tile kernel, or 16-row passes where
# the outputs are few.
PAIR_CASES = [
    ("f2", "f16", 32, 4096, 14336), ("f2", "f16", 17, 4096, 2048), ("f2", "f16", 40, 2048, 776),
    ("f2", "f16", 24, 4096, 1001), ("f2", "f16", 33, 6144, 264),
    ("f2", "fp8", 32, 4096, 14336), ("f2", "fp8", 20, 2048, 1792), ("f2", "fp8", 48, 4096, 520),
    ("f2n", "f16", 32, 4096, 14336), ("f2n", "f16", 17, 2048, 1000), ("f2n", "f16", 40, 4096, 264),
    ("f2n", "fp8", 24, 4096, 14336), ("f2n", "fp8", 33, 2048, 776),
    # one group (a tile whose second half repeats it) and two groups
    ("f2", "f16", 17, 2048, 8), ("f2n", "fp8", 32, 4096, 16),
]


@pytest.mark.parametrize("mode,dtype,B,K,N", PAIR_CASES)
def test_gateup_pair_streamed_parity(mode, dtype, B, K, N):
    from decodebench_amd.quant import quantize_e4m3_rows

    print(f"[pair] {mode} {dtype} B={B} K={K} N={N}", flush=True)
    gen = torch.Generator().manual_seed(9000 + B + K + N)
    x = randn(gen, (B, K))
    g = randn(gen, (K,), std=0.1, mean=1.0)
    Wg = randn(gen, (N, K), std=0.02)
    Wu = randn(gen, (N, K), std=0.02)
    norm = mode == "f2n"
    xin = stages.rmsnorm(x, g, 1e-6) if norm else x
    xin_np = cref.rmsnorm(x.numpy(), g.numpy(), 1e-6) if norm else x.numpy()
    if dtype == "fp8":
        Gq, sg = quantize_e4m3_rows(Wg)
        Uq, su = quantize_e4m3_rows(Wu)
        if norm:
            y = ops.f2_rmsnorm_gateup_swiglu(x.cuda(), g.cuda(), Gq.cuda(), Uq.cuda(),
                                             sg=sg.cuda(), su=su.cuda(), eps=1e-6)
        else:
            y = ops.f2_gateup_swiglu(x.cuda(), Gq.cuda(), Uq.cuda(), sg.cuda(), su.cuda())
        ref = stages.f2_fp8(xin, Gq, sg, Uq, su)
        exact = cref.f2_fp8_exact(xin_np, Gq.view(torch.uint8).numpy(), sg.numpy(),
                                  Uq.view(torch.uint8).numpy(), su.numpy())
    else:
        if norm:
            y = ops.f2_rmsnorm_gateup_swiglu(x.cuda(), g.cuda(), Wg.cuda(), Wu.cuda(), eps=1e-6)
        else:
            y = ops.f2_gateup_swiglu(x.cuda(), Wg.cuda(), Wu.cuda())
        ref, exact = stages.f2(xin, Wg, Wu), cref.f2_exact(xin_np, Wg.numpy(), Wu.numpy())
    torch.cuda.synchronize()
    assert y.shape == (B, N)
    assert_parity(y, ref, exact, 5e-3, f"pair {mode} {dtype} B={B} K={K} N={N}")


def test_gateup_pair_launch_shapes_agree():
    """The config-2 gate/up pair, with and without the fused RMSNorm, at 16 and
    32 rows through the tile kernel and through the 16-row passes agrees to fp32
    summation order, fp16 and e4m3."""
    from decodebench_amd.quant import quantize_e4m3_rows

    gen = torch.Generator().manual_seed(80)
    lib = ops.load_library()
    Wg = randn(gen, (14336, 4096), std=0.02)
    Wu = randn(gen, (14336, 4096), std=0.02)
    g = randn(gen, (4096,), std=0.1, mean=1.0).cuda()
    Gq, sg = (t.cuda() for t in quantize_e4m3_rows(Wg))
    Uq, su = (t.cuda() for t in quantize_e4m3_rows(Wu))
    Wg, Wu = Wg.cuda(), Wu.cuda()
    try:
        for B in (16, 32):
            x = randn(gen, (B, 4096)).cuda()
            def calls():
                return (ops.f2_gateup_swiglu(x, Wg, Wu), ops.f2_gateup_swiglu(x, Gq, Uq, sg, su),
                        ops.f2_rmsnorm_gateup_swiglu(x, g, Wg, Wu),
                        ops.f2_rmsnorm_gateup_swiglu(x, g, Gq, Uq, sg=sg, su=su))

            assert lib.db_tune(b"gemv_pair_min_batch", 1 << 20) == 0
            base = calls()
            assert lib.db_tune(b"gemv_pair_min_batch", 2) == 0
            for a, b in zip(calls(), base):
                err = rel_l2(a.float().cpu().numpy(), b.float().cpu().numpy())
                assert err < 1e-3, f"B={B}: rel-L2 {err:.2e}"
    finally:
        lib.db_tune(b"gemv_pair_min_batch", 0)


# --------------------------------------------------- GEMV edge shapes
# The smallest K (one 16-byte chunk per row), a single output row, and the
# largest K the ABI accepts (the activation row fills the 152 KB LDS
# budget), for fp16 and e4m3 weights.
EDGE_CASES = [("f1", 1, 8, 1, "f16"), ("plain", 3, 8, 5, "f16"), ("f2", 2, 16, 1, "f16"),
              ("f1", 1, 77824, 64, "f16"), ("plain", 1, 77824, 33, "fp8"),
              ("f2", 1, 77824, 17, "fp8"), ("plain", 1, 16, 1, "fp8"),
              # e4m3 row whose 8-chunk k-steps would pad past the LDS budget
              ("plain", 1, 77808, 9, "fp8"), ("f2", 2, 77808, 5, "fp8")]


@pytest.mark.parametrize("mode,B,K,N,dtype", EDGE_CASES)
def test_gemv_edge_shapes(mode, B, K, N, dtype):
    from decodebench_amd.quant import quantize_e4m3_rows

    print(f"[edge] {mode} {dtype} B={B} K={K} N={N}", flush=True)
    gen = torch.Generator().manual_seed(7000 + B + K + N)
    x = randn(gen, (B, K))
    g = randn(gen, (K,), std=0.1, mean=1.0)
    w_std = 1.0 / math.sqrt(K)
    W, W2 = randn(gen, (N, K), std=w_std), randn(gen, (N, K), std=w_std)
    xd, gd = x.cuda(), g.cuda()
    if dtype == "fp8":
        Wq, s = quantize_e4m3_rows(W)
        W2q, s2 = quantize_e4m3_rows(W2)
        bits, bits2 = Wq.view(torch.uint8).numpy(), W2q.view(torch.uint8).numpy()
        if mode == "plain":
            y = ops.gemv(xd, Wq.cuda(), w_scale=s.cuda())
            ref, exact = stages.gemv_fp8(x, Wq, s), cref.gemv_fp8_exact(x.numpy(), bits, s.numpy())
        else:
            y = ops.f2_gateup_swiglu(xd, Wq.cuda(), W2q.cuda(), s.cuda(), s2.cuda())
            ref = stages.f2_fp8(x, Wq, s, W2q, s2)
            exact = cref.f2_fp8_exact(x.numpy(), bits, s.numpy(), bits2, s2.numpy())
    elif mode == "f1":
        y = ops.f1_rmsnorm_gemv(xd, gd, W.cuda())
        ref, exact = stages.f1(x, g, W), cref.f1_exact(x.numpy(), g.numpy(), W.numpy())
    elif mode == "f2":
        y = ops.f2_gateup_swiglu(xd, W.cuda(), W2.cuda())
        ref, exact = stages.f2(x, W, W2), cref.f2_exact(x.numpy(), W.numpy(), W2.numpy())
    else:
        y = ops.gemv(xd, W.cuda())
        ref, exact = stages.gemv(x, W), cref.gemv_exact(x.numpy(), W.numpy())
    torch.cuda.synchronize()
    assert y.shape == (B, N)
    assert_parity(y, ref, exact, 5e-3, f"edge {mode} {dtype} B={B} K={K} N={N}")


# ------------------------------------------- RMSNorm -> gate/up + SwiGLU
# One kernel for the decode chain's post-attention half; batch 1 takes the
# VALU kernel, batches of 2..16 (and passes of 16) the MFMA kernel.
F2N_CASES = [(1, 4096, 14336), (1, 1024, 300), (1, 4104, 64), (4, 4096, 1000),
             (17, 4096, 600), (2, 2048, 777), (9, 512, 40),
             # x staged through LDS on the batched kernel: one and two batch
             # tiles at K = 2048 and 4096, up to 7 row groups per workgroup
             (3, 2048, 333), (12, 2048, 520), (16, 4096, 14336)]


@pytest.mark.parametrize("B,K,N", F2N_CASES)
def test_f2_rmsnorm_gateup_swiglu_parity(B, K, N):
    print(f"[f2n] B={B} K={K} N={N}", flush=True)
    gen = torch.Generator().manual_seed(5000 + B + K + N)
    x = randn(gen, (B, K))
    g = randn(gen, (K,), std=0.1, mean=1.0)
    Wg = randn(gen, (N, K), std=0.02)
    Wu = randn(gen, (N, K), std=0.02)
    y = ops.f2_rmsnorm_gateup_swiglu(x.cuda(), g.cuda(), Wg.cuda(), Wu.cuda(), eps=1e-6)
    torch.cuda.synchronize()
    assert y.shape == (B, N)
    ref = stages.f2_rmsnorm(x, g, Wg, Wu, 1e-6)
    xh = cref.rmsnorm(x.numpy(), g.numpy(), 1e-6)
    exact = cref.f2_exact(xh, Wg.numpy(), Wu.numpy())
    assert_parity(y, ref, exact, 5e-3, f"f2n B={B} K={K} N={N}")


# ------------------------------------------------------- fp8 e4m3 weights
# OCP e4m3 weights with per-row fp32 scales (quantize_e4m3_rows), the four
# GEMV modes, decode-chain shapes (QKV, O, gate/up, down) plus ragged ones:
# K not a multiple of the 1 KB row step, N not a multiple of the row group,
# batches that take several passes.
FP8_CASES = [
    ("f1", 1, 4096, 6144), ("f1", 1, 4096, 4096), ("f1", 3, 4112, 131), ("f1", 9, 1024, 64),
    ("f2", 1, 4096, 14336), ("f2", 2, 2048, 333), ("f2", 8, 4096, 1000),
    ("f2n", 1, 4096, 14336), ("f2n", 5, 4096, 257),
    ("plain", 1, 14336, 4096), ("plain", 1, 4096, 4096), ("plain", 4, 14336, 512),
    ("plain", 1, 16, 5), ("plain", 12, 4096, 300),
    # rows longer than 4096 at one batch row: 8-wave workgroups of one row per wave
    ("plain", 1, 4112, 777), ("plain", 1, 6000, 1),
    # batched e4m3 on the MFMA kernel (K in {2048, 4096}, batches from 2 / 3 rows)
    ("f1", 16, 4096, 6144), ("f1", 32, 2048, 1032), ("f2", 17, 4096, 600),
    ("f2n", 9, 2048, 100), ("plain", 3, 2048, 8), ("plain", 16, 4096, 4100),
    ("f2", 2, 4096, 520), ("f2n", 2, 4096, 1000),
    ("f1", 32, 4096, 6144), ("plain", 20, 4096, 777), ("f1", 40, 2048, 520),
    ("f1", 6, 2048, 333), ("f1", 8, 4096, 4096),
    # two rows on the MFMA kernel: e4m3 F1 (the QKV shape and a ragged one)
    ("f1", 2, 4096, 6144), ("f1", 2, 2048, 1001),
]


@pytest.mark.parametrize("mode,B,K,N", FP8_CASES)
def test_fp8_weight_gemv_parity(mode, B, K, N):
    from decodebench_amd.quant import quantize_e4m3_rows

    print(f"[fp8] {mode} B={B} K={K} N={N}", flush=True)
    gen = torch.Generator().manual_seed(6000 + B + K + N)
    x = randn(gen, (B, K))
    g = randn(gen, (K,), std=0.1, mean=1.0)
    Wq, s = quantize_e4m3_rows(randn(gen, (N, K), std=0.02))
    W2q, s2 = quantize_e4m3_rows(randn(gen, (N, K), std=0.02))
    bits, bits2 = Wq.view(torch.uint8).numpy(), W2q.view(torch.uint8).numpy()
    xd, gd = x.cuda(), g.cuda()
    if mode == "f1":
        y = ops.f1_rmsnorm_gemv(xd, gd, Wq.cuda(), w_scale=s.cuda())
        ref = stages.f1_fp8(x, g, Wq, s)
        exact, bound = cref.f1_fp8_exact(x.numpy(), g.numpy(), bits, s.numpy()), F12_REL_L2
    elif mode in ("f2", "f2n"):
        if mode == "f2":
            y = ops.f2_gateup_swiglu(xd, Wq.cuda(), W2q.cuda(), s.cuda(), s2.cuda())
            xin, xin_np = x, x.numpy()
        else:
            y = ops.f2_rmsnorm_gateup_swiglu(xd, gd, Wq.cuda(), W2q.cuda(), sg=s.cuda(),
                                             su=s2.cuda())
            xin = stages.rmsnorm(x, g)
            xin_np = cref.rmsnorm(x.numpy(), g.numpy())
        ref = stages.f2_fp8(xin, Wq, s, W2q, s2)
        exact, bound = cref.f2_fp8_exact(xin_np, bits, s.numpy(), bits2, s2.numpy()), 5e-3
    else:
        y = ops.gemv(xd, Wq.cuda(), w_scale=s.cuda())
        ref = stages.gemv_fp8(x, Wq, s)
        exact, bound = cref.gemv_fp8_exact(x.numpy(), bits, s.numpy()), F12_REL_L2
    torch.cuda.synchronize()
    assert y.shape == (B, N)
    assert_parity(y, ref, exact, bound, f"fp8 {mode} B={B} K={K} N={N}")


def test_fp8_mfma_and_valu_paths_agree():
    """A batch of 8 on e4m3 weights through both kernels (the MFMA threshold
    raised to force the VALU path) differs only by fp32 summation order."""
    from decodebench_amd.quant import quantize_e4m3_rows

    gen = torch.Generator().manual_seed(78)
    x = randn(gen, (8, 4096)).cuda()
    g = randn(gen, (4096,), std=0.1, mean=1.0).cuda()
    Wq, s = (t.cuda() for t in quantize_e4m3_rows(randn(gen, (6144, 4096), std=0.02)))
    Uq, su = (t.cuda() for t in quantize_e4m3_rows(randn(gen, (6144, 4096), std=0.02)))
    lib = ops.load_library()
    try:
        outs = []
        for thr in (2, 1 << 20):
            assert lib.db_tune(b"gemv_mfma_min_batch", thr) == 0
            outs.append((ops.f1_rmsnorm_gemv(x, g, Wq, w_scale=s),
                         ops.f2_gateup_swiglu(x, Wq, Uq, s, su), ops.gemv(x, Wq, w_scale=s),
                         ops.f2_rmsnorm_gateup_swiglu(x, g, Wq, Uq, sg=s, su=su)))
    finally:
        lib.db_tune(b"gemv_mfma_min_batch", 0)
    for a, b in zip(*outs):
        assert rel_l2(a.float().cpu().numpy(), b.float().cpu().numpy()) < 1e-3


def test_fp8_raw_byte_weights_equal_float8_tensor():
    """A uint8 view of the same e4m3 bytes is accepted and gives identical
    results (callers may hold fp8 weights as raw bytes)."""
    from decodebench_amd.quant import quantize_e4m3_rows

    gen = torch.Generator().manual_seed(61)
    x = randn(gen, (1, 4096)).cuda()
    Wq, s = quantize_e4m3_rows(randn(gen, (4096, 4096), std=0.02))
    Wq, s = Wq.cuda(), s.cuda()
    a = ops.gemv(x, Wq, w_scale=s)
    b = ops.gemv(x, Wq.view(torch.uint8), w_scale=s)
    assert torch.equal(a, b)


# ------------------------------------------------------------------- F4
def f4_inputs(B, Hq, Hkv, L, seed):
    gen = torch.Generator().manual_seed(seed)
    q = randn(gen, (B, Hq, 128))
    K = randn(gen, (B, Hkv, L, 128))
    V = randn(gen, (B, Hkv, L, 128))
    return q, K, V


F4_CASES = [
    # (B, Hq, Hkv, L, S)
    (1, 32, 8, 1024, None), (1, 32, 8, 1024, 1), (1, 32, 8, 1024, 4),
    (1, 32, 8, 8192, None), (1, 32, 8, 8192, 16), (1, 32, 8, 8192, 64),
    (1, 32, 8, 32768, None), (1, 32, 8, 32768, 64),
    (4, 32, 8, 1024, None), (4, 32, 8, 8192, 16), (8, 32, 8, 1024, 4),
    (1, 8, 8, 300, 3), (2, 16, 8, 257, 5), (1, 64, 8, 100, None),
    (1, 32, 8, 1, None), (1, 32, 8, 15, 4), (1, 32, 8, 17, 2), (3, 32, 8, 4097, 7),
    (1, 4, 4, 2000, 256),
    # Tile-stream edges: with S = 1 each of the 8 waves walks 3 tiles (L = 384), 3-4 with a
    # partial last tile (391), 4-5 (528) or 5-6 (720) tiles through the two register sets.
    (1, 32, 8, 384, 1), (1, 32, 8, 391, 1), (1, 32, 8, 528, 1), (1, 32, 8, 720, 1),
    (2, 32, 8, 1040, 2),
]


@pytest.mark.parametrize("B,Hq,Hkv,L,S", F4_CASES)
def test_f4_splitkv_parity(B, Hq, Hkv, L, S):
    print(f"[f4] B={B} Hq={Hq} Hkv={Hkv} L={L} S={S}", flush=True)
    q, K, V = f4_inputs(B, Hq, Hkv, L, 3000 + B * 7 + L + (S or 0))
    o = ops.f4_flashdecode(q.cuda(), K.cuda(), V.cuda(), n_splits=S)
    torch.cuda.synchronize()
    assert o.shape == (B, Hq, 128)
    ref = stages.f4(q, K, V)
    exact = cref.attention(q.numpy(), K.numpy(), V.numpy())
    assert_parity(o, ref, exact, F4_REL_L2, f"f4 B={B} Hq={Hq} Hkv={Hkv} L={L} S={S}")


# Shapes run with each score-operand layout forced (db_tune "f4_line": 1 = whole-line K
# loads, 2 = 16 keys x 64 bytes); the launcher otherwise picks by tiles per wave.
F4_LAYOUT_CASES = [(1, 32, 8, 1024, None), (1, 32, 8, 8192, None), (4, 32, 8, 4096, 4),
                   (1, 64, 8, 100, None), (1, 8, 8, 300, 3), (1, 32, 8, 17, 2),
                   (2, 16, 8, 257, 5), (1, 16, 16, 2000, 8), (1, 32, 8, 720, 1)]


@pytest.mark.parametrize("B,Hq,Hkv,L,S", F4_LAYOUT_CASES)
def test_f4_score_layouts(B, Hq, Hkv, L, S):
    print(f"[f4-layout] B={B} Hq={Hq} Hkv={Hkv} L={L} S={S}", flush=True)
    q, K, V = f4_inputs(B, Hq, Hkv, L, 3500 + B * 7 + L + (S or 0))
    exact = cref.attention(q.numpy(), K.numpy(), V.numpy())
    ref = stages.f4(q, K, V)
    outs = []
    try:
        for layout in (1, 2):
            ops.tune("f4_line", layout)
            o = ops.f4_flashdecode(q.cuda(), K.cuda(), V.cuda(), n_splits=S)
            torch.cuda.synchronize()
            assert_parity(o, ref, exact, F4_REL_L2, f"f4 layout {layout} B={B} L={L} S={S}")
            outs.append(o.float().cpu().numpy())
    finally:
        ops.tune("f4_line", 0)
    assert rel_l2(outs[0], outs[1]) < 2e-3


# Shapes of the 8-wave whole-line kernel (at least 8 tiles per split, at most 8 (batch,
# kv-head) pairs; "f4_depth" applies to that kernel only) run with one and with two tiles
# in flight per wave: 8 tiles per wave (config 4, L = 32768), 2, 3-4 with a partial last
# tile, 5-6, 2-3 with G = 1, and 39-40.
F4_DEPTH_CASES = [(1, 32, 8, 32768, None), (1, 32, 8, 8192, None), (1, 32, 8, 391, 1),
                  (1, 32, 8, 720, 1), (1, 8, 8, 300, 1), (1, 16, 4, 5000, 1)]


@pytest.mark.parametrize("B,Hq,Hkv,L,S", F4_DEPTH_CASES)
def test_f4_tile_depths(B, Hq, Hkv, L, S):
    """The two tile streams change when loads are issued, not what is
    computed: the outputs are bit-identical and match the exact oracle."""
    print(f"[f4-depth] B={B} Hq={Hq} Hkv={Hkv} L={L} S={S}", flush=True)
    q, K, V = f4_inputs(B, Hq, Hkv, L, 3700 + B * 7 + L + (S or 0))
    exact = cref.attention(q.numpy(), K.numpy(), V.numpy())
    ref = stages.f4(q, K, V)
    outs = []
    try:
        for depth in (1, 2):
            ops.tune("f4_depth", depth)
            o = ops.f4_flashdecode(q.cuda(), K.cuda(), V.cuda(), n_splits=S)
            torch.cuda.synchronize()
            assert_parity(o, ref, exact, F4_REL_L2, f"f4 depth {depth} B={B} L={L} S={S}")
            outs.append(o.cpu())
    finally:
        ops.tune("f4_depth", 0)
    assert torch.equal(outs[0], outs[1])


@pytest.mark.parametrize("L", [8192, 32768])
def test_f4_full_batch_split_invariance(L):
    """B = 8 at full length: every split count gives the same answer, and
    batch row 0 matches the exact oracle (size-independent properties)."""
    print(f"[f4-inv] B=8 L={L}", flush=True)
    q, K, V = f4_inputs(8, 32, 8, L, 77 + L)
    qd, Kd, Vd = q.cuda(), K.cuda(), V.cuda()
    outs = [ops.f4_flashdecode(qd, Kd, Vd, n_splits=s).float().cpu().numpy()
            for s in (1, 4, 16, 64, None)]
    for o in outs[1:]:
        assert rel_l2(o, outs[0]) < 2e-3
    exact0 = cref.attention(q[:1].numpy(), K[:1].numpy(), V[:1].numpy())
    assert rel_l2(outs[-1][:1], exact0) < F4_REL_L2
    exact7 = cref.attention(q[7:].numpy(), K[7:].numpy(), V[7:].numpy())
    assert rel_l2(outs[-1][7:], exact7) < F4_REL_L2


def test_f4_config4_batch4_full_length():
    """Config 4 at B = 4, L = 32768: batch rows 0 and 3 against the exact
    oracle (relative L2, which zeros would fail: |o| is about 0.009 here)
    and the same answer for every split count."""
    print("[f4-cfg4] B=4 L=32768", flush=True)
    q, K, V = f4_inputs(4, 32, 8, 32768, 4321)
    qd, Kd, Vd = q.cuda(), K.cuda(), V.cuda()
    outs = {s: ops.f4_flashdecode(qd, Kd, Vd, n_splits=s).float().cpu().numpy()
            for s in (None, 1, 4, 16, 64)}
    for s, o in outs.items():
        assert rel_l2(o, outs[None]) < 2e-3, f"S={s}"
    for row in (0, 3):
        exact = cref.attention(q[row:row + 1].numpy(), K[row:row + 1].numpy(),
                               V[row:row + 1].numpy())
        assert rel_l2(outs[None][row:row + 1], exact) < F4_REL_L2, f"row {row}"
        assert rel_l2(np.zeros_like(exact), exact) > 0.5   # the bound rejects zeros


def test_f4_workspace_reuse_is_deterministic():
    """One zero-filled workspace serves any number of calls: repeated calls
    (and a different split count on the same workspace, whose stale records
    must not leak into the result) give bitwise-identical results; partial
    records full of garbage (NaN bytes) before the first call change nothing;
    every call leaves the split ticket lines at zero."""
    q, K, V = f4_inputs(1, 32, 8, 8192, 5)
    qd, Kd, Vd = q.cuda(), K.cuda(), V.cuda()
    nbytes = ops.load_library().db_f4_workspace_bytes(1, 32, 8, 8192, 128, 64)
    ws = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device="cuda")
    ws[:8 * 256] = 0                    # the ticket lines of the 8 pairs (256 bytes each)
    first = ops.f4_flashdecode(qd, Kd, Vd, n_splits=64, workspace=ws)
    for _ in range(20):
        again = ops.f4_flashdecode(qd, Kd, Vd, n_splits=64, workspace=ws)
        assert torch.equal(first, again)
    other = ops.f4_flashdecode(qd, Kd, Vd, n_splits=16, workspace=ws)
    assert rel_l2(other.float().cpu().numpy(), first.float().cpu().numpy()) < 2e-3
    exact = cref.attention(q.numpy(), K.numpy(), V.numpy())
    assert rel_l2(first.float().cpu().numpy(), exact) < F4_REL_L2
    torch.cuda.synchronize()
    assert int(ws[:8 * 256].count_nonzero()) == 0     # tickets at zero, no pair recomputed


def test_f4_concurrent_streams_get_their_own_workspace():
    """Two streams running F4 of one shape at the same time: the cached
    workspace is per stream, so neither stream's split partials are
    overwritten by the other's, and both match their single-stream result."""
    inputs = [f4_inputs(1, 32, 8, 8192, 11 + i) for i in range(2)]
    dev = [tuple(t.cuda() for t in inp) for inp in inputs]
    ref = [ops.f4_flashdecode(*d) for d in dev]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for s in streams:
        s.wait_stream(torch.cuda.current_stream())
    outs = [[], []]
    for _ in range(10):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                outs[i].append(ops.f4_flashdecode(*dev[i]))
    torch.cuda.synchronize()
    ws = [ops.f4_workspace(1, 32, 8, 8192, 128, ops.f4_default_splits(1, 8, 8192), "cuda")]
    with torch.cuda.stream(streams[0]):
        ws.append(ops.f4_workspace(1, 32, 8, 8192, 128, ops.f4_default_splits(1, 8, 8192),
                                   "cuda"))
    assert ws[0].data_ptr() != ws[1].data_ptr()
    for i in range(2):
        for o in outs[i]:
            assert torch.equal(o, ref[i])


@pytest.mark.parametrize("merge", [2, 0])
def test_f4_graphs_replayed_concurrently_use_their_own_workspaces(merge):
    """Two graphs captured on torch's capture stream, each holding F4 calls
    of the same shape, replayed at the same time on two streams: each
    capture has its own workspace, so both graphs give their eager
    results on every replay (with the split merge in a second launch, and
    with the default in-launch merge, whose tickets must start at zero)."""
    inputs = [tuple(t.cuda() for t in f4_inputs(1, 32, 8, 8192, 41 + i)) for i in range(2)]
    try:
        ops.tune("f4_merge", merge)
        want = [ops.f4_flashdecode(*d) for d in inputs]
        torch.cuda.synchronize()
        graphs, outs = [], []
        for d in inputs:
            ops.f4_flashdecode(*d)          # warm-up outside the capture
            torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                o = [ops.f4_flashdecode(*d) for _ in range(4)]
            graphs.append(g)
            outs.append(o)
        streams = [torch.cuda.Stream(), torch.cuda.Stream()]
        for rep in range(6):
            for s in streams:
                s.wait_stream(torch.cuda.current_stream())
            for g, s in zip(graphs, streams):
                with torch.cuda.stream(s):
                    g.replay()
            for s in streams:
                torch.cuda.current_stream().wait_stream(s)
            torch.cuda.synchronize()
            for i in range(2):
                for o in outs[i]:
                    assert torch.equal(o, want[i]), f"graph {i}, replay {rep}"
        del graphs
        torch.cuda.synchronize()
        assert ops.release_captured_workspaces() >= 2     # one per capture
    finally:
        ops.tune("f4_merge", 0)


@pytest.mark.parametrize("L", [1024, 8192, 32768])
def test_f4_two_launch_halves_make_the_pair(L):
    """The measurement hook behind the per-half timings: with the merge in a
    second launch, f4_launch = 1 launches the split kernel alone and
    f4_launch = 2 the merge alone; run one after the other on one workspace
    they give bitwise the output of the two-launch call, and each reports a
    single launch."""
    print(f"[f4-halves] L={L}", flush=True)
    q, K, V = f4_inputs(1, 32, 8, L, 4200 + L)
    qd, Kd, Vd = q.cuda(), K.cuda(), V.cuda()
    S = ops.f4_default_splits(1, 8, L)
    ws = torch.zeros(ops.load_library().db_f4_workspace_bytes(1, 32, 8, L, 128, S),
                     dtype=torch.uint8, device="cuda")
    try:
        ops.tune("f4_merge", 2)
        S_run = ops.f4_launch_info(1, 32, 8, L, S)[0]
        assert ops.f4_launch_info(1, 32, 8, L, S) == (S_run, 2)
        want = ops.f4_flashdecode(qd, Kd, Vd, workspace=ws)
        torch.cuda.synchronize()
        ws.zero_()
        ops.tune("f4_launch", 1)
        assert ops.f4_launch_info(1, 32, 8, L, S) == (S_run, 1)
        ops.f4_flashdecode(qd, Kd, Vd, workspace=ws)
        ops.tune("f4_launch", 2)
        assert ops.f4_launch_info(1, 32, 8, L, S) == (S_run, 1)
        got = ops.f4_flashdecode(qd, Kd, Vd, workspace=ws)
        torch.cuda.synchronize()
    finally:
        ops.tune("f4_launch", 0)
        ops.tune("f4_merge", 0)
    assert torch.equal(got, want)
    exact = cref.attention(q.numpy(), K.numpy(), V.numpy())
    assert rel_l2(want.float().cpu().numpy(), exact) < F4_REL_L2


@pytest.mark.parametrize("B,L", [(1, 1024), (1, 8192), (4, 8192), (8, 300)])
def test_f4_in_launch_merge_matches_two_launch_merge(B, L):
    """The split merge done by the last split's workgroup (the default on an
    8-XCD device when B * Hkv is a multiple of 8) and by a second launch
    (f4_merge = 2) agree to fp32 summation order, and 100 back-to-back calls
    of the in-launch merge are bitwise identical (the ticket of every pair is
    taken exactly once per call and reset)."""
    print(f"[f4-merge] B={B} L={L}", flush=True)
    q, K, V = f4_inputs(B, 32, 8, L, 90 + B + L)
    qd, Kd, Vd = q.cuda(), K.cuda(), V.cuda()
    lib = ops.load_library()
    S = ops.f4_default_splits(B, 8, L)
    S_run = ops.f4_launch_info(B, 32, 8, L, S)[0]
    assert ops.f4_launch_info(B, 32, 8, L, S) == (S_run, 1)   # merged in the first launch
    ws = torch.zeros(lib.db_f4_workspace_bytes(B, 32, 8, L, 128, S), dtype=torch.uint8,
                     device="cuda")
    one = ops.f4_flashdecode(qd, Kd, Vd, workspace=ws)
    outs = [ops.f4_flashdecode(qd, Kd, Vd, workspace=ws) for _ in range(100)]
    torch.cuda.synchronize()
    # every pair's splits ran on one XCD in all 101 calls: nothing was recomputed
    assert int(ws[:B * 8 * 256].count_nonzero()) == 0
    try:
        assert lib.db_tune(b"f4_merge", 2) == 0
        assert ops.f4_launch_info(B, 32, 8, L, S) == (S, 2)
        two = ops.f4_flashdecode(qd, Kd, Vd)
        torch.cuda.synchronize()
    finally:
        assert lib.db_tune(b"f4_merge", 0) == 0
    assert rel_l2(one.float().cpu().numpy(), two.float().cpu().numpy()) < 1e-3
    for o in outs:
        assert torch.equal(o, one)
    exact = cref.attention(q.numpy(), K.numpy(), V.numpy())
    assert rel_l2(one.float().cpu().numpy(), exact) < F4_REL_L2


@pytest.mark.parametrize("Hq,L,S", [(64, 4096, 16), (16, 4096, 16), (8, 4096, 32), (8, 8192, 48),
                                    (32, 8192, 20), (32, 8192, 40),
                                    # 4 tiles per split: 4-wave workgroups, so G = 8 has one
                                    # split group and G = 1 eight
                                    (64, 1024, 16), (32, 1024, 16), (8, 1024, 16)])
def test_f4_in_launch_grouped_merge_head_groups(Hq, L, S):
    """The in-launch merge of more than 8 splits (split groups meeting in
    LDS, the (m, l) pairs handed between the lanes of each half-wave) at
    every query-head group size G = Hq / 8: G = 8, 2 and 1 lay out the
    output slots over the half-waves differently from G = 4 (G = 1 puts two
    split groups in one wave), and 20, 40 and 48 splits leave the last chunk
    of a group partly past S.  Checked against the second-launch merge and
    the fp64 oracle."""
    print(f"[f4-grouped] Hq={Hq} L={L} S={S}", flush=True)
    q, K, V = f4_inputs(1, Hq, 8, L, 5100 + Hq + L + S)
    qd, Kd, Vd = q.cuda(), K.cuda(), V.cuda()
    S_run, launches = ops.f4_launch_info(1, Hq, 8, L, S)
    assert S_run > 8 and launches == 1       # merged in the first launch, grouped
    one = ops.f4_flashdecode(qd, Kd, Vd, n_splits=S)
    torch.cuda.synchronize()
    lib = ops.load_library()
    try:
        assert lib.db_tune(b"f4_merge", 2) == 0
        assert ops.f4_launch_info(1, Hq, 8, L, S) == (S_run, 2)
        two = ops.f4_flashdecode(qd, Kd, Vd, n_splits=S)
        torch.cuda.synchronize()
    finally:
        assert lib.db_tune(b"f4_merge", 0) == 0
    assert rel_l2(one.float().cpu().numpy(), two.float().cpu().numpy()) < 1e-3
    ref = stages.f4(q, K, V)
    exact = cref.attention(q.numpy(), K.numpy(), V.numpy())
    assert_parity(one, ref, exact, F4_REL_L2, f"f4 grouped Hq={Hq} L={L} S={S}")


@pytest.mark.parametrize("B,L,k", [(1, 8192, 1), (1, 8192, 2), (1, 8192, 7), (4, 1024, 3),
                                   (8, 300, 2), (1, 32768, 5)])
def test_f4_misplaced_splits_are_recomputed_by_the_merger(B, L, k):
    """In-launch merge with workgroups reporting a foreign XCD, forced from
    the host (f4_misplace = k: split s reports another XCD when
    s % k == k - 1; k = 1 makes every split report a different one).  The
    merger of such a pair recomputes every split with the same code, so the
    output is bitwise the one of a call with every workgroup in place; calls
    after it (tickets cleared) are too."""
    print(f"[f4-misplace] B={B} L={L} k={k}", flush=True)
    q, K, V = f4_inputs(B, 32, 8, L, 300 + B + L + k)
    qd, Kd, Vd = q.cuda(), K.cuda(), V.cuda()
    S = ops.f4_default_splits(B, 8, L)
    assert ops.f4_launch_info(B, 32, 8, L, S)[1] == 1
    lib = ops.load_library()
    ws = torch.zeros(lib.db_f4_workspace_bytes(B, 32, 8, L, 128, S), dtype=torch.uint8,
                     device="cuda")
    want = ops.f4_flashdecode(qd, Kd, Vd, workspace=ws)
    try:
        assert lib.db_tune(b"f4_misplace", k) == 0
        got = [ops.f4_flashdecode(qd, Kd, Vd, workspace=ws) for _ in range(5)]
    finally:
        assert lib.db_tune(b"f4_misplace", 0) == 0
    after = ops.f4_flashdecode(qd, Kd, Vd, workspace=ws)
    torch.cuda.synchronize()
    for o in got + [after]:
        assert torch.equal(o, want)
    lines = ws[:B * 8 * 256].view(torch.int32).view(B * 8, 64).cpu()
    assert int(lines[:, :2].count_nonzero()) == 0         # tickets left at zero
    assert int(lines[:, 3:].count_nonzero()) == 0
    # the recompute counter: the normal calls (want, after) recomputed nothing; the
    # forced calls recomputed every pair holding a split that reported another XCD
    S_run = ops.f4_launch_info(B, 32, 8, L, S)[0]
    hooked = any(s % k == k - 1 for s in range(S_run))
    assert lines[:, 2].tolist() == [5 if hooked else 0] * (B * 8)
    exact = cref.attention(q.numpy(), K.numpy(), V.numpy())
    assert rel_l2(want.float().cpu().numpy(), exact) < F4_REL_L2


def test_f4_gqa_equals_mha_on_gpu():
    q, K, V = f4_inputs(1, 32, 8, 1000, 9)
    gqa = ops.f4_flashdecode(q.cuda(), K.cuda(), V.cuda())
    Kr = K.repeat_interleave(4, dim=1).contiguous()
    Vr = V.repeat_interleave(4, dim=1).contiguous()
    mha = ops.f4_flashdecode(q.cuda(), Kr.cuda(), Vr.cuda())
    assert rel_l2(gqa.float().cpu().numpy(), mha.float().cpu().numpy()) < 1e-3


# ------------------------------------------------- decode-layer chain
def c_oracle_layer(inp, Hq, fp8):
    """The chain on the C oracle: fp16 rounding at every stage boundary (as
    the torch stages round), each stage computed in double."""
    np_ = {k: (v.view(torch.uint8).numpy() if v.dtype == torch.float8_e4m3fn else v.numpy())
           for k, v in inp.items()}

    def proj(a, key, skey):
        if fp8:
            return cref.f2h(cref.gemv_fp8_exact(a, np_[key], np_[skey]))
        return cref.gemv(a, np_[key])

    B = np_["x"].shape[0]
    qkv = proj(cref.rmsnorm(np_["x"], np_["g1"]), "Wqkv", "s_qkv")
    q = np.ascontiguousarray(qkv[:, : Hq * 128].reshape(B, Hq, 128))
    attn = cref.f2h(cref.attention(q, np_["K"], np_["V"])).reshape(B, Hq * 128)
    h = proj(attn, "Wo", "s_o")
    hn = cref.rmsnorm(h, np_["g2"])
    if fp8:
        g = cref.f2h(cref.gemv_fp8_exact(hn, np_["Wg"], np_["s_gate"]))
        u = cref.f2h(cref.gemv_fp8_exact(hn, np_["Wu"], np_["s_up"]))
        ff = cref.swiglu(g, u)
    else:
        ff = cref.f2(hn, np_["Wg"], np_["Wu"])
    return proj(ff, "Wd", "s_down").astype(np.float64)


@pytest.mark.parametrize("dtype,B,L", [("f16", 1, 1024), ("fp8", 1, 1024), ("f16", 2, 520),
                                       ("fp8", 3, 300),
                                       # config 5 itself: batch 1, KV length 8192
                                       ("f16", 1, 8192), ("fp8", 1, 8192)])
def test_decode_layer_chain_parity(dtype, B, L):
    """Config-5 chain at Llama-3-8B width through the fused HIP kernels
    (F1 -> F4 -> O GEMV -> RMSNorm+F2 -> down GEMV) against the torch stage
    chain on the CPU and against the C oracle chain.

    Bar: each kernel meets rtol/atol 1e-2 on its own (the tests above); the
    twelve fp16 rounding points of the chain compound, and the second
    RMSNorm rescales the small O-projection output back to unit size, so two
    valid implementations of the chain already differ by more: the torch
    stages and the C oracle chain (same rounding points, double arithmetic
    per stage) differ by up to 1.6e-2 and miss rtol/atol 1e-2 at 1-3 of 4096
    outputs for these seeds.  The chain is held to rtol/atol 2e-2 against
    both, and to rel-L2 <= 5e-3 against the C oracle chain."""
    from decodebench_amd.demos.llama_decode import build_config

    print(f"[layer] {dtype} B={B} L={L}", flush=True)
    case = build_config("layer", batch=B, L=L, device="cpu", replicas=1, dtype=dtype,
                        seed=700 + B + L)
    cpu = case.inputs
    gpu = {k: v.cuda() for k, v in cpu.items()}
    y = case.fused(gpu)
    torch.cuda.synchronize()
    assert y.shape == (B, 4096)
    fp8 = dtype == "fp8"
    scales = ({k: cpu["s_" + k] for k in ("qkv", "o", "gate", "up", "down")} if fp8 else None)
    ref = stages.decode_layer(cpu["x"], cpu["g1"], cpu["Wqkv"], cpu["K"], cpu["V"], cpu["Wo"],
                              cpu["g2"], cpu["Wg"], cpu["Wu"], cpu["Wd"], 32, scales=scales)
    exact = c_oracle_layer(cpu, 32, fp8)
    assert_parity(y, ref, exact, 5e-3, f"layer {dtype} B={B} L={L}", tol=CHAIN_TOL)
    got = y.float().cpu().numpy().astype(np.float64)
    assert np.isclose(got, exact, rtol=CHAIN_TOL, atol=CHAIN_TOL).all()


# ------------------------------------------------------------ graph replay
@pytest.mark.parametrize("dtype", ["f16", "fp8"])
def test_decode_layer_replays_correctly_in_a_graph(dtype):
    """The six launches of the decode layer captured into one graph: five
    replays, with eager work in between, are bitwise equal to the eager
    call (the F4 workspace needs no reset between replays)."""
    from decodebench_amd.demos.llama_decode import build_config

    case = build_config("layer", batch=1, L=2048, replicas=1, dtype=dtype, seed=31)
    inp = case.inputs
    eager = case.fused(inp).clone()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        case.fused(inp)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = case.fused(inp)
    for i in range(5):
        inp["x"].add_(0.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager), f"{dtype} replay {i} differs from eager"


def test_streamed_gemv_kernels_replay_correctly_in_a_graph():
    """The kernels that stream their activations (the gate/up pair with and
    without the RMSNorm above 16 rows, the long-row down projection) captured
    in one hipGraph replay bit-identically to eager, with eager work between
    replays."""
    from decodebench_amd.quant import quantize_e4m3_rows

    gen = torch.Generator().manual_seed(12)
    x32 = randn(gen, (32, 4096)).cuda()
    x24 = randn(gen, (24, 4096)).cuda()
    x16 = randn(gen, (16, 14336)).cuda()
    g = randn(gen, (4096,), std=0.1, mean=1.0).cuda()
    Wg = randn(gen, (14336, 4096), std=0.02)
    Wu = randn(gen, (14336, 4096), std=0.02)
    Gq, sg = (t.cuda() for t in quantize_e4m3_rows(Wg))
    Uq, su = (t.cuda() for t in quantize_e4m3_rows(Wu))
    Wg, Wu = Wg.cuda(), Wu.cuda()
    Wd = randn(gen, (4096, 14336), std=1.0 / 128).cuda()

    def body():
        return (ops.f2_gateup_swiglu(x32, Wg, Wu),
                ops.f2_rmsnorm_gateup_swiglu(x24, g, Gq, Uq, sg=sg, su=su),
                ops.gemv(x16, Wd))

    eager = [t.clone() for t in body()]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        body()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = body()
    for i in range(5):
        x32.add_(0.0)                    # eager work between replays
        graph.replay()
        torch.cuda.synchronize()
        for e, o in zip(eager, outs):
            assert torch.equal(e, o), f"replay {i} differs from eager"


def test_ops_replay_correctly_in_a_graph():
    gen = torch.Generator().manual_seed(11)
    x = randn(gen, (1, 4096)).cuda()
    g = randn(gen, (4096,), std=0.1, mean=1.0).cuda()
    W = randn(gen, (4096, 4096), std=1 / 64).cuda()
    Wg = randn(gen, (2048, 4096), std=0.02).cuda()
    Wu = randn(gen, (2048, 4096), std=0.02).cuda()
    q, K, V = (t.cuda() for t in f4_inputs(1, 32, 8, 4096, 12))

    def body():
        return (ops.f1_rmsnorm_gemv(x, g, W), ops.f2_gateup_swiglu(x, Wg, Wu),
                ops.f4_flashdecode(q, K, V))

    eager = [t.clone() for t in body()]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        body()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        outs = body()
    for i in range(5):
        x.add_(0.0)                      # eager work between replays
        graph.replay()
        torch.cuda.synchronize()
        for e, o in zip(eager, outs):
            assert torch.equal(e, o), f"replay {i} differs from eager"
