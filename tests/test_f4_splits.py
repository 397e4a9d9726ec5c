"""The F4 split policy: how full its rounds of workgroups are, what stays
accepted, and (GPU) that odd split counts give the attention."""

import pytest

from decodebench_amd import ops

CUS = 256


@pytest.fixture(scope="module")
def lib():
    if not ops.LIB_PATH.exists():
        from decodebench_amd import build

        build.build()
    return ops.load_library()


def _used(L, S):
    nt = -(-L // 16)
    tps = -(-nt // min(S, nt))
    return -(-nt // tps), tps


@pytest.mark.parametrize("hkv", [1, 2, 4, 8, 16])
def test_default_splits_stay_in_range(lib, hkv):
    """Any batch and length: 1 to 256 splits of at least one tile, and records
    that db_f4_splitkv_noalloc accepts for every head group."""
    for B in (1, 2, 3, 5, 7, 12, 20, 33, 48, 64, 100, 300):
        for L in (1, 16, 17, 63, 64, 65, 300, 1024, 3001, 8192, 32768, 131072):
            S = lib.db_f4_default_splits(B, hkv, L, CUS)
            assert 1 <= S <= 256 and S <= max(1, -(-L // 16))
            for G in (1, 2, 4, 8):
                assert lib.db_f4_workspace_bytes(B, hkv * G, hkv, L, 128, S) <= 4 << 20


def test_default_splits_fill_their_rounds(lib):
    """Long contexts: at least 3/4 of the slots of the rounds that a split
    count takes are busy wherever few enough pairs let one choose."""
    for pairs in (8, 16, 24, 40, 56, 72, 80, 96, 112, 144, 160, 192):
        used, _ = _used(12000, lib.db_f4_default_splits(pairs // 8, 8, 12000, CUS))
        rounds = -(-pairs * used // CUS)
        assert pairs * used >= 0.75 * rounds * CUS, (pairs, used)


def test_contexts_that_a_merge_costs_more_than(lib):
    """Below 16 tiles one split, whatever the batch; one where the pairs alone
    fill the chip and shorter rounds hardly shorten the whole; and no fewer splits
    for a merge of eight where that takes a launch of its own."""
    for pairs in (1, 2, 3, 5, 8, 12, 16, 40, 64, 96, 128, 200, 300, 512):
        for L in (1, 64, 128, 177, 192, 208, 239, 240):
            assert lib.db_f4_default_splits(pairs, 1, L, CUS) == 1, (pairs, L)
    assert lib.db_f4_default_splits(75, 4, 448, CUS) == 1
    assert lib.db_f4_default_splits(48, 8, 496, CUS) == 1
    assert lib.db_f4_default_splits(3, 4, 1400, CUS) >= 11
    assert lib.db_f4_default_splits(1, 8, 300, CUS) > 1


def test_tuned_split_targets_keep_their_rule(lib):
    """Either knob away from its default: a workgroup per CU (times
    f4_blocks_per_cu), no fewer tiles per split than f4_min_tiles."""
    try:
        assert lib.db_tune(b"f4_blocks_per_cu", 2) == 0
        assert lib.db_f4_default_splits(5, 8, 8192, CUS) == -(-2 * CUS // 40)
        assert lib.db_tune(b"f4_blocks_per_cu", 1) == 0
        assert lib.db_tune(b"f4_min_tiles", 16) == 0
        assert lib.db_f4_default_splits(1, 8, 1024, CUS) == 4
    finally:
        lib.db_tune(b"f4_blocks_per_cu", 1)
        lib.db_tune(b"f4_min_tiles", 8)


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,L", [(1, 32, 8, 64), (1, 32, 8, 80), (5, 32, 8, 333),
                                        (20, 32, 8, 777), (3, 8, 8, 2001), (7, 16, 2, 1000),
                                        (36, 64, 8, 257), (9, 4, 4, 1500)])
def test_default_splits_attention(B, Hq, Hkv, L):
    """Against fp64 attention: probabilities and V in fp16 (2^-11 each of
    sum p |v|) and the output rounding, fp32 sums."""
    torch = pytest.importorskip("torch")
    print(f"[f4-splits] B={B} Hq={Hq} Hkv={Hkv} L={L}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(B + L)
    q, K, V = (torch.randn(*s, generator=gen, device="cuda").half()
               for s in ((B, Hq, 128), (B, Hkv, L, 128), (B, Hkv, L, 128)))
    o = ops.f4_flashdecode(q, K, V).double()
    G = Hq // Hkv
    Kt = K.double().transpose(-1, -2).contiguous()
    p = torch.softmax(torch.matmul(q.double().view(B, Hkv, G, 128), Kt) / 128 ** 0.5, dim=-1)
    ref = torch.matmul(p, V.double()).view(B, Hq, 128)
    mag = torch.matmul(p, V.double().abs()).view(B, Hq, 128)
    u = 2.0 ** -11
    # the scores' fp32 sums shift each exponent by at most 128 2^-24 |q||k| / sqrt(128)
    bound = 2 * u * mag + u * ref.abs() + 2.0 ** -13 * mag
    assert ((o - ref).abs() <= bound).all()


@pytest.mark.gpu
def test_a_workspace_for_one_workgroup_per_cu_still_serves():
    """A caller's workspace sized for a workgroup per CU, where the default
    now takes more splits; one too small for that is still refused."""
    torch = pytest.importorskip("torch")
    lib = ops.load_library()
    B, Hq, Hkv, L = 12, 32, 8, 3001
    gen = torch.Generator(device="cuda").manual_seed(1)
    q, K, V = (torch.randn(*s, generator=gen, device="cuda").half()
               for s in ((B, Hq, 128), (B, Hkv, L, 128), (B, Hkv, L, 128)))
    S0 = -(-ops.cu_count() // (B * Hkv))
    assert ops.f4_default_splits(B, Hkv, L) > S0
    need = lib.db_f4_workspace_bytes(B, Hq, Hkv, L, 128, S0)
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    assert torch.equal(ops.f4_flashdecode(q, K, V, workspace=ws),
                       ops.f4_flashdecode(q, K, V, n_splits=S0))
    with pytest.raises(ValueError, match="required"):
        ops.f4_flashdecode(q, K, V, workspace=ws[:need - 256])
