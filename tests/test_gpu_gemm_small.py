"""The few-row GEMM kernel (kernels_gemm_small.hip) against the large tiles, on the GPU.

bf16: every output must have the bits of the large-tile kernel (a pinned tile configuration keeps a
launch there), whatever variant its rule picks: sizes on both sides of the 16-, 32-, 64- and 128-row
tiles, K of one stage, an odd number of stages and more stages than the ring holds, N that a tile does
not divide, and the rule's own upper ends.  fp32: those of the generic kernel.
Rows past M (a guard behind C) must stay untouched.  Whole passes, with the QKV, GeGLU and split-K
epilogues the hook does not reach: one question in an engine pinned to a large tile and in the default
one, and in fp32 alone and inside a batch."""
import numpy as np
import pytest

from layamd_amd import checkpoint as ck
from layamd_amd import engine as le
from layamd_amd import workloads as wl

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1024, 1024), (31, 1024, 64), (33, 72, 192), (64, 8, 128), (65, 4096, 1024), (127, 1024, 2624),
          (129, 768, 1152), (200, 1024, 2624), (255, 5248, 1024), (257, 3072, 768), (513, 1024, 4096),
          (1024, 1024, 1024), (1025, 1024, 2624)]


def _operands(M, N, K, dtype, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    t = torch.bfloat16 if dtype == "bf16" else torch.float32
    A = torch.randn(M, K, generator=g, device="cuda").to(t)
    W = (torch.randn(N, K, generator=g, device="cuda") * 0.02).to(t)
    b = torch.randn(N, generator=g, device="cuda")
    X = torch.randn(M + 8, N, generator=g, device="cuda")
    return A, W, b, X


def _all(lib, A, W, b, X):
    """Plain store, bias + ReLU, bias + GELU, residual with and without bias; 8 guard rows behind each."""
    import torch
    M, N = A.shape[0], W.shape[0]
    out = []
    for bias, act in ((None, 0), (b, 1), (b, 2)):
        C = torch.full((M + 8, N), 7.0, dtype=A.dtype, device="cuda")
        le.gemm(lib, A, W, C, bias=bias, act=act)
        out.append(C)
    for bias in (None, b):
        C = X.clone()
        le.gemm(lib, A, W, C, bias=bias, residual=True)
        out.append(C)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_bf16_bits_of_the_large_tiles(M, N, K):
    import torch
    lib = le.load_library()
    ops = _operands(M, N, K, "bf16", M + N + K)
    prev = le.gemm_config(lib, 3)
    try:
        want = _all(lib, *ops)
        le.gemm_config(lib, -1)
        got = _all(lib, *ops)
    finally:
        le.gemm_config(lib, prev)
    for w, g in zip(want, got):
        assert torch.isfinite(g[:M].float()).all()
        assert torch.equal(w, g)
    assert all((g[M:] == 7.0).all() for g in got[:3]) and torch.equal(got[3][M:], ops[3][M:])


@pytest.mark.parametrize("M,N,K", SHAPES + [(2500, 1024, 1024), (4096, 768, 768)])
def test_fp32_bits_of_the_generic_kernel(M, N, K):
    """An output 4 bytes off its alignment keeps the generic kernel."""
    import torch
    lib = le.load_library()
    A, W, b, X = _operands(M, N, K, "fp32", M + N + K)

    def off(t):
        o = torch.empty(t.numel() + 1, device="cuda")[1:].view(t.shape)
        return o.copy_(t)

    for bias, act, residual in ((None, 0, False), (b, 1, False), (b, 2, False), (None, 0, True), (b, 0, True)):
        start = X if residual else torch.full((M + 8, N), 7.0, device="cuda")
        got, want = start.clone(), off(start)
        assert want.data_ptr() % 16 == 4
        le.gemm(lib, A, W, got, bias=bias, act=act, residual=residual)
        le.gemm(lib, A, W, want, bias=bias, act=act, residual=residual)
        torch.cuda.synchronize()
        assert torch.isfinite(got[:M]).all()
        assert torch.equal(got, want)


@pytest.mark.parametrize("preset,lens", [("large", [16]), ("large", [128]), ("large", [300, 77]), ("large", [512, 400, 333]),
                                         ("base", [41]), ("base", [200, 260])])
def test_bf16_passes_of_a_pinned_engine(preset, lens):
    d = ck.cached_checkpoint(preset, ln_jitter=0.05)
    b = wl.make_batch(ck.PRESETS[preset], lens, [5] * len(lens), seed=len(lens))
    env = {"LAYA_MAX_TOKENS": 4096, "LAYA_GRAPHS": 0}
    want = le.Engine(None, d, precision="bf16", env=dict(env, LAYA_GEMM_CFG=3)).forward_flat(*b.flat())
    got = le.Engine(None, d, precision="bf16", env=env).forward_flat(*b.flat())
    assert np.isfinite(want[0]).all() and np.array_equal(want[0], got[0]) and np.array_equal(want[1], got[1])


# the tile that the rule picks for each of SHAPES, store and residual alike: the smallest whose grid is one
# round of 256 CUs; -1: past the rule's upper end, where the tests above compare the large tiles with themselves
# (fp32: by the load of the busiest CU)
PICKS_BF16 = [0, 0, 0, 0, 2, 0, 0, 1, -1, 3, 3, 3, -1]


def test_rule_takes_the_shapes():
    lib = le.load_library()
    for epi in (0, 1):
        assert [lib.laya_ext_gemm_small_pick(1, epi, M, N, K, 0) for M, N, K in SHAPES] == PICKS_BF16
        assert all(0 <= lib.laya_ext_gemm_small_pick(0, epi, M, N, K, 0) <= 3 for M, N, K in SHAPES)
        assert [lib.laya_ext_gemm_small_pick(1, epi, M, N, K, ks) for M, N, K, ks in SPLITS] == PICKS_SPLIT
    prev = le.gemm_config(lib, 3)
    try:
        assert lib.laya_ext_gemm_small_pick(1, 0, 1, 1024, 1024, 0) == -1
    finally:
        le.gemm_config(lib, prev)


def _all_tile(lib, A, W, b, X, tile, ksplit=0):
    """What _all gives, on one tile of the few-row kernel."""
    import torch
    M, N = A.shape[0], W.shape[0]
    out = [torch.full((M + 8, N), 7.0, dtype=A.dtype, device="cuda") for _ in range(3)] + [X.clone(), X.clone()]
    for C, bias, act, residual in zip(out, (None, b, b, None, b), (0, 1, 2, 0, 0), (False,) * 3 + (True,) * 2):
        le.gemm_small(lib, A, W, C, tile, bias=bias, act=act, residual=residual, ksplit=ksplit)
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("M,N,K", [(1, 72, 64), (31, 1024, 192), (33, 72, 2624), (64, 128, 64), (65, 1024, 1024), (129, 136, 1152),
                                   (513, 1024, 1024)])
def test_every_tile_gives_the_same_bits(M, N, K):
    """Each tile on shapes that it does not divide, whatever the rule would pick: bf16 against the large tiles,
    fp32 against the others (the rule's tile is compared with the generic kernel above)."""
    import torch
    lib = le.load_library()
    for dtype in ("bf16", "fp32"):
        ops = _operands(M, N, K, dtype, M + N + K)
        want = None
        if dtype == "bf16":
            prev = le.gemm_config(lib, 3)
            try:
                want = _all(lib, *ops)
            finally:
                le.gemm_config(lib, prev)
        for v in range(4):
            got = _all_tile(lib, *ops, v)
            want = want or got
            for w, g in zip(want, got):
                assert torch.isfinite(g[:M].float()).all() and torch.equal(w, g), (dtype, v)
            assert all((g[M:] == 7.0).all() for g in got[:3]) and torch.equal(got[3][M:], ops[3][M:])
        for v in (4, 5, -1):                               # 128x64: split-K (and QKV) only
            with pytest.raises(ValueError):
                _all_tile(lib, *ops, v)


SPLITS = [(M, 1024, K, ks) for M in (1, 67, 513, 1025, 2600) for K, ks in ((1024, 8), (4096, 16), (2624, 7), (2624, 11))]
PICKS_SPLIT = [0] * 8 + [3] * 4 + [4] * 8


@pytest.mark.parametrize("M,N,K,ks", SPLITS)
def test_split_k_bits_of_the_workspace_path(M, N, K, ks):
    """Split-K in registers against the slices' reduction (laya_ext_gemm_ksplit): every tile, the 128x64 one in
    more than one round too, chunks of equal length and with a shorter last one (2624: 41 stages in 6 chunks of 6
    and one of 5, or 10 of 4 and one of 1)."""
    import torch
    lib = le.load_library()
    ops = _operands(M, N, K, "bf16", M + K + ks)
    ws = torch.empty(16 << 20, dtype=torch.float32, device="cuda")   # (the engine's 64 MB: several row chunks at M = 2600)
    prev = le.gemm_ksplit(lib, ks, ws)
    try:
        want = _all(lib, *ops)
    finally:
        le.gemm_ksplit(lib, prev)
    for v in range(5):
        got = _all_tile(lib, *ops, v, ks)
        for w, g in zip(want, got):
            assert torch.isfinite(g[:M].float()).all() and torch.equal(w, g), v
        assert all((g[M:] == 7.0).all() for g in got[:3]) and torch.equal(got[3][M:], ops[3][M:])
    # (the split is there: one sum over all of K has other bits)
    assert M == 1 or not torch.equal(want[3], _all_tile(lib, *ops, 3)[3])


def test_fp32_question_alone_and_in_a_batch():
    b = wl.c3(0)
    e = le.Engine(None, ck.cached_checkpoint("large", ln_jitter=0.05), precision="fp32", env={"LAYA_MAX_TOKENS": 16384, "LAYA_GRAPHS": 0})
    logits, act = e.forward_flat(*b.flat())
    at = np.concatenate([[0], np.cumsum(b.nmark)])
    for i in (0, 7, int(np.argmin(b.lens)), int(np.argmax(b.lens))):
        lo, ac = e.forward_flat(*b.subset([i]).flat())
        assert np.array_equal(lo, logits[at[i]:at[i + 1]]) and np.array_equal(ac[0], act[i]), i
