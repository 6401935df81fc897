"""How smx_matmul runs a call (smx_matmul_plan), on the 256 CUs of an MI355X:
whole tiles, K shares, read-ahead workgroups or the streaming kernel. Needs no
GPU; what the plans compute is checked in test_gpu_stream.py and
test_gpu_tail_split.py."""

import ctypes
import os
import subprocess
import sys

import pytest

from strassen_tpu_amd import _lib

CUS = 256


def plan(m, k, n, *, algo=7, bm=None, bn=256, epilogue=None, formula="classical", flags=None, cus=CUS):
    d = _lib.SmxGemmDesc()
    d.m, d.n, d.k, d.lda, d.ldb = m, n, k, k, k
    d.ldc = n // 2 if epilogue in ("swiglu", "geglu") else n
    d.ldr = n
    d.bm, d.bn, d.bk = bm or (256 if m % 256 == 0 else 16), bn, 512
    d.algo, d.epilogue, d.formula = algo, _lib.SMX_EPI[epilogue], _lib.SMX_FORMULA[formula]
    d.a_layout, d.b_layout = _lib.SMX_A_ROWMAJOR, _lib.SMX_B_PACKED
    d.flags = _lib.SMX_FLAG_PRODUCT_MAJOR_ROUNDS if flags is None and algo == 7 else flags or 0
    d.rope_head_dim = 128
    p = _lib.SmxMatmulLaunch()
    _lib.check(_lib.load().smx_matmul_plan(d, _lib.SMX_DTYPE_BF16, 1, cus, ctypes.byref(p)))
    return p


# tile rows x tile columns of 128 x 128 product tiles
@pytest.mark.parametrize("rows,cols", [(1, 100), (1, 196), (2, 80), (2, 100), (3, 70), (4, 50), (64, 3), (100, 2)])
@pytest.mark.parametrize("k", [512, 2048, 5120, 8192])
def test_no_read_ahead_where_the_readers_fall_behind(rows, cols, k):
    """More panels than an eighth of the CUs reads as fast as the tiles take
    them: the readers then only add traffic (1 x 196 at K = 5120: 562 us against 210)."""
    p = plan(256 * rows, k, 256 * cols)
    assert not p.readers


@pytest.mark.parametrize("rows,cols", [(3, 44), (5, 27), (6, 30), (12, 17)])
def test_no_read_ahead_over_half_the_cus_off_the_xcds(rows, cols):
    assert not plan(256 * rows, 5120, 256 * cols).readers


@pytest.mark.parametrize("rows,cols", [(4, 34), (5, 32), (8, 17), (8, 20), (8, 24), (12, 12), (16, 14), (32, 5)])
@pytest.mark.parametrize("k", [1024, 4096, 5120, 8192, 12288])
def test_whole_tiles_with_read_ahead(rows, cols, k):
    p = plan(256 * rows, k, 256 * cols)
    assert (p.streaming, p.whole_tiles, p.split_tiles, p.readers) == (0, rows * cols, 0, CUS // 8)


@pytest.mark.parametrize("rows,cols,k,shares", [(16, 8, 5120, 2), (32, 4, 5120, 2), (32, 4, 8192, 2), (3, 26, 5120, 3),
                                                (5, 16, 5120, 3), (4, 24, 8192, 2), (8, 17, 25600, 3),
                                                (8, 20, 25600, 3)])
def test_shares_that_fit_the_chip_stay(rows, cols, k, shares):
    """Up to half the CUs, where the shares fit one round, and at depths whose
    panels no cache holds."""
    p = plan(256 * rows, k, 256 * cols)
    assert (p.streaming, p.whole_tiles, p.split_tiles, p.readers) == (0, 0, rows * cols, 0) and p.shares >= shares


def test_block_projections_keep_their_shares():
    """k of 8 x 1024 tokens, and the rest of the attention output behind its
    product-major head: 128 tiles in two shares."""
    p = plan(8192, 5120, 1024, bm=1024, bn=1024, epilogue="qk_norm_rope")
    assert (p.head_columns, p.whole_tiles, p.split_tiles, p.shares) == (0, 0, 128, 2)
    p = plan(8192, 8192, 5120, bm=1024, bn=1024, epilogue="residual_add")
    assert (p.head_columns, p.whole_tiles, p.split_tiles, p.shares) == (8, 0, 128, 2)


@pytest.mark.parametrize("algo", [7, 8])
@pytest.mark.parametrize("cus", [64, 228, 256, 304])
def test_plans_cover_the_call(algo, cus):
    for m in (16, 48, 96, 144, 256, 272, 512, 1808, 2048, 8192):
        for n in (256, 1024, 5120, 13824, 25600):
            for k in (512, 2048, 5120, 25600):
                p = plan(m, k, n, algo=algo, cus=cus)
                rows, cols = -(-(m // 2) // p.tile_rows), n // 2 // p.tile_cols
                assert p.whole_tiles + p.split_tiles + rows * 2 * p.head_columns == rows * cols
                assert 1 <= p.shares <= 16 and (p.shares > 1) == (p.split_tiles > 0)
                assert k // 32 >= (8 if p.streaming else 16) * p.shares or p.shares == 1
                assert p.readers == 0 or rows * cols + p.readers <= cus
                if algo == 8:
                    assert not p.readers and not p.head_columns


def test_streaming_tests_reach_every_tiling():
    """The calls of test_gpu_stream.py run on the streaming kernel, and its
    tilings are all those that a grid of calls gets, each with K in one share
    and in several."""
    import test_gpu_stream as g

    for algo, (m, k, n), tiling in g.TILINGS:
        p = plan(m, k, n, algo=algo, bm=16)
        assert p.streaming and (p.tile_rows, p.tile_cols, p.shares) == tiling
    key = lambda algo, m, rows, cols, shares: (algo, rows, cols, m // 2 <= rows, shares > 1)  # noqa: E731
    tested = {key(algo, m, *tiling) for algo, (m, _, _), tiling in g.TILINGS}
    for algo in (7, 8):
        for m in (16, 64, 80, 128, 144, 256, 272, 1024):
            for n in [256, 512, 1024, 1536, 2816, 4352, 5120, 8192, 12288, 17664, 25600, 33792, 51200]:
                for k in (512, 1024, 2048, 4608, 10240, 25600):
                    p = plan(m, k, n, algo=algo, bm=16)
                    if p.streaming:
                        assert key(algo, m, p.tile_rows, p.tile_cols, p.shares) in tested, (algo, m, k, n)
    for algo in (7, 8):
        for (m, k, n), (bm, bn, _) in g.SHAPES:
            assert plan(m, k, n, algo=algo, bm=bm, bn=bn).streaming
        for m, k, n, bm in ((48, 4608, 512, 16), (272, 512, 512, 272)):
            for epilogue in ("swiglu", "geglu", "residual_add", "bias_add"):
                assert plan(m, k, n, algo=algo, bm=bm, epilogue=epilogue).streaming
        assert plan(48, 2048, 1024, algo=algo, bm=16, epilogue="qk_norm_rope").streaming
    for m, k in ((16, 512), (272, 4608)):
        for formula in _lib.SMX_FORMULA:
            assert plan(m, k, 512, bm=m, formula=formula).streaming


def test_tail_split_off_keeps_every_tile_whole():
    """SMX_TAIL_SPLIT=0 (read once per process): no kernel divides K."""
    script = """
import test_matmul_plan as t
for algo in (7, 8):
    for m in (16, 80, 256, 1024, 2048):
        for n in (256, 5120, 17664):
            for k in (512, 4608, 25600):
                p = t.plan(m, k, n, algo=algo)
                assert p.shares == 1 and p.split_tiles == 0, (algo, m, k, n)
"""
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, SMX_TAIL_SPLIT="0",
               PYTHONPATH=os.pathsep.join([here, os.path.dirname(here), os.environ.get("PYTHONPATH", "")]))
    subprocess.run([sys.executable, "-c", script], env=env, check=True)


@pytest.mark.parametrize("algo", [7, 8])
def test_recorded_shares_are_those_of_the_call(algo):
    """On the streaming kernel too, whose shares differ from smx_gemm's (12 here)."""
    for m, k, n in ((16, 25600, 5120), (256, 25600, 5120), (8192, 5120, 5120)):
        bm = min(m, 256)
        assert _lib.k_shares(m, k, n, (bm, 256, 512), algo, CUS) == plan(m, k, n, algo=algo, bm=bm).shares
    assert _lib.k_shares(16, 25600, 5120, (16, 256, 512), algo, CUS) == 6


def test_plan_checks_its_arguments():
    lib, d = _lib.load(), _lib.SmxGemmDesc()
    p = _lib.SmxMatmulLaunch()
    assert lib.smx_matmul_plan(d, 0, 1, CUS, None) == _lib.SMX_ERR_INVALID
    assert lib.smx_matmul_plan(None, 0, 1, CUS, ctypes.byref(p)) == _lib.SMX_ERR_INVALID
    assert lib.smx_matmul_plan(d, 0, 1, -1, ctypes.byref(p)) == _lib.SMX_ERR_INVALID
    assert lib.smx_matmul_plan(d, 0, 1, CUS, ctypes.byref(p)) == _lib.SMX_ERR_UNSUPPORTED  # an unpacked B
