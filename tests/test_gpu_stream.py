"""GPU parity of the streaming kernel (kernel_stream.hpp), which smx_matmul runs
on launches of few product rows or few tiles: every tiling it has, with K in
one share and in several, and its edges (padding rows, the last columns),
against exact integer products, and every epilogue, formula and block
permutation against the 128 x 128 tile kernels (smx_gemm on the same
operands) within one bf16 ulp. That these calls run on it is checked in
test_matmul_plan.py.
"""

import ctypes

import numpy as np
import pytest
import torch

import oracle as o
import strassen_tpu_amd as smx
from strassen_tpu_amd import _lib
from test_gpu_parity import DEV, _qk_problem, assert_ulp_close, dev, dev_weight, host, say
from test_gpu_tail_split import _pack, _problem, abi_gemm
from test_matmul_plan import plan as launch_plan

pytestmark = pytest.mark.gpu

# (m, k, n), tile: product rows M/2 of 8 and 32 (one 32-row block, the second
# with more columns than 256 tiles of 64), 40, 64, 72, 128 and 136 (padding rows
# in the last tile row) and 512.
SHAPES = [
    ((16, 512, 256), (16, 256, 512)),
    ((64, 4608, 1024), (64, 512, 512)),
    ((64, 512, 34816), (16, 512, 512)),
    ((80, 3072, 512), (16, 256, 512)),
    ((128, 512, 34816), (128, 512, 512)),
    ((144, 2560, 256), (48, 256, 512)),
    ((256, 512, 768), (256, 256, 512)),
    ((272, 1024, 512), (272, 256, 512)),
    ((1024, 1024, 1024), (1024, 1024, 512)),
]


# algo, (m, k, n), the tiling that 256 CUs get: product rows and columns per
# workgroup, shares of K. One tile row (M/2 up to the tile's rows) loads B past
# the L2, several read it through. Row tiles of 16: M/2 of 8, 40 and 72 leaves
# padding rows in the last 32-row block, and in the second of a tile of two.
TILINGS = [
    (7, (16, 512, 256), (32, 64, 2)), (7, (16, 512, 17664), (32, 64, 1)),
    (7, (16, 3072, 17664), (32, 128, 3)), (7, (16, 512, 33792), (32, 128, 1)),
    (7, (80, 2048, 2816), (64, 64, 8)), (7, (80, 512, 17664), (64, 64, 1)),
    (7, (80, 1536, 17664), (64, 128, 3)), (7, (80, 512, 33792), (64, 128, 1)),
    (7, (80, 512, 256), (32, 32, 2)), (7, (80, 512, 4352), (32, 32, 1)),
    (7, (144, 2048, 1536), (64, 64, 8)), (7, (144, 512, 12288), (64, 64, 1)),
    (8, (16, 512, 256), (32, 64, 2)), (8, (16, 512, 17664), (32, 64, 1)),
    (8, (16, 1024, 12288), (32, 128, 4)), (8, (16, 512, 33792), (32, 128, 1)),
    (8, (80, 2048, 2816), (64, 64, 8)), (8, (80, 512, 17664), (64, 64, 1)),
    (8, (80, 512, 256), (32, 32, 2)), (8, (80, 512, 4352), (32, 32, 1)),
    (8, (144, 1536, 2048), (64, 64, 6)), (8, (144, 512, 12288), (64, 64, 1)),
]


@pytest.fixture(autouse=True)
def _announce(request):
    say(f"\n[gpu] {request.node.nodeid}")
    yield
    torch.cuda.synchronize()


def _call(algo, a, b, tile, **kw):
    fn = smx.strassen_matmul if algo == 7 else smx.cubic_matmul
    return fn(a, b, bm=tile[0], bn=tile[1], bk=tile[2], **kw)


@pytest.mark.parametrize("algo", [7, 8])
@pytest.mark.parametrize("shape,tile", SHAPES)
def test_integer_products_are_exact(algo, shape, tile):
    """Operand sums and FP32 sums of small integers are exact, so any fragment
    missed, repeated or misplaced shows."""
    m, k, n = shape
    rng = np.random.default_rng(m + n)
    a = rng.integers(-2, 3, (m, k)).astype(np.float32)
    b = rng.integers(-2, 3, (k, n)).astype(np.float32)
    pa, pb = _pack(algo, a, b, tile)
    want = torch.from_numpy(a).to(DEV).double() @ torch.from_numpy(b).to(DEV).double()
    for left in (dev(a), pa):  # packed by the call, and packed before it
        got = _call(algo, left, pb, tile, output_dtype=torch.float32)
        assert torch.equal(got.double(), want)


@pytest.mark.parametrize("algo,shape,tiling", TILINGS)
def test_every_tiling_is_exact(algo, shape, tiling):
    m, k, n = shape
    plan = launch_plan(m, k, n, algo=algo, bm=16, cus=0)  # this device's
    if torch.cuda.get_device_properties(DEV).multi_processor_count == 256:
        assert plan.streaming and (plan.tile_rows, plan.tile_cols, plan.shares) == tiling
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a = torch.randint(-2, 3, (m, k), device=DEV, generator=g).to(torch.bfloat16)
    b = torch.randint(-2, 3, (n, k), device=DEV, generator=g).to(torch.bfloat16).t()
    want = a.double() @ b.double()
    layout = smx.strassen_weight_layout if algo == 7 else smx.cubic_weight_layout
    got = _call(algo, a, layout(b, 256, 512), (16, 256, 512), output_dtype=torch.float32)
    assert torch.equal(got.double(), want)


@pytest.mark.parametrize("epilogue", ["swiglu", "geglu", "residual_add", "bias_add"])
@pytest.mark.parametrize("shape,tile", [((48, 4608, 512), (16, 256, 512)), ((272, 512, 512), (272, 256, 512))])
@pytest.mark.parametrize("algo", [7, 8])
def test_epilogues_match_the_tile_kernels(algo, shape, tile, epilogue):
    m, k, n = shape
    rng, a, b = _problem(7 + algo, m, k, n)
    aux = {}
    if epilogue == "residual_add":
        aux["residual"] = dev(o.bf16_round(rng.standard_normal((m, n)).astype(np.float32)))
    elif epilogue == "bias_add":
        aux["bias"] = dev(o.bf16_round(rng.standard_normal(n).astype(np.float32)))
    pa, pb = _pack(algo, a, b, tile)
    want, _ = abi_gemm(algo, pa, pb, m, n, k, tile, epilogue, workspace=True, **aux)
    got = host(_call(algo, dev(a), pb, tile, epilogue=epilogue, **aux))
    assert_ulp_close(got, host(want), k=k)
    # float32 epilogue operands
    aux32 = {key: v.float() for key, v in aux.items()}
    assert_ulp_close(host(_call(algo, pa, pb, tile, epilogue=epilogue, **aux32)), got, k=k)


@pytest.mark.parametrize("algo", [7, 8])
def test_qk_norm_rope_matches_the_tile_kernels(algo):
    batch, seq, heads, k, bn = 1, 48, 8, 2048, 256
    m, n, tile = batch * seq, heads * 128, (16, bn, 512)
    x, w, laid, tcos, tsin, scale = _qk_problem(17, batch, seq, heads, k, bn)
    pa, pb = _pack(algo, x, laid, tile)
    rope = (dev(tcos), dev(tsin), torch.from_numpy(scale).to(DEV).to(torch.bfloat16))
    want, _ = abi_gemm(algo, pa, pb, m, n, k, tile, "qk_norm_rope", workspace=True, rope=rope)
    got = _call(algo, dev(x), pb, tile, epilogue="qk_norm_rope", rope_cos=rope[0], rope_sin=rope[1],
                rope_scale=rope[2], rope_eps=1e-6)
    assert_ulp_close(host(got), host(want), k=k)


@pytest.mark.parametrize("formula", ["classical", "dual", "powers"])
@pytest.mark.parametrize("perm", range(8))
@pytest.mark.parametrize("m,k", [(16, 512), (272, 4608)])
def test_formulas_and_permutations_are_exact(m, k, formula, perm):
    n, tile = 512, (m, 256, 512)
    rng = np.random.default_rng(perm)
    a = rng.integers(-2, 3, (m, k)).astype(np.float32) * 4  # the powers formula halves and quarters
    b = rng.integers(-2, 3, (k, n)).astype(np.float32) * 4
    w = smx.strassen_weight_layout(dev_weight(b), 256, 512, formula_variant=formula, block_permutation=perm)
    got = _call(7, dev(a), w, tile, formula_variant=formula, block_permutation=perm, output_dtype=torch.float32)
    assert np.array_equal(host(got), a @ b)


def test_matmul_checks_its_arguments():
    """smx_matmul refuses a short workspace, an unpacked B and bad layouts
    before it launches anything."""
    lib, tile, (m, k, n) = _lib.load(), (16, 256, 512), (16, 5120, 1024)
    _, a, b = _problem(3, m, k, n)
    _, pb = _pack(7, a, b, tile)
    a_dev, c = dev(a), torch.full((m, n), 7.0, dtype=torch.bfloat16, device=DEV)
    d = _lib.SmxGemmDesc()
    d.m, d.n, d.k, d.lda, d.ldb, d.ldc = m, n, k, k, k, n
    d.bm, d.bn, d.bk = tile
    d.algo, d.a_layout, d.b_layout = 7, _lib.SMX_A_ROWMAJOR, _lib.SMX_B_PACKED
    d.flags, d.rope_head_dim, d.rope_eps = _lib.SMX_FLAG_PRODUCT_MAJOR_ROUNDS, 128, 1e-6
    need = ctypes.c_int64()
    _lib.check(lib.smx_matmul_workspace_bytes(d, _lib.SMX_DTYPE_BF16, 1, ctypes.byref(need)))
    assert need.value > smx.packing.packed_bytes(7, m, k)  # the packed A, then the FP32 shares
    ws = torch.empty(need.value, dtype=torch.uint8, device=DEV)
    args = (a_dev.data_ptr(), pb.data.data_ptr(), c.data_ptr(), None, None, None, None, None,
            torch.cuda.current_stream(DEV).cuda_stream)
    d.workspace, d.workspace_bytes = ws.data_ptr(), need.value - 16
    assert lib.smx_matmul(d, 0, 1, *args) == _lib.SMX_ERR_INVALID and "workspace" in _lib.last_error()
    d.workspace_bytes = need.value
    assert lib.smx_matmul(d, 2, 1, *args) == _lib.SMX_ERR_INVALID
    assert lib.smx_matmul(d, 0, 2, *args) == _lib.SMX_ERR_INVALID
    d.a_layout = 5
    assert lib.smx_matmul(d, 0, 1, *args) == _lib.SMX_ERR_INVALID
    d.a_layout, d.b_layout = _lib.SMX_A_ROWMAJOR, _lib.SMX_B_KCONTIG
    assert lib.smx_matmul(d, 0, 1, *args) == _lib.SMX_ERR_UNSUPPORTED
    torch.cuda.synchronize()
    assert (c == 7.0).all()
