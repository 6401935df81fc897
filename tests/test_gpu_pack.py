"""GPU packing kernels at their edges: row-major and transposed sources of
both operands pack to the same bytes, for every source type, number of
passes, panel map and block permutation, with K below, at and past a
workgroup's stages and rows that pad the last product tile. (The layout
itself is pinned against the oracle in test_gpu_parity and test_gpu_thin.)
"""

import numpy as np
import pytest
import torch

import oracle as o
import strassen_tpu_amd as smx
from strassen_tpu_amd.packing import ExactSchedule, pack_operand
from test_gpu_parity import DEV, host, say

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    say(f"\n[gpu] {request.node.nodeid}")
    yield
    torch.cuda.synchronize()


def _source(rows, k, dtype, seed=3):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randn(rows, k, device=DEV, generator=g).to(dtype)


# K of 64 (two stages), 320 (ten: a group of eight and a part) and 1536
@pytest.mark.parametrize("k,bk", [(64, 64), (320, 64), (1536, 512)])
@pytest.mark.parametrize("dtype,precision", [(torch.bfloat16, None), (torch.float32, None), (torch.float32, "high"),
                                             (torch.float32, "highest")])
@pytest.mark.parametrize("algo,perm", [(7, 0), (7, 6), (8, 0)])
def test_row_major_right_operand_packs_as_the_transposed_one(algo, perm, dtype, precision, k, bk):
    n = 768
    b = _source(n, k, dtype).t()  # [K, N], K contiguous
    kw = dict(algo=algo, side="rhs", tile_rows=256, bk=bk, block_permutation=perm, dot_precision=precision)
    want = pack_operand(b, **kw)
    got = pack_operand(b.contiguous(), **kw)  # row-major
    assert torch.equal(got.data.view(torch.int16), want.data.view(torch.int16)) and got.shape == want.shape
    if algo == 7 and not perm:
        expected = o.packed_operand(host(b.float()), 7, "rhs", 256, bk, **(
            {} if dtype == torch.bfloat16 else dict(input_dtype="float32", **(
                {} if precision is None else dict(dot_precision=precision)))))
        assert np.array_equal(host(want.data), expected)


@pytest.mark.parametrize("ld_pad", [0, 8, 3])
@pytest.mark.parametrize("m,bm", [(16, 16), (144, 48), (512, 256)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_transposed_left_operand_with_any_row_stride(dtype, m, bm, ld_pad):
    """Row strides that are not whole 128-byte lines take the gathering kernel,
    the others the one that moves 16-byte chunks."""
    k = 576
    a = _source(m, k, dtype)
    wide = torch.zeros(k, m + ld_pad, dtype=dtype, device=DEV)
    wide[:, :m] = a.t()
    kw = dict(algo=7, tile_rows=bm, bk=64)
    want = pack_operand(a, side="lhs", **kw)
    got = pack_operand(wide[:, :m], side="lhs_t", **kw)
    assert torch.equal(got.data.view(torch.int16), want.data.view(torch.int16))


@pytest.mark.parametrize("algo", [7, 8])
@pytest.mark.parametrize("m,bm,ld", [(16, 16, 64), (144, 48, 192), (512, 256, 512), (512, 256, 576)])
def test_transposed_left_operand_in_whole_lines(algo, m, bm, ld):
    """Row strides of whole 128-byte lines, which the 16-byte-chunk kernel
    takes, with padding rows in the last product tile."""
    a = _source(m, 576, torch.bfloat16)
    wide = torch.zeros(576, ld, dtype=torch.bfloat16, device=DEV)
    wide[:, :m] = a.t()
    kw = dict(algo=algo, tile_rows=bm, bk=64)
    want, got = pack_operand(a, side="lhs", **kw), pack_operand(wide[:, :m], side="lhs_t", **kw)
    assert torch.equal(got.data.view(torch.int16), want.data.view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_exact_panels_of_a_row_major_right_operand(dtype):
    b = _source(512, 2048, dtype).t()
    schedule = ExactSchedule(4, (0, 2))
    kw = dict(algo=7, side="rhs", tile_rows=256, bk=512, panel_schedule=schedule)
    want, got = pack_operand(b, **kw), pack_operand(b.contiguous(), **kw)
    for part in ("ordinary", "exact"):
        assert torch.equal(getattr(got, part).data.view(torch.int16), getattr(want, part).data.view(torch.int16))


def test_views_that_cannot_be_read_in_place_pack_alike():
    """A row-major view whose rows are not 16-byte aligned, and one of a
    wider matrix whose rows are."""
    b = _source(256, 512, torch.bfloat16).t()
    want = smx.strassen_weight_layout(b, 256, 512)
    for pad, offset in ((4, 0), (8, 8), (8, 1)):
        wide = torch.zeros(512, 256 + 2 * pad, dtype=torch.bfloat16, device=DEV)
        view = wide[:, offset:offset + 256]
        view.copy_(b)
        got = smx.strassen_weight_layout(view, 256, 512)
        assert torch.equal(got.data.view(torch.int16), want.data.view(torch.int16))
