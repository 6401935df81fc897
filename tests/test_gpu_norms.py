"""GPU row norms (smx_rms_norm, smx_norm_residual_add's chunked pass) against
their FP32 definition, at widths below, at and past what a workgroup keeps in
registers, and the block's attention against its head-by-head layout."""

import pytest
import torch

import strassen_tpu_amd.qwen3_block as qb
from strassen_tpu_amd import _lib
from test_gpu_parity import DEV, say

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _announce(request):
    say(f"\n[gpu] {request.node.nodeid}")
    yield
    torch.cuda.synchronize()


def _ulp_close(got, want):
    """Within one bf16 ulp: FP32 sums of n squares in another order differ by
    under n 2^-24, far below half an ulp (2^-9)."""
    assert ((got.double() - want).abs() <= want.abs() * 2.0 ** -7 + 1e-30).all()


@pytest.mark.parametrize("m,n", [(1, 8), (3, 2040), (5, 5120), (2, 8192), (2, 8200), (1, 25600)])
@pytest.mark.parametrize("scale_dtype", [torch.bfloat16, torch.float32])
def test_rms_norm(m, n, scale_dtype):
    g = torch.Generator(device=DEV).manual_seed(n)
    x = (torch.randn(m, n, device=DEV, generator=g) * 3).to(torch.bfloat16)
    scale = torch.randn(n, device=DEV, generator=g).to(scale_dtype)
    x64 = x.double()
    want = x64 * torch.rsqrt(x64.square().mean(-1, keepdim=True) + 1e-6) * scale.double()
    _ulp_close(qb._row_rms_norm(x, scale, 1e-6), want)
    _ulp_close(qb.rms_norm(x, scale, 1e-6), want)


@pytest.mark.parametrize("m,n", [(1, 8), (3, 2040), (64, 5120), (2, 8200), (8192, 5120), (1, 25600)])
@pytest.mark.parametrize("scale_dtype", [torch.bfloat16, torch.float32])
def test_block_norm_has_the_bits_of_the_torch_form(m, n, scale_dtype):
    """Rows over 40 binades, zero rows, and rows with an infinity or a NaN."""
    g = torch.Generator(device=DEV).manual_seed(m + n)
    x = torch.randn(m, n, device=DEV, generator=g) * torch.exp2(torch.rand(m, 1, device=DEV, generator=g) * 40 - 20)
    for row, value in ((1, 0.0), (2, float("inf")), (3, float("nan"))):
        if row < m:
            x[row, slice(None) if value == 0 else n // 2] = value
    x = x.to(torch.bfloat16)
    scale = torch.randn(n, device=DEV, generator=g).to(scale_dtype)
    got, want = qb._row_rms_norm(x, scale, 1e-6), qb.rms_norm(x, scale, 1e-6)
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got[~got.isnan()], want[~want.isnan()])


def test_block_norm_records_gradients():
    x = torch.randn(4, 128, device=DEV).to(torch.bfloat16).requires_grad_()
    scale = torch.randn(128, device=DEV).to(torch.bfloat16)
    qb._row_rms_norm(x, scale, 1e-6).float().sum().backward()
    assert x.grad is not None


def test_rms_norm_in_one_pass():
    """smx_rms_norm itself, rows apart and at widths past the registers."""
    for n in (2040, 8200):
        x = torch.randn(3, n + 8, device=DEV).to(torch.bfloat16)[:, :n]
        scale, out = torch.randn(n, device=DEV), torch.empty(3, n, dtype=torch.bfloat16, device=DEV)
        _lib.check(_lib.load().smx_rms_norm(3, n, x.data_ptr(), x.stride(0), scale.data_ptr(), _lib.SMX_NRA_SCALE_F32,
                                            1e-6, out.data_ptr(), n, torch.cuda.current_stream(DEV).cuda_stream))
        x64 = x.double()
        _ulp_close(out, x64 * torch.rsqrt(x64.square().mean(-1, keepdim=True) + 1e-6) * scale.double())


def test_rms_norm_keeps_other_layouts():
    """Widths and views that are not whole 16-byte chunks take the torch form."""
    x = torch.randn(4, 100, device=DEV).to(torch.bfloat16)
    scale = torch.randn(100, device=DEV).to(torch.bfloat16)
    assert torch.equal(qb._row_rms_norm(x, scale, 1e-6), qb.rms_norm(x, scale, 1e-6))
    wide = torch.randn(4, 130, device=DEV).to(torch.bfloat16)[:, 1:129]
    scale = torch.randn(128, device=DEV).to(torch.bfloat16)
    assert torch.equal(qb._row_rms_norm(wide, scale, 1e-6), qb.rms_norm(wide, scale, 1e-6))


# chunked rows, and rows that are not (odd width, odd stride)
@pytest.mark.parametrize("m,n,pad", [(3, 256, 0), (2, 8192, 0), (2, 8448, 8), (3, 250, 0), (3, 256, 1)])
@pytest.mark.parametrize("f32", [False, True])
def test_norm_residual_add(m, n, pad, f32):
    g = torch.Generator(device=DEV).manual_seed(n + pad)
    dtype = torch.float32 if f32 else torch.bfloat16
    x = torch.randn(m, n + pad, device=DEV, generator=g)[:, :n]
    residual = torch.randn(m, n + pad, device=DEV, generator=g).to(dtype)[:, :n]
    scale = torch.randn(n, device=DEV, generator=g).to(dtype)
    out = torch.empty(m, n, device=DEV, dtype=dtype)
    bits = _lib.SMX_NRA_SCALE_F32 | _lib.SMX_NRA_RESIDUAL_F32 | _lib.SMX_NRA_OUT_F32 if f32 else 0
    _lib.check(_lib.load().smx_norm_residual_add(
        m, n, x.data_ptr(), x.stride(0), residual.data_ptr(), residual.stride(0), scale.data_ptr(), bits, 1e-6,
        out.data_ptr(), out.stride(0), torch.cuda.current_stream(DEV).cuda_stream))
    x64 = x.double()
    product = x64 * torch.rsqrt(x64.square().mean(-1, keepdim=True) + 1e-6) * scale.double()
    want = product + residual.double()
    # one rounding of the result, FP32 rounding of its terms
    eps = 2.0 ** -23 if f32 else 2.0 ** -8
    bound = want.abs() * eps + (product.abs() + residual.double().abs()) * 2.0 ** -20
    assert ((out.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("heads,kv", [(8, 8), (16, 2)])
def test_attention_reads_heads_in_place(heads, kv):
    g = torch.Generator(device=DEV).manual_seed(1)
    q, k, v = (torch.randn(2, 256, h, 128, device=DEV, generator=g).to(torch.bfloat16) for h in (heads, kv, kv))
    with torch.enable_grad():
        want = qb.attention(q.detach().requires_grad_(), k, v).detach()  # laid out and repeated
    assert torch.equal(qb.attention(q, k, v), want)


@pytest.mark.parametrize("offset,pad", [(0, 8), (8, 0), (1, 7), (0, 1)])
def test_attention_on_views(offset, pad):
    """Heads inside wider rows: read in place where their rows are aligned, laid
    out first where they are not, with the same bits."""
    g = torch.Generator(device=DEV).manual_seed(2)
    q, k, v = (torch.randn(2, 128, h, 128 + offset + pad, device=DEV, generator=g).to(torch.bfloat16)
               [..., offset:offset + 128] for h in (8, 2, 2))
    want = qb.attention(*(t.contiguous() for t in (q, k, v)))
    assert torch.equal(qb.attention(q, k, v), want)


def test_attention_under_transforms():
    """Batched by vmap and traced, with the bits of the plain call."""
    from torch.fx.experimental.proxy_tensor import make_fx

    g = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.randn(3, 2, 64, h, 128, device=DEV, generator=g).to(torch.bfloat16) for h in (8, 2, 2))
    want = torch.stack([qb.attention(*t) for t in zip(q, k, v)])
    assert torch.equal(torch.vmap(qb.attention)(q, k, v), want)
    traced = make_fx(qb.attention, tracing_mode="fake")(q[0], k[0], v[0])
    # the traced call lays out what it is given: rows that are not 16-byte aligned too
    odd = [torch.nn.functional.pad(t[1], (1, 7))[..., 1:129] for t in (q, k, v)]
    assert torch.equal(traced(*odd), want[1])
