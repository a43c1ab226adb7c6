"""Row L2 norm kernels: the row-group form (rows of 64, 128, 256 at 16-byte
aligned pointers) and the general one, against float64.

Bounds: the outputs are rounded once to the dtype (half a unit: 2^-9 bf16,
2^-12 fp16 of the value) after fp32 arithmetic over at most 256 products;
doubled here, with 1e-6 for float32."""

import pytest
import torch

pytestmark = pytest.mark.gpu

BOUND = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 1e-6}


def _at(x, shift):
    """x's values at an address `shift` elements past a 16-byte boundary."""
    buf = torch.empty(x.numel() + 16, dtype=x.dtype, device="cuda")
    v = buf[shift:shift + x.numel()].view(x.shape)
    v.copy_(x)
    return v


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,d,shift", [(1, 64, 0), (127, 64, 0), (129, 64, 0), (5, 128, 0), (65, 128, 0), (33, 256, 0),
                                       (31, 64, 1), (31, 128, 3), (7, 96, 0), (9, 512, 0)])
def test_l2norm_fwd_bwd(n, d, shift, dtype):
    from linatt_amd.delta_rule import l2norm
    g = torch.Generator().manual_seed(n * 1000 + d)
    x = _at(torch.randn(n, d, generator=g).to(dtype), shift).requires_grad_(True)
    dy = _at(torch.randn(n, d, generator=g).to(dtype), shift)
    y = l2norm(x, 1e-6)
    dx, = torch.autograd.grad(y, x, dy)
    xr = x.detach().double()
    r = torch.rsqrt((xr * xr).sum(-1, keepdim=True) + 1e-6)
    assert (y.double() - xr * r).abs().max() <= BOUND[dtype] * (xr * r).abs().max()
    # the backward starts from the stored (rounded) y
    yr, gr = y.detach().double(), dy.double()
    ref = r * (gr - yr * (yr * gr).sum(-1, keepdim=True))
    assert (dx.double() - ref).abs().max() <= BOUND[dtype] * ref.abs().max()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("n,d", [(1, 64), (6000, 64), (3001, 128), (1501, 256)])
def test_l2norm_bits_independent_of_alignment(n, d, dtype):
    """The row-group kernels keep the general kernel's summation order: the
    same values at 16-byte aligned and at other addresses give the same bits."""
    from linatt_amd.delta_rule import l2norm
    g = torch.Generator().manual_seed(n + d)
    x, dy = (torch.randn(n, d, generator=g).to(dtype) for _ in range(2))
    out = []
    for shift in (0, 1):
        xs = _at(x, shift).requires_grad_(True)
        y = l2norm(xs, 1e-6)
        out.append((y, *torch.autograd.grad(y, xs, _at(dy, shift))))
    for a, b in zip(*out):
        assert torch.equal(a, b)


@pytest.mark.parametrize("d", [64, 128, 256])
def test_l2norm_float32_outputs_at_16_mod_32(d):
    """float32 outputs at addresses that are 16-byte but not 32-byte aligned
    take the row-group kernels too: the same bits as at 32-byte aligned ones,
    and nothing outside them is written."""
    from linatt_amd import _lib
    L, p, n = _lib.load(), _lib.ptr, 67
    g = torch.Generator().manual_seed(d)
    x, dy = (torch.randn(n, d, generator=g).cuda() for _ in range(2))
    out, sp = [], _lib.stream_of(x)
    for off in (8, 4):
        bufs = [torch.full((n * d + 16,), float("nan"), device="cuda") for _ in range(2)]
        assert all(b.data_ptr() % 32 == 0 for b in bufs)
        y, dx = (b[off:off + n * d].view(n, d) for b in bufs)
        rstd = torch.empty(n, device="cuda")
        _lib.check("fwd", L.linatt_l2norm_fwd(p(x), p(y), p(rstd), n, d, 1e-6, 0, sp))
        _lib.check("bwd", L.linatt_l2norm_bwd(p(y), p(rstd), p(dy), p(dx), n, d, 0, sp))
        for b in bufs:
            assert b[:off].isnan().all() and b[off + n * d:].isnan().all() and not b[off:off + n * d].isnan().any()
        out.append((y, rstd, dx))
    for a, b in zip(*out):
        assert torch.equal(a, b)
