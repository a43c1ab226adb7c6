"""The forward with its key tiles split over workgroups
(``linatt_kata_fwd_split``) against the unsplit call on the same inputs, at
the sizes where the split engages, with ragged last tiles.

Bounds: both sum the same non-negative weights (den) and the same products
(o) in float32, n <= T terms in two orders, so den agrees to 2 T 2^-24 of
itself and o den to 2 T 2^-24 max|v| den; o is then rounded to the dtype (one
spacing, 2^-7 bf16, 2^-10 fp16, 2^-23 fp32, of its value).  fp16 rounds the
weights after a row scale that follows each piece's own maximum: up to one
fp16 spacing of each weight, 2^-10 of max|v| in o and of den."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu
SPACING = {torch.bfloat16: 2.0 ** -7, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -23}


@pytest.mark.parametrize("B,T,HQ,H,dk,M,variant,decay,dtype", [
    (1, 300, 2, 2, 64, 4, "concat", False, torch.float32), (1, 512, 4, 2, 64, 2, "sum", False, torch.float32),
    (1, 257, 1, 1, 128, 2, "concat", True, torch.float32), (1, 1985, 2, 1, 64, 2, "concat", False, torch.float16),
    (1, 2049, 3, 3, 64, 4, "sum", False, torch.bfloat16), (2, 2500, 4, 2, 64, 4, "concat", False, torch.bfloat16),
    (1, 3000, 2, 2, 64, 1, "concat", False, torch.bfloat16), (1, 1900, 4, 4, 128, 2, "concat", True, torch.bfloat16),
    (1, 3100, 2, 2, 64, 2, "concat", True, torch.float16), (1, 2100, 2, 2, 128, 2, "sum", False, torch.float16)])
def test_split_forward_equals_unsplit(B, T, HQ, H, dk, M, variant, decay, dtype):
    from linatt_amd import _lib
    print(f"\nsplit forward B{B} T{T} HQ{HQ} H{H} dk{dk} M{M} {variant} decay={decay} {dtype}", flush=True)
    L, p = _lib.load(), _lib.ptr
    g = torch.Generator().manual_seed(T + dk)
    q = torch.randn(B, T, HQ, dk, generator=g).to(dtype).cuda()
    k = torch.randn(B, T, H, dk, generator=g).to(dtype).cuda()
    v = torch.randn(B, T, H, 64, generator=g).to(dtype).cuda()
    c = (-torch.rand(B, T, HQ, generator=g) * 0.05).cumsum(1).cuda() if decay else None
    var, code = int(variant == "sum"), _lib.dtype_code(dtype)
    shape = (B, T, HQ, H, dk, 64, M)
    nws = L.linatt_kata_fwd_workspace_bytes(*shape, var, int(decay), code)
    assert nws > 0
    ws = torch.empty(nws, device="cuda", dtype=torch.uint8)
    out = []
    for split in (False, True):
        o = torch.full((B, T, HQ, 64), float("nan"), device="cuda", dtype=dtype)
        den = torch.full((B, T, HQ), float("nan"), device="cuda")
        head, tail = (p(q), p(k), p(v), p(c), p(o), p(den)), (*shape, 1 / math.sqrt(dk // M), var, code, _lib.stream_of(q))
        if split:
            _lib.check("split", L.linatt_kata_fwd_split(*head, p(ws), nws, *tail))
        else:
            _lib.check("fwd", L.linatt_kata_fwd(*head, *tail))
        out.append((o.double(), den.double()))
    torch.cuda.synchronize()
    (o1, d1), (o2, d2) = out
    acc = 2 * T * 2.0 ** -24 + (2.0 ** -10 if dtype == torch.float16 else 0.0)
    assert ((d1 - d2).abs() <= acc * d1).all()
    # o = (o den) / den: both sums' error
    assert ((o1 - o2).abs() <= SPACING[dtype] * o1.abs() + 2 * acc * v.double().abs().max()).all()


def test_split_forward_workspace_checked():
    from linatt_amd import _lib
    L, p = _lib.load(), _lib.ptr
    x = torch.zeros(1, 512, 4, 64, device="cuda")
    den = torch.zeros(1, 512, 4, device="cuda")
    shape = (1, 512, 4, 4, 64, 64, 4)
    nws = L.linatt_kata_fwd_workspace_bytes(*shape, 0, 0, 0)
    ws = torch.empty(nws, device="cuda", dtype=torch.uint8)
    tail = (*shape, 0.25, 0, 0, _lib.stream_of(x))
    for w, n in ((None, 0), (ws, nws - 1), (ws[4:], nws)):
        assert L.linatt_kata_fwd_split(p(x), p(x), p(x), None, p(x), p(den), p(w), n, *tail) == -1
