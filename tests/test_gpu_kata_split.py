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


def test_split_forward_fp16_tiny_weights():
    """float16 rows whose every weight lies below 2^-128 (four small keys, then
    a decay of e^-84.5 and zero keys): the row scale keeps them through the
    pieces, as in the unsplit kernel.  The four weights are equal, so o is the
    mean of their v rows to one float16 spacing."""
    from linatt_amd import _lib
    L, p = _lib.load(), _lib.ptr
    B, T, H, dk, M = 1, 3100, 2, 64, 2
    print(f"\nsplit forward, weights below 2^-128, B{B} T{T} H{H}", flush=True)
    q = torch.full((B, T, H, dk), 2.0 ** -5, dtype=torch.float16, device="cuda")
    k = torch.zeros_like(q)
    k[:, :4] = 2.0 ** -5
    v = torch.randn(B, T, H, 64, generator=torch.Generator().manual_seed(0)).half().cuda()
    c = torch.zeros(B, T, H, device="cuda")
    c[:, 64:] = -84.5
    shape = (B, T, H, H, dk, 64, M)
    nws = L.linatt_kata_fwd_workspace_bytes(*shape, 0, 1, 2)
    assert nws > 0
    ws = torch.empty(nws, device="cuda", dtype=torch.uint8)
    out = []
    for split in (False, True):
        o, den = torch.full_like(v, float("nan")), torch.full((B, T, H), float("nan"), device="cuda")
        head, tail = (p(q), p(k), p(v), p(c), p(o), p(den)), (*shape, 1.0, 0, 2, _lib.stream_of(q))
        if split:
            _lib.check("split", L.linatt_kata_fwd_split(*head, p(ws), nws, *tail))
        else:
            _lib.check("fwd", L.linatt_kata_fwd(*head, *tail))
        out.append((o.double(), den.double()))
    torch.cuda.synchronize()
    (o1, d1), (o2, d2) = out
    assert 0 < d1[:, 64:].max() < 2.0 ** -128
    mean = v[:, :4].double().mean(1, keepdim=True)
    for o in (o1, o2):
        assert ((o[:, 64:] - mean).abs() <= 2.0 ** -10 * mean.abs() + 2.0 ** -24).all()
    assert torch.equal(d1, d2) and torch.equal(o1, o2)


def _special(q, k, v):
    """Rows without weights (zero queries, the first key included), then a NaN
    key and an infinite value, each well inside a cut list."""
    T = q.shape[1]
    q[:, 0] = q[:, 700:760] = 0
    k[:, T // 2 + 7, 0, 3] = float("nan")
    v[:, T // 2 - 130, -1, 5] = float("inf")


def _same_special(a, b, tol):
    a, b = a.double(), b.double()
    assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isinf(), b.isinf())
    fin = a.isfinite()
    assert fin.any() and not fin.all()
    assert torch.equal(a[a.isinf()], b[a.isinf()])
    a, b = torch.where(fin, a, 0.0), torch.where(fin, b, 0.0)
    assert ((a - b).abs() <= tol(a)).all()


@pytest.mark.parametrize("T,HQ,H,dk,M,variant,decay,dtype", [
    (2049, 3, 3, 64, 4, "sum", False, torch.bfloat16), (2600, 4, 2, 64, 4, "concat", False, torch.bfloat16),
    (3100, 2, 2, 64, 2, "concat", True, torch.float16), (2100, 2, 2, 128, 2, "sum", False, torch.float16),
    (2000, 4, 2, 64, 2, "concat", False, torch.float32)])
def test_split_forward_special_values(T, HQ, H, dk, M, variant, decay, dtype):
    """Zero denominators, NaN and infinities come out of the split forward where
    the unsplit one has them, and nowhere else."""
    from linatt_amd import _lib
    print(f"\nsplit forward, special values, T{T} HQ{HQ} H{H} dk{dk} M{M} {variant} decay={decay} {dtype}", flush=True)
    L, p = _lib.load(), _lib.ptr
    g = torch.Generator().manual_seed(T)
    q = torch.randn(1, T, HQ, dk, generator=g).to(dtype).cuda()
    k, v = (torch.randn(1, T, H, d, generator=g).to(dtype).cuda() for d in (dk, 64))
    _special(q, k, v)
    c = (-torch.rand(1, T, HQ, generator=g) * 0.05).cumsum(1).cuda() if decay else None
    var, code, shape = int(variant == "sum"), _lib.dtype_code(dtype), (1, T, HQ, H, dk, 64, M)
    nws = L.linatt_kata_fwd_workspace_bytes(*shape, var, int(decay), code)
    assert nws > 0
    ws = torch.empty(nws, device="cuda", dtype=torch.uint8)
    out = []
    for split in (False, True):
        o, den = torch.empty(1, T, HQ, 64, device="cuda", dtype=dtype), torch.empty(1, T, HQ, device="cuda")
        head, tail = (p(q), p(k), p(v), p(c), p(o), p(den)), (*shape, 1 / math.sqrt(dk // M), var, code, _lib.stream_of(q))
        if split:
            _lib.check("split", L.linatt_kata_fwd_split(*head, p(ws), nws, *tail))
        else:
            _lib.check("fwd", L.linatt_kata_fwd(*head, *tail))
        out.append((o, den))
    torch.cuda.synchronize()
    (o1, d1), (o2, d2) = out
    assert (d1[:, 700:760] == 0).all() and (o1[:, 700:760].float() == 0).all()
    vmax = v[v.isfinite()].double().abs().max()
    acc = 2 * T * 2.0 ** -24 + (2.0 ** -10 if dtype == torch.float16 else 0.0)
    _same_special(d1, d2, lambda a: acc * a)
    _same_special(o1, o2, lambda a: SPACING[dtype] * a.abs() + 2 * acc * vmax)


@pytest.mark.parametrize("B,T,HQ,H,M,variant", [(1, 2048, 3, 3, 4, "concat"), (1, 1985, 6, 2, 1, "concat"), (1, 1930, 2, 1, 4, "sum")])
def test_split_backward_special_values(B, T, HQ, H, M, variant):
    """The same for dk and dv (bounds as in the plain comparison)."""
    from linatt_amd import _lib
    print(f"\nsplit backward, special values, B{B} T{T} HQ{HQ} H{H} M{M} {variant}", flush=True)
    L, p = _lib.load(), _lib.ptr
    g = torch.Generator().manual_seed(T + M)
    q, do = (torch.randn(B, T, HQ, 64, generator=g).bfloat16().cuda() for _ in range(2))
    k, v = (torch.randn(B, T, H, 64, generator=g).bfloat16().cuda() for _ in range(2))
    o, den = torch.empty_like(q), torch.empty(B, T, HQ, device="cuda")
    var, sp, sc, shape = int(variant == "sum"), _lib.stream_of(q), math.sqrt(M) / 8, (B, T, HQ, H, 64, 64, M)
    q[:, 0] = q[:, 700:760] = 0
    _lib.check("fwd", L.linatt_kata_fwd(p(q), p(k), p(v), None, p(o), p(den), *shape, sc, var, 1, sp))
    do[:, T // 2 + 7, 0, 3], do[:, T // 3, -1, 5] = float("nan"), float("inf")
    ns = L.linatt_kata_bwd_split_workspace_bytes(*shape, var, 1)
    assert ns > L.linatt_kata_bwd_workspace_bytes(B, T, HQ, 64, 1) + 256  # the split engages
    ws = torch.empty(ns, device="cuda", dtype=torch.uint8)
    out = []
    for split in (False, True):
        gr = [torch.empty_like(x) for x in (q, k, v)]
        head, tail = (p(q), p(k), p(v), p(o), p(den), p(do), *map(p, gr), p(ws)), (*shape, sc, var, 1, sp)
        if split:
            _lib.check("split", L.linatt_kata_bwd_split(*head, ns, *tail))
        else:
            _lib.check("bwd", L.linatt_kata_bwd(*head, *tail))
        out.append(gr)
    torch.cuda.synchronize()
    assert torch.equal(out[0][0].isnan(), out[1][0].isnan())
    for a, b in zip(out[0][1:], out[1][1:]):
        top = a[a.isfinite()].double().abs().max()
        _same_special(a, b, lambda x: 2.0 ** -7 * x.abs() + 2.0 ** -12 * top)


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


@pytest.mark.parametrize("B,T,HQ,H,M,variant", [(6, 1403, 12, 4, 2, "sum"), (1, 2048, 3, 3, 4, "concat"),
                                                (1, 2100, 4, 1, 4, "concat"), (1, 1985, 6, 2, 1, "concat"),
                                                (1, 1930, 2, 1, 4, "sum"), (2, 2048, 16, 8, 4, "concat")])
def test_split_backward_equals_unsplit(B, T, HQ, H, M, variant):
    """``linatt_kata_bwd_split`` (dk/dv's query tiles over several workgroups)
    against ``linatt_kata_bwd``: dq is the same kernel (bit for bit); dk, dv
    add the same products in another order, in float32 far below the bf16
    spacing they are then rounded to, so a value moves by one spacing (2^-7 of
    it) at most, and the whole by less than that in the 2-norm."""
    from linatt_amd import _lib
    print(f"\nsplit backward B{B} T{T} HQ{HQ} H{H} M{M} {variant}", flush=True)
    L, p = _lib.load(), _lib.ptr
    g = torch.Generator().manual_seed(T + M)
    q, do = (torch.randn(B, T, HQ, 64, generator=g).bfloat16().cuda() for _ in range(2))
    k, v = (torch.randn(B, T, H, 64, generator=g).bfloat16().cuda() for _ in range(2))
    o, den = torch.empty_like(q), torch.empty(B, T, HQ, device="cuda")
    var, sp, sc, shape = int(variant == "sum"), _lib.stream_of(q), math.sqrt(M) / 8, (B, T, HQ, H, 64, 64, M)
    _lib.check("fwd", L.linatt_kata_fwd(p(q), p(k), p(v), None, p(o), p(den), *shape, sc, var, 1, sp))
    nb = L.linatt_kata_bwd_workspace_bytes(B, T, HQ, 64, 1)
    ns = L.linatt_kata_bwd_split_workspace_bytes(*shape, var, 1)
    assert ns > nb + 256  # the split engages
    ws = torch.empty(ns, device="cuda", dtype=torch.uint8)
    out = []
    for split in (False, True):
        gr = [torch.full_like(x, float("nan")) for x in (q, k, v)]
        head, tail = (p(q), p(k), p(v), p(o), p(den), p(do), *map(p, gr), p(ws)), (*shape, sc, var, 1, sp)
        if split:
            _lib.check("split", L.linatt_kata_bwd_split(*head, ns, *tail))
        else:
            _lib.check("bwd", L.linatt_kata_bwd(*head, *tail))
        out.append(gr)
    assert L.linatt_kata_bwd_split(*head, ns - 1, *tail) == -1
    torch.cuda.synchronize()
    assert torch.equal(out[0][0], out[1][0])
    for a, b in zip(out[0][1:], out[1][1:]):
        a, b = a.double(), b.double()
        print("  rel %.1e" % ((a - b).norm() / a.norm()).item(), flush=True)
        assert (a - b).norm() <= 2.0 ** -8 * a.norm()
        assert ((a - b).abs() <= 2.0 ** -7 * a.abs() + 2.0 ** -12 * a.abs().max()).all()


@pytest.mark.parametrize("B,T,HQ,H,M,variant,decay", [(1, 2048, 12, 12, 4, "concat", False), (1, 2100, 4, 1, 1, "concat", False),
                                                      (1, 1930, 3, 3, 4, "sum", False), (1, 300, 2, 2, 2, "concat", True)])
def test_split_onorm_backward_equals_unsplit(B, T, HQ, H, M, variant, decay):
    """The same with the output norm in the dq pass (the decayed score: never
    split).  dq, dc and the weight's gradient come from the same launches."""
    from linatt_amd import _lib
    print(f"\nsplit onorm backward B{B} T{T} HQ{HQ} H{H} M{M} {variant} decay={decay}", flush=True)
    L, p = _lib.load(), _lib.ptr
    g = torch.Generator().manual_seed(T + M)
    q, dy = (torch.randn(B, T, HQ, 64, generator=g).bfloat16().cuda() for _ in range(2))
    k, v = (torch.randn(B, T, H, 64, generator=g).bfloat16().cuda() for _ in range(2))
    w = (torch.rand(64, generator=g) + 0.5).cuda()
    c = (-torch.rand(B, T, HQ, generator=g) * 0.05).cumsum(1).cuda() if decay else None
    o, y = torch.empty_like(q), torch.empty_like(q)
    den, rstd = (torch.empty(B, T, HQ, device="cuda") for _ in range(2))
    var, sp, sc, shape = int(variant == "sum"), _lib.stream_of(q), math.sqrt(M) / 8, (B, T, HQ, H, 64, 64, M)
    _lib.check("fwd", L.linatt_kata_fwd_onorm(p(q), p(k), p(v), p(c), p(o), p(den), p(w), 1e-5, p(y), p(rstd), *shape,
                                              sc, var, 1, sp))
    nb = L.linatt_kata_bwd_onorm_workspace_bytes(B, T, HQ, 64, 1)
    ns = L.linatt_kata_bwd_onorm_split_workspace_bytes(*shape, var, int(decay), 1)
    assert (ns > nb + 256) == (not decay)
    ws = torch.empty(ns, device="cuda", dtype=torch.uint8)
    out = []
    for split in (False, True):
        gr = [torch.full_like(x, float("nan")) for x in (q, w, k, v)] + ([torch.full_like(c, float("nan"))] if decay else [])
        dq, dw, dk, dv = gr[:4]
        dc = gr[4] if decay else None
        head = (p(q), p(k), p(v), p(c), p(o), p(den), p(rstd), p(w), p(dy), p(dq), p(dk), p(dv), p(dc), p(dw), p(ws))
        tail = (*shape, sc, var, 1, sp)
        if split:
            _lib.check("split", L.linatt_kata_bwd_onorm_split(*head, ns, *tail))
        else:
            _lib.check("bwd", L.linatt_kata_bwd_onorm(*head, *tail))
        out.append(gr)
    if not decay:
        assert L.linatt_kata_bwd_onorm_split(*head, ns - 1, *tail) == -1
    torch.cuda.synchronize()
    assert all(torch.equal(out[0][i], out[1][i]) for i in (0, 1))
    for a, b in zip(out[0][2:4], out[1][2:4]):
        a, b = a.double(), b.double()
        print("  rel %.1e" % ((a - b).norm() / a.norm()).item(), flush=True)
        assert (a - b).norm() <= 2.0 ** -8 * a.norm()
        assert ((a - b).abs() <= 2.0 ** -7 * a.abs() + 2.0 ** -12 * a.abs().max()).all()
