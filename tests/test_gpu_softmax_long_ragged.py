"""softmax / log_softmax of long rows that are no whole number of packs: one workgroup of 1024 lanes holds the row in 3
to 20 whole packs a lane (TAIL of softmax_fwd_resident_kernel, softmax_bwd_resident_kernel and
log_softmax_bwd_grad_resident_kernel), few rows are held by teams of workgroups whose last chunk starts early
(softmax_fwd_team_kernel, softmax_bwd_team_kernel).  The regime of the reference's vocabulary-sized rows
(src/ATen/native/xpu/sycl/SoftMaxKernels.cpp:546-684, 991-1150).  Against float64: the last pack one element to one
short of whole, the last one of a lane round or the only one in it, off a 16-byte boundary, in place, rows without a
finite element and with infinities and NaN where neighbouring packs meet, and every wait given up."""
import math

import pytest
import torch

from helpers import gen, offset_view

pytestmark = pytest.mark.gpu

UNIT = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -10, torch.float32: 2.0 ** -22}
TINY = {torch.bfloat16: 1e-37, torch.float16: 6e-8, torch.float32: 1e-37}  # a step of the smallest numbers


def _near(a, ref, tol, what):
    a, ref, tol = a.double(), ref.double(), tol.double()
    bad = ~((a == ref) | (a.isnan() & ref.isnan()) | ((a - ref).abs() <= tol))
    assert not bool(bad.any()), "%s: %d wrong, first at %s" % (what, int(bad.sum()), bad.nonzero()[0].tolist())


def _sum(n):
    """The sums' float32 error relative to the sum of magnitudes: the terms of a lane (of 512 at least) and a tree."""
    return (n / 512 + 32) * 2.0 ** -24


def _forward(cabi, x, is_log, what, y=None):
    v = x.double()
    ref = torch.log_softmax(v, -1) if is_log else torch.softmax(v, -1)
    y = cabi.softmax_fwd(x, is_log, y=y)
    # exp's and log's own error against float64: 4 units of float32 over arguments up to 2^7
    own = 2.0 ** -15 if not is_log else 2.0 ** -20
    _near(y, ref, UNIT[y.dtype] * ref.abs() + (own + _sum(x.shape[-1])) * (torch.ones_like(ref) if is_log else ref) + TINY[y.dtype], what)
    return y


def _backward(cabi, grad, y, is_log, what, gi=None, gi_dtype=None):
    g, v = grad.double(), y.double()
    terms = g if is_log else g * v
    s, m = terms.sum(-1, keepdim=True), terms.abs().sum(-1, keepdim=True)
    ref = g - v.exp() * s if is_log else v * (g - s)
    w = v.exp() if is_log else v
    out = cabi.softmax_bwd(grad, y, is_log, gi=gi, gi_dtype=gi_dtype)
    slack = w * (_sum(y.shape[-1]) * m) + 2.0 ** -20 * (w * s.abs() + (0 if is_log else w * g.abs()))
    _near(out, ref, UNIT[out.dtype] * ref.abs() + slack + TINY[out.dtype], what)
    return out


def _rows(M, N, dtype, seed):
    g = gen(seed)
    return (3 * torch.randn(M, N, generator=g)).to(dtype), torch.randn(M, N, generator=g).to(dtype)


def _all(cabi, gpu, M, N, dtype, seed):
    x, grad = (t.to(gpu) for t in _rows(M, N, dtype, seed))
    for is_log in (False, True):
        what = "[%d, %d] %s log %d" % (M, N, dtype, is_log)
        print("case", what, flush=True)
        y = _forward(cabi, x, is_log, what)
        gi = _backward(cabi, grad, y, is_log, "backward " + what)
        assert torch.equal(y, cabi.softmax_fwd(x, is_log)), "run to run " + what
        assert torch.equal(gi, cabi.softmax_bwd(grad, y, is_log)), "run to run, backward " + what
        _forward(cabi, offset_view(x, 3), is_log, "off a boundary " + what)
        _backward(cabi, offset_view(grad, 1), offset_view(y, 5), is_log, "off a boundary, backward " + what)
        over = x.clone()
        _forward(cabi, over, is_log, "in place " + what, y=over)
        over_g, over_y = grad.clone(), y.clone()
        _backward(cabi, over_g, y, is_log, "gi over grad " + what, gi=over_g)
        _backward(cabi, grad, over_y, is_log, "gi over y " + what, gi=over_y)


# packs beyond whole lane rounds of 1024, and the elements of the last pack
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=str)
def test_every_pack_count(cabi, gpu, dtype):
    E = 4 if dtype == torch.float32 else 8
    for v in range(3 if E == 8 else 5, 22):
        packs = (1024 * v, 1024 * (v - 1) + 1, 1024 * (v - 1) + 517)[v % 3]
        _all(cabi, gpu, 130 if v in (4, 9) else 129, (packs - 1) * E + 1 + v % (E - 1), dtype, 7000 + v)


@pytest.mark.parametrize("M", [1, 3, 64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=str)
def test_teams(cabi, gpu, dtype, M):
    E = 4 if dtype == torch.float32 else 8
    # (packs: the fewest; the last chunk one pack; the last chunk whole; two rounds of a full machine)
    for packs in (4096, 4097, 9 * 512 + 1, 16 * 512 * (1 if M > 8 else 64) + 300):
        N = (packs - 1) * E + 1 + packs % (E - 1)
        _all(cabi, gpu, M, N, dtype, 7100 + packs)
        x, grad = (t.to(gpu) for t in _rows(M, N, dtype, 7200 + packs))
        try:
            cabi.set_team_wait_us(0)
            for is_log in (False, True):
                y = _forward(cabi, x, is_log, "every wait given up %s" % ((M, N),))
                _backward(cabi, grad, y, is_log, "every wait given up, backward %s" % ((M, N),))
                torch.cuda.synchronize()
        finally:
            cabi.set_team_wait_us()


@pytest.mark.parametrize("M", [5, 200])
def test_other_dtypes_and_special_rows(cabi, gpu, M):
    for packs, over in ((5000, 3), (9217, 1), (18000, 7)):
        N = packs * 8 - 8 + over
        x, _ = (t.to(gpu) for t in _rows(M, N, torch.float16, packs))
        for is_log in (False, True):
            y = cabi.softmax_fwd(x, is_log, out_dtype=torch.float32)
            ref = torch.log_softmax(x.double(), -1) if is_log else torch.softmax(x.double(), -1)
            tol = 2.0 ** -20 * (ref.abs() + 1) + _sum(N) if is_log else (2.0 ** -18 + _sum(N)) * ref
            _near(y, ref, tol, "half to float %s log %d" % ((M, N), is_log))
            grad = torch.randn(M, N, generator=gen(5)).to(gpu)
            _backward(cabi, grad, y, is_log, "float to half %s log %d" % ((M, N), is_log), gi_dtype=torch.float16)
        b = x.to(torch.bfloat16)
        edge = N - 8  # the first element of the row's last whole pack; its last ones belong to both of the last packs
        b[0] = -math.inf
        b[1, edge] = math.inf
        b[2, edge + 1] = math.nan
        b[3, : N - 1] = -math.inf
        b[4, N - 1] = -math.inf
        for is_log in (False, True):
            y = cabi.softmax_fwd(b, is_log)
            assert bool(y[:3].isnan().all())
            if not is_log:
                assert float(y[3, N - 1]) == 1.0 and float(y[3, : N - 1].abs().max()) == 0.0
                assert float(y[4, N - 1]) == 0.0
            else:
                assert float(y[3, N - 1]) == 0.0 and float(y[4, N - 1]) == -math.inf
            rest = torch.log_softmax(b[4:].double(), -1) if is_log else torch.softmax(b[4:].double(), -1)
            _near(y[4:], rest, 2.0 ** -7 * rest.abs() + 1e-30, "rows beside special ones")
