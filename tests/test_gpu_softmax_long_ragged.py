"""softmax / log_softmax of long rows that are no whole number of packs: one workgroup of 1024 or 512 lanes holds the
row in 3 to 20 whole packs a lane (TAIL of softmax_fwd_resident_kernel, softmax_bwd_resident_kernel and
log_softmax_bwd_grad_resident_kernel), few rows are held by teams of workgroups whose last chunk starts early
(softmax_fwd_team_kernel, softmax_bwd_team_kernel).  The regime of the reference's vocabulary-sized rows
(src/ATen/native/xpu/sycl/SoftMaxKernels.cpp:546-684, 991-1150).  Against float64: the last pack one element to one
short of whole, the last one of a lane round or the only one in it, off a 16-byte boundary, in place, rows without a
finite element and with infinities and NaN where neighbouring packs meet, and every wait given up.  The plan says of
every case which lanes, packs or team it runs on."""
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
    slack = (own + _sum(x.shape[-1])) * (torch.ones_like(ref) if is_log else ref)
    _near(y, ref, UNIT[y.dtype] * ref.abs() + slack + TINY[y.dtype], what)
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


def _row(lanes, v, last, E):
    """The longest ragged row whose window has one pack in the last lane round, or (last) all of them."""
    window = lanes * v if last else lanes * (v - 1) + 1
    return next(n for n in range(window * E - E + 1, 0, -1) if n % E and (n + 2 * (E - 1)) // E == window)


def _held(cabi, backward, is_log, M, N, dtype, lanes, v):
    p = cabi.softmax_plan(backward, is_log, M, N, cabi.dtype_code(dtype))
    assert (p["team"], p["resident"], p["lanes_per_row"], p["packs_per_lane"]) == (0, 1, lanes, v), (M, N, p)


# (lanes, packs a lane, a number of rows for which the forward runs on these)
HELD16 = [(512, v, 129) for v in range(5, 15)] + [(1024, 3, 2100), (1024, 4, 2100)] + [(1024, v, 520) for v in (5, 6, 7)] + \
    [(1024, v, 129) for v in (8, 9, 10, 11, 12, 13, 14, 15, 16, 18, 20)]
HELD32 = [(512, v, 129) for v in range(9, 15)] + [(1024, v, 520) for v in (5, 6, 7)] + [(1024, v, 129) for v in range(8, 17)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=str)
def test_every_pack_count_forward(cabi, gpu, dtype):
    E = 4 if dtype == torch.float32 else 8
    for lanes, v, M in HELD32 if E == 4 else HELD16:
        for last in (False, True):
            if (lanes, v, last) == (1024, 3, False):
                continue  # (rows of up to 2560 packs run on 512 lanes)
            N = _row(lanes, v, last, E)
            x, _ = _rows(M, N, dtype, 7000 + v)
            x = x.to(gpu)
            for is_log in (False, True):
                what = "[%d, %d] %s log %d, %d packs on %d lanes" % (M, N, dtype, is_log, v, lanes)
                print("case", what, flush=True)
                _held(cabi, 0, is_log, M, N, dtype, lanes, v)
                y = _forward(cabi, x, is_log, what)
                assert torch.equal(y, cabi.softmax_fwd(x, is_log)), "run to run " + what
                _forward(cabi, offset_view(x, 3), is_log, "off a boundary " + what)
                over = x.clone()
                _forward(cabi, over, is_log, "in place " + what, y=over)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=str)
def test_every_pack_count_backward(cabi, gpu, dtype):
    E, M = 4 if dtype == torch.float32 else 8, 129
    for v in range(5 if E == 4 else 3, 21):
        for last in (False, True):
            N = _row(1024, v, last, E)
            x, grad = (t.to(gpu) for t in _rows(M, N, dtype, 7050 + v))
            for is_log in (False, True):
                if v > 8 and not is_log:
                    continue
                what = "[%d, %d] %s log %d backward, %d packs" % (M, N, dtype, is_log, v)
                print("case", what, flush=True)
                _held(cabi, 1, is_log, M, N, dtype, 1024, v)
                y = cabi.softmax_fwd(x, is_log)
                gi = _backward(cabi, grad, y, is_log, what)
                assert torch.equal(gi, cabi.softmax_bwd(grad, y, is_log)), "run to run " + what
                _backward(cabi, offset_view(grad, 3), offset_view(y, 3), is_log, "off a boundary " + what)
                _backward(cabi, offset_view(grad, 1), offset_view(y, 2), is_log, "windows apart " + what)
                over_g, over_y = grad.clone(), y.clone()
                _backward(cabi, over_g, y, is_log, "gi over grad " + what, gi=over_g)
                _backward(cabi, grad, over_y, is_log, "gi over y " + what, gi=over_y)


def test_float32_output_of_every_pack_count(cabi, gpu):
    """float16 -> float32: the held forward stores 32 bytes a lane and pack."""
    for lanes, v, M in HELD16:
        M = max(M, 200)  # (fewer rows: two passes, see the plan)
        N = _row(lanes, v, v == 3 or v % 2 == 0, 8)
        x, _ = _rows(M, N, torch.float16, 7300 + v)
        x = x.to(gpu)
        for is_log in (False, True):
            p = cabi.softmax_plan(0, is_log, M, N, cabi.F16, cabi.F32)
            if not is_log and p["resident"] == 0:
                continue
            assert (p["team"], p["lanes_per_row"], p["packs_per_lane"]) == (0, lanes, v), p
            y = cabi.softmax_fwd(x, is_log, out_dtype=torch.float32)
            ref = torch.log_softmax(x.double(), -1) if is_log else torch.softmax(x.double(), -1)
            tol = 2.0 ** -20 * (ref.abs() + 1) + _sum(N) if is_log else (2.0 ** -18 + _sum(N)) * ref
            _near(y, ref, tol, "half to float %s log %d" % ((M, N), is_log))


@pytest.mark.parametrize("M", [1, 3, 64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=str)
def test_teams(cabi, gpu, dtype, M):
    E = 4 if dtype == torch.float32 else 8
    # (packs: some of the fewest; the last chunk one pack; the last chunk whole; more than one workgroup holds, in the
    # backward two rounds of a full machine at 128 rows)
    for packs in {1: (4224, 4609, 5120), 3: (4224, 4609, 5120), 64: (7168, 12801, 14336),
                  128: (21505, 24577, 24576)}[M] + (16 * 512 * (8 if M > 8 else 64) + 300,):
        N = (packs - 1) * E + 1 + packs % (E - 1)
        on = [(b, l) for b in (0, 1) for l in (0, 1) if cabi.softmax_plan(b, l, M, N, cabi.dtype_code(dtype))["team"] > 1]
        assert (0, 0) in on and (packs < 8192 or len(on) == 4), (M, N, on)
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
