"""softmax / log_softmax over a dimension that is not innermost, D beyond the one-workgroup tile:
softmax_strided_team_fwd_kernel / softmax_strided_team_bwd_kernel, where a team of workgroups holds
a strip of columns in registers and exchanges the columns' numbers through library-owned device
memory with a bounded wait.  Stands where the reference walks the D rows three times
(SpatialSoftmaxForwardKernelFunctor / SpatialSoftmaxBackwardKernelFunctor,
src/ATen/native/xpu/sycl/SoftMaxKernels.cpp:725-950, 1387-1564).
Through the extern "C" ABI against the float64 oracle (float32 rtol = atol = 1e-5; 16-bit atol 1e-2,
rtol 1.6e-2), against the path a workgroup takes when its wait gives up (forced from the host by a
wait of zero: no kernel hangs), and for run-to-run determinism."""
import numpy as np
import pytest
import torch

from helpers import assert_close, gen, rowsum_slack, to_np32

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]
# (outer, D, packs of inner): the shortest D; a workgroup with its last rows missing; strips one,
# three and sixteen packs wide with a narrow last strip; teams whose last workgroup holds one row; a
# strip over the largest teams; more strips than teams (rounds), the last round not full; the same on
# teams of one.  Beside each: whether the forward / backward call is the one-workgroup tile's, a
# team's of one workgroup or of several.
SHAPES = {(3, 257, 20): "tile tile", (2, 513, 16): "several several", (1, 1025, 1): "tile tile",
          (3, 2300, 3): "several several", (1, 1025, 40): "several several",
          (2, 4097, 17): "several several", (1, 60000, 2): "several several", (700, 1025, 1): "tile tile",
          (1, 520, 4120): "several several", (300, 300, 17): "several several",
          (2, 9000, 33): "several several", (1, 262000, 1): "several several",
          (1000, 300, 8): "one one"}


def _runs(cabi, backward, shape, dtype):
    inner = shape[2] * (4 if dtype == torch.float32 else 8)
    team = cabi.strided_team_plan(backward, shape[0], shape[1], inner, cabi.dtype_code(dtype))["team"]
    return "tile" if team == 0 else "one" if team == 1 else "several"


def _last(a):
    return np.ascontiguousarray(np.moveaxis(a, 1, -1))


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("shape", list(SHAPES), ids=str)
def test_team_strips_against_oracle_and_the_give_up_path(cabi, oracle, gpu, dtype, shape):
    outer, D, packs = shape
    inner = packs * (4 if dtype == torch.float32 else 8)
    print("case strided softmax teams", dtype, (outer, D, inner), flush=True)
    assert [_runs(cabi, b, shape, dtype) for b in (0, 1)] == SHAPES[shape].split()
    g = gen(2400 + D)
    x = (3.0 * torch.randn(outer, D, inner, generator=g)).to(dtype)
    x[0, D // 3:, 0] = float("-inf")      # a masked tail: whole workgroups without a finite element
    x[0, :, 1] = float("-inf")            # a column without one
    x[-1, D - 1, 2] = float("nan")        # a NaN poisons its column
    grad = torch.randn(outer, D, inner, generator=g).to(dtype)
    xg, gg = x.to(gpu), grad.to(gpu)

    def given_up(fn):
        try:
            cabi.set_team_wait_us(0)
            return fn()
        finally:
            cabi.set_team_wait_us()

    for mode, is_log in ((cabi.SOFTMAX, False), (cabi.LOG_SOFTMAX, True)):
        what = "%s %s %s" % ("log_softmax" if is_log else "softmax", shape, dtype)
        fwd = lambda: cabi.softmax_strided_fwd(xg, 1, mode)  # noqa: E731
        y = fwd()
        oy = np.moveaxis(oracle.softmax_fwd(_last(to_np32(x)), is_log), -1, 1)
        assert_close(y, oy, dtype, what)
        assert torch.equal(y.view(torch.uint8), fwd().view(torch.uint8)), what + ": run to run"
        assert_close(given_up(fwd), oy, dtype, what + ", every wait given up")
        bwd = lambda: cabi.softmax_strided_bwd(gg, y, 1, mode)  # noqa: E731
        gi = bwd()
        ogi = np.moveaxis(oracle.softmax_bwd(_last(to_np32(grad)), _last(to_np32(y)), is_log), -1, 1)
        yy = y.float().cpu().movedim(1, -1)
        terms = grad.float().movedim(1, -1)
        sl = rowsum_slack(terms, torch.exp(yy)) if is_log else rowsum_slack(yy * terms, yy)
        sl = sl.movedim(-1, 1)
        assert_close(gi, ogi, dtype, what + " backward", slack=sl)
        assert torch.equal(gi.view(torch.uint8), bwd().view(torch.uint8)), what + ": run to run"
        assert_close(given_up(bwd), ogi, dtype, what + " backward, every wait given up", slack=sl)
    ys = cabi.softmax_strided_fwd(xg, 1, cabi.SAFE_SOFTMAX)
    assert bool((ys[0, :, 1] == 0).all()), "safe softmax: zeros for a column without a finite element"
    if dtype == torch.float16:
        y32 = cabi.softmax_strided_fwd(xg, 1, cabi.SOFTMAX, out_dtype=torch.float32)
        assert_close(y32, np.moveaxis(oracle.softmax_fwd(_last(to_np32(x)), False), -1, 1),
                     torch.float32, "float16 -> float32")
        g32 = grad.float().to(gpu)
        gi16 = cabi.softmax_strided_bwd(g32, y32, 1, cabi.SOFTMAX, gi_dtype=torch.float16)
        assert_close(gi16, cabi.softmax_strided_bwd(g32, y32, 1, cabi.SOFTMAX), torch.float16,
                     "float32 -> float16")


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("shape,runs", [((1000, 300, 8), "one one"), ((300, 300, 17), "several several"),
                                        ((2, 2048, 33), "several several"), ((40, 480, 8), "tile tile")], ids=str)
def test_in_place(cabi, gpu, shape, runs, dtype):
    """The output over an input: a team of one workgroup holds its strip before it writes it; several would
    read one another's strips again, so such a call keeps the launches that exchange nothing."""
    outer, D, packs = shape
    inner = packs * (4 if dtype == torch.float32 else 8)
    print("case strided softmax in place", dtype, (outer, D, inner), flush=True)
    assert [_runs(cabi, b, shape, dtype) for b in (0, 1)] == runs.split()
    g = gen(2450 + D)
    x = (3.0 * torch.randn(outer, D, inner, generator=g)).to(dtype).to(gpu)
    grad = torch.randn(outer, D, inner, generator=g).to(dtype).to(gpu)
    for mode, fn in ((cabi.SOFTMAX, torch.softmax), (cabi.LOG_SOFTMAX, torch.log_softmax)):
        xin = x.clone()
        cabi.softmax_strided_fwd(xin, 1, mode, y=xin)
        assert_close(xin, to_np32(fn(x.double(), 1).float()), dtype, "in place y")
        y = cabi.softmax_strided_fwd(x, 1, mode)
        p, gd = y.double(), grad.double()
        want = p * (gd - (p * gd).sum(1, keepdim=True))
        # (a few ulps of the sum of the magnitudes, as for any float32 sum in another order)
        slack = p * (p * gd).abs().sum(1, keepdim=True) * 2.0 ** -21
        if mode == cabi.LOG_SOFTMAX:
            want = gd - p.exp() * gd.sum(1, keepdim=True)
            slack = p.exp() * gd.abs().sum(1, keepdim=True) * 2.0 ** -21
        for over in (0, 1):
            a, b = grad.clone(), y.clone()
            gi = cabi.softmax_strided_bwd(a, b, 1, mode, gi=(a, b)[over])
            assert_close(gi, to_np32(want.float()), dtype, "in place gi over %d" % over, slack=slack.float().cpu())


@pytest.mark.parametrize("shape,runs", [((2, 2048, 33), "several several"), ((1000, 300, 8), "one one"),
                                        ((64, 400, 17), "several several")], ids=str)
def test_under_capture(cabi, gpu, shape, runs):
    """A captured call runs no exchange (a replay would carry the id of the capture): replays, with eager
    work between them, give what an eager call gives to rounding, on other inputs too."""
    outer, D, packs = shape
    dtype, inner = torch.bfloat16, packs * 8
    assert [_runs(cabi, b, shape, dtype) for b in (0, 1)] == runs.split()
    g = gen(2470 + D)
    x, grad = (torch.randn(outer, D, inner, generator=g).to(dtype).to(gpu) for _ in range(2))
    y, gi = torch.empty_like(x), torch.empty_like(x)

    def both():
        cabi.softmax_strided_fwd(x, 1, y=y)
        cabi.softmax_strided_bwd(grad, y, 1, gi=gi)

    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        both()
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        both()
    for k in range(4):
        x.copy_(torch.randn(outer, D, inner, generator=g).to(dtype))
        graph.replay()
        torch.cuda.synchronize()
        got = y.clone(), gi.clone()
        ey = cabi.softmax_strided_fwd(x, 1)
        egi = cabi.softmax_strided_bwd(grad, ey, 1)
        assert_close(got[0], to_np32(ey.float()), dtype, "replay %d y" % k)
        assert_close(got[1], to_np32(egi.float()), dtype, "replay %d gi" % k)


def test_more_than_two_to_the_31_elements(cabi, gpu):
    """[8, 8192, 33000] bfloat16: byte offsets beyond 32 bits, strips in more rounds than a tag counts (64)."""
    outer, D, inner = 8, 8192, 33000
    for b in (0, 1):
        t = cabi.strided_team_plan(b, outer, D, inner, cabi.BF16)
        strips = outer * -(-inner // (8 * t["lanes_per_row"]))
        assert t["team"] > 1 and strips > 64 * (t["grid_blocks"] // t["team"])
    g = torch.Generator(device=gpu).manual_seed(2490)
    x = torch.empty(outer, D, inner, dtype=torch.bfloat16, device=gpu).normal_(0, 3, generator=g)
    grad = torch.empty_like(x).normal_(generator=g)
    y = cabi.softmax_strided_fwd(x, 1)
    gi = cabi.softmax_strided_bwd(grad, y, 1)
    for o in range(outer):
        for c in range(0, inner, 11000):
            cols = slice(c, c + 11000)
            want = torch.softmax(x[o, :, cols].float(), 0)
            err = (y[o, :, cols].float() - want).abs() - 1.6e-2 * want.abs()
            assert float(err.max()) <= 1e-5, (o, c)
            p, gd = y[o, :, cols].float(), grad[o, :, cols].float()
            want = p * (gd - (p * gd).sum(0, keepdim=True))
            err = (gi[o, :, cols].float() - want).abs() - 1.6e-2 * want.abs()
            assert float(err.max()) <= 1e-5, (o, c)
