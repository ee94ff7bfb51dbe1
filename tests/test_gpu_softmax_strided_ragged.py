"""softmax / log_softmax over a dimension that is not innermost, rows of `inner` that are no whole number of
16-byte packs: the last pack of a row is read and written E elements before the row's end, over columns that a
neighbouring lane -- of another workgroup or another team, where strips meet -- holds as well.  Stands where the
reference walks element by element (SpatialSoftmaxForwardKernelFunctor,
src/ATen/native/xpu/sycl/SoftMaxKernels.cpp:725-950; backward :1387-1564).  Against the float64 oracle, apart and in
place (where the output overlaps the input, no pack may reach into a neighbour's columns), with every wait given up
and from run to run."""
import numpy as np
import pytest
import torch

from helpers import assert_close, gen, rowsum_slack, to_np32

pytestmark = pytest.mark.gpu

# (outer, D, columns beyond whole packs, whole packs): one pack and an element; a strip's last pack alone in a strip
# of its own; the one-workgroup tile at its largest D and beyond; teams of one, of several, of whole compute units.
# Beside each: the workgroups of a team in the forward and backward.
SHAPES = {(3, 5, 1, 1): (0, 0), (2, 40, 3, 4): (0, 0), (2, 256, 1, 16): (0, 0), (1, 300, 1, 1): (0, 0),
          (2, 600, 2, 16): (19, 19), (2, 2300, 3, 32): (18, 18), (600, 300, 1, 8): (1, 2), (1000, 300, 1, 7): (1, 1),
          (1, 8200, 3, 512): (13, 43)}


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", list(SHAPES), ids=str)
def test_rows_of_no_whole_packs(cabi, oracle, gpu, dtype, shape):
    outer, D, over, packs = shape
    inner = packs * (4 if dtype == torch.float32 else 8) + over
    teams = tuple(cabi.strided_team_plan(b, outer, D, inner, cabi.dtype_code(dtype))["team"] for b in (0, 1))
    assert teams == SHAPES[shape]
    print("case strided softmax, ragged", dtype, (outer, D, inner), flush=True)
    g = gen(3100 + D)
    x = (3.0 * torch.randn(outer, D, inner, generator=g)).to(dtype)
    x[0, D // 3:, inner - 1] = float("-inf")  # a masked tail of a column that two lanes hold
    x[0, :, inner - 2] = float("-inf")        # a column without a finite element
    x[-1, D - 1, 2] = float("nan")            # a NaN poisons its column
    grad = torch.randn(outer, D, inner, generator=g).to(dtype)
    xg, gg = x.to(gpu), grad.to(gpu)

    def last(a):
        return np.ascontiguousarray(np.moveaxis(a, 1, -1))

    def given_up(fn):
        try:
            cabi.set_team_wait_us(0)
            return fn()
        finally:
            cabi.set_team_wait_us()

    for mode, is_log in ((cabi.SOFTMAX, False), (cabi.LOG_SOFTMAX, True)):
        what = "%s %s %s" % ("log_softmax" if is_log else "softmax", (outer, D, inner), dtype)
        fwd = lambda: cabi.softmax_strided_fwd(xg, 1, mode)  # noqa: E731
        y = fwd()
        oy = np.moveaxis(oracle.softmax_fwd(last(to_np32(x)), is_log), -1, 1)
        assert_close(y, oy, dtype, what)
        assert torch.equal(y.view(torch.uint8), fwd().view(torch.uint8)), what + ": run to run"
        assert_close(given_up(fwd), oy, dtype, what + ", every wait given up")
        over_x = xg.clone()
        assert_close(cabi.softmax_strided_fwd(over_x, 1, mode, y=over_x), oy, dtype, what + ", in place")
        bwd = lambda: cabi.softmax_strided_bwd(gg, y, 1, mode)  # noqa: E731
        gi = bwd()
        yy = y.float().cpu().movedim(1, -1)
        ogi = np.moveaxis(oracle.softmax_bwd(last(to_np32(grad)), last(to_np32(y)), is_log), -1, 1)
        terms = grad.float().movedim(1, -1)
        sl = (rowsum_slack(terms, torch.exp(yy)) if is_log else rowsum_slack(yy * terms, yy)).movedim(-1, 1)
        assert_close(gi, ogi, dtype, what + " backward", slack=sl)
        assert torch.equal(gi.view(torch.uint8), bwd().view(torch.uint8)), what + " backward: run to run"
        assert_close(given_up(bwd), ogi, dtype, what + " backward, every wait given up", slack=sl)
        over_g, over_y = gg.clone(), y.clone()
        assert_close(cabi.softmax_strided_bwd(over_g, y, 1, mode, gi=over_g), ogi, dtype, what + ", gi over grad", slack=sl)
        assert_close(cabi.softmax_strided_bwd(gg, over_y, 1, mode, gi=over_y), ogi, dtype, what + ", gi over y", slack=sl)
    if dtype == torch.float16:
        y32 = cabi.softmax_strided_fwd(xg, 1, cabi.SOFTMAX, out_dtype=torch.float32)
        assert_close(y32, np.moveaxis(oracle.softmax_fwd(last(to_np32(x)), False), -1, 1), torch.float32,
                     "float16 -> float32")
