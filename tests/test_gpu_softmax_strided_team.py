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
# strip over hundreds of workgroups; more strips than teams (rounds), the last round not full
SHAPES = [(3, 257, 20), (2, 513, 16), (1, 1025, 1), (3, 2300, 3), (1, 1025, 40), (2, 4097, 17),
          (1, 60000, 2), (700, 1025, 1), (1, 520, 4120)]


def _last(a):
    return np.ascontiguousarray(np.moveaxis(a, 1, -1))


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_team_strips_against_oracle_and_the_give_up_path(cabi, oracle, gpu, dtype, shape):
    outer, D, packs = shape
    inner = packs * (4 if dtype == torch.float32 else 8)
    print("case strided softmax teams", dtype, (outer, D, inner), flush=True)
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
