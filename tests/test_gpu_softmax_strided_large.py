"""Strided softmax on workgroups that have a compute unit each: packs of a lane in registers and, beyond 48
(backward 24 of each tensor), in LDS.  Every instance, full and with rows missing from the last workgroup,
against the float64 oracle on some columns of every strip (float32 rtol = atol = 1e-5, 16-bit atol 1e-2, rtol
1.6e-2), bit for bit from run to run, and against the path a workgroup takes when its wait gives up."""
import numpy as np
import pytest
import torch

from helpers import assert_close, rowsum_slack, to_np32

pytestmark = pytest.mark.gpu

# (outer, D, packs of inner): packs a lane of the forward, the backward and the float32 forward there (0: two
# workgroups a compute unit)
SHAPES = {(1, 5000, 1024): (40, 20, 0), (4, 4500, 230): (40, 0, 40), (1, 12899, 484): (56, 28, 56),
          (1, 8191, 1024): (64, 32, 0), (40, 4286, 28): (48, 24, 48), (1, 8192, 1022): (64, 32, 0),
          (40, 5686, 18): (64, 32, 64), (6, 323, 1285): (0, 24, 0)}


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("shape", list(SHAPES), ids=str)
def test_large_teams_against_oracle_and_the_give_up_path(cabi, oracle, gpu, dtype, shape):
    outer, D, packs = shape
    E = 4 if dtype == torch.float32 else 8
    inner = packs * E
    print("case strided softmax, large teams", dtype, (outer, D, inner), flush=True)
    plans = [cabi.strided_team_plan(b, outer, D, inner, cabi.dtype_code(dtype)) for b in (0, 1)]
    packs_a_lane = SHAPES[shape][2 if dtype == torch.float32 else 0], SHAPES[shape][1]
    for p, v, small in zip(plans, packs_a_lane, (16, 8)):
        assert p["packs_per_lane"] == v if v else p["packs_per_lane"] <= small, (plans, packs_a_lane)
    g = torch.Generator(device=gpu).manual_seed(D + packs)
    x = torch.empty(outer, D, inner, device=gpu, dtype=dtype).normal_(0, 3.0, generator=g)
    grad = torch.empty_like(x).normal_(0, 1.0, generator=g)
    x[0, D // 3:, 0] = float("-inf")
    x[0, :, 1] = float("-inf")
    x[-1, D - 1, 2] = float("nan")
    x[-1, :, 3] = torch.finfo(dtype).min
    # two columns of every pack that begins or ends a 16-pack piece, and the last ones
    cols = sorted({c for p in range(0, packs, 15) for c in (p * E, p * E + E - 1)} | {0, 1, 2, 3, inner - 1})[:97] + [inner - 1]
    cols = sorted(set(cols))
    pick = lambda t: t[:, :, cols].cpu()  # noqa: E731
    last = lambda a: np.ascontiguousarray(np.moveaxis(to_np32(a), 1, -1))  # noqa: E731
    back = lambda a: np.moveaxis(a, -1, 1)  # noqa: E731

    def given_up(fn):
        try:
            cabi.set_team_wait_us(0)
            return fn()
        finally:
            cabi.set_team_wait_us()

    for mode, is_log in ((cabi.SOFTMAX, False), (cabi.LOG_SOFTMAX, True)):
        what = "%s %s %s" % ("log_softmax" if is_log else "softmax", shape, dtype)
        fwd = lambda: cabi.softmax_strided_fwd(x, 1, mode)  # noqa: E731
        y = fwd()
        oy = back(oracle.softmax_fwd(last(pick(x)), is_log))
        assert_close(pick(y), oy, dtype, what)
        assert torch.equal(y.view(torch.uint8), fwd().view(torch.uint8)), what + ": run to run"
        assert_close(pick(given_up(fwd)), oy, dtype, what + ", every wait given up")
        bwd = lambda: cabi.softmax_strided_bwd(grad, y, 1, mode)  # noqa: E731
        gi = bwd()
        ogi = back(oracle.softmax_bwd(last(pick(grad)), last(pick(y)), is_log))
        yy, terms = pick(y).float().movedim(1, -1), pick(grad).float().movedim(1, -1)
        sl = (rowsum_slack(terms, torch.exp(yy)) if is_log else rowsum_slack(yy * terms, yy)).movedim(-1, 1)
        assert_close(pick(gi), ogi, dtype, what + " backward", slack=sl)
        assert torch.equal(gi.view(torch.uint8), bwd().view(torch.uint8)), what + ": run to run"
        assert_close(pick(given_up(bwd)), ogi, dtype, what + " backward, every wait given up", slack=sl)


@pytest.mark.parametrize("dtype,shape", [(torch.float32, (112, 497, 51)), (torch.bfloat16, (6, 323, 1285))], ids=str)
def test_a_team_of_one_has_no_conditions(cabi, gpu, dtype, shape):
    """A backward whose strips one workgroup holds runs on it in place, under capture and on any stream, with the
    bits of the plain call, and its inputs may be the outputs."""
    outer, D, packs = shape
    inner = packs * (4 if dtype == torch.float32 else 8)
    print("case strided softmax, large teams of one", dtype, (outer, D, inner), flush=True)
    p = cabi.strided_team_plan(1, outer, D, inner, cabi.dtype_code(dtype))
    assert p["team"] == 1 and p["packs_per_lane"] > 8, p
    g = torch.Generator(device=gpu).manual_seed(D)
    grad = torch.empty(outer, D, inner, device=gpu, dtype=dtype).normal_(0, 1.0, generator=g)
    y = torch.softmax(torch.empty(outer, D, inner, device=gpu).normal_(0, 3.0, generator=g), 1).to(dtype)
    for mode in (cabi.SOFTMAX, cabi.LOG_SOFTMAX):
        want = cabi.softmax_strided_bwd(grad, y, 1, mode)
        yd, gd = y.double(), grad.double()
        ref = gd - yd.exp() * gd.sum(1, keepdim=True) if mode else yd * (gd - (yd * gd).sum(1, keepdim=True))
        # (a few ulps of the magnitudes' sum, as for any float32 sum in another order)
        mag = yd.exp() * gd.abs().sum(1, keepdim=True) if mode else yd * (yd * gd).abs().sum(1, keepdim=True)
        assert_close(want, ref.float().cpu().numpy(), dtype, "mode %d" % mode, slack=(mag * 2.0 ** -21).float().cpu())
        del yd, gd, ref, mag
        for over in (0, 1):
            a, b = grad.clone(), y.clone()
            assert torch.equal(cabi.softmax_strided_bwd(a, b, 1, mode, gi=(a, b)[over]), want), "in place over %d" % over
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            assert torch.equal(cabi.softmax_strided_bwd(grad, y, 1, mode), want)
        torch.cuda.current_stream().wait_stream(s)
        gi = torch.empty_like(grad)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            cabi.softmax_strided_bwd(grad, y, 1, mode, gi=gi)
        for _ in range(3):
            gi.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(gi, want), "replayed"


@pytest.mark.parametrize("shape", [(40, 5686, 18), (40, 4286, 28), (1, 12899, 484)], ids=str)
def test_safe_softmax_and_outputs_of_another_type(cabi, gpu, shape):
    """Safe softmax and float32 gradients with a float16 grad_input on large teams, and a float16 forward with a
    float32 output, which keeps to small ones, at the same sizes: against float64 on the GPU, and with every wait
    given up."""
    outer, D, packs = shape
    print("case strided softmax, large teams, other types", shape, flush=True)
    g = torch.Generator(device=gpu).manual_seed(D + 5)

    def both(fn):
        a = fn()
        try:
            cabi.set_team_wait_us(0)
            return a, fn()
        finally:
            cabi.set_team_wait_us()

    for dtype in (torch.float16, torch.float32):
        inner = packs * (4 if dtype == torch.float32 else 8)
        x = torch.empty(outer, D, inner, device=gpu, dtype=dtype).normal_(0, 3.0, generator=g)
        x[0, D // 3:, 0] = float("-inf")
        x[-1, :, 1] = float("-inf")
        assert cabi.strided_team_plan(0, outer, D, inner, cabi.dtype_code(dtype))["packs_per_lane"] > 16
        want = torch.softmax(x.double(), 1)
        nan = want.isnan()
        assert int(nan.sum()) == D
        for y in both(lambda: cabi.softmax_strided_fwd(x, 1, cabi.SAFE_SOFTMAX)):
            assert bool((y[-1, :, 1] == 0).all()), "zeros for a column without a finite element"
            assert_close(y, want.masked_fill(nan, 0).float().cpu().numpy(), dtype, "safe softmax")
        if dtype == torch.float16:
            for y in both(lambda: cabi.softmax_strided_fwd(x, 1, cabi.SOFTMAX, out_dtype=torch.float32)):
                assert_close(y, want.float().cpu().numpy(), torch.float32, "float16 -> float32")
            for y in both(lambda: cabi.softmax_strided_fwd(x, 1, cabi.LOG_SOFTMAX, out_dtype=torch.float32)):
                ref = torch.log_softmax(x.double(), 1)
                assert_close(y, ref.float().cpu().numpy(), torch.float32, "float16 -> float32, log")
            continue
        y = torch.softmax(torch.empty(outer, D, inner, device=gpu).normal_(0, 3.0, generator=g), 1)
        grad = torch.empty(outer, D, inner, device=gpu).normal_(generator=g)
        assert cabi.strided_team_plan(1, outer, D, inner, cabi.F32)["packs_per_lane"] > 8
        yd, gd = y.double(), grad.double()
        for mode in (cabi.SOFTMAX, cabi.LOG_SOFTMAX):
            want = gd - yd.exp() * gd.sum(1, keepdim=True) if mode else yd * (gd - (yd * gd).sum(1, keepdim=True))
            mag = yd.exp() * gd.abs().sum(1, keepdim=True) if mode else yd * (yd * gd).abs().sum(1, keepdim=True)
            # (a few ulps of the magnitudes' sum, as for any float32 sum in another order)
            for gi in both(lambda: cabi.softmax_strided_bwd(grad, y, 1, mode, gi_dtype=torch.float16)):
                assert_close(gi, want.float().cpu().numpy(), torch.float16, "float32 -> float16 mode %d" % mode,
                             slack=(mag * 2.0 ** -21).float().cpu())
