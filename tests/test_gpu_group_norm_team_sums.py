"""GroupNorm backward by teams that write dgamma / dbeta themselves (gn_bwd_team_kernel with SUMS): one and several
samples, one and several groups a team, one and several workgroups a channel, beside shapes whose teams leave
partial rows; against float64 on the GPU, from run to run, with every wait given up, and with one of the two wanted."""
import ctypes
import os
import subprocess

import pytest
import torch

from helpers import assert_close, colsum_slack

pytestmark = pytest.mark.gpu

# (N, C, side, groups): whether a team sees all samples of its channels
SHAPES = {(1, 128, 200, 32): True, (2, 256, 256, 32): True, (3, 96, 144, 12): False, (2, 128, 504, 8): True,
          (4, 128, 256, 32): False}


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    here = os.path.dirname(os.path.abspath(__file__))
    out = str(tmp_path_factory.mktemp("rules") / "libplan_rules.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wno-unknown-pragmas", "-shared", "-fPIC",
                    os.path.join(here, "native", "plan_rules.cpp"), "-o", out], check=True)
    return ctypes.CDLL(out)


@pytest.mark.parametrize("dtype,wdtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32),
                                          (torch.float32, torch.float32)], ids=str)
@pytest.mark.parametrize("shape", list(SHAPES), ids=str)
def test_teams_that_sum_their_channels(cabi, gpu, rules, shape, dtype, wdtype):
    N, C, side, groups = shape
    print("case group norm team sums", dtype, shape, flush=True)
    D, hw, i64 = C // groups, side * side, ctypes.c_int64
    plan = (i64 * 5)()
    rules.rule_gn_bwd_team(i64(N * groups), i64(D), i64(hw * dtype.itemsize // 16), dtype.itemsize, plan)
    if dtype != torch.float32:
        assert plan[0] > 0 and not plan[3]
        assert rules.rule_gn_team_sums(i64(N * groups), i64(groups), i64(plan[4] // plan[0])) == SHAPES[shape]
    g = torch.Generator(device=gpu).manual_seed(C + side)
    x = torch.empty(N, C, side, side, device=gpu).normal_(0.3, 1.0, generator=g).to(dtype)
    dy = torch.empty(N, C, side, side, device=gpu).normal_(generator=g).to(dtype)
    w = (1 + 0.1 * torch.empty(C, device=gpu).normal_(generator=g)).to(wdtype)
    _, mean, rstd = cabi.group_norm_fwd(x, w, None, groups, 1e-5)
    run = lambda **k: cabi.group_norm_bwd(dy, x, mean, rstd, w, groups, **k)  # noqa: E731
    dx, dg, db = run()
    xh = (x.double().view(N, groups, -1) - mean.double().view(N, groups, 1)) * rstd.double().view(N, groups, 1)
    terms = (dy.double() * xh.view_as(dy)).view(N, C, hw).transpose(0, 1).reshape(C, -1).t().cpu()
    dyt = dy.double().view(N, C, hw).transpose(0, 1).reshape(C, -1).t().cpu()
    gy = (dy.double() * w.double().view(1, C, 1, 1)).view(N, groups, -1)
    rdx = (gy - gy.mean(-1, keepdim=True) - xh * (gy * xh).mean(-1, keepdim=True)) * rstd.double().view(N, groups, 1)
    what = "%s %s" % (shape, dtype)

    def check(dx, dg, db, what):
        assert_close(dx, rdx.view_as(dx).float().cpu().numpy(), dtype, "dx " + what)
        assert_close(dg, terms.sum(0).float().numpy(), wdtype, "dgamma " + what, slack=colsum_slack(terms))
        assert_close(db, dyt.sum(0).float().numpy(), wdtype, "dbeta " + what, slack=colsum_slack(dyt))

    check(dx, dg, db, what)
    for a, b in zip(run(), (dx, dg, db)):
        assert torch.equal(a, b), "run to run " + what
    assert torch.equal(run(want=(True, True, False))[1], dg) and torch.equal(run(want=(True, False, True))[2], db)
    try:
        cabi.set_team_wait_us(0)
        check(*run(), what + ", every wait given up")
    finally:
        cabi.set_team_wait_us()
