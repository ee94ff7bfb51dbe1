"""GroupNorm backward where a team of workgroups works through several slabs, the next one on its
way while one is exchanged and written (the reference reads dY and X twice,
src/ATen/native/xpu/sycl/GroupNormKernels.cpp:1088-1165 and 1353-1589): one to eight slabs a
team, channels that end inside a workgroup's packs, teams too large for it, and
the path of a workgroup whose wait gives up, against the oracle."""
import pytest
import torch

from helpers import assert_close, gen, to_np32

pytestmark = pytest.mark.gpu

# (N, C, packs a channel, groups, dtype), of 512 workgroups: teams of 8, 140 slabs on 64 of them
# (three rounds, the last for 12 teams), channels one pack short of their workgroup's; 80 slabs
# (two rounds); 4 teams of 128, 32 slabs (eight rounds); one team of 440 and seven slabs, the last
# workgroup of a channel half full; one slab a team; one team of 264 with eight packs a lane; 224
# slabs on 42 teams of 12, eight packs a lane (six rounds), and 96 on 10 of 48 (ten), where the
# layout that looks ahead would fill its workgroups less well
SHAPES = [(70, 16, 2047, 2, torch.bfloat16), (40, 16, 1100, 2, torch.float16),
          (4, 128, 16384, 8, torch.float32), (7, 8, 55 * 2048 - 1000, 1, torch.float32),
          (2, 16, 1025, 2, torch.float32), (1, 16, 65 * 2048 - 10, 2, torch.float32),
          (28, 96, 2704, 8, torch.float32), (3, 512, 11552, 32, torch.bfloat16)]


@pytest.mark.parametrize("N,C,packs,groups,dtype", SHAPES, ids=str)
def test_several_slabs_a_team(cabi, oracle, gpu, N, C, packs, groups, dtype):
    HxW = packs * (4 if dtype == torch.float32 else 8)
    print("case group norm backward rounds", dtype, (N, C, HxW, groups), flush=True)
    g = gen(2400 + packs)
    x = (0.5 + torch.randn(N, C, HxW, generator=g)).to(dtype)
    dy = torch.randn(N, C, HxW, generator=g).to(dtype)
    gamma = (1 + 0.1 * torch.randn(C, generator=g)).to(dtype)
    xg, dyg, gg = x.to(gpu), dy.to(gpu), gamma.to(gpu)
    what = "[%d, %d, %d] in %d groups %s" % (N, C, HxW, groups, dtype)
    _, mean, rstd = cabi.group_norm_fwd(xg, gg, None, groups, 1e-5)
    odx, odg, odb = oracle.group_norm_bwd(to_np32(dy), to_np32(x), groups, to_np32(mean.float()),
                                          to_np32(rstd.float()), to_np32(gamma))
    D = C // groups
    mu = mean.float().cpu().reshape(N, groups, 1, 1)
    rs = rstd.float().cpu().reshape(N, groups, 1, 1)
    xhat = ((x.float().reshape(N, groups, D, HxW) - mu) * rs).reshape(N, C, HxW)
    # (float32 partial sums: a few ulps of the sum of the magnitudes, per channel)
    sl_g = (dy.float() * xhat).abs().sum(dim=(0, 2)) * 2.0 ** -22
    sl_b = dy.float().abs().sum(dim=(0, 2)) * 2.0 ** -22
    first = None
    for wait in (None, None, 0):
        try:
            if wait is not None:
                cabi.set_team_wait_us(wait)
            dx, dg, db = cabi.group_norm_bwd(dyg, xg, mean, rstd, gg, groups)
            torch.cuda.synchronize()
        finally:
            cabi.set_team_wait_us()
        assert_close(dx, odx, dtype, "dx %s wait %s" % (what, wait))
        assert_close(dg.float(), odg, dtype, "dgamma %s wait %s" % (what, wait), slack=sl_g)
        assert_close(db.float(), odb, dtype, "dbeta %s wait %s" % (what, wait), slack=sl_b)
        if first is None:
            first = (dx, dg, db)
        elif wait is None:
            assert all(torch.equal(a, b) for a, b in zip(first, (dx, dg, db))), "twice " + what
