"""LayerNorm / RMSNorm over few rows beyond one workgroup's registers: the backward in two launches
(norm_bwd_few_rows_kernel: dX, dgamma and dbeta complete, no partial rows) and the forward of fewer than eight rows
by small teams of workgroups (norm_fwd_team_kernel).  The regime of the reference's split-row kernels
(src/ATen/native/xpu/sycl/Norm.h:632-812; column sums LayerNormKernels.cpp:1140-1406).  Against the CPU oracle:
rows ragged and whole, off a 16-byte boundary, in place (where no pack may reach into a neighbour's columns), with a
residual gradient, one of dgamma / dbeta alone, a workspace without the row sums' part, and every wait given up."""
import pytest
import torch

from helpers import assert_close, colsum_slack, gen, offset_view, to_np32

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.float16, torch.bfloat16]
# (rows, elements beyond whole packs, whole packs): the wavefronts that share a piece of columns.  Fewer rows than a
# wavefront takes at once, rows missing in its last turn, the most rows; the last piece one pack or one element
SHAPES = {(2, 0, 8200): 8, (3, 1, 6000): 8, (9, 0, 12800): 8, (33, 3, 8193): 8, (64, 0, 5121): 8, (128, 1, 4160): 8,
          (11, 0, 20001): 4, (10, 1, 20000): 4, (7, 0, 40001): 2, (3, 3, 40000): 2, (3, 0, 70001): 1, (5, 1, 100000): 1}


def _inputs(M, N, dtype, seed):
    g = gen(seed)
    x = (0.5 + torch.randn(M, N, generator=g)).to(dtype)
    dy = torch.randn(M, N, generator=g).to(dtype)
    return x, dy, (1 + 0.1 * torch.randn(N, generator=g)).to(dtype), (0.1 * torch.randn(N, generator=g)).to(dtype)


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("shape", list(SHAPES), ids=str)
def test_backward_against_oracle(cabi, oracle, gpu, dtype, shape):
    M, over, packs = shape
    N = packs * (4 if dtype == torch.float32 else 8) + over
    print("case few rows", dtype, (M, N), flush=True)
    code = cabi.dtype_code(dtype)
    for op in (cabi.OP_LAYER_NORM_BWD, cabi.OP_RMS_NORM_BWD):
        assert cabi.few_rows_plan(op, M, N, code, code)["waves"] == SHAPES[shape]
    x, dy, gamma, beta = _inputs(M, N, dtype, 4100 + M)
    xg, dyg, gg = x.to(gpu), dy.to(gpu), gamma.to(gpu)
    _, mean, rstd = cabi.layer_norm_fwd(xg, gg, None, 1e-5)
    odx, odg, odb = oracle.layer_norm_bwd(to_np32(dy), to_np32(x), (N,), to_np32(mean), to_np32(rstd), to_np32(gamma))
    xhat = (x.double() - mean.cpu().double().reshape(M, 1)) * rstd.cpu().double().reshape(M, 1)
    slack = (None, colsum_slack(dy.double() * xhat), colsum_slack(dy)) if dtype == torch.float32 else (None,) * 3

    def check(got, what):
        for name, a, o, s in zip(("dx", "dgamma", "dbeta"), got, (odx, odg, odb), slack):
            if a is not None:
                assert_close(a, o, dtype, "%s %s %s" % (name, (M, N), what), slack=s)

    first = cabi.layer_norm_bwd(dyg, xg, mean, rstd, gg)
    check(first, "")
    for a, b in zip(first, cabi.layer_norm_bwd(dyg, xg, mean, rstd, gg)):
        assert torch.equal(a, b), "run to run"
    check(cabi.layer_norm_bwd(offset_view(dyg, 1), offset_view(xg, 3), mean, rstd, offset_view(gg, 1)), "off a boundary")
    check(cabi.layer_norm_bwd(dyg, xg, mean, rstd, gg, want=(True, True, False)), "without dbeta")
    check(cabi.layer_norm_bwd(dyg, xg, mean, rstd, gg, want=(True, False, True)), "without dgamma")
    over_dy, over_x = dyg.clone(), xg.clone()
    check(cabi.layer_norm_bwd(over_dy, xg, mean, rstd, gg, dx=over_dy), "dx over dy")
    check(cabi.layer_norm_bwd(dyg, over_x, mean, rstd, gg, dx=over_x), "dx over x")
    p = cabi.plan(cabi.OP_LAYER_NORM_BWD, M, N, code, code)
    columns = torch.empty(2 * p["partial_rows"] * N * 4, dtype=torch.uint8, device=gpu)
    check(cabi.layer_norm_bwd(dyg, xg, mean, rstd, gg, workspace=columns), "workspace of the column sums alone")
    up = torch.randn(M, N, generator=gen(7)).to(dtype)
    dh, dg, db = cabi.add_layer_norm_bwd(dyg, up.to(gpu), xg, mean, rstd, gg)
    assert_close(dh, torch.as_tensor(odx) + up.float(), dtype, "residual gradient %s" % ((M, N),))
    check((None, dg, db), "with a residual gradient")
    _, rr = cabi.rms_norm_fwd(xg, gg, 1e-6)
    rdx, rdg = cabi.rms_norm_bwd(dyg, xg, rr, gg)
    ordx, ordg = oracle.rms_norm_bwd(to_np32(dy), to_np32(x), (N,), to_np32(rr), to_np32(gamma))
    terms = dy.double() * x.double() * rr.cpu().double().reshape(M, 1)
    assert_close(rdx, ordx, dtype, "rms dx %s" % ((M, N),))
    assert_close(rdg, ordg, dtype, "rms dgamma %s" % ((M, N),), slack=None if slack[1] is None else colsum_slack(terms))


@pytest.mark.parametrize("M,N,dtype", [(48, 112000, torch.float32), (48, 320000, torch.bfloat16)], ids=str)
def test_rows_of_teams_where_no_team_can_run(cabi, oracle, gpu, M, N, dtype):
    """Rows beyond the line of the teams, dX over an input or captured: the two launches again, whose bits the call
    with a residual gradient of zeros shows (it never has teams; -0 equals 0)."""
    print("case few rows, no team", dtype, (M, N), flush=True)
    code = cabi.dtype_code(dtype)
    assert cabi.few_rows_plan(cabi.OP_LAYER_NORM_BWD, M, N, code, code)["waves"] == 0
    assert cabi.plan(cabi.OP_LAYER_NORM_BWD, M, N, code, code)["row_chunks"] > 1
    x, dy, gamma, _ = _inputs(M, N, dtype, 4300 + M)
    xg, dyg, gg = x.to(gpu), dy.to(gpu), gamma.to(gpu)
    _, mean, rstd = cabi.layer_norm_fwd(xg, gg, None, 1e-5)
    two = cabi.add_layer_norm_bwd(dyg, torch.zeros_like(xg), xg, mean, rstd, gg)
    o = oracle.layer_norm_bwd(to_np32(dy), to_np32(x), (N,), to_np32(mean), to_np32(rstd), to_np32(gamma))
    xhat = (x.double() - mean.cpu().double().reshape(M, 1)) * rstd.cpu().double().reshape(M, 1)
    slack = (None, colsum_slack(dy.double() * xhat), colsum_slack(dy)) if dtype == torch.float32 else (None,) * 3
    for name, a, b, s in zip(("dx", "dgamma", "dbeta"), two, o, slack):
        assert_close(a, b, dtype, name, slack=s)
    for which in (0, 1):
        pair = [dyg.clone(), xg.clone()]
        got = cabi.layer_norm_bwd(*pair, mean, rstd, gg, dx=pair[which])
        assert all(torch.equal(a, b) for a, b in zip(got, two)), "dx over %s" % ("dy", "x")[which]
    torch.cuda.synchronize()
    out = torch.empty_like(xg), torch.empty_like(gg), torch.empty_like(gg)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        cabi.layer_norm_bwd(dyg, xg, mean, rstd, gg, dx=out[0], dgamma=out[1], dbeta=out[2])
    for k in range(3):
        for t in out:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, two)), "replay %d" % k
        for name, a, b, s in zip(("dx", "dgamma", "dbeta"), cabi.layer_norm_bwd(dyg, xg, mean, rstd, gg), o, slack):
            assert_close(a, b, dtype, name + " by teams", slack=s)


@pytest.mark.parametrize("dtype", DTYPES, ids=str)
@pytest.mark.parametrize("M,packs", [(1, 32769), (2, 40000), (3, 300001), (7, 20000), (7, 70000)], ids=str)
def test_forward_by_small_teams(cabi, oracle, gpu, dtype, M, packs):
    """Fewer than eight rows: teams of at most 64 workgroups, and what a workgroup does without its team."""
    N = packs * (4 if dtype == torch.float32 else 8)
    print("case few rows forward", dtype, (M, N), flush=True)
    p = cabi.plan(cabi.OP_LAYER_NORM_FWD, M, N, cabi.dtype_code(dtype), cabi.dtype_code(dtype))
    assert p["resident"] == 0 and 2 <= p["row_chunks"] <= 64 and p["grid_blocks"] == M * p["row_chunks"], p
    x, _, gamma, beta = _inputs(M, N, dtype, 4200 + M)
    xg, gg, bg = x.to(gpu), gamma.to(gpu), beta.to(gpu)
    oy, om, orr = oracle.layer_norm_fwd(to_np32(x), (N,), to_np32(gamma), to_np32(beta), 1e-5)
    ory, orr2 = oracle.rms_norm_fwd(to_np32(x), (N,), to_np32(gamma), 1e-6)

    def check(what):
        y, mean, rstd = cabi.layer_norm_fwd(xg, gg, bg, 1e-5)
        assert_close(y, oy, dtype, "y " + what)
        assert_close(mean, om.reshape(-1), dtype, "mean " + what)
        assert_close(rstd, orr.reshape(-1), dtype, "rstd " + what)
        ry, rr = cabi.rms_norm_fwd(xg, gg, 1e-6)
        assert_close(ry, ory, dtype, "rms y " + what)
        assert_close(rr, orr2.reshape(-1), dtype, "rms rstd " + what)
        return y, mean, rstd, ry, rr

    for a, b in zip(check(""), check("again")):
        assert torch.equal(a, b), "run to run"
    try:
        cabi.set_team_wait_us(0)
        check("every wait given up")
    finally:
        cabi.set_team_wait_us()
    over = xg.clone()
    y, _, _ = cabi.layer_norm_fwd(over, gg, bg, 1e-5, y=over)
    assert_close(y, oy, dtype, "in place")
