"""Long norm forward rows whose teams share the rows out evenly over two or three rounds, beside calls whose teams
are as many as fit: full and nearly empty last chunks, against float64."""
import pytest
import torch

from helpers import assert_close, gen

pytestmark = pytest.mark.gpu

EPS = 1e-5


@pytest.mark.parametrize("dtype,wdtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32),
                                          (torch.float32, torch.float32)], ids=str)
@pytest.mark.parametrize("M,packs,even", [(140, 27072, "all"), (139, 27073, "all"), (131, 3 * 8192 - 511, ""),
                                          (259, 16385, ""), (33, 137936, "same"), (358, 20480, "all")])
def test_even_rounds(cabi, gpu, dtype, wdtype, M, packs, even):
    """even: whether the rule takes the call, with all weights or only those of the rows' type."""
    N = packs * (4 if dtype == torch.float32 else 8)
    print("case even rounds of teams", dtype, wdtype, (M, N), flush=True)
    p = cabi.plan(cabi.OP_LAYER_NORM_FWD, M, N, cabi.dtype_code(dtype), cabi.dtype_code(wdtype))
    teams, most = p["grid_blocks"] // p["row_chunks"], min(M, 512 // -(-packs // 8192))
    assert (teams < most) == (even == "all" or (even == "same" and dtype == wdtype)), (p, most)
    assert -(-M // teams) == -(-M // most)
    g = gen(M + packs)
    base = (torch.randn(M, 997, generator=g) + 0.5).to(gpu)
    x = base.repeat(1, -(-N // 997))[:, :N].mul(torch.linspace(0.5, 1.5, N, device=gpu)).to(dtype).contiguous()
    w = (1 + 0.1 * torch.randn(N, generator=g)).to(gpu, wdtype)
    b = (0.1 * torch.randn(N, generator=g)).to(gpu, wdtype)
    y, mean, rstd = cabi.layer_norm_fwd(x, w, b, EPS)
    yr, rr = cabi.rms_norm_fwd(x, w, EPS)
    for r in sorted({0, 1, M // 3, M // 2, 2 * M // 3, M - 2, M - 1}):
        xd, what = x[r].double(), "row %d of [%d, %d] %s %s" % (r, M, N, dtype, wdtype)
        mu, var = xd.mean(), xd.var(unbiased=False)
        rs, rq = (var + EPS).rsqrt(), (xd.square().mean() + EPS).rsqrt()
        assert_close(y[r], ((xd - mu) * rs * w.double() + b.double()).cpu().numpy(), dtype, "y " + what)
        assert_close(yr[r], (xd * rq * w.double()).cpu().numpy(), dtype, "rms y " + what)
        stats = torch.stack((mu, rs, rq)).cpu().numpy()
        assert_close(torch.stack((mean[r], rstd[r], rr[r])), stats, torch.float32, "statistics " + what)
