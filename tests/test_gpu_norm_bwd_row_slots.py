"""Norm backward where a workgroup works on several rows at a time: the row slots' column sums are
added through LDS into one partial row (src/ATen/native/xpu/sycl/LayerNormKernels.cpp:1312-1314
sums block buffers likewise).  Lane groups of 8 to 256 lanes, rows that end inside a pack, fewer
rows than slots, and several row blocks a workgroup, against the float64 oracle."""
import pytest
import torch

from helpers import assert_close, gen, to_np32

pytestmark = pytest.mark.gpu

# (row length, dtype): 8 lanes of one pack up to 256 lanes, whole and ragged packs
ROWS = [(16, torch.float32), (61, torch.float32), (256, torch.float32), (1021, torch.float32),
        (1024, torch.float32), (2048, torch.float32), (2112, torch.float32),
        (64, torch.bfloat16), (161, torch.float16), (520, torch.float16), (1001, torch.bfloat16),
        (2560, torch.bfloat16), (4097, torch.float16)]


@pytest.mark.parametrize("N,dtype", ROWS, ids=lambda v: str(v).replace("torch.", ""))
@pytest.mark.parametrize("M", [1, 3, 300, 5003])
def test_column_sums_of_several_row_slots(cabi, oracle, gpu, N, dtype, M):
    print("case norm backward row slots", dtype, (M, N), flush=True)
    g = gen(2300 + N + M)
    x = (0.5 + torch.randn(M, N, generator=g)).to(dtype)
    dy = torch.randn(M, N, generator=g).to(dtype)
    gamma = (1 + 0.1 * torch.randn(N, generator=g)).to(dtype)
    xg, dyg, gg = x.to(gpu), dy.to(gpu), gamma.to(gpu)
    what = "[%d, %d] %s" % (M, N, dtype)
    _, mean, rstd = cabi.layer_norm_fwd(xg, gg, None, 1e-5)
    xhat = (x.float() - mean.float().cpu()[:, None]) * rstd.float().cpu()[:, None]
    # float32 sums over the rows, in another order: a few ulps of the magnitudes' sum
    slack_g = (dy.float() * xhat).abs().sum(dim=0) * 2.0 ** -21
    slack_b = dy.float().abs().sum(dim=0) * 2.0 ** -21
    dx, dg, db = cabi.layer_norm_bwd(dyg, xg, mean, rstd, gg)
    odx, odg, odb = oracle.layer_norm_bwd(to_np32(dy), to_np32(x), (N,), to_np32(mean),
                                          to_np32(rstd), to_np32(gamma))
    assert_close(dx, odx, dtype, "layer_norm dx " + what)
    assert_close(dg, odg, dtype, "layer_norm dgamma " + what, slack=slack_g)
    assert_close(db, odb, dtype, "layer_norm dbeta " + what, slack=slack_b)
    _, rr = cabi.rms_norm_fwd(xg, gg, 1e-6)
    slack_g = (dy.float() * x.float() * rr.float().cpu()[:, None]).abs().sum(dim=0) * 2.0 ** -21
    rdx, rdg = cabi.rms_norm_bwd(dyg, xg, rr, gg)
    ordx, ordg = oracle.rms_norm_bwd(to_np32(dy), to_np32(x), (N,), to_np32(rr), to_np32(gamma))
    assert_close(rdx, ordx, dtype, "rms_norm dx " + what)
    assert_close(rdg, ordg, dtype, "rms_norm dgamma " + what, slack=slack_g)
