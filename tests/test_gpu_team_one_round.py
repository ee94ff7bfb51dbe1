"""LayerNorm / RMSNorm forward of rows held by teams of workgroups (norm_fwd_team_kernel) on both sides of the line
between rows that are all done in one round, whose sums cross as self-validating words, and rows in several, whose
sums cross beside a tag.  The regime of the reference's split-row kernels (src/ATen/native/xpu/sycl/Norm.h:632-812).
Against float64, from run to run, and with every wait given up."""
import pytest
import torch

from helpers import assert_close, gen

pytestmark = pytest.mark.gpu

# teams of 4 to 64 workgroups in a grid of at most 512: each list has counts of rows in one round and in two or more
CASES = [(262144, (8, 32, 60, 64, 86, 102, 128, 129)), (1048576, (8, 10, 15, 16, 17, 32))]


def _check(x, w, b, y, mean, rstd, dtype, what):
    for r in {0, 1, x.shape[0] // 2, x.shape[0] - 1}:
        v = x[r].double()
        mu = v.mean() if mean is not None else torch.zeros((), dtype=torch.float64, device=x.device)
        rs = torch.rsqrt((v - mu).square().mean() + 1e-5)
        e = (v - mu) * rs * w.double() + (b.double() if b is not None else 0)
        assert_close(y[r].cpu(), e.float().cpu(), dtype, "y row %d %s" % (r, what))
        # two roundings to float32 and the square root's own
        assert abs(rstd.reshape(-1)[r].double() - rs) <= 4e-7 * rs, "rstd row %d %s" % (r, what)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=str)
@pytest.mark.parametrize("case", CASES, ids=str)
def test_rounds(cabi, gpu, dtype, case):
    N, counts = case
    g = gen(N)
    x0 = (0.5 + torch.randn(max(counts), N, generator=g)).to(dtype).to(gpu)
    w = (1 + 0.1 * torch.randn(N, generator=g)).to(dtype).to(gpu)
    b = (0.1 * torch.randn(N, generator=g)).to(dtype).to(gpu)
    for M in counts:
        what = "%s %s" % ((M, N), dtype)
        print("case", what, flush=True)
        x = x0[:M]
        run = lambda: (cabi.layer_norm_fwd(x, w, b, 1e-5), cabi.rms_norm_fwd(x, w, 1e-5))
        (y, mean, rstd), (ry, rr) = first = run()
        _check(x, w, b, y, mean, rstd, dtype, what)
        _check(x, w, None, ry, None, rr, dtype, "rms " + what)
        again = run()
        for a, c in zip(first[0] + first[1], again[0] + again[1]):
            assert torch.equal(a, c), "run to run " + what
        try:
            cabi.set_team_wait_us(0)
            (y, mean, rstd), (ry, rr) = run()
            torch.cuda.synchronize()
        finally:
            cabi.set_team_wait_us()
        _check(x, w, b, y, mean, rstd, dtype, what + " every wait given up")
        _check(x, w, None, ry, None, rr, dtype, "rms " + what + " every wait given up")
