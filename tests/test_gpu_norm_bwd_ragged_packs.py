"""Norm backward of ragged rows (N not a whole number of packs) off a 16-byte boundary: a row's last
pack is read as the last whole pack inside the row and moved into place.  Every remainder, rows just
above a pack, rows shorter than one (a forced layout included), NaN on both sides of every input,
against the float64 oracle (the reference's unaligned path: can_vectorize() false,
src/ATen/native/xpu/sycl/LayerNormKernels.cpp:1121-1163)."""
import pytest
import torch

from helpers import assert_close, gen, to_np32

pytestmark = pytest.mark.gpu


def _inside(t, off, gpu):
    buf = torch.full((t.numel() + 64,), float("nan"), dtype=t.dtype, device=gpu)
    v = buf[16 + off:16 + off + t.numel()].view(t.shape)
    v.copy_(t)
    return v


def _check(cabi, oracle, gpu, M, N, dtype, offs):
    print("case ragged norm backward", dtype, (M, N), offs, flush=True)
    g = gen(2500 + N + offs[0])
    x = (0.5 + torch.randn(M, N, generator=g)).to(dtype)
    dy = torch.randn(M, N, generator=g).to(dtype)
    gamma = (1 + 0.1 * torch.randn(N, generator=g)).to(dtype)
    xg, dyg = _inside(x, offs[0], gpu), _inside(dy, offs[1], gpu)
    gg = _inside(gamma, 1, gpu)
    what = "[%d, %d] %s offsets %s" % (M, N, dtype, offs)
    _, mean, rstd = cabi.layer_norm_fwd(xg, gg, None, 1e-5)
    xhat = (x.float() - mean.float().cpu()[:, None]) * rstd.float().cpu()[:, None]
    # float32 sums over the rows, in another order: a few ulps of the magnitudes' sum
    slack_g = (dy.float() * xhat).abs().sum(dim=0) * 2.0 ** -21
    slack_b = dy.float().abs().sum(dim=0) * 2.0 ** -21
    odx, odg, odb = oracle.layer_norm_bwd(to_np32(dy), to_np32(x), (N,), to_np32(mean),
                                          to_np32(rstd), to_np32(gamma))
    over = _inside(dy, offs[1], gpu)
    for dx_out, dyt in ((None, dyg), (over, over)):
        dx, dg, db = cabi.layer_norm_bwd(dyt, xg, mean, rstd, gg, dx=dx_out)
        assert_close(dx, odx, dtype, "layer_norm dx " + what)
        assert_close(dg, odg, dtype, "layer_norm dgamma " + what, slack=slack_g)
        assert_close(db, odb, dtype, "layer_norm dbeta " + what, slack=slack_b)
    _, rr = cabi.rms_norm_fwd(xg, gg, 1e-6)
    slack_g = (dy.float() * x.float() * rr.float().cpu()[:, None]).abs().sum(dim=0) * 2.0 ** -21
    rdx, rdg = cabi.rms_norm_bwd(dyg, xg, rr, gg)
    ordx, ordg = oracle.rms_norm_bwd(to_np32(dy), to_np32(x), (N,), to_np32(rr), to_np32(gamma))
    assert_close(rdx, ordx, dtype, "rms_norm dx " + what)
    assert_close(rdg, ordg, dtype, "rms_norm dgamma " + what, slack=slack_g)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=str)
@pytest.mark.parametrize("offs", [(2, 2), (1, 7), (5, 0)], ids=str)
def test_ragged_rows_off_a_boundary(cabi, oracle, gpu, dtype, offs):
    widths = [3, 9, 129, 130, 131, 132, 133, 134, 135, 257, 1001, 1027, 2050, 2801, 4097, 8195]
    for N in widths:
        _check(cabi, oracle, gpu, 7 if N % 2 else 1100, N, dtype, offs)


@pytest.mark.parametrize("M,N,dtype", [(1, 8193, torch.float16), (300, 10005, torch.bfloat16),
                                       (300, 12295, torch.float16), (270, 13311, torch.bfloat16),
                                       (270, 16383, torch.float16), (270, 12289, torch.float32),
                                       (8150, 6145, torch.float32)], ids=str)
def test_both_ways_of_reading_a_ragged_row(cabi, oracle, gpu, M, N, dtype):
    """Rows on 1024 lanes on both sides of the line between whole packs and element loads; two of the calls run on
    whole wavefronts, whose last pack is the row's last whole pack."""
    code = cabi.dtype_code(dtype)
    w = cabi.waves_plan(cabi.OP_LAYER_NORM_BWD, M, N, code, code)["waves"]
    assert (w > 0) == ((M, N) in ((300, 10005), (8150, 6145)))
    _check(cabi, oracle, gpu, M, N, dtype, (1, 3))


@pytest.mark.parametrize("M,N", [(33000, 3071 + 64), (16500, 6145), (13100, 7777)], ids=str)
def test_element_loads_of_float_tensors_beyond_100_million_elements(cabi, gpu, M, N):
    """Float32 rows that fill most of their lanes, in tensors far beyond the caches, keep the element loads: against
    float64 on the GPU, NaN on both sides of the inputs."""
    print("case float32 element loads", (M, N), flush=True)
    for op in (cabi.OP_LAYER_NORM_BWD, cabi.OP_RMS_NORM_BWD):
        p = cabi.plan(op, M, N, cabi.F32, cabi.F32)
        assert cabi.waves_plan(op, M, N, cabi.F32, cabi.F32)["waves"] == 0 and M * N > 100000000
        assert p["lanes_per_row"] in (256, 512) and 16 * N * 4 > 9 * 16 * p["lanes_per_row"] * p["packs_per_lane"]
    g = torch.Generator(device=gpu).manual_seed(2570 + N)
    x, dy = (_inside(torch.empty(M, N, device=gpu).normal_(generator=g), o, gpu) for o in (1, 3))
    w = _inside(1 + 0.1 * torch.empty(N, device=gpu).normal_(generator=g), 1, gpu)
    for rms in (False, True):
        # (a slab of columns or rows at a time in float64)
        xd = x.double()
        mu = xd.new_zeros(M, 1) if rms else xd.mean(1, keepdim=True)
        rs = (xd.sub_(mu).square().mean(1, keepdim=True) + 1e-5).rsqrt()
        xh = xd.mul_(rs)
        stats = rs.view(-1).float(), mu.view(-1).float()
        out = cabi.rms_norm_bwd(dy, x, stats[0], w) if rms else cabi.layer_norm_bwd(dy, x, stats[1], stats[0], w)
        terms = dy.double().mul_(xh)
        # (float32 sums over the rows of terms with the statistics' own rounding: a few ulps of the magnitudes' sum)
        assert_close(out[1], to_np32(terms.sum(0)), torch.float32, "dgamma", slack=(terms.abs().sum(0) * 2.0 ** -20).cpu())
        s2 = terms.mul_(w.double()).mean(1, keepdim=True)
        del terms
        if not rms:
            assert_close(out[2], to_np32(dy.double().sum(0)), torch.float32, "dbeta", slack=(dy.abs().sum(0) * 2.0 ** -21).cpu())
        gy = dy.double().mul_(w.double())
        want = gy.sub_(0 if rms else gy.mean(1, keepdim=True)).sub_(xh.mul_(s2)).mul_(rs)
        for r in range(0, M, 4096):
            assert_close(out[0][r:r + 4096], to_np32(want[r:r + 4096]), torch.float32, "dx from row %d" % r)
        del xd, xh, gy, want, out


@pytest.mark.parametrize("N,dtype", [(5, torch.float16), (7, torch.bfloat16), (3, torch.float32)],
                         ids=str)
def test_rows_shorter_than_a_pack_on_a_forced_layout(cabi, oracle, gpu, N, dtype):
    packs = 4 if dtype == torch.float32 else 2
    try:
        for op in (cabi.OP_LAYER_NORM_BWD, cabi.OP_RMS_NORM_BWD):
            cabi.set_override(op, 32, packs, 0, 0)
        _check(cabi, oracle, gpu, 300, N, dtype, (1, 3))
    finally:
        cabi.clear_overrides()


@pytest.mark.parametrize("M,N,dtype", [(40, 8193, torch.float16), (40, 16383, torch.bfloat16),
                                       (40, 5001, torch.float32), (8150, 6145, torch.float32)], ids=str)
def test_the_residual_gradient_on_either_way_of_reading(cabi, gpu, M, N, dtype):
    """The fused backward, dx + dh rounded once, on the same two ways: against the plain backward of the
    same rows in float64 on the GPU."""
    print("case ragged norm backward with the residual gradient", dtype, (M, N), flush=True)
    g = torch.Generator(device=gpu).manual_seed(2560 + N)
    h, dy, dh = (torch.empty(M, N, device=gpu).normal_(generator=g).to(dtype) for _ in range(3))
    gamma = (1 + 0.1 * torch.empty(N, device=gpu).normal_(generator=g)).to(dtype)
    _, mean, rstd = cabi.layer_norm_fwd(h, gamma, None, 1e-5)
    dx, dg, db = cabi.add_layer_norm_bwd(dy, dh, h, mean, rstd, gamma)[:3]
    xhat = (h.double() - mean.double().view(M, 1)) * rstd.double().view(M, 1)
    gy = dy.double() * gamma.double()
    want = (gy - gy.mean(1, keepdim=True) - xhat * (gy * xhat).mean(1, keepdim=True)) * rstd.double().view(M, 1) + dh.double()
    assert_close(dx, to_np32(want.float()), dtype, "dx [%d, %d]" % (M, N))
    # float32 sums over the rows: a few ulps of the magnitudes' sum
    for got, terms, what in ((dg, dy.double() * xhat, "dgamma"), (db, dy.double(), "dbeta")):
        assert_close(got, to_np32(terms.sum(0).float()), dtype, "%s [%d, %d]" % (what, M, N),
                     slack=(terms.abs().sum(0) * 2.0 ** -21).float().cpu())
