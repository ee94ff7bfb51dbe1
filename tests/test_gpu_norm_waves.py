"""LayerNorm / RMSNorm rows on whole wavefronts (norm_waves_kernels.hpp), forward and backward: rows at the edges
of a wavefront, of a lane's packs and of the layouts, more and fewer rows than a workgroup has slots, in tensors
at every alignment whose surroundings are NaN (nothing outside a row is used) and whose outputs' surroundings
stay as they are, against the float64 oracle; the column sums alone have the bits they have beside dX.  Calls of
many rows, whose row loops have steady rounds on one and several slots, against float64 on the GPU."""
import pytest
import torch

from helpers import assert_close, colsum_slack, gen, to_np32, xhat_slack

pytestmark = pytest.mark.gpu

EPS = 1e-5
# row lengths in elements, 16-bit and float32: one lane past a wavefront or a workgroup's layout, the row's last
# pack all but one element another lane's, whole packs, the longest the backward's instances take (calls of few
# rows: some of these run on the general layouts, see STEADY)
N16 = (521, 1025, 1031, 2049, 2304, 4095, 4097, 4608, 5119, 8191, 8193, 12287)
N32 = (1025, 1027, 2049, 3073, 4097, 4607, 6143, 6145, 9215)


def _inside(t, offset):
    """t at `offset` elements into a buffer of NaN."""
    buf = torch.full((t.numel() + offset + 16,), float("nan"), dtype=t.dtype, device=t.device)
    view = buf[offset:offset + t.numel()].view(t.shape)
    view.copy_(t)
    return buf, view


@pytest.mark.parametrize("dtype,wdtype", [(torch.float16, torch.float16), (torch.bfloat16, torch.float32),
                                          (torch.float32, torch.float32)], ids=str)
@pytest.mark.parametrize("M", [256, 331, 1000])
def test_rows_on_whole_wavefronts(cabi, oracle, gpu, dtype, wdtype, M):
    for j, N in enumerate(N32 if dtype == torch.float32 else N16):
        if M * N > 5_000_000:
            continue
        offset = j % 4 if N % 2 else 2 * (j % 2)
        print("case norm rows on whole wavefronts", dtype, wdtype, (M, N), "offset", offset, flush=True)
        g = gen(9000 + 7 * N + M)
        x = (torch.randn(M, N, generator=g) + 0.5).to(dtype)
        x[M // 2] = 0.5  # a constant row: y is beta bit for bit
        dy = torch.randn(M, N, generator=g).to(dtype)
        w = (1 + 0.1 * torch.randn(N, generator=g)).to(wdtype)
        b = (0.1 * torch.randn(N, generator=g)).to(wdtype)
        (_, xg), (_, dyg) = _inside(x.to(gpu), offset), _inside(dy.to(gpu), (offset + 1) % 4)
        (_, wg), (_, bg) = _inside(w.to(gpu), 1), _inside(b.to(gpu), 3)
        what = "[%d, %d] %s %s" % (M, N, dtype, wdtype)
        wn, bn = to_np32(w), to_np32(b)

        ybuf, y = _inside(torch.zeros_like(xg), 3)
        y, mean, rstd = cabi.layer_norm_fwd(xg, wg, bg, EPS, y=y)
        oy, om, orr = oracle.layer_norm_fwd(to_np32(x), (N,), wn, bn, EPS)
        assert_close(y, oy, dtype, "layer_norm y " + what)
        assert_close(mean, om.reshape(-1), torch.float32, "mean " + what)
        assert_close(rstd, orr.reshape(-1), torch.float32, "rstd " + what)
        assert torch.isnan(ybuf[:3]).all() and torch.isnan(ybuf[3 + M * N:]).all(), "outside y " + what
        assert torch.equal(y[M // 2], bg.to(dtype)), "constant row " + what
        _, xin = _inside(xg, 1)
        y2, _, _ = cabi.layer_norm_fwd(xin, wg, bg, EPS, y=xin)
        assert_close(y2, oy, dtype, "in place " + what)
        yr, rr = cabi.rms_norm_fwd(xg, wg, EPS)
        ory, orr = oracle.rms_norm_fwd(to_np32(x), (N,), wn, EPS)
        assert_close(yr, ory, dtype, "rms_norm y " + what)

        # (the backward on rows with a spread: a constant row's dX is all cancellation)
        x[M // 2] = torch.randn(N, generator=g).to(dtype)
        xg[M // 2] = x[M // 2].to(gpu)
        _, mean, rstd = cabi.layer_norm_fwd(xg, wg, bg, EPS)
        _, rr = cabi.rms_norm_fwd(xg, wg, EPS)
        dbuf, dx = _inside(torch.zeros_like(xg), 1)
        dx, dg, db = cabi.layer_norm_bwd(dyg, xg, mean, rstd, wg, dx=dx)
        odx, odg, odb = oracle.layer_norm_bwd(to_np32(dy), to_np32(x), (N,), to_np32(mean), to_np32(rstd), wn)
        assert_close(dx, odx, dtype, "layer_norm dx " + what)
        xhat = (x.float() - mean.cpu().reshape(M, 1)) * rstd.cpu().reshape(M, 1)
        assert_close(dg, odg, wdtype, "dgamma " + what, slack=colsum_slack(dy.float() * xhat) + xhat_slack(dy.float(), mean, rstd))
        assert_close(db, odb, wdtype, "dbeta " + what, slack=colsum_slack(dy.float()))
        assert torch.isnan(dbuf[:1]).all() and torch.isnan(dbuf[1 + M * N:]).all(), "outside dx " + what
        n, dg1, db1 = cabi.layer_norm_bwd(dyg, xg, mean, rstd, wg, want=(False, True, True))
        assert n is None and torch.equal(dg1, dg) and torch.equal(db1, db), "sums alone " + what
        dx1, _, _ = cabi.layer_norm_bwd(dyg, xg, mean, rstd, wg, want=(True, False, False))
        assert torch.equal(dx1, dx), "dX alone " + what
        _, din = _inside(dyg, 1)
        din, _, _ = cabi.layer_norm_bwd(din, xg, mean, rstd, wg, dx=din)
        assert torch.equal(din, dx), "dX over dY " + what
        rdx, rdg = cabi.rms_norm_bwd(dyg, xg, rr, wg)
        rodx, rodg = oracle.rms_norm_bwd(to_np32(dy), to_np32(x), (N,), to_np32(rr), wn)
        assert_close(rdx, rodx, dtype, "rms_norm dx " + what)
        assert_close(rdg, rodg, wdtype, "rms dgamma " + what,
                     slack=colsum_slack(dy.float() * x.float() * rr.cpu().reshape(M, 1)))


# (rows, elements): whether the LayerNorm forward and backward, the RMSNorm forward and backward run on whole
# wavefronts there.  16 bits: eight to two row slots with steady rounds and rows missing from the last one, one
# slot; the forward's two packs a lane at the edges of its range; whole packs from 8192 rows on
STEADY = {
    torch.float16: {(6003, 521): "-b-b", (6001, 1023): "-b-b", (6003, 1401): "fb-b", (5999, 1999): "fb-b",
                    (4100, 2501): "fb-b", (4099, 2999): "fbfb", (4097, 4095): "fbfb", (4099, 4097): "fbfb",
                    (4101, 4609): "fb-b", (8193, 5120 - 3): "fbfb", (4099, 6151): "fbfb", (8195, 2304): "-b-b",
                    (8193, 3080): "-b-b", (2050, 5448): "-b-b", (1031, 8191): "fb-b"},
    torch.float32: {(4103, 1025): "fb-b", (4099, 1535): "fb-b", (4101, 2049): "fb-b", (4097, 3071): "fb-b",
                    (4099, 4095): "fb-b", (4103, 4607): "fb-b", (1031, 6143): "-b-b", (1033, 6145): "-b-b"}}


@pytest.mark.parametrize("dtype,wdtype", [(torch.float16, torch.float16), (torch.bfloat16, torch.float32),
                                          (torch.float32, torch.float32)], ids=str)
def test_steady_rounds(cabi, gpu, dtype, wdtype):
    code, wcode = cabi.dtype_code(dtype), cabi.dtype_code(wdtype)
    ops = (cabi.OP_LAYER_NORM_FWD, cabi.OP_LAYER_NORM_BWD, cabi.OP_RMS_NORM_FWD, cabi.OP_RMS_NORM_BWD)
    for j, ((M, N), runs) in enumerate(STEADY[torch.float32 if dtype == torch.float32 else torch.float16].items()):
        offset = 1 + j % 3 if N % 2 else 2 * (j % 2)
        print("case steady rounds on whole wavefronts", dtype, wdtype, (M, N), "offset", offset, flush=True)
        plans = [cabi.waves_plan(op, M, N, code, wcode) for op in ops]
        for p, want in zip(plans, runs):
            # (an RMSNorm forward with float32 weights keeps its longest rows on them, too)
            if not (want == "-" and wdtype != dtype and p["waves"]):
                assert (p["waves"] > 0) == (want != "-"), (M, N, runs, plans)
            if p["waves"]:
                assert p["grid_blocks"] * p["rows_per_block"] < M, "a second round"
        g = torch.Generator(device=gpu).manual_seed(N + M)
        rand = lambda *s: torch.empty(*s, device=gpu).normal_(generator=g)  # noqa: E731
        _, x = _inside((rand(M, N) + 0.5).to(dtype), offset)
        _, dy = _inside(rand(M, N).to(dtype), (offset + 1) % 4)
        _, w = _inside((1 + 0.1 * rand(N)).to(wdtype), 1)
        _, b = _inside((0.1 * rand(N)).to(wdtype), 3)
        what = "[%d, %d] %s %s" % (M, N, dtype, wdtype)
        xd, dyd, wd = x.double(), dy.double(), w.double()
        cpu = lambda t: t.float().cpu().numpy()  # noqa: E731
        for rms in (False, True):
            mu = torch.zeros(M, 1, dtype=torch.float64, device=gpu) if rms else xd.mean(1, keepdim=True)
            rs = ((xd - mu).square().mean(1, keepdim=True) + EPS).rsqrt()
            xh = (xd - mu) * rs
            buf, y = _inside(torch.zeros_like(x), 3)
            if rms:
                y, rstd = cabi.rms_norm_fwd(x, w, EPS, y=y)
                dx, dg = cabi.rms_norm_bwd(dy, x, rstd, w)
                again = cabi.rms_norm_bwd(dy, x, rstd, w)
            else:
                y, mean, rstd = cabi.layer_norm_fwd(x, w, b, EPS, y=y)
                assert_close(mean, cpu(mu.view(-1)), torch.float32, "mean " + what)
                dx, dg, db = cabi.layer_norm_bwd(dy, x, mean, rstd, w)
                again = cabi.layer_norm_bwd(dy, x, mean, rstd, w)
                assert_close(db, cpu(dyd.sum(0)), wdtype, "dbeta " + what, slack=(dyd.abs().sum(0) * 2.0 ** -21).cpu())
                assert torch.equal(again[2], db), "run to run " + what
            assert torch.equal(again[0], dx) and torch.equal(again[1], dg), "run to run " + what
            assert_close(y, cpu(xh * wd + (0 if rms else b.double())), dtype, "y " + what)
            assert_close(rstd, cpu(rs.view(-1)), torch.float32, "rstd " + what)
            assert torch.isnan(buf[:3]).all() and torch.isnan(buf[3 + M * N:]).all(), "outside y " + what
            # (float32 sums over the rows, in another order, of terms with the statistics' own rounding: a few ulps
            # of the magnitudes' sum)
            terms = dyd * xh
            assert_close(dg, cpu(terms.sum(0)), wdtype, "dgamma " + what, slack=(terms.abs().sum(0) * 2.0 ** -21).cpu())
            gy = dyd * wd
            want = (gy - (0 if rms else gy.mean(1, keepdim=True)) - xh * (gy * xh).mean(1, keepdim=True)) * rs
            assert_close(dx, cpu(want), dtype, "dx " + what)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32], ids=str)
def test_infinities_and_nan_stay_in_their_rows(cabi, gpu, dtype):
    """A row with an inf or a NaN, in its head, in an element two lanes hold and in its last element, comes out
    NaN; the other rows do not change."""
    M, N = 300, 4097
    g = gen(77)
    x = torch.randn(M, N, generator=g).to(dtype).to(gpu)
    w = torch.ones(N, dtype=dtype, device=gpu)
    clean, m0, r0 = cabi.layer_norm_fwd(x, w, None, EPS)
    rows = [0, 3, 128, 299]
    for r, c, v in zip(rows, (0, 1, N - 3, N - 1), (float("inf"), float("nan"), float("inf"), float("nan"))):
        x[r, c] = v
    y, mean, rstd = cabi.layer_norm_fwd(x, w, None, EPS)
    other = torch.ones(M, dtype=torch.bool, device=gpu)
    other[rows] = False
    assert bool(torch.isnan(y[rows]).all()) and bool(torch.isnan(mean[rows]).all())
    assert torch.equal(y[other], clean[other]) and torch.equal(mean[other], m0[other])
    dx, _, _ = cabi.layer_norm_bwd(x, x, mean, rstd, w)
    assert bool(torch.isnan(dx[rows]).all()) and not bool(torch.isnan(dx[other]).any())
