"""Team launches on several streams at once: every stream has exchange memory of its own, and one such
launch at a time runs on the device, so nobody's wait runs out and the results are those that the calls
have alone; a stream beyond the slots takes the launches that exchange nothing.  (The reference's kernels
share nothing between calls: SpatialSoftmaxForward, src/ATen/native/xpu/sycl/SoftMaxKernels.cpp:725-950,
LayerNormKernels.cpp:360-470.)"""
import time

import pytest
import torch

from helpers import assert_close, gen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def streams(gpu):
    """Three streams for all tests of this file that need exchange memory: a stream keeps its slot of the strided
    softmax (eight a device) for the process, and calls on one that found none give other bits."""
    return [torch.cuda.Stream() for _ in range(3)]


def _calls(cabi, gpu, seed):
    """Thunks of one stream: strips on 64 workgroups, on a few, forward and backward, and rows of the
    norm and softmax kernels held by teams."""
    g = gen(seed)
    x = torch.randn(1, 32000, 64, generator=g).bfloat16().to(gpu)
    w = torch.randn(4, 1025, 1024, generator=g).bfloat16().to(gpu)
    y = torch.softmax(w.float(), 1).bfloat16()
    r = torch.randn(16, 140000, generator=g).bfloat16().to(gpu)
    gamma = torch.ones(140000, dtype=torch.bfloat16, device=gpu)
    return [lambda: cabi.softmax_strided_fwd(x, 1), lambda: cabi.softmax_strided_fwd(w, 1, cabi.LOG_SOFTMAX),
            lambda: cabi.softmax_strided_bwd(w, y, 1),
            lambda: cabi.layer_norm_fwd(r, gamma, None, 1e-5)[0], lambda: cabi.softmax_fwd(r)]


def test_calls_on_three_streams_do_not_wait_for_one_another(cabi, gpu, streams):
    calls = [_calls(cabi, gpu, 2600 + i) for i in range(3)]
    alone = [[f() for f in fs] for fs in calls]
    got = [[None] * len(fs) for fs in calls]
    for i, s in enumerate(streams):  # (the streams' slots, the allocator's blocks)
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            got[i] = [f() for f in calls[i]]
    torch.cuda.synchronize()
    print("case three streams, 40 rounds of five calls each", flush=True)
    t0 = time.perf_counter()
    for k in range(40):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                for j, f in enumerate(calls[i]):
                    # (every stream meets the others' calls at another place)
                    j = (j + k * (i + 1)) % len(calls[i])
                    got[i][j] = calls[i][j]()
    torch.cuda.synchronize()
    # (one wait that runs out is a second)
    assert time.perf_counter() - t0 < 0.9
    for i in range(3):
        for j in range(len(calls[i])):
            assert torch.equal(got[i][j].view(torch.uint8), alone[i][j].view(torch.uint8)), (i, j)


def _large_calls(cabi, gpu, seed):
    """Thunks of one stream: strips of workgroups that need a whole compute unit each, forward and backward, among
    teams of smaller workgroups and kernels without teams that fill the machine."""
    g = torch.Generator(device=gpu).manual_seed(seed)
    x = torch.empty(1, 8192, 8192, dtype=torch.bfloat16, device=gpu).normal_(0, 3, generator=g)
    y = torch.softmax(x.float(), 1).bfloat16()
    w = torch.empty(1, 12899, 3872, dtype=torch.bfloat16, device=gpu).normal_(generator=g)
    for backward, shape in ((0, (1, 8192, 8192)), (1, (1, 8192, 8192)), (0, (1, 12899, 3872))):
        p = cabi.strided_team_plan(backward, *shape, cabi.BF16)
        assert p["team"] > 1 and p["packs_per_lane"] > (8 if backward else 16), p
    small = torch.empty(4, 1025, 1024, dtype=torch.bfloat16, device=gpu).normal_(generator=g)
    rows = torch.empty(16, 140000, dtype=torch.bfloat16, device=gpu).normal_(generator=g)
    many = torch.empty(16384, 4096, dtype=torch.bfloat16, device=gpu).normal_(generator=g)
    gamma = torch.ones(140000, dtype=torch.bfloat16, device=gpu)
    return [lambda: cabi.softmax_strided_fwd(x, 1), lambda: cabi.softmax_strided_bwd(x, y, 1),
            lambda: cabi.softmax_strided_fwd(small, 1), lambda: cabi.softmax_strided_fwd(w, 1, cabi.LOG_SOFTMAX),
            lambda: cabi.layer_norm_fwd(rows, gamma, None, 1e-5)[0], lambda: cabi.softmax_fwd(many),
            lambda: cabi.layer_norm_fwd(many, gamma[:4096], None, 1e-5)[0]]


def test_workgroups_that_need_a_whole_compute_unit_on_three_streams(cabi, gpu, streams):
    """A large team takes turns with other streams' teams and shares the machine with kernels whose workgroups take any
    compute unit that has room: nobody's wait runs out."""
    calls = [_large_calls(cabi, gpu, 2700 + i) for i in range(3)]
    alone = [[f() for f in fs] for fs in calls]
    for i, s in enumerate(streams):  # (the streams' slots, the allocator's blocks)
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            for f in calls[i]:
                f()
    torch.cuda.synchronize()
    for k in range(24):
        print("case large teams on three streams, round", k, flush=True)
        t0 = time.perf_counter()
        got = [[None] * len(fs) for fs in calls]
        for step in range(len(calls[0])):
            for i, s in enumerate(streams):
                with torch.cuda.stream(s):
                    # (every stream meets the others' calls at another place)
                    j = (step + k * (i + 1)) % len(calls[i])
                    got[i][j] = calls[i][j]()
        torch.cuda.synchronize()
        # (one wait that runs out is a second; a round is a few milliseconds)
        assert time.perf_counter() - t0 < 0.5, k
        for i in range(3):
            for j in range(len(calls[i])):
                assert torch.equal(got[i][j].view(torch.uint8), alone[i][j].view(torch.uint8)), (k, i, j)


def test_more_streams_than_slots(cabi, gpu):
    """Twelve streams, eight of them with a slot of the strided softmax: the others' results come from
    the launches that exchange nothing."""
    g = gen(2650)
    x = (3 * torch.randn(2, 1500, 256, generator=g)).to(gpu)
    grad = torch.randn(2, 1500, 256, generator=g).to(gpu)
    want = torch.softmax(x.double(), 1)
    wgrad = want * (grad.double() - (want * grad.double()).sum(1, keepdim=True))
    torch.cuda.synchronize()
    outs = []
    for s in [torch.cuda.Stream() for _ in range(12)]:
        with torch.cuda.stream(s):
            y = cabi.softmax_strided_fwd(x, 1)
            outs.append((y, cabi.softmax_strided_bwd(grad, y, 1)))
    torch.cuda.synchronize()
    for k, (y, gi) in enumerate(outs):
        assert_close(y, want.float().cpu().numpy(), torch.float32, "y of stream %d" % k)
        assert_close(gi, wgrad.float().cpu().numpy(), torch.float32, "gi of stream %d" % k)
