"""The rule that lays norm rows out on whole wavefronts (norm_waves_layout() in plan.hpp), on the CPU."""
import ctypes
import random

from test_plan_rules import rules  # noqa: F401

i64 = ctypes.c_int64
INSTANCES = {(0, 2): {(1, 3, 1024), (2, 3, 1024)}, (0, 4): {(3, 2, 512)},
             (1, 2): {(1, 3, 1024), (2, 2, 768)}, (1, 4): {(3, 3, 512), (3, 2, 768)}}
FOLD_FLOATS = 8192


def _layout(rules, backward, M, N, esize, ln=1, wide=0, want_dx=1):  # noqa: F811
    out = (i64 * 7)()
    rules.rule_norm_waves(backward, i64(M), i64(N), esize, ln, wide, want_dx, out)
    return dict(zip(("waves", "v", "depth", "threads", "slots", "grid", "partial"), list(out)))


def test_rows_on_whole_wavefronts(rules):  # noqa: F811
    """Every row is held, only a lane's last pack may reach past it, the workgroup fits its instance, the column
    sums fit the memory they are folded through and the caller's partial rows, every workgroup has a row."""
    rng = random.Random(11)
    taken = {k: 0 for k in INSTANCES}
    for _ in range(60000):
        M = int(2 ** rng.uniform(6, 18))
        N = int(2 ** rng.uniform(6, 14.2))
        N = N // 8 * 8 if rng.random() < 0.3 else N
        esize, backward = rng.choice((2, 4)), rng.randint(0, 1)
        a = (backward, M, N, esize, rng.randint(0, 1), rng.randint(0, 1) if esize == 2 else 0)
        l = _layout(rules, *a)
        assert l["waves"] == 0 or M >= 256
        if l["waves"] == 0:
            continue
        taken[(backward, esize)] += 1
        E = 16 // esize
        packs = -(-N // E)
        assert (l["v"], l["depth"], l["threads"]) in INSTANCES[(backward, esize)]
        lanes = 64 * l["waves"]
        assert lanes * l["v"] >= packs and (l["v"] - 1) * lanes * E <= N and N >= E, (a, l)
        assert 1 <= l["slots"] and l["slots"] * lanes <= l["threads"] <= 1024
        assert 1 <= l["grid"] and (l["grid"] - 1) * l["slots"] < M, "a workgroup without a row"
        if backward:
            assert l["grid"] <= l["partial"]
            assert l["slots"] == 1 or 2 * lanes * l["v"] * E <= FOLD_FLOATS
            # the column sums alone run on the same layout
            assert _layout(rules, *a, want_dx=0) == dict(l, partial=_layout(rules, *a, want_dx=0)["partial"])
    assert all(n > 100 for n in taken.values()), taken


def test_rows_that_keep_their_layout(rules):  # noqa: F811
    """Widths an exact layout or a power of two of lanes serves as well, and rows too short or too long."""
    for N in (1024, 2048, 4096, 5120, 8192, 16384):
        for ln in (0, 1):
            for b in (0, 1):
                assert _layout(rules, b, 16384, N, 2, ln)["waves"] == 0 and _layout(rules, b, 16384, N, 4, ln)["waves"] == 0
    assert _layout(rules, 1, 8192, 16383, 2)["waves"] == 0 and _layout(rules, 0, 8192, 8195, 2)["waves"] == 0
    assert _layout(rules, 0, 8192, 4097, 4, 0)["waves"] == 0 and _layout(rules, 0, 1024, 4097, 4)["waves"] == 0
    assert _layout(rules, 1, 8192, 509, 2)["waves"] == 0 and _layout(rules, 0, 8192, 1021, 4)["waves"] == 0
    assert _layout(rules, 1, 8192, 4097, 2) == dict(waves=9, v=1, depth=3, threads=1024, slots=1, grid=256, partial=512)
    assert _layout(rules, 0, 8192, 4097, 2)["waves"] == 5


def test_short_rows_need_many_of_them(rules):  # noqa: F811
    """A ragged 16-bit backward whose row slots see a row or two each measured slower on whole wavefronts."""
    taken = lambda M, N, ln: _layout(rules, 1, M, N, 2, ln)["waves"] > 0  # noqa: E731
    for ln in (0, 1):
        assert not taken(881, 739, ln) and not taken(1830, 869, ln) and not taken(2395, 547, ln) and taken(3100, 850, ln)
        assert not taken(910, 1807, ln) and taken(1100, 1807, ln)
    assert not taken(1997, 1317, 0) and taken(2100, 1317, 0) and taken(600, 1317, 1)
    assert not taken(538, 2249, 0) and taken(800, 2249, 0) and taken(600, 2201, 1)
    assert not taken(412, 3791, 0) and taken(600, 3791, 0) and taken(300, 4097, 0)


def test_whole_packs_of_large_tensors(rules):  # noqa: F811
    """Backward rows of 513 to 768 whole packs beyond 50 million elements, and LayerNorm rows just below 512 beyond
    200 million, keep their layout, except LayerNorm rows that leave half of its lanes idle."""
    taken = lambda M, N, ln: _layout(rules, 1, M, N, 2, ln)["waves"] > 0  # noqa: E731
    for ln in (0, 1):
        for N in (4616, 4968, 5288, 5448, 6136):
            assert taken(8000, N, ln) and not taken(11000, N, ln) and not taken(100000, N, ln)
        for N in (6152, 7000, 8184):
            assert taken(300, N, ln) and taken(60000, N, ln)
        assert taken(60000, 3200, ln) and not taken(8191, 3200, ln)
    assert taken(100000, 4184, 1) and not taken(100000, 4184, 0)
    assert taken(40000, 4072, 1) and not taken(104347, 4072, 1) and taken(104347, 4072, 0)


def test_float_rows(rules):  # noqa: F811
    """Ragged float32 rows keep their layout in tensors far beyond the caches, and in the backward where a compute
    unit would get one long row or two."""
    fwd = lambda M, N: _layout(rules, 0, M, N, 4)["waves"] > 0  # noqa: E731
    for N in (1027, 2051, 2999, 4095):
        assert fwd(12000, N) and not fwd(70000, N) and not fwd(4000, N)
    assert fwd(9000, 1999) and not fwd(13000, 1999) and fwd(60000, 4097) and fwd(60000, 4607)
    bwd = lambda M, N, ln: _layout(rules, 1, M, N, 4, ln)["waves"] > 0  # noqa: E731
    for ln in (0, 1):
        assert bwd(65000, 3071, ln) and bwd(24000, 4097, ln) and not bwd(25000, 4097, ln) and not bwd(55957, 3777, ln)
        assert bwd(300, 6143, ln) and not bwd(300, 6145, ln) and bwd(400, 6145, ln)
        assert not bwd(485, 8743, ln) and bwd(700, 8743, ln) and not bwd(27414, 8269, ln)


def test_forward_rows(rules):  # noqa: F811
    """RMSNorm rows of 577 to 768 packs in calls of a middling number of rows, its longest rows, and LayerNorm rows
    whose slots leave wavefronts idle in large tensors, keep their layout."""
    taken = lambda M, N, ln, wide=0: _layout(rules, 0, M, N, 2, ln, wide)["waves"] > 0  # noqa: E731
    for wide in (0, 1):
        for N in (4617, 5001, 6143):
            assert taken(1000, N, 0, wide) and not taken(1100, N, 0, wide) and not taken(8000, N, 0, wide)
            assert taken(8192, N, 0, wide) and taken(4000, N, 1, wide)
        assert taken(4000, 4603, 0, wide) and taken(4000, 6151, 0, wide)
        assert taken(1000, 8001, 0, wide) and taken(30000, 8001, 0, wide) == (wide == 1) and taken(30000, 8001, 1, wide)
        assert taken(68064, 2577, 1, wide) == (wide == 1) and taken(94118, 1293, 1, wide) == (wide == 1)
        assert taken(30000, 1401, 1, wide) and taken(16821, 2669, 1, wide) and taken(100000, 2051, 1, wide)


def test_the_plan_query_reports_them(cabi, rules):  # noqa: F811
    """mi355x_rownorm_waves_plan says what runs: lanes, packs, rows a workgroup works on, workgroups, and the partial
    rows of a backward, which fit the workspace that the call asks for; nothing for forced fields, mi355x_rownorm_plan's
    layout where it reports none."""
    rng, taken = random.Random(13), 0
    for _ in range(4000):
        M, N = int(2 ** rng.uniform(7, 17)), int(2 ** rng.uniform(9, 14))
        dt, wd = rng.choice(((cabi.F32, cabi.F32), (cabi.F16, cabi.F16), (cabi.BF16, cabi.F32)))
        esize = 4 if dt == cabi.F32 else 2
        ln, backward = rng.randint(0, 1), rng.randint(0, 1)
        l = _layout(rules, backward, M, N, esize, ln, int(wd == cabi.F32 and esize == 2))
        op = ((cabi.OP_RMS_NORM_FWD, cabi.OP_LAYER_NORM_FWD), (cabi.OP_RMS_NORM_BWD, cabi.OP_LAYER_NORM_BWD))[backward][ln]
        p = cabi.waves_plan(op, M, N, dt, wd)
        assert p.pop("waves") == l["waves"]
        if l["waves"] == 0:
            q = cabi.plan(op, M, N, dt, wd)
            q.pop("row_chunks")
            assert p == q
            continue
        taken += 1
        assert p["resident"] == 1 and p["lanes_per_row"] == 64 * l["waves"]
        assert (p["packs_per_lane"], p["rows_per_block"], p["grid_blocks"]) == (l["v"], l["slots"], l["grid"])
        assert p["block_threads"] == 64 * l["waves"] * l["slots"]
        assert p["partial_rows"] == (l["grid"] if backward else 0)
        if backward:
            f = cabi.lib().mi355x_layer_norm_bwd_workspace_bytes if ln else cabi.lib().mi355x_rms_norm_bwd_workspace_bytes
            assert f(M, N, dt, wd, *((1, 1) if ln else (1,))) >= p["partial_rows"] * N * 4 * (1 + ln)
    assert taken > 300
    assert cabi.waves_plan(cabi.OP_SOFTMAX_FWD, 8192, 4097, cabi.F16, cabi.F16)["waves"] == 0
    try:
        cabi.set_override(cabi.OP_LAYER_NORM_BWD, 0, 0, 0, 3)
        assert cabi.waves_plan(cabi.OP_LAYER_NORM_BWD, 8192, 4097, cabi.F16, cabi.F16)["waves"] == 0
    finally:
        cabi.clear_overrides()
    assert cabi.waves_plan(cabi.OP_LAYER_NORM_BWD, 8192, 4097, cabi.F16, cabi.F16)["waves"] == 9
