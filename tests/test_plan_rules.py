"""The host-side rules behind the choice of a kernel, on the CPU: tests/native/plan_rules.cpp (the plan
header behind C functions) is compiled with g++ and called through ctypes."""
import ctypes
import os
import random
import subprocess
import threading

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rules") / "libplan_rules.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wno-unknown-pragmas", "-shared", "-fPIC", "-pthread",
                    os.path.join(HERE, "native", "plan_rules.cpp"), "-o", out], check=True)
    return ctypes.CDLL(out)


def test_how_a_ragged_row_of_the_norm_backward_is_read(cabi, rules):
    """Rows that leave much of 1024 lanes idle, and long rows of tensors far beyond the caches, keep the
    element loads that measured faster there; everything else reads whole packs."""
    f = rules.rule_norm_bwd_reads_elements
    i64 = ctypes.c_int64

    def reads_elements(dt, wdt, rms, M, N):
        es = 4 if dt == cabi.F32 else 2
        p = cabi.plan(cabi.OP_RMS_NORM_BWD if rms else cabi.OP_LAYER_NORM_BWD, M, N, dt, wdt)
        assert p["resident"] == 1
        return f(es, 4 if wdt == cabi.F32 else es, p["lanes_per_row"], p["packs_per_lane"], rms,
                 i64(M), i64(N))

    for dt in (cabi.F16, cabi.BF16):
        for M in (1, 4096, 32768):
            for N in (9, 100, 1401, 2049, 4097, 6143, 8191):
                assert not reads_elements(dt, dt, 0, M, N) and not reads_elements(dt, dt, 1, M, N)
            assert [reads_elements(dt, dt, 1, M, N) for N in (8193, 10001, 12289, 16383)] == [int(M > 12000)] * 2 + [0, 0]
            assert [reads_elements(dt, dt, 0, M, N) for N in (8193, 10001, 12289, 13001, 16383)] == [1, 1, 1, 0, 0]
            assert [reads_elements(dt, cabi.F32, 0, M, N) for N in (8193, 10001, 16383)] == [1, 0, 0]
    for rms in (0, 1):
        for M in (1, 4096):
            for N in (5, 1401, 3001, 4097, 6143, 7777, 8193, 16383):
                assert not reads_elements(cabi.F32, cabi.F32, rms, M, N)
        assert [reads_elements(cabi.F32, cabi.F32, rms, 32768, N) for N in (1401, 2049, 3001, 4097, 5001, 7777)] == [0, 0, 1, 0, 1, 1]


def _gn_team(rules, N, C, side, esize, groups=32):
    out = (ctypes.c_int64 * 5)()
    hw, E = side * side, 16 // esize
    assert hw % E == 0
    rules.rule_gn_bwd_team(ctypes.c_int64(N * groups), ctypes.c_int64(C // groups), ctypes.c_int64(hw // E),
                           esize, out)
    return dict(zip(("team", "wpc", "v", "ahead", "grid"), out))


def test_group_norm_backward_teams(rules):
    """Every plan holds its channels and fits the machine, and the next slab is on its way only where
    that neither idles workgroups nor runs clearly more rounds of packs."""
    for esize in (2, 4):
        for C in (32, 128, 256, 512, 1024):
            for side in range(16, 520, 8):
                cp = side * side * esize // 16
                for N in (1, 2, 3, 5, 8, 64):
                    t = _gn_team(rules, N, C, side, esize)
                    if t["team"] == 0:  # (short channels, or one slab beyond the machine)
                        continue
                    D, slots = C // 32, t["wpc"] * t["v"] * 512
                    assert t["v"] in (4, 8) and t["team"] == D * t["wpc"] >= 2
                    assert slots >= cp and 2 * cp >= slots, "a channel is held, its workgroups half full at least"
                    assert t["grid"] % t["team"] == 0 and t["team"] <= t["grid"] <= 512
                    if t["ahead"]:
                        assert t["v"] == 4 and N * 32 > t["grid"] // t["team"]
                        # against eight packs a lane: no fewer workgroups at work, pack-rounds within an eighth
                        wpc8 = -(-cp // 4096)
                        if cp > 2048 and D * wpc8 <= 512:
                            teams8 = min(512 // (D * wpc8), N * 32)
                            rounds8 = -(-N * 32 // teams8)
                            rounds = -(-N * 32 // (t["grid"] // t["team"]))
                            assert t["grid"] >= 480 and 4 * rounds <= 9 * rounds8, (N, C, side, t)
    # where the look-ahead kernel measured slower ...
    for N, C, sides, esize in ((1, 512, range(320, 345, 8), 2), (1, 512, range(368, 393, 8), 2),
                               (1, 512, range(408, 473, 8), 2), (1, 256, range(448, 481, 8), 2),
                               (3, 512, (232,), 2), (4, 512, (152,), 2), (7, 128, (248,), 2), (1, 512, (296, 312), 4), (7, 384, (104,), 4)):
        for side in sides:
            assert not _gn_team(rules, N, C, side, esize)["ahead"], (N, C, side)
    # ... and where faster
    for N, C, side, esize in ((1, 512, 480, 2), (1, 512, 496, 2), (1, 512, 512, 2), (16, 512, 128, 2), (4, 256, 128, 2),
                              (2, 512, 200, 2), (5, 256, 184, 2), (8, 128, 512, 2), (4, 256, 256, 4), (1, 512, 256, 4),
                              (4, 128, 200, 4), (8, 128, 136, 4), (1, 512, 248, 4), (1, 384, 232, 4)):
        assert _gn_team(rules, N, C, side, esize)["ahead"], (N, C, side)


def test_group_norm_backward_teams_that_sum_their_channels(rules):
    """Whole groups a team make no more rounds than slabs dealt out one by one, and of no more teams: a last round
    of at most half the teams keeps the second stage."""
    i64 = ctypes.c_int64
    f = lambda N, groups, teams: bool(rules.rule_gn_team_sums(i64(N * groups), i64(groups), i64(teams)))  # noqa: E731
    for groups in (1, 4, 8, 12, 32, 64):
        for N in range(1, 9):
            for teams in range(1, 513):
                rounds = -(-N * groups // teams)
                last = N * groups - (rounds - 1) * teams
                if f(N, groups, teams):
                    assert teams <= groups and -(-groups // teams) * N <= rounds
                    assert N == 1 or 2 * last > teams
    assert f(1, 32, 25) and f(2, 32, 32) and f(3, 32, 32)
    assert not f(2, 64, 25) and not f(2, 8, 5) and not f(2, 64, 42) and not f(4, 32, 64)


def test_every_stream_has_its_own_exchange_memory(rules):
    """Slots are handed out by stream, whatever the order and the number of calls: one stream always gets
    the same, two never share one, a stream beyond the last slot gets none; also from several threads."""
    rules.rule_slots_new.restype = ctypes.c_void_p
    n = rules.rule_team_slots()
    table = ctypes.c_void_p(rules.rule_slots_new())
    of = lambda key: rules.rule_slot_of(table, ctypes.c_size_t(key))  # noqa: E731
    try:
        keys = [1] + [0x7f0000001000 + 64 * i for i in range(n - 1)]
        got, start = [{} for _ in range(8)], threading.Barrier(8)

        def calls(mine, seed):
            order = keys * 20
            random.Random(seed).shuffle(order)
            start.wait()
            for k in order:
                s = of(k)
                assert mine.setdefault(k, s) == s, "a stream's slot changed"

        threads = [threading.Thread(target=calls, args=(got[i], i)) for i in range(8)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert all(g == got[0] for g in got) and sorted(got[0].values()) == list(range(n))
        assert of(0x7f1000000000) == -1 and of(0x7f1000000040) == -1
        assert all(of(k) == got[0][k] for k in keys)
    finally:
        rules.rule_slots_delete(table)


def _strided(rules, backward, outer, D, inner, esize):
    out = (ctypes.c_int64 * 10)()
    i64 = ctypes.c_int64
    rules.rule_strided_plan(backward, i64(outer), i64(D), i64(inner), esize, out)
    return dict(zip(("team", "v", "tx", "grid", "resident", "tile_tx", "tile_ty", "tile_v", "tile_grid",
                     "chunks"), out))


def test_strided_softmax_teams(rules):
    """Every row of a strip is held, on instances that exist, by teams of at most an eighth of the
    machine: launches on several streams always hold whole teams, which finish."""
    built = {0: (1, 2, 3, 4, 6, 8, 10, 12, 14, 16), 1: (1, 2, 3, 4, 5, 6, 7, 8)}
    rng = random.Random(31)
    shapes = [(o, D, px) for o in (1, 8, 200, 2000) for D in (257, 700, 2048, 8192, 60000, 262144, 1 << 20)
              for px in (1, 2, 3, 8, 17, 33, 40, 238, 1024)]
    shapes += [(rng.randint(1, 300), int(2 ** rng.uniform(8, 20)), int(2 ** rng.uniform(0, 14))) for _ in range(3000)]
    teams = 0
    for outer, D, px in shapes:
        for esize in (2, 4):
            for backward in (0, 1):
                p = _strided(rules, backward, outer, D, px * 16 // esize, esize)
                if p["team"] == 0:
                    continue
                teams += 1
                ty = 512 // p["tx"]
                assert p["tx"] in (1, 2, 4, 8, 16, 32) and p["v"] in built[backward]
                assert p["team"] * ty * p["v"] >= D > (p["team"] - 1) * ty * p["v"], "held, no workgroup without a row"
                assert p["team"] <= 64, (outer, D, px, esize, backward, p)
                assert p["grid"] % p["team"] == 0 and p["team"] <= p["grid"] <= 512
                assert p["grid"] // p["team"] <= outer * -(-px // p["tx"])
                assert ty * p["v"] * px * 16 < 2 ** 31
    assert teams > 3000


def test_strided_softmax_tile_or_teams(rules):
    """Teams where they measured faster than the one-workgroup tile, and strips of the width that measured
    faster: [outer, D, packs of inner], in 16 bits unless stated."""
    for outer, D, px in ((2000, 257, 1), (200, 512, 1), (2000, 300, 2), (200, 1025, 1), (2000, 512, 4),  # the tile spans the row
                         (8, 257, 8), (1, 257, 64), (200, 256, 238), (8, 450, 72), (8, 512, 100)):
        for esize in (2, 4):
            for backward in (0, 1):
                p = _strided(rules, backward, outer, D, px * 16 // esize, esize)
                assert p["team"] == 0 and p["resident"], (outer, D, px, esize, backward, p)
                assert p["tile_ty"] * p["tile_v"] >= D
    for outer, D, px, esize in ((200, 257, 40, 2), (40, 257, 72, 2), (40, 384, 72, 4), (1, 512, 1024, 4)):
        assert _strided(rules, 0, outer, D, px * 16 // esize, esize)["team"] == 0
    for outer, D, px in ((4, 512, 1024), (64, 300, 100), (200, 512, 17), (40, 512, 238), (1, 700, 4), (8, 2048, 2),
                         (1, 8192, 1024), (1, 30000, 8), (35, 1000, 238)):
        for esize in (2, 4):
            for backward in (0, 1):
                assert _strided(rules, backward, outer, D, px * 16 // esize, esize)["team"] >= 1, (outer, D, px)
    width = lambda *a: _strided(rules, *a)["tx"]  # noqa: E731
    assert width(0, 35, 1000, 1904, 2) == width(1, 35, 1000, 1904, 2) == 32
    assert width(0, 200, 700, 320, 2) == 16 and width(0, 200, 257, 800, 2) == 16  # a last strip mostly past the row
    assert width(1, 200, 700, 264, 2) == 32
    assert width(0, 1, 8192, 8192, 2) == width(1, 1, 8192, 8192, 2) == 16
    assert width(0, 1, 8192, 136, 2) == 8 and width(1, 1, 30000, 136, 2) == 8
    assert _strided(rules, 0, 8, 8192, 16, 4)["team"] == 16


def _team_order(rules, stream, captured=None, per_thread=None):
    n, streams = len(stream), max(stream) + 1
    ints = lambda v: (ctypes.c_int * n)(*(v or [0] * n))  # noqa: E731
    ran, counts = ints(None), (ctypes.c_int * 3)()
    rules.rule_team_order(n, ints(stream), ints(captured), ints(per_thread), streams, ran, counts)
    return list(ran), list(counts)


def test_one_team_launch_at_a_time(rules):
    """Launches whose workgroups wait for one another never run beside one another, whatever the streams' turns; a
    program on one stream records no event; nothing is recorded on a stream under capture."""
    ran, counts = _team_order(rules, [0] * 1000)
    assert ran == [1] * 1000 and counts == [0, 0, 0]
    ran, counts = _team_order(rules, [0, 0, 1, 0])  # the first turn: the event goes behind the earlier stream's work
    assert ran == [1] * 4 and counts == [3, 2, 0]
    rng = random.Random(7)
    for streams, stay in ((2, 1), (3, 1), (5, 4), (3, 40), (2, 300)):
        order = [s for _ in range(12 if stay > 40 else 40) for s in [rng.randrange(streams)] * rng.randint(1, stay)]
        ran, counts = _team_order(rules, order)
        assert ran == [1] * len(order) and counts[2] == 0
        ran, counts = _team_order(rules, order, per_thread=[1] * len(order))
        assert ran == [1] * len(order)
        under = [rng.randrange(1 << streams) & ~(1 << s) for s in order]  # (a stream's own capture is seen before)
        ran, counts = _team_order(rules, order, captured=under)
        assert 2 not in ran and counts[2] == 0
    # quiet again: a launch on the same stream records nothing, one elsewhere still finds its order
    ran, counts = _team_order(rules, [0, 1] + [1] * 600)
    assert ran == [1] * 602 and counts == [1 + 256, 1, 0]
    assert _team_order(rules, [0, 1] + [1] * 600 + [0]) == ([1] * 603, [1 + 256 + 2, 2, 0])
    # the earlier stream under capture before its event exists: without teams, until it is out
    assert _team_order(rules, [0, 1, 1, 1], captured=[0, 1, 0, 0])[0] == [1, 0, 1, 1]
    assert rules.rule_team_order_threads(8, 60) == 0


def test_a_slot_never_meets_an_id_twice(rules):
    """The tag of a word has room for 2^25 - 1 calls: a slot that a call before the ids came round has written to is
    cleared before the next one reads it, whatever calls other slots have had in between."""
    P = rules.rule_team_call_ids()
    rng = random.Random(11)
    slots, calls, n = 5, [], 0
    for _ in range(4000):
        n += rng.choice((1, 1, 1, 2, P // 3, P - 1, P, P + 1, 7 * P))
        calls.append((n, rng.randrange(slots)))
    calls = [(k, 0) for k in (0, P - 1, P, P + 1, 2 * P, 2 ** 32, 2 ** 32 + P)] + [(k + 2 ** 33, s) for k, s in calls]
    k = len(calls)
    ids, clear = (ctypes.c_uint * k)(), (ctypes.c_int * k)()
    rules.rule_team_ids(k, (ctypes.c_uint64 * k)(*[c[0] for c in calls]), (ctypes.c_int * k)(*[c[1] for c in calls]),
                        ids, clear)
    seen = [set() for _ in range(slots)]
    for i, (at, slot) in enumerate(calls):
        if clear[i]:
            seen[slot].clear()
        assert 1 <= ids[i] <= P and ids[i] << 6 < 2 ** 31 and ids[i] not in seen[slot]
        seen[slot].add(ids[i])
    assert list(clear[:7]) == [0, 0, 1, 0, 1, 1, 1] and (ids[0], ids[1], ids[2]) == (1, P, 1)


def _route(rules, backward, is_log, M, N, esize, widened=0):
    out = (ctypes.c_int64 * 2)()
    kind = rules.rule_softmax_route(backward, is_log, ctypes.c_int64(M), ctypes.c_int64(N), esize, widened, out)
    return ("two passes", "registers", "team", "held")[kind], out[0], out[1]


def test_softmax_rows_with_a_wider_output_have_teams(rules):
    """Few long float16 rows with a float32 output: teams for whole and ragged rows of any number, where one workgroup a
    row measured up to half as slow again."""
    f = lambda M, N, wide: _route(rules, 0, 0, M, N, 2, wide)[0]  # noqa: E731
    for M in (1, 30, 48, 64, 100, 128):
        for N in (32768, 36032, 40963, 45008, 60032, 60035, 140000):
            assert f(M, N, 1) == "team", (M, N)
    assert f(128, 32776, 0) == "registers" and f(129, 60032, 1) == "registers" and f(64, 32752, 1) == "registers"


def test_softmax_of_few_rows_by_teams_or_by_one_workgroup_each(rules):
    """Both sides of every line as they measured: (backward, log, rows, elements, bytes an element) -> team or not."""
    one = [(0, 0, 48, 32768, 2), (0, 0, 64, 36032, 2), (0, 0, 100, 40000, 2), (0, 0, 128, 50048, 2), (0, 1, 64, 40000, 2),
           (0, 0, 8, 17024, 4), (0, 0, 64, 20480, 4), (0, 0, 128, 20480, 4),
           (1, 0, 8, 32768, 2), (1, 0, 64, 36032, 2), (1, 1, 100, 36032, 2), (1, 0, 128, 50048, 2), (1, 1, 128, 55040, 2),
           (1, 0, 8, 16384, 4), (1, 0, 64, 20480, 4), (1, 1, 128, 25024, 4),
           # ragged: the slow side of the lines for whole rows was up to 1.4 times the two passes' time
           (0, 0, 64, 45051, 2), (0, 0, 100, 61435, 2), (0, 0, 128, 102403, 2), (0, 1, 48, 61435, 2), (0, 1, 128, 94203, 2),
           (0, 0, 128, 26619, 4), (0, 1, 30, 20475, 4),
           (1, 0, 30, 36859, 2), (1, 0, 64, 58155, 2), (1, 0, 100, 53243, 2), (1, 0, 128, 53243, 2), (1, 0, 128, 64707, 2),
           (1, 1, 48, 74539, 2), (1, 1, 64, 81091, 2), (1, 1, 128, 53243, 2), (1, 1, 128, 130243, 2),
           (1, 0, 64, 28027, 4), (1, 1, 64, 24571, 4), (1, 1, 128, 28027, 4)]
    team = [(0, 0, 8, 32768, 2), (0, 0, 48, 36032, 2), (0, 0, 64, 45056, 2), (0, 0, 100, 50048, 2), (0, 0, 100, 60032, 2),
            (0, 0, 128, 65536, 2), (0, 0, 8, 22528, 4), (0, 0, 64, 22528, 4),
            (1, 0, 8, 33792, 2), (1, 0, 30, 36032, 2), (1, 1, 48, 33792, 2), (1, 0, 64, 45056, 2), (1, 0, 128, 60032, 2),
            (1, 1, 30, 20480, 4), (1, 0, 64, 22528, 4),
            (0, 0, 8, 33579, 2), (0, 0, 64, 61435, 2), (0, 0, 100, 91000, 2), (0, 0, 128, 159739, 2), (0, 1, 64, 91003, 2),
            (0, 0, 48, 20067, 4), (0, 1, 64, 32643, 4),
            (1, 0, 8, 42000, 2), (1, 0, 30, 61435, 2), (1, 0, 128, 73475, 2), (1, 1, 8, 53243, 2), (1, 1, 64, 123691, 2),
            (1, 0, 100, 40835, 4), (1, 1, 64, 40835, 4), (1, 1, 128, 45055, 4)]
    for c in one:
        assert _route(rules, *c)[0] in ("registers", "held"), c
    for c in team:
        assert _route(rules, *c)[0] == "team", c
    for M in (1, 8, 48, 100, 128):  # without a held form there is nothing but teams or the two passes
        assert _route(rules, 1, 0, M, 80003, 2)[0] == "team" and _route(rules, 0, 0, M, 200003, 2)[0] == "team"


def test_which_ragged_softmax_rows_are_held(rules):
    """Both sides of the lines of softmax_tail_serves(), and no pack count for which no kernel is built."""
    held = [(0, 1, 3000, 53243, 2), (0, 1, 1000, 49963, 2), (0, 0, 2000, 53243, 2), (0, 1, 4096, 18431, 4), (0, 1, 2000, 26619, 4),
            (0, 0, 200, 159739, 2), (0, 0, 1000, 159739, 2), (0, 0, 1000, 61847, 4), (0, 1, 2000, 37271, 4), (0, 0, 200, 37271, 4),
            (1, 0, 2000, 32515, 2), (1, 0, 300, 29483, 2), (1, 0, 4096, 28003, 2), (1, 0, 2000, 16791, 4), (1, 1, 2000, 29483, 2),
            (1, 1, 4096, 18839, 4), (1, 1, 1000, 16791, 4)]
    passes = [(0, 1, 2000, 53243, 2), (0, 1, 1500, 61435, 2), (0, 1, 3000, 18431, 4), (0, 0, 300, 159739, 2),
              (0, 0, 1000, 133540, 2), (0, 0, 4096, 152001, 2), (0, 0, 300, 61847, 4), (0, 0, 2000, 37271, 4), (0, 1, 700, 37271, 4),
              (1, 0, 2000, 29483, 2), (1, 0, 2000, 31939, 2), (1, 1, 4096, 16791, 4), (0, 1, 700, 45463, 4),
              (1, 0, 2000, 34003, 2), (1, 0, 2000, 66003, 2), (0, 0, 2000, 163843, 2)]
    for c in held:
        assert _route(rules, *c)[0] == "held", c
    for c in passes:
        assert _route(rules, *c)[0] == "two passes", c
    wide = lambda M, N, log: _route(rules, 0, log, M, N, 2, 1)[0]  # noqa: E731
    assert [wide(*a) for a in ((130, 53243, 0), (200, 36859, 0), (200, 53243, 0), (130, 53243, 1), (300, 53243, 0),
                               (2000, 53243, 1))] == ["two passes"] * 2 + ["held"] * 4
    for es in (2, 4):
        E = 16 // es
        for packs in range(2049 if es == 2 else 4097, 20600, 13):
            for over in range(1, E, 3):
                N = packs * E - E + over
                for M in (129, 300, 513, 1100, 2050, 5000):
                    kind, g, v = _route(rules, 0, 0, M, N, es)
                    assert kind in ("held", "two passes")
                    if kind == "held":
                        window = (N + 2 * (E - 1)) // E
                        assert (v - 1) * g < window <= v * g
                        assert v in range(*((5, 15) if es == 2 else (9, 15))) if g == 512 else (
                            g == 1024 and v in range(3 if es == 2 else 5, 21 if es == 2 else 17) and v not in (17, 19))
                    kind, g, v = _route(rules, 1, 0, M, N, es)
                    assert kind == "two passes" or (g == 1024 and (3 if es == 2 else 5) <= v <= 8)


def test_backward_of_few_long_norm_rows(rules):
    """Both sides of the lines between the two launches without partial rows and the teams of whole-pack rows as they
    measured: (rows, elements, bytes an element, LayerNorm, float32 weights of 16-bit rows)."""

    def f(*c):
        out = (ctypes.c_int64 * 2)()
        rules.rule_norm_few_rows(*map(ctypes.c_int64, c[:2]), *c[2:], out)
        return list(out)

    few = [(40, 80000, 4, 1, 0), (24, 160000, 4, 1, 0), (16, 224000, 4, 1, 0), (64, 160000, 2, 1, 1), (48, 224000, 2, 1, 1),
           (64, 160000, 2, 1, 0), (40, 224000, 2, 1, 0), (128, 66400, 2, 1, 0), (24, 320000, 4, 1, 0), (16, 520000, 4, 1, 0),
           (80, 79997, 4, 1, 0), (100, 79997, 4, 1, 0), (24, 640000, 2, 1, 1), (64, 79997, 4, 0, 0), (16, 320000, 2, 0, 0)]
    team = [(128, 40000, 4, 1, 0), (100, 56000, 4, 1, 0), (80, 80000, 4, 1, 0), (48, 112000, 4, 1, 0), (32, 160000, 4, 1, 0),
            (48, 160000, 4, 1, 0), (24, 224000, 4, 1, 0), (80, 160000, 2, 1, 1), (64, 224000, 2, 1, 1), (40, 320000, 2, 1, 1),
            (32, 448000, 2, 1, 1), (48, 320000, 2, 1, 0), (32, 160000, 4, 0, 0), (100, 112000, 2, 0, 0)]
    for c in few:
        assert f(*c)[0] in (1, 2, 4, 8) and f(*c)[1] == 0, (c, f(*c))
    # (a LayerNorm call that cannot have its teams keeps the two launches, up to 32 MB)
    for c in team:
        assert f(*c)[1] >= 2 and (f(*c)[0] > 0) == bool(c[3] and c[0] * c[1] * c[2] <= 32 << 20), (c, f(*c))
    assert [f(2, N, 2, 1, 0)[0] for N in (66400, 163840, 300000, 600000)] == [8, 4, 2, 1] and f(129, 66401, 2, 1, 0)[0] == 0
    assert f(1, 66400, 2, 1, 0) == [0, 0] and f(2, 3000000, 2, 1, 0) == [0, 0]
