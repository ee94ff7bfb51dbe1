"""The rule that shares the rows of a long norm forward call out to its teams (make_plan() in plan.hpp), on the CPU."""
import ctypes
import random

from test_plan_rules import rules  # noqa: F401

i64 = ctypes.c_int64


def _team(rules, M, N, esize=2, wide=0):  # noqa: F811
    out = (i64 * 3)()
    rules.rule_norm_team(i64(M), i64(N), esize, wide, out)
    return tuple(out)


def test_every_layout_holds_the_row(rules):  # noqa: F811
    """At most two workgroups a compute unit, 16 packs a lane; the team holds the row and no team is without a row;
    the rounds are as many as those of the most teams that fit."""
    rng, evened = random.Random(3), 0
    for _ in range(20000):
        esize = rng.choice((2, 4))
        n = int(2 ** rng.uniform(14, 22)) // (16 // esize) * (16 // esize)
        M = int(2 ** rng.uniform(0, 11))
        team, v, teams = _team(rules, M, n, esize, rng.randint(0, 1) if esize == 2 else 0)
        if team == 0 or v == 0:
            continue
        packs = n * esize // 16
        assert 1 <= v <= 16 and 1 <= teams <= M and team * teams <= 512
        assert (team - 1) * v * 512 < packs <= team * v * 512
        most = min(M, 512 // -(-packs // 8192))
        assert -(-M // teams) == -(-M // most), (M, n, esize, team, v, teams)
        evened += teams < most
    assert evened > 50


def test_rounds_of_the_same_rows(rules):  # noqa: F811
    assert _team(rules, 140, 216576) == (7, 8, 70) and _team(rules, 33, 1103488) == (30, 9, 17)
    assert _team(rules, 358, 163840) == (4, 10, 120)
    # one round, four and more, a row that would not spread further, workgroups left over, an odd team beside
    # weights that fill the L2
    assert _team(rules, 64, 115200)[2] == 64 and _team(rules, 512, 401408) == (7, 14, 73)
    assert _team(rules, 389, 188800)[2] == 170 and _team(rules, 148, 291328)[2] == 102
    assert _team(rules, 71, 1284480)[2] == 25
    # packs that do not go down as far as the last round was short, weights an XCD's L2 does not hold
    assert _team(rules, 112, 686560)[2] == 46 and _team(rules, 241, 133440, wide=1)[2] == 170
    assert _team(rules, 20, 2036640, wide=1)[2] == 16 and _team(rules, 35, 2034192, wide=1)[2] == 16
