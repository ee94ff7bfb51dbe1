"""The rule that gives the strips of a strided softmax to workgroups with a compute unit each
(strided_large_team() in plan.hpp), on the CPU."""
import ctypes
import random

from test_plan_rules import _strided, rules  # noqa: F401

i64 = ctypes.c_int64


def _large(rules, backward, outer, D, inner, esize, widened=0):  # noqa: F811
    out = (i64 * 4)()
    rules.rule_strided_large(backward, i64(outer), i64(D), i64(inner), esize, out, widened)
    return dict(zip(("team", "v", "tx", "grid"), list(out)))


def test_large_teams(rules):  # noqa: F811
    """Every row of a strip is held on instances that exist, on a grid that is resident at one workgroup a
    compute unit, by teams of an eighth of the machine at most, in fewer rounds than two a compute unit."""
    rng = random.Random(7)
    built = {0: (40, 48, 56, 64), 1: (20, 24, 28, 32)}
    shapes = [(1, 8192, 1024), (12, 9602, 25), (6, 323, 1285), (1, 65536, 16384), (92, 2206, 32)]
    shapes += [(rng.randint(1, 300), int(2 ** rng.uniform(8, 17)), int(2 ** rng.uniform(1, 13))) for _ in range(4000)]
    taken = 0
    for outer, D, px in shapes:
        for esize in (2, 4):
            for backward in (0, 1):
                a = (backward, outer, D, px * 16 // esize, esize)
                p, l = _strided(rules, *a), _large(rules, *a)
                if l["team"] == 0:
                    continue
                taken += 1
                ty, strips = 512 // l["tx"], lambda t: outer * -(-px // t["tx"])
                assert p["team"] > 0 and l["tx"] in (16, 32) and l["v"] in built[backward]
                assert l["team"] * ty * l["v"] >= D > (l["team"] - 1) * ty * l["v"], "held, no workgroup without a row"
                assert l["team"] <= 32 and l["grid"] % l["team"] == 0 and l["team"] <= l["grid"] <= 256
                rounds = lambda t: -(-strips(t) // (t["grid"] // t["team"]))  # noqa: E731
                assert rounds(l) < rounds(p) and ty * l["v"] * px * 16 * (2 if esize == 2 else 1) < 2 ** 31
    assert taken > 300
    assert _large(rules, 0, 1, 8192, 8192, 2) == dict(team=8, v=64, tx=32, grid=256)
    assert _large(rules, 1, 1, 8192, 8192, 2) == dict(team=16, v=32, tx=32, grid=256)
    # where two a compute unit measured faster
    for a in ((0, 50, 954, 920, 2), (0, 6, 820, 10296, 2), (0, 4, 3419, 3912, 2), (1, 36, 2844, 384, 2), (0, 8, 2048, 2048, 2)):
        assert _large(rules, *a)["team"] == 0, a
    # strips no wider than the small teams', in a float32 forward also rows of 16 packs at most
    for a in ((0, 48, 3983, 592, 2), (0, 18, 4088, 2736, 2), (0, 47, 3854, 472, 4), (1, 14, 3068, 1336, 2), (1, 45, 3068, 488, 4),
              (0, 34, 12457, 60, 4), (0, 62, 14919, 56, 4)):
        assert _large(rules, *a)["team"] == 0, a
    # in 16 bits rows of 16 packs at most for a single round only
    for a, one in (((0, 55, 14117, 120, 2), 32), ((0, 56, 15618, 104, 2), 28), ((0, 49, 14836, 80, 2), 24)):
        assert _large(rules, *a)["team"] == 0 and _large(rules, 0, one, *a[2:])["team"] > 0, a
    # forward rows of whole lines, several rounds, in float32 any
    for a in ((0, 62, 6587, 256, 2), (0, 4, 9431, 2304, 2), (0, 40, 10726, 128, 4), (0, 16, 11602, 128, 4), (0, 2, 5884, 1824, 4)):
        assert _large(rules, *a)["team"] == 0, a
    # float32 forward rows on small teams whose neighbouring strips meet on one XCD
    for a in ((0, 14, 6942, 376, 4), (0, 4, 8964, 632, 4), (0, 4, 12060, 492, 4)):
        assert _strided(rules, *a)["team"] % 8 == 0 and _large(rules, *a)["team"] == 0, a
    # float32 backward strips no wider, of an odd number of packs, rounds not halved
    for a in ((1, 9, 4084, 524, 4), (1, 53, 3929, 236, 4)):
        assert _large(rules, *a)["team"] == 0 and _large(rules, *a[:3], a[3] + 4, 4)["team"] > 0, a


def test_not_for_an_output_wider_than_the_input(rules):  # noqa: F811
    """A float16 forward with a float32 output is slower on them at every size."""
    rng, plain = random.Random(8), 0
    for _ in range(3000):
        a = (0, rng.randint(1, 64), int(2 ** rng.uniform(8, 15)), 8 * int(2 ** rng.uniform(1, 12)), 2)
        plain += _large(rules, *a)["team"] > 0
        assert _large(rules, *a, widened=1)["team"] == 0, a
    assert plain > 300
