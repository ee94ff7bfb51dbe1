"""The host-side rules behind the choice of a kernel, on the CPU: tests/native/plan_rules.cpp (the plan
header behind C functions) is compiled with g++ and called through ctypes."""
import ctypes
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("rules") / "libplan_rules.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wno-unknown-pragmas", "-shared", "-fPIC",
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
