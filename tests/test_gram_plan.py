"""How a chain's Gram launches are cut (gram_plan.hpp, compiled here for the host): no launch of a call uses more rows
of the Gram workspace or of the shared counts than the plan reserves for it."""
import ctypes as C
import itertools
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "bayesrrcmd_amd" / "csrc"
SHIM = """
#include "gram_plan.hpp"
extern "C" void cohort_plan(uint32_t n, const uint32_t* M, const uint32_t* B, uint32_t total, uint64_t most, uint64_t* out)
{
    const brr::CohortPlan p = brr::cohort_plan(std::vector<uint32_t>(M, M + n), std::vector<uint32_t>(B, B + n), total, most);
    out[0] = p.step; out[1] = p.parts; out[2] = p.rows;
    out[3] = out[4] = 0;                     // markers of an iteration, largest rows of a step
    for (uint32_t part = 0; part < p.parts; ++part) {
        uint64_t rows = 0;
        for (uint32_t q = 0; q < n; ++q) {
            const uint32_t a = p.first(M[q], B[q], part), b = p.first(M[q], B[q], part + 1);
            if (b < a || (b > a && a % B[q])) out[3] = 1ull << 62;
            rows += b - a;
        }
        out[3] += rows;
        if (rows * p.step > out[4]) out[4] = rows * p.step;
    }
}
extern "C" void plan(uint32_t N, uint32_t M, uint32_t B, uint32_t total, uint64_t most, uint64_t* out)
{
    const brr::GramPlan p = brr::gram_plan(N, M, B, total, most);
    out[0] = p.step; out[1] = p.splits; out[2] = p.rows; out[3] = p.acc_rows; out[4] = p.parts;
    out[5] = out[6] = out[7] = out[8] = 0;   // markers swept, launches, largest rows, rows of split launches
    for (uint32_t it = 0; it < p.total; it += p.step)
        for (uint32_t q = 0; q < p.parts; ++q) {
            const uint64_t rows = (uint64_t)p.iterations(it) * p.markers(M, q);
            out[5] += rows;
            out[6] += 1;
            if (rows == 0 || q * p.part % B) out[5] = ~0ull;   // an empty part, or one that starts inside a block
            if (rows > out[7]) out[7] = rows;
            if (p.splits > 1 && rows > out[8]) out[8] = rows;
        }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("gram_plan")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{CSRC}", str(d / "shim.cpp"), "-o",
                    str(d / "shim.so")], check=True)
    lib = C.CDLL(str(d / "shim.so"))

    def cohorts(ms, bs, total, most):
        out = (C.c_uint64 * 5)()
        arr = C.c_uint32 * len(ms)
        lib.cohort_plan(len(ms), arr(*ms), arr(*bs), total, C.c_uint64(most), out)
        return dict(zip(("step", "parts", "rows", "swept", "used"), out))

    def call(n, m, b, total, most=262144):
        out = (C.c_uint64 * 9)()
        lib.plan(n, m, b, total, C.c_uint64(most), out)
        return dict(zip(("step", "splits", "rows", "acc_rows", "parts", "swept", "launches", "used", "used_acc"), out))
    call.cohorts = cohorts
    return call


# the last launch of a chain is shorter than the others and may hold few blocks
@pytest.mark.parametrize("n", [500, 5000, 100000])
def test_launches_stay_inside_their_workspace(plan, n):
    ms = [1, 63, 64, 65, 200, 500, 700, 1000, 3000, 4095, 8128, 8192, 9000, 33000, 65536, 65537, 300000]
    for m, b, total in itertools.product(ms, [1, 2, 33, 64], [1, 2, 3, 7, 9, 23, 67, 100, 200, 400, 1000, 5000]):
        p = plan(n, m, b, total)
        at = (n, m, b, total, p)
        assert p["swept"] == total * m, at
        assert p["used"] <= p["rows"] <= max(min(m, 262144), 65536), at
        assert p["used_acc"] <= p["acc_rows"], at
        assert p["acc_rows"] == 0 or p["acc_rows"] <= 128 * 64, at
        # nearly equal launches, no more of them than their bound asks for
        assert p["launches"] <= -(-total // max(1, 65536 // m)) * p["parts"], at
        assert p["parts"] == 1 or m > 262144, at


# a workspace smaller than an iteration: the iteration in parts of whole blocks
@pytest.mark.parametrize("most", [64, 100, 4096, 8192, 65536, 262144])
def test_parts_stay_inside_a_small_workspace(plan, most):
    for m, b, total in itertools.product([1, 63, 64, 65, 129, 4097, 8192, 8193, 70000, 300001], [1, 2, 33, 64], [1, 2, 5]):
        p = plan(5000, m, b, total, most)
        at = (most, m, b, total, p)
        assert p["swept"] == total * m, at
        assert p["used"] <= p["rows"] <= most, at
        assert p["used_acc"] <= p["acc_rows"] and (p["acc_rows"] == 0 or p["acc_rows"] <= 128 * 64), at


# the steps of several contexts: each holds every context's next iterations, or the next part of their blocks
@pytest.mark.parametrize("most", [8192, 65536, 524288])
def test_cohort_steps_stay_inside_their_workspace(plan, most):
    for ms, bs in (([5], [64]), ([200, 4001, 64], [64, 64, 2]), ([20000] * 8, [64] * 8), ([300000, 1, 70000], [64, 64, 33]),
                   ([100000] * 40, [64] * 40), ([64] * 9000, [64] * 9000), ([1] * 9000, [1] * 9000)):
        for total in (1, 2, 3, 10, 1000):
            p = plan.cohorts(ms, bs, total, most)
            at = (most, ms[:4], len(ms), total, p)
            assert 1 <= p["step"] <= total and (p["parts"] == 1 or p["step"] == 1), at
            assert p["swept"] == sum(ms) and p["used"] == p["rows"], at
            if max(ms) > 64 * len(ms):
                assert p["rows"] <= most + 64 * len(ms), at
