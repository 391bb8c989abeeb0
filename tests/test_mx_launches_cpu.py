"""What a block-scaled call launches, and that the workspace query counts on it: on the CPU, as test_dispatch_cpu.py does for plain operands."""
import json
import os
import random
import subprocess
import sys

import pytest

from tests import abi_ctypes as ac
from tests.test_dispatch_cpu import CHILD, GEMM, HERE, matrix_core

MX_CHILD = CHILD[:CHILD.index("for c in json.load")] + """
for M, N, K, room in json.load(sys.stdin):
    recorder.forget()
    need = L.mi355_gemm_mx_workspace_bytes(M, N, K, 1)
    room = need if room is None else room
    st = L.mi355_gemm_tn_mxfp8(1 << 44, 2 << 44, 3 << 44, M, N, K, K, K, N, 4 << 44, K // 32, 6 << 44, K // 32, 1, 0, (5 << 44) if room else None, room, None)
    out.append((st, need, [(recorder.recorded_name(i).decode(), recorder.recorded_values(i)[:12]) for i in range(recorder.recorded())]))
json.dump(out, sys.stdout)
"""


@pytest.fixture(scope="module")
def mx_launches(tmp_path_factory):
    """mx_launches(problems, room) -> [(status, workspace query, [(kernel, values)])], scales shuffled by the caller."""
    so = str(tmp_path_factory.mktemp("recorder") / "recorder.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-isystem", "/opt/rocm/include",
                    "-o", so, os.path.join(HERE, "launch_recorder.cpp")], check=True)

    def ask(problems, room=None):
        run = subprocess.run([sys.executable, "-c", MX_CHILD, so, os.path.dirname(HERE)], input=json.dumps([[*p, room] for p in problems]), text=True,
                             capture_output=True, check=True)
        return [(st, need, [(name, dict(zip(GEMM, v)) if "gemm_tn_" in name else None) for name, v in got]) for st, need, got in json.loads(run.stdout)]
    return ask


def problems_of(n, seed):
    rng = random.Random(seed)
    return [(int(2 ** rng.uniform(9, 13.2)), int(2 ** rng.uniform(9, 15.6)) // 4 * 4, int(2 ** rng.uniform(9, 13.8)) // 128 * 128) for _ in range(n)]


def test_launches_do_not_depend_on_more_room(mx_launches):
    problems = [(2163, 7716, 7552), (5371, 3328, 8192), (1043, 28160, 7168)] + problems_of(800, 6)
    cut = 0
    for p, (st, need, got), (_, _, more) in zip(problems, mx_launches(problems), mx_launches(problems, 1 << 30)):
        assert st == ac.OK and got == more, p
        cut += sum(matrix_core(name) for name, _ in got) > 1
    assert cut >= 60


def test_halves_cover_the_problem_and_stay_in_the_room(mx_launches):
    problems = [(6144, 4096, 4096), (1480, 12160, 8320)] + problems_of(800, 7)
    for room in (None, 0):
        for p, (st, need, got) in zip(problems, mx_launches(problems, room)):
            M, N, K = p
            products = [v for name, v in got if matrix_core(name)]
            assert st == ac.OK and sum(v["M"] * v["N"] for v in products) == M * N, p
            for v in products:
                m0, n0 = divmod((v["C"] - (3 << 44)) // 2, N)
                assert (v["A"], v["B"]) == ((1 << 44) + m0 * K, (2 << 44) + n0 * K) and m0 + v["M"] <= M and n0 + v["N"] <= N
                if v["splits"] > 1 and M > 64:
                    assert 4 * v["splits"] * v["M"] * v["N"] <= (need if room is None else 0), p


def test_what_is_cut_besides_what_the_queries_report(mx_launches):
    """As the header says: also problems that they give a tail split, and never more room than the query's."""
    abi, tails, cut_tails = ac.load(), 0, 0
    problems = [(6144, 4096, 4096)] + problems_of(1200, 9)
    for p, (st, need, got) in zip(problems, mx_launches(problems)):
        products = [v for name, v in got if matrix_core(name)]
        if ac.plan(abi, *p, ac.E4M3)[4] > 0 and abi.mi355_gemm_pieces(*p, ac.E4M3, ac.AUTO, None, None) == 1:
            tails += 1
            cut_tails += len(products) == 2
            assert need > 0 and len(products) <= 2, p
    assert tails >= 20 and cut_tails >= 10
