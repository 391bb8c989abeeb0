"""Problems of a few tiles more than whole rounds: cut in two by a call, whatever the number of k-steps; what each half is, on the CPU."""
import random
import re

import pytest

from tests import abi_ctypes as ac
from tests.test_dispatch_cpu import A, B, C, case, launches, matrix_core  # noqa: F401  (fixture)


def covered(c, got, es):
    """The products' rectangles of C make up all of it, each from its own rows of A and B."""
    rects = []
    for name, v in got:
        if matrix_core(name):
            m0, n0 = divmod((v["C"] - C) // 2, c["ldc"])
            assert v["A"] == A + m0 * c["lda"] * es and v["B"] == B + n0 * c["ldb"] * es and v["K"] == c["K"]
            rects.append((m0, n0, v["M"], v["N"]))
    assert sum(m * n for _, _, m, n in rects) == c["M"] * c["N"]
    assert all(m0 + m <= c["M"] and n0 + n <= c["N"] for m0, n0, m, n in rects)
    assert len(rects) in (1, 2) and (len(rects) == 1 or rects[0][:2] == (0, 0) and rects[1][:2] in ((rects[0][2], 0), (0, rects[0][3])))
    return len(rects)


@pytest.mark.parametrize("M,N,K,in_dt", [(1000, 50257, 768, ac.BF16), (1000, 50260, 768, ac.F16), (2123, 8032, 1408, ac.BF16), (1509, 11192, 3200, ac.E4M3),
                                         (6784, 2504, 1792, ac.BF16), (3748, 13208, 640, ac.BF16)])
def test_cut(launches, M, N, K, in_dt):  # noqa: F811
    es = 1 if in_dt == ac.E4M3 else 2
    cases = [case(M, N, K, in_dt), case(M, N, K, in_dt, room=0) if N % 4 == 0 else case(M, N, K, in_dt, room=256), case(M, N, K, in_dt, noalloc=True)]
    for c, (st, _, got) in zip(cases, launches(cases)):
        assert st == ac.OK and covered(c, got, es) == 2, c


def test_what_the_queries_call_one_launch_with_a_tail_split_is_one(launches):  # noqa: F811
    """Its result is the tile variant's to the bit."""
    abi, rng, tails = ac.load(), random.Random(4), 0
    problems = [(4352, 4352, 4096), (1056, 26704, 2176), (6784, 2504, 2304)]
    problems += [(rng.randint(1000, 7000), 4 * rng.randint(500, 3000), 64 * rng.randint(32, 90)) for _ in range(300)]
    cases = [case(*p) for p in problems]
    for p, c, (st, _, got) in zip(problems, cases, launches(cases)):
        if abi.mi355_gemm_pieces(*p, ac.BF16, ac.AUTO, None, None) == 1 and ac.plan(abi, *p, ac.BF16)[4] > 0:
            tails += 1
            assert st == ac.OK and covered(c, got, 2) == 1, p
    assert tails >= 20


def test_halves_cover_random_problems(launches):  # noqa: F811
    rng = random.Random(3)
    cases = []
    for _ in range(300):
        in_dt = rng.choice([ac.BF16, ac.E4M3])
        M, N, K = int(2 ** rng.uniform(8, 13.2)), int(2 ** rng.uniform(9, 15.6)) // 4 * 4, int(2 ** rng.uniform(7, 13)) // 16 * 16
        cases.append(case(M, N, K, in_dt, room=rng.choice([0, None])))
    seen = {covered(c, got, 1 if c["in_dt"] == ac.E4M3 else 2) for c, (st, _, got) in zip(cases, launches(cases)) if st == ac.OK}
    assert seen == {1, 2}


def launched(got):
    """What was launched, wherever the workspace lies."""
    return [(name, [v[k] for k in ("M", "N", "K", "lda", "ldb", "ldc", "A", "B", "C", "c_ragged", "splits", "tail_tiles")] if "gemm_tn_" in name else None) for name, v in got]


def test_halves_do_not_depend_on_the_workspace(launches):  # noqa: F811
    """The same kernels and splits, so the same sums, with the room that the query asks for, with more, and without allocation."""
    rng = random.Random(6)
    problems = [(3518, 14380, 7168, ac.BF16), (2167, 21868, 9792, ac.BF16), (3094, 16012, 12928, ac.BF16), (4139, 12620, 12224, ac.E4M3)]
    problems += [(int(2 ** rng.uniform(9, 13.2)), int(2 ** rng.uniform(9, 15.6)) // 4 * 4, int(2 ** rng.uniform(10, 13.8)) // 16 * 16, rng.choice([ac.BF16, ac.E4M3]))
                 for _ in range(800)]
    answers = [launches([case(*p, room=room, noalloc=noalloc) for p in problems]) for room, noalloc in ((None, False), (1 << 30, False), (None, True))]
    cut = 0
    for p, (st, _, got), more, without in zip(problems, *answers):
        assert (st, more[0], without[0]) == (ac.OK, ac.OK, ac.OK)
        assert launched(got) == launched(more[2]) == launched(without[2]), p
        cut += sum(matrix_core(name) for name, _ in got) > 1
    assert cut >= 60


def test_a_half_without_splits_has_tiles_for_that(launches):  # noqa: F811
    """Not the large tiles of a plan that would have cut K, on less than half of the compute units."""
    rng = random.Random(8)
    problems = [(3094, 16012, 12928, ac.BF16), (5436, 9524, 9920, ac.BF16), (4139, 12620, 12224, ac.E4M3), (565, 23296, 3712, ac.BF16)]
    problems += [(int(2 ** rng.uniform(9, 13.2)), int(2 ** rng.uniform(9, 15.6)) // 4 * 4, int(2 ** rng.uniform(12, 13.8)) // 16 * 16, rng.choice([ac.BF16, ac.E4M3]))
                 for _ in range(1500)]
    seen = 0
    for p, (st, _, got) in zip(problems, launches([case(*p) for p in problems])):
        products = [(name, v) for name, v in got if matrix_core(name)]
        for name, v in products if len(products) == 2 else []:
            tile = re.search(r"gemm_tn_tile_ring\w*?Li(\d+)ELi\d+ELi(\d+)E", name)
            if tile and v["splits"] == 1 and v["tail_tiles"] == 0:
                rows, cols = int(tile.group(1)), int(tile.group(2))
                seen += 1
                assert rows == 128 or -(-v["M"] // rows) * -(-v["N"] // cols) > 128, (p, name, v)
    assert seen >= 100
