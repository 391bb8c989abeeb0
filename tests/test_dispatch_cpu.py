"""What a call of the C ABI launches, looked at without a GPU: the built library's host code runs against a recorder in the
place of the HIP runtime (launch_recorder.cpp), in a process of its own."""
import json
import os
import subprocess
import sys

import pytest

from tests import abi_ctypes as ac

HERE = os.path.dirname(os.path.abspath(__file__))
A, B, C, WS = 1 << 44, 2 << 44, 3 << 44, 5 << 44      # addresses that nothing reads
GEMM = ["M", "N", "K", "lda", "ldb", "ldc", "A", "B", "C", "c_ragged", "splits", "tail_tiles"]
REPACK = ["rows", "src_ld", "src", "dst", "dst_ld", "blocks"]

CHILD = """
import ctypes, json, sys
recorder = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
from tests import abi_ctypes as ac
L = ac.load()
recorder.recorded_name.restype = ctypes.c_char_p
recorder.recorded_values.restype = ctypes.POINTER(ctypes.c_int64)
out = []
for c in json.load(sys.stdin):
    recorder.forget()
    args = [c["A"], c["B"], c["C"], c["M"], c["N"], c["K"], c["lda"], c["ldb"], c["ldc"], c["in_dt"], c["out_dt"], 1.0, c["variant"]]
    need = L.mi355_gemm_workspace_bytes(c["M"], c["N"], c["K"], c["in_dt"], c["variant"])
    room = need if c["room"] is None else c["room"]
    st = L.mi355_gemm_tn_noalloc(*args, None) if c["noalloc"] else L.mi355_gemm_tn(*args, c["ws"] if room else None, room, None)
    got = [(recorder.recorded_name(i).decode(), recorder.recorded_values(i)[:12]) for i in range(recorder.recorded())]
    out.append((st, need, got))
json.dump(out, sys.stdout)
"""


@pytest.fixture(scope="module")
def launches(tmp_path_factory):
    """launches(cases) -> [(status, workspace query, [(kernel, values)])]."""
    so = str(tmp_path_factory.mktemp("recorder") / "recorder.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-isystem", "/opt/rocm/include",
                    "-o", so, os.path.join(HERE, "launch_recorder.cpp")], check=True)

    def ask(cases):
        run = subprocess.run([sys.executable, "-c", CHILD, so, os.path.dirname(HERE)], input=json.dumps(cases), text=True,
                             capture_output=True, check=True)
        out = []
        for st, need, got in json.loads(run.stdout):
            shown = []
            for name, v in got:
                if "repack_rows" in name:
                    v = [dict(zip(REPACK, v[:6])), dict(zip(REPACK, v[6:]))]
                elif "gemm_tn_" in name:
                    v = dict(zip(GEMM, v))
                shown.append((name, v))
            out.append((st, need, shown))
        return out
    return ask


def case(M, N, K, in_dt=ac.BF16, lda=None, ldb=None, ldc=None, a=A, b=B, c=C, variant=ac.AUTO, room=None, noalloc=False, ws=WS):
    """room: bytes of workspace, None for what the query asks."""
    return dict(M=M, N=N, K=K, in_dt=in_dt, out_dt=ac.BF16 if in_dt == ac.E4M3 else in_dt, lda=lda or K, ldb=ldb or K, ldc=ldc or N,
                A=a, B=b, C=c, variant=variant, room=room, noalloc=noalloc, ws=ws)


def matrix_core(name):
    return "gemm_tn_" in name and "gemm_tn_simple" not in name and "gemm_tn_small" not in name


def panel_ok(v, es):
    return 256 * v["lda"] * es < 1 << 31 and 256 * v["ldb"] * es < 1 << 31


# 256 rows of B of 2 GiB and more, N not a multiple of 4: tile and streaming kernels, A aligned or not, K aligned or not.
@pytest.mark.parametrize("in_dt", [ac.BF16, ac.F16, ac.E4M3])
def test_no_kernel_gets_rows_of_b_it_cannot_address(launches, in_dt):
    es = 1 if in_dt == ac.E4M3 else 2
    limit = (1 << 31) // 256 // es
    cases = [case(M, N, K, in_dt, ldb=ldb, a=a, b=b, room=None if a == A else 1 << 34)    # the query counts on aligned rows of A
             for M, N, K in [(4096, 5, 4096), (1024, 257, 1024), (300, 130, 4096), (100, 1001, 2048), (17, 4099, 4096), (2048, 8191, 4100)]
             for ldb in (limit - 16, limit, limit + 3, 1 << 26, 1 << 29)
             for a, b in ((A, B), (A + es, B), (A, B + es))]
    for c, (st, need, got) in zip(cases, launches(cases)):
        assert st == ac.OK and got, c
        for name, v in got:
            if matrix_core(name):
                assert panel_ok(v, es), (c, name, v)
        # with that much workspace every one of these runs on the matrix cores
        assert any(matrix_core(name) for name, _ in got), (c, got)
        packed = [v for name, v in got if "repack_rows" in name]
        if c["ldb"] >= limit:
            assert packed and packed[0][1]["rows"] == c["N"] and packed[0][1]["src_ld"] == c["ldb"] * es


# Copies of 17 GB and of 36 and 40 GB (two launches: one counts below 2^31 chunks of 16 bytes), of B and of A; 34 GB of fp8.
@pytest.mark.parametrize("M,N,K,in_dt,copies", [(8192, 262144, 33001, ac.BF16, 1), (64, 600000, 33001, ac.BF16, 2), (550000, 40, 32801, ac.F16, 2),
                                                (300, 530001, 65001, ac.E4M3, 2)])
def test_copies_of_any_size_are_made(launches, M, N, K, in_dt, copies):
    es = 1 if in_dt == ac.E4M3 else 2
    cases = [case(M, N, K, in_dt), case(M, N, K, in_dt, noalloc=True)]
    (st, need, got), (st_noalloc, _, got_noalloc) = launches(cases)
    assert st == ac.OK and need > 17e9
    packed = [v for name, v in got if "repack_rows" in name]
    assert len(packed) == copies
    for i, (src, rows) in enumerate(((A, M), (B, N))):
        parts = [p[i] for p in packed if p[i]["rows"]]
        assert sum(p["rows"] for p in parts) == rows
        at, to = src, parts[0]["dst"]
        for p in parts:      # one after the other, without a gap
            chunks = p["rows"] * (p["dst_ld"] // 16)
            assert (p["src"], p["dst"], p["src_ld"]) == (at, to, K * es)
            assert chunks < 1 << 31 and p["blocks"] == -(-chunks // 1024)
            at, to = at + p["rows"] * p["src_ld"], to + p["rows"] * p["dst_ld"]
        assert WS <= parts[0]["dst"] and to <= WS + need
    assert any(matrix_core(name) for name, _ in got) and not any("simple" in name for name, _ in got)
    assert st_noalloc == ac.ERR_SCRATCH and not got_noalloc


# Rows of C of 2^21 elements and more: the tile kernels' 32-bit offsets do not reach them, a padded copy of C does.
@pytest.mark.parametrize("in_dt", [ac.BF16, ac.E4M3])
@pytest.mark.parametrize("M,N,K", [(300, 1003, 1024), (100, 4099, 4096), (4096, 5, 4096), (2048, 8190, 129), (8192, 16385, 128), (300, 1000, 1024)])
def test_rows_of_c_out_of_reach(launches, in_dt, M, N, K):
    limit = 1 << 21
    strides = (limit - 3, limit - 1, limit + 1, limit + 6, 1 << 24)     # none aligned where N is
    cases = [case(M, N, K, in_dt, ldc=ldc + (ldc % 4 == 0 and N % 4 == 0), room=1 << 31) for ldc in strides]
    for c, (st, need, got) in zip(cases, launches(cases)):
        assert st == ac.OK
        products = [v for name, v in got if matrix_core(name)]
        assert products and not any("simple" in name for name, _ in got), c
        assert all(256 * v["ldc"] * 4 < 1 << 31 for v in products), c
        out_of_reach = 256 * (-(-c["ldc"] // 4) * 4) * 4 >= 1 << 31
        assert ("copy_out" in got[-1][0]) == out_of_reach, (c, got)
        for v in products:
            if out_of_reach:      # whole quads of columns fit in a padded row
                assert WS <= v["C"] < WS + need + (1 << 31) and v["ldc"] >= -(-N // 4) * 4 and v["ldc"] % 64 == 0 and not v["c_ragged"]
            else:
                assert v["ldc"] == c["ldc"]


# Under 2^27 operations, everything aligned but the rows of C.
@pytest.mark.parametrize("M,N,K,ldc", [(1, 129, 128, 129), (16, 1001, 4096, 1001), (64, 71, 14336, 71), (257, 501, 512, 501), (100, 128, 1024, 130),
                                       (3, 30001, 64, 30001), (1, 4, 16, 5)])
def test_small_fp8_products_keep_their_fp32_sums(launches, M, N, K, ldc):
    cases = [case(M, N, K, ac.E4M3, ldc=ldc, room=room, noalloc=noalloc) for room in (0, None, 1 << 26) for noalloc in (False, True)]
    for st, need, got in launches(cases):
        assert st == ac.OK and (need == 0 or N % 4 == 0)
        assert [("gemm_tn_small" if K >= 128 else "gemm_tn_simple") in name for name, _ in got] == [True]
    for st, need, got in launches([case(M, N, K, ac.BF16, ldc=ldc)]):
        assert st == ac.OK and all(not matrix_core(name) or v["c_ragged"] for name, v in got) and matrix_core(got[0][0])


@pytest.mark.parametrize("M,N,K,split", [(16, 14336, 4096, False), (16, 14333, 4096, False), (17, 4100, 4096, True), (17, 4099, 4096, True),
                                         (64, 16896, 2048, False), (64, 16897, 2048, False)])
def test_streaming_kernel_has_a_form_for_each_kind_of_rows(launches, M, N, K, split):
    """The form for rows of any alignment is launched for those only, and nothing is decided about C inside a kernel."""
    (st, _, got), = launches([case(M, N, K)])
    assert st == ac.OK and len(got) == 1 + split and "gemm_tn_stream" in got[0][0]
    ragged = N % 4 != 0
    writes_c = got[-1][0]      # the reduction of a K split, else the product itself
    assert ("splitk_reduce" in writes_c) == split
    assert ("Lb1E" in writes_c) == ragged
    if split:
        assert "Lb1E" not in got[0][0]


# Rows at odd 2-byte addresses under a plan with tiles of 256 rows are stored directly, with or without room for a padded copy of C
# (which took 3-21 % longer on 80 sizes).
@pytest.mark.parametrize("M,N,K,in_dt,padded", [(4096, 14337, 2048, ac.BF16, False), (8192, 8193, 4096, ac.F16, False), (2048, 4097, 8192, ac.E4M3, False),
                                                (1000, 50257, 768, ac.BF16, False), (8192, 8193, 512, ac.BF16, False), (9335, 9969, 1536, ac.BF16, False)])
def test_rows_of_c_at_odd_addresses(launches, M, N, K, in_dt, padded):
    cases = [case(M, N, K, in_dt), case(M, N, K, in_dt, c=C + 2), case(M, N, K, in_dt, room=256), case(M, N, K, in_dt, noalloc=True),
             case(M, N + 1 - N % 4, K, in_dt, ldc=N + 4), case(M, N, K + 1, in_dt), case(M, N, K, in_dt, ldc=N + 1)]
    for c, (st, need, got) in zip(cases, launches(cases)):
        assert st == ac.OK
        products = [v for name, v in got if matrix_core(name)]
        assert products and not any("simple" in name for name, _ in got)
        room = need if c["room"] is None else c["room"]
        odd = c["ldc"] % 2 != 0 or c["C"] % 4 != 0
        fits = room > 2 * M * N and (not c["noalloc"] or 2 * M * -(-N // 64) * 64 <= ac.NOALLOC_SCRATCH_BYTES)
        assert ("copy_out" in got[-1][0]) == (padded and odd and fits), (c, got)
        for v in products:
            assert v["c_ragged"] == 0 or v["C"] >= c["C"] and v["ldc"] == c["ldc"]
            if "copy_out" in got[-1][0]:      # inside the workspace, behind the copies of the operands if there are any
                packed = [p for name, p in got if "repack_rows" in name]
                end = max([o["dst"] + o["rows"] * o["dst_ld"] for p in packed for o in p], default=WS) if not c["noalloc"] else 0
                assert v["C"] >= end and v["C"] + 2 * ((v["M"] - 1) * v["ldc"] + v["N"]) <= (WS if not c["noalloc"] else 1 << 30) + max(room, 64 << 20)
        # no row or column is left to nobody
        assert sum(v["M"] * v["N"] for v in products) == M * c["N"]


@pytest.mark.parametrize("M,N,K,in_dt", [(908, 10640, 832, ac.F16), (3612, 1516, 4016, ac.E4M3), (8192, 8192, 512, ac.BF16), (1024, 1032, 512, ac.BF16)])
def test_rows_of_less_than_64_bytes_are_stored_plainly(launches, M, N, K, in_dt):
    cases = [case(M, N, K, in_dt, ldc=N + pad, c=C + off) for pad in (0, 4, 32) for off in (0, 8, 64)]
    for c, (st, _, got) in zip(cases, launches(cases)):
        assert st == ac.OK
        plain = M * N >= 4 << 20 and (c["ldc"] * 2 % 64 != 0 or c["C"] % 64 != 0)
        for name, v in got:
            if "gemm_tn_tile_ring" in name:
                assert bool(v["c_ragged"]) == plain
