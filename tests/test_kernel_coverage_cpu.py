"""That the cases of kernel_coverage_cases.py reach what they are there for: what their calls launch, on the CPU."""
import re

from tests import abi_ctypes as ac
from tests.kernel_coverage_cases import MX, ODD_ROWS, REPACKED
from tests.test_dispatch_cpu import case, launches  # noqa: F401  (fixture)
from tests.test_mx_launches_cpu import mx_launches  # noqa: F401  (fixture)


def kernels(answers):
    """(kernel and tile, whether K is split, whether the last round is) of every product; the other launches by name."""
    out = set()
    for st, _, got in answers:
        assert st == ac.OK
        for name, v in got:
            tile = re.search(r"gemm_tn_tile_ring\w*?Li(\d+)ELi\d+ELi(\d+)E", name)
            stream = re.search(r"gemm_tn_stream\w*?Li(\d+)ELi(\d+)ELi(\d)E", name)
            if tile:
                out.add(("tile", int(tile.group(1)), int(tile.group(2)), v["splits"] > 1, v["tail_tiles"] > 0))
            elif stream:      # blocks of 16 rows, over the waves that share them
                out.add(("stream", int(stream.group(1)) * int(stream.group(3)), len(got) > 1 and "splitk_reduce" in got[-1][0]))
            else:
                out.add(re.search(r"(splitk_reduce|tail_reduce|repack_rows|copy_out|gemm_tn_\w+?)(?=I|E)", name).group(1))
    return out


TILES = {("tile", 128, 128, False, False), ("tile", 128, 128, True, False), ("tile", 256, 128, False, False), ("tile", 256, 128, True, False),
         ("tile", 256, 256, False, False)}


def test_block_scaled(mx_launches):  # noqa: F811
    got = kernels(mx_launches(MX))
    assert got >= TILES | {("stream", rows, split) for rows in (1, 2, 4) for split in (False, True)} | {("tile", 256, 256, False, True), "tail_reduce"}


def test_rows_of_c_of_any_alignment(launches):  # noqa: F811
    for dt in (ac.BF16, ac.E4M3):
        got = kernels(launches([case(*c) for c in ODD_ROWS if c[3] == dt]))
        assert got >= TILES | {("stream", rows, split) for rows in (1, 2, 4, 8) for split in (False, True)}
    assert ("tile", 256, 256, False, True) in kernels(launches([case(*c) for c in ODD_ROWS]))


def test_repacked(launches):  # noqa: F811
    answers = launches([case(*c) for c in REPACKED])
    assert all("repack_rows" in got[0][0] for _, _, got in answers)
    assert kernels(answers) >= TILES | {("stream", 4, True), ("stream", 8, True)}
