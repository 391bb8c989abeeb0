"""Which problems go to the kernel for products of few outputs, and with which form of it: what a call launches, on the CPU."""
import re

import pytest

from tests import abi_ctypes as ac
from tests.few_outputs_cases import ANY_ROWS, PLAIN
from tests.test_dispatch_cpu import A, B, C, case, launches  # noqa: F401  (fixture)


def form(name):
    m = re.search(r"gemm_tn_slices\w*?Li(\d)ELi(\d)ELi(\d)ELb(\d)ELb(\d)E", name)
    return m and tuple(int(x) for x in m.groups())


def test_every_form_is_among_the_cases(launches):  # noqa: F811
    got = [form(got[0][0]) for _, _, got in launches([case(*c) for c in PLAIN])]
    assert {f[:3] for f in got if f} == {(1, 1, 4), (1, 1, 8), (1, 2, 4), (2, 2, 2), (2, 2, 4), (2, 4, 4), (4, 4, 4)}
    assert sum(f is not None for f in got) >= 0.9 * len(PLAIN)


def test_one_launch_without_a_workspace_and_with_it(launches):  # noqa: F811
    for room in (0, None):
        for noalloc in (False, True):
            for c, (st, _, got) in zip(PLAIN, launches([case(*c, room=room, noalloc=noalloc) for c in PLAIN])):
                if form(got[0][0]):
                    assert st == ac.OK and len(got) == 1 and not form(got[0][0])[3], c


@pytest.mark.parametrize("in_dt", [ac.BF16, ac.E4M3])
def test_rows_of_c_of_any_alignment_have_a_form_of_their_own(launches, in_dt):  # noqa: F811
    for c, (st, _, got) in zip(PLAIN, launches([case(*c[:3], in_dt, ldc=c[1] + 1, c=C + 2, room=1 << 26) for c in PLAIN])):
        assert st == ac.OK
        f = form(got[0][0])
        assert f is None or f[3] == 1, c


@pytest.mark.parametrize("variant", [ac.BASIC, ac.SKINNY, ac.PINGPONG, ac.SIMPLE])
def test_explicit_variants_stay_on_their_kernels(launches, variant):  # noqa: F811
    cases = [case(*c, variant=variant) for c in PLAIN if variant != ac.SKINNY or c[0] <= 256]
    assert all(form(name) is None for _, _, got in launches(cases) for name, _ in got)


def test_large_products_stay_where_they_were(launches):  # noqa: F811
    large = [(16, 14336, 4096), (64, 4096, 14336), (256, 4096, 4096), (2048, 2048, 2048), (17, 4100, 4096), (512, 6144, 4096), (8192, 128, 4096)]
    assert all(form(name) is None for _, _, got in launches([case(*c) for c in large]) for name, _ in got)


def test_rows_of_any_alignment(launches):  # noqa: F811
    """16-bit products of few outputs always, e4m3 ones where they would be copied for the matrix cores; with the same refusals."""
    es = {ac.BF16: 2, ac.F16: 2, ac.E4M3: 1}
    cases = [case(m, n, k, dt, lda=k + gap, ldb=k + gap, a=A + off * es[dt], b=B + off * es[dt], room=1 << 27) for m, n, k, dt, off, gap in ANY_ROWS]
    forms = set()
    for c, (st, _, got) in zip(cases, launches(cases)):
        f = form(got[0][0])
        assert st == ac.OK and f and f[4] == 1 and len(got) == 1, (c, got)
        forms.add(f[:3])
    assert len(forms) >= 6
    for c in cases:
        c["variant"] = ac.SIMPLE
    assert all(form(got[0][0]) is None for _, _, got in launches(cases))


def test_rows_of_any_alignment_go_elsewhere(launches):  # noqa: F811
    cases = [case(16, 1001, 1001, ac.E4M3), case(16, 1001, 7), case(64, 1001, 1001, ldb=1 << 26),          # fp32 sums; short rows; out of reach
             case(515, 2050, 4100, room=0), case(4096, 4096, 4098), case(3154, 878, 7747)]            # no workspace; large
    for c, (st, _, got) in zip(cases, launches(cases)):
        assert st == ac.OK and all(form(name) is None or form(name)[4] == 0 for name, _ in got), (c, got)
    for c in (case(10, 10028, 12846), case(515, 2050, 4100)):     # the copies of the first are beyond the library's own scratch memory
        (st, need, got), = launches([dict(c, noalloc=True)])
        assert (st, len(got)) == ((ac.ERR_SCRATCH, 0) if need > ac.NOALLOC_SCRATCH_BYTES else (ac.OK, 1))
