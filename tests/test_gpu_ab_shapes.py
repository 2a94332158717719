"""The alpha-beta kernel at the edges of its launch shapes, through the C-ABI: one beta string,
the last column count of each workgroup size and the first of the next, several ket chunks, a
beta list beyond one batch, and alpha rows cut into several segments (their partial rows joined
in order), FP64 and FP32 against the oracle on the same inputs.

Bars: FP64 within 1e-12 of the oracle relative to its largest element, FP32 within 2e-5 (the
bars of the other sigma tests: sums of some hundred terms of unit size, in 53 and 24 bits)."""
import numpy as np
import pytest

import oracle
import sbdg
from helpers import workload_small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("norb,nel,na,nb", [
    (18, 5, 90, 1), (18, 5, 90, 2), (18, 5, 90, 256), (18, 5, 90, 257), (18, 5, 60, 512), (18, 5, 60, 513),
    (18, 5, 60, 1024), (18, 5, 60, 1025), (22, 6, 40, 2047), (22, 6, 40, 6000), (22, 6, 40, 6001),
    (58, 6, 80, 600), (64, 4, 70, 300), (64, 4, 60, 1024), (40, 8, 30, 8193),
])
def test_sigma_at_launch_shape_edges(norb, nel, na, nb):
    c = workload_small(norb, nel, nel, na, nb, 41)
    s = sbdg.Solver(c["norb"], c["core"], c["h1"], c["eri"], c["astr"], c["bstr"])
    p = oracle.Problem(c["norb"], c["core"], c["h1"], c["astr"], c["bstr"], eri=c["eri"])
    x = np.random.default_rng(7).normal(size=s.ndet)
    want = p.sigma(x)
    top = np.abs(want).max()
    longest = int(np.diff(s.table(0)[0]).max())
    e64 = np.abs(s.sigma(x) - want).max() / top
    e32 = np.abs(s.sigma(x, precision=1) - want).max() / top
    print(f"norb {norb}, {na} x {nb}, longest alpha row {longest}: FP64 {e64:.1e}, FP32 {e32:.1e}", flush=True)
    assert longest > 8  # several segments
    assert e64 <= 1e-12 and e32 <= 2e-5
    s.set_options(overlap=0)
    assert np.abs(s.sigma(x) - want).max() <= 1e-12 * top
    s.close()


def test_sigma_with_more_joined_rows_than_a_grid_dimension():
    """All strings of 8 electrons in 19 orbitals: 75,582 alpha rows of 88 singles, each cut after
    64, so that more than 65,535 rows are joined.  Rows at both ends and around that count against
    the oracle, every row on one stream against two."""
    c = workload_small(19, 8, 3, 0, 5, 79)
    s = sbdg.Solver(c["norb"], c["core"], c["h1"], c["eri"], c["astr"], c["bstr"])
    p = oracle.Problem(c["norb"], c["core"], c["h1"], c["astr"], c["bstr"], eri=c["eri"])
    assert s.na > 65535 and int(np.diff(s.table(0)[0]).min()) > 64
    x = np.random.default_rng(8).normal(size=s.ndet)
    hii = p.hii()
    got = {}
    for overlap in (0, 1):
        s.set_options(overlap=overlap)
        for precision in (0, 1):
            got[overlap, precision] = s.sigma(x, precision=precision).reshape(s.na, s.nb)
    top = np.abs(got[0, 0]).max()
    for r0 in (0, 40000, 65520, s.na - 30):
        want = p.sigma_rows(x, hii, r0, r0 + 30).reshape(s.na, s.nb)[r0:r0 + 30]
        for (overlap, precision), y in got.items():
            err = np.abs(y[r0:r0 + 30] - want).max() / top
            print(f"rows {r0}+30, overlap {overlap}, precision {precision}: {err:.1e}", flush=True)
            assert err <= (2e-5 if precision else 1e-12)
    for precision, bar in ((0, 1e-12), (1, 2e-5)):
        assert np.abs(got[0, precision] - got[1, precision]).max() <= bar * top
    s.close()


@pytest.mark.parametrize("norb,nel,na,nb", [
    (12, 4, 200, 2), (18, 5, 90, 63), (18, 5, 90, 64), (18, 5, 90, 65), (18, 5, 90, 128), (18, 5, 90, 129),
    (29, 5, 80, 128), (30, 5, 80, 33), (45, 5, 80, 128), (46, 5, 80, 3), (58, 6, 80, 128),
])
def test_sigma_at_narrow_row_shapes(norb, nel, na, nb):
    """Rows of up to 128 columns: workgroups of 64, 128 and 256 threads by the number of slice
    vectors (406 at norb=29, 990 at 45, 1,035 at 46), and the first row length beyond."""
    test_sigma_at_launch_shape_edges(norb, nel, na, nb)
