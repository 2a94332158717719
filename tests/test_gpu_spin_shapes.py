"""The spin phases (row products, core products, transposes) at the edges of their shapes,
through the C-ABI against the oracle: rows narrower than one vector, odd row lengths (every row
starts at its own alignment, the last lanes repeat the last columns), lists split over four
waves and the first size that is not, and core-product passes whose last column range holds a
single column, FP64 and FP32, in one stream and beside the alpha-beta kernel.

Bars: FP64 within 1e-12 of the oracle relative to its largest element, FP32 within 2e-5 (the
bars of the other sigma tests)."""
import numpy as np
import pytest

import oracle
import sbdg
from helpers import core_split, workload_small

pytestmark = pytest.mark.gpu


def check(case, **options):
    s = sbdg.Solver(case["norb"], case["core"], case["h1"], case["eri"], case["astr"], case["bstr"], **options)
    p = oracle.Problem(case["norb"], case["core"], case["h1"], case["astr"], case["bstr"], eri=case["eri"])
    x = np.random.default_rng(11).normal(size=s.ndet)
    want = p.sigma(x)
    top = np.abs(want).max()
    for overlap in (0, 1):
        s.set_options(overlap=overlap)
        e64 = np.abs(s.sigma(x) - want).max() / top
        e32 = np.abs(s.sigma(x, precision=1) - want).max() / top
        print(f"{s.na} x {s.nb}, {options}, overlap {overlap}: FP64 {e64:.1e}, FP32 {e32:.1e}", flush=True)
        assert e64 <= 1e-12 and e32 <= 2e-5
    return s


@pytest.mark.parametrize("na,nb", [(3, 1), (1, 3), (2, 5), (7, 2), (63, 65), (129, 67), (511, 515), (1021, 1027),
                                   (1025, 1025), (300, 4001)])
def test_sigma_at_row_lengths(na, nb):
    check(workload_small(20, 4, 4, na, nb, 43)).close()


@pytest.mark.parametrize("doubles", [1, 2])
def test_sigma_odd_rows_by_table_and_by_core(doubles):
    check(workload_small(16, 5, 4, 601, 703, 47), doubles=doubles).close()


def test_core_pass_of_one_column():
    """The core workspace capped at one 512-column pass over rows of 1,025 and 513 columns."""
    case = workload_small(18, 5, 5, 513, 1025, 53)
    s = check(case, doubles=2)
    members = max(s.stats()["core_members"])
    s.close()
    assert members > 0
    s = check(case, doubles=2, core_gib=(members * 512 * 8 + 4096) / 2**30)
    s.close()


@pytest.mark.parametrize("norb,nb,capped", [(10, 129, False), (11, 203, False), (12, 65, False), (13, 1025, True)])
def test_core_sizes_around_the_workspace_cut(norb, nb, capped):
    """All alpha strings of five electrons: cores of 21, 28, 36 and 45 members, either side of
    the size from which they go through the workspace (28), and a last pass of one column."""
    case = workload_small(norb, 5, 5, 0, nb, 59)
    s = check(case, doubles=2)
    members = max(s.stats()["core_members"])
    s.close()
    if capped:
        check(case, doubles=2, core_gib=(members * 512 * 8 + 4096) / 2**30).close()


@pytest.mark.parametrize("na", [3, 256, 257, 513])
def test_core_pass_of_few_columns_and_many_blocks(na):
    """Rows of up to 128 vectors (256 columns in FP64, 512 in FP32) over the 2,800 product blocks
    of all strings of five electrons in 16 orbitals, and the first row length beyond."""
    check(workload_small(16, 5, 5, na, 0, 73), doubles=2).close()


def test_core_passes_end_with_one_column():
    """1,025 of the 1,287 strings of five electrons in 13 orbitals on either side, most of whose
    cores go through the workspace, with the workspace capped at one 512-column pass of the cores
    of ten members and more: both precisions take several passes, the last of a single column."""
    case = workload_small(13, 5, 5, 1025, 1025, 89)
    s = check(case, doubles=2)
    members = s.stats()["core_members"]
    s.close()
    cap = max(members) * 512 * 8
    for strs, kept in zip((case["astr"], case["bstr"]), members):
        assert core_split(strs)[0] == kept
        through = core_split(strs, 28)[0]
        for size in (8, 4):
            columns = cap // (size * through) // 512 * 512
            assert 512 <= columns < 1025 and 1025 % columns == 1
    check(case, doubles=2, core_gib=(cap + 64) / 2**30).close()
