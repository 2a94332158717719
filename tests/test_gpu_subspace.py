"""The small eigenproblem of the Davidson steps at its sizes: bases of 3 up to the 48 allowed (odd
and even, up to more 2 x 2 blocks than lanes), grown to their end before a restart.

Bars: the solver stops at a residual norm of 1e-7, so the energy is within 1e-10 of the dense
one (residual squared over a gap of some tenths, and rounding), and the residual of the returned
vector, by the oracle's sigma, within 2e-7."""
import numpy as np
import pytest

import oracle
import sbdg
from helpers import workload_small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_nb", [3, 4, 7, 10, 17, 33, 47, 48])
def test_davidson_with_bases_of(max_nb):
    c = workload_small(10, 3, 3, 24, 21, 71)
    p = oracle.Problem(c["norb"], c["core"], c["h1"], c["astr"], c["bstr"], eri=c["eri"])
    n = len(c["astr"]) * len(c["bstr"])
    h = np.stack([p.sigma(e) for e in np.eye(n)])
    want = np.linalg.eigvalsh(h)[0]
    s = sbdg.Solver(c["norb"], c["core"], c["h1"], c["eri"], c["astr"], c["bstr"], max_it=400, max_nb=max_nb,
                    eps=1e-7, init=1, seed=3)
    e = s.run()
    w = s.vector()
    r = np.linalg.norm(p.sigma(w) - e * w)
    print(f"max_nb {max_nb}: energy off by {abs(e - want):.1e}, residual {r:.1e}", flush=True)
    assert abs(e - want) < 1e-10 and r < 2e-7
    s.close()
