"""The RDM kernels at the edges of their shapes, through the C-ABI against the oracle on the same
vector: one to three beta strings, odd row lengths, few beta pairs (one and four alpha pairs per
step) and many, the last row length of one column chunk and the first of two and of three, alpha
sets with a single string, and same-spin parts on rows of one column.

Bars: 1e-11 on the RDMs, their partial traces and Hermiticity (sums of at most some ten thousand
products of a unit vector's elements: a few hundred units of 1e-16), bit-identical on repetition
(every sum has a fixed order)."""
import numpy as np
import pytest

import oracle
import sbdg
from helpers import rdm_close, rdm_invariants, workload_small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("norb,nel,na,nb", [
    (12, 4, 40, 1), (12, 4, 1, 40), (12, 4, 30, 2), (12, 4, 30, 3), (16, 5, 65, 129), (16, 5, 30, 638),
    (26, 5, 25, 641), (26, 5, 20, 2001), (18, 5, 20, 5116), (18, 5, 20, 5117), (22, 5, 9, 10241), (64, 3, 50, 70),
])
def test_rdm_at_shape_edges(norb, nel, na, nb):
    c = workload_small(norb, nel, nel, na, nb, 61)
    w = np.random.default_rng(5).normal(size=na * nb)
    w /= np.linalg.norm(w)
    p = oracle.Problem(c["norb"], c["core"], c["h1"], c["astr"], c["bstr"], eri=c["eri"])
    one_o, two_o = p.rdm(w)
    for doubles in (0, 1):
        s = sbdg.Solver(c["norb"], c["core"], c["h1"], c["eri"], c["astr"], c["bstr"], doubles=doubles, max_it=1,
                        max_nb=2, eps=1e10, init=2, do_rdm=1)
        s.set_vector(w)
        s.run()
        one, two = s.rdm()
        print(f"norb {norb}, {na} x {nb}, doubles {doubles}: one {np.abs(one - one_o).max():.1e}, "
              f"two {np.abs(two[[0, 3]] - two_o[[0, 3]]).max():.1e} "
              f"{np.abs(two[1] + two[2] - two_o[1] - two_o[2]).max():.1e}", flush=True)
        rdm_close(one, two, one_o, two_o, 1e-11, mixed_sum=True)
        rdm_invariants(one, two, nel, nel, norb, 1e-11)
        one2, two2 = s.rdm(compute=True)
        assert np.array_equal(one, one2) and np.array_equal(two, two2)
        dens = s.density()
        assert np.abs(dens[0::2] - one[0].reshape(norb, norb).diagonal()).max() < 1e-12
        assert np.abs(dens[1::2] - one[1].reshape(norb, norb).diagonal()).max() < 1e-12
        s.close()


@pytest.mark.parametrize("norb,nel,na,nb", [(12, 4, 40, 1), (16, 5, 65, 129), (18, 5, 900, 700)])
def test_rdm_same_bits_whatever_memory_is_idle(norb, nel, na, nb):
    """The transient buffers come out of the idle Davidson vectors and, where those have no room,
    from allocations: the same RDMs and gradients with a basis of 2 and of 40 vectors, and the
    solution intact afterwards."""
    c = workload_small(norb, nel, nel, na, nb, 67)
    w = np.random.default_rng(6).normal(size=na * nb)
    w /= np.linalg.norm(w)
    got = []
    for max_nb, precision in ((2, 0), (40, 0), (40, 1)):
        s = sbdg.Solver(c["norb"], c["core"], c["h1"], c["eri"], c["astr"], c["bstr"], max_it=1, max_nb=max_nb,
                        eps=1e10, init=2, do_rdm=1)
        s.set_vector(w)
        s.run()
        s.set_options(precision=precision)
        before = s.vector()
        one, two = s.rdm(compute=True)
        got.append((one, two, *s.rdm_backward(2.0), s.density()))
        assert np.array_equal(s.vector(), before)
        s.close()
    for other in got[1:]:
        assert all(np.array_equal(x, y) for x, y in zip(got[0], other))


def test_rdm_after_new_integrals_and_new_strings():
    """The beta-pair tables belong to the beta strings and norb: one context taken through new
    integrals on its strings, other alpha strings, other beta strings of the same number, and
    another norb gives the bits of a context made for each."""
    first = workload_small(14, 4, 4, 60, 300, 83)
    steps = [first, dict(workload_small(14, 4, 4, 60, 300, 84), astr=first["astr"], bstr=first["bstr"])]
    steps.append(dict(steps[1], astr=workload_small(14, 4, 4, 55, 300, 85)["astr"]))
    steps.append(dict(steps[2], bstr=workload_small(14, 4, 4, 55, 300, 86)["bstr"]))
    steps.append(dict(workload_small(16, 4, 4, 55, 300, 87), astr=steps[3]["astr"], bstr=steps[3]["bstr"]))
    options = dict(max_it=1, max_nb=2, eps=1e10, init=1, seed=9, do_rdm=1)
    s = None
    for c in steps:
        fresh = sbdg.Solver(c["norb"], c["core"], c["h1"], c["eri"], c["astr"], c["bstr"], **options)
        if s is None:
            s = sbdg.Solver(c["norb"], c["core"], c["h1"], c["eri"], c["astr"], c["bstr"], **options)
        else:
            s.norb, s.astr, s.bstr, s.na, s.nb = c["norb"], c["astr"], c["bstr"], len(c["astr"]), len(c["bstr"])
            s.set_integrals(c["core"], c["h1"], c["eri"])
        for x in (s, fresh):
            x.run()
        got, want = (*s.rdm(), s.density()), (*fresh.rdm(), fresh.density())
        assert all(np.array_equal(x, y) for x, y in zip(got, want))
        assert abs(got[0][1].reshape(c["norb"], -1).trace() - 4) < 1e-11
        fresh.close()
    s.close()


@pytest.mark.parametrize("refresh_k", [3, 0])
@pytest.mark.parametrize("norb,nel,na,nb", [(16, 5, 65, 129), (18, 5, 300, 251)])
def test_rdm_out_of_a_mixed_solves_vectors(norb, nel, na, nb, refresh_k):
    """A mixed solve leaves its basis and the FP32 sigma vectors idle (no FP64 ones): the RDMs'
    buffers come out of those, the vector stays, repeats give the same bits, and the RDMs and
    gradients are those of an FP64 context that holds the vector (its norm is formed again there:
    a unit in the last place of every element, so 1e-12 instead of the same bits)."""
    c = workload_small(norb, nel, nel, na, nb, 97)
    args = c["norb"], c["core"], c["h1"], c["eri"], c["astr"], c["bstr"]
    s = sbdg.Solver(*args, max_it=20, max_nb=6, eps=1e-5, precision=1, refresh_k=refresh_k, do_rdm=1)
    s.run()
    assert s.stats()["sigma_fp32"] > 0
    w = s.vector()
    one, two = s.rdm()
    grad = s.rdm_backward(1.0)
    again = (*s.rdm(compute=True), *s.rdm_backward(1.0))
    assert all(np.array_equal(x, y) for x, y in zip((one, two, *grad), again))
    assert np.array_equal(s.vector(), w)
    r = sbdg.Solver(*args, max_it=1, max_nb=2, eps=1e10, init=2, do_rdm=1)
    r.set_vector(w)
    r.run()
    for x, y in zip((one, two, *grad, s.density()), (*r.rdm(), *r.rdm_backward(1.0), r.density())):
        assert np.abs(x - y).max() < 1e-12
    rdm_invariants(one, two, nel, nel, norb, 1e-11)
    s.close()
    r.close()


def test_rdm_after_the_doubles_option_changed():
    """Core tables of an earlier string set must not serve a later one that was built without:
    a context with cores of 1,287 strings, then 200 strings by excitation table, then the option
    set back before the RDMs of that solution are asked for."""
    big = workload_small(13, 5, 5, 0, 60, 101)
    small = workload_small(13, 5, 5, 200, 60, 102)
    options = dict(max_it=1, max_nb=2, eps=1e10, init=1, seed=9)
    s = sbdg.Solver(13, big["core"], big["h1"], big["eri"], big["astr"], big["bstr"], doubles=2, **options)
    s.run()
    s.astr, s.na = small["astr"], len(small["astr"])
    s.bstr, s.nb = small["bstr"], len(small["bstr"])
    s.set_options(doubles=1, **options)
    s.set_integrals(small["core"], small["h1"], small["eri"])
    s.run()
    s.set_options(doubles=0, **options)
    got = s.rdm(compute=True)
    fresh = sbdg.Solver(13, small["core"], small["h1"], small["eri"], small["astr"], small["bstr"], doubles=1, **options)
    fresh.run()
    want = fresh.rdm(compute=True)
    assert all(np.array_equal(x, y) for x, y in zip(got, want))
    s.close()
    fresh.close()
