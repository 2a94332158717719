"""The work a user of this library has it do, as measurable cases.

Five kinds of call, each through the public Python binding of the C-ABI:

* ``sigma``     H c on device-resident vectors (``Solver.sigma_device``), FP64 or FP32;
* ``davidson``  a fixed number of Davidson steps on a built problem (``Solver.run``), FP64 or
                mixed precision, energy and orbital occupations out;
* ``diag``      the whole of ``sbdg.diag``: context, tables, Davidson to convergence, RDMs;
* ``gradient``  ``ground_state_energy`` forward and backward (energy and its derivatives with
                respect to the integrals: tables, Davidson, RDMs, contraction);
* ``rdm``       the 1- and 2-RDMs of a vector the program holds (``Solver.rdm(compute=True)``).

Inputs are problems of the kind ``sbdg.synthetic`` makes: a symmetric one-electron matrix with
a rising diagonal, a positive semidefinite two-electron tensor with exact 8-fold symmetry
(here scaled so that the Hartree-Fock determinant has the lowest diagonal element and the
largest weight, as in a molecule near its equilibrium geometry), and either every string of a space or strings sampled around the Hartree-Fock one with the
excitation level k drawn in proportion to 0.5**k.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sbd-ykt_amd"))
import sbdg  # noqa: E402

DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
SIGMA64_MAX, SIGMA32_MAX = 8_388_608, 13_421_772  # determinants sigma_device takes


def _case(name, kind, norb, nalpha, nbeta, na, nb, **more):
    return dict(name=name, kind=kind, norb=norb, nalpha=nalpha, nbeta=nbeta, na=na, nb=nb, **more)


def listed():
    return [
        # the N2 6-31G dataset's shape at its loosest threshold: one short sigma, all latency
        _case("sigma_57k", "sigma", 18, 7, 7, 239, 239, fp32=False),
        # odd string counts at norb=26, near the most that sigma_device takes in FP64
        _case("sigma_7m_odd", "sigma", 26, 5, 5, 2801, 2749, fp32=False),
        # FP32 sigma (the mixed iteration's) at norb=36 with equal sets
        _case("sigma_12m_fp32", "sigma", 36, 9, 9, 3600, 3500, fp32=True),
        # a block of alpha rows of the largest workload (norb=58, 40,000 beta strings)
        _case("sigma_8m_wide", "sigma", 58, 12, 12, 200, 40000, fp32=False),
        # a small problem from strings to RDMs in one call (norb=12, 4+4, every string)
        _case("diag_245k_full", "diag", 12, 4, 4, 495, 495),
        # a geometry step: energy and gradient at the H2O cc-pVDZ dataset's shape
        _case("gradient_75k", "gradient", 24, 5, 5, 275, 275),
        # the reference's default solve (one block of 10) at norb=26, 4,000 x 4,000
        _case("davidson_16m", "davidson", 26, 5, 5, 4000, 4000, steps=10, mixed=False),
        # mixed precision, an exact sigma every 4 steps, at norb=36 with odd sets
        _case("mixed_25m_odd", "davidson", 36, 9, 9, 5001, 4999, steps=8, mixed=True),
        # the first steps of the headline workload (norb=36, 20,000 x 20,000) in FP64
        _case("davidson_400m", "davidson", 36, 9, 9, 20000, 20000, steps=3, mixed=False),
        # and in mixed precision with its first exact refresh
        _case("mixed_400m", "davidson", 36, 9, 9, 20000, 20000, steps=4, mixed=True),
        # RDMs of a full space (norb=16, 5+5: dense excitation lists)
        _case("rdm_19m_full", "rdm", 16, 5, 5, 4368, 4368),
        # RDMs over wide beta rows (norb=36)
        _case("rdm_80m_wide", "rdm", 36, 9, 9, 4000, 20000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sigma", "sigma", "sigma", "davidson", "davidson", "diag", "gradient", "rdm"])
    fp32 = kind == "sigma" and rng.random() < 0.4
    lo_l, hi_l, lo_n, hi_n, most = {
        "sigma": (12, 58, 2e4, SIGMA32_MAX if fp32 else SIGMA64_MAX, 40000),
        "davidson": (16, 40, 1e5, 1.2e8, 20000),
        "diag": (10, 26, 1e4, 1e6, 2000),
        "gradient": (10, 24, 1e4, 2e5, 1000),
        "rdm": (12, 36, 1e5, 6e7, 20000),
    }[kind]
    while True:
        norb = rng.randint(lo_l, hi_l)
        nalpha = rng.randint(3, min(12, norb // 2))
        nbeta = nalpha if rng.random() < 0.6 else rng.randint(3, min(12, norb // 2))
        n = math.exp(rng.uniform(math.log(lo_n), math.log(hi_n)))
        na = max(60, _log_int(rng, math.sqrt(n) / 5, math.sqrt(n) * 3))
        nb = int(n / na)
        if na <= most and 60 <= nb <= most and 2 * na <= math.comb(norb, nalpha) and 2 * nb <= math.comb(norb, nbeta):
            break
    c = _case("", kind, norb, nalpha, nbeta, na, nb)
    del c["name"]
    if kind == "sigma":
        c["fp32"] = fp32
    if kind == "davidson":
        c["steps"] = rng.randint(3, 10)
        c["mixed"] = rng.random() < 0.5
    return c


# ------------------------------------------------------------------ inputs

def _integrals(norb, rng):
    h = np.zeros((norb, norb))
    iu = np.triu_indices(norb, 1)
    h[iu] = rng.normal(0.0, 0.05, size=len(iu[0]))
    h = h + h.T
    h[np.diag_indices(norb)] = np.linspace(-4.0, 2.0, norb)
    iu = np.triu_indices(norb)
    b = rng.normal(0.0, 0.03, size=(2 * norb, len(iu[0])))
    m = b.T @ b
    m = np.tril(m) + np.tril(m, -1).T
    pair = np.zeros((norb, norb), dtype=np.int64)
    pair[iu] = pair[iu[::-1]] = np.arange(len(iu[0]))
    pair = pair.reshape(-1)
    return h, np.ascontiguousarray(m[pair][:, pair].reshape((norb,) * 4))


def _strings(norb, nel, count, rng):
    if count == math.comb(norb, nel):
        return _full_space(norb, nel)
    levels = np.arange(1, min(nel, norb - nel) + 1)
    p = 0.5 ** levels
    one = np.uint64(1)
    hf = np.uint64((1 << nel) - 1)
    got = np.array([hf], dtype=np.uint64)
    while len(got) < count:
        m = 2 * count + 1000
        k = rng.choice(levels, size=m, p=p / p.sum())[:, None]
        holes = np.argsort(rng.random((m, nel)), axis=1)[:, : levels[-1]].astype(np.uint64)
        parts = (np.argsort(rng.random((m, norb - nel)), axis=1)[:, : levels[-1]] + nel).astype(np.uint64)
        use = levels[None, :] <= k
        s = (hf - np.where(use, one << holes, 0).sum(axis=1, dtype=np.uint64)) \
            + np.where(use, one << parts, 0).sum(axis=1, dtype=np.uint64)
        got = np.concatenate([got, s])
        got = got[np.sort(np.unique(got, return_index=True)[1])]
    return np.sort(got[:count])


def _full_space(norb, nel):
    """Every string of nel electrons in norb orbitals, ascending."""
    s = np.array([0], dtype=np.uint64)
    for o in range(norb):
        s = np.concatenate([s, s | np.uint64(1 << o)])
        s = s[np.bitwise_count(s) <= nel]
    return np.sort(s[np.bitwise_count(s) == nel])


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    h, eri = _integrals(case["norb"], rng)
    a = _strings(case["norb"], case["nalpha"], case["na"], rng)
    b = _strings(case["norb"], case["nbeta"], case["nb"], rng)
    return h, eri, a, b


def _vector(case, a, b, seed):
    """A correlated vector's look: random signs and sizes that fall with the excitation level
    from the Hartree-Fock determinant; unit norm, on the GPU."""
    g = torch.Generator(device=DEVICE).manual_seed(int(seed))
    v = torch.randn(case["na"], case["nb"], dtype=torch.float64, device=DEVICE, generator=g)
    for s, nel, axis in ((a, case["nalpha"], 0), (b, case["nbeta"], 1)):
        level = np.bitwise_count(s >> np.uint64(nel)).astype(np.float64)
        w = torch.from_numpy(0.5 ** level).to(DEVICE)
        v *= w[:, None] if axis == 0 else w[None, :]
    return v.div_(v.norm()).reshape(-1)


def _solver(case, h, eri, a, b, **options):
    return sbdg.Solver(case["norb"], 0.0, h, eri, a, b, **options)


CONVERGE = dict(max_it=40, max_nb=10, restart_keep=2, eps=1e-9)


def prepare(case, seed):
    h, eri, a, b = _inputs(case, seed)
    kind = case["kind"]
    st = {"case": case, "h": h, "eri": eri, "a": a, "b": b}
    if kind == "sigma":
        st["solver"] = _solver(case, h, eri, a, b)
        st["solver"].build()
        st["x"] = _vector(case, a, b, seed)
        st["y"] = torch.zeros_like(st["x"])
    elif kind == "davidson":
        st["solver"] = _solver(case, h, eri, a, b, max_it=1, max_nb=case["steps"], eps=1e-12,
                               precision=1 if case["mixed"] else 0, refresh_k=4)
        st["solver"].build()
    elif kind == "gradient":
        st["solver"] = _solver(case, h, eri, a, b, **CONVERGE)
        st["h"] = torch.from_numpy(h)
        st["eri"] = torch.from_numpy(eri)
    elif kind == "rdm":
        # a wavefunction of an earlier run, taken as the solution (the tolerance stops at once)
        s = _solver(case, h, eri, a, b, max_it=1, max_nb=2, eps=1e10, init=2)
        s.set_vector(_vector(case, a, b, seed).cpu().numpy())
        s.run()
        st["solver"] = s
    return st


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "sigma":
        state["solver"].sigma_device(state["x"].data_ptr(), state["y"].data_ptr(), int(case["fp32"]))
        # an FP32 product is kept in FP32, as a mixed iteration keeps it
        return state["y"].float() if case["fp32"] else state["y"]
    if kind == "davidson":
        energy = state["solver"].run()
        density = state["solver"].density()
        # FP32 sigmas shape the mixed iteration's vector: its occupations are FP32 numbers
        return {"energy": energy, "density": density.astype(np.float32) if case["mixed"] else density}
    if kind == "diag":
        r = sbdg.diag(case["norb"], 0.0, state["h"], state["eri"], state["a"], state["b"], do_rdm=1, **CONVERGE)
        return {"energy": r.energy, "density": r.density, "one": r.one_p_rdm, "two": r.two_p_rdm}
    if kind == "gradient":
        h = state["h"].clone().requires_grad_()
        eri = state["eri"].clone().requires_grad_()
        energy = sbdg.ground_state_energy(h, eri, state["solver"])
        energy.backward()
        return {"energy": energy.detach(), "dh": h.grad, "deri": eri.grad}
    one, two = state["solver"].rdm(compute=True)
    return {"one": one, "two": two}


# ------------------------------------------------------------------ the work of one pass

def _pairs(s):
    """Estimated (singles, doubles) table entries of a string set, from a sample of its rows."""
    rows = s[:: max(1, len(s) // 200)]
    d = np.bitwise_count(rows[:, None] ^ s[None, :])
    f = len(s) / len(rows)
    return float((d == 2).sum()) * f, float((d == 4).sum()) * f


def work(case):
    _, _, a, b = _inputs(dict(case, norb=case["norb"]), 1)
    na, nb, n = len(a), len(b), float(len(a) * len(b))
    (sa, da), (sb, db) = _pairs(a), _pairs(b)
    l4 = float(case["norb"]) ** 4
    sigma = {"bytes": 16 * n + 8 * l4, "flops": 2 * (n + (sa + da) * nb + (sb + db) * na + sa * sb)}
    rdm = {"bytes": 8 * n + 32 * l4, "flops": 2 * (2 * n + (sa + da) * nb + (sb + db) * na + sa * sb) / 2}
    kind = case["kind"]
    if kind == "sigma":
        return sigma
    if kind == "rdm":
        return rdm
    # Davidson steps: a sigma each and one for the final energy; a converged solve takes about 30
    steps = case["steps"] + 1 if kind == "davidson" else 30
    w = {k: steps * sigma[k] for k in sigma}
    return w if kind == "davidson" else {k: w[k] + rdm[k] for k in w}


# ------------------------------------------------------------------ the same in plain 64-bit torch

class _Space:
    """One spin's strings: the pairs (bra, ket) one and two excitations apart, with the signs
    of the strings' own creator order."""

    def __init__(self, strings, norb, device):
        self.n, self.norb = len(strings), norb
        self.s = torch.from_numpy(strings.astype(np.int64)).to(device)
        self.occ = ((self.s[:, None] >> torch.arange(norb, device=device)) & 1).bool()
        self.below = torch.zeros(self.n, norb + 1, dtype=torch.int64, device=device)
        self.below[:, 1:] = self.occ.long().cumsum(1)
        of = self.occ.float()
        nel = int(self.occ[0].sum())
        bra, ket, level = [], [], []
        step = max(1, (1 << 27) // max(1, self.n))
        for r in range(0, self.n, step):
            diff = nel - (of[r:r + step] @ of.T).round().int()
            i, j = torch.nonzero((diff == 1) | (diff == 2), as_tuple=True)
            bra.append(i + r)
            ket.append(j)
            level.append(diff[i, j])
        bra, ket, level = torch.cat(bra), torch.cat(ket), torch.cat(level)
        one = level == 1
        self.bra1, self.ket1 = bra[one], ket[one]
        self.a, self.i = self._top(self.s[self.bra1] & ~self.s[self.ket1]), self._top(self.s[self.ket1] & ~self.s[self.bra1])
        self.sign1 = self._sign(self.ket1, self.i, self.a)
        self.bra2, self.ket2 = bra[~one], ket[~one]
        up, dn = self.s[self.bra2] & ~self.s[self.ket2], self.s[self.ket2] & ~self.s[self.bra2]
        self.B, self.J = self._top(up), self._top(dn)
        self.A, self.I = self._top(up ^ (1 << self.B)), self._top(dn ^ (1 << self.J))
        # a+_A a_I a+_B a_J on the ket: J -> B first, then I -> A on what that leaves
        lo, hi = torch.minimum(self.I, self.A), torch.maximum(self.I, self.A)
        moved = ((self.J > lo) & (self.J < hi)).long() + ((self.B > lo) & (self.B < hi)).long()
        self.sign2 = self._sign(self.ket2, self.J, self.B) * self._sign(self.ket2, self.I, self.A) * (1 - 2 * (moved & 1))
        # E_pq entries, the number operators among them
        r, p = torch.nonzero(self.occ, as_tuple=True)
        self.ebra, self.eket = torch.cat([self.bra1, r]), torch.cat([self.ket1, r])
        self.epq = torch.cat([self.a * norb + self.i, p * norb + p])
        self.esign = torch.cat([self.sign1, torch.ones_like(p)]).double()

    @staticmethod
    def _top(x):
        return torch.frexp(x.double())[1].long() - 1  # highest set bit

    def _sign(self, ket, i, a):
        lo, hi = torch.minimum(i, a), torch.maximum(i, a)
        between = self.below[ket, hi] - self.below[ket, lo + 1]
        return (1 - 2 * (between & 1)).double()

    def matrix(self, h, eri):
        """The same-spin Hamiltonian among the strings (dense)."""
        n, occ = self.n, self.occ.double()
        coul = torch.einsum("ppqq->pq", eri) - torch.einsum("pqqp->pq", eri)
        m = torch.zeros(n, n, dtype=torch.float64, device=h.device)
        m.diagonal().copy_(occ @ h.diagonal() + 0.5 * ((occ @ coul) * occ).sum(1))
        mean = torch.einsum("aikk->aik", eri) - torch.einsum("akki->aik", eri)  # k = i cancels
        step = 1 << 20
        for q in range(0, len(self.bra1), step):
            t = slice(q, q + step)
            a, i = self.a[t], self.i[t]
            v = h[a, i] + (mean[a, i] * occ[self.ket1[t]]).sum(1)
            m[self.bra1[t], self.ket1[t]] = self.sign1[t] * v
        for q in range(0, len(self.bra2), step):
            t = slice(q, q + step)
            A, B, i, j = self.A[t], self.B[t], self.I[t], self.J[t]
            m[self.bra2[t], self.ket2[t]] = self.sign2[t] * (eri[A, i, B, j] - eri[A, j, B, i])
        return m


class _Exact:
    def __init__(self, norb, h, eri, a, b):
        self.norb = norb
        self.h, self.eri = torch.from_numpy(h).to(DEVICE), torch.from_numpy(eri).to(DEVICE)
        self.A, self.B = _Space(a, norb, DEVICE), _Space(b, norb, DEVICE)
        self.Ha, self.Hb = self.A.matrix(self.h, self.eri), self.B.matrix(self.h, self.eri)
        # creators interleaved by orbital (alpha first) against all alpha, then all beta
        par = (self.A.occ.double() @ self.B.below[:, :norb].double().T).long() & 1
        self.phase = (1 - 2 * par).double()
        order = torch.argsort(self.A.epq, stable=True)
        self.groups = []
        pq, cnt = torch.unique_consecutive(self.A.epq[order], return_counts=True)
        end = 0
        for p, k in zip(pq.tolist(), cnt.tolist()):
            self.groups.append((p, order[end:end + k]))
            end += k
        self.chunk = max(1, (1 << 27) // max(1, len(self.B.epq)))

    def _alpha_groups(self):
        for p, idx in self.groups:
            for q in range(0, len(idx), self.chunk):
                e = idx[q:q + self.chunk]
                yield p, self.A.ebra[e], self.A.eket[e], self.A.esign[e]

    def separated(self, c):
        B = self.B
        y = self.Ha @ c + c @ self.Hb
        L2 = self.norb ** 2
        eri = self.eri.reshape(L2, L2)
        for p, bra, ket, sign in self._alpha_groups():
            t = c[ket][:, B.eket] * (eri[p, B.epq] * B.esign)
            o = torch.zeros(len(bra), B.n, dtype=torch.float64, device=DEVICE).index_add_(1, B.ebra, t)
            y.index_add_(0, bra, o * sign[:, None])
        return y

    def ground_state(self):
        """Davidson to a residual of 1e-11, from the first determinant."""
        L2 = self.norb ** 2
        coul = torch.einsum("ppqq->pq", self.eri)
        diag = self.Ha.diagonal()[:, None] + self.Hb.diagonal()[None, :] \
            + self.A.occ.double() @ coul @ self.B.occ.double().T
        v = torch.zeros_like(diag)
        v[0, 0] = 1.0
        V, S = [v], [self.separated(v)]
        for _ in range(300):
            T = torch.stack([x.reshape(-1) for x in V])
            Y = torch.stack([x.reshape(-1) for x in S])
            m = T @ Y.T
            e, u = torch.linalg.eigh((m + m.T).cpu() / 2)
            u = u.to(DEVICE)
            w, hw = (u[:, 0] @ T).reshape_as(v), (u[:, 0] @ Y).reshape_as(v)
            r = hw - e[0].item() * w
            if float(r.norm()) < 1e-11:
                break
            if len(V) >= 16:
                V = [x.reshape_as(v) for x in u[:, :4].T @ T]
                S = [x.reshape_as(v) for x in u[:, :4].T @ Y]
            d = e[0].item() - diag
            t = r / torch.where(d.abs() > 1e-8, d, torch.full_like(d, 1e-8))
            for _ in range(2):
                for x in V:
                    t = t - (x * t).sum() * x
            V.append(t / t.norm())
            S.append(self.separated(V[-1]))
        return float((w * hw).sum() / (w * w).sum()), w / w.norm()

    def rdms(self, w):
        """one (2, L^2) and two (4, L^4) in the library's layout, from separated phases."""
        L = self.norb
        one = torch.zeros(2, L, L, dtype=torch.float64, device=DEVICE)       # [s][j][i]
        two = torch.zeros(4, L, L, L, L, dtype=torch.float64, device=DEVICE)  # [block][l][k][j][i]
        for s, sp, x in ((0, self.A, w), (1, self.B, w.T)):
            gram = x @ x.T
            one[s].view(-1).index_add_(0, (sp.epq % L) * L + sp.epq // L, sp.esign * gram[sp.ebra, sp.eket])
            blk = two[3 * s].view(-1)

            def put(i, j, k, l, v):
                blk.index_add_(0, i + L * j + L * L * k + L ** 3 * l, v)

            v = sp.sign2 * gram[sp.bra2, sp.ket2]
            put(sp.A, sp.B, sp.I, sp.J, v)
            put(sp.B, sp.A, sp.J, sp.I, v)
            put(sp.A, sp.B, sp.J, sp.I, -v)
            put(sp.B, sp.A, sp.I, sp.J, -v)
            v1 = sp.sign1 * gram[sp.bra1, sp.ket1]
            for k in range(L):
                on = (sp.occ[sp.ket1, k] & sp.occ[sp.bra1, k])
                a, i, v = sp.a[on], sp.i[on], v1[on]
                kk = torch.full_like(a, k)
                put(a, kk, i, kk, v)
                put(kk, a, kk, i, v)
                put(a, kk, kk, i, -v)
                put(kk, a, i, kk, -v)
            occ = sp.occ.double()
            nn = occ.T @ (gram.diagonal()[:, None] * occ)
            i, j = torch.nonzero(~torch.eye(L, dtype=torch.bool, device=DEVICE), as_tuple=True)
            put(i, j, i, j, nn[i, j])
            put(i, j, j, i, -nn[i, j])
        B = self.B
        T = torch.zeros(L * L, L * L, dtype=torch.float64, device=DEVICE)  # <E_ik(alpha) E_jl(beta)>
        for p, bra, ket, sign in self._alpha_groups():
            t = ((w[bra] * sign[:, None])[:, B.ebra] * w[ket][:, B.eket]).sum(0) * B.esign
            T[p].index_add_(0, B.epq, t)
        T = T.reshape(L, L, L, L)  # [i][k][j][l]
        two[2] = T.permute(3, 1, 2, 0)
        two[1] = T.permute(1, 3, 0, 2)
        return one.reshape(2, -1), two.reshape(4, -1)


def exact(case, seed):
    kind = case["kind"]
    big = case["na"] * case["nb"]
    if kind == "davidson" or (kind == "rdm" and big > 3e7):
        return None  # the state of an unfinished iteration; too long in plain torch
    h, eri, a, b = _inputs(case, seed)
    X = _Exact(case["norb"], h, eri, a, b)
    if kind == "sigma":
        x = _vector(case, a, b, seed).reshape(len(a), len(b))
        return (X.separated(x * X.phase) * X.phase).reshape(-1)
    if kind == "rdm":
        one, two = X.rdms(_vector(case, a, b, seed).reshape(len(a), len(b)) * X.phase)
        return {"one": one, "two": two}
    energy, w = X.ground_state()
    one, two = X.rdms(w)
    L = case["norb"]
    if kind == "gradient":
        G = two.sum(0).reshape(L, L, L, L)  # [s][q][r][p]
        return {"energy": torch.tensor(energy, dtype=torch.float64), "dh": (one[0] + one[1]).reshape(L, L).T, "deri": 0.5 * G.permute(3, 1, 2, 0)}
    density = torch.stack([one[0].reshape(L, L).diagonal(), one[1].reshape(L, L).diagonal()], 1).reshape(-1)
    return {"energy": energy, "density": density, "one": one, "two": two}
