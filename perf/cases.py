"""The work that users of sbdx have it do, as measurable cases.

Every case is one call (or the few calls) of the public interface that a
program makes in the middle of a selected-CI calculation: a Hamiltonian
product, a ground-state solve, several roots at once, the reduced density
matrices, the operator build of a new string set.  The integrals are those
of a molecule-like system (ascending orbital energies, a closed-shell or
open-shell determinant that dominates the ground state); a seed changes the
"geometry" a little and picks other excitations into the string sets.  The
string sets are the Hartree-Fock string, its singles and a subset of its
doubles, as a selected-CI step produces them.

`exact` evaluates the same quantities in float64 from the definitions with
plain torch: string occupations, Slater-Condon rules, a dense (pq|rs)
contraction.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "sbd-pub_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import sbdx  # noqa: E402
from sbdx import instances  # noqa: E402

# Solves go to a residual at which the vector is good to about 1e-10 or
# better, as properties of the state need it.
EPS = 4e-12


def listed():
    return [
        # a minimal active space: one product is a handful of launches
        dict(name="sigma_3k", op="sigma", norb=10, ea=3, na=60, eb=3, nb=60),
        # open shell, different and ragged string sets, the usual size of an
        # active-space calculation: a user's own eigensolver calls the product
        dict(name="sigma_open_2m", op="sigma", norb=24, ea=5, na=1543, eb=4, nb=1387),
        # the 64M-determinant problem that the benchmark is quoted on
        dict(name="sigma_64m", op="sigma", norb=36, ea=8, na=8000, eb=8, nb=8000),
        # the largest product: more strings and more orbitals than that
        dict(name="sigma_121m", op="sigma", norb=40, ea=8, na=11003, eb=8, nb=11003),
        # ground state of a small open-shell problem with the default solver
        # (FP64, restart from the Ritz vector alone)
        dict(name="solve_plain_66k", op="solve", norb=16, ea=5, na=275, eb=4, nb=239, solver="plain"),
        # ground state in mixed precision with spin-flip sectors, small ...
        dict(name="solve_mixed_250k", op="solve", norb=16, ea=5, na=500, eb=5, nb=500, solver="lowest"),
        # ... and large, with a coarse start, as the benchmark runs it
        dict(name="solve_mixed_16m", op="solve", norb=36, ea=8, na=4001, eb=8, nb=4001, solver="lowest"),
        # the lowest states together by the block solver
        dict(name="roots_block_1m", op="roots", norb=24, ea=5, na=1001, eb=5, nb=1001, roots=3, block=4),
        # density matrices of a solution: small closed shell, ragged open
        # shell, and the benchmark's size
        dict(name="rdm_250k", op="rdm", norb=16, ea=5, na=500, eb=5, nb=500),
        dict(name="rdm_open_4m", op="rdm", norb=29, ea=6, na=2583, eb=5, nb=1387),
        dict(name="rdm_64m", op="rdm", norb=36, ea=8, na=8000, eb=8, nb=8000),
        # a new string set: excitation tables and the diagonal
        dict(name="build_7m", op="build", norb=29, ea=7, na=2583, eb=7, nb=2583),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["sigma", "sigma", "sigma", "solve", "solve", "roots", "rdm", "rdm", "build"])
    # strings: small active spaces to the largest listed sets, by operation
    top = {"sigma": 9000, "solve": 3500, "roots": 1200, "rdm": 7000, "build": 4000}[op]
    na = _log_int(rng, 60, top)
    # orbitals: enough singles and doubles for the set, up to 40
    lo = 10 if na <= 120 else 16 if na <= 550 else 24 if na <= 1500 else 29 if na <= 3000 else 36
    norb = rng.randint(lo, min(40, lo + 6))
    ea = 3 if lo == 10 else 5 if lo <= 24 else rng.choice([6, 7]) if lo == 29 else 8
    case = dict(op=op, norb=norb, ea=ea, na=na, eb=ea, nb=na)
    if op == "roots":
        case.update(roots=rng.choice([2, 3]), block=4)
        return case
    if op == "solve":
        case.update(solver=rng.choice(["plain", "lowest"]))
    # open shell: other beta strings (the smallest orbital spaces hold too few of them)
    closed = lo == 10 or op == "solve" and case["solver"] == "lowest"
    if not closed and rng.random() < 0.5:
        case.update(eb=ea - 1, nb=max(40, int(na * rng.uniform(0.5, 1.0))))
    return case


# ---------------------------------------------------------------- inputs
def _integrals(norb, n, seed):
    """h and (pq|rs) of a molecule-like system: a base system per (norb, n)
    and a small displacement of it per seed."""
    base, move = np.random.default_rng([norb, n]), np.random.default_rng([seed, 7])
    nv = max(1, norb - n)
    off = 0.06 * math.sqrt(55.0 / (n * nv))

    def pair(rng, scale):
        Lk = rng.normal(0.0, off * scale, size=(40, norb, norb))
        Lk = np.triu(Lk, 1)
        Lk = Lk + np.transpose(Lk, (0, 2, 1))
        i = np.arange(norb)
        Lk[:, i, i] = rng.normal(0.0, 0.08 * scale, size=(40, norb)) + (0.09 if scale == 1.0 else 0.0)
        hh = np.triu(rng.normal(0.0, 0.01 * scale, size=(norb, norb)), 1)
        return Lk, hh + hh.T

    L0, h0 = pair(base, 1.0)
    L1, h1 = pair(move, 0.02)
    Lf = (L0 + L1).reshape(40, norb * norb)
    eri = (Lf.T @ Lf).reshape(norb, norb, norb, norb)
    h = h0 + h1
    # orbital energies -3 .. on the occupied, a gap, then the virtuals; h is
    # what remains once the Hartree-Fock string's mean field is taken off
    i = np.arange(norb)
    e = np.where(i < n, -0.5 - 0.22 * (n - 1 - i), 0.35 + 0.11 * (i - n)) + 0.02 * base.normal(size=norb)
    mean = 2.0 * np.einsum("pqkk->pq", eri[:, :, :n, :n]) - np.einsum("pkkq->pq", eri[:, :n, :n, :])
    h = h + np.diag(e) - mean
    return 0.5 * (h + h.T), eri


def _strings(case, seed):
    a = instances.make_strings(case["norb"], case["ea"], case["na"], 100 + seed)
    if case["eb"] == case["ea"] and case["nb"] == case["na"]:
        return a, a.copy()
    return a, instances.make_strings(case["norb"], case["eb"], case["nb"], 500000 + seed)


def _problem(case, seed):
    h, eri = _integrals(case["norb"], case["ea"], seed)
    a, b = _strings(case, seed)
    return h, eri, a, b


def _vector(na, nb, seed):
    """A normalized CI vector on the GPU: magnitudes over several decades,
    the leading determinants the largest."""
    g = torch.Generator(device="cuda").manual_seed(1 + seed)
    x = torch.randn(na * nb, dtype=torch.float64, device="cuda", generator=g)
    x *= torch.exp(-6.0 * torch.rand(na * nb, dtype=torch.float64, device="cuda", generator=g))
    x[0] = 3.0 * math.sqrt(float(x.square().sum()))
    return x / x.norm()


def _operator(case, seed):
    h, eri, a, b = _problem(case, seed)
    I0, I1, I2 = instances.pack_integrals(case["norb"], h, eri)
    return sbdx.TPBOperator(case["norb"], I0, I1, I2, a, b)


def prepare(case, seed):
    op = case["op"]
    if op == "build":  # a new string set of a known molecule: integrals and strings are in host memory
        h, eri, a, b = _problem(case, seed)
        return dict(op=op, args=(case["norb"], *instances.pack_integrals(case["norb"], h, eri), a, b))
    H = _operator(case, seed)
    s = dict(op=op, H=H)
    if op == "sigma":  # the caller's eigensolver keeps its vectors on the GPU
        s["x"] = _vector(H.na, H.nb, seed)
        s["y"] = torch.empty_like(s["x"])
        torch.cuda.synchronize()
    elif op == "rdm":  # a solution in host memory, as the solves return it
        s["W"] = _vector(H.na, H.nb, seed).cpu().numpy()
    elif op == "solve":
        s["nb"], s["it"] = 12, 100
        if case["solver"] == "lowest":
            H.set_precision(sbdx.PREC_MIXED)
            H.set_restart(3)
            H.set_symmetry("lowest")
            H.set_coarse_start(1000 if case["na"] > 2000 else 0, 1e-2)
            s["nb"] = 16
    elif op == "roots":
        H.configure("block")
        H.set_symmetry("lowest")
        s["roots"], s["block"] = case["roots"], case["block"]
    return s


# ---------------------------------------------------------------- the passes
def _phased(W, nb):
    """A state is defined up to its sign: the largest coefficient of the
    first alpha string's row is made positive."""
    k = int(np.argmax(np.abs(W[:nb])))
    if W[k] < 0.0:
        torch.from_numpy(W).neg_()
    return W


def run(state):
    op = state["op"]
    if op == "build":
        H = sbdx.TPBOperator(*state["args"])
        hii = H.make_diag()
        H.close()
        return hii
    H = state["H"]
    if op == "sigma":
        L = sbdx.lib()
        if L.sbdx_sigma_device(H.h, state["x"].data_ptr(), state["y"].data_ptr(), 0) != 0:
            raise RuntimeError(L.sbdx_last_error().decode())
        return state["y"]
    if op == "rdm":
        one, two = H.correlation(state["W"])
        return dict(one=one, two=two)
    if op == "solve":
        E, W, _, ok = sbdx.davidson(H, max_it=state["it"], nb=state["nb"], eps=EPS)
        if not ok:
            raise RuntimeError("the solve did not converge")
        return dict(E=E, W=_phased(W, H.nb))
    E, W, _, ok = H.davidson_block(state["roots"], state["block"], max_it=400, eps=EPS)
    if not ok:
        raise RuntimeError("the block solve did not converge")
    return dict(E=E, W=np.stack([_phased(w, H.nb) for w in W]))


# ---------------------------------------------------------------- work
_counts = {}


def _pair_counts(norb, n, nstr, seed=100):
    """Ordered single and double pairs within one string set."""
    key = (norb, n, nstr, seed)
    if key not in _counts:
        O = _occ(instances.make_strings(norb, n, nstr, seed), norb, torch.float32, "cpu")
        s = d = 0
        for i in range(0, nstr, 1024):
            c = O[i:i + 1024] @ O.T
            s += int((c == n - 1).sum())
            d += int((c == n - 2).sum())
        _counts[key] = (s, d)
    return _counts[key]


def work(case):
    """Bytes: vectors, tables' strings and integrals once in and once out.
    Flops: a multiply-add for every matrix element that is not zero."""
    na, nb, L = case["na"], case["nb"], case["norb"]
    N = float(na) * nb
    sa, da = _pair_counts(L, case["ea"], na)
    sb, db = _pair_counts(L, case["eb"], nb, 100 if (case["eb"], nb) == (case["ea"], na) else 500000)
    product = 2.0 * (float(sa) * sb + (sa + da) * float(nb) + (sb + db) * float(na) + N)
    inp = 8.0 * (na + nb + float(L) ** 4 / 8)
    op = case["op"]
    if op == "sigma":
        return {"bytes": 16.0 * N + inp, "flops": product}
    if op == "rdm":
        return {"bytes": 8.0 * N + inp + 8.0 * (2 * L * L + 4.0 * L ** 4), "flops": product}
    if op == "build":
        return {"bytes": 8.0 * N + inp, "flops": 2.0 * N}
    # a solve: some ten corrections per state at the least, each a product
    # and the update and orthogonalization of a vector
    k = 10 * case.get("roots", 1)
    return {"bytes": k * 32.0 * N + inp, "flops": k * product}


# ---------------------------------------------------------------- float64 reference
def _occ(strs, norb, dtype, dev):
    s = torch.from_numpy(np.asarray(strs).astype(np.int64)).to(dev)
    return ((s[:, None] >> torch.arange(norb, device=dev)) & 1).to(dtype)


def _parity(k):
    return 1.0 - 2.0 * (k.to(torch.int64) & 1).to(torch.float64)


class _Spin:
    """Excitations within one string set, from its occupations."""

    def __init__(self, strs, norb, h, eri, dev):
        self.O = O = _occ(strs, norb, torch.float64, dev)
        self.n, self.ne, self.L = O.shape[0], int(O[0].sum()), norb
        self.cum = torch.cumsum(O, 1) - O  # occupied orbitals below each one
        self.h, self.eri = h, eri
        I1, J1, I2, J2 = [], [], [], []
        for i in range(0, self.n, 2048):
            c = O[i:i + 2048] @ O.T
            for want, I, J in ((self.ne - 1, I1, J1), (self.ne - 2, I2, J2)):
                a, b = torch.nonzero(c == want, as_tuple=True)
                I.append(a + i)
                J.append(b)
        self._singles(torch.cat(I1), torch.cat(J1))
        self.dI, self.dJ = torch.cat(I2), torch.cat(J2)

    def _singles(self, I, J):
        self.I, self.J = I, J
        self.p = torch.empty_like(I)
        self.q = torch.empty_like(I)
        self.s = torch.empty(I.numel(), dtype=torch.float64, device=I.device)
        for a in range(0, I.numel(), 1 << 20):
            z = slice(a, a + (1 << 20))
            OI, OJ = self.O[I[z]], self.O[J[z]]
            p, q = (OI * (1 - OJ)).argmax(1), (OJ * (1 - OI)).argmax(1)
            lo, hi = torch.minimum(p, q), torch.maximum(p, q)
            between = (torch.gather(self.cum[J[z]], 1, hi[:, None]) - torch.gather(self.cum[J[z]], 1, lo[:, None])
                       - torch.gather(OJ, 1, lo[:, None]))[:, 0]
            self.p[z], self.q[z], self.s[z] = p, q, _parity(between)

    def doubles(self):
        """Chunks (I, J, p1, p2, q1, q2, sign) of the double excitations
        |I> = sign a+_p1 a+_p2 a_q2 a_q1 |J>, p1 < p2, q1 < q2."""
        for a in range(0, self.dI.numel(), 1 << 20):
            I, J = self.dI[a:a + (1 << 20)], self.dJ[a:a + (1 << 20)]
            OI, OJ = self.O[I], self.O[J]
            C = OI * OJ
            p = torch.topk((OI - C) * torch.arange(1, self.L + 1, device=I.device), 2, 1).indices
            q = torch.topk((OJ - C) * torch.arange(1, self.L + 1, device=I.device), 2, 1).indices
            p2, p1, q2, q1 = p[:, 0], p[:, 1], q[:, 0], q[:, 1]
            cJ, cC = self.cum[J], torch.cumsum(C, 1) - C
            at = lambda m, k: torch.gather(m, 1, k[:, None])[:, 0]  # noqa: E731
            yield I, J, p1, p2, q1, q2, _parity(at(cJ, q1) + at(cJ, q2) - 1 + at(cC, p2) + at(cC, p1))

    def block(self):
        """The same-spin part of H between the strings, dense."""
        h, eri, O = self.h, self.eri, self.O
        J = torch.einsum("ppqq->pq", eri)
        X = torch.einsum("pqqp->pq", eri)
        H = torch.diag(O @ torch.diagonal(h) + 0.5 * ((O @ (J - X)) * O).sum(1))
        F = torch.einsum("pqkk->pqk", eri) - torch.einsum("pkkq->pqk", eri)
        for a in range(0, self.I.numel(), 1 << 20):
            z = slice(a, a + (1 << 20))
            I, p, q = self.I[z], self.p[z], self.q[z]
            H[I, self.J[z]] = self.s[z] * (h[p, q] + (F[p, q] * O[I]).sum(1))
        for I, K, p1, p2, q1, q2, s in self.doubles():
            H[I, K] = s * (eri[p1, q1, p2, q2] - eri[p1, q2, p2, q1])
        return H

    def extended(self):
        """Singles and the occupation numbers: (I, J, p, q, sign)."""
        i, k = torch.nonzero(self.O, as_tuple=True)
        return (torch.cat([self.I, i]), torch.cat([self.J, i]), torch.cat([self.p, k]), torch.cat([self.q, k]),
                torch.cat([self.s, torch.ones(i.numel(), dtype=torch.float64, device=i.device)]))


class _Reference:
    """The problem of a case in plain torch."""

    def __init__(self, case, seed):
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        h, eri, a, b = _problem(case, seed)
        self.h, self.eri = (torch.from_numpy(v).to(self.dev) for v in (h, eri))
        self.L = case["norb"]
        self.A = _Spin(a, self.L, self.h, self.eri, self.dev)
        self.B = self.A if a.size == b.size and bool((a == b).all()) else _Spin(b, self.L, self.h, self.eri, self.dev)
        # the interleaved order of spin orbitals against alpha before beta:
        # a sign for each beta orbital below an occupied alpha orbital
        self.S = _parity(torch.round(self.A.O @ self.B.cum.T))
        self.Ha = self.A.block()
        self.Hb = self.Ha if self.B is self.A else self.B.block()

    def diagonal(self):
        J = torch.einsum("ppqq->pq", self.eri)
        return (torch.diagonal(self.Ha)[:, None] + torch.diagonal(self.Hb)[None, :] + self.A.O @ J @ self.B.O.T)

    def sigma(self, x):
        L, dev = self.L, self.dev
        na, nb = self.A.n, self.B.n
        X = self.S * x.reshape(na, nb)
        Y = self.Ha @ X + X @ self.Hb.T
        tri = lambda p, q: torch.maximum(p, q) * (torch.maximum(p, q) + 1) // 2 + torch.minimum(p, q)  # noqa: E731
        hi, lo = torch.tril_indices(L, L, device=dev)
        V = self.eri[hi, lo][:, hi, lo]
        Kt = V.shape[0]
        aI, aJ, ap, aq, as_ = self.A.extended()
        r, j, p, q, s = self.B.extended()
        order = torch.argsort(r, stable=True)
        r, j, t, s = r[order], j[order], tri(p, q)[order], s[order]
        start = torch.searchsorted(r, torch.arange(nb + 1, device=dev)).tolist()
        ta = tri(ap, aq)
        B = max(1, min(nb, int(2e9 // (8 * Kt * na))))
        XT = X.T.contiguous()
        for r0 in range(0, nb, B):
            w = min(B, nb - r0)
            z = slice(start[r0], start[r0 + w])
            D = torch.zeros(Kt, w, na, dtype=torch.float64, device=dev)
            D[t[z], r[z] - r0] = s[z, None] * XT[j[z]]
            G = (V @ D.view(Kt, -1)).view(Kt, w, na).transpose(1, 2).contiguous()
            part = torch.zeros(na, w, dtype=torch.float64, device=dev)
            step = max(1, int(1e9 // (8 * w)))
            for a in range(0, aI.numel(), step):
                e = slice(a, a + step)
                part.index_add_(0, aI[e], as_[e, None] * G[ta[e], aJ[e]])
            Y[:, r0:r0 + w] += part
        return (self.S * Y).reshape(-1)

    def rdm(self, x):
        L, dev = self.L, self.dev
        X = self.S * x.reshape(self.A.n, self.B.n)
        one = torch.zeros(2, L * L, dtype=torch.float64, device=dev)
        two = torch.zeros(4, L ** 4, dtype=torch.float64, device=dev)

        def add(block, a, b, i, j, v):
            two[block].index_add_(0, a + L * b + L * L * i + L ** 3 * j, v)

        for spin, (T, w) in enumerate(((self.A, X), (self.B, X.T.contiguous()))):
            G, bs = w @ w.T, 3 * spin
            rho = torch.diagonal(G).contiguous()
            one[spin].index_add_(0, torch.arange(L, device=dev) * (L + 1), T.O.T @ rho)
            pr = (T.O * rho[:, None]).T @ T.O
            p, r = torch.nonzero(~torch.eye(L, dtype=torch.bool, device=dev), as_tuple=True)
            add(bs, p, r, p, r, pr[p, r])
            add(bs, p, r, r, p, -pr[p, r])
            v = T.s * G[T.I, T.J]
            one[spin].index_add_(0, T.p + L * T.q, v)
            e, k = torch.nonzero(T.O[T.I] * T.O[T.J], as_tuple=True)  # k: occupied in both
            p, q, v = T.p[e], T.q[e], v[e]
            add(bs, q, k, p, k, v)
            add(bs, k, q, k, p, v)
            add(bs, q, k, k, p, -v)
            add(bs, k, q, p, k, -v)
            for I, J, i, j, a, b, s in T.doubles():
                v = s * G[I, J]
                add(bs, a, b, i, j, v)
                add(bs, b, a, j, i, v)
                add(bs, a, b, j, i, -v)
                add(bs, b, a, i, j, -v)
        # alpha-beta: T[pq][rs] over the extended singles of both spins
        aI, aJ, ap, aq, as_ = self.A.extended()
        bI, bJ, bp, bq, bs_ = self.B.extended()
        rs = bp * L + bq
        order = torch.argsort(rs, stable=True)
        bI, bJ, bs_ = bI[order], bJ[order], bs_[order]
        start = torch.searchsorted(rs[order], torch.arange(L * L + 1, device=dev)).tolist()
        T = torch.zeros(L * L, L * L, dtype=torch.float64, device=dev)
        for k in range(L * L):
            z = slice(start[k], start[k + 1])
            if z.stop > z.start:
                M = (X[:, bI[z]] * bs_[z]) @ X[:, bJ[z]].T
                T[:, k].index_add_(0, ap * L + aq, as_ * M[aI, aJ])
        p, q, r, s = (v.reshape(-1) for v in torch.meshgrid(*[torch.arange(L, device=dev)] * 4, indexing="ij"))
        v = T.reshape(-1)
        # of two excitations, the element goes to the block of its lower
        # created spin orbital (2p alpha, 2r+1 beta) with the annihilated
        # ones in ascending order
        swap = (p != q) & (r != s) & ((p <= r) != (q <= s))
        for m, ab, ba in ((~swap, 2, 1), (swap, 1, 2)):
            add(ab, q[m], s[m], p[m], r[m], v[m])
            add(ba, s[m], q[m], r[m], p[m], v[m])
        return one.reshape(-1), two.reshape(-1)

    def ground(self):
        """The lowest eigenpair: Davidson with full reorthogonalization from
        the Hartree-Fock determinant and a little of everything else."""
        d = self.diagonal().reshape(-1)
        g = torch.Generator(device="cpu").manual_seed(3)
        v = 1e-3 * torch.randn(d.numel(), dtype=torch.float64, generator=g).to(self.dev) / math.sqrt(d.numel())
        v[0] += 1.0
        V, HV = [v / v.norm()], []
        for _ in range(200):
            HV.append(self.sigma(V[-1]))
            Vm, Hm = torch.stack(V), torch.stack(HV)
            E, U = torch.linalg.eigh(Vm @ Hm.T)
            e, u = E[0], U[:, 0]
            W, HW = u @ Vm, u @ Hm
            r = e * W - HW
            if float(r.norm()) < 2e-13 * max(1.0, abs(float(e))):
                break
            if len(V) == 24:
                V, HV = [W / W.norm()], [HW / W.norm()]
                Vm = torch.stack(V)
            den = e - d
            t = r / torch.where(den.abs() < 1e-8, torch.full_like(den, -1e-8), den)
            for _ in range(2):
                t = t - (Vm @ t) @ Vm
                t = t / t.norm()
            V.append(t)
        W = W / W.norm()
        return float(e), W


def exact(case, seed):
    if case["op"] in ("solve", "roots") and (case["op"] == "roots" or case["na"] * case["nb"] > 400_000):
        return None
    ref = _Reference(case, seed)
    if case["op"] == "build":
        return ref.diagonal().reshape(-1).cpu().numpy()
    if case["op"] == "solve":
        E, W = ref.ground()
        return dict(E=E, W=_phased(W.cpu().numpy(), ref.B.n))
    x = _vector(ref.A.n, ref.B.n, seed)
    if case["op"] == "sigma":
        return ref.sigma(x)
    one, two = ref.rdm(x)
    return dict(one=one.cpu().numpy(), two=two.cpu().numpy())
