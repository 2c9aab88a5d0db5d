"""Gauge generation and smearing at their launch forms' edges: lattices below
and above a workgroup's sites, ragged extents, and both sides of the smearing's
line between one and four spins a lane.  The heatbath is followed link by link
in numpy (same counter-based random numbers, same order of updates)."""
import numpy as np
import pytest

import oracle as O
from baylorlqcd_amd import diracops, gauge, lattice

pytestmark = pytest.mark.gpu


def smix(z):
    with np.errstate(over="ignore"):
        z = z + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def sweep(n, U, beta, seed, sw):
    """One pseudo-heatbath sweep on U (V, 4, 3, 3), sites x0 + n0 (x1 + n1 (x2 + n2 x3))."""
    V = int(np.prod(n))
    lex = np.arange(V).reshape(n[::-1])
    up = [np.roll(lex, -1, 3 - m).ravel() for m in range(4)]
    dn = [np.roll(lex, 1, 3 - m).ravel() for m in range(4)]
    odd = O.parity_mask(n)
    dag = lambda a: np.conj(np.swapaxes(a, -1, -2))
    for par in (0, 1):
        s = np.nonzero(odd if par else ~odd)[0]
        for mu in range(4):
            A = 0
            for nu in range(4):
                if nu != mu:
                    pm, mn = up[mu][s], dn[nu][s]
                    A = A + U[pm, nu] @ dag(U[up[nu][s], mu]) @ dag(U[s, nu])
                    A = A + dag(U[dn[nu][pm], nu]) @ dag(U[mn, mu]) @ U[mn, nu]
            W = U[s, mu]
            with np.errstate(over="ignore"):
                key = (np.uint64(sw * 8 + par * 4 + mu) * np.uint64(1 << 32)) + (s >> 1).astype(np.uint64)
            st = smix(np.uint64(seed) ^ smix(key))

            def uni(mask):
                st[mask] = smix(st[mask])
                return ((st[mask] >> np.uint64(11)).astype(np.float64) + 1.0) / 9007199254740992.0

            for p, q in ((0, 1), (1, 2), (0, 2)):
                w = W @ A
                a = np.array([0.5 * (w[:, p, p].real + w[:, q, q].real), 0.5 * (w[:, p, q].imag + w[:, q, p].imag),
                              0.5 * (w[:, p, q].real - w[:, q, p].real), 0.5 * (w[:, p, p].imag - w[:, q, q].imag)])
                k = np.sqrt((a * a).sum(0))
                x0, todo = np.ones(len(s)), np.ones(len(s), bool)
                while todo.any():
                    r1, r2, r3, r4 = (uni(todo) for _ in range(4))
                    X = -(np.log(r1) + np.cos(2 * np.pi * r2) ** 2 * np.log(r3)) / (2 * beta * k[todo] / 3)
                    ok = r4 * r4 <= 1 - 0.5 * X
                    at = np.nonzero(todo)[0][ok]
                    x0[at] = 1 - X[ok]
                    todo[at] = False
                every = np.ones(len(s), bool)
                ct = 2 * uni(every) - 1
                ph = 2 * np.pi * uni(every)
                rr, sn = np.sqrt(np.maximum(0, 1 - x0 * x0)), np.sqrt(np.maximum(0, 1 - ct * ct))
                sig = lambda c: np.array([[c[0] + 1j * c[3], c[2] + 1j * c[1]],
                                          [-c[2] + 1j * c[1], c[0] - 1j * c[3]]]).transpose(2, 0, 1)
                R = sig([x0, rr * sn * np.cos(ph), rr * sn * np.sin(ph), rr * ct]) @ dag(sig(a / k))
                W = W.copy()
                W[:, [p, q]] = R @ W[:, [p, q]]
            W[:, 0] /= np.linalg.norm(W[:, 0], axis=1)[:, None]
            W[:, 1] -= (np.conj(W[:, 0]) * W[:, 1]).sum(1)[:, None] * W[:, 0]
            W[:, 1] /= np.linalg.norm(W[:, 1], axis=1)[:, None]
            W[:, 2] = np.conj(np.cross(W[:, 0], W[:, 1]))
            U[s, mu] = W


@pytest.mark.parametrize("n", [(4, 4, 4, 4), (12, 4, 8, 4), (4, 8, 4, 20), (12, 8, 20, 28)])
def test_heatbath_sweep(n):
    # a link's rounding (about 1e-15) grows by at most the staples' condition a sweep: 1e-11 after two
    print(f"[forms] heatbath {n}", flush=True)
    lattice.init(n, (1, 1, 1, -1))
    try:
        co = O.coact_array()
        diracops.gauge_heatbath(5.7, 0, 77, 1, co)
        U = diracops.gauge_get_canonical(n)
        for sw in range(2):
            sweep(n, U, 5.7, 77, sw)
        diracops.gauge_heatbath(5.7, 2, 77, 1, co)
        assert np.max(np.abs(diracops.gauge_get_canonical(n) - U)) < 1e-11
    finally:
        lattice.finalize()


@pytest.mark.parametrize("n", [(4, 4, 4, 4), (12, 4, 8, 4), (4, 8, 20, 4), (20, 20, 20, 24), (20, 20, 20, 28)])
def test_smear_forms(n):
    bc, a, ns = (-1, 1, 0, 1), 0.15, 3
    print(f"[forms] smear {n}", flush=True)
    lattice.init(n, bc)
    try:
        U = gauge.haar(n, 8)
        V = int(np.prod(n))
        psi = np.random.default_rng(9).standard_normal(24 * V).view(np.complex128).reshape(V, 4, 3)
        ge, go = O.spinor_canon_to_ref(n, psi)
        he, ho = np.zeros_like(ge), np.zeros_like(go)
        diracops.smear(he, ho, O.links_canon_to_ref(n, U), ge, go, a, ns, bc)
        want = O.smear(n, U, bc, psi, a, ns)
        assert np.linalg.norm(O.spinor_ref_to_canon(n, he, ho) - want) < 1e-13 * np.linalg.norm(want)
    finally:
        lattice.finalize()
