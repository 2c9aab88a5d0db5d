"""Batched Arnoldi steps in blocks of four over the FP16 basis, against one
step at a time: basis sizes that leave a block of one to three steps and that
take the pass of dots in two launches, one to two slot blocks, with and without
a twisted mass.  Both end below the tolerance, so the solutions differ by at
most twice it times the operator's condition number (below 100 here)."""
import numpy as np
import pytest

import oracle as O
from baylorlqcd_amd import _lib, diracops, disconloops, lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nrhs,gmres,kappa", [((4, 4, 4, 8), 2, (13, 6), (0.13, 0.0)),
                                                ((4, 8, 4, 12), 10, (18, 8), (0.13, 0.02)),
                                                ((8, 4, 12, 4), 18, (15, 4), (0.125, 0.0)),
                                                ((8, 8, 8, 16), 5, (60, 11), (0.15, 0.0)),
                                                ((4, 4, 4, 4), 70, (16, 8), (0.12, 0.01))])
def test_blocks(n, nrhs, gmres, kappa):
    bc, tol = (1, 1, 1, -1), 1e-10
    lattice.init(n, bc)
    lib = _lib.lib()
    try:
        co = O.coact_array()
        diracops.gauge_random(1, 0.4, 3, co)
        u = diracops.gauge_get_ref(n)
        U = diracops.gauge_get_canonical(n)
        V = int(np.prod(n))
        psi = np.random.default_rng(5).standard_normal(24 * V * nrhs).view(np.complex128).reshape(nrhs, V, 4, 3)
        src = [O.spinor_canon_to_ref(n, p) for p in psi]
        sols = {}
        for steps in (1, 2):
            print(f"[blocks] {n} {nrhs} {gmres} {kappa} steps {steps}", flush=True)
            _lib.check(lib.qqcd_set_arnoldi_steps(steps))
            xe, xo, it, rr = disconloops.fermprop_multi([s[0] for s in src], [s[1] for s in src], kappa, co, bc, tol,
                                                        gmres, u)
            sols[steps] = [O.spinor_ref_to_canon(n, xe[r], xo[r]) for r in range(nrhs)]
            assert disconloops.batch_stats()["fallback"] == 0
        one = [1.0] * 4
        for r in range(nrhs):
            x = sols[2][r]
            res = np.linalg.norm(psi[r] - O.full_m(n, U, bc, one, one, kappa, x)) / np.linalg.norm(psi[r])
            assert res < tol, (r, res)
            assert np.linalg.norm(x - sols[1][r]) < 200 * tol * np.linalg.norm(x), r
    finally:
        _lib.check(lib.qqcd_set_arnoldi_steps(2))
        lattice.finalize()


@pytest.mark.parametrize("eps", [0.0, 1e-5, 1e-4, 1e-3, 1e-2])
@pytest.mark.parametrize("nrhs,gmres", [(3, (20, 6)), (9, (27, 6))])
def test_invariant_sources(nrhs, gmres, eps):
    """Free field, periodic: constant sources are eigenvectors, so a slot's Krylov space has one dimension, or two
    for a sum of two eigenvectors, plus what eps of noise adds; a generic source shares the batch.  The blocks give
    up inside such a slot, which keeps what it has: every slot ends in the batch, in as many outer steps (one more
    at most) as one step at a time."""
    n, bc, tol, kappa = (8, 4, 4, 8), (1, 1, 1, 1), 1e-10, (0.11, 0.0)
    lattice.init(n, bc)
    lib = _lib.lib()
    try:
        co = O.coact_array()
        diracops.gauge_random(1, 0.0, 3, co)
        u = diracops.gauge_get_ref(n)
        U = diracops.gauge_get_canonical(n)
        V = int(np.prod(n))
        rng = np.random.default_rng(6)
        noise = rng.standard_normal(24 * V * nrhs).view(np.complex128).reshape(nrhs, V, 4, 3)
        s = np.arange(V)
        wave = np.where((s % n[0]) % 4 < 2, 1.0, -1.0)[:, None, None]
        const = np.broadcast_to(np.arange(1, 13).reshape(4, 3).astype(complex), (V, 4, 3))
        psi = np.empty_like(noise)
        for r in range(nrhs):
            psi[r] = (r + 1) * const * (1.0 + wave if r % 3 == 2 else 1.0)
            psi[r] += eps * noise[r] * np.linalg.norm(psi[r]) / np.linalg.norm(noise[r])
        psi[nrhs // 2] = noise[nrhs // 2]
        src = [O.spinor_canon_to_ref(n, p) for p in psi]
        outer = {}
        for steps in (1, 2):
            print(f"[blocks] invariant {nrhs} {gmres} eps {eps} steps {steps}", flush=True)
            _lib.check(lib.qqcd_set_arnoldi_steps(steps))
            xe, xo, it, rr = disconloops.fermprop_multi([p[0] for p in src], [p[1] for p in src], kappa, co, bc, tol,
                                                        gmres, u)
            st = disconloops.batch_stats()
            outer[steps] = st["outer"]
            assert st["fallback"] == 0, st
            for r in range(nrhs):
                x = O.spinor_ref_to_canon(n, xe[r], xo[r])
                res = np.linalg.norm(psi[r] - O.full_m(n, U, bc, [1.0] * 4, [1.0] * 4, kappa, x))
                # the solve stops at tol of its even-odd source b_e + kappa H b_o, at most (1 + 8 kappa) of the
                # whole one, and the odd residual is rounding
                assert res < (1 + 8 * kappa[0]) * tol * np.linalg.norm(psi[r]), (r, res)
        assert outer[2] <= outer[1] + 1, outer
    finally:
        _lib.check(lib.qqcd_set_arnoldi_steps(2))
        lattice.finalize()


def block_dots(nrhs, nb, nq, s, re):
    out = np.zeros(2 * s * (nq + s))
    _lib.check(_lib.lib().qqcd_block_dots(nrhs, nb, nq, s, _lib.dp(np.array(re)), _lib.dp(out)))
    return out.view(complex).reshape(nq + s, s)


# a sum of equal terms in FP32 is off by at most half a unit in the last place of 24 bits a term, here with one sign;
# the runs are of 48 terms at most (batched: 32), whatever the volume, and the rest is FP64


# (43 basis vectors or 64 slots a block on the largest lattice would be tens of GB: the smaller ones have them)
SUMS = [(n, r, nb, nq, s) for n in ((4, 4, 4, 4), (12, 8, 4, 8), (24, 24, 24, 48))
        for r, nb in ((0, 0), (3, 1), (3, 2), (6, 4), (8, 8), (18, 16), (20, 32), (5, 64))
        for nq, s in ((1, 4), (5, 3), (13, 2), (6, 1), (43, 4)) if n[0] < 24 or r == 0 or (nq < 43 and nb < 64)]


@pytest.mark.parametrize("n,nrhs,nb,nq,s", SUMS)
def test_long_sums(n, nrhs, nb, nq, s):
    print(f"[blocks] sums {n} {nrhs} {nb} {nq} {s}", flush=True)
    lattice.init(n, (1, 1, 1, -1))
    try:
        re = [0.3, 0.7, 0.11, 1.3, 0.9]
        got = block_dots(nrhs, nb, nq, s, re)
    finally:
        lattice.finalize()
    N = 12 * int(np.prod(n)) // 2
    f = np.array(re, np.float32).astype(float)
    if nrhs:
        f[0] = 1.0 / np.sqrt(N)  # of unit length: 1 as stored
    want = np.empty((nq + s, s))
    want[:nq] = N * f[0] * f[1:s + 1]
    want[nq:] = N * np.outer(f[1:s + 1], f[1:s + 1])
    run = 32 if nrhs else 48
    assert np.all(np.abs(got - want) <= (run + 4) * 2.0 ** -24 * want), np.abs(got / want - 1).max()
