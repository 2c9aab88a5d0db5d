"""Arnoldi steps in blocks (two passes over the basis for up to four steps)
against one step at a time: the same Krylov steps, restarts and deflation
space, so the same counts and solutions to the solve's tolerance, and true
residuals by the oracle's operator.  Sizes where a block is cut: cycle lengths
and deflation counts that leave remainders of 1..3, iteration floors and cycles
shorter than a block, the smallest lattice, strides with padding sites, and a
right-hand side whose Krylov space ends at once."""
import numpy as np
import pytest

import oracle as O
from baylorlqcd_amd import _lib, diracops, inverters, lattice

pytestmark = pytest.mark.gpu

BC = (1, 1, 1, -1)


def setup(n, kind=1, eps=0.3, bc=BC):
    lattice.init(n, bc)
    co = O.coact_array()
    diracops.gauge_random(kind, eps, 11, co)
    U = diracops.gauge_get_canonical(n)
    u = O.links_canon_to_ref(n, U)
    diracops.gauge_load(u, co)
    return U, u, co


def rhs(n, seed):
    V = int(np.prod(n))
    psi = np.random.default_rng(seed).standard_normal(24 * V).view(np.complex128).reshape(V, 4, 3)
    psi[O.parity_mask(n)] = 0
    return psi, O.spinor_canon_to_ref(n, psi)[0]


def residual(n, U, kap, psi, x, bc=BC):
    xe = O.spinor_ref_to_canon(n, x, None)
    even = ~O.parity_mask(n)
    r = psi - O.schur(n, U, bc, [1] * 4, [1] * 4, 0, kap, xe)
    return np.linalg.norm(r[even]) / np.linalg.norm(psi[even])


def both(f):
    """f() one step at a time, then in blocks."""
    out = []
    try:
        for steps in (1, 2):
            _lib.check(_lib.lib().qqcd_set_arnoldi_steps(steps))
            out.append(f())
    finally:
        _lib.check(_lib.lib().qqcd_set_arnoldi_steps(2))
    return out


@pytest.mark.parametrize("n", [(4, 4, 4, 4), (12, 4, 8, 4), (8, 8, 8, 16)])
@pytest.mark.parametrize("gm,kap", [((40, 10), (0.12, 0.0)), ((7, 2), (0.12, 0.01)), ((3, 1), (0.10, 0.0)),
                                    ((21, 0), (0.12, 0.0)), ((23, 5), (0.125, 0.02)), ((60, 20), (0.125, 0.0))])
def test_gmresdr_and_proj(n, gm, kap):
    print(f"[arnoldi] {n} GMRES{gm} kappa {kap}", flush=True)
    U, u, co = setup(n)
    try:
        psi, phi = rhs(n, 3)
        psi2, phi2 = rhs(n, 4)

        def solve():
            x = np.zeros_like(phi)
            it = inverters.gmresdr(None, phi, x, gm, 1e-11, 0, u, None, -1, kap, co, BC)
            if gm[1] == 0:
                return it, x
            y = np.zeros_like(phi)
            mvp = np.zeros(1, np.int32)
            gdr = np.full((4000, 1), -1.0, order="F")
            it2 = inverters.gmresproject(None, phi2, y, (gm[0] - gm[1], gm[1]), 1e-11, 0, u, None, -1, kap, co, BC,
                                         isignal=2, mvp=mvp, gdr=gdr)
            h = gdr[:, 0]
            assert np.sum(h != -1.0) == it2 and np.all(h[int(mvp[0]):] == -1.0)
            return it, x, it2, y, h[h != -1.0]

        one, blk = both(solve)
    finally:
        lattice.finalize()
    # a solution at relative residual 1e-11 is off by at most that times the condition number (below 1e2 here)
    assert blk[0] == one[0]
    assert np.linalg.norm(blk[1] - one[1]) < 2e-9 * np.linalg.norm(one[1])
    assert residual(n, U, kap, psi, blk[1]) < 1e-11
    if gm[1]:
        assert blk[2] == one[2]
        assert residual(n, U, kap, psi2, blk[3]) < 1e-11
        # the history entries are residual norms of the same steps, down to 1e-11 of the first
        assert np.allclose(blk[4], one[4], rtol=1e-4, atol=1e-13 * one[4][0])


def test_iteration_floor():
    """itermin keeps a converged solve going to the given step, also inside a block."""
    n = (8, 8, 8, 16)
    U, u, co = setup(n)
    try:
        psi, phi = rhs(n, 5)
        for itermin in (0, 1, 37, 38, 39):
            one, blk = both(lambda: inverters.gmresdr(None, phi, np.zeros_like(phi), (40, 10), 1e-6, itermin, u, None,
                                                      -1, (0.12, 0.0), co, BC))
            assert one == blk and blk >= itermin
    finally:
        lattice.finalize()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_invariant_start(prec):
    """Free field, periodic, constant right-hand side: an eigenvector of the operator, whose Krylov space has one
    dimension (every new vector is rounding), and a sum of two, whose space has two."""
    n, bc = (8, 4, 4, 8), (1, 1, 1, 1)
    U, u, co = setup(n, kind=1, eps=0.0, bc=bc)
    kap = (0.11, 0.0)
    try:
        even = ~O.parity_mask(n)
        s = np.arange(int(np.prod(n)))
        const = np.zeros((len(s), 4, 3), complex)
        const[even] = np.arange(1, 13).reshape(4, 3)
        wave = const * np.where((s % n[0]) % 4 < 2, 1.0, -1.0)[:, None, None]
        for psi in (const, const + wave):
            phi, _ = O.spinor_canon_to_ref(n, psi)
            x = np.zeros_like(phi)
            if prec == "fp64":
                inverters.gmresdr(None, phi, x, (20, 4), 1e-10, 0, u, None, -1, kap, co, bc)
            else:
                inverters.solve_mixed(phi, x, (20, 4), 1e-10, 1, 1, 18, 0.0, 0, u, co, kap, bc)
            assert residual(n, U, kap, psi, x, bc) < 1e-10
    finally:
        lattice.finalize()


@pytest.mark.parametrize("basis,prec,recon", [(1, 1, 18), (1, 1, 12), (1, 2, 12), (2, 2, 12), (2, 2, 18), (2, 1, 18)])
@pytest.mark.parametrize("n,gm", [((8, 8, 8, 16), (40, 16)), ((8, 8, 8, 16), (21, 6)), ((4, 4, 4, 4), (10, 3)),
                                  ((12, 4, 8, 4), (60, 20))])
def test_mixed_low_basis(basis, prec, recon, n, gm):
    """Blocks over an FP32 or FP16 basis, operator in FP32 or FP16: the FP64 residual is met, in about the steps
    of one at a time (an inner solve may end a check later)."""
    kap = (0.125, 0.01)
    U, u, co = setup(n)
    try:
        psi, phi = rhs(n, 6)

        def solve():
            x = np.zeros_like(phi)
            return inverters.solve_mixed(phi, x, gm, 1e-10, basis, prec, recon, 0.0, 0, u, co, kap, BC), x

        one, blk = both(solve)
    finally:
        lattice.finalize()
    assert residual(n, U, kap, psi, blk[1]) < 1e-10
    assert np.linalg.norm(blk[1] - one[1]) < 1e-8 * np.linalg.norm(one[1])
    # an inner solve ends with a block, all of whose vectors are used: whole blocks of four where the cycles are
    if (gm[0] - gm[1]) % 4 == 0:
        assert blk[0] % 4 == 0, blk[0]
    # not more steps, to an inner check's granularity per outer step; fewer only where the inner target (1e-6 with
    # the FP32 operator) is below what an FP16 basis carries (11 bits), so that inner solves run to their cap
    assert blk[0] <= 1.15 * one[0] + 8, (one[0], blk[0])
    if (basis, prec) != (2, 1):
        assert blk[0] >= 0.85 * one[0] - 8, (one[0], blk[0])


def check_basis(phi, m, u, co, kap, bc):
    steps, out = np.zeros(1, np.int32), np.zeros(3)
    _lib.check(_lib.lib().qqcd_arnoldi_check(_lib.dp(phi), m, _lib.dp(u), _lib.dp(np.asarray(co).ravel(order="F")),
                                             _lib.dp(np.array(kap)), _lib.ints(bc).ctypes.data_as(_lib._ip),
                                             steps.ctypes.data_as(_lib._ip), _lib.dp(out)))
    return int(steps[0]), *out


@pytest.mark.parametrize("m", [6, 23])
@pytest.mark.parametrize("eps", [0.0, 1e-9, 1e-7, 1e-6, 1e-5, 3e-5, 5e-5, 1e-4, 3e-4, 1e-3, 1e-2, 1.0])
def test_near_invariant_basis(m, eps):
    """An eigenvector with a little noise: the first block's vectors cancel against it to any number of digits, so
    that none, some or all of them are taken.  The basis stays orthogonal and the Arnoldi relation holds."""
    n, bc, kap = (8, 4, 4, 8), (1, 1, 1, 1), (0.11, 0.0)
    U, u, co = setup(n, kind=1, eps=0.0, bc=bc)
    try:
        even = ~O.parity_mask(n)
        const = np.zeros((int(np.prod(n)), 4, 3), complex)
        const[even] = np.arange(1, 13).reshape(4, 3)
        noise, _ = rhs(n, 8)
        psi = const + eps * noise * np.linalg.norm(const) / np.linalg.norm(noise)
        phi, _ = O.spinor_canon_to_ref(n, psi)
        steps, loss, bound, rel = check_basis(phi, m, u, co, kap, bc)
    finally:
        lattice.finalize()
    print(f"[arnoldi] near invariant {m} {eps}: {steps} steps, loss {loss:.2e} <= {bound:.2e}, relation {rel:.2e}",
          flush=True)
    # the bound that the solver keeps, and what it says of the basis; the relation to the rounding of vectors that
    # cancelled to the least that is taken (1e-6 of the squared norm)
    assert loss < 1e-12 and loss <= bound <= 1e-8
    assert rel < 1e-15 / 1e-3


@pytest.mark.parametrize("n,m", [((4, 4, 4, 4), 11), ((8, 8, 8, 16), 40), ((12, 4, 8, 4), 61), ((8, 8, 8, 16), 120)])
def test_basis(n, m):
    U, u, co = setup(n)
    try:
        psi, phi = rhs(n, 9)
        steps, loss, bound, rel = check_basis(phi, m, u, co, (0.125, 0.01), BC)
    finally:
        lattice.finalize()
    print(f"[arnoldi] basis {n} {m}: {steps} steps, loss {loss:.2e} <= {bound:.2e}, relation {rel:.2e}", flush=True)
    assert steps == m and loss < 1e-12 and loss <= bound <= 1e-8 and rel < 1e-14
