"""The launch forms of the single-right-hand-side hop that the size picks: one
hop per wavefront (fields in the last-level cache), pipelined without and with
streaming.  Each storage format against the oracle's hop and twisted Schur
operator (so the epilogue with and without the local spinor) on both parities,
for both signs and every boundary condition, at the smallest lattice, at
extents below a wavefront and ragged ones; and the two sides of the dispatch's
lines against each other at their sizes."""
import numpy as np
import pytest

import oracle as O
from baylorlqcd_amd import _lib, diracops, inverters, lattice

pytestmark = pytest.mark.gpu

FORMATS = ((0, 18, 1e-14), (0, 12, 1e-13), (1, 18, 1e-6), (1, 12, 1e-6), (2, 18, 3e-3), (2, 12, 3e-3))


def rel2(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def field(n, seed):
    V = int(np.prod(n))
    return np.random.default_rng(seed).standard_normal(24 * V).view(np.complex128).reshape(V, 4, 3)


@pytest.mark.parametrize("bc", [(1, 1, 1, -1), (0, -1, 1, 0)])
@pytest.mark.parametrize("n", [(4, 4, 4, 4), (4, 12, 8, 20), (20, 4, 4, 8), (12, 8, 20, 28)])
def test_formats(n, bc):
    print(f"[hop forms] {n} {bc}", flush=True)
    lattice.init(n, bc)
    try:
        co = O.coact_array()
        diracops.gauge_random(0, 0.0, 3, co)
        U = diracops.gauge_get_canonical(n)
        psi = field(n, 1)
        odd = O.parity_mask(n)
        for prec, recon, tol in FORMATS:
            for par in (0, 1):
                for idag in (0, 1):
                    want = O.hop(n, U, bc, [1] * 4, [1] * 4, idag, par, psi)
                    got = diracops.hop_canonical(psi, par, idag, prec, recon)
                    at = odd if par else ~odd
                    assert rel2(got[at], want[at]) < tol, (prec, recon, par, idag)
            for kap in ((0.15, 0.0), (0.156, 0.05)):
                want = O.schur(n, U, bc, [1] * 4, [1] * 4, 0, kap, psi)[~odd]
                got = diracops.schur_canonical(psi, kap, 0, prec, recon)[~odd]
                assert rel2(got, want) < tol, (prec, recon, kap)
    finally:
        lattice.finalize()


# FP64/18 fits the cache up to 166k sites of a parity (20^3x40: 160k, 20^2x24x40: 192k does not); FP32/18 to 24^3x48;
# FP16 takes the pipelined form past 200k sites and streams past the cache
@pytest.mark.parametrize("n,formats", [((20, 20, 20, 40), ((0, 18), (0, 12), (2, 12))),
                                       ((20, 20, 24, 40), ((0, 18), (1, 18), (2, 18))),
                                       ((24, 24, 24, 48), ((1, 18), (1, 12), (2, 12), (2, 18)))])
def test_both_sides_of_the_lines(n, formats):
    print(f"[hop forms] {n}", flush=True)
    lattice.init(n, (1, 1, 1, -1))
    try:
        diracops.gauge_random(1, 0.3, 5, O.coact_array())
        psi = field(n, 2)
        even = ~O.parity_mask(n)
        for prec, recon in formats:
            out = []
            for depth in (2, 1):  # the size's own choice, the pipelined streaming kernel
                _lib.check(_lib.lib().qqcd_set_dslash_tune(1, 0, depth, 1))
                out.append(diracops.schur_canonical(psi, (0.15, 0.01), 0, prec, recon)[even])
            # sums in another order; FP16 results rounded to 11 bits of the site's largest (an ulp may flip)
            assert rel2(out[0], out[1]) < (2e-15, 5e-7, 3e-4)[prec], (prec, recon)
    finally:
        _lib.check(_lib.lib().qqcd_set_dslash_tune(1, 0, 2, 1))
        lattice.finalize()


def test_fp16_result_in_both_precisions():
    """The FP16 hop's FP32 copy and its own rounded result (both used by the mixed solver's chains of operator
    applications): a mixed solve on the form reaches the FP64 residual."""
    n, bc, kap = (12, 8, 20, 4), (1, 1, 1, -1), (0.12, 0.02)
    lattice.init(n, bc)
    try:
        co = O.coact_array()
        diracops.gauge_random(1, 0.3, 8, co)
        U = diracops.gauge_get_canonical(n)
        u = O.links_canon_to_ref(n, U)
        diracops.gauge_load(u, co)
        even = ~O.parity_mask(n)
        psi = field(n, 4) * even[:, None, None]
        phi, _ = O.spinor_canon_to_ref(n, psi)
        for basis in (1, 2):
            x = np.zeros_like(phi)
            inverters.solve_mixed(phi, x, (20, 6), 1e-11, basis, 2, 12, 0.0, 0, u, co, kap, bc)
            r = psi - O.schur(n, U, bc, [1] * 4, [1] * 4, 0, kap, O.spinor_ref_to_canon(n, x, None))
            assert np.linalg.norm(r[even]) < 1e-11 * np.linalg.norm(psi)
    finally:
        lattice.finalize()
