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
