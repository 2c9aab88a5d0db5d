"""BiCGStab with its scalars on the device against the same recurrence in
numpy on the oracle's operator: iteration counts, the logged residual history
and the solution, at vector lengths of a few workgroups and of the full grid,
with an iteration floor inside and past the queued iterations, and starts that
are already good enough."""
import numpy as np
import pytest

import oracle as O
from baylorlqcd_amd import diracops, inverters, lattice

pytestmark = pytest.mark.gpu

BC = (1, 1, 1, -1)


def reference(op, b, x, tol, itermin):
    r = b - op(x)
    r0 = rr = np.linalg.norm(r)
    rh, p, v = r.copy(), np.zeros_like(r), np.zeros_like(r)
    rho = alpha = omega = 1.0
    hist = []
    while not (rr < tol * r0 and len(hist) >= itermin):
        old, rho = rho, np.vdot(rh, r)
        beta = rho / old * (alpha / omega)
        p = r + beta * (p - omega * v)
        v = op(p)
        alpha = rho / np.vdot(rh, v)
        r = r - alpha * v
        t = op(r)
        omega = np.vdot(t, r) / np.vdot(t, t)
        x = x + omega * r + alpha * p
        r = r - omega * t
        rr = np.linalg.norm(r)
        hist.append(rr * rr / r0)
    return x, hist


@pytest.mark.parametrize("n,kap", [((4, 4, 4, 4), (0.12, 0.0)), ((12, 4, 8, 4), (0.12, 0.02)),
                                   ((8, 8, 8, 16), (0.12, 0.01)), ((16, 8, 12, 8), (0.115, 0.0))])
@pytest.mark.parametrize("tol,itermin,start", [(1e-9, 0, 0.0), (1e-4, 21, 0.5), (1e-4, 40, 0.0), (2.0, 0, 1.0),
                                               (2.0, 3, 1.0)])
def test_against_numpy(n, kap, tol, itermin, start):
    print(f"[bicgstab] {n} {kap} {tol} {itermin}", flush=True)
    lattice.init(n, BC)
    try:
        co = O.coact_array()
        diracops.gauge_random(1, 0.3, 21, co)
        U = diracops.gauge_get_canonical(n)
        u = O.links_canon_to_ref(n, U)
        diracops.gauge_load(u, co)
        even = ~O.parity_mask(n)
        V = int(np.prod(n))
        rng = np.random.default_rng(9)
        psi = np.zeros((V, 4, 3), complex)
        psi[even] = rng.standard_normal((V // 2, 4, 3)) + 1j * rng.standard_normal((V // 2, 4, 3))

        def op(w):
            f = np.zeros((V, 4, 3), complex)
            f[even] = w.reshape(-1, 4, 3)
            return O.schur(n, U, BC, [1] * 4, [1] * 4, 0, kap, f)[even].ravel()

        x0 = np.full((V, 4, 3), start, complex) * even[:, None, None]
        want, hist = reference(op, psi[even].ravel(), x0[even].ravel(), tol, itermin)
        phi, _ = O.spinor_canon_to_ref(n, psi)
        x, _ = O.spinor_canon_to_ref(n, x0)
        it = inverters.bicgstab(None, phi, x, tol, itermin, u, None, -1, kap, co, BC)
        log = inverters.solve_log()
    finally:
        lattice.finalize()
    got = O.spinor_ref_to_canon(n, x, None)[even].ravel()
    assert it == len(hist) and [v[1] for v in log] == list(range(1, it + 1))
    # the recurrences part by rounding, which BiCGStab's residuals amplify as they fall: the history to 1e-3 of
    # itself while it is above 1e-12 of its start, the solution to the residual
    h = np.array(hist)
    keep = h > 1e-12 * (h[0] if len(h) else 1.0)
    assert np.allclose(np.array([v[2] for v in log])[keep], h[keep], rtol=1e-3)
    scale = np.linalg.norm(want)
    assert np.linalg.norm(got - want) <= max(1e-8, 1e-2 * tol if tol < 1 else 1e-12) * max(scale, 1e-300)


@pytest.mark.parametrize("scale", [1e-90, 1e-75, 1e80])
def test_source_scale(scale):
    """The recurrence is linear in the source: a source scaled by a power of ten far from 1, whose squared scalars
    leave the range of FP64 while its norms do not, takes the same iterations to the scaled solution."""
    n, kap, tol = (8, 8, 8, 16), (0.12, 0.01), 1e-9
    lattice.init(n, BC)
    try:
        co = O.coact_array()
        diracops.gauge_random(1, 0.3, 21, co)
        u = diracops.gauge_get_ref(n)
        diracops.gauge_load(u, co)
        psi = np.random.default_rng(9).standard_normal(24 * int(np.prod(n))).view(complex).reshape(-1, 4, 3)
        phi, _ = O.spinor_canon_to_ref(n, psi)
        x1, xs = np.zeros_like(phi), np.zeros_like(phi)
        it1 = inverters.bicgstab(None, phi, x1, tol, 0, u, None, -1, kap, co, BC)
        its = inverters.bicgstab(None, scale * phi, xs, tol, 0, u, None, -1, kap, co, BC)
    finally:
        lattice.finalize()
    # the scale is no power of two: both runs round differently and end within an iteration or two of each other
    assert abs(its - it1) <= 2
    # residuals below 1e-9 each, condition number below 1e2
    assert np.linalg.norm(xs / scale - x1) < 2e-7 * np.linalg.norm(x1)
