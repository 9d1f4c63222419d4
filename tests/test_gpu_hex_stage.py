"""One-kernel stages of affine hexes under every integrator and order (each
order has its own thread count), inviscid, BR1 and BR2, and with the channel's
bulk forcing, whose update runs after a domain-wide mean: against the CPU
oracle.
"""
import numpy as np
import pytest

from dgm_amd import dgx, mesh as meshgen
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

# rounding of one step: residuals agree to 1e-12 (test_gpu_parity) and enter
# with dt |R| / |U| << 1, amplified about 55 times by LSRK14's weights
TOL = 1e-11
WALL = (1.0, 4.0)


def _state(x, H):
    s = [np.sin(x[0] + 0.3 * k) * np.cos(x[1] - 0.2 * k) * np.cos(2 * np.pi * x[2] / H + 0.1 * k) for k in range(5)]
    return np.stack([1.0 + 0.1 * s[0], 0.3 + 0.1 * s[1], 0.1 * s[2] - 0.1, 0.1 * s[3], 2.5 + 0.1 * s[4]])


def _rel(a, b):
    return np.sqrt(((a - b) ** 2).sum((1, 2)) / (b ** 2).sum((1, 2)))


@pytest.mark.parametrize("inttype", [dgx.DGX_TVD, dgx.DGX_RK4, dgx.DGX_LSRK14])
@pytest.mark.parametrize("p,eqn,viscous", [(1, 9, 1), (2, 8, 0), (2, 9, 0), (3, 9, 1), (4, 8, 0), (4, 9, 0), (5, 9, 1),
                                           (6, 9, 0), (7, 8, 0), (7, 9, 1), (8, 9, 0), (9, 8, 0), (9, 9, 0), (10, 8, 0)])
def test_one_step_matches_the_oracle(p, eqn, viscous, inttype):
    print(f"[hex stage] p={p} eqn={eqn} viscous={viscous} inttype={inttype}", flush=True)
    vis = 0.02 if eqn == 9 else 0.0
    m = meshgen.periodic_hexes(3, 2, 2, (0, 0, 0), (2 * np.pi, 2 * np.pi, 2.0))
    orc = Oracle(m, p, eqn, vis=vis, flux=p % 2, viscous=viscous, br2_eta=6.0)
    orc.set_state(_state(orc.coords(), 2.0))
    orc.project_state()
    gpu = dgx.GPUDomain(m, p, eqn, vis=vis, flux=p % 2, viscous=viscous, br2_eta=6.0)
    gpu.upload(orc.state())
    dt = 0.05 / ((p + 1) ** 2 * 2.5)
    orc.advance(inttype, dt, 1)
    gpu.advance(inttype, dt, 1)
    err = _rel(gpu.download(), orc.state())
    gpu.close()
    print(f"[hex stage] rel L2 per field: {err}", flush=True)
    assert np.all(err <= TOL), err


@pytest.mark.parametrize("inttype", [dgx.DGX_TVD, dgx.DGX_RK4, dgx.DGX_LSRK14])
@pytest.mark.parametrize("p", [1, 3, 7])
def test_bulk_forcing_steps_match_stage_by_stage_residuals(p, inttype):
    """The forced step against the same integrator run on the host from the
    domain's own forced residuals (dgx_rhs, checked against the oracle in
    test_gpu_ns_walls)."""
    print(f"[hex stage] bulk p={p} inttype={inttype}", flush=True)
    m = meshgen.channel_hexes(3, 2, 3, (0, 0, 0), (2 * np.pi, 2 * np.pi, 2.0), bc_bottom=3, bc_top=3)
    g = dgx.GPUDomain(m, p, 9, vis=0.02, wall=WALL, bulk_forcing=True)
    g.upload(_state(g.coords(), 2.0))
    U = g.download(dgx.DGX_MODAL)
    dt = 0.05 / ((p + 1) ** 2 * 2.5)
    h = dgx.GPUDomain(m, p, 9, vis=0.02, wall=WALL, bulk_forcing=True)

    def f(V):
        h.upload(V, dgx.DGX_MODAL)
        return -h.rhs(dgx.DGX_MODAL)

    if inttype == dgx.DGX_TVD:
        a = U + dt * f(U)
        b = 0.75 * U + 0.25 * (a + dt * f(a))
        want = U / 3 + 2 / 3 * (b + dt * f(b))
    elif inttype == dgx.DGX_RK4:
        k1 = f(U)
        k2 = f(U + 0.5 * dt * k1)
        k3 = f(U + 0.5 * dt * k2)
        k4 = f(U + dt * k3)
        want = U + dt / 6 * (k1 + 2 * k2 + 2 * k3 + k4)
    else:
        from acoustic_ref import LSRK_A, LSRK_B
        want, Ut = U.copy(), np.zeros_like(U)
        for A, B in zip(LSRK_A, LSRK_B):
            Ut = A * Ut + dt * f(want)
            want = want + B * Ut
    g.advance(inttype, dt, 1)
    err = _rel(g.download(dgx.DGX_MODAL), want)
    g.close()
    h.close()
    print(f"[hex stage] rel L2 per field: {err}", flush=True)
    assert np.all(err <= TOL), err


def test_a_residual_between_stages_leaves_the_step_unchanged():
    m = meshgen.periodic_hexes(2, 2, 2)
    out = []
    for between in (False, True):
        g = dgx.GPUDomain(m, 3, dgx.DGX_EULER3D)
        g.upload(_state(g.coords(), 1.0))
        for st in range(3):
            g.stage(dgx.DGX_TVD, st, 1e-3)
            if between:
                g.rhs()
        out.append(g.download(dgx.DGX_MODAL))
        g.close()
    assert np.array_equal(out[0], out[1])


def test_free_stream_residual_is_that_of_plain_tables():
    """The even-odd derivative of a constant leaves the rounding of its table's
    rows, like the plain table's: with halves rounded once, p = 4 leaves less
    than the plain tables do (PLAIN, the residual's norms per field); halves
    formed from rounded entries left up to twice as much."""
    PLAIN = np.array([5.63e-16, 1.38e-13, 7.52e-14, 7.81e-14, 1.68e-13])
    m = meshgen.periodic_hexes(3, 3, 3, (0, 0, 0), (2 * np.pi,) * 3)
    g = dgx.GPUDomain(m, 4, dgx.DGX_EULER3D)
    x = g.coords()
    g.upload(np.stack([0 * x[0] + v for v in (1.0, 0.3, -0.2, 0.7, 250.0)]))
    F = g.rhs(dgx.DGX_MODAL)
    g.close()
    norms = np.sqrt((F ** 2).sum((1, 2)) / m.ne)
    print(f"[hex stage] free stream residual {norms}", flush=True)
    assert np.all(norms <= PLAIN), norms
