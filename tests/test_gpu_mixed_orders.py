"""The mixed-precision hex kernels at every order (each has its own thread
count), inviscid, BR1 and BR2: residual and one LSRK14 step against the FP64
path, on a box with different sizes and element counts per direction.
"""
import numpy as np
import pytest

from dgm_amd import dgx, mesh as meshgen

pytestmark = pytest.mark.gpu

# FP32 sums (eps 6e-8) of terms up to (p + 1)^2 times the deviation, whose
# residual they are summed into: a few 1e-5 of it at p = 8; a step multiplies
# that by dt |R| / |U| < 1e-2
TOL_RHS, TOL_STEP = 1e-4, 1e-6


def _domain(p, eqn, viscous, precision):
    m = meshgen.periodic_hexes(3, 2, 4, (0, 0, 0), (2 * np.pi, 2 * np.pi, 4.0))
    g = dgx.GPUDomain(m, p, eqn, gamma=1.4, vis=0.02 if eqn == dgx.DGX_NAVIER_STOKES3D else 0.0, Pr=0.71, precision=precision,
                      flux=p % 2, viscous=viscous, br2_eta=6.0)
    x = g.coords()
    s = [np.sin(x[0] + 0.3 * k) * np.cos(x[1] - 0.2 * k) * np.cos(np.pi * x[2] / 2 + 0.1 * k) for k in range(5)]
    g.upload(np.stack([1.0 + 0.1 * s[0], 0.3 + 0.1 * s[1], 0.1 * s[2] - 0.1, 0.1 * s[3], 2.5 + 0.1 * s[4]]))
    return g


def _rel(a, b):
    return np.sqrt(((a - b) ** 2).sum((1, 2)) / (b ** 2).sum((1, 2)))


@pytest.mark.parametrize("p", [1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("eqn,viscous", [(dgx.DGX_EULER3D, 0),
                                         (dgx.DGX_NAVIER_STOKES3D, dgx.DGX_VISCOUS_BR1),
                                         (dgx.DGX_NAVIER_STOKES3D, dgx.DGX_VISCOUS_BR2)])
def test_residual_and_step_match_fp64(p, eqn, viscous):
    print(f"[mixed orders] p={p} eqn={eqn} viscous={viscous}", flush=True)
    a, b = _domain(p, eqn, viscous, dgx.DGX_MIXED), _domain(p, eqn, viscous, dgx.DGX_FP64)
    e_rhs = _rel(a.rhs(), b.rhs())
    dt = 0.02 / (p + 1) ** 2
    for g in (a, b):
        g.advance(dgx.DGX_LSRK14, dt, 1)
    e_step = _rel(a.download(), b.download())
    a.close()
    b.close()
    print(f"[mixed orders] residual {e_rhs} step {e_step}", flush=True)
    assert np.all(e_rhs <= TOL_RHS), e_rhs
    assert np.all(e_step <= TOL_STEP), e_step
