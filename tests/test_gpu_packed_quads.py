"""Stages of affine quads with several elements per wavefront, on graded
meshes (no two neighbours of one size, so that a clamped or misplaced element's
metric shows) just beyond the size from which meshes are packed, the last
wavefront short; and the same on a few elements, one to a wavefront:
Navier-Stokes, Euler with walls, the mixed precision, and the acoustic system
forward and reversed.
"""
import numpy as np
import pytest

from acoustic_ref import AcousticRef
from dgm_amd import acoustic, dgx, mesh as meshgen
from oracle_lib import Oracle
from test_oracle_acoustic import stretched_quads

pytestmark = pytest.mark.gpu

# rounding of one step: the stages' residuals agree to 1e-14 (test_gpu_parity),
# LSRK14's weights amplify that about 55 times and a small momentum field about
# ten times more
TOL = 1e-11
# p, nx, ny: packed by 5, 4, 3 and 2 elements with 4, 2, 2 and 1 in the last
# wavefront, then one element to a wavefront
SIZES = [(1, 67, 62), (2, 67, 62), (3, 67, 62), (4, 91, 91), (1, 3, 2), (2, 5, 3), (6, 3, 2), (10, 2, 3)]


def _graded(m):
    """The mesh of [0, 2 pi]^2 with its lines moved: element sizes vary threefold."""
    m.vert[:, 0] += 0.5 * np.sin(m.vert[:, 0])
    m.vert[:, 1] += 0.4 * np.sin(m.vert[:, 1] + 1.0) - 0.4 * np.sin(1.0)
    return m


def _state(x):
    s = [np.sin(x[0] + 0.3 * k) * np.cos(x[1] - 0.2 * k) for k in range(4)]
    return np.stack([1.0 + 0.1 * s[0], 0.4 + 0.1 * s[1], 0.2 * s[2] - 0.1, 2.2 + 0.1 * s[3]])


def _rel(a, b):
    return np.sqrt(((a - b) ** 2).sum((1, 2)) / (b ** 2).sum((1, 2)))


def _dt(m, p, vis=0.0):
    h = (m.vert.max(2) - m.vert.min(2)).min()
    adv = 0.1 * h / ((p + 1) ** 2 * 2.0)
    return min(adv, 0.1 * h * h / (vis * 2.0 * (p + 1) ** 4)) if vis else adv


@pytest.mark.parametrize("inttype", [dgx.DGX_TVD, dgx.DGX_RK4, dgx.DGX_LSRK14])
@pytest.mark.parametrize("p,nx,ny", SIZES)
def test_navier_stokes_step_matches_the_oracle(p, nx, ny, inttype):
    print(f"[packed quads] Navier-Stokes p={p} {nx}x{ny} inttype={inttype}", flush=True)
    m = _graded(meshgen.periodic_quads(nx, ny, 0.0, 2 * np.pi, 0.0, 2 * np.pi))
    orc = Oracle(m, p, 2, vis=0.02, flux=p % 2)
    orc.set_state(_state(orc.coords()))
    orc.project_state()
    gpu = dgx.GPUDomain(m, p, dgx.DGX_NAVIER_STOKES, vis=0.02, flux=p % 2)
    gpu.upload(orc.state())
    dt = _dt(m, p, 0.02)
    orc.advance(inttype, dt, 1)
    gpu.advance(inttype, dt, 1)
    err = _rel(gpu.download(), orc.state())
    gpu.close()
    print(f"[packed quads] rel L2 per field: {err}", flush=True)
    assert np.all(err <= TOL), err


@pytest.mark.parametrize("p,nx,ny", SIZES)
def test_euler_step_with_walls_matches_the_oracle(p, nx, ny):
    """Slip walls at the bottom and top, a free stream at the sides."""
    print(f"[packed quads] walls p={p} {nx}x{ny}", flush=True)
    free = [1.0, 0.4, 0.0, 2.2]
    m = _graded(meshgen.box_quads(nx, ny, 0.0, 2 * np.pi, 0.0, 2 * np.pi, bc=(0, 1, 0, 1)))
    orc = Oracle(m, p, 1)
    orc.set_bc_state(free)
    orc.set_state(_state(orc.coords()))
    orc.project_state()
    gpu = dgx.GPUDomain(m, p, dgx.DGX_EULER, bc_state=free + [0.0])
    gpu.upload(orc.state())
    dt = _dt(m, p)
    orc.advance(dgx.DGX_RK4, dt, 1)
    gpu.advance(dgx.DGX_RK4, dt, 1)
    err = _rel(gpu.download(), orc.state())
    gpu.close()
    print(f"[packed quads] rel L2 per field: {err}", flush=True)
    assert np.all(err <= TOL), err


@pytest.mark.parametrize("p,nx,ny", SIZES[:4] + SIZES[6:7])
@pytest.mark.parametrize("inttype", [dgx.DGX_TVD, dgx.DGX_LSRK14])
@pytest.mark.parametrize("eqn", [dgx.DGX_EULER, dgx.DGX_SHALLOW])
def test_mixed_step_stays_near_fp64(eqn, p, nx, ny, inttype):
    """One step of the mixed precision against the FP64 one: FP32 contractions
    leave 1e-4 of the residual (test_gpu_mixed2d), of which a step takes
    dt |R| / |U| < 1e-2, LSRK14 with weights up to 39; against the norm of the
    whole state, as a momentum is a small part of it."""
    print(f"[packed quads] mixed eqn={eqn} p={p} {nx}x{ny} inttype={inttype}", flush=True)
    m = _graded(meshgen.periodic_quads(nx, ny, 0.0, 2 * np.pi, 0.0, 2 * np.pi))
    out = []
    for prec in (dgx.DGX_FP64, dgx.DGX_MIXED):
        g = dgx.GPUDomain(m, p, eqn, precision=prec, balance=False)
        U = _state(g.coords())
        g.upload(U if eqn == dgx.DGX_EULER else U[:3])
        g.advance(inttype, _dt(m, p), 1)
        out.append(g.download(dgx.DGX_MODAL))
        g.close()
    err = np.sqrt(((out[1] - out[0]) ** 2).sum((1, 2)) / (out[0] ** 2).sum())
    print(f"[packed quads] error against the whole state per field: {err}", flush=True)
    assert np.all(err <= 1e-5) and np.any(err > 0), err


@pytest.mark.parametrize("n,p", [((65, 64), 1), ((67, 62), 2), ((67, 62), 3), ((91, 91), 4), ((5, 4), 2)])
def test_acoustic_gradient_matches_the_oracle(n, p):
    """Forward observations and the gradient on graded quads, packed: the bars
    of the small meshes (test_gpu_acoustic)."""
    print(f"[packed quads] acoustic {n[0]}x{n[1]} p={p}", flush=True)
    m = stretched_quads(*n)
    mean, rec = (1.0, 0.3, -0.1, 1.0 / 1.4), [(0.13, 0.21), (0.77, 0.4), (0.5, 0.9)]
    dt, steps = 0.2 / max(n) / ((p + 1) ** 2 * 1.4), 3
    gpu = acoustic.AcousticProblem(m, p, mean, rec, 0.4 / dt, 0.5 * dt, dt, steps, nsnap=2, gamma=1.4)
    ref = AcousticRef(m, p, mean, rec, 0.4 / dt, 0.5 * dt, dt, steps, gamma=1.4)
    rng = np.random.default_rng(p)
    true, theta = rng.standard_normal(m.ne), rng.standard_normal(m.ne)
    y, y_ref = gpu.forward(true), ref.forward(true)
    J, g = gpu.gradient(theta, y_ref)
    J_ref, g_ref = ref.gradient(theta, y_ref)
    gpu.close()
    ey, eg = np.linalg.norm(y - y_ref) / np.linalg.norm(y_ref), np.linalg.norm(g - g_ref) / np.linalg.norm(g_ref)
    print(f"[packed quads] observations {ey:.2e}, J {abs(J - J_ref) / J_ref:.2e}, gradient {eg:.2e}", flush=True)
    assert ey <= 1e-12 and abs(J - J_ref) <= 1e-10 * J_ref and eg <= 1e-10
