"""One-launch stages of affine quads (k_quad2): every integrator, on meshes on
both sides of the packing rule (several elements per wavefront from 4096
elements at p <= 3, 8192 at p = 4) and with element counts that leave the last
wavefront short, against the CPU oracle; and in the serving loop, where the
packing depends on what shares the launch and the results must not.
"""
import numpy as np
import pytest

from dgm_amd import dgx, mesh as meshgen, serve
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu

# rounding of one step: the stages' residuals agree to 1e-14 (test_gpu_parity),
# LSRK14's weights amplify that about 55 times and a small momentum field about
# ten times more
TOL = 1e-11


def _state(x, eqn):
    s = [np.sin(x[0] + 0.3 * k) * np.cos(x[1] - 0.2 * k) for k in range(4)]
    if eqn == dgx.DGX_SHALLOW:
        return np.stack([1.0 + 0.1 * s[0], 0.2 + 0.1 * s[1], 0.1 * s[2] - 0.1])
    return np.stack([1.0 + 0.1 * s[0], 0.4 + 0.1 * s[1], 0.2 * s[2] - 0.1, 2.2 + 0.1 * s[3]])


@pytest.mark.parametrize("eqn", [dgx.DGX_EULER, dgx.DGX_SHALLOW])
@pytest.mark.parametrize("p,nx,ny", [(1, 5, 3), (2, 63, 65), (2, 64, 64), (3, 67, 62), (4, 90, 91), (4, 91, 91),
                                     (6, 3, 2), (10, 2, 3)])
@pytest.mark.parametrize("inttype", [dgx.DGX_TVD, dgx.DGX_RK4, dgx.DGX_LSRK14])
def test_one_step_matches_the_oracle(eqn, p, nx, ny, inttype):
    print(f"[quad stage] eqn={eqn} p={p} {nx}x{ny} inttype={inttype}", flush=True)
    m = meshgen.periodic_quads(nx, ny, 0.0, 2 * np.pi, 0.0, 2 * np.pi)
    orc = Oracle(m, p, eqn)
    orc.set_balance(False)
    orc.set_state(_state(orc.coords(), eqn))
    orc.project_state()
    gpu = dgx.GPUDomain(m, p, eqn, balance=False)
    gpu.upload(orc.state())
    dt = 0.1 * (2 * np.pi / max(nx, ny)) / ((p + 1) ** 2 * 2.0)
    orc.advance(inttype, dt, 1)
    gpu.advance(inttype, dt, 1)
    U, ref = gpu.download(), orc.state()
    gpu.close()
    err = np.sqrt(((U - ref) ** 2).sum((1, 2)) / (ref ** 2).sum((1, 2)))
    print(f"[quad stage] rel L2 per field: {err}", flush=True)
    assert np.all(err <= TOL), err


def test_a_residual_between_stages_leaves_the_step_unchanged():
    """dgx_rhs between dgx_stage calls takes the traces of the step's state; the
    next stage must not use them for its own intermediate state (TVD-RK3 keeps
    nothing else that dgx_rhs writes)."""
    m = meshgen.periodic_quads(4, 3, 0.0, 2 * np.pi, 0.0, 2 * np.pi)
    out = []
    for between in (False, True):
        g = dgx.GPUDomain(m, 4, dgx.DGX_EULER)
        g.upload(_state(g.coords(), dgx.DGX_EULER))
        for st in range(3):
            g.stage(dgx.DGX_TVD, st, 1e-2)
            if between:
                g.rhs()
        out.append(g.download(dgx.DGX_MODAL))
        g.close()
    assert np.array_equal(out[0], out[1])


@pytest.mark.parametrize("precision", [dgx.DGX_FP64, dgx.DGX_MIXED])
@pytest.mark.parametrize("p,n", [(2, 64), (3, 64), (4, 91)])
def test_served_results_do_not_depend_on_packing(p, n, precision):
    """A small request alone runs one element per wavefront, beside a large one
    several: the same bits."""
    def job(k, eqn):
        m = meshgen.periodic_quads(k, k, 0.0, 2 * np.pi, 0.0, 2 * np.pi)
        U = _state(meshgen.quad_nodes(m, p), eqn)
        return dict(mesh=m, p=p, eqntype=eqn, U0=U, inttype=dgx.DGX_LSRK14, dt=1e-3 / k, nsteps=3,
                    precision=precision, balance=False)

    for eqn in (dgx.DGX_EULER, dgx.DGX_SHALLOW):
        print(f"[quad stage] served p={p} eqn={eqn} precision={precision}", flush=True)
        got = []
        for sizes in ((7,), (7, n)):
            srv = serve.Server(hbm_budget=1 << 34, max_active=4)
            ids = [srv.submit(**job(k, eqn)) for k in sizes]
            srv.run_until_done(timeout_s=60.0)
            got.append(srv.result(ids[0])[0])
            srv.close()
        assert np.array_equal(got[0], got[1])
