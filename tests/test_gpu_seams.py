"""The step, vField and optimisation seams through the C ABI on the GPU.

* dgx_stage: running the stages of a step one call at a time is bitwise the
  same as dgx_advance (LSRK14 fused and unfused, RK4, TVD-RK3), and the stage
  order is enforced.
* dgx_vfield_sizes: vField::size/qtot/nmodes/ndof/sdof/nsd of the state
  (src/vField.hpp:330-376) for quads and hexes, through the pydgm mirror.
* ReoOptProblem over the acoustic problem: computeState / computeAdjoint /
  getGradient agree with the direct entry points, and a few descent steps
  lower the objective.
"""
import ctypes

import numpy as np
import pytest

from dgm_amd import dgx, ic, mesh as meshgen
from dgm_amd import problem as dgm

pytestmark = pytest.mark.gpu


def _tgv_domain(p=3, eqn=9, **kw):
    m = meshgen.periodic_hexes(2, 2, 2, (0, 0, 0), (2 * np.pi,) * 3)
    d = dgx.GPUDomain(m, p, eqn, vis=0.01 if eqn == 9 else 0.0, **kw)
    x = d.coords()
    U = ic.taylor_green(x[0], x[1], x[2])
    U[1:4] *= 1.0 + 0.02 * np.sin(x[0] + 2 * x[1])
    d.upload(U)
    return d


@pytest.mark.parametrize("inttype,eqn,kw", [(14, 9, {}), (14, 9, {"bulk_forcing": True}), (4, 8, {}), (3, 9, {})])
def test_stages_equal_advance(inttype, eqn, kw):
    print(f"[stage] inttype={inttype} eqn={eqn} {kw}", flush=True)
    a, b = _tgv_domain(eqn=eqn, **kw), _tgv_domain(eqn=eqn, **kw)
    dt, ns = 1e-3, {3: 3, 4: 4, 14: 14}[inttype]
    a.advance(inttype, dt, 2)
    for _ in range(2):
        for s in range(ns):
            b.stage(inttype, s, dt)
    a.synchronize()
    b.synchronize()
    assert np.array_equal(a.download(dgx.DGX_MODAL), b.download(dgx.DGX_MODAL))
    assert a.time == b.time and a.stage_count == b.stage_count
    a.close()
    b.close()


def _write_state(d, U):
    """U into the domain's modal state through its device pointer."""
    hip = ctypes.CDLL("libamdhip64.so.7")
    U = np.ascontiguousarray(U)
    rc = hip.hipMemcpy(ctypes.c_void_p(d.device_state_ptr()), U.ctypes.data_as(ctypes.c_void_p),
                       ctypes.c_size_t(U.nbytes), ctypes.c_int(1))   # hipMemcpyHostToDevice
    assert rc == 0, rc


def _stage_domain(kind):
    if kind == "quads":
        d = dgx.GPUDomain(meshgen.periodic_quads(4, 3, 0.0, 2 * np.pi, 0.0, 2 * np.pi), 4, 1)
        x = d.coords()
        s = [np.sin(x[0] + 0.3 * k) * np.cos(x[1]) for k in range(4)]
        d.upload(np.stack([1.0 + 0.1 * s[0], 0.3 + 0.1 * s[1], 0.1 * s[2], 2.5 + 0.1 * s[3]]))
        return d
    if kind == "curved hexes":
        m = meshgen.periodic_hexes(2, 2, 2, (0, 0, 0), (2 * np.pi,) * 3)
        bend = lambda x, y, z: (x, y + 0.1 * np.sin(x), z + 0.1 * np.sin(y))   # noqa: E731
        return _tgv_domain(eqn=8, xnodes=meshgen.mapped_nodes(m, 3, bend))
    return _tgv_domain(precision=dgx.DGX_MIXED if kind == "mixed hexes" else dgx.DGX_FP64)


@pytest.mark.parametrize("inttype", [dgx.DGX_TVD, dgx.DGX_LSRK14])
@pytest.mark.parametrize("kind", ["quads", "hexes", "mixed hexes", "curved hexes"])
def test_a_state_written_between_stages_is_the_next_stages_state(kind, inttype):
    """A filter between dgx_stage calls, through the state's device pointer and
    through dgx_state_upload: the same bits (a stage that kept the face
    traces of the state before the filter would differ by the filter's own
    size)."""
    print(f"[stage] filter between stages, {kind}, inttype={inttype}", flush=True)
    out = []
    for by_pointer in (True, False):
        d = _stage_domain(kind)
        keep = np.ones(d.nm)
        keep[-1] = 0.5
        keep[1] = 0.9
        for st in range(3 if inttype == dgx.DGX_TVD else 14):
            d.stage(inttype, st, 1e-3)
            d.synchronize()
            U = d.download(dgx.DGX_MODAL) * keep
            if by_pointer:
                _write_state(d, U)
            else:
                d.upload(U, dgx.DGX_MODAL)
        out.append(d.download(dgx.DGX_MODAL))
        d.close()
    assert np.array_equal(out[0], out[1]), np.abs(out[0] - out[1]).max()


def test_stage_order_is_enforced():
    d = _tgv_domain()
    with pytest.raises(dgx.DgxError):
        d.stage(14, 1, 1e-3)                 # a step starts at stage 0
    d.stage(14, 0, 1e-3)
    with pytest.raises(dgx.DgxError):
        d.advance(14, 1e-3, 1)               # the begun step is unfinished
    with pytest.raises(dgx.DgxError):
        d.stage(4, 1, 1e-3)                  # same integrator through the step
    for s in range(1, 14):
        d.stage(14, s, 1e-3)
    d.advance(14, 1e-3, 1)
    d.synchronize()
    d.close()


def test_vfield_sizes():
    for m, p, eqn, nf, nq, nm, ns, qs in (
            (meshgen.periodic_quads(3, 2), 4, 1, 4, 36, 25, 4, 5),
            (meshgen.periodic_hexes(2, 2, 3), 3, 8, 5, 125, 64, 6, 16),
            (meshgen.periodic_quads(2, 2), 2, 30, 3, 16, 9, 4, 3)):
        d = dgx.GPUDomain(m, p, eqn, balance=False)
        v = dgm.vField(d)
        ne = m.ne
        assert v.size() == nf and v.nsd() == m.nsd
        assert v.qtot() == nf * ne * nq and v.nmodes() == v.ndof() == nf * ne * nm
        assert v.sdof() == nf * ne * ns * qs
        assert v.numpy().shape == (nf, ne, nq)
        v.zero()
        assert not np.any(v.numpy(dgx.DGX_MODAL))
        d.close()


def test_opt_problem_seam():
    from dgm_amd.acoustic import AcousticProblem, ReoOptProblem
    m = meshgen.periodic_quads(8, 8, 0.0, 1.0, 0.0, 1.0)
    rng = np.random.default_rng(4)
    rec = rng.uniform(0.1, 0.9, (4, 2))
    prob = AcousticProblem(m, 3, (1.0, 0.2, 0.0, 1.0 / 1.4), rec, 8.0, 0.12, 2e-3, 120)
    true = rng.standard_normal(m.ne)
    data = prob.forward(true)
    opt = ReoOptProblem(prob, data)
    J0 = opt.computeState()
    opt.computeAdjoint()
    Jd, gd = prob.gradient(opt.getControl(), data)
    assert abs(J0 - Jd) <= 1e-13 * Jd and np.array_equal(opt.getGradient(), gd)
    J3 = opt.solve(iterations=3, step=1.0 / max(1e-300, float(np.abs(gd).max())))
    assert J3 < J0
    prob.close()
