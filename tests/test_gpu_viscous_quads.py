"""Stages of affine Navier-Stokes quads."""
import os

import numpy as np
import pytest

from dgm_amd import dgx, mesh as meshgen

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "viscous_quads.npz")


@pytest.mark.parametrize("inttype,name", [(dgx.DGX_TVD, "tvd"), (dgx.DGX_RK4, "rk4")])
def test_steps_beyond_the_viscous_limit_keep_the_plain_sums(inttype, name):
    """Five steps beyond the viscous limit (nu (p + 1)^4 dt / h^2 = 4.7 at p = 10)
    multiply a difference in the last bit by up to 1e8 (TVD-RK3) and 1e10 (RK4),
    so a kernel that forms its sums in another order or from other halves of the
    tables is off by 1e-8 and more.  The stored states are those of plain
    ascending sums; 2e-12 is the bound that a well conditioned run keeps."""
    print(f"[viscous quads] beyond the limit, {name}", flush=True)
    g = np.load(GOLDEN)
    m = meshgen.periodic_quads(2, 2, 0.0, 2 * np.pi, 0.0, 2 * np.pi)
    gpu = dgx.GPUDomain(m, 10, dgx.DGX_NAVIER_STOKES, vis=1.6)
    gpu.upload(g["U0"], dgx.DGX_MODAL)
    gpu.advance(inttype, 2e-3, 5)
    U, ref = gpu.download(dgx.DGX_MODAL), g[name]
    gpu.close()
    err = np.sqrt(((U - ref) ** 2).sum((1, 2)) / (ref ** 2).sum((1, 2)))
    print(f"[viscous quads] rel L2 per field: {err}", flush=True)
    assert np.all(err <= 2e-12), err
