"""The element block's one-wavefront kernels at every mode count they are built
for (2 and 3 modes pack 7 and 4 elements per wavefront, 4 modes two), with
element counts that leave the last group partly empty: the bits of the oracle.
"""
import numpy as np
import pytest

from dgm_amd.hexblock import HexKernels
from oracle_lib import hexblock_backward_transform, hexblock_inner_product

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_element", [False, True])
@pytest.mark.parametrize("nm,ne", [(2, 1), (2, 13), (2, 14), (2, 15), (3, 3), (3, 8), (3, 9), (4, 1), (4, 5), (5, 3),
                                   (6, 4), (7, 65), (8, 2), (9, 33), (10, 7), (11, 3)])
def test_bits_of_the_oracle(nm, ne, per_element):
    print(f"[hexblock waves] nm={nm} ne={ne} per_element={per_element}", flush=True)
    q = nm + 1
    rng = np.random.default_rng(100 * nm + ne)
    B = [rng.standard_normal((nm, q)) for _ in range(3)]
    wJ = rng.uniform(0.5, 2.0, (ne if per_element else 1, q ** 3))
    u = rng.standard_normal((ne, q ** 3))
    hk = HexKernels().initialize(ne, nm, q, q, q)
    hk.Basis(*B)
    hk.wJ(wJ, per_element)
    got, back = u.copy(), u.copy()
    hk.inner_product(got)
    hk.backward_transform(back)
    hk.close()
    assert np.array_equal(got, hexblock_inner_product(u, *B, wJ, per_element))
    assert np.array_equal(back, hexblock_backward_transform(u, *B))
