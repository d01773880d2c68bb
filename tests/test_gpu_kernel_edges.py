"""Kernels at the sizes where they can go wrong: remainders of their tiles, the smallest and largest
of their ranges, against the CPU restatement."""
from __future__ import annotations

import numpy as np
import pytest

from agal_amd import capi
from agal_amd.mesh import LbmMesh
from oracle_lib import MlpOracle, OracleMesh
from parity import compare_states, ldc_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 63, 64, 65, 129, 4096, 16387])
def test_forward_and_gradients_at_the_edges_of_row_groups(n):
    """Rows around a wavefront's group of four, the gradient's blocks of 64 rows and its pairs of
    blocks, and more rows than one pass of the largest launch: logits bit for bit, the gradient to the
    float rounding of n-term sums, n 2^-24 of the sum of magnitudes (bounded by the tensor's maximum)."""
    p = ldc_params(vs=capi.D3Q19, N=16, Re=40.0, levels=2, P_REFINE=15, S_CRITERION=2, N_REFINE_START=-2.0)
    g = LbmMesh(p, 1024)
    g.predictor_init(5, n)
    w = g.predictor_params()
    rng = np.random.default_rng(n)
    x = rng.normal(0, 1, (n, 12)).astype(np.float32)
    y = (rng.uniform(size=n) < 0.3).astype(np.float32)
    o = MlpOracle(w)
    z, _ = g.predictor_forward(x)
    np.testing.assert_array_equal(z, o.forward(x))
    lg, lo = g.predictor_train_step(x, y), o.train_step(x, y, lr=1e-3, pos_weight=4.0)
    assert abs(lg - lo) <= 1e-5 * max(1.0, abs(lo))
    np.testing.assert_allclose(g.predictor_params(2), o.g, rtol=0, atol=max(1e-6, n * 2.0 ** -24) * np.abs(o.g).max())
    g.close()


@pytest.mark.parametrize("vs,prec", [(capi.D3Q27, capi.FP16), (capi.D3Q27, capi.FP64), (capi.D3Q19, capi.BF16)])
def test_cubic_interpolation_of_other_sets_and_storage(vs, prec):
    """The cubic kernel's lanes are dealt by the number of directions (two index groups for 27, three
    for 19): interface and new children of three levels, bit for bit."""
    p = ldc_params(vs=vs, N=16, Re=40.0, levels=3, P_REFINE=8, prec=prec, interp_order=capi.INTERP_CUBIC,
                   N_REFINE_START=-2)
    g, o = LbmMesh(p, 8192), OracleMesh(p, 8192)
    for m in (g, o):
        m.S_SetIC(0)
        m.advance_loop(0, 24)
    assert g.refresh_sizes().n_ids[1] > 0
    bad = compare_states(g.state(), o.state())
    assert not bad, "\n".join(bad)
