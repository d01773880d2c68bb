"""Advance from a level below the root, against the CPU restatement."""
from __future__ import annotations

import numpy as np
import pytest

from agal_amd import capi
from agal_amd.mesh import LbmMesh
from oracle_lib import OracleMesh
from parity import compare_states, ldc_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vs,N,levels", [(capi.D3Q19, 16, 2), (capi.D3Q19, 16, 3), (capi.D2Q9, 32, 3)])
@pytest.mark.parametrize("guard", [False, True])
def test_advance_from_every_level(vs, N, levels, guard):
    """One coarse step of level L0 is two sub-steps of every level above the root, the finest included
    (solver_lbm_advance.cu:86-122); `guard`: with many links that fail the swap guard."""
    p = ldc_params(vs=vs, N=N, Re=40.0, levels=levels, P_REFINE=1 << 28)
    g, o = LbmMesh(p, 4096), OracleMesh(p, 4096)
    for m in (g, o):
        m.S_SetIC(0)
        for L in range(levels - 1):
            ids = m.id_set(L)
            m.mark_blocks(ids[m.coords()[0, ids] < 0.3 / (L + 1)], capi.REF_MARK_REFINE)
            m.M_RefineAndCoarsenBlocks()
        m.advance_loop(0, 2)
    if guard:
        f = o.populations()
        f = f * (1.0 + 1.5 * np.random.default_rng(7).standard_normal(f.shape).astype(f.dtype))
        for m in (g, o):
            m.set_populations(f)
    for L0 in (levels - 1, 0, 1, levels - 1, levels - 1, 0):
        for m in (g, o):
            m.S_Advance(L0)
        g.sync()
        bad = compare_states(g.state(), o.state())
        assert not bad, f"from level {L0}: " + "\n".join(bad)
    g.close()
