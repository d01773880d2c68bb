"""Linked blocks beside the matrix-core MRT."""
from __future__ import annotations

import numpy as np
import pytest

from agal_amd import capi
from agal_amd.mesh import LbmMesh
from parity import body, sphere_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vs,prec", [(capi.D3Q27, capi.FP32), (capi.D3Q19, capi.FP32), (capi.D3Q27, capi.FP16)])
def test_linked_blocks_keep_the_vector_operator(vs, prec):
    """One finest sub-step without and with AGAL_OPT_MRT_MFMA from the same flow, no force due: the rest
    populations, which no link moves, are the same bits in the linked blocks and not everywhere else."""
    p = sphere_params(vs=vs, N=16, levels=3, prec=prec, collision=capi.MRT, D=0.16, G_BIN_MAKE_LINKS=1,
                      G_BIN_DENSITY=4, G_BIN_LEVELS=3, G_BIN_SPEC=1, S_BC_TYPE=0, S_FORCE_TYPE=0, S_FORCE_ORDER=1)
    rest = []
    for mfma in (0, 1):
        m = LbmMesh(p, 20000)
        m.set_geometry(body(center=(0.3, 0.5, 0.5), radius=0.08, subdivisions=3, noise=0.0, seed=1))
        assert m.M_Advance_RefineNearWall() == capi.AGAL_OK
        m.advance_loop(0, 6)
        m.set_option(capi.OPT_MRT_MFMA, mfma)
        m.collide_stream(2)
        ids, rank = m.id_set(2), m.links()["onb_solid"]
        f0 = m.populations()[0].reshape(-1, 64)
        linked = rank[ids] >= 0
        assert linked.sum() > 10 and (~linked).sum() > 50
        rest.append((f0[ids[linked]], f0[ids[~linked]]))
        m.close()
    np.testing.assert_array_equal(rest[0][0], rest[1][0])
    assert (rest[0][1] != rest[1][1]).any()
