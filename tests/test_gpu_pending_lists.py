"""The stream guard's exception lists on refined meshes: which launch resolves them, and which records into
them, against the CPU restatement."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

from agal_amd import capi
from agal_amd.mesh import LbmMesh
from oracle_lib import OracleMesh
from parity import compare_states, ldc_params

pytestmark = pytest.mark.gpu

SETS = [(capi.D3Q19, capi.FP32, capi.BGK, 1.5), (capi.D3Q19, capi.FP16, capi.BGK, 0.35), (capi.D3Q27, capi.FP64, capi.MRT, 1.0)]


def _refined_pair(vs, prec, coll, N, x_max, solid):
    """The same three-level mesh in both contexts: blocks of level L left of x_max / (L + 1) refined; with
    `solid`, two cells of the finest level turned solid, which keeps its sub-steps out of the in-place form."""
    p = ldc_params(vs=vs, N=N, Re=40.0, levels=3, P_REFINE=1 << 28, prec=prec, collision=coll)
    p.L_fy = p.L_fz = 0.5
    g, o = LbmMesh(p, 16384), OracleMesh(p, 16384)  # lists of 2^20 entries
    for m in (g, o):
        m.S_SetIC(0)
        for L in range(2):
            ids = m.id_set(L)
            m.mark_blocks(ids[m.coords()[0, ids] < x_max / (L + 1)], capi.REF_MARK_REFINE)
            m.M_RefineAndCoarsenBlocks()
    if solid:
        mask, nb = o.cell_masks(), g.n_blocks()
        ids = o.id_set(2)
        mask[64 * ids[len(ids) // 3] + 21] = mask[64 * ids[len(ids) // 2] + 63] = capi.CELL_SOLID
        g._call("upload_cell_masks", capi.np_ptr(mask, ctypes.c_int), nb)
        o.set_cell_masks(mask)
    return g, o


def _perturb(g, o, amp):
    f = o.populations()
    f = f * (1.0 + amp * np.random.default_rng(5).standard_normal(f.shape).astype(f.dtype))
    g.set_populations(f)
    o.set_populations(f)


def _step_and_compare(g, o, calls):
    i = 0
    for n in calls:
        for m in (g, o):
            m.advance_loop(i, n)
        i += n
        g.sync()
        assert np.isfinite(o.populations()).all()
        bad = compare_states(g.state(), o.state())
        assert not bad, f"after {i} steps: " + "\n".join(bad)


@pytest.mark.parametrize("vs,prec,coll,amp", SETS)
@pytest.mark.parametrize("graphs", [1, 0])
def test_finest_pairs_under_a_wholly_refined_level(vs, prec, coll, amp, graphs):
    """Every block refined twice: no interface blocks, so nothing is averaged and no kernel lies between the
    second sub-step of a finest pair, which leaves its list pending, and the first of the next, which
    records into the extra list that is emptied with it.  40 workgroups a launch."""
    g, o = _refined_pair(vs, prec, coll, 8, 9.0, True)
    assert list(g.sizes.n_ids)[:3] == [2, 16, 128] and not g.block_ints(capi.BLK_MASK)[g.id_set(1)].any()
    g.set_option(capi.OPT_GRAPHS, graphs)
    _perturb(g, o, amp)
    _step_and_compare(g, o, (1, 2, 1))
    g.close()


@pytest.mark.parametrize("lv", [2, 7, 8, 9, 40, 1 << 29, (1 << 31) - 1, -1, -(1 << 31)])
def test_a_block_of_no_level_is_in_no_list(lv):
    """An uploaded block table may hold any level.  A block whose level is none of the mesh's is left out of
    every list: the averages and interpolations of the others are the restatement's, and with its level
    back the mesh steps as if nothing had been."""
    p = ldc_params(vs=capi.D3Q19, N=16, Re=40.0, levels=2, P_REFINE=1 << 28)
    g, o, q = LbmMesh(p, 1024), OracleMesh(p, 1024), OracleMesh(p, 1024)
    for m in (g, o):
        m.S_SetIC(0)
        ids = m.id_set(0)
        m.mark_blocks(ids[m.coords()[0, ids] < 0.3], capi.REF_MARK_REFINE)
        m.M_RefineAndCoarsenBlocks()
        m.advance_loop(0, 3)
    st = o.state()
    fine = st["id_sets"][1]
    level, b = st["level"].copy(), int(fine[len(fine) // 2])
    level[b] = lv
    g.set_block_ints(capi.BLK_LEVEL, level)
    sets = [st["id_sets"][0], fine[fine != b]]
    assert [g.id_set(L).tolist() for L in range(2)] == [s.tolist() for s in sets]
    q.import_state(dict(st, level=level, id_sets=sets, n_ids=[len(s) for s in sets]))
    for m in (g, q):
        m.S_Interpolate(0, capi.INTERP_INTERFACE)
        m.S_Average(0, capi.AVERAGE_INTERFACE)
    cells = (64 * np.concatenate(sets)[:, None] + np.arange(64)).ravel()
    np.testing.assert_array_equal(g.populations(st["id_max"])[:, cells], q.populations(st["id_max"])[:, cells])
    g.set_block_ints(capi.BLK_LEVEL, st["level"])
    g.set_populations(st["f"])
    for m in (g, o):
        m.advance_loop(3, 3)
    bad = compare_states(g.state(), o.state())
    assert not bad, "\n".join(bad)
    g.close()


@pytest.mark.parametrize("vs,prec,coll,amp", SETS)
@pytest.mark.parametrize("N,x_max,solid", [(16, 0.3, True), (16, 0.3, False), (16, 9.0, True)])
def test_finest_pairs_with_failed_links(vs, prec, coll, amp, N, x_max, solid):
    """Many failed links on every level.  With solid cells on the finest level its pairs are push pairs: the
    first sub-step links its entries per block and flags the blocks, the second applies them as it loads; 256
    blocks in launches that resolve what is pending themselves, and 1024 blocks, whose launches leave that to
    a fixup launch.  Without solid cells 256 blocks step in place, and the second sub-step resolves the first
    one's list."""
    g, o = _refined_pair(vs, prec, coll, N, x_max, solid)
    assert int(g.sizes.n_ids[2]) == (256 if x_max < 1 else 1024)
    _perturb(g, o, amp)
    _step_and_compare(g, o, (1, 2, 1))
    g.close()
