"""Kernels at the sizes where they can go wrong: remainders of their tiles, the smallest and largest
of their ranges, against the CPU restatement."""
from __future__ import annotations

import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import torch

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


def _perturbed(m, o, seed):
    """The same populations in both contexts, many of them non-positive."""
    f = o.populations()
    f = f * (1.0 + 1.5 * np.random.default_rng(seed).standard_normal(f.shape).astype(f.dtype))
    m.set_populations(f)
    o.set_populations(f)


@pytest.mark.parametrize("vs,prec,coll", [(capi.D3Q19, capi.FP32, capi.BGK), (capi.D3Q19, capi.FP64, capi.MRT),
                                          (capi.D3Q27, capi.FP16, capi.MRT), (capi.D3Q27, capi.BF16, capi.BGK)])
@pytest.mark.parametrize("periodic", [0, 1])
def test_in_place_pairs_on_one_level(vs, prec, coll, periodic):
    """One to nine steps in one call (in-place pairs, an odd one out, several recorded graphs) on a root
    grid of unequal sides, two blocks wide along z, with lid or periodic faces, from populations that
    fail the swap guard in many links: the exchange before each second sub-step and the fixups after
    it, bit for bit."""
    p = ldc_params(vs=vs, N=16, Re=20.0, levels=1, prec=prec, collision=coll)
    p.L_fy, p.L_fz = 0.75, 0.5
    p.PERIODIC_X = p.PERIODIC_Z = periodic
    g, o = LbmMesh(p, 1024), OracleMesh(p, 1024)  # lists of 65 536 entries
    for m in (g, o):
        m.S_SetIC(0)
    _perturbed(g, o, 11)
    i = 0
    for n in (1, 2, 3, 4, 9):
        for m in (g, o):
            m.advance_loop(i, n)
        i += n
        bad = compare_states(g.state(), o.state())
        assert not bad, f"after {n}: " + "\n".join(bad)
    g.close()


def test_pairs_leave_a_level_with_solid_cells_to_the_general_path():
    """A cell turned solid makes its neighbourhood general: the level's sub-steps then run one by one,
    and again in place once the cell is fluid."""
    p = ldc_params(vs=capi.D3Q19, N=16, Re=20.0, levels=1, prec=capi.FP32)
    g, o = LbmMesh(p, 128), OracleMesh(p, 128)
    for m in (g, o):
        m.S_SetIC(0)
        m.advance_loop(0, 4)
    mask = o.cell_masks()
    for solid in (True, False):
        mask[64 * 21 + 27] = capi.CELL_SOLID if solid else capi.CELL_INTERIOR
        nb = g.n_blocks()
        g._call("upload_cell_masks", capi.np_ptr(np.ascontiguousarray(mask[: 64 * nb]), ctypes.c_int), nb)
        o.set_cell_masks(mask[: 64 * nb])
        for m in (g, o):
            m.advance_loop(4 if solid else 10, 6)
        bad = compare_states(g.state(), o.state())
        assert not bad, f"solid {solid}: " + "\n".join(bad)
    g.close()


@pytest.mark.parametrize("vs,prec", [(capi.D2Q9, capi.FP32), (capi.D3Q19, capi.FP32)])
def test_pending_lists_resolved_by_the_next_kernel(vs, prec):
    """Guard failures on every level of a refined mesh: each kernel of the coarse step (fused step,
    in-place second sub-step, average, average + interpolation) finds lists to resolve, with several
    workgroups waiting for the one that does."""
    p = ldc_params(vs=vs, N=32 if vs == capi.D2Q9 else 16, Re=40.0, levels=3, P_REFINE=1 << 28, prec=prec)
    g, o = LbmMesh(p, 4096), OracleMesh(p, 4096)
    for m in (g, o):
        m.S_SetIC(0)
        for L in range(2):
            ids = m.id_set(L)
            m.mark_blocks(ids[m.coords()[0, ids] < 0.3 / (L + 1)], capi.REF_MARK_REFINE)
            m.M_RefineAndCoarsenBlocks()
    assert g.refresh_sizes().n_ids[2] > 0
    _perturbed(g, o, 5)
    for i in range(3):
        for m in (g, o):
            m.advance_loop(2 * i, 2)
        bad = compare_states(g.state(), o.state())
        assert not bad, "\n".join(bad)
    g.close()


@pytest.mark.parametrize("vs,prec,N,nb", [(capi.D3Q19, capi.FP32, 60, 4095), (capi.D3Q19, capi.FP32, 60, 4096),
                                          (capi.D3Q27, capi.FP64, 76, 8200), (capi.D2Q9, capi.FP16, 508, 16385)])
def test_large_downloads_in_pieces(vs, prec, N, nb):
    """Macroscopic fields and populations around the line between a direct copy and pinned pieces (4 MB),
    and rows that end within a piece: into pageable memory with a gap between the rows, into pinned memory
    (copied directly), and from two threads at once.  All must hold the same bytes; the gaps stay as they
    were."""
    m = LbmMesh(ldc_params(vs=vs, N=N, Re=40.0, levels=1, prec=prec), nb)
    q, nc = m.sizes.n_q, nb * m.sizes.cells_per_block
    m.set_populations(np.random.default_rng(nb).uniform(0.5 / q, 1.5 / q, (q, nc)))
    m.S_RefreshVariables(0)
    for what, rows in (("download_macros", 4), ("download_populations", q)):
        pinned = torch.full((rows, nc), -7.0, dtype=torch.float64 if m.dtype == np.float64 else torch.float32, pin_memory=True)
        m._call(what, capi.np_ptr(pinned.numpy()), nb, nc)
        ref = pinned.numpy().view(np.uint8)
        assert ref.any()

        def check():
            out = np.full((rows, nc + 3), -7, dtype=m.dtype)
            m._call(what, capi.np_ptr(out), nb, nc + 3)
            return np.array_equal(out[:, :nc].copy().view(np.uint8), ref) and bool((out[:, nc:] == -7).all())

        assert check()
        with ThreadPoolExecutor(2) as pool:
            assert all(f.result() for f in [pool.submit(check) for _ in range(4)])
    m.close()
