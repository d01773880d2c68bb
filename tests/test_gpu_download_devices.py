"""Large downloads with another GPU current than the context's."""
from __future__ import annotations

from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import torch

from agal_amd import capi
from agal_amd.mesh import LbmMesh
from parity import ldc_params

pytestmark = pytest.mark.gpu


def test_large_download_leaves_the_current_gpu():
    """The calling thread's current GPU is the same after a download in pieces."""
    m = LbmMesh(ldc_params(vs=capi.D3Q19, N=64, levels=1), 4608)
    m.S_SetIC(0)
    m.S_RefreshVariables(0)
    before = torch.cuda.current_device()
    assert m.macros(4608).nbytes >= 4 << 20 and torch.cuda.current_device() == before
    m.close()


@pytest.mark.skipif(torch.cuda.device_count() < 2, reason="needs two GPUs")
def test_large_download_with_another_gpu_current():
    """A context on GPU 1; the call comes from a thread whose current GPU is 0."""
    m = LbmMesh(ldc_params(vs=capi.D3Q19, N=64, levels=1), 4608, device=1)
    m.S_SetIC(0)
    m.S_RefreshVariables(0)
    m.sync()
    ref = m.macros(512)

    def fetch():
        torch.cuda.set_device(0)
        out = m.macros(4608)
        return out, torch.cuda.current_device()

    with ThreadPoolExecutor(1) as pool:
        out, dev = pool.submit(fetch).result()
    assert dev == 0
    np.testing.assert_array_equal(out[:, :64 * 512], ref)
    m.close()
