"""Device memory that handles hold and leave behind."""
import gc

import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu


def _handle(nbf, naux, ncol=0):
    from psi4_amd.core import JK
    jk = JK.build_tensor(nbf, naux)
    jk.set_print(0)
    jk.initialize()
    if ncol:
        jk.fill_synthetic(1)
        jk.C_left_add(np.random.default_rng(0).standard_normal((nbf, ncol)))
        jk.compute()
    return jk


def _free():
    import torch
    return torch.cuda.mem_get_info()[0]


def test_small_handles_are_small(gpu_available):
    """64 handles of 8 functions, a build each.  A build of host arrays keeps 9 workspace arrays of 256 KiB, 8 tables and B
    (below 0.2 MiB together): 2.5 MiB, so 4 MiB leave room for the allocator's own granularity."""
    from psi4_amd.core import trim_memory
    announce("64 handles of 8 functions")
    first = _handle(8, 8, 2)
    gc.collect()
    trim_memory()
    before = _free()
    held = [_handle(8, 8, 2) for _ in range(64)]
    each = (before - _free()) / len(held) / 2 ** 20
    print(f"  {each:.2f} MiB per handle", flush=True)
    assert each < 4.0
    del first, held
