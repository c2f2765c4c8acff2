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


def test_the_pool_keeps_to_its_setting(gpu_available):
    """A handle with 0.5 GiB of B leaves it behind for the next one by default, and nothing with a pool of 0 bytes."""
    from psi4_amd.core import set_memory_pool, trim_memory
    announce("a finished handle of 0.5 GiB, pool of 0 bytes and by default")
    gc.collect()
    trim_memory()
    size = 68 * 990 * 8192             # naux x tile pairs of 44 x 32 functions x 8 KiB
    try:
        for pool, kept in ((0, False), (12 << 30, True)):
            set_memory_pool(pool)
            before = _free()
            jk = _handle(44 * 32, 68)
            assert before - _free() > size
            del jk
            gc.collect()
            assert (before - _free() > size // 2) == kept
        set_memory_pool(1 << 20)       # what is held beyond a new bound goes back
        assert before - _free() < size // 2
    finally:
        set_memory_pool(12 << 30)


def test_the_pool_gives_way_on_a_full_card(gpu_available):
    """With about 16 GiB free, 3 GiB of a finished handle are more than an eighth of it and go back to the device."""
    import torch

    from psi4_amd.core import trim_memory
    announce("a finished handle of 3 GiB with 16 GiB free")
    gc.collect()
    trim_memory()
    torch.cuda.empty_cache()
    rest = _free() - (16 << 30)
    if rest < 0:
        pytest.skip("less than 16 GiB free on this device")
    fill = torch.empty(rest, dtype=torch.uint8, device="cuda")
    try:
        before = _free()
        jk = _handle(1408, 400)        # 44 x 45 / 2 tiles of 8 KiB per Q: 3.02 GiB
        assert before - _free() > 3 << 30
        del jk
        gc.collect()
        assert before - _free() < 1 << 30
    finally:
        del fill
        torch.cuda.empty_cache()


def test_two_threads_share_the_pools(gpu_available):
    """Handles made, used and dropped by two threads at once: memory, staging and side queues go from one to the other.
    Every build of every thread has to finish, whatever kind of error would stop it.  J against numpy at the
    rounding of its sums, on sums of absolute values."""
    import threading

    announce("two threads, six handles each")
    shapes = [(100, 90, 20), (61, 90, 20), (150, 70, 33), (24, 116, 5), (256, 250, 24), (97, 40, 8)]
    done, errors = [], []

    def work(t):
        try:
            for i in range(len(shapes)):
                nbf, naux, ncol = shapes[(i + 3 * t) % len(shapes)]
                jk = _handle(nbf, naux)
                jk.fill_synthetic(nbf)
                B = jk.get_B_dense(0, naux)
                C = np.random.default_rng(i).standard_normal((nbf, ncol))
                jk.C_left_add(C)
                jk.compute()
                flat, D = B.reshape(naux, -1), (C @ C.T).reshape(-1)
                Da = (np.abs(C) @ np.abs(C).T).reshape(-1)
                tol = 2 * (nbf * nbf + naux + ncol + 2) * 2.0 ** -53 * ((np.abs(flat) @ Da) @ np.abs(flat))
                assert np.all(np.abs(jk.J()[0].reshape(-1) - (flat @ D) @ flat) <= tol)
                done.append((t, i))
        except Exception as e:  # noqa: BLE001
            errors.append((t, repr(e)))

    threads = [threading.Thread(target=work, args=(t,)) for t in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors and sorted(done) == [(t, i) for t in range(2) for i in range(len(shapes))]
