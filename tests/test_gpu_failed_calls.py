"""Calls on host arrays that the library refuses after their operands were sent to the device (a declared cross form
with an odd number of columns)."""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

NBF, NAUX = 90, 40


def _handle():
    from psi4_amd.core import JK
    jk = JK.build_tensor(NBF, NAUX)
    jk.set_print(0)
    jk.initialize()
    jk.fill_synthetic(5)
    return jk


def _refused(jk, rng, ncol=601):
    jk.C_clear()
    jk.C_left_add(rng.standard_normal((NBF, ncol)))
    jk.C_right_add(rng.standard_normal((NBF, ncol)))
    jk.set_pair_form("CROSS")
    with pytest.raises(RuntimeError, match="even column count"):
        jk.compute()
    jk.set_pair_form("DETECT")


def test_the_call_after_a_refused_one(gpu_available):
    """The staging that a refused call filled serves the next call, and another handle's once this one is gone."""
    announce("refused host calls, each followed by a good one")
    jk = _handle()
    rng = np.random.default_rng(0)
    B = jk.get_B_dense(0, NAUX)
    for other in (False, False, True):
        _refused(jk, rng)
        if other:
            del jk
            jk = _handle()
        C = rng.standard_normal((NBF, 12))
        jk.C_clear()
        jk.C_left_add(C)
        jk.compute()
        d = np.einsum("qmn,mn->q", B, C @ C.T)
        # rounding of sums of at most nbf^2 + naux terms, on sums of absolute values
        a = np.einsum("qmn,mn->q", np.abs(B), np.abs(C) @ np.abs(C).T)
        tol = 2 * (NBF * NBF + NAUX + 14) * 2.0 ** -53 * np.einsum("q,qmn->mn", a, np.abs(B))
        assert np.all(np.abs(jk.J()[0] - np.einsum("q,qmn->mn", d, B)) <= tol)


def test_outputs_of_a_refused_call_are_zero(gpu_available):
    """J and K hold zeros after a refused call, not memory that nothing has written."""
    announce("J and K after a refused call")
    jk = _handle()
    rng = np.random.default_rng(1)
    for _ in range(3):
        jk.C_clear()
        jk.C_left_add(rng.standard_normal((NBF, 12)))
        jk.compute()               # results that the next arrays' memory may still hold
        assert jk.J()[0].any()
        _refused(jk, rng, 11)
        assert not jk.J()[0].any() and not jk.K()[0].any()
