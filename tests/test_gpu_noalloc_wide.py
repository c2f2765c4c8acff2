"""dfjk_compute_device_noalloc, a general pair with several times as many columns as functions, near the end of the
scratch array: both sides' operands and X do not fit it at once, and the sides are transformed one after the
other.  Against numpy on the same tensor.

Tolerance: the bound of the rounding of sums of n terms, n * 2^-53 on the same sums of absolute values, once for the
device and once for numpy.
"""
import numpy as np
import pytest

from conftest import announce
from test_zz_no_alloc import _call, _lib

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53


def _ref(B, L, R):
    naux, nbf, _ = B.shape
    d = np.einsum("qmn,mn->q", B, L @ R.T)
    K = np.zeros((nbf, nbf))
    for b in B:
        K += (b @ L) @ (b @ R).T
    return np.einsum("q,qmn->mn", d, B), K


@pytest.mark.parametrize("nbf,naux,ncol", [(373, 16, 6653), (580, 7, 4299), (736, 5, 3433), (289, 1, 8118)])
def test_more_columns_than_functions(gpu_available, nbf, naux, ncol):
    from psi4_amd.core import JK
    announce(f"noalloc, general pair: nbf {nbf}, naux {naux}, {ncol} columns")
    jk = JK.build_tensor(nbf, naux)
    jk.set_print(0)
    jk.initialize()
    jk.fill_synthetic(11)
    B = jk.get_B_dense(0, naux)
    rng = np.random.default_rng(nbf)
    L, R = rng.standard_normal((nbf, ncol)), rng.standard_normal((nbf, ncol))
    D, J, K = _call(_lib(), "dfjk_compute_device_noalloc", jk.handle(), L, R)
    Jo, Ko = _ref(B, L, R)
    Ja, Ka = _ref(np.abs(B), np.abs(L), np.abs(R))
    assert np.all(np.abs(D - L @ R.T) <= 2 * (ncol + 1) * EPS * (np.abs(L) @ np.abs(R).T))
    assert np.all(np.abs(J - Jo) <= 2 * (nbf * nbf + naux + ncol + 2) * EPS * Ja)
    assert np.all(np.abs(K - Ko) <= 2 * (2 * nbf + naux * ncol + 3) * EPS * Ka)
