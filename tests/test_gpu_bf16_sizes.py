"""BF16x3 J and K of small tensor handles at the edges of the kernels' tiles against numpy in FP64 on the same tensor:
1 to 6 column tiles of 32 (the half-transform's steps, odd and even), row blocks of 128 with every number of valid
fragments, column counts around 32 and 320, every pair form, a partial auxiliary range and more than 64 column tiles.

Tolerance, first order, on the same sums over absolute values.  A value is split into BF16 hi = RNE(x) and
lo = RNE(x - hi), so |x - hi| <= 2^-9 |x| and |x - hi - lo| <= 2^-18 |x|; of a product, lo lo and the two
remainders are missing: 3 * 2^-18.  FP32 roundings of B and C, 2^-24 each.  Additions in the matrix unit, three per
product: 2^-23 each (2^-24 rounded; the unit may cut off instead) - nbf terms in X, at most 512 and one step of
32 in a sum of K before it is folded, then the folds of a sum in FP32.  J: the FP32 copy of B in two uses, FP64 sums.
1 % for the second order.
"""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

U, UM, EPS = 2.0 ** -24, 2.0 ** -23, 2.0 ** -53
SPLIT = 3 * 2.0 ** -18


def _tensor(nbf, naux, seed):
    from psi4_amd.core import JK, PREC_BF16X3
    jk = JK.build_tensor(nbf, naux)
    jk.set_print(0)
    jk.initialize()
    jk.fill_synthetic(seed)
    jk.set_precision(PREC_BF16X3)
    return jk, jk.get_B_dense(0, naux)


def _check(jk, B, L, R):
    naux, nbf, _ = B.shape
    ncol = L.shape[1]
    jk.C_clear()
    jk.C_left_add(L)
    if R is not L:
        jk.C_right_add(R)
    jk.compute()

    def sums(B, L, R):
        d = np.einsum("qmn,mn->q", B, L @ R.T)
        return np.einsum("q,qmn->mn", d, B), np.einsum("qmi,qni->mn", B @ L, B @ R, optimize=True)

    Jo, Ko = sums(B, L, R)
    Ja, Ka = sums(np.abs(B), np.abs(L), np.abs(R))
    D, J, K = jk.D()[0], jk.J()[0], jk.K()[0]
    assert np.all(np.abs(D - L @ R.T) <= 2 * (ncol + 1) * EPS * (np.abs(L) @ np.abs(R).T))
    assert np.all(np.abs(J - Jo) <= 1.01 * (2 * U + 2 * (nbf * nbf + naux + ncol + 2) * EPS) * Ja)
    terms = naux * (ncol + 31)
    x = SPLIT + 2 * U + 3 * nbf * UM
    k = SPLIT + (3 * min(512 + 32, terms) + terms // 512 + 2) * UM
    assert np.all(np.abs(K - Ko) <= 1.01 * (2 * x + k + 2 * terms * EPS) * Ka)
    return K


@pytest.mark.parametrize("nbf,naux", [(1, 1), (32, 3), (33, 9), (65, 17), (97, 8), (128, 5), (129, 41), (190, 70)])
def test_symmetric_sizes(gpu_available, nbf, naux):
    announce(f"BF16x3 symmetric pairs, nbf {nbf} naux {naux}")
    jk, B = _tensor(nbf, naux, 7)
    rng = np.random.default_rng(nbf)
    for ncol in (1, 2, 32, 33, 82, 330):
        C = rng.standard_normal((nbf, ncol))
        K = _check(jk, B, C, C)
        assert np.array_equal(K, K.T)


@pytest.mark.parametrize("nbf,naux", [(1, 2), (33, 5), (65, 20), (97, 33), (129, 12), (161, 7)])
@pytest.mark.parametrize("ncol", [2, 18, 82, 330])
def test_pair_forms(gpu_available, nbf, naux, ncol):
    announce(f"BF16x3 general, cross and signed pairs, nbf {nbf} naux {naux} columns {ncol}")
    jk, B = _tensor(nbf, naux, 8)
    rng = np.random.default_rng(ncol)
    L, R = rng.standard_normal((2, nbf, ncol))
    _check(jk, B, L, R)
    A, V = rng.standard_normal((2, nbf, ncol // 2))
    K = _check(jk, B, np.hstack([A, V]), np.hstack([V, A]))
    assert np.array_equal(K, K.T)
    for s in (np.where(np.arange(ncol) % 3 == 1, -1.0, 1.0), -np.ones(ncol)):
        K = _check(jk, B, L, L * s)
        assert np.array_equal(K, K.T)


def test_partial_auxiliary_range(gpu_available):
    nbf, naux = 66, 50
    announce("BF16x3, auxiliary range 7..31 of 50")
    jk, B = _tensor(nbf, naux, 10)
    C = np.random.default_rng(4).standard_normal((nbf, 20))
    jk.set_aux_range(7, 31)
    _check(jk, B[7:31], C, C)


def test_more_than_64_column_tiles(gpu_available):
    """nbf 2100 is 66 column tiles: the step list's entries come from more than one wave."""
    announce("nbf 2100 naux 2, BF16x3")
    jk, B = _tensor(2100, 2, 12)
    C = np.random.default_rng(5).standard_normal((2100, 3))
    _check(jk, B, C, C)
