"""J, K and the energy adjoint of a basis whose B lacks most tiles: seven waters in a row, 25 bohr apart, where only the
pairs of a water with itself survive the screening (nbf 168: 6 rows of 32 x 32 tiles, stored next to the
diagonal only).  A half-transform wave of two tile rows then meets columns where either row has no tile.
Against numpy on the device's own B, in every precision and pair form.

Tolerances: the first-order bounds on sums of absolute values of the tests at tile edges.  FP64: 2^-53 a term.  FP32:
2^-24 for each rounding of B and C and each term of a chain.  BF16x3: 3 * 2^-18 a product (the missing terms of the
split) and 2^-23 an addition of the matrix unit, three per product.
"""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

EPS, U, UM, SPLIT = 2.0 ** -53, 2.0 ** -24, 2.0 ** -23, 3 * 2.0 ** -18


@pytest.fixture(scope="module")
def system(gpu_available):
    from helpers import gpu_jk
    from psi4_amd.basisset import BasisSet
    from psi4_amd.molecule import Molecule
    one = np.array([[0.0, 0.0, 0.22], [0.0, 1.43, -0.89], [0.0, -1.43, -0.89]])
    mol = Molecule(["O", "H", "H"] * 7, np.vstack([one + [25.0 * i, 0.0, 0.0] for i in range(7)]))
    announce("seven waters in a row: set-up")
    jk = gpu_jk(BasisSet.build(mol, "cc-pvdz"), BasisSet.build(mol, "cc-pvdz-jkfit"))
    assert jk.info()["nbf"] == 168 and jk.info()["ntile_pairs"] <= 11   # of 21
    return jk, jk.get_B_dense(0, jk.info()["naux"])


def _sums(B, L, R):
    d = np.einsum("qmn,mn->q", B, L @ R.T, optimize=True)
    X, Y = B @ L, B @ R
    n = B.shape[1]
    K = X.transpose(1, 0, 2).reshape(n, -1) @ Y.transpose(1, 0, 2).reshape(n, -1).T
    return np.einsum("q,qmn->mn", d, B, optimize=True), K


@pytest.mark.parametrize("precision", ["FP64", "FP32", "BF16X3"])
@pytest.mark.parametrize("ncol", [6, 150])
def test_pair_forms(system, precision, ncol):
    import psi4_amd.core as core
    jk, B = system
    naux, nbf, _ = B.shape
    announce(f"screened B, {precision}, {ncol} columns")
    jk.set_precision(getattr(core, "PREC_" + precision))
    rng = np.random.default_rng(ncol)
    L, R = rng.standard_normal((2, nbf, ncol))
    half = ncol // 2
    X = np.hstack([L[:, :half], R[:, :half]])
    Y = np.hstack([R[:, :half], L[:, :half]])
    pairs = [(L, L), (L, R), (X, Y), (L, L * np.where(np.arange(ncol) % 3 == 1, -1.0, 1.0))]
    terms = naux * (ncol + 31)
    f64 = 2 * (2 * nbf + terms + 3) * EPS
    tj = 2 * (nbf * nbf + naux + ncol + 2) * EPS + (0 if precision == "FP64" else 2.02 * U)
    tk = {"FP64": f64, "FP32": 1.01 * ((2 * (nbf + 2) + 512 + 16 + 1) * U + f64),
          "BF16X3": 1.01 * (2 * (SPLIT + 2 * U + 3 * nbf * UM) + SPLIT + (3 * 544 + terms // 512 + 2) * UM + f64)}[precision]
    try:
        for l, r in pairs:
            jk.C_clear()
            jk.C_left_add(l)
            if r is not l:
                jk.C_right_add(r)
            jk.compute()
            Jo, Ko = _sums(B, l, r)
            Ja, Ka = _sums(np.abs(B), np.abs(l), np.abs(r))
            assert np.all(np.abs(jk.J()[0] - Jo) <= tj * Ja)
            assert np.all(np.abs(jk.K()[0] - Ko) <= tk * Ka)
    finally:
        jk.set_precision(core.PREC_FP64)


@pytest.mark.parametrize("nocc", [6, 150])
def test_adjoint(system, nocc):
    jk, B = system
    naux, nbf, _ = B.shape
    announce(f"screened B, adjoint, {nocc} columns")
    C = np.random.default_rng(nocc).standard_normal((nbf, nocc)) / np.sqrt(nbf)

    def ref(B, C):
        D = C @ C.T
        d = np.einsum("qmn,mn->q", B, D, optimize=True)
        DBD = (D @ B.reshape(-1, nbf, nbf)) @ D
        J, K = _sums(B, C, C)
        return 2 * np.sum(d * d), np.sum(DBD * B), 8 * (J @ C), 4 * (K @ C), 4 * d[:, None, None] * D, 2 * DBD

    E, dC, dB = jk.energy_adjoint(C, True)
    r, a = ref(B, C), ref(np.abs(B), np.abs(C))
    c = 4 * (2 * nbf * nbf + 2 * nbf + nocc + naux * nocc + 8) * EPS
    assert abs(E - (r[0] - r[1])) <= c * (a[0] + a[1])
    assert np.all(np.abs(dC - (r[2] - r[3])) <= c * (a[2] + a[3]))
    assert np.all(np.abs(dB - (r[4] - r[5])) <= c * (a[4] + a[5]))
