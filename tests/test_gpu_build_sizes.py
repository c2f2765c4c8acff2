"""FP64 J and K of small tensor handles at the edges of the kernels' tiles against numpy on the
same tensor: basis sizes around the 16-, 32- and 64-row blocks, one and a few auxiliary
functions, column counts around 8, 16 and 80, every pair form (symmetric, signed, cross,
general), several pairs in one call and a partial auxiliary range.

Tolerance: with every product replaced by its absolute value the same sums bound the rounding
error of any summation order, |error| <= (number of additions in a chain) * 2^-53 * (sum of
absolute values); the device and numpy each contribute one such term.
"""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53


def _tensor(nbf, naux, seed):
    from psi4_amd.core import JK
    jk = JK.build_tensor(nbf, naux)
    jk.set_print(0)
    jk.initialize()
    jk.fill_synthetic(seed)
    return jk, jk.get_B_dense(0, naux)


def _ref(B, L, R):
    d = np.einsum("qmn,mn->q", B, L @ R.T)
    J = np.einsum("q,qmn->mn", d, B)
    X, Y = B @ L, B @ R
    return J, np.einsum("qmi,qni->mn", X, Y)


def _check(B, L, R, D, J, K):
    naux, nbf, _ = B.shape
    ncol = L.shape[1]
    Jo, Ko = _ref(B, L, R)
    Ja, Ka = _ref(np.abs(B), np.abs(L), np.abs(R))
    assert np.all(np.abs(D - L @ R.T) <= 2 * (ncol + 1) * EPS * (np.abs(L) @ np.abs(R).T))
    assert np.all(np.abs(J - Jo) <= 2 * (nbf * nbf + naux + ncol + 2) * EPS * Ja)
    assert np.all(np.abs(K - Ko) <= 2 * (2 * nbf + naux * ncol + 3) * EPS * Ka)


def _compute(jk, lefts, rights=None):
    jk.C_clear()
    for c in lefts:
        jk.C_left_add(c)
    for c in rights or []:
        jk.C_right_add(c)
    jk.compute()
    return jk.D(), jk.J(), jk.K()


@pytest.mark.parametrize("nbf,naux", [(1, 1), (15, 3), (32, 1), (33, 9), (64, 5), (65, 17), (97, 8), (129, 41),
                                      (190, 70)])
def test_symmetric_sizes(gpu_available, nbf, naux):
    announce(f"symmetric pairs, nbf {nbf} naux {naux}")
    jk, B = _tensor(nbf, naux, 7)
    rng = np.random.default_rng(nbf)
    for ncol in (1, 8, 9, 17, 80, 81, 130):
        C = rng.standard_normal((nbf, ncol))
        D, J, K = _compute(jk, [C])
        _check(B, C, C, D[0], J[0], K[0])
        assert np.array_equal(K[0], K[0].T) and np.array_equal(J[0], J[0].T)


@pytest.mark.parametrize("nbf,naux", [(1, 2), (31, 5), (48, 64), (100, 33)])
@pytest.mark.parametrize("ncol", [2, 18, 82])
def test_pair_forms(gpu_available, nbf, naux, ncol):
    announce(f"general, cross and signed pairs, nbf {nbf} naux {naux} columns {ncol}")
    jk, B = _tensor(nbf, naux, 8)
    rng = np.random.default_rng(ncol)
    L, R = rng.standard_normal((2, nbf, ncol))
    D, J, K = _compute(jk, [L], [R])
    _check(B, L, R, D[0], J[0], K[0])
    A, V = rng.standard_normal((2, nbf, ncol // 2))
    X, Y = np.hstack([A, V]), np.hstack([V, A])
    D, J, K = _compute(jk, [X], [Y])
    _check(B, X, Y, D[0], J[0], K[0])
    assert np.array_equal(K[0], K[0].T)
    S = L * np.where(np.arange(ncol) % 3 == 1, -1.0, 1.0)
    D, J, K = _compute(jk, [L], [S])
    _check(B, L, S, D[0], J[0], K[0])
    assert np.array_equal(K[0], K[0].T)


def test_many_pairs_in_one_call(gpu_available):
    """Pairs of different widths and forms in one call: shared left matrices (the same array), an
    empty pair among them, more pairs than the kernels take at once."""
    nbf, naux = 70, 45
    announce("twelve pairs in one call")
    jk, B = _tensor(nbf, naux, 9)
    rng = np.random.default_rng(3)
    C0 = rng.standard_normal((nbf, 13))
    lefts, rights = [], []
    for i in range(12):
        if i % 4 == 0:
            L = R = rng.standard_normal((nbf, 5 + i))
        elif i % 4 == 1:
            L, R = C0, rng.standard_normal((nbf, 13))
        elif i == 6:
            L = R = np.zeros((nbf, 0))
        elif i % 4 == 2:
            A, V = rng.standard_normal((2, nbf, 9))
            L, R = np.hstack([A, V]), np.hstack([V, A])
        else:
            L, R = C0, -C0
        lefts.append(L)
        rights.append(R)
    D, J, K = _compute(jk, lefts, rights)
    for i in range(12):
        if lefts[i].shape[1]:
            _check(B, lefts[i], rights[i], D[i], J[i], K[i])
        else:
            assert not D[i].any() and not J[i].any() and not K[i].any()


def test_partial_auxiliary_range(gpu_available):
    nbf, naux = 66, 50
    announce("auxiliary range 7..31 of 50")
    jk, B = _tensor(nbf, naux, 10)
    C = np.random.default_rng(4).standard_normal((nbf, 20))
    jk.set_aux_range(7, 31)
    D, J, K = _compute(jk, [C])
    _check(B[7:31], C, C, D[0], J[0], K[0])


@pytest.mark.parametrize("nbf,naux,nocc", [(1, 1, 1), (33, 7, 5), (64, 12, 16), (70, 20, 33), (97, 9, 65), (100, 31, 81),
                                           (129, 6, 100), (40, 11, 60)])
def test_adjoint_sizes(gpu_available, nbf, naux, nocc):
    """E, dE/dC = 4 (2J - K) C and dE/dB = 4 d D - 2 D B D at block edges and for more columns than rows.
    The tolerance is that of the chains the device sums (rows, columns and auxiliary functions in
    turn) on the sums of absolute values; dE/dB is exactly symmetric, and a partial auxiliary range
    gives the same slice."""
    announce(f"adjoint, nbf {nbf} naux {naux} columns {nocc}")
    jk, B = _tensor(nbf, naux, 11)
    C = np.random.default_rng(nocc).standard_normal((nbf, nocc)) / np.sqrt(nbf)

    def ref(B, C):
        D = C @ C.T
        d = np.einsum("qmn,mn->q", B, D)
        DBD = D @ B @ D
        ej, ek = 2 * np.sum(d * d), np.einsum("qmn,qmn->", DBD, B)
        J, K = np.einsum("q,qmn->mn", d, B), np.einsum("qmk,qnk->mn", B @ C, B @ C)
        return ej, ek, 8 * (J @ C), 4 * (K @ C), 4 * d[:, None, None] * D, 2 * DBD

    E, dC, dB = jk.energy_adjoint(C, True)
    r, a = ref(B, C), ref(np.abs(B), np.abs(C))
    c = 4 * (2 * nbf * nbf + 2 * nbf + nocc + naux * nocc + 8) * EPS
    assert abs(E - (r[0] - r[1])) <= c * (a[0] + a[1])
    assert np.all(np.abs(dC - (r[2] - r[3])) <= c * (a[2] + a[3]))
    assert np.all(np.abs(dB - (r[4] - r[5])) <= c * (a[4] + a[5]))
    assert np.array_equal(dB, dB.transpose(0, 2, 1))
    if naux > 6:
        jk.set_aux_range(2, 5)
        E2, dC2, dB2 = jk.energy_adjoint(C, True)
        assert E2 == E and np.array_equal(dC2, dC) and np.array_equal(dB2, dB[2:5])


def test_memory_of_finished_handles_is_reused_and_given_back(gpu_available):
    """Buffers that earlier handles left behind (their contents too) serve later ones of other shapes,
    also from two threads at once; trim_memory gives the memory back to the device."""
    import gc
    import threading

    import torch

    from psi4_amd.core import trim_memory

    announce("handles after handles on reused memory")

    def one(nbf, naux, ncol, bad):
        jk, B = _tensor(nbf, naux, nbf)
        C = np.random.default_rng(naux).standard_normal((nbf, ncol))
        D, J, K = _compute(jk, [C])
        try:
            _check(B, C, C, D[0], J[0], K[0])
        except AssertionError as e:
            bad.append((nbf, naux, ncol, e))

    bad = []
    for shape in ((150, 200, 40), (40, 300, 9), (129, 150, 70)):
        one(*shape, bad)
    threads = [threading.Thread(target=one, args=(n, 90, 20, bad)) for n in (100, 61)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
    gc.collect()
    before = torch.cuda.mem_get_info()[0]
    trim_memory()
    assert torch.cuda.mem_get_info()[0] > before


def test_j_beside_k_on_a_caller_stream(gpu_available):
    """A build large enough (B 72 MB) for J's second pass to run on its own stream: results, and repeated
    builds queued back to back on a caller's stream with the outputs read on that stream."""
    import torch

    announce("nbf 256 naux 245 on a side stream")
    nbf, naux = 256, 245
    jk, B = _tensor(nbf, naux, 12)
    rng = np.random.default_rng(6)
    Cs = [rng.standard_normal((nbf, 24)) for _ in range(3)]
    s = torch.cuda.Stream()
    jk.set_stream(s.cuda_stream)
    with torch.cuda.stream(s):
        dC = [torch.tensor(C, device="cuda") for C in Cs]
        outs = []
        for C in dC:
            D, J, K = (torch.empty(nbf, nbf, dtype=torch.float64, device="cuda") for _ in range(3))
            jk.compute_device([C.data_ptr()], [], [24], [D.data_ptr()], [J.data_ptr()], [K.data_ptr()])
            outs.append([x.clone() for x in (D, J, K)])
    s.synchronize()
    for C, o in zip(Cs, outs):
        _check(B, C, C, *(x.cpu().numpy() for x in o))
    jk.set_stream(0)
