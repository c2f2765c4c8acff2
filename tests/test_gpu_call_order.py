"""Device calls whose arrays overlap: the pairs of a call are taken in order, and so are the outputs D, J, K of a
pair, as if each were finished before the next is begun.

The reference replays a call on a numpy copy of the same memory.  Tolerance: arrays that a pair reads may be
results of an earlier one, so an error bound would have to follow the chain; the products of at most two
pairs of 60 x 60 matrices are compared at 1e-11 of the largest element instead (their own rounding is
about 1e-13 of it, and a wrong order changes the leading digits).
"""
import numpy as np
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

NBF, NAUX = 60, 37
NN = NBF * NBF


@pytest.fixture(scope="module")
def jk(gpu_available):
    from psi4_amd.core import JK
    jk = JK.build_tensor(NBF, NAUX)
    jk.set_print(0)
    jk.initialize()
    jk.fill_synthetic(21)
    return jk, jk.get_B_dense(0, NAUX)


def _replay(B, mem, pairs, accumulate):
    for p in pairs:
        n = NBF * p["ncol"]
        L = mem[p["L"]:p["L"] + n].reshape(NBF, -1).copy()
        R = mem[p["R"]:p["R"] + n].reshape(NBF, -1).copy() if "R" in p else L
        d = np.einsum("qmn,mn->q", B, L @ R.T)
        res = {"D": L @ R.T, "J": np.einsum("q,qmn->mn", d, B), "K": np.einsum("qmi,qni->mn", B @ L, B @ R)}
        for k in "DJK":
            if k in p:
                out = mem[p[k]:p[k] + NN]
                out[:] = res[k].ravel() + (out if accumulate and k != "D" else 0.0)


def _run(jk, size, pairs, accumulate=False):
    import torch
    jk, B = jk
    start = np.random.default_rng(size).standard_normal(size)
    mem = torch.tensor(start, device="cuda")
    base = mem.data_ptr()
    at = lambda k: [base + 8 * p[k] if k in p else 0 for p in pairs]  # noqa: E731
    torch.cuda.synchronize()
    jk.compute_device(at("L"), at("R") if "R" in pairs[0] else [], [p["ncol"] for p in pairs], at("D"), at("J"),
                      at("K"), accumulate)
    torch.cuda.synchronize()
    _replay(B, start, pairs, accumulate)
    assert np.abs(mem.cpu().numpy() - start).max() <= 1e-11 * np.abs(start).max()


@pytest.mark.parametrize("read", ["L", "R"])
def test_later_output_over_an_earlier_input(jk, read):
    """D of the second pair lies where the first pair's left or right matrix was."""
    announce(f"D of pair 1 over {read} of pair 0")
    pairs = [{"L": 0, "R": NN, "ncol": NBF, "D": 2 * NN, "J": 3 * NN, "K": 4 * NN},
             {"L": 5 * NN, "R": 6 * NN, "ncol": 11, "J": 7 * NN, "K": 8 * NN}]
    pairs[1]["D"] = pairs[0][read]
    _run(jk, 9 * NN, pairs)


def test_outputs_that_reach_into_the_next_input(jk):
    """K of the first pair ends inside the second pair's left matrix, D of the second inside the first's right one."""
    announce("partly overlapping arrays")
    pairs = [{"L": 0, "R": NN, "ncol": 17, "D": 2 * NN, "J": 3 * NN, "K": 4 * NN},
             {"L": 5 * NN - 100, "R": 6 * NN, "ncol": 17, "D": NN - 300, "J": 7 * NN, "K": 8 * NN}]
    _run(jk, 9 * NN, pairs)


@pytest.mark.parametrize("accumulate", [False, True])
def test_outputs_of_one_pair_in_one_array(jk, accumulate):
    """J and K added up in one array, and D, J and K all written to one array (K stays)."""
    announce(f"outputs of a pair in one array, accumulate {accumulate}")
    _run(jk, 5 * NN, [{"L": 0, "ncol": 9, "D": NN, "J": 2 * NN, "K": 2 * NN},
                      {"L": 3 * NN, "ncol": 9, "D": 4 * NN, "J": 4 * NN, "K": 4 * NN}], accumulate)
