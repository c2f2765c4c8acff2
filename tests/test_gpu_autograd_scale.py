"""Gradients of s E(C, B) that are differentiated again in the factor s (create_graph): d<dE/dC, v>/ds.

Tolerance: both sides sum the same products s dE/dC_i v_i, |error| <= 2 n 2^-53 sum |dE/dC_i v_i| for n terms.
"""
import pytest

from conftest import announce

pytestmark = pytest.mark.gpu

EPS = 2.0 ** -53


@pytest.mark.parametrize("scale", [1.0, -0.5])
@pytest.mark.parametrize("with_B", [False, True])
def test_gradients_differentiate_in_the_factor(gpu_available, scale, with_B):
    import torch
    from psi4_amd.autograd import scf_energy_2e
    from psi4_amd.core import JK

    announce(f"create_graph, factor {scale}, {'C and B' if with_B else 'C'}")
    nbf, naux, nocc = 50, 30, 7
    jk = JK.build_tensor(nbf, naux)
    jk.set_print(0)
    jk.initialize()
    jk.fill_synthetic(3)
    g = torch.Generator(device="cuda").manual_seed(1)
    C = torch.randn(nbf, nocc, dtype=torch.float64, device="cuda", generator=g, requires_grad=True)
    x = [C]
    if with_B:
        B = torch.randn(naux, nbf, nbf, dtype=torch.float64, device="cuda", generator=g)
        x.append((0.5 * (B + B.transpose(1, 2))).contiguous().requires_grad_())
    plain = torch.autograd.grad(scf_energy_2e(jk, *x), x)
    v = [torch.randn(t.shape, dtype=torch.float64, device="cuda", generator=g) for t in x]
    s = torch.tensor(scale, dtype=torch.float64, device="cuda", requires_grad=True)
    grads = torch.autograd.grad(s * scf_energy_2e(jk, *x), x, create_graph=True)
    for got, want in zip(grads, plain):
        assert torch.equal(got.detach(), want * scale)
    ds, = torch.autograd.grad(sum((a * b).sum() for a, b in zip(grads, v)), s)
    terms = torch.cat([(a * b).reshape(-1) for a, b in zip(plain, v)])
    assert abs(float(ds - terms.sum())) <= 2 * terms.numel() * EPS * float(terms.abs().sum())
