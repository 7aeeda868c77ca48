"""How a layer hands its generator to the kernels: a_scale of every shape that broadcasts against A, numbers on the
parameters' rows and tensors of A's shape on the entries read off A; a generator that is the module's own storage (the
kernels' operand, saved for the backward, is no alias of it while gradients are recorded); a parametrisation whose
forward was replaced on the instance."""

import numpy as np
import pytest
import torch

import ews_mi355x as E
from ews_mi355x.params import kernel_rows

CPU = torch.device("cpu")
D = 6


def _layers():
    g = torch.Generator().manual_seed(0)
    v, u, th = (torch.randn(n, generator=g) for n in (D // 2, D // 2, D))
    return [E.EWS(E.AParamDampedRotation(v, u, D), N=2, leaf="plane_closed", combine="block_kernel"),
            E.EWS(E.AParamEFM(th), N=2, leaf="series", series_q=8)]


def _read(structure, A):
    if structure == "planes":
        i = torch.arange(0, D, 2)
        return torch.stack([A[i, i], A[i, i + 1]], -1)
    return torch.diagonal(A)


@pytest.mark.parametrize("scale", [1.0, 2, 0.5, np.float32(0.25), torch.tensor(0.3), torch.tensor([0.3]),
                                   torch.tensor([[0.3]]), torch.tensor(0.3, dtype=torch.float64),
                                   torch.linspace(0.2, 1.0, D), torch.linspace(0.2, 1.0, D)[:, None],
                                   torch.linspace(0.2, 1.0, D * D).reshape(D, D)])
def test_scales_of_every_shape(scale):
    for layer in _layers():
        A = layer.A_param() * torch.as_tensor(scale, dtype=torch.float32)
        got, want = layer._diag_params(CPU, scale), _read(layer.structure, A)
        assert got.shape == want.shape and got.is_contiguous()
        assert torch.equal(got, want)


def test_learned_scale_gets_its_gradient():
    for layer in _layers():
        for shape in ((), (1,), (1, 1), (D, D)):
            s = torch.full(shape, 0.7, requires_grad=True)
            r = s.detach().clone().requires_grad_()
            layer._diag_params(CPU, s).square().sum().backward()
            _read(layer.structure, layer.A_param() * r).square().sum().backward()
            assert torch.allclose(s.grad, r.grad, rtol=1e-6)


def test_no_alias_of_the_modules_own_storage():
    for p in (E.AParamConstant(torch.randn(4, 4)), E.AParamGeneral(torch.randn(4, 4))):
        own = next(iter(p.state_dict().values()))
        A = E.EWS._scaled(p(), 1.0, CPU)
        assert A.data_ptr() != own.data_ptr()
        with torch.no_grad():  # nothing is saved: the tensor itself serves
            assert E.EWS._scaled(p(), 1.0, CPU).data_ptr() == own.data_ptr()


def test_forward_replaced_on_the_instance():
    p = E.AParamEFM(torch.randn(D))
    assert kernel_rows(p) is not None
    p.forward = lambda: torch.diag(p.theta.exp())
    assert kernel_rows(p) is None
