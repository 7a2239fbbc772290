"""The differentiable form of backward passes that run as kernels, on the CPU: the library calls are replaced by
equivalents that, like the kernels, leave no graph."""

import pytest
import torch

from oracle import bdm_oracle as O


@pytest.fixture
def router(monkeypatch):
    from bdm_amd import ops, routing

    @torch.no_grad()
    def select(projected, *, bank_count, selected_banks):
        return tuple(t.clone() for t in O.product_key_route(projected, bank_count=bank_count,
                                                            selected_banks=selected_banks))

    @torch.no_grad()
    def backward(weights, indices, grad_weights, factors):
        w, dw = weights.float(), grad_weights.float()
        values = (w * (dw - (w * dw).sum(-1, keepdim=True))).to(weights.dtype).float()
        grad = torch.zeros(*weights.shape[:-1], sum(factors))
        grad[..., :factors[0]].scatter_add_(-1, indices // factors[1], values)
        grad[..., factors[0]:].scatter_add_(-1, indices % factors[1], values)
        return grad.to(weights.dtype)

    monkeypatch.setattr(ops, 'router_select', select)
    monkeypatch.setattr(ops, 'router_backward', backward)
    return routing.product_key_route


@pytest.mark.parametrize('banks,selected', [(64, 4), (12, 3), (6, 1)])
def test_route_weights_second_derivative(router, banks, selected):
    """A penalty on the first gradient reaches the scores, against autograd of the selection in float64."""
    factors = O.near_square_factors(banks)
    gen = torch.Generator().manual_seed(banks)
    scores = torch.randn(2, 7, sum(factors), generator=gen, requires_grad=True)
    coefficient = torch.randn(2, 7, selected, generator=gen)

    def penalized(leaf, weights):
        loss = (weights * coefficient.to(weights.dtype)).sum()
        grad, = torch.autograd.grad(loss, leaf, create_graph=True)
        return torch.autograd.grad(loss + 100 * grad.square().sum(), leaf, allow_unused=True)[0]

    weights, index = router(scores, bank_count=banks, selected_banks=selected)
    leaf = scores.detach().double().requires_grad_(True)
    values = leaf[..., :factors[0]].gather(-1, index // factors[1]) + leaf[..., factors[0]:].gather(-1, index % factors[1])
    ref = penalized(leaf, values.softmax(-1))
    # FP32 sums of at most 2K terms of the two adjoints: a few dozen roundings of 2^-24 of the largest term
    torch.testing.assert_close(penalized(scores, weights).double(), ref, rtol=0, atol=64 * 2 ** -24 * 100)
