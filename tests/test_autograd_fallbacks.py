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


@pytest.fixture
def layer():
    from bdm_amd import BSDMConfig, BankedDeltaMemory
    config = BSDMConfig(dim=64, bank_count=64, bank_size=8, selected_banks=4, value_width=128, num_heads=2)
    return BankedDeltaMemory(config, seed=3).to(torch.bfloat16)


def subclass(layer, name):
    base = type(layer)
    layer.__class__ = type('Own', (base,), {name: lambda self, *args: getattr(base, name)(self, *args)})


def replace_forward(module):
    module.forward = lambda x, forward=module.forward: forward(x)


class Marked(torch.Tensor):
    """A tensor type of its own, as quantized or sharded weights are."""


OWN_BEHAVIOUR = {
    'forward of an instance': lambda m: replace_forward(m.q_proj),
    'forward of the factor pair': lambda m: replace_forward(m.f_proj),
    'own read map': lambda m: setattr(m.shared_router, 'read', m.shared_router.read),
    'hook': lambda m: m.w_proj.register_forward_hook(lambda *a: None),
    'another module': lambda m: setattr(m, 'v_proj', torch.nn.Sequential(m.v_proj)),
    'another factor pair': lambda m: setattr(m, 'f_proj', torch.nn.Linear(64, 16, bias=False, dtype=torch.bfloat16)),
    'another router': lambda m: setattr(m, 'shared_router', torch.nn.Identity()),
    'method of the instance': lambda m: setattr(m, '_controllers', m._controllers),
    'another weight type': lambda m: setattr(m.k_proj, 'weight', torch.nn.Parameter(
        m.k_proj.weight.detach().as_subclass(Marked))),
    **{'subclass ' + n: lambda m, n=n: subclass(m, n)
       for n in ('bank_reads', '_controllers', '_route_projections', '_project_bank_output', '_normalize_qk')},
}


@pytest.mark.parametrize('change', OWN_BEHAVIOUR)
def test_training_path_gives_way_to_own_behaviour(layer, change):
    """Calls that the fused training path would pass by keep the modules' path."""
    x = torch.zeros(1, 3, 64, dtype=torch.bfloat16)
    assert layer._fused_training_supported(x)
    OWN_BEHAVIOUR[change](layer)
    assert not layer._fused_training_supported(x)


@pytest.mark.parametrize('register', ['register_module_forward_hook', 'register_module_forward_pre_hook',
                                      'register_module_full_backward_hook'])
def test_training_path_gives_way_to_global_hooks(layer, register):
    x = torch.zeros(1, 3, 64, dtype=torch.bfloat16)
    handle = getattr(torch.nn.modules.module, register)(lambda *a: None)
    try:
        assert not layer._fused_training_supported(x)
    finally:
        handle.remove()
    assert layer._fused_training_supported(x)
