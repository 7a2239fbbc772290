"""The layer's training kernels against float64 autograd of the same equations on the same BF16 inputs.

The reference rounds where the forward kernels store BF16 (straight through); a gradient is then FP32 arithmetic and
one rounding, half a BF16 ulp = 2^-9 of its value, and the l2 norm's and the normalization's differences of nearly equal
terms are judged on their row's scale: 1e-2 of the row's largest value (``_inputs.rel_err``).  Sums over tokens are
FP32 and rounded once: 1e-2 of the tensor's largest value."""

import pytest
import torch
import torch.nn.functional as F

from _inputs import global_rel_err, rel_err

pytestmark = pytest.mark.gpu
TOL = 1e-2


def rounded(x):
    return x + (x.detach().to(torch.bfloat16).double() - x.detach())


@pytest.mark.parametrize('tokens,heads,s,hv,routes,qk', [
    (1, 1, 8, 8, 16, 'nvidia'), (5, 3, 8, 24, 32, 'original'), (33, 2, 16, 64, 48, 'nvidia'), (7, 1, 32, 256, 8, 'original'),
    (3, 8, 8, 128, 96, 'nvidia')])
def test_controller_backward(device, tokens, heads, s, hv, routes, qk):
    from bdm_amd import ops
    gen = torch.Generator().manual_seed(tokens * 10 + s)
    hs, total = heads * s, heads * hv
    widths = dict(q=hs, k=hs, v=total, f=hv, b=hs, w=total, read=routes, write=routes, gate=total)
    columns, at = {}, 0
    for name, width in widths.items():
        columns[name], at = at, at + width
    proj = (2 * torch.randn(tokens, at, generator=gen)).to(torch.bfloat16)
    proj[0, columns['q']:columns['q'] + s] = 0  # a zero row: the norm's guard
    f = (4 * torch.randn(tokens, hs, generator=gen)).to(torch.bfloat16)
    f[-1, 0] = 40.0  # above the softplus threshold
    a_log, dt_bias = (torch.randn(n, generator=gen).to(torch.bfloat16) for n in (heads, hs))
    shapes = [(tokens, heads, s)] * 2 + [(tokens, heads, hv), (tokens, heads, s), (tokens, heads, s), (tokens, heads, hv),
                                         (tokens, routes), (tokens, routes), (tokens, total)]
    grads = [torch.randn(*shape, generator=gen).to(torch.float32 if i == 3 else torch.bfloat16)
             for i, shape in enumerate(shapes)]
    p64, f64, a64, dt64 = (t.double().requires_grad_(True) for t in (proj, f, a_log, dt_bias))
    part = {n: p64[:, columns[n]:columns[n] + w] for n, w in widths.items()}

    def unit(x):
        x = rounded(F.silu(x)).reshape(tokens, heads, s)
        norm2 = x.square().sum(-1, keepdim=True)
        return x * torch.rsqrt(norm2 + 1e-6) if qk == 'nvidia' else x / norm2.clamp_min(1e-24).sqrt()

    g = -a64.exp()[:, None] * F.softplus((f64 + dt64).reshape(tokens, heads, s))
    outs = (unit(part['q']), unit(part['k']), F.silu(part['v']).reshape(tokens, heads, hv), g,
            part['b'].sigmoid().reshape(tokens, heads, s), part['w'].sigmoid().reshape(tokens, heads, hv),
            part['read'], part['write'], part['gate'])
    ref_p, ref_f, ref_a, ref_dt = torch.autograd.grad(outs, (p64, f64, a64, dt64), [t.double() for t in grads])
    print('CASE controller backward', tokens, heads, s, hv, routes, qk, flush=True)
    dp, df, terms = ops.controller_backward(*(t.to(device) for t in (proj, f)), columns, a_log.to(device),
                                            dt_bias.to(device), [t.to(device) for t in grads], heads=heads, bank_size=s,
                                            head_width=hv, route_width=routes, qk_norm=qk)
    torch.cuda.synchronize()
    for name, width in widths.items():
        if name != 'f':  # those columns are the caller's
            cut = slice(columns[name], columns[name] + width)
            err = rel_err(dp[:, cut], ref_p[:, cut], block=s if name in 'qkb' else None)
            assert err < TOL, (name, err)
    assert rel_err(df, ref_f) < TOL
    dt, rate = terms.sum(0)
    assert global_rel_err(dt, ref_dt) < TOL and global_rel_err(rate.view(heads, s).sum(-1), ref_a) < TOL


@pytest.mark.parametrize('tokens,width,kind', [(1, 8, 'layer'), (5, 520, 'rms'), (33, 512, 'layer'), (70, 1032, 'layer'),
                                               (3, 4096, 'rms'), (64, 2048, 'layer')])
def test_output_backward(device, tokens, width, kind):
    from bdm_amd import ops
    gen = torch.Generator().manual_seed(width + tokens)
    raw, wide, dy = (torch.randn(tokens, n, generator=gen).to(torch.bfloat16) for n in (width, width + 16, width))
    weight, bias = ((1 + 0.3 * torch.randn(width, generator=gen)).to(torch.bfloat16) for _ in range(2))
    leaves = [t.double().requires_grad_(True) for t in (raw, wide[:, 8:8 + width], weight, bias)]
    r, gt, wt, bs = leaves
    n = F.layer_norm(r, (width,), wt, bs, 1e-5) if kind == 'layer' else r * torch.rsqrt(r.square().mean(-1, keepdim=True) + 1e-5) * wt
    ref = torch.autograd.grad(rounded(n) * gt.sigmoid(), leaves, dy.double(), allow_unused=True)
    print('CASE output backward', tokens, width, kind, flush=True)
    got = ops.output_backward(raw.to(device), wide.to(device)[:, 8:8 + width], weight.to(device),
                              bias.to(device) if kind == 'layer' else None, dy.to(device), eps=1e-5, kind=kind)
    torch.cuda.synchronize()
    assert (got[3] is None) == (kind == 'rms')
    for ours, theirs, err in zip(got, ref, (rel_err, rel_err, global_rel_err, global_rel_err)):
        if ours is not None:
            assert err(ours, theirs) < TOL, err(ours, theirs)


@pytest.mark.parametrize('banks,selected,dtype', [(256, 8, torch.bfloat16), (12, 3, torch.float32), (2048, 8, torch.float32),
                                                  (6, 1, torch.bfloat16)])
def test_router_backward(device, banks, selected, dtype):
    from bdm_amd.config import near_square_factors
    from bdm_amd import product_key_route
    gen = torch.Generator().manual_seed(banks)
    j1, j2 = near_square_factors(banks)
    scores = torch.randn(2, 77, j1 + j2, generator=gen).to(dtype).to(device).requires_grad_(True)
    dw = torch.randn(2, 77, selected, generator=gen).to(dtype).to(device)
    print('CASE router backward', banks, selected, dtype, flush=True)
    weights, index = product_key_route(scores, bank_count=banks, selected_banks=selected)
    grad, = torch.autograd.grad(weights, scores, dw)
    leaf = scores.detach().double().requires_grad_(True)
    values = leaf[..., :j1].gather(-1, index // j2) + leaf[..., j1:].gather(-1, index % j2)
    ref, = torch.autograd.grad(values.softmax(-1), leaf, dw.double())
    # BF16: the weights, the K terms and their sum are each rounded
    assert rel_err(grad, ref) < (4e-2 if dtype == torch.bfloat16 else 1e-5)


LAYERS = [  # config class, heads, rows, options
    ('BSDMConfig', 2, 8, {}),
    ('BSDMConfig', 1, 16, {}),
    ('BSDMConfig', 4, 8, dict(output_bias=False, qk_normalization='original')),
    ('BDMConfig', 2, 8, {}),
    ('BDMConfig', 1, 32, dict(output_normalization='layer', routed_decay=True))]


def trained_layer(device, kind, heads, rows, options, tokens=50):
    """A BF16 layer and its input.  Input and router are small multiples of powers of two, so that the route scores are
    the same however a product sums them: no route depends on the path."""
    import bdm_amd
    cfg = getattr(bdm_amd, kind)(dim=64, bank_count=64, bank_size=rows, selected_banks=4, value_width=128, num_heads=heads,
                                 **options)
    gen = torch.Generator().manual_seed(rows + heads)
    layer = bdm_amd.BankedDeltaMemory(cfg, seed=3)
    with torch.no_grad():
        for p in layer.shared_router.parameters():
            p.copy_(torch.randint(-32, 33, p.shape, generator=gen) / 128)
        layer.dt_bias += 3  # decays that are felt within the sequence
        for p in (layer.output_norm_weight, getattr(layer, 'output_norm_bias', None), layer.output_gate.bias):
            if p is not None:
                p += 0.2 * torch.randn(p.shape, generator=gen)
    layer = layer.to(device=device, dtype=torch.bfloat16)
    x = (torch.randint(-8, 9, (2, tokens, 64), generator=gen) / 4).to(torch.bfloat16).to(device).requires_grad_(True)
    dy = torch.randn(2, tokens, 64, generator=gen).to(torch.bfloat16).to(device)
    return layer, x, dy


def both_paths(layer, x, work):
    """``work()`` with the fused training path and, behind a hook that changes nothing, with the modules' own calls."""
    assert layer._fused_training_supported(x)
    fused = work()
    handle = layer.v_proj.register_forward_hook(lambda m, i, o: None)
    assert not layer._fused_training_supported(x)
    plain = work()
    handle.remove()
    torch.cuda.synchronize()
    return fused, plain


def norm_err(a, b):
    a, b = a.double(), b.double()
    return float((a - b).norm() / b.norm().clamp_min(1e-30))


@pytest.mark.parametrize('kind,heads,rows,options', LAYERS)
def test_layer_gradients(device, kind, heads, rows, options):
    """The fused training path against autograd of the modules' own calls: the output and the gradients of the input
    and of every parameter.  Both round to BF16 at up to ten places between a parameter and the loss, 2^-9 each and
    independent of one another: 2.5e-2 in the 2-norm is four times their root sum (each was 0.2 to 1.4 % off float64)."""
    layer, x, dy = trained_layer(device, kind, heads, rows, options)
    names = [n for n, _ in layer.named_parameters()] + ['input']
    leaves = [*layer.parameters(), x]
    print('CASE layer gradients', kind, heads, rows, options, flush=True)

    def gradients():
        y = layer(x)
        return [y.detach(), *torch.autograd.grad(y, leaves, dy)]

    fused, plain = both_paths(layer, x, gradients)
    assert len(names) >= 22
    for name, ours, theirs in zip(['output', *names], fused, plain):
        assert ours.dtype == theirs.dtype and ours.shape == theirs.shape
        assert float(theirs.double().norm()) > 0, name
        assert norm_err(ours, theirs) < 2.5e-2, (name, norm_err(ours, theirs))


def test_layer_second_derivatives(device):
    """Gradients of gradients reach what they reach without the fused path: those of the parameters behind the operator
    are whole, those that pass the operator's own backward keep its first-order part."""
    layer, x, dy = trained_layer(device, 'BSDMConfig', 2, 8, {})
    behind = [layer.o_proj.weight, layer.output_norm_weight, layer.output_norm_bias, layer.output_gate.weight]
    leaves = [*behind, layer.output_gate.bias, layer.q_proj.weight, layer.f_proj[1].weight, layer.A_log,
              layer.shared_router.base.weight, x]
    print('CASE second derivatives', flush=True)

    def penalized(first):
        def run():
            loss = (layer(x).float() * dy.float()).sum()
            grads = torch.autograd.grad(loss, first, create_graph=True)
            penalty = sum(g.float().square().sum() for g in grads)
            assert all(g.requires_grad for g in grads)
            return torch.autograd.grad(penalty, leaves, allow_unused=True)
        return run

    for first in (behind, [x]):
        fused, plain = both_paths(layer, x, penalized(first))
        for leaf, ours, theirs in zip(leaves, fused, plain):
            assert (ours is None) == (theirs is None), leaf.shape
            if theirs is not None:
                # twice the roundings of a first gradient, and the penalty doubles their share
                assert norm_err(ours, theirs) < 5e-2, (leaf.shape, norm_err(ours, theirs))


def test_layer_batched_gradients(device):
    """Several output gradients at once (is_grads_batched), for the parameters whose gradients don't pass the operator."""
    layer, x, dy = trained_layer(device, 'BSDMConfig', 2, 8, {})
    leaves = [layer.o_proj.weight, layer.output_norm_weight, layer.output_gate.weight]
    several = torch.stack([dy, -0.5 * dy, dy.flip(1)])
    print('CASE batched gradients', flush=True)
    fused, plain = both_paths(layer, x, lambda: torch.autograd.grad(layer(x), leaves, several, is_grads_batched=True))
    for ours, theirs in zip(fused, plain):
        assert ours.shape == theirs.shape and norm_err(ours, theirs) < 2.5e-2


GATES = {  # what a hook on the output gate returns
    'another stride': lambda o: torch.cat([o, o], -1)[..., :o.shape[-1]],
    'another order': lambda o: o.transpose(1, 2).contiguous().transpose(1, 2),
    'unaligned': lambda o: torch.cat([o, o], -1)[..., 3:3 + o.shape[-1]],
    'FP32': lambda o: o.float(),
    'broadcast': lambda o: o[..., :1]}


@pytest.mark.parametrize('kind', GATES)
def test_hooked_output_gate(device, kind):
    """The output gate is called as a module on the fused path too: whatever its hook makes of the projection."""
    layer, x, dy = trained_layer(device, 'BSDMConfig', 2, 8, {})
    layer.output_gate.register_forward_hook(lambda m, i, o: GATES[kind](o))
    leaves = [x, layer.output_gate.weight, layer.output_norm_weight, layer.q_proj.weight]
    print('CASE hooked gate', kind, flush=True)

    def gradients():
        y = layer(x)
        return [y.detach(), *torch.autograd.grad(y, leaves, dy)]

    for ours, theirs in zip(*both_paths(layer, x, gradients)):
        assert ours.shape == theirs.shape and norm_err(ours, theirs) < 2.5e-2


def test_output_side_leaves_the_operator(device, monkeypatch):
    """Gradients of the parameters behind the operator alone, by freezing the others or by asking for these, neither run
    the operator's backward nor take snapshots for it."""
    from bdm_amd import ops
    layer, x, dy = trained_layer(device, 'BSDMConfig', 2, 8, {})
    side = {n: p for n, p in layer.named_parameters() if n.startswith('output') or n.startswith('o_proj')}
    assert len(side) == 6
    print('CASE output side', flush=True)
    whole = torch.autograd.grad(layer(x), list(side.values()), dy)
    monkeypatch.setattr(ops, 'routed_backward', None)
    asked = torch.autograd.grad(layer(x), list(side.values()), dy)
    monkeypatch.setattr(ops, 'snapshot_buffer', None)
    for n, p in layer.named_parameters():
        p.requires_grad_(n in side)
    frozen = torch.autograd.grad(layer(x.detach()), list(side.values()), dy)
    for a, b, c in zip(whole, asked, frozen):
        assert torch.equal(a, b) and torch.equal(a, c)


def test_training_forward_keeps_module_hooks(device):
    """A projection that is hooked is called as a module, with the same output to BF16 rounding (read and write routes
    from one projection or several agree here: well separated scores)."""
    from bdm_amd import BSDMConfig, BankedDeltaMemory
    cfg = BSDMConfig(dim=64, bank_count=64, bank_size=8, selected_banks=4, value_width=128, num_heads=2)
    layer = BankedDeltaMemory(cfg, seed=3).to(device=device, dtype=torch.bfloat16)
    x = torch.randn(2, 50, 64, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(device)
    seen = []
    print('CASE training hooks', flush=True)
    assert layer._fused_training_supported(x)
    first = layer(x)
    handle = layer.v_proj.register_forward_hook(lambda m, i, o: seen.append(o.shape))
    assert not layer._fused_training_supported(x)
    second = layer(x)
    handle.remove()
    assert len(seen) == 1 and rel_err(first, second) < 5e-2
