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


def test_training_forward_keeps_module_hooks(device):
    """A projection that is hooked or replaced is called as a module, with the same gradients to BF16 rounding (read
    and write routes from one projection or several agree here: well separated scores)."""
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
