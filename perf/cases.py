"""Performance cases of the routed-memory framework.

Each case is one piece of work that a program built on this package asks for
through its public entry points:

``operator``  the routed bank operator (``bank_training`` with routed decay,
              ``role_bank_training`` without): forward, or forward and the
              gradients of every controller, route weight and the state;
``layer``     the memory layer ``BankedDeltaMemory``: ``forward`` under
              no_grad, ``prefill`` (reads and the new cache), or a training
              pass with the gradients of the input and every parameter;
``step``      one decode token of a layer for a batch of sequences
              (``GraphDecoder``, or ``BankedDeltaMemory.step``);
``mlp``       the language model's normalization and feed-forward sublayer,
              forward and backward;
``lm_step``   one decode token of a whole ``BDMLanguageModel``
              (``LanguageModelGraphDecoder``), returning logits.

``listed`` are the sizes of this repository's configurations, benchmark and
tests; ``draw`` gives others of the same ranges.  ``exact`` restates each path
in float64 with plain torch.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

DTYPES = {'bf16': torch.bfloat16, 'fp32': torch.float32}


def listed():
    return [
        # the layer without gradients at the size of the FP32 module check: a small, latency-bound call
        dict(name='layer_small_fp32', kind='layer', mode='forward', dtype='fp32', batch=1, time=512, dim=512, heads=4,
             rows=8, width=64, banks=256, selected=8, state='fp32', defaults='bsdm'),
        # serving: one token for each of 64 sequences against resident caches, replayed from a graph
        dict(name='step_batch64', kind='step', graph=True, dtype='bf16', batch=64, dim=1024, heads=8, rows=8,
             width=128, banks=256, selected=8, state='bf16', defaults='bsdm'),
        # serving: the prompt of 8 sequences through one layer, reads and the new cache
        dict(name='layer_prefill', kind='layer', mode='prefill', dtype='bf16', batch=8, time=4096, dim=1024, heads=8,
             rows=8, width=128, banks=256, selected=8, state='bf16', defaults='bsdm'),
        # training: one layer, forward and backward, every parameter gradient
        dict(name='layer_train', kind='layer', mode='train', dtype='bf16', batch=4, time=2048, dim=1024, heads=8,
             rows=8, width=128, banks=256, selected=8, state='bf16', defaults='bsdm'),
        # evaluation: the routed operator on a large batch with the training state's rounding
        dict(name='operator_forward', kind='operator', grads=False, dtype='bf16', batch=8, time=4096, heads=8, rows=8,
             width=128, banks=256, selected=8, state='bf16', decay=True, zipf=0.0),
        # many banks, a few of which take most events: long chains beside many short ones; the FP32 state of
        # the prefill policy, and the rounded state of the training policy
        dict(name='operator_skewed_fp32_state', kind='operator', grads=False, dtype='bf16', batch=4, time=8192,
             heads=8, rows=8, width=128, banks=2048, selected=8, state='fp32', decay=True, zipf=1.1),
        dict(name='operator_skewed', kind='operator', grads=False, dtype='bf16', batch=4, time=8192, heads=8, rows=8,
             width=128, banks=2048, selected=8, state='bf16', decay=True, zipf=1.1),
        # training at the package's default geometry: 4 rows a bank, one head, 1024 banks, no routed decay
        dict(name='operator_train_default', kind='operator', grads=True, dtype='bf16', batch=8, time=2048, heads=1,
             rows=4, width=128, banks=1024, selected=8, state='bf16', decay=False, zipf=0.0),
        # larger banks, a few heads, an odd length
        dict(name='operator_train_rows16', kind='operator', grads=True, dtype='bf16', batch=2, time=1001, heads=4,
             rows=16, width=64, banks=64, selected=8, state='bf16', decay=True, zipf=0.0),
        # training the whole model's layer: one head of width 2048 over 1024 banks
        dict(name='operator_train_wide', kind='operator', grads=True, dtype='bf16', batch=1, time=8192, heads=1,
             rows=8, width=2048, banks=1024, selected=8, state='bf16', decay=True, zipf=0.0),
        # training: the feed-forward sublayer of the whole model (activations recomputed, its default)
        dict(name='mlp_train', kind='mlp', dtype='bf16', tokens=8192, dim=2048),
        # serving: one token of a model of 4 layers of the whole model's widths, batch 1, replayed from a graph
        dict(name='lm_step', kind='lm_step', dtype='bf16', batch=1, layers=4, vocab=50257, dim=2048, heads=1, rows=8,
             width=2048, banks=1024, selected=8, state='bf16', defaults='bsdm'),
    ]


def _spread(rng, low, high):
    """A size spread over the logarithm of its range, odd or even."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(['operator', 'operator', 'operator', 'layer', 'layer', 'step', 'mlp'])
    if kind == 'mlp':
        return dict(kind='mlp', dtype='bf16', tokens=_spread(rng, 64, 8192), dim=rng.choice([512, 1024, 2048]))
    if kind == 'step':
        heads, width = rng.choice([(8, 128), (4, 64), (4, 128), (1, 2048)])
        return dict(kind='step', graph=rng.random() < 0.7, dtype='bf16', batch=_spread(rng, 1, 96 if heads > 1 else 8),
                    dim=rng.choice([512, 1024, 2048]), heads=heads, rows=8, width=width,
                    banks=rng.choice([256, 1024]), selected=8, state='bf16', defaults='bsdm')
    if kind == 'layer':
        mode = rng.choice(['forward', 'prefill', 'train'])
        dtype = 'fp32' if rng.random() < 0.25 else 'bf16'
        heads, width, dim = rng.choice([(8, 128, 1024), (4, 64, 512), (2, 64, 256), (1, 1024, 1024)])
        batch = rng.randint(1, 8)
        return dict(kind='layer', mode=mode, dtype=dtype, batch=batch,
                    time=_spread(rng, 64, (16384 if mode == 'prefill' else 8192) // batch), dim=dim, heads=heads,
                    rows=8, width=width, banks=rng.choice([256, 512, 1024]), selected=8,
                    state='fp32' if dtype == 'fp32' else 'bf16', defaults=rng.choice(['bsdm', 'bsdm', 'bdm']))
    grads = rng.random() < 0.6
    rows = rng.choice([4, 8, 8, 16])
    heads, width = rng.choice([(1, 128), (2, 64), (4, 64), (8, 128), (1, 512), (1, 2048 if rows == 8 else 256)])
    dtype = 'fp32' if rng.random() < 0.2 else 'bf16'
    batch = rng.randint(1, 8)
    most = 8192 if grads or dtype == 'fp32' else 32768
    if rows * width * heads > 8192:
        most //= rows * width * heads // 8192
    return dict(kind='operator', grads=grads, dtype=dtype, batch=batch, time=_spread(rng, 33, max(64, most // batch)),
                heads=heads, rows=rows, width=width, banks=rng.choice([64, 256, 1024, 2048]), selected=rng.choice([4, 8]),
                state='fp32' if dtype == 'fp32' else rng.choice(['bf16', 'bf16', 'fp32']), decay=rng.random() < 0.7,
                zipf=rng.choice([0.0, 0.0, 1.1]) if not grads else 0.0)


# ---------------------------------------------------------------------------------------------- inputs

def _generator(seed, salt=0):
    gen = torch.Generator(device='cuda')
    gen.manual_seed(int(seed) * 1009 + salt)
    return gen


def _near_square(value):
    first = math.isqrt(value)
    while value % first:
        first -= 1
    return first, value // first


def _route(scores, banks, selected):
    """Product-key selection of [..., J1 + J2] scores: the best ``selected`` of
    the pair sums of each factor's best, added in the score type, ties to the
    lower index; (float64 softmax weights, indices)."""
    j1, j2 = _near_square(banks)
    s = min(selected, j1, j2)

    def best(x, k):
        values, index = torch.sort(x, dim=-1, descending=True, stable=True)
        return values[..., :k], index[..., :k]

    first, fi = best(scores[..., :j1], s)
    second, si = best(scores[..., j1:], s)
    values, pair = best((first.unsqueeze(-1) + second.unsqueeze(-2)).flatten(-2), min(selected, s * s))
    row = torch.gather(fi, -1, torch.div(pair, s, rounding_mode='floor'))
    return torch.softmax(values.double(), -1), row * j2 + torch.gather(si, -1, pair.remainder(s))


def _operator_inputs(c, seed):
    """Controllers as a layer's projections give them, routes of normal scores
    (with a Zipf bias over each factor where the case is skewed), a small
    initial state, and the upstream gradient."""
    gen, dtype = _generator(seed), DTYPES[c['dtype']]
    lead = (c['batch'], c['time'])
    h, s, v, j = c['heads'], c['rows'], c['width'], c['banks']

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device='cuda')

    q, k = (F.normalize(F.silu(normal(*lead, h, s)), dim=-1).to(dtype) for _ in range(2))
    val = F.silu(normal(*lead, h, v)).to(dtype)
    rate = torch.empty(h, 1, device='cuda').uniform_(1, 16, generator=gen)
    steps = torch.empty(h, s, device='cuda').uniform_(math.log(1e-3), math.log(0.1), generator=gen)
    g = -rate * F.softplus(steps.exp().expm1().log() + 0.3 * normal(*lead, h, s))
    b = torch.sigmoid(normal(*lead, h, s)).to(dtype)
    w = torch.sigmoid(normal(*lead, h, v)).to(dtype)
    j1, j2 = _near_square(j)
    bias = torch.cat([-c['zipf'] * torch.log1p(torch.randperm(n, generator=gen, device='cuda').float())
                      for n in (j1, j2)])
    routes = []
    for _ in range(2):
        weights, index = _route((normal(*lead, j1 + j2) + bias).to(dtype), j, c['selected'])
        routes += [index, weights.to(dtype)]
    wi, ww, ri, rw = routes
    state = (normal(j, h, s, v) * 0.05).to(dtype)
    dy = normal(*lead, h * v).to(dtype)
    return q, k, val, g, b, w, wi, ww, ri, rw, state, dy


def _layer_weights(c, seed, salt=1):
    """A memory layer's parameters at the scale of a trained layer's (the read
    and write routers apart by their residuals), by name."""
    gen, dtype = _generator(seed, salt), DTYPES[c['dtype']]
    d, h, s, v, j = c['dim'], c['heads'], c['rows'], c['width'], c['banks']
    total, keys, routes = h * v, h * s, sum(_near_square(j))
    p, q = _near_square(j * h * s)

    def normal(*shape, std):
        return (torch.randn(*shape, generator=gen, device='cuda') * std).to(dtype)

    def uniform(*shape, low, high):
        return torch.empty(*shape, device='cuda').uniform_(low, high, generator=gen)

    std = d ** -0.5
    out = {'A_log': uniform(h, low=1, high=16).log().to(dtype),
           'dt_bias': uniform(keys, low=math.log(1e-3), high=math.log(0.1)).exp().expm1().log().to(dtype),
           'initial_row_factor': normal(p, v, std=0.05), 'initial_column_factor': normal(q, v, std=0.05),
           'output_norm_weight': 1 + normal(total, std=0.1), 'f_proj.0.weight': normal(v, d, std=0.5 * std),
           'f_proj.1.weight': normal(keys, v, std=0.5 * v ** -0.5), 'output_gate.weight': normal(total, d, std=std),
           'output_gate.bias': normal(total, std=0.1), 'o_proj.weight': normal(d, total, std=total ** -0.5)}
    for name, width in (('q_proj', keys), ('k_proj', keys), ('v_proj', total), ('b_proj', keys), ('w_proj', total)):
        out[name + '.weight'] = normal(width, d, std=std)
    for name, scale in (('base', 1.0), ('read_residual', 0.5), ('write_residual', 0.5)):
        out[f'shared_router.{name}.weight'] = normal(routes, d, std=scale * std)
        out[f'shared_router.{name}.bias'] = normal(routes, std=0.1 * scale)
    if c['defaults'] == 'bsdm':
        out['output_norm_bias'] = normal(total, std=0.1)
        out['o_proj.bias'] = normal(d, std=0.1)
    return out


def _memory_config(c):
    from bdm_amd import BDMConfig, BSDMConfig
    kind = BSDMConfig if c['defaults'] == 'bsdm' else BDMConfig
    return kind(dim=c['dim'], bank_count=c['banks'], bank_size=c['rows'], selected_banks=c['selected'],
                value_width=c['heads'] * c['width'], num_heads=c['heads'],
                training_state_dtype={'bf16': 'bfloat16', 'fp32': 'float32'}[c['state']])


def _layer(c, weights):
    from bdm_amd import BankedDeltaMemory
    with torch.device('cuda'):
        layer = BankedDeltaMemory(_memory_config(c))
    layer = layer.to(DTYPES[c['dtype']])
    layer.load_state_dict(weights)
    return layer


def _hidden(c, seed, *lead):
    return torch.randn(*lead, c['dim'], generator=_generator(seed, 2), device='cuda').to(DTYPES[c['dtype']])


def _cache(c, seed, salt=3):
    """A resident decode cache, as the states of a running service."""
    shape = (c['batch'], c['banks'], c['heads'], c['rows'], c['width'])
    cache = torch.empty(shape, device='cuda', dtype=DTYPES[c['state']])
    gen = _generator(seed, salt)
    for i in range(c['batch']):
        cache[i] = torch.randn(shape[1:], generator=gen, device='cuda') * 0.02
    return cache if c['heads'] > 1 else cache.squeeze(2)


def _ffn_width(dim):
    return 256 * (-(-int(2 * 4 * dim / 3) // 256))


def _ffn_weights(c, seed, salt=4):
    gen, dtype, d = _generator(seed, salt), DTYPES[c['dtype']], c['dim']
    f = _ffn_width(d)

    def normal(*shape, std):
        return (torch.randn(*shape, generator=gen, device='cuda') * std).to(dtype)

    return {'norm': 1 + normal(d, std=0.1), 'w1': normal(f, d, std=d ** -0.5), 'w3': normal(f, d, std=d ** -0.5),
            'w2': normal(d, f, std=f ** -0.5)}


def _lm_weights(c, seed):
    gen, dtype, d = _generator(seed, 5), DTYPES[c['dtype']], c['dim']

    def normal(*shape, std):
        return (torch.randn(*shape, generator=gen, device='cuda') * std).to(dtype)

    out = {'tok_embeddings.weight': normal(c['vocab'], d, std=1.0), 'norm.weight': 1 + normal(d, std=0.1),
           'output.weight': normal(c['vocab'], d, std=d ** -0.5)}
    for i in range(c['layers']):
        out.update({f'layers.{i}.attention.{n}': t for n, t in _layer_weights(c, seed, 100 + i).items()})
        ffn = _ffn_weights(c, seed, 200 + i)
        out.update({f'layers.{i}.feed_forward.{n}.weight': ffn[n] for n in ('w1', 'w2', 'w3')})
        out[f'layers.{i}.ffn_norm.weight'] = ffn['norm']
        out[f'layers.{i}.attention_norm.weight'] = 1 + normal(d, std=0.1)
    return out


def _lm_inputs(c, seed):
    tokens = torch.randint(0, c['vocab'], (c['batch'], 1), generator=_generator(seed, 6), device='cuda')
    return tokens, [_cache(c, seed, 300 + i) for i in range(c['layers'])]


# ---------------------------------------------------------------------------------------------- the calls

def prepare(case, seed):
    c, kind = case, case['kind']
    if kind == 'operator':
        *args, dy = _operator_inputs(c, seed)
        if c['grads']:
            args = [t.requires_grad_(True) if t.is_floating_point() else t for t in args]
        return dict(case=c, args=args, dy=dy)
    if kind == 'layer':
        layer = _layer(c, _layer_weights(c, seed))
        x = _hidden(c, seed, c['batch'], c['time'])
        state = dict(case=c, layer=layer, x=x)
        if c['mode'] == 'train':
            x.requires_grad_(True)
            state['dy'] = torch.randn(x.shape, generator=_generator(seed, 7), device='cuda').to(x.dtype)
        return state
    if kind == 'step':
        from bdm_amd import GraphDecoder
        layer = _layer(c, _layer_weights(c, seed)).requires_grad_(False)
        cache = _cache(c, seed)
        decoder = GraphDecoder(layer, cache) if c['graph'] else None
        return dict(case=c, layer=layer, cache=cache, decoder=decoder, x=_hidden(c, seed, c['batch'], 1))
    if kind == 'mlp':
        from bdm_amd.lm import FeedForward, RMSNorm
        w, dtype = _ffn_weights(c, seed), DTYPES[c['dtype']]
        with torch.device('cuda'):
            norm = RMSNorm(c['dim'], eps=1e-5).to(dtype)
            ffn = FeedForward(c['dim'], 4 * c['dim'], 256, None, recompute_activations=True).to(dtype)
        norm.load_state_dict({'weight': w['norm']})
        ffn.load_state_dict({n + '.weight': w[n] for n in ('w1', 'w2', 'w3')})
        x = _hidden(c, seed, 1, c['tokens']).requires_grad_(True)
        dy = torch.randn(x.shape, generator=_generator(seed, 7), device='cuda').to(dtype)
        return dict(case=c, norm=norm, ffn=ffn, x=x, dy=dy)
    from bdm_amd import LanguageModelGraphDecoder
    from bdm_amd.lm import BDMLanguageModel, LanguageModelConfig
    config = LanguageModelConfig(memory=_memory_config(c), vocab_size=c['vocab'], layers=c['layers'])
    with torch.device('cuda'):
        model = BDMLanguageModel(config)
    model = model.to(DTYPES[c['dtype']]).requires_grad_(False)
    model.load_state_dict(_lm_weights(c, seed))
    tokens, caches = _lm_inputs(c, seed)
    return dict(case=c, model=model, tokens=tokens, decoder=LanguageModelGraphDecoder(model, caches))


def _call_operator(c, args):
    from bdm_amd import bank_training, role_bank_training
    operator = bank_training if c['decay'] else role_bank_training
    return operator(*args, c['banks'], c['rows'] ** -0.5, state_dtype=DTYPES[c['state']])


def run(state):
    c, kind = state['case'], state['case']['kind']
    if kind == 'operator':
        if not c['grads']:
            with torch.no_grad():
                return _call_operator(c, state['args'])
        y = _call_operator(c, state['args'])
        leaves = [t for t in state['args'] if t.requires_grad]
        return [y.detach(), *torch.autograd.grad(y, leaves, state['dy'])]
    if kind == 'layer':
        layer, x = state['layer'], state['x']
        if c['mode'] == 'train':
            y, leaves = layer(x), dict(layer.named_parameters(), input=x)
            return dict(zip(leaves, torch.autograd.grad(y, list(leaves.values()), state['dy'])), output=y.detach())
        with torch.no_grad():
            return list(layer.prefill(x)) if c['mode'] == 'prefill' else layer(x)
    if kind == 'step':
        if state['decoder'] is not None:
            return [state['decoder'].step(state['x']), state['cache']]
        with torch.no_grad():
            return list(state['layer'].step(state['x'], state['cache']))
    if kind == 'mlp':
        norm, ffn, x = state['norm'], state['ffn'], state['x']
        y = x + ffn(norm(x))
        return [y.detach(), *torch.autograd.grad(y, [x, norm.weight, ffn.w1.weight, ffn.w3.weight, ffn.w2.weight],
                                                 state['dy'])]
    return [state['decoder'].step(state['tokens']), *state['decoder'].caches]


# ---------------------------------------------------------------------------------------------- what a pass needs

def _size(c):
    return DTYPES[c['dtype']].itemsize


def _routed_work(c, tokens, grads, state_bytes):
    """The recurrence and the combine: a write is 5 and a read 2 operations a
    state element, their adjoints 11 and 4."""
    e, h, s, v, k = _size(c), c['heads'], c['rows'], c['width'], c['selected']
    inputs = tokens * (h * s * (3 * e + 4) + 2 * h * v * e + 2 * k * (8 + e)) + state_bytes
    moved = inputs + tokens * h * v * e
    if grads:  # dy in; the gradients of all but the indices out
        moved += tokens * h * v * e + inputs - tokens * 2 * k * 8
    return moved, tokens * h * k * s * v * (22 if grads else 7)


def _layer_parameters(c):
    h, s, v, d = c['heads'], c['rows'], c['width'], c['dim']
    total, keys, routes = h * v, h * s, sum(_near_square(c['banks']))
    maps = d * (3 * keys + 4 * total + 2 * routes + v) + v * keys
    return maps, maps + d * routes + sum(_near_square(c['banks'] * h * s)) * v


def work(case):
    c, kind, e = case, case['kind'], _size(case)
    if kind == 'mlp':
        n, d, f = c['tokens'], c['dim'], _ffn_width(c['dim'])
        return {'bytes': e * (4 * n * d + 2 * (3 * d * f + d)), 'flops': 18 * n * d * f}
    if kind == 'operator':
        elements = c['banks'] * c['heads'] * c['rows'] * c['width']
        moved, flops = _routed_work(c, c['batch'] * c['time'], c['grads'], elements * e)
        return {'bytes': moved, 'flops': flops}
    bank = c['heads'] * c['rows'] * c['width'] * DTYPES[c['state']].itemsize
    maps, weights = _layer_parameters(c)
    if kind == 'layer':
        n, train = c['batch'] * c['time'], c['mode'] == 'train'
        flops = 2 * n * maps * (3 if train else 1) + _routed_work(c, n, train, 0)[1]
        moved = e * (2 * n * c['dim'] + weights) * (2 if train else 1)
        if c['mode'] == 'prefill':
            moved += c['batch'] * c['banks'] * bank
        return {'bytes': moved, 'flops': flops}
    n = c['batch']
    moved = e * (2 * n * c['dim'] + weights) + n * 2 * 2 * c['selected'] * bank  # banks written: in and out; read: about half more
    flops = 2 * n * maps + _routed_work(c, n, False, 0)[1]
    if kind == 'step':
        return {'bytes': moved, 'flops': flops}
    ffn, head = 3 * c['dim'] * _ffn_width(c['dim']), c['vocab'] * c['dim']
    return {'bytes': c['layers'] * (moved + e * ffn) + e * head, 'flops': c['layers'] * (flops + 2 * n * ffn) + 2 * n * head}


def tolerance(case):
    """Measured against ``exact``: FP32 paths 1e-7 to 1.2e-6 off; in BF16 the operator and the feed-forward 0.2 to
    0.5 %, a layer 0.8 % and its parameter gradients up to 1.4 % (a gradient passes more BF16 roundings), four layers
    in a row 1.3 to 6 % (a rounded route score that flips one bank).  The largest single value is 0.15 of the root mean
    square off (a state row of a token whose route flipped)."""
    if case['dtype'] == 'fp32':
        return {'rel': 1e-5, 'max': 2e-3}
    return {'rel': {'layer': 2e-2, 'step': 2e-2, 'lm_step': 3e-2}.get(case['kind'], 1e-2), 'max': 0.25}


# ---------------------------------------------------------------------------------------------- float64 restatement

def _recurrence64(q, k, v, g, b, w, wi, ww, ri, rw, state, banks, scale, decay):
    """The routed recurrence in float64: (reads [B, T, H*v], final state [B, J, H, S, v]).  Events of a (sequence,
    bank) run in order, a token's write before its read; step p advances every segment of more than p events."""
    batch, time, kw = wi.shape
    kr, nt = ri.shape[-1], batch * time
    device = q.device
    token = torch.arange(nt, device=device)
    tokens = torch.cat([token.repeat_interleave(kw), token.repeat_interleave(kr)])
    bank = torch.cat([wi.reshape(-1), ri.reshape(-1)])
    reads = torch.arange(tokens.numel(), device=device) >= nt * kw
    weight = torch.cat([ww.reshape(-1), rw.reshape(-1)]).double()
    segment = tokens // time * banks + bank
    order = torch.argsort((segment * time + tokens % time) * 2 + reads)
    tokens, reads, weight = tokens[order], reads[order], weight[order]
    lengths = torch.bincount(segment, minlength=batch * banks)
    starts = lengths.cumsum(0) - lengths
    longest = torch.argsort(lengths, descending=True)
    starts = starts[longest]
    most = int(lengths.max())
    live = (lengths[None, :] > torch.arange(0, most, 1024, device=device)[:, None]).sum(1).tolist()  # every 1024 steps
    ordered = lengths[longest]
    q, k, g, b = (t.reshape(nt, *t.shape[2:]).double() for t in (q, k, g, b))
    v, w = (t.reshape(nt, *t.shape[2:]) for t in (v, w))
    state = state.double()
    if state.ndim == 4:
        state = state.expand(batch, *state.shape)
    whole = state.reshape(batch * banks, *state.shape[2:])[longest]
    heads, rows, width = whole.shape[1:]
    training = torch.is_grad_enabled()
    step_bytes = 6 * tokens.numel() * heads * rows * 8 if training else 1  # kept for the backward, a column
    columns = max(1, min(width, int(40e9 // step_bytes)))
    outs, finals = [], []
    for lo in range(0, width, columns):
        m, z, done = whole[..., lo:lo + columns], [], []
        vc, wc = (t[..., lo:lo + columns].double() for t in (v, w))
        for p in range(most):
            if p % 1024 == 0:
                counts = (ordered[None, :live[p // 1024]] > p + torch.arange(min(1024, most - p), device=device)[:, None]
                          ).sum(1).tolist()
            n = counts[p % 1024]
            if n < m.shape[0]:
                done.append(m[n:])
                m = m[:n]
            e = starts[:n] + p
            t, r, pw = tokens[e], reads[e][:, None, None], weight[e][:, None, None]
            kt = k[t].masked_fill(r, 0)
            log_decay = (g[t] * pw if decay else g[t]).masked_fill(r, 0)
            m = m * log_decay.exp().unsqueeze(-1)
            u = wc[t] * pw * vc[t] - ((b[t] * pw * kt).unsqueeze(-1) * m).sum(-2)
            m = m + kt.unsqueeze(-1) * u.unsqueeze(-2)
            z.append((t, ((q[t] * pw * scale).masked_fill(~r, 0).unsqueeze(-1) * m).sum(-2)))
        out = torch.zeros(nt, heads, m.shape[-1], dtype=torch.float64, device=device)
        outs.append(out.index_add(0, torch.cat([t for t, _ in z]), torch.cat([x for _, x in z])))
        finals.append(torch.cat([m, *done[::-1]]))
    final = torch.cat(finals, -1)[torch.argsort(longest)].reshape(batch, banks, heads, rows, width)
    return torch.cat(outs, -1).reshape(batch, time, heads * width), final


def _rounded(x, dtype):
    """float64 values rounded to the layer's data type; the gradient passes."""
    return x + (x.detach().to(dtype).double() - x.detach())


def _routes64(scores, c):
    """Selection on the scores in the layer's type, weights in float64 with their gradient."""
    _, index = _route(scores.detach().to(DTYPES[c['dtype']]), c['banks'], c['selected'])
    j1, j2 = _near_square(c['banks'])
    values = torch.gather(scores[..., :j1], -1, torch.div(index, j2, rounding_mode='floor')) \
        + torch.gather(scores[..., j1:], -1, index.remainder(j2))
    return torch.softmax(values, -1), index


def _layer64(c, p, hidden, cache=None):
    """The memory layer in float64 from its parameters ``p``: (output, final state).  The values that the layer
    defines in its own type are rounded to it: the sums of parameters, and the route scores, which select."""
    lead, h, s, v = hidden.shape[:2], c['heads'], c['rows'], c['width']
    bsdm, dtype = c['defaults'] == 'bsdm', DTYPES[c['dtype']]
    x = hidden.double()

    def linear(name):
        bias = p.get(name + '.bias')
        return F.linear(x, p[name + '.weight'].double(), None if bias is None else bias.double())

    def total(first, second):
        return _rounded(first.double() + second.double(), dtype)

    def unit(t):
        t = F.silu(t).reshape(*lead, h, s)
        norm2 = t.square().sum(-1, keepdim=True)
        return t * torch.rsqrt(norm2 + 1e-6) if bsdm else t / norm2.sqrt().clamp_min(1e-12)

    def scores(role):
        r = 'shared_router.'
        weight, bias = (total(p[f'{r}base.{n}'], p[f'{r}{role}_residual.{n}']) for n in ('weight', 'bias'))
        return _rounded(F.linear(x, weight, bias), dtype)

    q, k = unit(linear('q_proj')), unit(linear('k_proj'))
    val = F.silu(linear('v_proj')).reshape(*lead, h, v)
    f = F.linear(linear('f_proj.0'), p['f_proj.1.weight'].double())
    g = -p['A_log'].double().exp()[:, None] * F.softplus((f + p['dt_bias'].double()).reshape(*lead, h, s))
    b = linear('b_proj').sigmoid().reshape(*lead, h, s)
    w = linear('w_proj').sigmoid().reshape(*lead, h, v)
    ww, wi = _routes64(scores('write'), c)
    rw, ri = _routes64(scores('read'), c)
    if cache is None:
        cache = total(p['initial_row_factor'][:, None, :], p['initial_column_factor'][None, :, :]).reshape(
            c['banks'], h, s, v)
    else:
        cache = cache.reshape(c['batch'], c['banks'], h, s, v)
    raw, final = _recurrence64(q, k, val, g, b, w, wi, ww, ri, rw, cache, c['banks'], s ** -0.5, bsdm)
    weight, eps = p['output_norm_weight'].double(), 1e-5
    if bsdm:
        normed = F.layer_norm(raw, (h * v,), weight, p['output_norm_bias'].double(), eps)
    else:
        normed = raw * torch.rsqrt(raw.square().mean(-1, keepdim=True) + eps) * weight
    x = normed * torch.sigmoid(linear('output_gate'))
    return linear('o_proj'), final


def _rms64(x, weight, eps=1e-5):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * weight.double()


def _ffn64(x, w1, w3, w2):
    return F.linear(F.silu(F.linear(x, w1.double())) * F.linear(x, w3.double()), w2.double())


def exact(case, seed):
    c, kind = case, case['kind']
    if kind == 'operator':
        *args, dy = _operator_inputs(c, seed)
        args = [t.double() if t.is_floating_point() else t for t in args]
        with torch.set_grad_enabled(c['grads']):
            leaves = [t.requires_grad_(c['grads']) for t in args if t.is_floating_point()]
            y, _ = _recurrence64(*args, c['banks'], c['rows'] ** -0.5, c['decay'])
            return [y.detach(), *torch.autograd.grad(y, leaves, dy.double())] if c['grads'] else y
    if kind == 'layer':
        p, x = _layer_weights(c, seed), _hidden(c, seed, c['batch'], c['time'])
        if c['mode'] != 'train':
            with torch.no_grad():
                y, final = _layer64(c, p, x)
            return [y, final if c['heads'] > 1 else final.squeeze(2)] if c['mode'] == 'prefill' else y
        dy = torch.randn(x.shape, generator=_generator(seed, 7), device='cuda').to(x.dtype)
        leaves = {n: t.double().requires_grad_(True) for n, t in {'input': x, **p}.items()}
        y, _ = _layer64(c, leaves, leaves['input'])
        return dict(zip(leaves, torch.autograd.grad(y, list(leaves.values()), dy.double())), output=y.detach())
    if kind == 'step':
        with torch.no_grad():
            y, final = _layer64(c, _layer_weights(c, seed), _hidden(c, seed, c['batch'], 1), _cache(c, seed))
        return [y, final if c['heads'] > 1 else final.squeeze(2)]
    if kind == 'mlp':
        w, x = _ffn_weights(c, seed), _hidden(c, seed, 1, c['tokens'])
        dy = torch.randn(x.shape, generator=_generator(seed, 7), device='cuda').to(x.dtype)
        leaves = [t.double().requires_grad_(True) for t in (x, w['norm'], w['w1'], w['w3'], w['w2'])]
        y = leaves[0] + _ffn64(_rms64(leaves[0], leaves[1]), *leaves[2:])
        return [y.detach(), *torch.autograd.grad(y, leaves, dy.double())]
    p = _lm_weights(c, seed)
    tokens, caches = _lm_inputs(c, seed)
    finals = []
    with torch.no_grad():
        x = p['tok_embeddings.weight'][tokens].double()
        for i, cache in enumerate(caches):
            own = {n.split('.attention.')[1]: t for n, t in p.items() if n.startswith(f'layers.{i}.attention.')}
            y, final = _layer64(c, own, _rms64(x, p[f'layers.{i}.attention_norm.weight']), cache)
            x = x + y
            ffn = [p[f'layers.{i}.feed_forward.{n}.weight'] for n in ('w1', 'w3', 'w2')]
            x = x + _ffn64(_rms64(x, p[f'layers.{i}.ffn_norm.weight']), *ffn)
            finals.append(final if c['heads'] > 1 else final.squeeze(2))
        return [F.linear(_rms64(x, p['norm.weight']), p['output.weight'].double()), *finals]
