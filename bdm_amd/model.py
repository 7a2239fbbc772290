"""The BDM layer module on the HIP path.

``BankedDeltaMemory`` keeps the reference module's constructor, parameter
names/shapes, seeded initialisation and ``forward``/``prefill``/``step``
methods (implementation/bdm/model.py:15-140, _parameters.py, heads.py,
inference.py) so state dicts and call sites interchange.  The routed-memory
path (router selection, dispatch, recurrence, combine, decode) runs in
``libbdm_hip.so``; the controller and output projections stay torch GEMMs.

``backend`` accepts ``'hip'`` and, as an alias so that reference call sites
keep working, ``'role'`` (the reference's GPU backend name).
"""

from __future__ import annotations

import functools
import hashlib
import math

import torch
import torch.nn.functional as F
from torch import nn

from . import ops
from .config import BDMConfig, near_square_factors
from .routed_update import _round_interval, bank_training, role_bank_training
from .routing import SharedResidualRouter, product_key_route

Tensor = torch.Tensor


def _unit_rows(value: Tensor, kind: str) -> Tensor:
    """l2 normalization of q and k: 'nvidia': x * rsqrt(sum x^2 + 1e-6) in FP32
    (the in-file formula of _parameters.py:219; the reference calls FLA's l2norm
    on GPU, which is not available here); 'original': F.normalize (:220)."""
    if kind == 'nvidia':
        xf = value.float()
        return (xf * torch.rsqrt(xf.square().sum(-1, keepdim=True) + 1e-6)).to(value.dtype)
    return F.normalize(value.float(), dim=-1).to(value.dtype)


def _controller_ops(q, k, v, f, b, w, a_log, dt_bias, normalize, *, heads, bank_size, head_width):
    """The controllers (heads.py:11-22) in torch ops of their projections
    [..., width]: q, k, g, b [..., H, S]; v, w [..., H, v]."""
    shape = (*q.shape[:-1], heads)
    q = normalize(F.silu(q).reshape(*shape, bank_size))
    k = normalize(F.silu(k).reshape(*shape, bank_size))
    v = F.silu(v).reshape(*shape, head_width)
    g = -a_log.float().exp()[:, None] * F.softplus((f.float() + dt_bias.float()).reshape(*shape, bank_size))
    b = b.sigmoid().reshape(*shape, bank_size)
    w = w.sigmoid().reshape(*shape, head_width)
    return q, k, v, g, b, w


def _output_ops(raw, gate, weight, bias, eps, kind):
    """norm(raw) * sigmoid(gate), the input of o_proj (_parameters.py:222-232), in torch ops."""
    if kind == 'layer':
        normalized = F.layer_norm(raw, (raw.shape[-1],), weight, bias, eps)
    else:
        variance = raw.float().square().mean(dim=-1, keepdim=True)
        normalized = raw * torch.rsqrt(variance + eps).to(raw.dtype)
        normalized = normalized * weight.to(raw.dtype)
    return normalized * torch.sigmoid(gate).to(raw.dtype)


# Tests for the wrapped tensors of batched gradients, as far as this torch has them, and the one for global module
# hooks (without it every module counts as hooked).
_WRAPPED = [f for f in (getattr(getattr(torch._C, '_functorch', None), name, None)
                        for name in ('is_legacy_batchedtensor', 'is_functorch_wrapped_tensor')) if f is not None]
_global_hooks = getattr(nn.modules.module, '_has_any_global_hook', lambda: True)


def _differentiable(grads) -> bool:
    """Whether a backward has to run in torch ops: its result is differentiated
    again (create_graph; a kernel's would end the graph), or the gradients are
    batched (is_grads_batched)."""
    return torch.is_grad_enabled() or any(wrapped(t) for t in grads for wrapped in _WRAPPED)


def _torch_gradients(form, inputs, grads):
    """Gradients of ``form(*inputs)`` by autograd; None for an input that takes none."""
    create = torch.is_grad_enabled()
    with torch.enable_grad():
        outputs = form(*inputs)
        wanted = [t for t in inputs if t is not None and t.requires_grad]
        found = iter(torch.autograd.grad(outputs, wanted, grads, create_graph=create))
    return tuple(next(found) if t is not None and t.requires_grad else None for t in inputs)


class _LayerInputs(torch.autograd.Function):
    """The controllers and route scores of a layer from one projection [N, P] of
    its input: f_proj's second factor and the controller epilogue forward;
    backward, every column of the projection's gradient in one kernel around the
    two products of that factor."""

    @staticmethod
    def forward(ctx, proj, f_weight, a_log, dt_bias, columns, geometry):
        hv, rw = geometry['head_width'], geometry['route_width']
        f = F.linear(proj[:, columns['f']:columns['f'] + hv], f_weight)
        controllers = ops.controller_epilogue(proj, f, columns, a_log, dt_bias, heads=geometry['heads'],
                                              bank_size=geometry['bank_size'], head_width=hv,
                                              qk_norm=geometry['qk_norm'])
        ctx.save_for_backward(proj, f, f_weight, a_log, dt_bias)
        ctx.columns, ctx.geometry = columns, geometry
        # copies, not views: an output that shares an input's storage could not be saved or changed in place apart
        scores = (proj[:, columns[n]:columns[n] + rw].contiguous() for n in ('read', 'write'))
        return (*controllers, *scores)

    @staticmethod
    def backward(ctx, *grads):
        proj, f, f_weight, a_log, dt_bias = ctx.saved_tensors
        columns, geometry = ctx.columns, ctx.geometry
        if _differentiable(grads):
            form = functools.partial(_layer_inputs_ops, columns=columns, **geometry)
            return (*_torch_gradients(form, (proj, f_weight, a_log, dt_bias), grads), None, None)
        grad_proj, grad_f, terms = ops.controller_backward(proj, f, columns, a_log, dt_bias, (*grads, None), **geometry)
        at = slice(columns['f'], columns['f'] + geometry['head_width'])
        torch.mm(grad_f, f_weight, out=grad_proj[:, at])
        grad_weight = grad_f.t() @ proj[:, at]
        grad_dt, rate = terms.sum(0)
        grad_a = rate.view(geometry['heads'], geometry['bank_size']).sum(-1)
        return grad_proj, grad_weight, grad_a.to(a_log.dtype), grad_dt.to(dt_bias.dtype), None, None


def _layer_inputs_ops(proj, f_weight, a_log, dt_bias, *, columns, heads, bank_size, head_width, route_width, qk_norm):
    """_LayerInputs' forward in torch ops."""
    keys, total = heads * bank_size, heads * head_width
    widths = dict(q=keys, k=keys, v=total, f=head_width, b=keys, w=total, read=route_width, write=route_width)
    part = {n: proj[:, columns[n]:columns[n] + width] for n, width in widths.items()}
    controllers = _controller_ops(part['q'], part['k'], part['v'], F.linear(part['f'], f_weight), part['b'], part['w'],
                                  a_log, dt_bias, lambda x: _unit_rows(x, qk_norm), heads=heads, bank_size=bank_size,
                                  head_width=head_width)
    return (*controllers, part['read'], part['write'])


class _OutputInterface(torch.autograd.Function):
    """norm(raw) * sigmoid(gate) before o_proj (_parameters.py:222-232)."""

    @staticmethod
    def forward(ctx, raw, gate, weight, bias, eps, kind):
        ctx.save_for_backward(raw, gate, weight, bias)
        ctx.eps, ctx.kind = eps, kind
        return ops.output_epilogue(raw, gate, weight, bias, eps=eps, kind=kind)

    @staticmethod
    def backward(ctx, grad_out):
        raw, gate, weight, bias = ctx.saved_tensors
        if _differentiable([grad_out]):
            form = functools.partial(_output_ops, eps=ctx.eps, kind=ctx.kind)
            return (*_torch_gradients(form, (raw, gate, weight, bias), grad_out), None, None)
        return (*ops.output_backward(raw, gate, weight, bias, grad_out, eps=ctx.eps, kind=ctx.kind), None, None)


# The methods of a layer whose work its fused training path does in another way.
_TRAINING_METHODS = ('bank_reads', '_controllers', '_normalize_qk', '_route_projections', '_project_bank_output')


class BankedDeltaMemory(nn.Module):
    """Shared-residual product routing around dense GDN2 memory banks."""

    # Inference steps run the controller epilogue, both routes and the decode
    # kernel as one launch (``ops.decode_fused``) where the geometry allows;
    # False keeps the three separate kernels.  The fused launch also forms
    # f_proj's second factor, in another FP32 summation order than the GEMM,
    # so f may differ by one BF16 rounding and y and the cache match the
    # separate kernels within tolerance rather than bit for bit.
    fused_decode = True

    def __init__(self, config: BDMConfig, *, layer_id=0, seed=0, backend='hip', compact_replay=None):
        super().__init__()
        if backend not in ('hip', 'role'):
            raise ValueError("backend must be hip (or its alias role); the CPU equation oracle lives in oracle/")
        if min(seed, layer_id) < 0:
            raise ValueError(f'seed and layer_id must be >= 0, got seed={seed}, layer_id={layer_id}')
        if not (compact_replay is None or isinstance(compact_replay, bool)):
            raise ValueError(f'compact_replay takes None or a bool, not {compact_replay!r}')
        self.compact_replay = compact_replay
        self.config, self.backend = config, 'hip'
        self.hidden_size, self.bank_count, self.bank_size = config.dim, config.bank_count, config.bank_size
        self.value_width, self.kernel_key_width = config.value_width, config.bank_size
        self.num_heads = config.num_heads
        self.head_value_width = config.head_value_width
        key_width = config.num_heads * config.bank_size
        self.num_reads = self.num_writes = config.selected_banks
        self.layer_id, self.initialization_seed = layer_id, seed * 100_000 + 6000 + layer_id
        self.norm_eps = config.norm_eps
        self.shared_residual_router = True
        self.initial_state_mode = 'product_key'
        self.routing_mode = 'product_topk'
        route_width = sum(near_square_factors(config.bank_count))
        self.factor_route_width = self.route_projection_width = route_width
        self.q_proj = nn.Linear(config.dim, key_width, bias=False)
        self.k_proj = nn.Linear(config.dim, key_width, bias=False)
        self.v_proj = nn.Linear(config.dim, config.value_width, bias=False)
        self.shared_router = SharedResidualRouter(config.dim, route_width)
        self.read_route_proj = self.write_route_proj = None
        self.f_proj = nn.Sequential(nn.Linear(config.dim, config.head_value_width, bias=False),
                                    nn.Linear(config.head_value_width, key_width, bias=False))
        self.b_proj = nn.Linear(config.dim, key_width, bias=False)
        self.w_proj = nn.Linear(config.dim, config.value_width, bias=False)
        self.A_log = nn.Parameter(torch.empty(config.num_heads, dtype=torch.float32))
        self.dt_bias = nn.Parameter(torch.empty(key_width, dtype=torch.float32))
        self.A_log._no_weight_decay = self.dt_bias._no_weight_decay = True
        rows, columns = near_square_factors(config.logical_rows)
        self.register_parameter('initial_state', None)
        self.initial_row_factor = nn.Parameter(torch.zeros(rows, config.head_value_width))
        self.initial_column_factor = nn.Parameter(torch.zeros(columns, config.head_value_width))
        self.initial_row_factor._sdm_memory_bank = self.initial_column_factor._sdm_memory_bank = True
        self.output_gate = nn.Linear(config.dim, config.value_width, bias=True)
        self.output_norm_weight = nn.Parameter(torch.ones(config.value_width))
        if config.output_normalization == 'layer':
            self.output_norm_bias = nn.Parameter(torch.zeros(config.value_width))
        self.o_proj = nn.Linear(config.value_width, config.dim, bias=config.output_bias)
        self._fused_cache = None  # concatenated inference projection, keyed by the parameters' storage
        self.init_weights(initialization_seed=self.initialization_seed)

    # -- geometry helpers (_parameters.py:11-38) ------------------------------------
    @property
    def total_rows(self) -> int:
        return self.bank_count * self.num_heads * self.bank_size

    @property
    def touched_rows(self) -> int:
        return self.num_writes * self.num_heads * self.bank_size

    @property
    def logical_reads(self) -> int:
        return self.num_reads * self.num_heads * self.bank_size

    @property
    def logical_writes(self) -> int:
        return self.num_writes * self.num_heads * self.bank_size

    @property
    def initial_state_parameter_count(self) -> int:
        return sum(p.numel() for p in (self.initial_state, self.initial_row_factor, self.initial_column_factor)
                   if p is not None)

    def materialize_initial_state(self) -> Tensor:
        """M0 from the product factors (_parameters.py:40-67): row n = j*H*S + h*S + s
        starts at U[n // Q] + Z[n % Q].  [J, H, S, v] for H > 1, [J, S, V] for H = 1."""
        total = self.initial_row_factor[:, None, :] + self.initial_column_factor[None, :, :]
        if self.num_heads != 1:
            return total.reshape(self.bank_count, self.num_heads, self.bank_size, self.head_value_width)
        return total.reshape(self.bank_count, self.bank_size, self.value_width)

    # -- initialisation (_parameters.py:69-180) --------------------------------------
    def _role_generator(self, role: str, parameter: Tensor, initialization_seed):
        if initialization_seed is None:
            return None
        key = f'bank_sparse_gdn2.{self.layer_id}.{role}'.encode()
        digest = int.from_bytes(hashlib.blake2b(key, digest_size=8).digest(), byteorder='little')
        generator = torch.Generator(device=parameter.device)
        generator.manual_seed((initialization_seed ^ digest) % (1 << 63))
        return generator

    def init_weights(self, init_std=None, factor: float = 1.0, width_scaling=None, *,
                     initialization_seed=None) -> None:
        del width_scaling
        if initialization_seed is None:
            initialization_seed = self.initialization_seed
        if initialization_seed is not None and initialization_seed < 0:
            raise ValueError('initialization_seed must be non-negative')
        for name, module in self.named_modules():
            if isinstance(module, nn.Linear) and not name.startswith('shared_router.'):
                nn.init.xavier_uniform_(module.weight, gain=2 ** -2.5,
                                        generator=self._role_generator(f'{name}.weight', module.weight,
                                                                       initialization_seed))
                if module.bias is not None:
                    nn.init.zeros_(module.bias)
        route_std = (init_std or self.hidden_size ** -0.5) / factor
        base = self.shared_router.base.weight
        self.shared_router.initialize_from_independent(
            std=route_std,
            read_generator=self._role_generator('read_router.weight', base, initialization_seed),
            write_generator=self._role_generator('write_router.weight', base, initialization_seed))
        with torch.no_grad():
            self.A_log.uniform_(1.0, 16.0, generator=self._role_generator('decay_rate', self.A_log,
                                                                         initialization_seed)).log_()
            log_dt = torch.empty_like(self.dt_bias).uniform_(
                math.log(0.001), math.log(0.1),
                generator=self._role_generator('time_step', self.dt_bias, initialization_seed))
            dt = log_dt.exp().clamp_min(1e-4)
            self.dt_bias.copy_(dt + torch.log(-torch.expm1(-dt)))
            for role, parameter in (('initial_state.row', self.initial_row_factor),
                                    ('initial_state.column', self.initial_column_factor)):
                std = (init_std or self.hidden_size ** -0.5) / factor
                nn.init.trunc_normal_(parameter, mean=0.0, std=std, a=-3 * std, b=3 * std,
                                      generator=self._role_generator(role, parameter, initialization_seed))
                parameter.mul_(1 / math.sqrt(2))
            self.output_norm_weight.fill_(1.0)
            if hasattr(self, 'output_norm_bias'):
                self.output_norm_bias.zero_()

    def reset_parameters(self) -> None:
        self.init_weights(initialization_seed=self.initialization_seed)

    # -- controllers, routes and output interface -----------------------------------
    def _route_projections(self, hidden: Tensor) -> tuple[Tensor, Tensor]:
        return self.shared_router.read(hidden), self.shared_router.write(hidden)

    def _route(self, projected: Tensor, selected_banks: int):
        return product_key_route(projected, bank_count=self.bank_count, selected_banks=selected_banks)

    def _route_both(self, write_routes: Tensor, read_routes: Tensor):
        """Both roles' routes, ``(ww, wi), (rw, ri)``: one launch when no
        gradient flows to the scores and the roles select equally many banks."""
        needs_grad = torch.is_grad_enabled() and (write_routes.requires_grad or read_routes.requires_grad)
        if not needs_grad and self.num_writes == self.num_reads:
            return ops.router_select_pair(write_routes, read_routes, bank_count=self.bank_count,
                                          selected_banks=self.num_writes)
        return self._route(write_routes, self.num_writes), self._route(read_routes, self.num_reads)

    def _route_and_dispatch(self, write_routes: Tensor, read_routes: Tensor):
        """Both roles' routes and the dispatch over them: one library call
        (ops.route_dispatch) when no gradient flows to the scores and the
        roles select equally many banks, else the two steps."""
        needs_grad = torch.is_grad_enabled() and (write_routes.requires_grad or read_routes.requires_grad)
        if (not needs_grad and self.num_writes == self.num_reads and write_routes.ndim == 3
                and write_routes.shape == read_routes.shape and write_routes.dtype == read_routes.dtype):
            return ops.route_dispatch(write_routes, read_routes, bank_count=self.bank_count,
                                      selected_banks=self.num_writes)
        (ww, wi), (rw, ri) = self._route_both(write_routes, read_routes)
        return (ww, wi), (rw, ri), ops.dispatch_build(wi, ri, self.bank_count)

    def _normalize_qk(self, value: Tensor) -> Tensor:
        return _unit_rows(value, self.config.qk_normalization)

    def _controllers(self, hidden: Tensor):
        """Per-head controllers (heads.py:11-22): q,k,g,b [B,T,H,S]; v,w [B,T,H,v]."""
        return _controller_ops(self.q_proj(hidden), self.k_proj(hidden), self.v_proj(hidden), self.f_proj(hidden),
                               self.b_proj(hidden), self.w_proj(hidden), self.A_log, self.dt_bias, self._normalize_qk,
                               heads=self.num_heads, bank_size=self.bank_size, head_width=self.head_value_width)

    # -- fused inference path -----------------------------------------------------------
    def _fused_weights(self):
        """One weight and bias for every linear map of ``hidden`` the layer makes
        (q, k, v, the first f_proj factor, b, w, both route roles, the output
        gate), concatenated along the outputs and cached while the parameters
        keep their storage and version.  Returns (weight, bias, column offsets)."""
        router = self.shared_router
        parts = [self.q_proj.weight, self.k_proj.weight, self.v_proj.weight, self.f_proj[0].weight,
                 self.b_proj.weight, self.w_proj.weight]
        tracked = parts + [router.base.weight, router.base.bias, router.read_residual.weight,
                           router.read_residual.bias, router.write_residual.weight, router.write_residual.bias,
                           self.output_gate.weight, self.output_gate.bias]
        key = tuple((t.data_ptr(), t._version, t.dtype) for t in tracked)
        if self._fused_cache is None or self._fused_cache[0] != key:
            with torch.no_grad():
                read_w = router.base.weight + router.read_residual.weight
                write_w = router.base.weight + router.write_residual.weight
                weight = torch.cat(parts + [read_w, write_w, self.output_gate.weight], 0).contiguous()
                plain = sum(t.shape[0] for t in parts)
                bias = torch.cat([torch.zeros(plain, device=weight.device, dtype=weight.dtype),
                                  router.base.bias + router.read_residual.bias,
                                  router.base.bias + router.write_residual.bias, self.output_gate.bias])
            names = ('q', 'k', 'v', 'f', 'b', 'w', 'read', 'write', 'gate')
            widths = [t.shape[0] for t in parts] + [read_w.shape[0], write_w.shape[0], self.output_gate.weight.shape[0]]
            columns, at = {}, 0
            for name, width in zip(names, widths):
                columns[name] = at
                at += width
            self._fused_cache = (key, weight, bias, columns)
        return self._fused_cache[1:]

    def _fused_supported(self, hidden: Tensor) -> bool:
        return (hidden.dtype in (torch.bfloat16, torch.float32) and self.A_log.dtype == self.dt_bias.dtype
                and self.bank_size in (8, 16, 32) and self.value_width % 8 == 0 and self.value_width <= 4096
                and self.output_norm_weight.dtype in (torch.bfloat16, torch.float32))

    def _fused_controllers(self, hidden: Tensor, proj: Tensor | None = None):
        """Inference controllers, route scores and the output-gate projection from
        one projection GEMM and the controller epilogue (heads.py:11-22).
        ``proj``: the projection already computed (hidden then only gives the
        leading shape)."""
        weight, bias, cols = self._fused_weights()
        lead = hidden.shape[:-1]
        if proj is None:
            proj = ops.linear(hidden.reshape(-1, self.hidden_size), weight, bias)
        hv, rw = self.head_value_width, self.factor_route_width
        f = ops.linear(proj[:, cols['f']:cols['f'] + hv], self.f_proj[1].weight)
        q, k, v, g, b, w = ops.controller_epilogue(proj, f, cols, self.A_log, self.dt_bias, heads=self.num_heads,
                                                   bank_size=self.bank_size, head_width=hv,
                                                   qk_norm=self.config.qk_normalization)
        heads = (*lead, self.num_heads)
        controllers = (q.view(*heads, self.bank_size), k.view(*heads, self.bank_size), v.view(*heads, hv),
                       g.view(*heads, self.bank_size), b.view(*heads, self.bank_size), w.view(*heads, hv))
        read_scores = proj[:, cols['read']:cols['read'] + rw].view(*lead, rw)
        write_scores = proj[:, cols['write']:cols['write'] + rw].view(*lead, rw)
        gate = proj[:, cols['gate']:cols['gate'] + self.value_width]
        return controllers, (read_scores, write_scores), gate

    def _inference_inputs(self, hidden: Tensor):
        """The controllers and route scores prefill and step use: the fused
        projection and epilogue where the geometry allows, the torch ops
        otherwise.  Returns ((q, k, v, g, b, w), (read scores, write scores),
        the output-gate projection or None)."""
        if self._fused_supported(hidden):
            return self._fused_controllers(hidden)
        return self._controllers(hidden), self._route_projections(hidden), None

    def _inference_output(self, hidden: Tensor, gate, raw: Tensor) -> Tensor:
        return self._fused_output(gate, raw) if gate is not None else self._project_bank_output(hidden, raw)

    def _fused_output(self, gate: Tensor, raw: Tensor) -> Tensor:
        """_project_bank_output (_parameters.py:222-232) with the normalization
        and gate in one epilogue kernel, then o_proj."""
        layer = self.config.output_normalization == 'layer'
        normalized = ops.output_epilogue(raw.reshape(-1, self.value_width), gate, self.output_norm_weight,
                                         self.output_norm_bias if layer else None, eps=self.norm_eps,
                                         kind='layer' if layer else 'rms')
        return ops.linear(normalized, self.o_proj.weight, self.o_proj.bias).view(*raw.shape[:-1], -1)

    def _output_norm(self):
        """The output normalization's weight, bias (None for RMS), eps and kind."""
        layer = self.config.output_normalization == 'layer'
        return (self.output_norm_weight, self.output_norm_bias if layer else None, self.norm_eps,
                'layer' if layer else 'rms')

    def _project_bank_output(self, hidden: Tensor, raw: Tensor) -> Tensor:
        """LN (or RMS) x sigmoid gate -> o_proj (_parameters.py:222-232)."""
        return self.o_proj(_output_ops(raw, self.output_gate(hidden), *self._output_norm()))

    def _state_heads(self, state: Tensor) -> Tensor:
        return state.reshape(self.bank_count, self.num_heads, self.bank_size, self.head_value_width)

    # -- forward (model.py:88-140) ----------------------------------------------------
    def bank_reads(self, hidden: Tensor) -> Tensor:
        """The routed-memory path: concatenated head reads y [B, T, V]."""
        q, k, v, g, b, w = self._controllers(hidden)
        read_routes, write_routes = self._route_projections(hidden)
        (ww, wi), (rw, ri) = self._route_both(write_routes, read_routes)
        state = self._state_heads(self.materialize_initial_state())
        operator = bank_training if self.config.routed_decay else role_bank_training
        return operator(q, k, v, g, b, w, wi, ww, ri, rw, state, self.bank_count, self.bank_size ** -0.5,
                        compact_replay=self.compact_replay,
                        state_dtype=getattr(torch, self.config.training_state_dtype))

    def forward(self, hidden: Tensor) -> Tensor:
        if hidden.ndim != 3 or hidden.shape[-1] != self.hidden_size or hidden.shape[1] == 0:
            raise ValueError('hidden must be [batch, positive time, dim]')
        if not hidden.is_cuda:
            raise ValueError('the hip backend requires ROCm tensors; the CPU oracle lives in oracle/')
        if not torch.is_grad_enabled() and self._fused_supported(hidden):
            return self._forward_inference(hidden)
        if torch.is_grad_enabled() and self._fused_training_supported(hidden):
            return self._forward_training(hidden)
        return self._project_bank_output(hidden, self.bank_reads(hidden))

    def _fused_training_supported(self, hidden: Tensor) -> bool:
        """Whether the autograd forward may project once and run the fused
        controller and output kernels: BF16 throughout (FP32 keeps torch's exact
        exponentials and divisions), 16-byte column groups, and no call that the
        one product stands for is another than this file's: the projections are
        plain linear maps of plain tensors without hooks (their own or global
        ones) or a forward of their instance, and neither a subclass nor the
        instance has methods of its own for the path."""
        def plain(m, kind):
            return type(m) is kind and 'forward' not in m.__dict__ and not (
                m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks)

        if (hidden.dtype != torch.bfloat16 or torch.is_autocast_enabled('cuda') or not self._fused_supported(hidden)
                or self.head_value_width % 8 or self.factor_route_width % 8 or _global_hooks()
                or any(getattr(type(self), n) is not getattr(BankedDeltaMemory, n) or n in self.__dict__
                       for n in _TRAINING_METHODS)):
            return False
        pair, router = self.f_proj, self.shared_router
        if not (plain(pair, nn.Sequential) and len(pair) == 2 and plain(router, SharedResidualRouter)
                and not {'read', 'write'} & router.__dict__.keys()):
            return False
        unbiased = (self.q_proj, self.k_proj, self.v_proj, *pair, self.b_proj, self.w_proj)
        biased = (router.base, router.read_residual, router.write_residual)
        if not all(plain(m, nn.Linear) and m._parameters.keys() == {'weight', 'bias'}
                   and (m._parameters['bias'] is None) is without
                   for group, without in ((unbiased, True), (biased, False)) for m in group):
            return False
        own = [t for m in (self, *unbiased, *biased) for t in m._parameters.values() if t is not None]
        return (type(hidden) in (Tensor, nn.Parameter)
                and all(type(t) in (Tensor, nn.Parameter) and t.dtype == torch.bfloat16 and t.device == hidden.device
                        for t in own))

    def _forward_training(self, hidden: Tensor) -> Tensor:
        """forward under autograd: the projections that the operator reads as one,
        by the concatenated weights (so that their gradients are one product
        each), the controllers and the output interface as one kernel each way.
        The output gate stays a call of its own: its gradients then do not
        depend on the operator's, as those of o_proj and the norm."""
        router, lead = self.shared_router, hidden.shape[:-1]
        parts = [self.q_proj.weight, self.k_proj.weight, self.v_proj.weight, self.f_proj[0].weight,
                 self.b_proj.weight, self.w_proj.weight, router.base.weight + router.read_residual.weight,
                 router.base.weight + router.write_residual.weight]
        columns, at = {}, 0
        for name, part in zip(('q', 'k', 'v', 'f', 'b', 'w', 'read', 'write'), parts):
            columns[name], at = at, at + part.shape[0]
        bias = torch.cat([router.base.bias.new_zeros(columns['read']), router.base.bias + router.read_residual.bias,
                          router.base.bias + router.write_residual.bias])
        proj = F.linear(hidden.reshape(-1, self.hidden_size), torch.cat(parts), bias)
        hv, rw, heads = self.head_value_width, self.factor_route_width, (*lead, self.num_heads)
        geometry = dict(heads=self.num_heads, bank_size=self.bank_size, head_width=hv, route_width=rw,
                        qk_norm=self.config.qk_normalization)
        q, k, v, g, b, w, read, write = _LayerInputs.apply(proj, self.f_proj[1].weight, self.A_log, self.dt_bias,
                                                           columns, geometry)
        (ww, wi), (rw_, ri) = self._route_both(write.view(*lead, rw), read.view(*lead, rw))
        state = self._state_heads(self.materialize_initial_state())
        operator = bank_training if self.config.routed_decay else role_bank_training
        raw = operator(q.view(*heads, self.bank_size), k.view(*heads, self.bank_size), v.view(*heads, hv),
                       g.view(*heads, self.bank_size), b.view(*heads, self.bank_size), w.view(*heads, hv),
                       wi, ww, ri, rw_, state, self.bank_count, self.bank_size ** -0.5,
                       compact_replay=self.compact_replay,
                       state_dtype=getattr(torch, self.config.training_state_dtype))
        gate, raw = self.output_gate(hidden), raw.reshape(*lead, self.value_width)
        if type(gate) is not Tensor or gate.dtype != raw.dtype or gate.shape != raw.shape:  # a gate of another kind
            return self.o_proj(_output_ops(raw, gate, *self._output_norm()))
        normalized = _OutputInterface.apply(*(ops._aligned(t.reshape(-1, self.value_width)) for t in (raw, gate)),
                                            *self._output_norm())
        return self.o_proj(normalized.view(*lead, self.value_width))

    def _forward_inference(self, hidden: Tensor) -> Tensor:
        """forward without autograd: the projections through one GEMM and the
        controller epilogue, both routes in one launch, the routed operator's
        forward (the training state and rounding policy of bank_reads, no
        snapshots) and the output interface in one epilogue before o_proj --
        about a third of the launches of the autograd path."""
        controllers, (read_routes, write_routes), gate = self._fused_controllers(hidden)
        (ww, wi), (rw, ri), meta = self._route_and_dispatch(write_routes, read_routes)
        q, k, v, g, b, w = controllers
        state = self._state_heads(self.materialize_initial_state())
        # the routed operator's forward (bank_training, routed_update.py:16-53)
        # on this dispatch: its state policy, no snapshots under no_grad
        interval = _round_interval(self.bank_size, getattr(torch, self.config.training_state_dtype),
                                   self.compact_replay, q.dtype)
        raw = ops.routed_forward(q, k, v, g, b, w, wi, ww, ri, rw, state, meta, bank_count=self.bank_count,
                                 scale=self.bank_size ** -0.5, routed_decay=self.config.routed_decay,
                                 round_interval=interval)
        return self._fused_output(gate, raw)

    # -- stateful inference (inference.py:88-194) -----------------------------------
    def _cache_shape(self, batch: int) -> tuple[int, ...]:
        if self.num_heads == 1:
            return (batch, self.bank_count, self.bank_size, self.value_width)
        return (batch, self.bank_count, self.num_heads, self.bank_size, self.head_value_width)

    def _validate_stateful(self, hidden: Tensor, state: Tensor | None) -> None:
        if not hidden.is_cuda:
            raise ValueError('Stateful inference requires the HIP backend on a ROCm device')
        if hidden.ndim != 3 or hidden.shape[1] == 0 or hidden.shape[-1] != self.hidden_size:
            raise ValueError('hidden must be [batch, positive time, dim]')
        if state is not None and (tuple(state.shape) != self._cache_shape(hidden.shape[0])
                                  or state.dtype not in (torch.float32, torch.bfloat16)
                                  or state.device != hidden.device or not state.is_contiguous()):
            raise ValueError('state must be contiguous FP32 or BF16 [batch, banks, (heads,) rows, values] '
                             'on the input device')

    def create_state(self, batch: int, *, dtype=torch.bfloat16) -> Tensor:
        """Initial cache: factors added in parameter dtype, stored in ``dtype``
        (inference.py:100-107, product_routed_update.py:10-21)."""
        if dtype not in (torch.float32, torch.bfloat16):
            raise ValueError('cache dtype must be FP32 or BF16')
        with torch.no_grad():
            total = (self.initial_row_factor[:, None, :] + self.initial_column_factor[None, :, :])
            # the sum is in parameter dtype; widening BF16 to FP32 and back is
            # exact, so only a change of dtype converts
            initial = total if total.dtype == dtype else total.float().to(dtype)
            initial = initial.reshape(self._cache_shape(1)[1:]).unsqueeze(0)
            if batch == 1:
                return initial.contiguous()
            return initial.expand(batch, *initial.shape[1:]).contiguous()

    def prefill(self, hidden: Tensor, state: Tensor | None = None, *, state_dtype=None):
        """Process a prefix; BF16 cache storage (the default) rounds at handoff.
        Recurrence arithmetic is FP32 with no interior rounding (forward_rows.py:176-184)."""
        self._validate_stateful(hidden, state)
        if torch.is_grad_enabled():
            raise RuntimeError('Stateful inference requires no_grad or inference_mode')
        cache_dtype = state_dtype or (state.dtype if state is not None else torch.bfloat16)
        if cache_dtype not in (torch.float32, torch.bfloat16):
            raise ValueError('cache dtype must be FP32 or BF16')
        if state is None:
            work = torch.float32 if self.initial_row_factor.dtype != cache_dtype else cache_dtype
            state = self.create_state(hidden.shape[0], dtype=work)
        elif state_dtype is not None and state_dtype != state.dtype:
            raise ValueError('state_dtype must match the supplied cache')
        (q, k, v, g, b, w), (read_routes, write_routes), gate = self._inference_inputs(hidden)
        (ww, wi), (rw, ri), meta = self._route_and_dispatch(write_routes, read_routes)
        heads_view = state.view(hidden.shape[0], self.bank_count, self.num_heads, self.bank_size,
                                self.head_value_width)
        raw = ops.routed_forward(q, k, v, g, b, w, wi, ww, ri, rw, heads_view, meta,
                                 bank_count=self.bank_count, scale=self.bank_size ** -0.5,
                                 routed_decay=self.config.routed_decay, round_interval=0,
                                 final_state=heads_view)
        if state.dtype != cache_dtype:
            state = state.to(cache_dtype)
        return self._inference_output(hidden, gate, raw), state

    def step(self, hidden: Tensor, state: Tensor):
        """Advance an existing bank state by one token (inference only)."""
        self._validate_stateful(hidden, state)
        if torch.is_grad_enabled() or hidden.shape[1] != 1:
            raise ValueError('step requires one token under no_grad/inference_mode')
        if self._fused_supported(hidden):
            weight, bias, cols = self._fused_weights()
            proj = ops.linear(hidden.reshape(-1, self.hidden_size), weight, bias)
            gate = proj[:, cols['gate']:cols['gate'] + self.value_width]
            raw = self._decode_fused(proj, state)
            if raw is None:
                controllers, scores, gate = self._fused_controllers(hidden, proj=proj)
                raw = self._decode_banks(controllers, scores, hidden.shape[0], state)
            return self._fused_output(gate, raw.unsqueeze(1)), state
        (q, k, v, g, b, w), (read_routes, write_routes), gate = self._inference_inputs(hidden)
        raw = self._decode_banks((q, k, v, g, b, w), (read_routes, write_routes), hidden.shape[0], state)
        return self._inference_output(hidden, gate, raw.unsqueeze(1)), state

    def _decode_fused(self, proj: Tensor, state: Tensor) -> Tensor | None:
        """The step's controller epilogue, routes and decode kernel in one
        launch from the fused projection ``proj`` [B, P]: the bank reads [B, V],
        or None where ``ops.decode_fused`` does not take the geometry."""
        if not self.fused_decode or self.num_reads != self.num_writes:
            return None
        _, _, cols = self._fused_weights()
        rows, hv = proj.shape[0], self.head_value_width
        heads_view = state.view(rows, self.bank_count, self.num_heads, self.bank_size, hv)
        geometry = dict(heads=self.num_heads, bank_size=self.bank_size, head_width=hv, bank_count=self.bank_count,
                        selected_banks=self.num_writes)
        options = dict(qk_norm=self.config.qk_normalization, routed_decay=self.config.routed_decay,
                       scale=self.bank_size ** -0.5)
        f_weight = self.f_proj[1].weight
        # f_proj's second factor inside the launch where it takes it (one GEMM node fewer)
        if ops.decode_fused_supported(proj, None, cols, self.A_log, self.dt_bias, heads_view, **geometry,
                                      f_weight=f_weight):
            return ops.decode_fused(proj, None, cols, self.A_log, self.dt_bias, heads_view, **geometry, **options,
                                    f_weight=f_weight)
        f = ops.linear(proj[:, cols['f']:cols['f'] + hv], f_weight)
        if not ops.decode_fused_supported(proj, f, cols, self.A_log, self.dt_bias, heads_view, **geometry):
            return None
        return ops.decode_fused(proj, f, cols, self.A_log, self.dt_bias, heads_view, **geometry, **options)

    def _decode_banks(self, controllers, scores, batch: int, state: Tensor) -> Tensor:
        """Both routes and the decode kernel of one step: the bank reads [B, V]."""
        q, k, v, g, b, w = controllers
        read_routes, write_routes = scores
        width = read_routes.shape[-1]
        if (batch == 1 and self.num_reads == self.num_writes and read_routes.stride(-1) == 1
                and write_routes.data_ptr() == read_routes.data_ptr() + width * read_routes.element_size()):
            # one token: its read and write scores are adjacent slices of the
            # projection row, so both roles route in one launch, as two rows
            pair = torch.as_strided(read_routes, (1, 2, width), (2 * width, width, 1))
            weights, indices = self._route(pair, self.num_reads)
            rw, ww = weights[:, 0:1], weights[:, 1:2]
            ri, wi = indices[:, 0:1], indices[:, 1:2]
        else:
            (ww, wi), (rw, ri) = self._route_both(write_routes, read_routes)
        heads_view = state.view(batch, self.bank_count, self.num_heads, self.bank_size, self.head_value_width)
        return ops.decode_step(q[:, 0], k[:, 0], v[:, 0], g[:, 0], b[:, 0], w[:, 0], wi[:, 0], ww[:, 0],
                               ri[:, 0], rw[:, 0], heads_view, bank_count=self.bank_count,
                               scale=self.bank_size ** -0.5, routed_decay=self.config.routed_decay)

    def step_fused_norm(self, hidden: Tensor, delta: Tensor | None, norm_weight: Tensor, norm_eps: float,
                        state: Tensor):
        """The memory sublayer of a pre-norm block for one decode token, with the
        block's residual add and RMSNorm formed inside the projection GEMV and
        the output interface inside the o_proj GEMV (``bdm_gemv_ex``):
        h = hidden + delta (delta None: h = hidden), out = step(RMSNorm(h)).
        Returns (out, h).  It matches the unfused kernels within tolerance:
        the decode launch forms f itself in another summation order, and the
        layer-norm prologue may differ from the standalone kernel by an ulp."""
        weight, bias, _ = self._fused_weights()
        rows = hidden.shape[0]
        flat = hidden.reshape(rows, self.hidden_size)
        if delta is None:
            proj = ops.gemv_fused(flat, weight, bias, prologue='rms', norm_weight=norm_weight, eps=norm_eps)
            new_hidden = hidden
        else:
            proj, total = ops.gemv_fused(delta.reshape(rows, self.hidden_size), weight, bias, prologue='rms',
                                         residual=flat, norm_weight=norm_weight, eps=norm_eps)
            new_hidden = total.view_as(hidden)
        _, _, cols = self._fused_weights()
        gate = proj[:, cols['gate']:cols['gate'] + self.value_width]
        raw = self._decode_fused(proj, state)
        if raw is None:
            controllers, scores, gate = self._fused_controllers(new_hidden, proj=proj)
            raw = self._decode_banks(controllers, scores, rows, state)
        layer = self.config.output_normalization == 'layer'
        out = ops.gemv_fused(raw, self.o_proj.weight, self.o_proj.bias,
                             prologue='out_layer' if layer else 'out_rms', norm_weight=self.output_norm_weight,
                             norm_bias=self.output_norm_bias if layer else None, gate=gate, eps=self.norm_eps)
        return out.view(rows, 1, self.hidden_size), new_hidden

    def step_fused_norm_supported(self, hidden: Tensor, norm_weight: Tensor) -> bool:
        rows = hidden.shape[0]
        return (hidden.is_cuda and hidden.dim() == 3 and hidden.shape[1] == 1 and 1 <= rows <= ops.GEMV_MAX_ROWS
                and self._fused_supported(hidden) and self.hidden_size % 8 == 0
                and max(self.hidden_size, self.value_width) <= ops.GEMV_PROLOGUE_MAX_K
                and self.o_proj.weight.dtype == hidden.dtype and self.q_proj.weight.dtype == hidden.dtype
                and norm_weight.dtype in (torch.bfloat16, torch.float32)
                and (self.o_proj.bias is None or self.o_proj.bias.dtype == hidden.dtype))
