"""The bf16 channel-wise ``GatedDeltaLayer`` as one autograd node.

The layer is launch-bound between its kernels: as separate torch modules it is
about 80 launches and 20 autograd nodes forward and backward, 1.0 to 1.5 ms of
host time, as long as its GPU work at 8 clips.  Here

* the six maps that read x (q, k, v, f_proj_1, g_proj_1, b_proj) are one GEMM on
  their stacked weights, and one GEMM returns dx (no per-map dx sums);
* the stacking and the fp32 copies of the small parameters are one launch
  (``kda_layer_pack``), as are the bf16 roundings of their gradients;
* every weight gradient is formed by one launch (``weight_grads``).

``GatedDeltaLayer.forward`` runs this only where it is what the separate modules
compute (``fused_params``); everything else keeps the general path.
"""
from __future__ import annotations

from typing import List, Optional, Tuple

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.autograd import forward_ad
from torch.nn.modules import module as _nn_module

from . import _lib
from .kda import _DTYPE_CODE, _stream, chunk_kda, kda_backward, kda_backward_train, kda_forward, kda_forward_train

_PLAIN_TENSORS = (torch.Tensor, nn.Parameter)
# positions in ``fused_params``' order: those whose gradient comes through the
# recurrence (all but g_proj_1, g_proj_2, o_proj, the gate's bias and the norm
# weight)
_BEFORE_RECURRENCE = (0, 1, 2, 3, 5, 6, 10, 11, 12, 13, 14, 15, 17, 18)


def _plain_module(m: nn.Module, cls: type) -> bool:
    """m is exactly a cls whose call is its forward: no subclass (a
    parametrization makes one), hooks or instance override."""
    return (type(m) is cls and "forward" not in m.__dict__ and not m._forward_hooks and not m._forward_pre_hooks
            and not m._backward_hooks and not m._backward_pre_hooks)


def fused_params(layer, x: torch.Tensor, state: Optional[torch.Tensor]) -> Optional[Tuple[torch.Tensor, ...]]:
    """The layer's parameters in ``fused_layer``'s order, or None where the
    general path has to run: other dtypes than bf16 activations and weights,
    autocast or tracing, module hooks, replaced modules, tensor subclasses."""
    from .layer import GatedDeltaLayer, RMSNormGated, ShortCausalConv1d
    if x.dtype != torch.bfloat16 or x.device.type != "cuda" or x.numel() == 0 or type(x) not in _PLAIN_TENSORS:
        return None
    # a trace records the launches of an autograd node, none of those made outside one
    if torch.is_autocast_enabled("cuda") or torch.compiler.is_compiling() or torch._C._is_tracing():
        return None
    # forward-mode tangents: the autograd nodes refuse them, the kernels would drop them
    if forward_ad._current_level >= 0:
        return None
    if (_nn_module._global_forward_hooks or _nn_module._global_forward_pre_hooks
            or _nn_module._global_backward_hooks or _nn_module._global_backward_pre_hooks):
        return None
    if type(layer).produce is not GatedDeltaLayer.produce or "produce" in layer.__dict__:
        return None
    linears = (layer.q_proj, layer.k_proj, layer.v_proj, layer.f_proj_1, layer.g_proj_1, layer.b_proj,
               layer.f_proj_2, layer.g_proj_2, layer.o_proj)
    convs = (layer.q_conv1d, layer.k_conv1d, layer.v_conv1d)
    if not (all(_plain_module(m, nn.Linear) for m in linears) and all(type(c) is ShortCausalConv1d for c in convs)
            and _plain_module(layer.o_norm, RMSNormGated)):
        return None
    if any(m.bias is not None for m in linears if m is not layer.g_proj_2) or layer.g_proj_2.bias is None:
        return None
    if any(c.bias is None for c in convs):
        return None
    weights = [m.weight for m in linears] + [layer.g_proj_2.bias]
    small = [c.weight for c in convs] + [c.bias for c in convs] + [layer.o_norm.weight, layer.dt_bias, layer.A_log]
    dev = x.device
    for p in weights:
        if p.dtype != torch.bfloat16 or type(p) not in _PLAIN_TENSORS or p.device != dev or not p.is_contiguous():
            return None
    for p in small:
        if p.dtype not in _DTYPE_CODE or type(p) not in _PLAIN_TENSORS or p.device != dev or not p.is_contiguous():
            return None
    hidden, total, D, H = layer.hidden_size, layer.total_dim, layer.head_dim, layer.num_heads
    rank = layer.f_proj_1.weight.shape[0]
    shapes = [(total, hidden)] * 3 + [(rank, hidden), (D, hidden), (H, hidden), (total, rank), (total, D),
                                      (hidden, total), (total,)]
    if any(tuple(p.shape) != s for p, s in zip(weights, shapes)):
        return None
    # the weight-gradient kernel reads 8 columns at a time and forms rows of 8
    if hidden % 8 or rank % 8 or total % 8 or D % 8:
        return None
    if state is not None and (type(state) not in _PLAIN_TENSORS or state.device != dev):
        return None
    return (*weights, *small)


def _pack(jobs: List[Tuple[torch.Tensor, int, int]]) -> None:
    """One launch of copies with conversion: (source, destination address,
    destination dtype code)."""
    from .layer import _i64
    arr = _i64([(s.data_ptr(), dst, s.numel(), _DTYPE_CODE[s.dtype] | dd << 8) for s, dst, dd in jobs])
    _lib.check(_lib.load().kda_layer_pack(arr, len(jobs), _stream(jobs[0][0].device)), "kda_layer_pack")


def _views(fp: torch.Tensor, HD: int, D: int):
    """(conv_w, conv_b, norm weight, dt_bias, A_log) of the packed fp32 parameters."""
    from .layer import CONV_TAPS
    return (fp[:12 * HD].view(3, HD, CONV_TAPS), fp[12 * HD:15 * HD].view(3, HD), fp[15 * HD:15 * HD + D],
            fp[15 * HD + D:16 * HD + D], fp[16 * HD + D:])


def _forward(x, state, spec, params, train: bool, keep: bool):
    """(out, new_state, what the backward reads, the training pair's workspace).
    Without ``keep`` each tensor is given up after its last use."""
    from .layer import gated_rmsnorm_forward, producer_forward
    H, D, scale, mult, eps, chunk = spec
    wq, wk, wv, wf1, wg1, wb, wf2, wg2, wo, bg2 = params[:10]
    B, L, hidden = x.shape
    M, HD, rank = B * L, H * D, wf1.shape[0]
    N = 3 * HD + rank + D + H
    NP = -(-N // 8) * 8
    dev, bf = x.device, torch.bfloat16
    x2 = x.contiguous().view(M, hidden)
    # rows past N of the stacked weight are not written: the columns they give
    # are not read
    wcat = torch.empty((NP, hidden), dtype=bf, device=dev)
    fp = torch.empty(16 * HD + D + H, dtype=torch.float32, device=dev)
    jobs, at = [], wcat.data_ptr()
    for w in (wq, wk, wv, wf1, wg1, wb):
        jobs.append((w, at, 1))
        at += 2 * w.numel()
    at = fp.data_ptr()
    for p in params[10:]:   # conv weights, conv biases, norm weight, dt_bias, A_log
        jobs.append((p, at, 0))
        at += 4 * p.numel()
    _pack(jobs)
    conv_w, conv_b, nw, dt_bias, A_log = _views(fp, HD, D)

    P = torch.mm(x2, wcat.t())
    P3 = P.view(B, L, NP)
    xf = torch.mm(P[:, 3 * HD:3 * HD + rank], wf2.t()).view(B, L, HD)
    z = torch.addmm(bg2, P[:, 3 * HD + rank:3 * HD + rank + D], wg2.t()).view(B, L, HD)
    q, k, v, g, beta = producer_forward(P3[..., :3 * HD], xf, P3[..., N - H:N], conv_w, conv_b, dt_bias, A_log,
                                        H, D, scale, mult, torch.float32)
    if not keep:
        x2 = P = P3 = xf = wcat = None
    ws = None
    if train:
        o, s_final, ws = kda_forward_train(q, k, v, g, beta, state, chunk)
    else:
        o, s_final = kda_forward(q, k, v, g, beta, state, chunk)
    if not keep:
        q = k = v = g = beta = None
    y = gated_rmsnorm_forward(o, z, nw, eps)
    if not keep:
        o = z = None
    # no view of the product: a node's output that is one refuses in-place operations
    out = F.linear(y, wo)
    return out, s_final, (x2, P, xf, z, q, k, v, g, beta, state, o, y, wcat, fp, wf2, wg2, wo), ws


def _by_modules(x, state, spec, params):
    """What ``GatedDeltaLayer.forward`` computes map by map, one autograd node each."""
    from .layer import CONV_TAPS, GatedRMSNormFunction, ProducerFunction
    H, D, scale, mult, eps, chunk = spec
    wq, wk, wv, wf1, wg1, wb, wf2, wg2, wo, bg2, *small = params
    conv_w = torch.stack([w.reshape(H * D, CONV_TAPS) for w in small[:3]])
    nw, dt_bias, A_log = small[6:]
    q, k, v, g, beta = ProducerFunction.apply(
        F.linear(x, torch.cat([wq, wk, wv])), F.linear(F.linear(x, wf1), wf2), F.linear(x, wb), conv_w,
        torch.stack(small[3:6]), dt_bias, A_log, H, D, scale, mult, torch.float32)
    o, s_final = chunk_kda(q, k, v, g, beta, state, chunk)
    gate = F.linear(F.linear(x, wg1), wg2, bg2)
    return F.linear(GatedRMSNormFunction.apply(o, gate, nw, eps), wo), s_final


def fused_layer(x, state, spec, params):
    """(out, new_state) of the layer for x (B, L, hidden).  ``spec`` = (H, D, scale,
    beta_mult, eps, chunk_size); ``params`` as ``fused_params`` orders them."""
    if torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in (x, state, *params)):
        if x.is_inference():
            return _by_modules(x, state, spec, params)   # a node cannot save it
        return FusedLayerFunction.apply(x, state, spec, *params)
    return _forward(x, state, spec, params, False, False)[:2]


class FusedLayerFunction(torch.autograd.Function):
    """``fused_layer`` with a gradient for every input.  A part of the backward runs
    only where a gradient needs it (frozen parameters, as autograd would skip
    its modules); with nothing before the output norm trained the forward keeps
    no factors, and the new state does not require grad."""

    @staticmethod
    def forward(ctx, x, state, spec, *params):
        need = ctx.needs_input_grad
        # what reaches the recurrence: x, every map and gate of its operands, the state
        ctx.need_prod = need[0] or any(need[3 + i] for i in _BEFORE_RECURRENCE)
        ctx.need_rec = ctx.need_prod or need[1]
        out, s_final, saved, ctx.ws = _forward(x, state, spec, params, ctx.need_rec, True)
        ctx.need_norm = ctx.need_rec or need[19] or any(need[3 + i] for i in (4, 7, 9))   # or the gate's maps
        if not ctx.need_rec:
            ctx.mark_non_differentiable(s_final)
            x2, P, xf, z, q, k, v, g, beta, s0, o, *rest = saved
            saved = (x2 if need[7] else None, P if need[10] or need[12] else None, None, z if ctx.need_norm else None,
                     None, None, None, None, None, None, o if ctx.need_norm else None, *rest)
        ctx.save_for_backward(*saved, x, state)
        ctx.params, ctx.versions = params, [p._version for p in params]
        ctx.spec, ctx.shape = spec, (*x.shape, params[3].shape[0])
        ctx.small = [(p.dtype, p.shape) for p in params[10:]]
        ctx.set_materialize_grads(False)
        return out, s_final

    @staticmethod
    def backward(ctx, dout, ds_final):
        if torch.is_grad_enabled():
            return FusedLayerFunction._backward_with_graph(ctx, dout, ds_final)
        return FusedLayerFunction._backward(ctx, dout, ds_final)

    @staticmethod
    def _backward_with_graph(ctx, dout, ds_final):
        """``create_graph``: through the separate nodes, whose gradients keep a graph
        where theirs do (the linear maps; the kernels' adjoints have none)."""
        x, state = ctx.saved_tensors[-2:]
        if [p._version for p in ctx.params] != ctx.versions:
            raise RuntimeError("a parameter of the layer was modified in place before its backward")
        outs = zip(_by_modules(x, state, ctx.spec, ctx.params), (dout, ds_final))
        outs, cots = zip(*[(t, c) for t, c in outs if c is not None])
        inputs = (x, state, None, *ctx.params)
        got = iter(torch.autograd.grad(outs, [t for t, n in zip(inputs, ctx.needs_input_grad) if n], cots,
                                       create_graph=True, allow_unused=True))
        return tuple(next(got) if n else None for n in ctx.needs_input_grad)

    @staticmethod
    def _backward(ctx, dout, ds_final):
        from .layer import gated_rmsnorm_backward, producer_backward, weight_grads
        x2, P, xf, z, q, k, v, g, beta, s0, o, y, wcat, fp, wf2, wg2, wo, _, _ = ctx.saved_tensors
        H, D, scale, mult, eps, chunk = ctx.spec
        B, L, hidden, rank = ctx.shape
        M, HD, NP = B * L, H * D, wcat.shape[0]
        N = 3 * HD + rank + D + H
        f1, g1 = slice(3 * HD, 3 * HD + rank), slice(3 * HD + rank, 3 * HD + rank + D)
        dev, dt = wo.device, wo.dtype
        need_x, need_ds0, need = ctx.needs_input_grad[0], ctx.needs_input_grad[1], ctx.needs_input_grad[3:]
        conv_w, conv_b, nw, dt_bias, A_log = _views(fp, HD, D)
        grads: List[Optional[torch.Tensor]] = [None] * 19
        small: List[Optional[torch.Tensor]] = [None] * 9   # the gradients of params[10:], fp32
        used = dout is not None   # else: only the new state was, and the maps behind the output get no gradient
        if used:
            dout2 = dout.to(dt).contiguous().view(M, hidden)
            if ctx.need_norm:
                dy = torch.mm(dout2, wo).view(B, L, HD)
                do, dz, small[6] = gated_rmsnorm_backward(o, z, nw, eps, dy)
                dz2 = dz.view(M, HD)
                del dy, dz
        elif ctx.need_rec:
            do = torch.zeros_like(o)
        dx = ds0 = None
        if ctx.need_rec:
            if ctx.ws is not None:
                dq, dk, dv, dg, dbeta, ds0 = kda_backward_train(q, k, v, g, beta, s0, do, ds_final, ctx.ws, chunk,
                                                                _need_ds0=need_ds0)
                ctx.ws = None
            else:   # another backward of a retained graph
                dq, dk, dv, dg, dbeta, ds0 = kda_backward(q, k, v, g, beta, s0, do, ds_final, chunk,
                                                          _need_ds0=need_ds0)
            do = None
        if ctx.need_prod or need[4]:
            dP = torch.empty((M, NP), dtype=dt, device=dev)
        if ctx.need_prod:
            P3, dP3 = P.view(B, L, NP), dP.view(B, L, NP)
            _, dxf, _, dcw, dcb, ddt, dA = producer_backward(
                P3[..., :3 * HD], xf, P3[..., N - H:N], conv_w, conv_b, dt_bias, A_log, dq, dk, dv, dg, dbeta, H, D,
                scale, mult, _dqkv=dP3[..., :3 * HD], _dxb=dP3[..., N - H:N])
            small[:6], small[7:] = [*dcw, *dcb], [ddt, dA]
            dq = dk = dv = dg = None
            dxf2 = dxf.view(M, HD)
            if need_x or need[3]:
                torch.mm(dxf2, wf2, out=dP[:, f1])
        if need_x or need[4]:
            if used:
                torch.mm(dz2, wg2, out=dP[:, g1])
            else:
                dP[:, g1].zero_()
        if need_x:
            dx = torch.mm(dP[:, :N], wcat[:N]).view(B, L, hidden)

        # the weight gradients: one problem for each run of adjacent maps of x that need one
        sizes = [HD, HD, HD, rank, D, H]
        if used and all(need[:10]):
            (dwcat, _), (grads[6], _), (grads[7], grads[9]), (grads[8], _) = weight_grads(
                [(dP[:, :N], x2, False), (dxf2, P[:, f1], False), (dz2, P[:, g1], True),
                 (dout2, y.view(M, HD), False)], M)
            grads[:6] = dwcat.split(sizes)
        elif any(need[:10]):
            runs: List[List[int]] = []   # first column and end of P, first map and end
            at = 0
            for i, j, want in ((0, 3, any(need[:3])), (3, 4, need[3]), (4, 5, need[4] and used), (5, 6, need[5])):
                end = at + (3 * HD if j == 3 else sizes[i])
                if want and runs and runs[-1][3] == i:
                    runs[-1][1], runs[-1][3] = end, j
                elif want:
                    runs.append([at, end, i, j])
                at = end
            problems = [(dP[:, a:b], x2, False) for a, b, _, _ in runs]
            into = []
            if need[6]:
                into.append(6)
                problems.append((dxf2, P[:, f1], False))
            if used and (need[7] or need[9]):
                into.append(7)
                problems.append((dz2, P[:, g1], True))
            if used and need[8]:
                into.append(8)
                problems.append((dout2, y.view(M, HD), False))
            dw = weight_grads(problems, M) if problems else []
            for (_, _, i, j), (d, _) in zip(runs, dw):
                grads[i:j] = d.split(sizes[i:j])
            for m, (d, db) in zip(into, dw[len(runs):]):
                grads[m] = d
                if db is not None:
                    grads[9] = db
        jobs = []
        for i, (t, (dtype, shape)) in enumerate(zip(small, ctx.small)):
            if t is None or not need[10 + i]:
                continue
            if dtype == torch.float32:
                grads[10 + i] = t.view(shape)
            else:
                grads[10 + i] = torch.empty(shape, dtype=dtype, device=dev)
                jobs.append((t, grads[10 + i].data_ptr(), _DTYPE_CODE[dtype]))
        if jobs:
            _pack(jobs)
        return (dx, ds0, None, *(t if n else None for t, n in zip(grads, need)))
