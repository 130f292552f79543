"""The body the reference's models repeat: outer step, then LayerNorm, ``outer`` times.

gridnet/scripts/train_mnist.py:62-64 and gridnet/scripts/train_imagenet.py:76-86 (including
the ``outer_residual`` variant ``n = norm(h); h = h + (net(n) - n)``); parameters are shared
across the outer iterations.  Embedding and readout are the callers' business.
"""

import torch
import torch.nn as nn
from torch.autograd.function import once_differentiable


class FusedBodyOp(torch.autograd.Function):
    """The whole loop as ONE autograd node on the entry points that fold the LayerNorm into the
    step kernels (``gridnet_hip_fused_*`` / ``gridnet_hip_chain_backward``): what
    ``BodyRunner(fused=True)`` does on buffers of its own, with torch's autograd around it.
    float32, ``normalize=False``, at least one inner iteration; other set-ups keep to the
    op-by-op loop.  ``params`` is one (weight, bias, residual_scale) triple shared by all outer
    steps, or ``outer_iterations`` triples in a row (the reference's ``--separate_params``).
    Every call owns its buffers (the raw outputs of all outer steps are what the backward needs),
    so several forwards may be outstanding before their backwards run."""

    @staticmethod
    def forward(ctx, x0, gamma, beta, inner_iterations, outer_iterations, block_size, activation,
                outer_residual, *params):
        from .runner import BodyRunner

        if len(params) not in (3, 3 * outer_iterations):
            raise ValueError("one (weight, bias, residual_scale) triple, or one per outer step")
        need_grad = any(ctx.needs_input_grad)
        for name, t in [("norm.weight", gamma), ("norm.bias", beta)] + \
                [(("weight", "bias", "residual_scale")[k % 3], t) for k, t in enumerate(params)]:
            if not t.is_contiguous():
                raise RuntimeError(f"{name} must be contiguous")
        detached = [t.detach() for t in params]
        separate = len(params) > 3
        sets = [detached[k::3] for k in range(3)] if separate else detached
        run = BodyRunner(*sets, gamma.detach(), beta.detach(), x0.shape[0], inner_iterations,
                         outer_iterations, block_size, activation, backward=need_grad, fused=True,
                         outer_residual=outer_residual)
        y = run.forward(x0.detach().contiguous())
        ctx.run = run if need_grad else None
        ctx.separate = separate
        if need_grad:
            # the runner reads these tensors again in the backward (it recomputes from them):
            # registering them lets autograd refuse a backward after an in-place change, such as
            # an optimizer step taken while this forward was still outstanding
            ctx.save_for_backward(x0, gamma, beta, *params)
        return y

    @staticmethod
    @once_differentiable
    def backward(ctx, grad_out):
        run, ctx.run = ctx.run, None
        if run is None:
            raise RuntimeError("FusedBodyOp: the buffers of this forward were released by its first "
                               "backward; a second backward (retain_graph=True) is not supported")
        ctx.saved_tensors  # raises if an input was modified in place since the forward
        # checked: the one-launch chain backward reports through a status word whether its bounded
        # waits held (read after a synchronisation; a failed launch is repeated step by step)
        dw, db, dr, dgamma, dbeta, dx0 = run.backward_checked(grad_out.contiguous())
        if ctx.separate:
            grads = [g for triple in zip(dw, db, dr) for g in triple]
        else:
            grads = [dw, db, dr]
        return (dx0, dgamma, dbeta, None, None, None, None, None, *grads)


def fused_body(h, network, norm, outer_iterations: int, outer_residual: bool = False):
    """``outer_iterations`` x (``network``, ``norm``) on ``h`` through :class:`FusedBodyOp`.
    ``network``: a :class:`gridnet_amd.Gridnet` with ``normalize=False`` whose parameters all
    iterations share, or a sequence of ``outer_iterations`` of them (one per iteration, alike
    but for their parameter values); ``norm`` a :class:`gridnet_amd.GridLayerNorm`."""
    nets = list(network) if isinstance(network, (list, tuple, nn.ModuleList)) else [network]
    if len(nets) not in (1, outer_iterations):
        raise ValueError("one network, or one per outer iteration")
    first = nets[0]
    for net in nets:
        if net.normalize:
            raise RuntimeError("the fused body covers normalize=False only")
        if (net.inner_iterations, net.block_size, net.activation) != \
                (first.inner_iterations, first.block_size, first.activation):
            raise ValueError("the networks of a fused body differ only in their parameter values")
    params = [p for net in nets for p in (net.weight, net.bias, net.residual_scale)]
    return FusedBodyOp.apply(h, norm.weight, norm.bias, first.inner_iterations, outer_iterations,
                             first.block_size, first.activation, outer_residual, *params)


class GatedBodyOp(torch.autograd.Function):
    """The loop over a gated step with one inner iteration and its LayerNorm as one autograd node, on
    ``gridnet_hip_rows_chain_*``: a kernel per step and direction, the LayerNorm and the accumulation of
    the shared parameters' gradients inside them.  It keeps four tensors per step for the backward where
    the modules one after the other keep two (8.6 GB at 32^3, batch 256, 64 steps)."""

    @staticmethod
    def forward(ctx, x0, weight, bias, gamma, beta, outer_iterations, activation, eps):
        from . import native as _n

        x0 = x0.contiguous()
        batch, (m, n, k) = x0.shape[0], x0.shape[1:]
        keep = any(ctx.needs_input_grad)
        act = _n.activation_id(activation)
        out = torch.empty_like(x0)
        y_raw = stats = saved = None
        if keep:
            y_raw = torch.empty((outer_iterations, *x0.shape), dtype=x0.dtype, device=x0.device)
            saved = torch.empty((outer_iterations, 3, *x0.shape), dtype=x0.dtype, device=x0.device)
            stats = torch.empty((outer_iterations, batch, 2), dtype=x0.dtype, device=x0.device)
        with torch.cuda.device(x0.device):
            nbytes = _n.lib.gridnet_hip_rows_chain_workspace_bytes(batch, m, n, k, 1, int(keep), 0)
            ws = _n.workspace(nbytes, x0.device)
            _n.check(_n.lib.gridnet_hip_rows_chain_forward(
                weight.data_ptr(), bias.data_ptr(), None, gamma.data_ptr(), beta.data_ptr(), x0.data_ptr(),
                *([t.data_ptr() for t in (y_raw, stats, saved)] if keep else [None] * 3), out.data_ptr(),
                batch, m, n, k, outer_iterations, 1, float(eps), act, ws.data_ptr(), nbytes,
                _n.current_stream(x0)))
        if keep:
            ctx.save_for_backward(x0, weight, bias, gamma, beta, y_raw, stats, saved)
            ctx.outer_iterations, ctx.act = outer_iterations, act
        return out

    @staticmethod
    @once_differentiable
    def backward(ctx, grad_out):
        from . import native as _n

        x0, weight, bias, gamma, beta, y_raw, stats, saved = ctx.saved_tensors
        batch, (m, n, k) = x0.shape[0], x0.shape[1:]
        dy = grad_out.contiguous()
        grads = [torch.empty_like(t) for t in (x0, weight, bias, gamma, beta)]
        dx, dw, db, dgamma, dbeta = (t.data_ptr() for t in grads)
        with torch.cuda.device(x0.device):
            nbytes = _n.lib.gridnet_hip_rows_chain_workspace_bytes(batch, m, n, k, 1, 1, 1)
            ws = _n.workspace(nbytes, x0.device)
            _n.check(_n.lib.gridnet_hip_rows_chain_backward(
                weight.data_ptr(), None, gamma.data_ptr(), beta.data_ptr(), x0.data_ptr(), y_raw.data_ptr(),
                stats.data_ptr(), saved.data_ptr(), dy.data_ptr(), dw, db, None, dgamma, dbeta, dx,
                batch, m, n, k, ctx.outer_iterations, 1, ctx.act, _n.OVERWRITE_PARAMS, ws.data_ptr(), nbytes,
                _n.current_stream(x0)))
        return (*grads, None, None, None)


_HOOKS = ("forward", "forward_pre", "backward", "backward_pre")


def _as_defined(module, cls):
    """Nothing is passed by where ``module.forward`` is not called: ``cls`` itself and no subclass, no
    ``forward`` of the instance's own, not compiled, and no hook, its own or for all modules."""
    hooks = [getattr(module, f"_{kind}_hooks", None) for kind in _HOOKS]
    hooks += [getattr(nn.modules.module, f"_global_{kind}_hooks") for kind in _HOOKS]
    return (type(module) is cls and "forward" not in vars(module) and not any(hooks) and
            getattr(module, "_compiled_call_impl", None) is None)


def _rows_cover(h, network, norm, outer_iterations):
    """Whether :class:`GatedBodyOp` computes what the modules, called one after the other, would."""
    from . import GatedGridnet
    from . import native as _n
    from .layernorm import GridLayerNorm

    if not (_as_defined(network, GatedGridnet) and _as_defined(norm, GridLayerNorm)):
        return False
    params = (network.weight, network.bias, norm.weight, norm.bias)
    if outer_iterations < 1 or not (h.is_cuda and h.is_contiguous() and h.dim() == 4 and h.shape[0]):
        return False
    shape = tuple(h.shape[1:])
    if not all(isinstance(t, torch.Tensor) and t.is_contiguous() and t.dtype == h.dtype == torch.float32 and
               t.device == h.device for t in params):
        return False
    return (tuple(t.shape for t in params) == ((27, 2, *shape), (2, *shape), shape, shape) and
            network.block_size in (4, 8) and not any(n % network.block_size for n in shape) and
            bool(_n.lib.gridnet_hip_rows_chain_supported(_n.F32, *shape, network.inner_iterations, 0, 1)))


def gated_body(h, network, norm, outer_iterations: int, rows=None):
    """``outer_iterations`` x (``network``, ``norm``) on ``h``: a :class:`gridnet_amd.GatedGridnet` and a
    :class:`gridnet_amd.GridLayerNorm`, through :class:`GatedBodyOp` where that covers the problem and, with
    a backward to come, there is room for what it keeps (``rows=True``: without asking for room; ``False``:
    never); one after the other where not."""
    from .runner import room_for

    if rows is not False and _rows_cover(h, network, norm, outer_iterations) and (
            rows or not torch.is_grad_enabled() or
            room_for(4 * outer_iterations * h.numel() * h.element_size(), h.device)):
        return GatedBodyOp.apply(h, network.weight, network.bias, norm.weight, norm.bias, outer_iterations,
                                 network.activation, norm.eps)
    for _ in range(outer_iterations):
        h = norm(network(h))
    return h


class GridnetBody(nn.Module):
    def __init__(self, shape, inner_iterations: int, outer_iterations: int, block_size: int,
                 device, activation: str = "leaky_relu", normalize: bool = False,
                 init_scale: float = 1.0, residual_scale: float = 1.0,
                 outer_residual: bool = False, dtype=None, fused: bool = False):
        super().__init__()

        from . import Gridnet
        from .layernorm import GridLayerNorm

        dtype = dtype or torch.float32
        self.outer_iterations = outer_iterations
        self.outer_residual = outer_residual
        self.fused = fused  # one autograd node over the whole loop, see FusedBodyOp
        self.network = Gridnet(shape, inner_iterations, block_size, device=device, dtype=dtype,
                               init_scale=init_scale, residual_scale=residual_scale,
                               normalize=normalize, activation=activation)
        self.norm = GridLayerNorm(shape, device=device, dtype=dtype)

    def forward(self, h):
        if self.fused:
            return fused_body(h, self.network, self.norm, self.outer_iterations, self.outer_residual)
        for _ in range(self.outer_iterations):
            if self.outer_residual:
                nh = self.norm(h)
                h = h + (self.network(nh) - nh)
            else:
                h = self.norm(self.network(h))
        return h
