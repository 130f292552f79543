"""The native operators (csrc/torch_ops.cpp) against the Python ones on the same kernels: same bits,
forward and gradients; calls they decline reach the Python operator's checks."""

import pytest
import torch

from helpers import make_acts, make_params

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("batch", [1, 3])
@pytest.mark.parametrize("op", ["step", "gated", "norm"])
def test_native_operator_equals_the_python_operator(op, batch, dtype):
    import gridnet_amd as ga
    from gridnet_amd.layernorm import GridLayerNormFn

    w, b, r = (t.to(DEV, dtype) for t in make_params((8, 16, 8), seed=3))
    x, gy = (make_acts(batch, (8, 16, 8), seed=s).to(DEV, dtype) for s in (4, 5))
    if op == "step":
        native, python, params = ga.gridnet_step, ga.GridnetCudaOp.apply, [w, b, r, x]
        rest = (2, 8, 1e-5, True, "silu")
    elif op == "gated":
        native, python = ga.gated_gridnet_step, ga.GatedGridnetCudaOp.apply
        params, rest = [torch.stack([w, w.flip(0)], 1), torch.stack([b, r]), x], (2, 8, "tanh")
    else:
        native, python, params, rest = ga.grid_layer_norm, GridLayerNormFn.apply, [x, r, b], (1e-5,)
    results = []
    for f in (native, python):
        leaves = [p.clone().requires_grad_(True) for p in params]
        y = f(*leaves, *rest)
        y.backward(gy)
        results.append([y.detach(), *[p.grad for p in leaves]])
    tol = dict(rtol=0, atol=0) if dtype is torch.float32 or op == "norm" else dict(rtol=1e-12, atol=1e-12)
    for got, want in zip(*results):  # fp64 dx is built with atomics
        torch.testing.assert_close(got, want, **tol)
    with torch.no_grad():
        assert not native(*params, *rest).requires_grad


def test_native_step_refuses_what_the_python_operator_refuses():
    import gridnet_amd as ga

    w, b, r = (t.to(DEV) for t in make_params((8, 8, 8), seed=3))
    x = make_acts(2, (8, 8, 8), seed=4).to(DEV)
    with pytest.raises(AssertionError, match="mismatching dtypes"):
        ga.gridnet_step(w, b.double(), r, x, 1, 8)
    assert ga.gridnet_step(w, b, r, x[:0], 1, 8).shape == (0, 8, 8, 8)
    y = ga.gridnet_step(w.requires_grad_(True), b, r, x, 1, 8)
    with pytest.raises(RuntimeError, match="outGrads must be contiguous"):
        y.sum().backward()  # an expanded gradient
    y = ga.gridnet_step(w, b, r, x, 1, 8)
    with torch.no_grad():
        w.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        y.backward(torch.ones_like(y))


def operators():
    """(native operator, Python operator, tensor arguments, the rest) of each."""
    import gridnet_amd as ga
    from gridnet_amd.layernorm import GridLayerNormFn

    w, b, r = (t.to(DEV) for t in make_params((8, 8, 8), seed=3))
    x = make_acts(2, (8, 8, 8), seed=4).to(DEV)
    return [(ga.gridnet_step, ga.GridnetCudaOp.apply, [w, b, r, x], (1, 8, 1e-5, False, "silu")),
            (ga.gated_gridnet_step, ga.GatedGridnetCudaOp.apply, [torch.stack([w, w.flip(0)], 1), torch.stack([b, r]), x],
             (1, 8, "tanh")),
            (ga.grid_layer_norm, GridLayerNormFn.apply, [x, r, b], (1e-5,))]


def forward_mode(f, tensors, rest, k):
    import torch.autograd.forward_ad as fwd

    with fwd.dual_level():
        args = [fwd.make_dual(t, torch.ones_like(t)) if i == k else t for i, t in enumerate(tensors)]
        return fwd.unpack_dual(f(*args, *rest)).tangent


def jvp(f, tensors, rest, k):
    def of(t):
        return f(*tensors[:k], t, *tensors[k + 1:], *rest)

    return torch.func.jvp(of, (tensors[k],), (torch.ones_like(tensors[k]),))[1]


def reverse(f, tensors, rest, k):
    return torch.func.grad(lambda t: f(*tensors[:k], t, *tensors[k + 1:], *rest).square().sum())(tensors[k])


def batched(f, tensors, rest, k):
    return torch.func.vmap(lambda t: f(*tensors[:k], t, *tensors[k + 1:], *rest))(torch.stack([tensors[k]] * 2))


@pytest.mark.parametrize("through", [forward_mode, jvp, reverse, batched], ids=lambda f: f.__name__)
@pytest.mark.parametrize("which", [0, 1, 2], ids=["step", "gated", "norm"])
def test_what_the_python_operators_refuse_is_not_answered_without_derivatives(which, through):
    """The operators have no forward-mode rule and no rule for function transforms: the Python ones say
    so, and the native ones leave such calls to them, whichever argument is concerned."""
    native, python, tensors, rest = operators()[which]
    for k in range(len(tensors)):
        raised = []
        for f in (native, python):
            with pytest.raises((RuntimeError, NotImplementedError)) as info:
                through(f, tensors, rest, k)
            raised.append(info.type)
        assert raised[0] is raised[1]


class Marked(torch.Tensor):
    pass


@pytest.mark.parametrize("which", [0, 1, 2], ids=["step", "gated", "norm"])
def test_tracing_and_subclasses_see_the_operator(which):
    native, python, tensors, rest = operators()[which]
    k = 0 if which == 2 else len(tensors) - 1  # the activations
    marked = [t.as_subclass(Marked) if i == k else t for i, t in enumerate(tensors)]
    assert type(native(*marked, *rest)) is type(python(*marked, *rest)) is Marked
    with torch.no_grad():
        # a trace that does not see the operator would hold its result as a constant
        traced = torch.jit.trace(lambda t: native(*tensors[:k], t, *tensors[k + 1:], *rest), tensors[k], check_trace=False)
        other = 2 * tensors[k] + 1
        assert torch.equal(traced(other), python(*tensors[:k], other, *tensors[k + 1:], *rest))


@pytest.mark.parametrize("which", [0, 1, 2], ids=["step", "gated", "norm"])
def test_saved_tensor_hooks_see_everything_that_is_kept(which):
    native, python, tensors, rest = operators()[which]
    results = []
    for f in (native, python):
        kept = []

        def pack(t):
            kept.append(tuple(t.shape))
            return t.cpu()

        leaves = [t.clone().requires_grad_(True) for t in tensors]
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t.to(DEV)):
            y = f(*leaves, *rest)
        y.backward(torch.ones_like(y))
        results.append((kept, [t.grad for t in leaves]))
    assert results[0][0] == results[1][0]
    for got, want in zip(results[0][1], results[1][1]):
        assert torch.equal(got, want)
