"""``gated_body`` takes the loop over as one autograd node only where the modules, called one after the
other, would do the same: whatever a user hangs on them, or puts in their place, is still called."""

import pytest
import torch
import torch.nn as nn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def model(seed=0):
    from gridnet_amd.models import MnistGridModel

    torch.manual_seed(seed)
    return MnistGridModel(1, 3, 1.0, 0.5, "tanh", True, 1.0, torch.device(DEV))


def images(batch=2):
    return torch.rand(batch, 1, 28, 28, generator=torch.Generator().manual_seed(1)).to(DEV)


def by_modules(m, x):
    h = m.embed(x)
    for _ in range(m.outer_iters):
        h = m.norm(m.network(h))
    return m.readout(h)


def nodes(y):
    seen, todo = set(), [y.grad_fn]
    while todo:
        f = todo.pop()
        if f is not None and f not in seen:
            seen.add(f)
            todo += [g for g, _ in f.next_functions]
    return {f.name() for f in seen}


def test_the_model_as_it_is_takes_one_node():
    m = model()
    assert "GatedBodyOpBackward" in nodes(m(images()))


def doubled(forward):
    return lambda *args: 2 * forward(*args)


@pytest.mark.parametrize("part", ["network", "norm"])
@pytest.mark.parametrize("how", ["subclass", "own forward", "hook", "pre-hook", "hook of all modules"])
def test_what_stands_in_the_place_of_a_module_is_called(part, how):
    from torch.nn.modules.module import register_module_forward_hook

    m, x, calls = model(), images(), []
    module = getattr(m, part)

    def hook(*args):
        calls.append(1)

    handle = None
    if how == "subclass":
        cls = type(module)
        module.__class__ = type("Own", (cls,), {"forward": lambda self, h: 2 * cls.forward(self, h)})
    elif how == "own forward":
        module.forward = doubled(module.forward)
    elif how == "hook":
        module.register_forward_hook(hook)
    elif how == "pre-hook":
        module.register_forward_pre_hook(hook)
    else:
        handle = register_module_forward_hook(hook)
    try:
        y = m(x)
        called = len(calls)
        assert torch.equal(y, by_modules(m, x))
    finally:
        if handle is not None:
            handle.remove()
    if how in ("hook", "pre-hook"):
        assert called == m.outer_iters
    elif how == "hook of all modules":
        assert called > 2 * m.outer_iters


def test_another_norm_and_a_strided_input():
    from gridnet_amd.network import gated_body

    m, x = model(), images()
    m.norm = nn.LayerNorm((32, 32, 32), elementwise_affine=False, device=DEV)
    assert torch.equal(m(x), by_modules(m, x))
    m = model()
    h = m.embed(x).transpose(1, 2)
    with pytest.raises(RuntimeError, match="must be contiguous"):
        gated_body(h, m.network, m.norm, 2)
