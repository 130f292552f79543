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


def test_without_room_the_shorter_history_is_kept(monkeypatch):
    """The loop by whole rows keeps twice the tensors: where they would take more than half of what is
    free, and where it is told not to, the modules (plain: the two-kernel chain) run, with the same results."""
    from gridnet_amd import runner

    m, x = model(), images()
    want = m(x)
    m.rows = False
    assert "GatedBodyOpBackward" not in nodes(m(x))
    m.rows = None
    params = [torch.ones(n, 8, 8, 16, device=DEV).squeeze(0) / 9 for n in (27, 1, 1, 1, 1)]
    acts = torch.randn(2, 8, 8, 16, generator=torch.Generator().manual_seed(2)).to(DEV)
    plain = runner.BodyRunner(*params, 2, 1, 3, 8, "silu", fused=True)
    assert plain.rows

    monkeypatch.setattr(runner, "UNASKED", 0)
    need = 4 * m.outer_iters * x.shape[0] * 32 ** 3 * 4
    for free, fits in ((3 * need, True), (need, False)):
        cached = torch.cuda.memory_reserved() - torch.cuda.memory_allocated()
        monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device: (free - cached, 0))
        y = m(x)
        assert ("GatedBodyOpBackward" in nodes(y)) == fits
        torch.testing.assert_close(y, want, rtol=1e-5, atol=1e-5)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda device: (1 << 60, 0))
    total = torch.cuda.get_device_properties(DEV).total_memory
    for more, fits in ((3 * need, True), (need, False)):  # within what the process may use
        share = (torch.cuda.memory_allocated() + more) / total
        monkeypatch.setattr(torch.cuda, "get_per_process_memory_fraction", lambda device: share)
        assert ("GatedBodyOpBackward" in nodes(m(x))) == fits
    with torch.no_grad():  # nothing is kept
        assert torch.equal(m(x), want)
    monkeypatch.setattr(runner, "room_for", lambda nbytes, device: False)
    short = runner.BodyRunner(*params, 2, 1, 3, 8, "silu", fused=True)
    assert not short.rows and runner.BodyRunner(*params, 2, 1, 3, 8, "silu", fused=True, rows=True).rows
    assert runner.BodyRunner(*params, 2, 1, 3, 8, "silu", fused=True, backward=False).rows
    torch.testing.assert_close(short.forward(acts), plain.forward(acts), rtol=1e-5, atol=1e-5)
    for a, b in zip(short.backward(acts), plain.backward(acts)):
        torch.testing.assert_close(a, b, rtol=1e-4, atol=1e-5)
