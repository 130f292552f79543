"""What this framework's performance is measured on: the calls its users make, from one small
inference step to a training step of the largest chain, each with the sizes it is used at.

A case is a dict of plain values.  ``kind`` says which entry point it goes through:

  ``step``      ``Gridnet`` on a grid of its own: one outer step, forward or forward + backward
  ``chain``     ``BodyRunner(fused=True)``: the loop step, LayerNorm on buffers the caller keeps
  ``mnist``     ``MnistGridModel``: embedding, loop, readout; serving, or a training step
  ``imagenet``  ``ImageNetGridModel``: the same with a patch embedding, both shapes of the loop,
                parameters shared by the outer steps or one set for each
"""

import math

import torch
import torch.nn.functional as F

import gridnet_amd
from gridnet_amd.models import ImageNetGridModel, MnistGridModel
from gridnet_amd.runner import BodyRunner

DEVICE = "cuda"
ACTIVATIONS = ("silu", "leaky_relu", "relu", "tanh")


def _step(name, m, n, k, batch, inner, block=8, train=True, normalize=True, activation="silu", dtype="float32"):
    return dict(name=name, kind="step", m=m, n=n, k=k, block=block, batch=batch, inner=inner, train=train,
                normalize=normalize, activation=activation, dtype=dtype)


def _chain(name, grid, batch, inner, outer, train, block=8, activation="leaky_relu"):
    return dict(name=name, kind="chain", m=grid, n=grid, k=grid, block=block, batch=batch, inner=inner,
                outer=outer, train=train, activation=activation)


def _mnist(name, batch, inner, outer, train, gated=False, activation="silu"):
    return dict(name=name, kind="mnist", batch=batch, inner=inner, outer=outer, train=train, gated=gated,
                activation=activation)


def _imagenet(name, grid, batch, inner, outer, residual, separate, train=True, activation="leaky_relu"):
    return dict(name=name, kind="imagenet", grid=grid, batch=batch, inner=inner, outer=outer,
                residual=residual, separate=separate, train=train, activation=activation)


def listed():
    return [
        # the smallest call: one step of a small grid on one sample, the module's defaults
        _step("step_serve_16", 16, 16, 16, batch=1, inner=2, train=False),
        # the shape of the reference's own benchmark of the op: two samples, ten inner iterations
        _step("step_train_32", 32, 32, 32, batch=2, inner=10),
        # a grid that is no cube and no power of two, an odd batch, the module's defaults
        _step("step_train_ragged", 40, 48, 56, batch=13, inner=4),
        # double precision: what gradient checks and reference runs use
        _step("step_train_f64", 24, 32, 32, batch=6, inner=3, normalize=False, activation="tanh", dtype="float64"),
        # one digit classified by the MNIST model at its script's defaults: 64 outer steps
        _mnist("mnist_serve_1", batch=1, inner=1, outer=64, train=False),
        # a training step of the same model at its script's batch size
        _mnist("mnist_train_256", batch=256, inner=1, outer=64, train=True),
        # the same script's gated network
        _mnist("mnist_train_gated", batch=256, inner=1, outer=64, train=True, gated=True, activation="tanh"),
        # batched inference on a small and on the largest grid
        _chain("chain_infer_32", 32, batch=64, inner=4, outer=8, train=False),
        _chain("chain_infer_128", 128, batch=8, inner=4, outer=16, train=False),
        # the benchmark's training chain, and the largest one, in 4^3 blocks
        _chain("chain_train_64", 64, batch=32, inner=4, outer=12, train=True),
        _chain("chain_train_64_block4", 64, batch=128, inner=8, outer=16, train=True, block=4),
        # the ImageNet script with its two options: residual loop, parameters of each step's own
        _imagenet("imagenet_train_64", 64, batch=32, inner=8, outer=12, residual=True, separate=True),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def _fits(case, most):
    return _cells(case) * case["batch"] * case["inner"] * case.get("outer", 1) <= most


def draw(rng):
    kind = rng.choice(("step", "step", "step_f64", "mnist", "gated", "infer", "train", "train", "imagenet"))
    if kind in ("step", "step_f64"):
        f64 = kind == "step_f64"
        block = rng.choice((4, 8, 8))
        low, high = 16 // block, (40 if f64 else 64) // block
        m, n, k = (block * rng.randint(low, high) for _ in range(3))
        batch = _log_int(rng, 1, 12 if f64 else 32)
        return _unnamed(_step("", m, n, k, batch, rng.randint(1, 10 if not f64 else 4), block,
                              train=rng.random() < 0.7, normalize=rng.random() < 0.6,
                              activation=rng.choice(ACTIVATIONS), dtype="float64" if f64 else "float32"))
    if kind in ("mnist", "gated"):
        gated = kind == "gated"
        return _unnamed(_mnist("", _log_int(rng, 1, 256), rng.choice((1, 1, 2, 3)) if not gated else 1,
                               _log_int(rng, 8, 64), train=rng.random() < 0.6, gated=gated,
                               activation="tanh" if gated else rng.choice(("silu", "leaky_relu"))))
    if kind == "imagenet":
        return _unnamed(_imagenet("", rng.choice((32, 64)), _log_int(rng, 2, 32), rng.randint(2, 8),
                                  rng.randint(4, 12), residual=rng.random() < 0.5,
                                  separate=rng.random() < 0.5, train=rng.random() < 0.8))
    train = kind == "train"
    while True:
        block = rng.choice((4, 8, 8)) if train else 8
        m, n, k = (block * rng.randint(32 // block, (64 if train else 128) // block) for _ in range(3))
        case = _chain("", 0, _log_int(rng, 2, 128), rng.randint(1, 8), rng.randint(4, 16), train, block,
                      activation=rng.choice(("leaky_relu", "silu")))
        case.update(m=m, n=n, k=k)
        # no more than the largest listed chain of its direction
        if _fits(case, 1 << 32 if train else 1 << 30) and m * n * k * case["batch"] <= (1 << 25 if train else 1 << 24):
            return _unnamed(case)


def _unnamed(case):
    del case["name"]
    return case


def _cells(case):
    if case["kind"] == "mnist":
        return 32 ** 3
    if case["kind"] == "imagenet":
        return case["grid"] ** 3
    return case["m"] * case["n"] * case["k"]


class _Inputs:
    """Random tensors on the GPU from one seed."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def normal(self, *shape, mean=0.0, std=1.0, dtype=torch.float32):
        return torch.randn(*shape, generator=self.gen, device=DEVICE, dtype=dtype).mul_(std).add_(mean)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.gen, device=DEVICE)

    def labels(self, batch, classes):
        return torch.randint(0, classes, (batch,), generator=self.gen, device=DEVICE)


def _fill_parameters(module, rnd):
    """Parameters as they are some way into a training run: at the scale of their initialisation,
    no two alike, biases off zero and LayerNorm weights off one."""
    with torch.no_grad():
        for name, p in module.named_parameters():
            if name.endswith("residual_scale"):
                p.copy_(rnd.normal(*p.shape, mean=0.5, std=0.05, dtype=p.dtype))
            elif name.endswith("norm.weight"):
                p.copy_(rnd.normal(*p.shape, mean=1.0, std=0.1, dtype=p.dtype))
            elif name.endswith("bias"):
                p.copy_(rnd.normal(*p.shape, std=0.1, dtype=p.dtype))
            elif name == "init_in":
                p.copy_(rnd.normal(*p.shape, dtype=p.dtype))
            else:
                fan_in = p[0].numel() if p.dim() in (2, 4) and "network" not in name and p.shape[0] != 27 else 27
                p.copy_(rnd.normal(*p.shape, std=1.0 / math.sqrt(fan_in), dtype=p.dtype))


def prepare(case, seed):
    rnd = _Inputs(seed)
    kind, batch = case["kind"], case["batch"]
    state = {"case": case}
    if kind == "step":
        dtype = getattr(torch, case["dtype"])
        shape = (case["m"], case["n"], case["k"])
        net = gridnet_amd.Gridnet(shape, case["inner"], case["block"], device=DEVICE, dtype=dtype,
                                  normalize=case["normalize"], activation=case["activation"])
        _fill_parameters(net, rnd)
        state.update(model=net, x=rnd.normal(batch, *shape, dtype=dtype))
        if case["train"]:
            state["x"].requires_grad_(True)
            state["grad"] = rnd.normal(batch, *shape, dtype=dtype)
    elif kind == "chain":
        shape = (case["m"], case["n"], case["k"])
        weight = rnd.normal(27, *shape, std=1.0 / math.sqrt(27))
        bias, scale = rnd.normal(*shape, std=0.1), rnd.normal(*shape, mean=1.0, std=0.1)
        gamma, beta = rnd.normal(*shape, mean=1.0, std=0.1), rnd.normal(*shape, std=0.1)
        if case["train"]:
            x = rnd.normal(batch, *shape)
            state["grad"] = rnd.normal(batch, *shape)
        else:  # an image on the first face of an empty grid
            x = torch.zeros(batch, *shape, device=DEVICE)
            x[..., 0] = rnd.normal(batch, *shape[:2])
        state["x"] = x
        state["model"] = BodyRunner(weight, bias, scale, gamma, beta, batch, case["inner"], case["outer"],
                                    case["block"], case["activation"], backward=case["train"], fused=True)
    elif kind == "mnist":
        model = MnistGridModel(case["inner"], case["outer"], 1.0, 0.5, case["activation"], case["gated"], 1.0,
                               torch.device(DEVICE), fused_body=not case["gated"])
        _fill_parameters(model, rnd)
        state.update(model=model, x=rnd.uniform(batch, 1, 28, 28), labels=rnd.labels(batch, 10))
    else:
        model = ImageNetGridModel(inner_iters=case["inner"], outer_iters=case["outer"],
                                  outer_residual=case["residual"], init_scale=1.0, residual_scale=0.5,
                                  emb_channels=16, grid_size=case["grid"], activation=case["activation"],
                                  separate_params=case["separate"], device=torch.device(DEVICE), fused_body=True)
        _fill_parameters(model, rnd)
        state.update(model=model, x=rnd.normal(batch, 3, 256, 256), labels=rnd.labels(batch, 1000))
    return state


def run(state):
    case, model, x = state["case"], state["model"], state["x"]
    if case["kind"] == "chain":
        y = model.forward(x)
        return [y, *model.backward(state["grad"])] if case["train"] else [y]
    if not case["train"]:
        with torch.no_grad():
            return [model(x)]
    model.zero_grad(set_to_none=True)
    if case["kind"] == "step":
        x.grad = None
        y = model(x)
        y.backward(state["grad"])
        return [y.detach(), x.grad] + [p.grad for p in model.parameters()]
    logits = model(x)
    F.cross_entropy(logits, state["labels"]).backward()
    return [logits.detach()] + [p.grad for p in model.parameters()]


def work(case):
    kind, cells, batch = case["kind"], _cells(case), case["batch"]
    size = 8 if case.get("dtype") == "float64" else 4
    gated, outer = case.get("gated", False), case.get("outer", 1)
    sets = outer if case.get("separate") else 1
    planes = sets * (56 if gated else 29)           # weights, bias, scale (the gated net: two nets, no scale)
    taps = 54 if gated else 27
    flops = 2.0 * taps * cells * batch * case["inner"] * outer
    if kind != "step":
        planes += 2                                 # the LayerNorm's weight and bias
    if kind in ("step", "chain"):
        ends_in, ends_out, extra = batch * cells, batch * cells, 0
    else:                                           # images in, logits out; embedding and readout parameters
        g = 32 if kind == "mnist" else case["grid"]
        image, classes = (784, 10) if kind == "mnist" else (3 * 65536, 1000)
        patch = 0 if kind == "mnist" else 16 * (3 * (256 // g) ** 2 + 1)
        ends_in, ends_out, extra = batch * image, batch * classes, cells + g * g * (classes + 2) + classes + patch
    params = planes * cells + extra
    if not case["train"]:
        return {"bytes": float(size * (params + ends_in + ends_out)), "flops": flops}
    # the backward: gradient of the inputs and of the weights, twice the forward's operations
    if kind in ("step", "chain"):                   # and the gradient in, the gradient of the input out
        ends_in, ends_out = 2 * ends_in, 2 * ends_out
    return {"bytes": float(size * (2 * params + ends_in + ends_out)), "flops": 3 * flops}


def tolerance(case):
    if case.get("dtype") == "float64":
        return {"rel": 1e-12}
    if case["train"] and case["activation"] in ("relu", "leaky_relu"):
        # The derivative jumps at zero: a pre-activation that rounds to the other side of it changes
        # its cell's gradients outright.  Two ways of computing the same chain in fp32 (step by step
        # with torch's autograd, LayerNorm folded in) differ by up to 9e-4 here, single entries by 0.25.
        return {"rel": 2e-3, "max": 0.5}
    # fp32 sums, iterated; a chain carries the rounding of every step through all later ones
    return {"rel": 1e-5}
