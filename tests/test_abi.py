"""CPU checks of the drop-in boundary: the library loads, exports what the header declares,
answers its host-only entry points, and the Python shim has the reference's call surface."""

import ctypes
import inspect
import os
import re
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HEADER = os.path.join(ROOT, "include", "gridnet_hip.h")


def declared_symbols():
    text = open(HEADER).read()
    text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
    return sorted(set(re.findall(r"\b(gridnet_hip_\w+)\s*\(", text)))


def test_header_declares_the_expected_entry_points():
    names = declared_symbols()
    for want in ("gridnet_hip_forward", "gridnet_hip_backward", "gridnet_hip_layernorm_forward",
                 "gridnet_hip_layernorm_backward", "gridnet_hip_last_error"):
        assert want in names


def test_library_exports_every_declared_symbol():
    from gridnet_amd import native

    lib = ctypes.CDLL(native.LIB_PATH)
    for name in declared_symbols():
        assert hasattr(lib, name), f"{name} declared in include/gridnet_hip.h but not exported"
    assert set(native.EXPORTS) == set(declared_symbols())


def test_host_only_entry_points():
    from gridnet_amd import native

    assert native.lib.gridnet_hip_version() >= 1
    assert [native.activation_id(n) for n in ("relu", "leaky_relu", "silu", "tanh")] == [0, 1, 2, 3]
    with pytest.raises(RuntimeError, match="unknown activation function: gelu"):
        native.activation_id("gelu")
    # argument validation happens before anything touches a device
    rc = native.lib.gridnet_hip_forward(0, 8, 8, 8, 8, 8, 2, 12, 8, 8, 1, 8, 1e-5, 0, 0, None)
    assert rc == 1 and "incompatible" in native.last_error()
    rc = native.lib.gridnet_hip_forward(0, 8, 8, 8, 8, 8, 2, 8, 8, 8, 1, 2, 1e-5, 0, 0, None)
    assert rc == 1 and "block_size" in native.last_error()
    rc = native.lib.gridnet_hip_backward(0, 8, 8, 8, 8, 8, 8, 8, 8, 8, 2, 8, 8, 8, 33, 8, 1e-5, 0,
                                         0, 0, None, 0, None)
    assert rc == 3
    assert native.last_error() == "cannot backprop through more than 32 inner iterations"
    rc = native.lib.gridnet_hip_forward(0, 8, 8, 8, 8, 8, 2, 8, 8, 8, 1, 8, 1e-5, 0, 7, None)
    assert rc == 2 and "unknown activation function" in native.last_error()
    # 32-bit cell indexing inside a sample: 27 * 432^3 is past 2^31, 27 * 424^3 is not
    rc = native.lib.gridnet_hip_forward(0, 8, 8, 8, 8, 8, 1, 432, 432, 432, 1, 8, 1e-5, 0, 0, None)
    assert rc == 1 and "grid too large" in native.last_error()
    rc = native.lib.gridnet_hip_forward(0, None, 8, 8, 8, 8, 1, 424, 424, 424, 1, 8, 1e-5, 0, 0, None)
    assert rc == 1 and "null input pointer" in native.last_error()
    # backward workspaces: one activation tensor (D) for the plain step, two floats per block and
    # batch element more with normalize, two tensors (D0, D1) for the gated step; none in fp64
    act = 32 * 64 ** 3 * 4
    assert native.lib.gridnet_hip_backward_workspace_bytes(0, 32, 64, 64, 64, 4, 8, 0) == act
    assert native.lib.gridnet_hip_backward_workspace_bytes(0, 32, 64, 64, 64, 4, 8, 1) == act + 32 * 512 * 8
    assert native.lib.gridnet_hip_backward_workspace_bytes(1, 32, 64, 64, 64, 4, 8, 0) == 0
    assert native.lib.gridnet_hip_backward_gated_workspace_bytes(0, 32, 64, 64, 64, 4, 8) == 2 * act
    assert native.lib.gridnet_hip_backward_gated_workspace_bytes(1, 32, 64, 64, 64, 4, 8) == 0
    # the history of more than 21 inner iterations does not fit the LDS at 8^3 blocks: generic kernels
    assert native.lib.gridnet_hip_backward_gated_workspace_bytes(0, 32, 64, 64, 64, 22, 8) == 0
    rc = native.lib.gridnet_hip_backward_gated(0, 8, 8, 8, 8, 8, 8, 8, 2, 8, 8, 8, 2, 8, 0, 0, None, 0, None)
    assert rc == 4 and "workspace" in native.last_error()
    rc = native.lib.gridnet_hip_backward(0, 8, 8, 8, 8, 8, 8, 8, 8, 8, 2, 8, 8, 8, 2, 8, 1e-5, 1, 0, 0,
                                         None, 0, None)
    assert rc == 4 and "workspace" in native.last_error()
    # the entry point on static scratch refuses, before touching a device, what its array cannot hold
    assert native.lib.gridnet_hip_backward_workspace_bytes(0, 64, 64, 64, 64, 4, 8, 0) > native.STATIC_SCRATCH_BYTES
    rc = native.lib.gridnet_hip_backward_static(0, 8, 8, 8, 8, 8, 8, 8, 8, 8, 64, 64, 64, 64, 4, 8, 1e-5,
                                                0, 0, 0, None)
    assert rc == 4 and "static array holds" in native.last_error()
    assert native.lib.gridnet_hip_layernorm_workspace_bytes(0, 32, 64 ** 3) == (32 * 64 * 2 + 64) * 4
    rc = native.lib.gridnet_hip_layernorm_forward(0, 8, 8, 8, 8, 8, 8, 4, 4096, 1e-5, None, 0, None)
    assert rc == 4 and "workspace" in native.last_error()


@pytest.mark.parametrize("block_size", [0, -1, -8, 3, 5, 16])
def test_size_queries_of_block_sizes_that_are_refused(block_size):
    """Callers ask for the size before the call that checks the arguments: the answer is 0, in every
    precision.  In a process of its own, for what must not happen there is that it dies."""
    queries = [f"gridnet_hip_backward_workspace_bytes({dt}, 4, 16, 16, 16, {inner}, {block_size}, {norm})"
               for dt in (0, 1, 2) for inner in (1, 2, 2000000) for norm in (0, 1)]
    queries += [f"gridnet_hip_backward_gated_workspace_bytes({dt}, 4, 16, 16, 16, 2, {block_size})" for dt in (0, 1)]
    queries += [f"gridnet_hip_fused_workspace_bytes(4, 16, 16, 16, 2, {block_size}, {b})" for b in (0, 1)]
    queries += [f"gridnet_hip_fused_forward_chain_workspace_bytes(4, 16, 16, 16, 2, {block_size})",
                f"gridnet_hip_chain_all_workspace_bytes(4, 16, 16, 16, 2, 4, {block_size})"]
    assert answers(queries) == [0] * len(queries)


@pytest.mark.parametrize("side,block_size", [(1, 4), (3, 4), (1, 8), (4, 8), (7, 8)])
def test_size_queries_of_grids_without_a_block(side, block_size):
    grid = f"{side}, {side}, {side}"
    queries = [f"gridnet_hip_backward_workspace_bytes({dt}, 4, {grid}, {inner}, {block_size}, {norm})"
               for dt in (0, 1) for inner in (1, 2) for norm in (0, 1)]
    queries += [f"gridnet_hip_backward_gated_workspace_bytes(0, 4, {grid}, 2, {block_size})"]
    queries += [f"gridnet_hip_fused_workspace_bytes(4, {grid}, {inner}, {block_size}, {b})" for inner in (1, 2) for b in (0, 1)]
    queries += [f"gridnet_hip_fused_forward_chain_workspace_bytes(4, {grid}, 2, {block_size})",
                f"gridnet_hip_fused_forward_chain_merges(0, 4, {grid}, 2, {block_size})",
                f"gridnet_hip_chain_forward_all_supported(0, 4, {grid}, 2, 4, {block_size}, 0)",
                f"gridnet_hip_chain_all_supported(0, 4, {grid}, 2, 4, {block_size}, 0)",
                f"gridnet_hip_chain_all_workspace_bytes(4, {grid}, 2, 4, {block_size})"]
    assert answers(queries) == [0] * len(queries)


def answers(queries):
    code = f"from gridnet_amd.native import lib\nfor q in {queries!r}: print(eval('lib.' + q), flush=True)"
    run = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True)
    got = [int(v) for v in run.stdout.split()]
    assert run.returncode == 0, f"status {run.returncode} at {queries[len(got)]}: {run.stderr}"
    return got


def test_native_operators_decline_tensors_without_data():
    """Fake device tensors have no memory behind them: the native operators leave them to the Python ones."""
    import torch
    from torch._subclasses.fake_tensor import FakeTensorMode

    from gridnet_amd import native

    with FakeTensorMode():
        w, p, x = (torch.empty(*s, 8, 8, 8, device="cuda") for s in ((27,), (), (2,)))
        gw, gp = torch.empty(27, 2, 8, 8, 8, device="cuda"), torch.empty(2, 8, 8, 8, device="cuda")

        def calls():
            return (native.ops.step(w, p, p, x, 1, 8, 1e-5, False, "silu"),
                    native.ops.gated_step(gw, gp, x, 1, 8, "tanh"), native.ops.layer_norm(x, p, p, 1e-5))

        assert calls() == (None, None, None)
    assert calls() == (None, None, None)  # nor outside the mode


def test_native_operators_and_library_of_different_builds_do_not_go_together(tmp_path):
    from gridnet_amd import native

    for op in (native.ops.step, native.ops.gated_step, native.ops.layer_norm):
        with pytest.raises(TypeError, match="stale"):
            op(1, 2)
    other = tmp_path / "other.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-x", "c", "-", "-o", str(other)], check=True,
                   input=b"int gridnet_hip_version(void) { return 8; }")
    with pytest.raises(ImportError, match="version 8 of the C ABI"):
        try:
            native.ops.bind(str(other))
        finally:
            native.ops.bind(native.LIB_PATH)


def test_a_workspace_of_the_largest_batch_serves_the_smaller_ones():
    """Kernels and chunks are chosen by the batch too; what a call needs must not be more at a smaller one.
    (The fused backward's figure holds room to split the batch beside what it cannot do without: a smaller
    workspace is accepted there.)"""
    from gridnet_amd import native

    for m in (8, 40, 48, 64):
        for k in (8, 16, 24, 32, 40, 56, 64, 72, 80, 96, 104, 128):
            for bs in (4, 8):
                for inner in (1, 2):
                    need = [native.lib.gridnet_hip_fused_workspace_bytes(b, m, 48, k, inner, bs, 0) for b in range(1, 66)]
                    assert need == sorted(need), (m, k, bs, inner)
            for gated, backward in ((0, 0), (0, 1), (1, 0), (1, 1)):
                need = [native.lib.gridnet_hip_rows_chain_workspace_bytes(b, m, 48, k, gated, 1, backward)
                        for b in range(1, 300)]
                assert need == sorted(need), (m, k, gated, backward)


def test_short_batches_of_small_blocks_have_room_to_be_split():
    """4^3 blocks: batches of two and three are walked by a wave per sample, which takes a copy of the 31 gradient planes
    for each; no smaller batch gets more room than a larger one."""
    from gridnet_amd import native

    for shape in ((8, 8, 8), (16, 16, 16), (16, 24, 32)):
        cells, last = shape[0] * shape[1] * shape[2], 0
        for batch in range(1, 40):
            room = native.lib.gridnet_hip_backward_workspace_bytes(0, batch, *shape, 4, 4, 0) - 4 * batch * cells
            if batch in (2, 3):
                assert room >= batch * 31 * 4 * cells, (shape, batch)
            assert room >= last, (shape, batch)
            last = room


def test_shim_has_the_reference_call_surface():
    """Positional signatures of src/gridnet_cuda.cpp:61-72, 91-106, 133-141, 160-171."""
    import gridnet_cuda

    assert list(inspect.signature(gridnet_cuda.forward).parameters) == [
        "weight", "bias", "scale", "initActivations", "outActivations", "innerIterations",
        "blockSize", "eps", "normalize", "activation"]
    assert list(inspect.signature(gridnet_cuda.backward).parameters) == [
        "weight", "bias", "scale", "initActivations", "outGrads", "weightGradOut", "biasGradOut",
        "scaleGradOut", "activationsGradOut", "innerIterations", "blockSize", "eps", "normalize",
        "activation"]
    assert len(inspect.signature(gridnet_cuda.forward_gated).parameters) == 7
    assert len(inspect.signature(gridnet_cuda.backward_gated).parameters) == 10


def test_shim_rejects_host_tensors_like_the_reference_binding():
    import torch

    import gridnet_cuda

    t = torch.zeros(1, 8, 8, 8)
    w = torch.zeros(27, 8, 8, 8)
    p = torch.zeros(8, 8, 8)
    with pytest.raises(RuntimeError, match="weight must be a CUDA tensor"):
        gridnet_cuda.forward(w, p, p, t, t.clone(), 1, 8, 1e-5, False, "silu")


def test_shim_validates_dtypes_and_shapes_on_the_host(monkeypatch):
    """Raw pointers carry no dtype or size: what the reference's typed accessors would refuse
    (src/gridnet_cuda.cpp:103-107) is refused here before any native call.  The device check is
    patched out so that host tensors reach the checks behind it."""
    import torch

    import gridnet_cuda
    from gridnet_amd import native

    monkeypatch.setattr(native, "check_input", lambda t, name: None)

    def forbid(*a, **k):
        raise AssertionError("a native entry point was reached")

    for name in ("gridnet_hip_forward", "gridnet_hip_backward", "gridnet_hip_forward_gated",
                 "gridnet_hip_backward_gated"):
        monkeypatch.setattr(native.lib, name, forbid)
    w, p, x = torch.zeros(27, 8, 8, 16), torch.zeros(8, 8, 16), torch.zeros(2, 8, 8, 16)
    ok = (w, p, p, x, x.clone())
    cases = {
        "bias has dtype": (w, p.double(), p, x, x.clone()),
        "initActivations has dtype": (w, p, p, x.double(), x.clone()),
        "outActivations has shape": (w, p, p, x, x[:1].clone()),
        "weight has shape": (w[:, :, :, :8].contiguous(), p, p, x, x.clone()),
        "scale has shape": (w, p, p[:4].contiguous(), x, x.clone()),
    }
    for message, args in cases.items():
        with pytest.raises(RuntimeError, match=message):
            gridnet_cuda.forward(*args, 1, 8, 1e-5, False, "silu")
    grads = (torch.zeros_like(w), torch.zeros_like(p), torch.zeros_like(p), torch.zeros_like(x))
    with pytest.raises(RuntimeError, match="weightGradOut has shape"):
        gridnet_cuda.backward(w, p, p, x, x.clone(), grads[0][:26].contiguous(), *grads[1:], 1, 8, 1e-5,
                              False, "silu")
    with pytest.raises(RuntimeError, match="activationsGradOut has dtype"):
        gridnet_cuda.backward(w, p, p, x, x.clone(), *grads[:3], grads[3].double(), 1, 8, 1e-5, False,
                              "silu")
    with pytest.raises(RuntimeError, match="outGrads has shape"):
        gridnet_cuda.backward(w, p, p, x, x[:1].clone(), *grads, 1, 8, 1e-5, False, "silu")
    wg, pg = torch.zeros(27, 2, 8, 8, 16), torch.zeros(2, 8, 8, 16)
    with pytest.raises(RuntimeError, match="weight has shape"):
        gridnet_cuda.forward_gated(w, pg, x, x.clone(), 1, 8, "tanh")
    with pytest.raises(RuntimeError, match="biasGradOut has shape"):
        gridnet_cuda.backward_gated(wg, pg, x, x.clone(), torch.zeros_like(wg), torch.zeros_like(p),
                                    torch.zeros_like(x), 1, 8, "tanh")
    with pytest.raises(RuntimeError, match=r"must be \[B, M, N, K\]"):
        gridnet_cuda.forward(w, p, p, x[0], x[0].clone(), 1, 8, 1e-5, False, "silu")
    # and a well-formed call passes every check
    gridnet_cuda._check_call(tuple(zip(ok, "abcde", [(27, 8, 8, 16), (8, 8, 16), (8, 8, 16), x.shape, x.shape])), x)


def test_dispatcher_never_falls_back():
    import torch

    import gridnet_amd

    w, p, t = torch.zeros(27, 8, 8, 8), torch.zeros(8, 8, 8), torch.zeros(1, 8, 8, 8)
    with pytest.raises(NotImplementedError, match="HIP devices only"):
        gridnet_amd.gridnet_step(w, p, p, t, 1, 8)


def test_autograd_op_keeps_the_reference_contract():
    import torch

    from gridnet_amd.backend_cuda import GridnetCudaOp

    params = list(inspect.signature(GridnetCudaOp.forward).parameters)
    assert params == ["ctx", "weight", "bias", "residual_scale", "init_activations", "inner_iters",
                      "block_size", "eps", "normalize", "activation"]
    w, p = torch.zeros(27, 8, 8, 8), torch.zeros(8, 8, 8)
    # gridnet/backend_cuda.py:20-22 and :51-52
    with pytest.raises(AssertionError, match="incompatible"):
        GridnetCudaOp.apply(w, p, p, torch.zeros(1, 8, 8, 8), 1, 3, 1e-5, False, "silu")
    with pytest.raises(AssertionError, match="invalid"):
        GridnetCudaOp.apply(w[:26], p, p, torch.zeros(1, 8, 8, 8), 1, 8, 1e-5, False, "silu")
    with pytest.raises(AssertionError, match="mismatching dtypes"):
        GridnetCudaOp.apply(w, p.double(), p, torch.zeros(1, 8, 8, 8), 1, 8, 1e-5, False, "silu")
    empty = torch.zeros(0, 8, 8, 8)
    out = GridnetCudaOp.apply(w, p, p, empty, 1, 8, 1e-5, False, "silu")
    assert out.shape == empty.shape and out.data_ptr() != empty.data_ptr() or out.numel() == 0


def test_shim_matches_the_call_sites_in_the_reference_tree():
    """Where the reference is on disk (this container, not the GPU box): every call of the
    extension module in gridnet/backend_cuda.py, read as text and parsed, must fit the shim's
    function of that name -- same number of positional arguments, no keywords."""
    import ast
    import os

    import gridnet_cuda

    path = "/root/reference/gridnet/backend_cuda.py"
    if not os.path.exists(path):
        pytest.skip("the reference tree is not on this machine")
    with open(path) as fh:
        tree = ast.parse(fh.read())
    calls = [n for n in ast.walk(tree)
             if isinstance(n, ast.Call) and isinstance(n.func, ast.Attribute)
             and isinstance(n.func.value, ast.Name) and n.func.value.id == "gridnet_cuda"]
    assert {c.func.attr for c in calls} == {"forward", "backward", "forward_gated", "backward_gated"}
    for call in calls:
        params = inspect.signature(getattr(gridnet_cuda, call.func.attr)).parameters
        assert not call.keywords, call.func.attr
        assert len(call.args) == len(params), (call.func.attr, len(call.args), len(params))
