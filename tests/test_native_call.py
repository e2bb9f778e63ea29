"""The native call of one linear (csrc/host_linear.cpp) against the general
route of qwen_int4_hip.backends over the forms it accepts, and the forms it
leaves to that route."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import oracle as O
from qwen_int4_hip import PackingFormat, _lib, hip_w4g64_linear, kernels
from qwen_int4_hip.kernels import linear_canonical_w4g64_hip

pytestmark = pytest.mark.skipif(not _lib.library_built(), reason="HIP library not built (run __graft_entry__.build())")
gpu = [pytest.mark.gpu, pytest.mark.skipif(not torch.cuda.is_available(), reason="needs a ROCm GPU")]
N, K = 96, 256


def _native(x, weights, bias=None, n=N, k=K):
    return _lib.host_linear()(x, *weights, bias, n, k, kernels._workspaces, kernels.grow_current_workspace)


def _weights(device, n=N, k=K):
    q, s, z = O.asymmetric_weights(n, k, n + k)
    return tuple(torch.from_numpy(np.ascontiguousarray(t)).to(device) for t in (q, s, z))


def test_host_tensors_are_left_to_the_general_route():
    x, weights = torch.zeros(2, K, dtype=torch.float16), _weights("cpu")
    assert _native(x, weights) is None
    assert _native(None, weights) is None and _native(x, (weights[0], 3, weights[2])) is None
    with pytest.raises(TypeError, match="9 arguments"):
        _lib.host_linear()(x)


@pytest.mark.parametrize("marks", [pytest.param(None, marks=gpu)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [(K,), (1, K), (3, K), (2, 5, K), (2, 1, 40, K), (300, K)])
def test_native_call_equals_the_general_route(marks, shape, dtype):
    weights = _weights("cuda")
    gen = torch.Generator(device="cuda").manual_seed(len(shape))
    x = torch.randn(shape, generator=gen, device="cuda").to(dtype)
    for bias_dtype in (None, torch.float16, torch.bfloat16, torch.float32):
        bias = None if bias_dtype is None else torch.randn(N, generator=gen, device="cuda").to(bias_dtype)
        got = _native(x, weights, bias)
        want = linear_canonical_w4g64_hip(x.reshape(-1, K), *weights, bias)
        assert got.shape == (*shape[:-1], N) and got.dtype == dtype and not got.requires_grad
        assert torch.equal(got.reshape(-1, N), want)
    parameter = torch.nn.Parameter(bias, requires_grad=False)
    assert torch.equal(_native(x.clone().requires_grad_(), weights, parameter), got)
    with torch.inference_mode():
        assert _native(x, weights).is_inference()
    side = torch.cuda.Stream()  # the current stream's workspace and queue
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        other = _native(x, weights, bias)
    side.synchronize()
    assert torch.equal(other, got)


@pytest.mark.parametrize("marks", [pytest.param(None, marks=gpu)])
def test_native_call_leaves_other_forms_to_the_general_route(marks):
    weights = _weights("cuda")
    q, s, z = weights
    x = torch.randn(4, K, device="cuda", dtype=torch.float16)

    class Sub(torch.Tensor):
        pass

    wide = torch.randn(4, 2 * K, device="cuda", dtype=torch.float16)
    flat = torch.randn(4 * K + 1, device="cuda", dtype=torch.float16)
    odd_q = torch.empty(q.numel() + 1, dtype=torch.uint8, device="cuda")[1:].view_as(q).copy_(q)
    accepted = {  # forms that the general route computes
        "strided rows": (wide[:, :K], weights), "transposed": (torch.randn(K, 4, device="cuda").half().t(), weights),
        "misaligned rows": (flat[1:].view(4, K), weights), "misaligned weight": (x, (odd_q, s, z)),
        "no rows": (x[:0], weights), "subclass": (x.as_subclass(Sub), weights),
    }
    for name, (rows, ws) in accepted.items():
        assert _native(rows, ws) is None, name
        got = hip_w4g64_linear(rows, *ws, None, out_features=N, in_features=K, group_size=64,
                               packing=PackingFormat.CANONICAL)
        if rows.numel():
            plain = rows.as_subclass(torch.Tensor).contiguous().clone()
            assert torch.equal(got.as_subclass(torch.Tensor), linear_canonical_w4g64_hip(plain, q, s, z, None)), name
        assert got.shape == (rows.shape[0], N), name
    refused = {
        "int rows": (x.to(torch.int32), weights, None, N, K), "double rows": (x.double(), weights, None, N, K),
        "other K": (x[:, :128].contiguous(), weights, None, N, K), "scalar": (x[0, 0], weights, None, N, K),
        "short weight": (x, (q[:-1], s, z), None, N, K), "signed weight": (x, (q.view(torch.int8), s, z), None, N, K),
        "flat scales": (x, (q, s.view(-1), z), None, N, K), "bf16 scales": (x, (q, s.bfloat16(), z), None, N, K),
        "short zeros": (x, (q, s, z[:-1]), None, N, K), "host scales": (x, (q, s.cpu(), z), None, N, K),
        "long bias": (x, weights, torch.zeros(N + 1, device="cuda"), N, K),
        "int bias": (x, weights, torch.zeros(N, device="cuda", dtype=torch.int32), N, K),
        "K % 64": (x[:, :96].contiguous(), weights, None, N, 96), "no outputs": (x, weights, None, 0, K),
    }
    for name, (rows, ws, bias, n, k) in refused.items():
        assert _native(rows, ws, bias, n, k) is None, name
        with pytest.raises((TypeError, ValueError)):
            hip_w4g64_linear(rows, *ws, bias, out_features=n, in_features=k, group_size=64,
                             packing=PackingFormat.CANONICAL)
    assert _native(x, weights, None, True, K) is None
    # modes, tracing and functorch levels keep the interpreter's route
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    for mode in (Function(), Dispatch()):
        with mode:
            assert _native(x, weights) is None
    seen = []
    torch.func.vmap(lambda t: (seen.append(_native(x, weights)), seen.append(_native(t, weights)), t)[2])(x)
    torch.jit.trace(lambda t: (seen.append(_native(t, weights)), t + 0)[1], (x,), check_trace=False)
    assert len(seen) >= 3 and all(y is None for y in seen)


def test_what_follows_torch_operators_is_seen():
    """The states in which the attention layer keeps to torch's operators."""
    from torch.autograd import forward_ad
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    assert not kernels._operators_followed()
    with torch.device("cpu"):  # (a default device is no such state)
        assert not kernels._operators_followed()
    for mode in (TorchFunctionMode(), TorchDispatchMode(), forward_ad.dual_level()):
        with torch.device("cpu"), mode:
            assert kernels._operators_followed(), type(mode)
    seen = []
    torch.func.vmap(lambda t: (seen.append(kernels._operators_followed()), t)[1])(torch.zeros(2))
    torch.jit.trace(lambda t: (seen.append(kernels._operators_followed()), t + 0)[1], (torch.zeros(2),), check_trace=False)
    compiled = torch.compile(lambda t: t + int(kernels._operators_followed()), backend="eager")(torch.zeros(2))
    assert len(seen) >= 2 and all(seen) and compiled.tolist() == [1, 1]
    assert not kernels._operators_followed()


@pytest.fixture
def no_host_module(monkeypatch):
    import sys

    import qwen_int4_hip

    monkeypatch.setattr(_lib, "_host_linear", None)
    monkeypatch.delattr(qwen_int4_hip, "_host", raising=False)
    monkeypatch.setitem(sys.modules, "qwen_int4_hip._host", None)  # its import fails


def test_host_module_that_does_not_load_leaves_all_calls(no_host_module):
    with pytest.warns(RuntimeWarning, match="general route"):
        assert _native(torch.zeros(2, K, dtype=torch.float16), _weights("cpu")) is None


@pytest.mark.parametrize("marks", [pytest.param(None, marks=gpu)])
def test_linears_run_without_the_host_module(marks, no_host_module):
    weights = _weights("cuda")
    x = torch.randn(4, K, device="cuda", dtype=torch.float16)
    with pytest.warns(RuntimeWarning, match="general route"):
        got = hip_w4g64_linear(x, *weights, None, out_features=N, in_features=K, group_size=64,
                               packing=PackingFormat.CANONICAL)
    assert torch.equal(got, linear_canonical_w4g64_hip(x, *weights, None))
