"""The direct registration of each custom op (radiance::<name>_inference): the public op's schema and
body, taken only where no gradient can be asked for and nothing compiles, traces or watches ops by
name."""
import os
import subprocess
import sys

import pytest
import torch

from vllm_sly_radiance_amd import radiance_fused_norm as F
from vllm_sly_radiance_amd import radiance_mxfp4 as R

OPS = [R.mxfp4_linear, R.mxfp4_linear_pq, R.silu_mul_mxfp4_linear, F.add_rms_quant_op,
       F.silu_mul_quant_op, F.gdn_norm_quant_op]


@pytest.mark.parametrize("op", OPS, ids=lambda o: o._qualname)
def test_same_schema_and_fake(op):
    name = op._qualname.split("::")[1]
    public = getattr(torch.ops.radiance, name).default._schema
    direct = getattr(torch.ops.radiance, name + "_inference").default._schema
    assert str(direct) == str(public).replace(name + "(", name + "_inference(", 1)


def _probe(name):
    calls = []

    def body(x: torch.Tensor) -> torch.Tensor:
        calls.append(torch.is_grad_enabled())
        return x * 2

    op = torch.library.custom_op(f"radiance::{name}", body, mutates_args=())
    op.register_fake(lambda x: torch.empty_like(x))
    return R.inference_op(op, body, lambda x: torch.empty_like(x)), calls


def test_gradients_take_the_public_op():
    call, calls = _probe("probe_grad")
    x = torch.ones(3, requires_grad=True)
    y = call(x)
    assert y.requires_grad and len(calls) == 1
    with pytest.raises(RuntimeError):                # the public op has no backward formula
        y.sum().backward()
    with torch.no_grad():
        assert not call(x).requires_grad
    assert torch.equal(call(torch.ones(3)), torch.full((3,), 2.0))


def test_fake_tensors_and_tracing_see_the_op():
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    call, calls = _probe("probe_fake")
    with FakeTensorMode():
        assert call(torch.empty(4, 5)).shape == (4, 5)
    assert not calls
    for how in (dict(tracing_mode="real"), dict(tracing_mode="fake"), dict(pre_dispatch=True)):
        graph = make_fx(call, **how)(torch.ones(2))
        assert [str(n.target) for n in graph.graph.nodes][1:-1] == ["radiance.probe_fake.default"], how
    assert "radiance::probe_fake(" in str(torch.jit.trace(call, torch.ones(2), check_trace=False).graph)
    with torch.inference_mode():
        assert torch.equal(call(torch.ones(2)), torch.full((2,), 2.0))


def test_modes_and_subclasses_see_the_public_op():
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode
    call, _ = _probe("probe_modes")
    seen = []

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return super().__torch_function__(func, types, args, kwargs or {})

    x = torch.ones(2)
    for mode in (Dispatch, Function):
        with mode():
            call(x)
    call(x.as_subclass(Sub))
    assert [s.removesuffix(".default") for s in seen if "probe" in s] == ["radiance.probe_modes"] * 3
    with torch.device("cpu"):                    # a default device is a function mode, and not one
        assert not R._watched()                  # that looks at ops
    assert not R._watched()


def test_a_bias_that_something_differentiates_or_maps_is_added_outside(monkeypatch):
    """Forward-mode tangents of the bias, vmap over it and traced graphs need its add as an op of its
    own; a plain call takes the epilogue."""
    from types import SimpleNamespace

    import torch.autograd.forward_ad as fw
    from torch.fx.experimental.proxy_tensor import make_fx
    x, y = torch.ones(2, 32, dtype=torch.bfloat16), torch.full((2, 4), 3.0, dtype=torch.bfloat16)
    layer = SimpleNamespace(weight=None, weight_scale=None, radiance_wref=torch.empty(4, 32, 0))
    fused = []
    monkeypatch.setattr(R, "call_linear", lambda *args: y.clone())
    monkeypatch.setattr(R, "call_linear_bias", lambda *args: fused.append(1) or y + args[-1])
    bias = torch.arange(4.0).bfloat16()

    def apply(b):
        return R.kernel_class()().apply(layer, x, b)

    assert torch.equal(apply(bias), y + bias) and len(fused) == 1
    with fw.dual_level():
        out = fw.unpack_dual(apply(fw.make_dual(bias, torch.full_like(bias, 2.0))))
    assert torch.equal(out.primal, y + bias) and (out.tangent == 2).all()
    out, tangent = torch.func.jvp(apply, (bias,), (torch.full_like(bias, 2.0),))
    assert torch.equal(out, y + bias) and (tangent == 2).all()
    biases = torch.stack([bias, bias + 1])
    assert torch.equal(torch.func.vmap(apply)(biases), y + biases[:, None])
    names = [str(n.target) for n in make_fx(apply)(bias).graph.nodes]
    assert "aten.add.Tensor" in names
    assert len(fused) == 1


def test_the_modules_can_be_loaded_again():
    """importlib.reload and a fresh import register every op again: the newest body runs, also for
    calls through the earlier module, and reloading one module leaves the other's ops alone."""
    code = """
import gc, importlib, sys, torch
def check(R, F):
    gc.collect()
    x = torch.empty(3, 64, dtype=torch.bfloat16, device="meta")
    w, ws, ref = (torch.empty(s, dtype=torch.uint8, device="meta") for s in ((32, 32), (32, 2), (32, 64, 0)))
    assert R.call_linear(x, w, ws, ref).shape == torch.ops.radiance.mxfp4_linear(x, w, ws, ref).shape == (3, 32)
    assert R.call_linear_bias(x, w, ws, ref, x[0, :32]).shape == (3, 32)
    q, s = F.call_silu_mul_quant(x)
    assert q.shape == (3, 32) and s.shape == (3,)
from vllm_sly_radiance_amd import radiance_mxfp4 as R, radiance_fused_norm as F
check(R, F)
for module in (R, R, F, R):
    importlib.reload(module)
    check(R, F)
old = R, F
for name in [n for n in sys.modules if n.startswith("vllm_sly_radiance_amd")]:
    del sys.modules[name]
import vllm_sly_radiance_amd.radiance_mxfp4 as R, vllm_sly_radiance_amd.radiance_fused_norm as F
assert R is not old[0]
check(R, F)
check(*old)
del old
check(R, F)

def probe(factor):
    def body(x: torch.Tensor) -> torch.Tensor:
        return x * factor
    op = torch.library.custom_op("radiance::probe_again", body, mutates_args=())
    return R.inference_op(op, body, torch.empty_like)
first, second = probe(2.0), probe(3.0)
with torch.no_grad():
    assert first(torch.ones(1)).item() == second(torch.ones(1)).item() == 3.0
def wider(x: torch.Tensor, factor: float) -> torch.Tensor:
    return x * factor
op = torch.library.custom_op("radiance::probe_again", wider, mutates_args=())
assert R.inference_op(op, wider, lambda x, factor: torch.empty_like(x))(torch.ones(1), 5.0).item() == 5.0
first, second = probe(2.0), probe(3.0)
grad = torch.ones(1, requires_grad=True)
assert first(grad).item() == second(grad).item() == 3.0
print("ok")
"""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    run = subprocess.run([sys.executable, "-c", code], cwd=root, capture_output=True, text=True,
                         timeout=120)
    assert run.returncode == 0 and run.stdout.strip() == "ok", run.stderr
