"""The direct registration of each custom op (radiance::<name>_inference): the public op's schema and
body, taken only where no gradient can be asked for and nothing is compiled."""
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
    graph = make_fx(call, tracing_mode="fake")(torch.ones(2))
    assert any("probe_fake_inference" in str(n.target) for n in graph.graph.nodes)
    with torch.inference_mode():
        assert torch.equal(call(torch.ones(2)), torch.full((2,), 2.0))
