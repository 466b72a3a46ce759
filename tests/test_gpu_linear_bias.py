"""The linear with its bias in the GEMM epilogue against the linear followed by the elementwise add, bit
for bit, on each kernel of the automatic plan: the one-launch linear, the streaming GEMM (two
widths, K of whole and part k-groups), skinny with and without its K split, band, tiles with staged
and direct stores, the K-split tiles with their reduction, and the two-launch prefill; N off the
vector width, and biases the epilogue does not take."""
import pytest
import torch

from tests._check import bf16_dev, to_dev
from vllm_sly_radiance_amd import _native, synthetic
from vllm_sly_radiance_amd import radiance_mxfp4 as R

pytestmark = pytest.mark.gpu


class Layer(torch.nn.Module):
    def __init__(self, w, ws):
        super().__init__()
        self.weight = torch.nn.Parameter(to_dev(w), requires_grad=False)
        self.weight_scale = torch.nn.Parameter(to_dev(ws), requires_grad=False)


def loaded(N, K):
    layer = Layer(*synthetic.weights(N, K, seed=N + K))
    R.kernel_class()().process_weights_after_loading(layer)
    return layer


@pytest.mark.parametrize("M,N,K", [(1, 2064, 1024), (1, 5120, 4352), (4, 10240, 512), (8, 301, 1024),
                                   (13, 5120, 4352), (16, 1000, 640), (5, 40, 8320),
                                   (24, 5120, 8704), (40, 10240, 5120), (33, 1003, 640),
                                   (64, 2050, 512), (200, 5122, 512), (300, 2048, 640),
                                   (1111, 1288, 512), (4096, 4608, 256)])
def test_bias_epilogue_equals_the_add(gpu_lib, M, N, K):
    layer, kern = loaded(N, K), R.kernel_class()()
    x = bf16_dev(synthetic.activations(M, K, seed=M))
    bias = 0.1 * torch.randn(N, device="cuda").bfloat16()
    assert R._fuses_bias(bias, N, x)
    y = kern.apply(layer, x)
    before = R.STATS["calls"]
    assert torch.equal(kern.apply(layer, x, bias), y + bias), _native.plan(M, N, K)
    assert R.STATS["calls"] == before + 1
    x3 = x.reshape(1, M, K)
    assert torch.equal(kern.apply(layer, x3, bias), (y + bias).reshape(1, M, N))


def test_biases_the_epilogue_does_not_take(gpu_lib):
    M, N, K = 3, 512, 512
    layer, kern = loaded(N, K), R.kernel_class()()
    x = bf16_dev(synthetic.activations(M, K, seed=1))
    y = kern.apply(layer, x)
    wide = torch.randn(2 * N + 1, device="cuda")
    for bias in (wide[:N], wide.bfloat16()[1:N + 1], wide.bfloat16()[:2 * N:2], wide.bfloat16()[:1],
                 wide.bfloat16()[:N].reshape(1, N), wide.bfloat16()[:N].expand(M, N)):
        out = kern.apply(layer, x, bias)
        assert out.dtype == (y + bias).dtype and torch.equal(out, y + bias)
    grad = torch.zeros(N, device="cuda", dtype=torch.bfloat16, requires_grad=True)
    kern.apply(layer, x, grad).sum().backward()
    assert torch.equal(grad.grad, torch.full_like(grad, M))
    inf = torch.full((N,), float("inf"), device="cuda", dtype=torch.bfloat16)
    assert torch.isinf(kern.apply(layer, x, inf)).all()
    assert kern.apply(layer, x[:0], inf).shape == (0, N)
