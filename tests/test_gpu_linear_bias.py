"""The linear with its bias in the GEMM epilogue against the linear followed by the elementwise add, bit
for bit, on each kernel of the automatic plan: the one-launch linear, the streaming GEMM (two
widths, K of whole and part k-groups), skinny with and without its K split, band, tiles with staged
and direct stores, the K-split tiles with their reduction, and two tiles side by side in two
launches; N off the vector width, NaN, infinite and overflowing sums, and biases the epilogue does
not take. test_bias_epilogue_on_its_route holds each shape to the kernel it is there for."""
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


def route(M, N, K):
    """The epilogue that a biased linear of this shape runs through."""
    kernel, _, split = _native.plan(M, N, K)
    if kernel == _native.KERNEL_STREAM:
        return "one launch" if _native.linear_fused(M, N, K, K) else "stream"
    if kernel in (_native.KERNEL_SKINNY, _native.KERNEL_TILE) and split > 1:
        return ("skinny" if kernel == _native.KERNEL_SKINNY else "tile") + ", K split"
    if kernel == _native.KERNEL_TILE:
        two = ", two launches" if _native.plan_columns(M, N, K)[1] >= 0 else ""
        return ("tile, staged" if N % 8 == 0 else "tile, direct") + two
    return {_native.KERNEL_SKINNY: "skinny", _native.KERNEL_BAND: "band"}[kernel]


ROUTES = [(1, 5120, 4352, "one launch"), (2, 10240, 1024, "one launch"), (8, 301, 1024, "stream"),
          (13, 5120, 4352, "stream"), (16, 2070, 640, "skinny"), (16, 1000, 640, "skinny, K split"),
          (5, 40, 8288, "skinny, K split"), (16, 301, 8288, "skinny, K split"),
          (40, 10240, 5120, "band"), (33, 8195, 640, "band"),
          (24, 5120, 8704, "tile, K split"), (200, 1024, 640, "tile, staged"),
          (200, 1004, 640, "tile, direct"), (77, 1003, 640, "tile, direct"),
          (1111, 16384, 1024, "tile, staged, two launches"),
          (513, 13824, 2560, "tile, staged, two launches"),
          (520, 13852, 2560, "tile, direct, two launches"),
          (1300, 13827, 1024, "tile, direct, two launches")]


@pytest.mark.parametrize("M,N,K,path", ROUTES)
def test_bias_epilogue_on_its_route(gpu_lib, M, N, K, path):
    """Token 0 holds a NaN, token 1 zeros, the last token's activations are near bf16's largest so that
    outputs overflow, and the bias holds NaNs of either sign, infinities and zeros of both signs,
    the largest bf16 and a subnormal, at the first columns, the last and those of a second launch.
    Bits of the add, whose NaNs have no sign."""
    layer, kern = loaded(N, K), R.kernel_class()()
    assert route(M, N, K) == path
    x = bf16_dev(synthetic.activations(M, K, seed=M))
    x[M - 1] = torch.where(x[M - 1] < 0, -3.0e38, 3.0e38).bfloat16()
    if M > 1:
        x[0, K - 1] = float("nan")
    if M > 2:
        x[1] = 0
    bias = 0.1 * torch.randn(N, device="cuda").bfloat16()
    special = torch.tensor([0x7FC0, -0x40, 0x7F81, 0x7F80, -0x80, 0, -0x8000, 0x7F7F, -0x81, 1],
                           dtype=torch.int16, device="cuda").view(torch.bfloat16)
    for at in {0, 7, N - 10, _native.plan_columns(M, N, K)[0] % N}:
        bias[at:at + 10] = special
    assert R._fuses_bias(bias, N, x)
    y = kern.apply(layer, x)
    out, want = kern.apply(layer, x, bias), y + bias
    assert torch.isinf(y[M - 1]).any() and not torch.isnan(y[M - 1]).any()
    nan = torch.isnan(want)
    assert M == 1 or nan[0].all()
    assert torch.equal(out.view(torch.int16), want.view(torch.int16))
    assert (out.view(torch.int16)[nan] == 0x7FC0).all()


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
