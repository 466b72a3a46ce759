"""The streaming GEMM where K is whole k-tiles but not whole k-groups (the last k-group part zero
padding): every M it serves against the oracle, a forced variant of each kind against the plan, and
the one-launch linear against quantizer + GEMM. Tolerance: tests/_check.py."""
import pytest
import torch

from tests._check import assert_gemm_close, bf16_dev, host_u16, host_u8, to_dev
from vllm_sly_radiance_amd import _native, synthetic
from vllm_sly_radiance_amd import radiance_mxfp4 as R

pytestmark = pytest.mark.gpu


# 4352 = 8.5, 3968 = 7.75, 9472 = 18.5 and 4224 = 8.25 k-groups; N = 300 pads its last n-tile
@pytest.mark.parametrize("M,N,K", [(1, 5120, 4352), (2, 5120, 4352), (4, 300, 4224), (8, 5120, 3968),
                                   (9, 2048, 4352), (13, 5120, 4352), (16, 3584, 9472)])
def test_stream_ktail(gpu_lib, M, N, K):
    assert _native.plan(M, N, K)[0] == _native.KERNEL_STREAM
    w, ws = synthetic.weights(N, K, seed=N)
    x = synthetic.activations(M, K, seed=M)
    x[M - 1, K - 1] = 0x7FC0                      # a NaN in the last token's last column
    wq, sq = R.repack_weights(to_dev(w), to_dev(ws))
    q, s = R.quant_per_token(bf16_dev(x))
    out = R.gemm(q, s, wq, sq, N, K)
    assert torch.isnan(out[M - 1]).all() and not torch.isnan(out[:M - 1]).any()
    ref = R.layout_ref(N, K, "cuda")
    one = torch.ops.radiance.mxfp4_linear(bf16_dev(x), wq, sq, ref)
    assert torch.equal(one[:M - 1], out[:M - 1]) and torch.isnan(one[M - 1]).all()
    x[M - 1, K - 1] = 0x3F80
    q, s = R.quant_per_token(bf16_dev(x))
    out = R.gemm(q, s, wq, sq, N, K)
    assert_gemm_close(host_u16(out), host_u8(q), s.cpu().numpy(), w, ws, f"M={M} N={N} K={K}")
    assert torch.equal(torch.ops.radiance.mxfp4_linear(bf16_dev(x), wq, sq, ref), out)
    skinny = R.gemm(q, s, wq, sq, N, K, kernel=_native.KERNEL_SKINNY, variant=0, split_k=1)
    rel = (skinny.float() - out.float()).norm() / out.float().norm()
    assert rel <= 1e-3, float(rel)               # two roundings of one sum (rel-L2 of each <= 1e-3)


def test_stream_serves_at_most_an_eighth_of_padding(gpu_lib):
    for K, serves in [(640, False), (1152, False), (4224, True), (4240 - 16, True), (4256, False)]:
        any_v = any(_native.variant_serves(_native.KERNEL_STREAM, v, 8, 2048, K)
                    for v in range(len(_native.variants(_native.KERNEL_STREAM))))
        assert any_v == serves, K
