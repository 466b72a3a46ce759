"""The automatic path for 64 < M <= 1024: every tile gives the plan's bits (a tile's shape does not
change an output's accumulation order), at ragged M and N, with tile counts that do and do not
divide by the 8 XCDs."""
import pytest
import torch

from tests._check import bf16_dev, to_dev
from vllm_sly_radiance_amd import _native, synthetic
from vllm_sly_radiance_amd import radiance_mxfp4 as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(65, 2064, 640), (96, 1544, 512), (200, 4112, 1152),
                                   (333, 5120, 512), (512, 10240, 384), (1024, 1000, 256)])
def test_every_tile_gives_the_same_bits(gpu_lib, M, N, K):
    w, ws = synthetic.weights(N, K, seed=N)
    wq, sq = R.repack_weights(to_dev(w), to_dev(ws))
    q, s = R.quant_per_token(bf16_dev(synthetic.activations(M, K, seed=M)))
    auto = R.gemm(q, s, wq, sq, N, K)
    k, v, sp = _native.plan(M, N, K)
    assert k == _native.KERNEL_TILE and sp == 1
    for v in range(len(_native.variants(_native.KERNEL_TILE))):
        out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        R.gemm(q, s, wq, sq, N, K, out=out, kernel=_native.KERNEL_TILE, variant=v, split_k=1)
        assert torch.equal(out, auto), v
