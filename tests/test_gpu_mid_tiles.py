"""The automatic path above 64 tokens: every tile gives the plan's bits (a tile's shape does not
change an output's accumulation order), at ragged M and N, with tile counts that do and do not
divide by the 8 XCDs; and two tiles side by side in two launches."""
import numpy as np
import pytest
import torch

from oracle import mxfp4_oracle as O
from tests._check import assert_gemm_close, bf16_dev, host_u16, host_u8, stream, to_dev
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


# ragged M, N off the store widths, a last k-group part padding (K = 2688); the rest on 128 x 160,
# 64 x 160, 96 x 128 (4 waves), 64 x 64 and 128 x 128 tiles
@pytest.mark.parametrize("M,N,K,tail", [(1300, 13824, 1024, (128, 160)), (513, 13824, 2560, (64, 160)),
                                        (520, 13827, 2688, (64, 160)), (513, 14336, 2560, (96, 128)),
                                        (900, 17408, 2048, (64, 64)), (1111, 16388, 1024, (128, 128))])
def test_two_launches_give_the_bits_of_one(gpu_lib, M, N, K, tail):
    """Row-major and fragment-tiled activations against one launch of the first tile over all N, and
    sampled tokens against the oracle."""
    kernel, v, split = _native.plan(M, N, K)
    n_main, tv = _native.plan_columns(M, N, K)
    assert (kernel, split) == (_native.KERNEL_TILE, 1) and 0 < n_main < N
    assert _native.variants(_native.KERNEL_TILE)[tv][2:] == tail
    w, ws = synthetic.weights(N, K, seed=N)
    wq, sq = R.repack_weights(to_dev(w), to_dev(ws))
    q, s = R.quant_per_token(bf16_dev(synthetic.activations(M, K, seed=M)))
    one = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
    R.gemm(q, s, wq, sq, N, K, out=one, kernel=_native.KERNEL_TILE, variant=v, split_k=1)
    two = torch.full_like(one, float("nan"))
    R.gemm(q, s, wq, sq, N, K, out=two)
    assert torch.equal(two, one)
    codes = host_u8(q)
    tiled = to_dev(O.tile_q(codes))
    two.fill_(float("nan"))
    _native.gemm_at(tiled.data_ptr(), s.data_ptr(), wq.data_ptr(), sq.data_ptr(), two.data_ptr(), M, N,
                    K, stream())
    assert torch.equal(two, one)
    rows = np.unique(np.r_[0, M // 2, M - 1])
    assert_gemm_close(host_u16(two)[rows], codes[rows], s.cpu().numpy()[rows], w, ws,
                      f"two launches M={M} N={N} K={K}")
