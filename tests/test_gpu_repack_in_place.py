"""The one-workgroup-per-n-tile repack (N % 16 == 0, K % 512 == 0) against the oracle, out of place
and rewriting its own input, at the edges of its tiles: K one k-group up to the widest each load
count per thread holds and one k-group more, and past the widest it serves (the general
repack). Bytes are bit-exact."""
import numpy as np
import pytest
import torch

from oracle import mxfp4_oracle as O
from tests._check import host_u8, stream, to_dev
from vllm_sly_radiance_amd import _native, synthetic
from vllm_sly_radiance_amd import radiance_mxfp4 as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(16, 512), (48, 2048), (16, 2560), (32, 4096), (16, 4608),
                                 (16, 6656), (16, 10752), (16, 16896), (16, 19968), (16, 20480)])
def test_repack_in_place_bit_exact(gpu_lib, N, K):
    w, ws = synthetic.weights(N, K, seed=N + K)
    owq, osq = O.repack(w, ws)
    wd, sd = to_dev(w), to_dev(ws)
    wq, sq = R.repack_weights(wd, sd)
    assert wq.data_ptr() != wd.data_ptr() and torch.equal(wd, to_dev(w))
    assert np.array_equal(host_u8(wq).reshape(-1), owq)
    assert np.array_equal(host_u8(sq).reshape(-1), osq)
    wq, sq = R.repack_weights(wd, sd, in_place=True)
    assert (wq.data_ptr() == wd.data_ptr()) == (K <= R.REPACK_IN_PLACE_MAX_K)
    assert np.array_equal(host_u8(wq).reshape(-1), owq)
    assert np.array_equal(host_u8(sq).reshape(-1), osq)


def test_repack_refuses_in_place_where_it_pads(gpu_lib):
    """A padded shape has no room in its own storage; scales off a 16-byte boundary take the
    general repack, which reads while others write."""
    w, ws = synthetic.weights(32, 640, seed=1)
    wd, sd = to_dev(w), to_dev(ws)
    with pytest.raises(RuntimeError, match="in place"):
        _native.repack(wd.data_ptr(), sd.data_ptr(), wd.data_ptr(), sd.data_ptr(), 32, 640, stream())
    w, ws = synthetic.weights(16, 512, seed=2)
    buf = torch.zeros(4 + ws.size, dtype=torch.uint8, device="cuda")
    buf[4:] = to_dev(ws).reshape(-1)
    wq, sq = R.repack_weights(to_dev(w), buf[4:].view(16, 16), in_place=True)
    owq, osq = O.repack(w, ws)
    assert np.array_equal(host_u8(wq).reshape(-1), owq)
    assert np.array_equal(host_u8(sq).reshape(-1), osq)
