"""The table form of SiLU-mul + quant (more than 128 rows) against the same rows in calls of at most 128,
which compute every silu: the same codes and scales, bit for bit, for every bf16 gate (zeros,
subnormals, infinities and NaNs among them) and at the edges of its rows: one to four groups per
thread, ragged last groups, fewer and more rows than workgroups, row-major and fragment-tiled."""
import pytest
import torch

from vllm_sly_radiance_amd import _native
from vllm_sly_radiance_amd import radiance_fused_norm as F
from vllm_sly_radiance_amd import radiance_mxfp4 as R

pytestmark = pytest.mark.gpu


def by_parts(x):
    parts = [F.silu_mul_quant_op(x[a:a + 128]) for a in range(0, x.shape[0], 128)]
    return torch.cat([p[0].view(torch.uint8) for p in parts]), torch.cat([p[1] for p in parts])


def same(x):
    q, s = F.silu_mul_quant_op(x)
    q0, s0 = by_parts(x)
    assert torch.equal(s.view(torch.int32), s0.view(torch.int32))
    assert torch.equal(q.view(torch.uint8), q0)


@pytest.mark.parametrize("M,N", [(129, 8200), (130, 8704), (257, 10240), (1024, 5128), (1111, 8192),
                                 (131, 10248), (300, 14336), (515, 17408), (140, 18432),
                                 (2048, 4104), (2049, 5120)])
@pytest.mark.parametrize("std", [1.0, 25.0])
def test_same_bits_as_the_computed_form(gpu_lib, M, N, std):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = (std * torch.randn(M, 2 * N, device="cuda", generator=g)).bfloat16()
    x[1, :N] = 0
    x[2] = 0
    same(x)


def test_every_gate(gpu_lib):
    """Every bf16 pattern as a gate: the finite ones in order of magnitude, 64 to a row beside ordinary
    ones (a row's scale then follows its own gates), and rows that hold infinities and NaNs."""
    N = 8704
    bits = torch.arange(1 << 16, device="cuda")
    order = bits[torch.argsort(bits & 0x7FFF)].to(torch.int16).view(torch.bfloat16)
    x = torch.randn(1024, 2 * N, device="cuda").bfloat16()
    x[:, 3:N:136] = order.reshape(1024, 64)
    same(x)
    same(order.reshape(-1).repeat(1 + 256 * 2 * N // order.numel())[:256 * 2 * N].reshape(256, 2 * N))


def test_fragment_tiled(gpu_lib):
    M, N = 200, 8704
    x = (3 * torch.randn(M, 2 * N, device="cuda")).bfloat16()
    q = R.alloc_tiled_q(M, N, "cuda")
    s = torch.empty(M, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    _native.silu_mul_quant(x.data_ptr(), q.data_ptr(), s.data_ptr(), M, N, st, _native.Q_TILED)
    q0, s0 = by_parts(x)
    t = torch.as_strided(q.view(torch.uint8), (-(-M // 16), N // 128, 2, 4, 16, 16),
                         (16 * N, 2048, 1024, 256, 16, 1))
    rows = t.permute(0, 4, 1, 2, 3, 5).reshape(-1, N)[:M]
    assert torch.equal(rows, q0) and torch.equal(s, s0)
