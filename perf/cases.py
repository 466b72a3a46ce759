"""Performance cases of the MXFP4 W4A8 linear path: the linear layers of a decoder, as a serving
program has them run.

A case is a block of a decoder layer at M tokens, over `layers` layers with weights of their own
(a decode pass streams every layer's weights from HBM; one layer alone would sit in the 256 MB
last-level cache):

  mlp     residual add + RMSNorm + quantizer, gate_up projection, SiLU-and-mul + down projection
  attn    residual add + RMSNorm + quantizer, qkv projection; gated per-head norm + quantizer on the
          attention output, o_proj
  linear  one projection on bf16 activations (quantizer inside), with or without a bias
  load    the load-time repack of one layer's four projections

`graph`: the pass is captured once into a HIP graph and replayed, as serving engines run decode and
small batches; otherwise the calls are made one by one. Sizes are those of the benchmark's
5120-hidden decoder, its tensor-parallel shares, and generic decoder shapes; M covers one token to a
4096-token prefill. Weights and activations have the distributions of the benchmark's synthetic
operands, made on the GPU.
"""
from __future__ import annotations

from types import SimpleNamespace

import torch

from vllm_sly_radiance_amd import radiance_fused_norm as F
from vllm_sly_radiance_amd import radiance_mxfp4 as R

EPS = 1e-6
# name -> (hidden, qkv outputs, attention output width, MLP intermediate width)
SHAPES = {
    "h5120": (5120, 10240, 6144, 8704),         # the benchmark's layer (bench.py)
    "h5120-half": (5120, 5120, 3072, 4352),     # one of two ranks' share of it; 4352 = 8.5 x 512
    "h5120-whole": (5120, 16384, 6144, 17408),  # the unsharded MLP
    "h4096": (4096, 6144, 4096, 14336),         # generic decoders
    "h3584": (3584, 4608, 3584, 9472),          # 9472 = 18.5 x 512
    "h2048": (2048, 3072, 2048, 6144),
}
COST_MAX = 4096 * (17408 * 5120 + 5120 * 8704)  # tokens x weights of the largest listed case


def _linears(case):
    """(N, K) of each projection that the block runs."""
    hidden, qkv, attn, inter = SHAPES[case["shape"]]
    mlp = [(2 * inter, hidden), (hidden, inter)]
    att = [(qkv, hidden), (hidden, attn)]
    if case["block"] == "linear":
        return [dict(qkv=att[0], o_proj=att[1], gate_up=mlp[0], down=mlp[1])[case["proj"]]]
    return {"mlp": mlp, "attn": att, "load": att + mlp}[case["block"]]


def listed():
    return [
        # one token through one projection, called from Python: the smallest call, latency and host
        dict(name="qkv_m1_eager", block="linear", proj="qkv", shape="h5120", M=1, layers=1,
             bias=False, graph=False),
        # single-stream decode
        dict(name="mlp_m1", block="mlp", shape="h5120", M=1, layers=6, graph=True),
        # speculative verify: a handful of drafted tokens
        dict(name="mlp_m8", block="mlp", shape="h5120", M=8, layers=6, graph=True),
        # a small odd batch on a tensor-parallel share whose K is not whole k-groups, with a bias
        dict(name="down_half_m13", block="linear", proj="down", shape="h5120-half", M=13, layers=24,
             bias=True, graph=True),
        # batched decode
        dict(name="attn_m24", block="attn", shape="h5120", M=24, layers=8, graph=True),
        dict(name="mlp_m40", block="mlp", shape="h4096", M=40, layers=6, graph=True),
        dict(name="mlp_m64", block="mlp", shape="h5120", M=64, layers=6, graph=True),
        # large decode batches and mixed steps (decode rows beside a prefill chunk)
        dict(name="mlp_m200", block="mlp", shape="h5120", M=200, layers=4, graph=True),
        dict(name="attn_m512", block="attn", shape="h5120", M=512, layers=4, graph=True),
        # prefill: a prompt of odd length, and a full chunk
        dict(name="mlp_m1111", block="mlp", shape="h5120", M=1111, layers=1, graph=False),
        dict(name="mlp_m4096", block="mlp", shape="h5120", M=4096, layers=1, graph=False),
        # model load: every layer's projections go through this once
        dict(name="load", block="load", shape="h5120", M=0, layers=1, graph=False),
    ]


def draw(rng):
    block = rng.choices(["mlp", "attn", "linear", "load"], [8, 5, 5, 1])[0]
    shape = rng.choice(sorted(SHAPES))
    case = dict(block=block, shape=shape, M=0, layers=1, graph=False)
    if block == "load":
        hidden, qkv, attn, inter = SHAPES[shape]
        case["layers"] = 1 if hidden * inter > 60 << 20 else rng.randint(1, 2)
        return case
    if block == "linear":
        case["proj"] = rng.choice(["qkv", "o_proj", "gate_up", "down"])
        case["bias"] = rng.random() < 0.3
    weights = sum(n * k for n, k in _linears(case))
    top = min(4096, COST_MAX // weights)
    M = int(round(2.0 ** rng.uniform(0.0, 12.0)))
    M = M + rng.randint(0, 1) if M > 4 else M       # odd ones among them
    case["M"] = max(1, min(M, top))
    case["graph"] = case["M"] <= 512 and rng.random() < 0.85
    # enough layers that a decode pass's weights outgrow the last-level cache
    if case["M"] <= 512:
        case["layers"] = max(1, min(24, (768 << 20) // weights))
    return case


class _Layer(torch.nn.Module):
    """A linear as a checkpoint loader leaves it: e2m1 bytes [N, K/2] and e8m0 bytes [N, K/32]."""

    def __init__(self, weight, weight_scale):
        super().__init__()
        self.weight = torch.nn.Parameter(weight, requires_grad=False)
        self.weight_scale = torch.nn.Parameter(weight_scale, requires_grad=False)


class _Inputs:
    """The seeded inputs of a case, drawn on the GPU in a fixed order."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def weight(self, N, K):
        return (torch.randint(0, 256, (N, K // 2), dtype=torch.uint8, device="cuda",
                              generator=self.g),
                torch.randint(119, 126, (N, K // 32), dtype=torch.uint8, device="cuda",
                              generator=self.g))

    def activation(self, M, K):
        """N(0, 1) with one outlier of 20x in a thousand."""
        x = torch.randn((M, K), device="cuda", generator=self.g)
        far = torch.rand((M, K), device="cuda", generator=self.g) < 1e-3
        return torch.where(far, 20 * x, x).bfloat16()

    def near(self, mean, n):
        return (mean + 0.1 * torch.randn(n, device="cuda", generator=self.g)).bfloat16()


def _make(case, seed):
    """Per layer: the checkpoint weights and the tensors that the block reads."""
    hidden, _, attn, _ = SHAPES[case["shape"]]
    M, src = case["M"], _Inputs(seed)
    for _ in range(case["layers"]):
        d = SimpleNamespace(ckpt=[src.weight(n, k) for n, k in _linears(case)])
        if case["block"] == "linear":
            n, k = _linears(case)[0]
            d.x = src.activation(M, k)
            d.bias = src.near(0.0, n) if case["bias"] else None
        elif case["block"] != "load":
            d.h, d.res = src.activation(M, hidden), src.activation(M, hidden)
            d.norm_w = src.near(0.0, hidden)        # the Gemma convention: the kernel adds the 1
        if case["block"] == "attn":
            d.core = src.activation(M, attn)
            # the gate is a column slice of the wider input projection
            d.z = src.activation(M, 2 * attn)[:, attn:]
            d.gate_w = src.near(1.0, 128)
        yield d


def prepare(case, seed):
    kernel = R.kernel_class()()
    state = SimpleNamespace(kernel=kernel, block=case["block"], layers=[], graph=None)
    for d in _make(case, seed):
        if case["block"] != "load":
            d.lin = [_Layer(*c) for c in d.ckpt]
            for layer in d.lin:
                kernel.process_weights_after_loading(layer)
            del d.ckpt
        if case["block"] in ("mlp", "attn"):
            d.norm = SimpleNamespace(weight=d.norm_w, variance_epsilon=EPS)
        if case["block"] == "attn":
            d.attn = SimpleNamespace(norm=SimpleNamespace(weight=d.gate_w, eps=EPS))
        state.layers.append(d)
    if case["graph"]:
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _pass(state)
        torch.cuda.current_stream().wait_stream(side)
        state.graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state.graph):
            state.out = _pass(state)
    return state


def _pass(state):
    kernel, out = state.kernel, []
    for d in state.layers:
        if state.block == "load":
            lin = [_Layer(w.clone(), s.clone()) for w, s in d.ckpt]     # what the loader filled
            for layer in lin:
                kernel.process_weights_after_loading(layer)
            out.append([(layer.weight, layer.weight_scale) for layer in lin])
        elif state.block == "linear":
            out.append(kernel.apply(d.lin[0], d.x, d.bias))
        else:
            qs, res = F.add_rms_quant(d.norm, d.h, d.res)
            first = kernel.apply(d.lin[0], qs)
            if state.block == "mlp":
                last, _ = F.silu_mul_down(d.lin[1], first)
            else:
                last = kernel.apply(d.lin[1], F.gdn_norm_quant(d.attn, d.core, d.z))
            out.append((res, first, last))
    return out


def run(state):
    if state.graph is None:
        return _pass(state)
    state.graph.replay()
    return state.out


def work(case):
    hidden, _, attn, inter = SHAPES[case["shape"]]
    M, lin = case["M"], _linears(case)
    weights = sum(n * k * 17 / 32 for n, k in lin)
    if case["block"] == "load":
        return dict(bytes=case["layers"] * 2 * weights, flops=0)
    flops = sum(2 * M * n * k for n, k in lin)
    moved = weights + sum(2 * M * n for n, k in lin)                    # each projection's output
    if case["block"] == "linear":
        moved += 2 * M * lin[0][1] + (2 * lin[0][0] if case["bias"] else 0)
    else:
        moved += 6 * M * hidden + 2 * hidden                            # h, residual in and out
        moved += 2 * M * 2 * inter if case["block"] == "mlp" else 4 * M * attn
    return dict(bytes=case["layers"] * moved, flops=case["layers"] * flops)


def tolerance(case):
    if case["block"] == "load":
        return "exact"
    # Four times the distance from 64 bits: 1.7e-3 for one projection (its bf16 outputs round), up to
    # 2.5e-3 where a projection's rounding goes through the second quantizer of an MLP.
    return {"rel": 1e-2 if case["block"] == "mlp" else 7e-3}


# ---- the same in 64 bits ------------------------------------------------------------------------
_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _dequant(w, ws):
    n, k2 = w.shape
    table = torch.tensor(_E2M1, dtype=torch.float64, device=w.device)
    v = torch.stack([table[(w & 15).int()], table[(w >> 4).int()]], dim=-1)
    scale = torch.exp2(ws.double() - 127)
    return (v.reshape(n, k2 // 16, 32) * scale[..., None]).reshape(n, 2 * k2)


def _quantized(x):
    """The per-token e4m3 quantizer on bf16 values, put back: its scale is defined in 32 bits."""
    x = x.bfloat16().float()
    s = (x.abs().amax(1) * (1.0 / 448.0)).clamp_min(1.0 / (448.0 * 512.0))
    q = (x / s[:, None]).clamp(-448.0, 448.0).to(torch.float8_e4m3fn)
    return q.double() * s[:, None].double()


def _product(x, ckpt, chunk=4096):
    """_quantized(x) @ weight^T, a chunk of output columns at a time."""
    a, (w, ws) = _quantized(x), ckpt
    return torch.cat([a @ _dequant(w[n:n + chunk], ws[n:n + chunk]).T
                      for n in range(0, w.shape[0], chunk)], dim=1)


def _silu(x):
    return x / (1 + torch.exp(-x))


def _granules(w, ws):
    """The repacked order: 16 columns x 128 k of weights, lane l holding column l % 16 and 32-element
    block l / 16; one dword of scales per lane for every four of them. N is padded to 16 and K to 512
    with zero weights of scale 127."""
    n, k = w.shape[0], 2 * w.shape[1]
    pn, pk = -n % 16, -k % 512
    w = torch.nn.functional.pad(w, (0, pk // 2, 0, pn))
    ws = torch.nn.functional.pad(ws, (0, pk // 32, 0, pn), value=127)
    nt, kg = w.shape[0] // 16, w.shape[1] // 256
    wq = w.reshape(nt, 16, kg * 4, 4, 16).permute(0, 2, 3, 1, 4).reshape(w.shape)
    sq = ws.reshape(nt, 16, kg, 4, 4).permute(0, 2, 4, 1, 3).reshape(ws.shape)
    return wq, sq


def exact(case, seed):
    out = []
    for d in _make(case, seed):
        if case["block"] == "load":
            out.append([_granules(*c) for c in d.ckpt])
            continue
        if case["block"] == "linear":
            y = _product(d.x, d.ckpt[0])
            out.append(y if d.bias is None else y + d.bias.double())
            continue
        r = d.h.double() + d.res.double()
        n = r * torch.rsqrt(r.square().mean(1, keepdim=True) + EPS) * (1 + d.norm_w.double())
        first = _product(n, d.ckpt[0])
        if case["block"] == "mlp":
            gate, up = first.bfloat16().double().chunk(2, dim=1)
            t = _silu(gate).bfloat16().double() * up
        else:
            x = d.core.double().reshape(case["M"], -1, 128)
            t = x * torch.rsqrt(x.square().mean(2, keepdim=True) + EPS) * d.gate_w.double()
            t = t.reshape(case["M"], -1) * _silu(d.z.double())
        out.append((r, first, _product(t, d.ckpt[1])))
    return out
