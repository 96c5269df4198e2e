"""The decode work that performance is measured on: single projections, the gated MLP, the two decoder layers, the MoE
feed-forward, the sampler and one whole model step, each through the entry point a serving program calls.

A serving program holds its weights packed, its states and KV caches resident and its step captured into a HIP graph
that it replays once per token (``hip.Graph``, as ``StepProgram`` does); one-off calls go through ``kernels`` directly.
``prepare`` makes what such a program keeps, ``run`` is one replay (or one direct call). M is the rows of a step: 1 for
plain decoding, 2 to 16 for the rows of a speculative verify pass or a small batch of positions.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "lithos-metal_amd"))

from monolith_mi355 import kernels  # noqa: E402
from monolith_mi355.formats import DequantSpec  # noqa: E402
from monolith_mi355.formats import device as DV  # noqa: E402
from monolith_mi355.layers import AttnDecoderLayer, GatedMLP, GdnDecoderLayer, MoeBlock, QuantizedMatrix  # noqa: E402
from monolith_mi355.runtime import hip  # noqa: E402

DEV = "cuda"
EPS = 1e-6
THETA = 1e6
BF16, F64 = torch.bfloat16, torch.float64


# ---- the cases ------------------------------------------------------------------------------------------------------
def listed():
    return [
        # one 4-bit affine projection of a small model, called directly from Python: the smallest call there is, where
        # the launch and the wrapper count
        dict(name="int4_proj_m1", kind="gemv", fmt="int4_affine", n=4096, k=4096, m=1, epilogue="", norm=False,
             graph=False),
        # the 27B checkpoint keeps its mixer projections in FP8: the Gated DeltaNet input projection with its norm, on
        # the eight rows of a verify pass
        dict(name="fp8_in_proj_m8", kind="gemv", fmt="fp8_e4m3", n=16480, k=5120, m=8, epilogue="", norm=True,
             graph=True),
        # a 4-bit affine checkpoint's gate|up projection on a verify pass
        dict(name="int4_gate_up_m8", kind="gemv", fmt="int4_affine", n=34816, k=5120, m=8, epilogue="silu_mul",
             norm=False, graph=True),
        # the 27B gated MLP at the widest step the kernels take
        dict(name="mlp_27b_m16", kind="mlp", hidden=5120, inter=17408, m=16),
        # the 27B Gated DeltaNet layer: three of four layers of the model; one token, and a verify pass
        dict(name="gdn_27b_m1", kind="gdn", hidden=5120, inter=17408, k_heads=16, v_heads=48, m=1),
        dict(name="gdn_27b_m8", kind="gdn", hidden=5120, inter=17408, k_heads=16, v_heads=48, m=8),
        # the gated attention layer over a long int8 context, one token
        dict(name="attn_int8_32k_m1", kind="attn", hidden=5120, inter=17408, heads=24, kv_heads=4, head_dim=128,
             kv="int8", ctx=32768, pos=32750, m=1),
        # the 27B model's own attention geometry (heads of 256, BF16 cache) at a ragged context, a short verify pass
        dict(name="attn_bf16_16k_m4", kind="attn", hidden=5120, inter=17408, heads=24, kv_heads=4, head_dim=256,
             kv="bf16", ctx=16384, pos=16001, m=4),
        # the 35B-A3B hybrid's feed-forward: 256 experts, eight chosen and a shared one; one token, and a verify pass
        dict(name="moe_35b_m1", kind="moe", hidden=2048, experts=256, top_k=8, inter=512, m=1),
        dict(name="moe_35b_m8", kind="moe", hidden=2048, experts=256, top_k=8, inter=512, m=8),
        # drawing the next token from a 248320-token vocabulary, called directly
        dict(name="sample_248k_m1", kind="sample", rows=1, vocab=248320, temperature=0.8, top_k=0, top_p=0.95,
             min_p=0.0),
        # a whole step of a small stack, embedding to logits: a Gated DeltaNet and an attention layer and the BF16 head
        dict(name="model_step_m1", kind="model", hidden=5120, inter=17408, k_heads=16, v_heads=48, heads=24, kv_heads=4,
             head_dim=128, kv="int8", ctx=8192, pos=8000, vocab=248320, m=1),
    ]


def _log(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step))


def draw(rng):
    """One more case: every format, epilogue and norm, M = 1..16, hidden sizes 1024..5120 in steps of 128, row counts
    that are not whole tiles, contexts of 200 to 128K tokens, 16 to 256 experts, vocabularies of 32K to 256K."""
    kind = rng.choice(("gemv", "gemv", "gemv", "mlp", "gdn", "gdn", "attn", "attn", "attn", "moe", "moe", "sample",
                       "model"))
    m = rng.choice((1, 1, 1, 2, 2, 3, 4, 4, 5, 6, 7, 8, 8, 9, 12, 13, 16))
    hidden = _log(rng, 1024, 5120, 128)
    inter = _log(rng, 1536, 17408, 128)
    if kind == "gemv":
        epilogue = rng.choice(("", "", "residual", "silu_mul"))
        n = _log(rng, 1024, 34816, {"": 1, "residual": 8, "silu_mul": 16}[epilogue])
        down = rng.random() < 0.3                        # a down projection: long K, no norm
        return dict(kind=kind, fmt=rng.choice(("nvfp4", "int4_affine", "fp8_e4m3", "bf16")), n=n,
                    k=_log(rng, 2048, 17408, 128) if down else hidden, m=m, epilogue=epilogue,
                    norm=not down and rng.random() < 0.6, graph=rng.random() < 0.75)
    if kind == "mlp":
        return dict(kind=kind, hidden=hidden, inter=inter, m=m)
    if kind == "gdn":
        kh = rng.choice((4, 8, 12, 16))
        return dict(kind=kind, hidden=hidden, inter=inter, k_heads=kh, v_heads=kh * rng.choice((1, 2, 3)), m=m)
    if kind == "attn":
        kv, rep = rng.choice((1, 2, 4, 8)), rng.choice((1, 2, 4, 6, 8))
        m = min(m, 64 // rep)
        ctx = _log(rng, 256, 131072, 64)
        return dict(kind=kind, hidden=hidden, inter=inter, heads=kv * rep, kv_heads=kv,
                    head_dim=rng.choice((128, 128, 256)), kv=rng.choice(("int8", "bf16")), ctx=ctx,
                    pos=ctx - m - rng.randrange(48), m=m)
    if kind == "moe":
        experts = rng.choice((16, 64, 128, 160, 256))
        return dict(kind=kind, hidden=_log(rng, 1024, 4096, 128), experts=experts, top_k=rng.choice((2, 4, 6, 8)),
                    inter=rng.choice((256, 384, 512, 768)), m=m)
    if kind == "sample":
        top_k, top_p, min_p = rng.choice(((0, 0.95, 0.0), (50, 0.0, 0.0), (40, 0.9, 0.0), (0, 0.0, 0.05), (0, 0.0, 0.0)))
        return dict(kind=kind, rows=m, vocab=_log(rng, 32000, 262144), temperature=rng.choice((0.7, 0.8, 1.0)),
                    top_k=top_k, top_p=top_p, min_p=min_p)
    kh = rng.choice((8, 16))
    return dict(kind=kind, hidden=hidden, inter=_log(rng, 1536, 12288, 128), k_heads=kh, v_heads=2 * kh, heads=16,
                kv_heads=rng.choice((2, 4)), head_dim=rng.choice((128, 256)), kv=rng.choice(("int8", "bf16")),
                ctx=8192, pos=8000 - rng.randrange(4000), vocab=_log(rng, 32000, 160000, 8), m=rng.choice((1, 1, 2, 4)))


# ---- inputs: checkpoint-shaped weights and activations, from the seed alone -----------------------------------------
def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * int(seed) + 7919 * salt + 1)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV)


def _rows_bf16(g, m, k):
    return _randn(g, m, k).to(BF16)


def _norm_weight(g, k):
    return 1.0 + 0.1 * _randn(g, k)


E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


class Nvfp4:
    """N(0, 0.02) weights as an NVFP4 checkpoint holds them: E2M1 codes (two a byte, low nibble first), an E4M3 scale
    per 16 columns and a tensor scale. ``parts`` equal row blocks have tensor scales of their own."""

    def __init__(self, g, n, k, parts=1):
        per = n // parts
        codes, scales, tensor = [], [], []
        for _ in range(parts):
            w = _randn(g, per, k) * 0.02
            s2 = w.abs().amax() / (6.0 * 448.0)
            sc = (w.view(per, k // 16, 16).abs().amax(-1) / 6.0 / s2).to(torch.float8_e4m3fn)
            v = w.view(per, k // 16, 16) / (sc.float() * s2).clamp_min(1e-30)[..., None]
            mids = torch.tensor([(a + b) / 2 for a, b in zip(E2M1, E2M1[1:])], device=DEV)
            c = torch.bucketize(v.abs(), mids, out_int32=True).to(torch.uint8) | ((v < 0).to(torch.uint8) << 3)
            c = c.view(per, k)
            codes.append(c[:, 0::2] | (c[:, 1::2] << 4))
            scales.append(sc.view(torch.uint8))
            tensor.append(s2.expand(per))
        self.n, self.k = n, k
        self.codes, self.scales, self.rows = torch.cat(codes), torch.cat(scales), torch.cat(tensor).contiguous()

    def interleaved(self):
        """[gate; up] as the silu·mul epilogue takes it: 8 gate rows, 8 up rows, …"""
        self.codes, self.scales = DV.interleave_rows(*self.codes.chunk(2)), DV.interleave_rows(*self.scales.chunk(2))
        self.rows = DV.interleave_rows(*self.rows[:, None].chunk(2)).reshape(-1).contiguous()
        return self

    def matrix(self, experts=1):
        """The packed weight (``experts`` equal matrices stored back to back) as a layer holds it."""
        n = self.n // experts
        pad = -self.n % 16
        rows = torch.cat([self.rows, self.rows.new_ones(pad)]) if pad else self.rows
        return QuantizedMatrix(self.codes, self.scales, self.rows, kernels.PackedWeight(
            "nvfp4", n, self.k, experts, DV.pack_nvfp4(self.codes, self.scales), rows.contiguous()))

    def rows64(self, lo=0, hi=None):
        hi = self.n if hi is None else hi
        lut = torch.tensor(E2M1 + tuple(-v for v in E2M1), dtype=F64, device=DEV)
        c = self.codes[lo:hi]
        w = torch.stack([lut[(c & 15).long()], lut[(c >> 4).long()]], -1).view(hi - lo, self.k // 16, 16)
        s = self.scales[lo:hi].view(torch.float8_e4m3fn).float().double() * self.rows[lo:hi].double()[:, None]
        return (w * s[..., None]).view(hi - lo, self.k)


class Affine4:
    """N(0, 0.02) weights in 4 bits with a BF16 (scale, bias) per 64 columns: w = scale·code + bias."""

    def __init__(self, g, n, k):
        w = (_randn(g, n, k) * 0.02).view(n, k // 64, 64)
        lo, hi = w.amin(-1), w.amax(-1)
        self.n, self.k = n, k
        self.scale, self.bias = ((hi - lo) / 15).to(BF16), lo.to(BF16)
        c = torch.round((w - self.bias.float()[..., None]) / self.scale.float()[..., None]).clamp(0, 15)
        self.codes = c.to(torch.uint8).view(n, k)

    def packed(self):
        t = {"weight": (self.codes[:, 0::2] | (self.codes[:, 1::2] << 4)).cpu().numpy(),
             "scales": self.scale.float().cpu().numpy(), "biases": self.bias.float().cpu().numpy()}
        return kernels.upload(DequantSpec("int4_affine", (self.n, self.k), t, {"group": 64}), device=DEV)

    def rows64(self, lo=0, hi=None):
        c = self.codes[lo:hi].double().view(-1, self.k // 64, 64)
        return (c * self.scale[lo:hi].double()[..., None] + self.bias[lo:hi].double()[..., None]).view(-1, self.k)


class Fp8:
    """N(0, 0.02) weights in E4M3 with one tensor scale."""

    def __init__(self, g, n, k):
        w = _randn(g, n, k) * 0.02
        self.n, self.k = n, k
        self.scale = float(w.abs().amax() / 448.0)
        self.codes = (w / self.scale).to(torch.float8_e4m3fn).view(torch.uint8)

    def packed(self):
        t = {"weight": self.codes.cpu().numpy()}
        return kernels.upload(DequantSpec("fp8_e4m3", (self.n, self.k), t, {"weight_scale": self.scale}), device=DEV)

    def rows64(self, lo=0, hi=None):
        s = float(torch.tensor(self.scale, dtype=torch.float32))
        return self.codes[lo:hi].view(torch.float8_e4m3fn).float().double() * s


class Bf16:
    """N(0, 0.02) weights in BF16."""

    def __init__(self, g, n, k):
        self.n, self.k = n, k
        self.w = (_randn(g, n, k) * 0.02).to(BF16)

    def packed(self):
        return kernels.PackedWeight("bf16", self.n, self.k, 1, DV.pack_bf16(self.w), None)

    def rows64(self, lo=0, hi=None):
        return self.w[lo:hi].double()


FORMATS = {"nvfp4": Nvfp4, "int4_affine": Affine4, "fp8_e4m3": Fp8, "bf16": Bf16}


def _matmul64(x, w):
    """x·Wᵀ in 64 bits, a block of rows of W at a time."""
    return torch.cat([x @ w.rows64(i, min(i + 8192, w.n)).T for i in range(0, w.n, 8192)], -1)


def _rms64(x, w, eps=EPS):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _silu64(x):
    return x * torch.sigmoid(x)


# ---- a captured step ------------------------------------------------------------------------------------------------
_STREAM = []


def _stream():
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0]


def _record(fn):
    """``fn`` recorded into a graph (an eager call of the same work has grown the library's workspaces)."""
    s = _stream()
    torch.cuda.synchronize()
    g = hip.Graph(s)
    with torch.cuda.stream(s), g:
        fn()
    return g


def _eager(fn):
    s = _stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        fn()
    s.synchronize()


class State:
    """What one case keeps: ``graphs`` replayed in turn (a Gated DeltaNet layer's conv slots alternate) or ``call``, and
    the buffers that hold the outputs afterwards."""

    def __init__(self, outputs, *, graphs=None, call=None, keep=()):
        self.outputs, self.graphs, self.call, self.keep, self.turn = outputs, graphs, call, keep, 0


def run(state):
    if state.call is not None:
        state.call()
    else:
        state.graphs[state.turn].launch(torch.cuda.current_stream())
        state.turn = (state.turn + 1) % len(state.graphs)
    return state.outputs


def prepare(case, seed):
    return KINDS[case["kind"]][0](case, seed)


def work(case):
    nbytes, flops = KINDS[case["kind"]][1](case)
    return {"bytes": int(nbytes), "flops": int(flops)}


def exact(case, seed):
    with torch.no_grad():
        return KINDS[case["kind"]][2](case, seed)


def tolerance(case):
    return KINDS[case["kind"]][3](case)


def _weight_bytes(fmt, n, k):
    return n * k * {"nvfp4": 9, "int4_affine": 9, "fp8_e4m3": 16, "bf16": 32}[fmt] / 16


# ---- one projection -------------------------------------------------------------------------------------------------
def _gemv_inputs(c, seed):
    g = _gen(seed)
    w = FORMATS[c["fmt"]](g, c["n"], c["k"])
    x = _rows_bf16(g, c["m"], c["k"])
    nw = _norm_weight(g, c["k"]) if c["norm"] else None
    res = _rows_bf16(g, c["m"], c["n"]) if c["epilogue"] == "residual" else None
    return w, x, nw, res


def _gemv_prepare(c, seed):
    w, x, nw, res = _gemv_inputs(c, seed)
    if c["epilogue"] == "silu_mul" and c["fmt"] == "nvfp4":
        w.interleaved()
    packed = w.matrix().packed if c["fmt"] == "nvfp4" else w.packed()
    out = torch.empty(c["m"], c["n"] // 2 if c["epilogue"] == "silu_mul" else c["n"], dtype=BF16, device=DEV)

    def call():
        kernels.gemv(packed, x, epilogue=c["epilogue"] or None, residual=res, norm_w=nw, eps=EPS, out=out)
    if not c["graph"]:
        return State(out, call=call, keep=(packed, x, nw, res))
    _eager(call)
    return State(out, graphs=[_record(call)], keep=(packed, x, nw, res))


def _gemv_work(c):
    n_out = c["n"] // 2 if c["epilogue"] == "silu_mul" else c["n"]
    rows = c["m"] * (2 * c["k"] + 2 * n_out + (2 * n_out if c["epilogue"] == "residual" else 0))
    return _weight_bytes(c["fmt"], c["n"], c["k"]) + rows + (4 * c["k"] if c["norm"] else 0), 2 * c["m"] * c["n"] * c["k"]


def _gemv_exact(c, seed):
    w, x, nw, res = _gemv_inputs(c, seed)
    xd = _rms64(x.double(), nw) if nw is not None else x.double()
    if c["epilogue"] == "silu_mul" and c["fmt"] == "nvfp4":
        w.interleaved()
    y = _matmul64(xd, w)
    if c["epilogue"] == "silu_mul":                      # rows in blocks of 8 gate, 8 up
        y = y.view(c["m"], c["n"] // 16, 2, 8)
        return (_silu64(y[:, :, 0]) * y[:, :, 1]).reshape(c["m"], -1)
    return y + res.double() if res is not None else y


def _gemv_tolerance(c):
    # one BF16 rounding of a 32-bit sum (and, behind a norm, of its inputs, which the matrix averages out), 1.7e-3
    # from 64 bits: another order of the sum moves a value to the next BF16 number now and then
    return {"rel": 4e-3, "max": 4e-2}


# ---- the gated MLP --------------------------------------------------------------------------------------------------
class _Mlp:
    def __init__(self, g, hidden, inter):
        self.norm = _norm_weight(g, hidden)
        self.gate_up = Nvfp4(g, 2 * inter, hidden, parts=2)
        self.down = Nvfp4(g, hidden, inter)

    def into(self, mlp):
        mlp.norm_w, mlp.gate_up, mlp.down = self.norm, self.gate_up.interleaved().matrix(), self.down.matrix()

    def exact(self, h):
        y = _matmul64(_rms64(h, self.norm), self.gate_up)
        gate, up = y.chunk(2, -1)
        return h + _matmul64(_silu64(gate) * up, self.down)


def _gen_small(seed):
    return _gen(seed, 1)


def _mlp_inputs(c, seed):
    g = _gen(seed)
    return _Mlp(g, c["hidden"], c["inter"]), _rows_bf16(g, c["m"], c["hidden"])


def _mlp_prepare(c, seed):
    w, h = _mlp_inputs(c, seed)
    mlp = GatedMLP(c["hidden"], c["inter"], _gen_small(seed), DEV, EPS)
    w.into(mlp)
    act = torch.empty(c["m"], c["inter"], dtype=BF16, device=DEV)
    out = torch.empty_like(h)

    def call():
        mlp(h, act=act, out=out)
    _eager(call)
    return State(out, graphs=[_record(call)], keep=(mlp, h, act))


def _mlp_bytes(hidden, inter, m):
    return _weight_bytes("nvfp4", 3 * inter, hidden) + 4 * hidden + m * 4 * hidden


def _mlp_work(c):
    return (_mlp_bytes(c["hidden"], c["inter"], c["m"]), 6 * c["m"] * c["hidden"] * c["inter"])


def _mlp_exact(c, seed):
    w, h = _mlp_inputs(c, seed)
    return w.exact(h.double())


def _layer_tolerance(c):
    # BF16 activations between the projections: a value rounded the other way travels through the ones after it. The
    # MLP and the attention layer are 3e-3 to 4e-3 from 64 bits, the Gated DeltaNet layer 8e-3, the whole step 1.1e-2
    return {"rel": 2e-2 if c["kind"] in ("gdn", "model") else 1e-2, "max": 1e-1}


# ---- the Gated DeltaNet layer ---------------------------------------------------------------------------------------
class _Gdn:
    """Weights, parameters and states of one layer: projection rows z | q | k | v | a | b, heads of 128, conv width 4."""

    def __init__(self, g, c):
        self.hk, self.hv, self.hidden = c["k_heads"], c["v_heads"], c["hidden"]
        self.conv_dim = 128 * (2 * self.hk + self.hv)
        self.n_proj = 128 * self.hv + self.conv_dim + 2 * self.hv
        self.norm = _norm_weight(g, self.hidden)
        self.w_in = Nvfp4(g, self.n_proj, self.hidden)
        self.w_out = Nvfp4(g, self.hidden, 128 * self.hv)
        self.conv_w = (0.3 * _randn(g, self.conv_dim, 4)).to(BF16)
        self.a_log = (torch.rand(self.hv, generator=g, device=DEV) * 3 - 2).to(BF16).float()
        self.dt_bias = _randn(g, self.hv).to(BF16).float()
        self.head_norm = (1.0 + 0.2 * _randn(g, 128)).to(BF16).float()
        self.mlp = _Mlp(g, self.hidden, c["inter"])
        self.conv = (0.5 * _randn(g, self.conv_dim, 3)).to(BF16)
        self.rec = 0.1 * _randn(g, self.hv, 128, 128)

    def layer(self, c, seed):
        layer = GdnDecoderLayer(hidden=self.hidden, k_heads=self.hk, v_heads=self.hv, inter=c["inter"], eps=EPS, device=DEV,
                                seed=seed % (1 << 31))
        layer.norm_w, layer.w_in, layer.w_out = self.norm, self.w_in.matrix(), self.w_out.matrix()
        layer.conv_w, layer.a_log, layer.neg_exp_a = self.conv_w, self.a_log, -torch.exp(self.a_log)
        layer.dt_bias, layer.gdn_norm_w = self.dt_bias, self.head_norm
        self.mlp.into(layer.mlp)
        self.restore(layer)
        return layer

    def restore(self, layer):
        layer.conv_state[0].copy_(self.conv)
        layer.conv_state[1].zero_()
        layer.rec.copy_(self.rec)
        layer.parity = 0

    def exact(self, h):
        m, hv, hk = h.shape[0], self.hv, self.hk
        p = _matmul64(_rms64(h, self.norm), self.w_in)
        z, x, a, b = p.split([128 * hv, self.conv_dim, hv, hv], -1)
        xs = torch.cat([self.conv.double().T, x])                                    # [3 + m, channels]
        w = self.conv_w.double()
        y = _silu64(sum(xs[j: j + m] * w[:, j] for j in range(4)))
        q, k, v = y.split([128 * hk, 128 * hk, 128 * hv], -1)

        def heads(t):
            t = t.view(m, hk, 128)
            return (t * torch.rsqrt(t.square().sum(-1, keepdim=True) + 1e-6)).repeat_interleave(hv // hk, 1)
        q, k, v = heads(q) / math.sqrt(128.0), heads(k), v.view(m, hv, 128)
        beta = torch.sigmoid(b)
        decay = torch.exp(-torch.exp(self.a_log.double()) * torch.nn.functional.softplus(a + self.dt_bias.double()))
        s, o = self.rec.double().clone(), []
        for t in range(m):
            s = s * decay[t][:, None, None]
            delta = (v[t] - torch.einsum("hkv,hk->hv", s, k[t])) * beta[t][:, None]
            s = s + k[t][:, :, None] * delta[:, None, :]
            o.append(torch.einsum("hkv,hk->hv", s, q[t]))
        o = _rms64(torch.stack(o), self.head_norm) * _silu64(z.view(m, hv, 128))
        h1 = h + _matmul64(o.reshape(m, -1), self.w_out)
        return self.mlp.exact(h1), s, xs[-3:].T

    def nbytes(self, m):
        states = 8 * self.hv * 128 * 128 + 12 * self.conv_dim
        return (_weight_bytes("nvfp4", self.n_proj + 128 * self.hv, self.hidden) + 4 * self.hidden + states
                + 8 * self.conv_dim + 8 * self.hv + 512 + m * 4 * self.hidden)


def _gdn_inputs(c, seed):
    g = _gen(seed)
    return _Gdn(g, c), _rows_bf16(g, c["m"], c["hidden"])


def _gdn_prepare(c, seed):
    w, h = _gdn_inputs(c, seed)
    layer = w.layer(c, seed)
    out = torch.empty_like(h)

    def call():
        layer.step(h, out=out)
    _eager(call)
    w.restore(layer)
    graphs = [_record(call), _record(call)]              # one for each conv slot, replayed in turn
    layer.parity = 0
    # the conv state has two slots and a pass writes the other one
    return State({"y": out, "rec": layer.rec, "conv": layer.conv_state}, graphs=graphs, keep=(layer, h))


def _gdn_sizes(c):
    conv_dim = 128 * (2 * c["k_heads"] + c["v_heads"])
    return conv_dim, 128 * c["v_heads"] + conv_dim + 2 * c["v_heads"]


def _gdn_bytes(c):
    conv_dim, n_proj = _gdn_sizes(c)
    hv, hidden, m = c["v_heads"], c["hidden"], c["m"]
    return (_weight_bytes("nvfp4", n_proj + 128 * hv, hidden) + 4 * hidden + 8 * hv * 128 * 128 + 12 * conv_dim
            + 8 * conv_dim + 8 * hv + 512 + m * 2 * hidden + _mlp_bytes(hidden, c["inter"], m) - m * 2 * hidden)


def _gdn_flops(c):
    _, n_proj = _gdn_sizes(c)
    return 2 * c["m"] * (c["hidden"] * (n_proj + 128 * c["v_heads"] + 3 * c["inter"]) + 4 * c["v_heads"] * 128 * 128)


def _gdn_work(c):
    return _gdn_bytes(c), _gdn_flops(c)


def _gdn_exact(c, seed):
    w, h = _gdn_inputs(c, seed)
    y, rec, conv = w.exact(h.double())
    return {"y": y, "rec": rec, "conv": torch.stack([w.conv.double(), conv])}


# ---- the attention layer --------------------------------------------------------------------------------------------
class _Attn:
    """Weights and cache of one layer: projection rows q|gate per head, then k, v; RoPE over 64 dims."""

    ROT = 64

    def __init__(self, g, c):
        self.c, self.hidden, self.heads, self.kv, self.d = c, c["hidden"], c["heads"], c["kv_heads"], c["head_dim"]
        self.n_proj = self.heads * 2 * self.d + 2 * self.kv * self.d
        self.norm = _norm_weight(g, self.hidden)
        self.w_qkv = Nvfp4(g, self.n_proj, self.hidden)
        self.w_o = Nvfp4(g, self.hidden, self.heads * self.d)
        self.q_norm = (1.0 + 0.1 * _randn(g, self.d)).to(BF16).float()
        self.k_norm = (1.0 + 0.1 * _randn(g, self.d)).to(BF16).float()
        self.mlp = _Mlp(g, self.hidden, c["inter"])
        shape = (self.kv, c["ctx"], self.d)
        self.k, self.v = _randn(g, *shape), _randn(g, *shape)
        self.k_scale = self.v_scale = None
        if c["kv"] == "int8":                            # codes and an f16 scale per token and KV head
            self.k_scale, self.v_scale = ((t.abs().amax(-1) / 127).to(torch.float16) for t in (self.k, self.v))
            self.k, self.v = (torch.round(t / s.float()[..., None]).clamp(-127, 127).to(torch.int8)
                              for t, s in ((self.k, self.k_scale), (self.v, self.v_scale)))
        else:
            self.k, self.v = self.k.to(BF16), self.v.to(BF16)

    def layer(self, c, seed):
        layer = AttnDecoderLayer(hidden=self.hidden, heads=self.heads, kv_heads=self.kv, head_dim=self.d,
                                 rotary_dim=self.ROT, theta=THETA, ctx=c["ctx"], inter=c["inter"], eps=EPS, device=DEV,
                                 seed=seed % (1 << 31), kv_dtype=c["kv"])
        layer.norm_w, layer.w_qkv, layer.w_o = self.norm, self.w_qkv.matrix(), self.w_o.matrix()
        layer.q_norm, layer.k_norm = self.q_norm, self.k_norm
        self.mlp.into(layer.mlp)
        cache = layer.cache
        cache.k_codes.copy_(self.k)
        cache.set_v_token_major(self.v)
        if self.k_scale is not None:
            cache.k_scales.copy_(self.k_scale)
            cache.v_scales.copy_(self.v_scale)
        return layer

    def cache64(self, n):
        k, v = self.k[:, :n].double(), self.v[:, :n].double()
        if self.k_scale is not None:
            k, v = k * self.k_scale[:, :n].double()[..., None], v * self.v_scale[:, :n].double()[..., None]
        return k, v

    def exact(self, h):
        m, pos, d = h.shape[0], self.c["pos"], self.d
        p = _matmul64(_rms64(h, self.norm), self.w_qkv)
        qg, k, v = p.split([2 * self.heads * d, self.kv * d, self.kv * d], -1)
        q, gate = qg.view(m, self.heads, 2, d).unbind(2)
        inv = 1.0 / THETA ** (torch.arange(0, self.ROT, 2, dtype=F64, device=DEV) / self.ROT)
        ang = (pos + torch.arange(m, dtype=F64, device=DEV))[:, None] * inv
        # the tables are BF16 by contract
        cos, sin = (torch.cat([f, f], -1).to(BF16).double()[:, None] for f in (ang.cos().float(), ang.sin().float()))

        def rope(x, w):
            x = _rms64(x, w)
            r, rest = x[..., : self.ROT], x[..., self.ROT:]
            a, b = r.chunk(2, -1)
            return torch.cat([r * cos + torch.cat([-b, a], -1) * sin, rest], -1)
        q, k = rope(q, self.q_norm), rope(k.view(m, self.kv, d), self.k_norm)
        ck, cv = self.cache64(pos)
        ck = torch.cat([ck, k.transpose(0, 1)], 1)                                   # [kv, pos + m, d]
        cv = torch.cat([cv, v.view(m, self.kv, d).transpose(0, 1)], 1)
        o = torch.empty(m, self.heads, d, dtype=F64, device=DEV)
        rep = self.heads // self.kv
        for t in range(m):
            n = pos + t + 1
            for j in range(self.kv):
                s = q[t, j * rep: (j + 1) * rep] @ ck[j, :n].T / math.sqrt(d)
                o[t, j * rep: (j + 1) * rep] = torch.softmax(s, -1) @ cv[j, :n]
        o = o * torch.sigmoid(gate)
        return self.mlp.exact(h + _matmul64(o.reshape(m, -1), self.w_o))


def _attn_inputs(c, seed):
    g = _gen(seed)
    return _Attn(g, c), _rows_bf16(g, c["m"], c["hidden"])


def _attn_outputs(layer, out):
    cache = layer.cache
    got = {"y": out, "k": cache.k_codes, "v": cache.v_codes}
    if cache.k_scales is not None:
        got.update(k_scale=cache.k_scales, v_scale=cache.v_scales)
    return got


def _attn_prepare(c, seed):
    w, h = _attn_inputs(c, seed)
    layer = w.layer(c, seed)
    out = torch.empty_like(h)

    def call():
        layer.step(h, c["pos"], out=out)
    _eager(call)
    return State(_attn_outputs(layer, out), graphs=[_record(call)], keep=(layer, h))


def _attn_bytes(c):
    heads, kv, d, hidden, m = c["heads"], c["kv_heads"], c["head_dim"], c["hidden"], c["m"]
    key = kv * (2 * d + 4 if c["kv"] == "int8" else 4 * d)
    return (_weight_bytes("nvfp4", 3 * heads * d + 2 * kv * d, hidden) + 4 * hidden + c["pos"] * key + 2 * m * key
            + _mlp_bytes(hidden, c["inter"], m))


def _attn_flops(c):
    heads, kv, d = c["heads"], c["kv_heads"], c["head_dim"]
    return 2 * c["m"] * (c["hidden"] * (3 * heads * d + 2 * kv * d + 3 * c["inter"]) + 2 * heads * d * c["pos"])


def _attn_work(c):
    return _attn_bytes(c), _attn_flops(c)


def _attn_exact(c, seed):
    w, h = _attn_inputs(c, seed)
    got = {"y": w.exact(h.double()), "k": None, "v": None}
    if c["kv"] == "int8":
        got.update(k_scale=None, v_scale=None)
    return got


def _attn_tolerance(c):
    # besides the activations' rounding: an int8 code of a new row may round to its neighbour
    return dict(_layer_tolerance(c), differ=min(0.5, 0.5 * c["m"] / c["ctx"]))


# ---- the MoE feed-forward -------------------------------------------------------------------------------------------
class _Moe:
    """Router, routed experts and the shared expert after them, with the router's row for the shared expert's gate."""

    def __init__(self, g, c):
        self.e, self.top_k, self.hidden, self.inter = c["experts"], c["top_k"], c["hidden"], c["inter"]
        self.norm = _norm_weight(g, self.hidden)
        self.router = (_randn(g, self.e + 1, self.hidden) * 0.02).to(BF16)
        self.gate_up = Nvfp4(g, (self.e + 1) * 2 * self.inter, self.hidden)          # per expert: 8 gate, 8 up, …
        self.down = Nvfp4(g, (self.e + 1) * self.hidden, self.inter)

    def block(self, c, seed):
        block = MoeBlock(hidden=self.hidden, experts=self.e, top_k=self.top_k, inter=self.inter, shared_inter=self.inter,
                         eps=EPS, device=DEV, seed=seed % (1 << 31))
        block.norm_w = self.norm
        block.router_gate = kernels.PackedWeight("bf16", self.e + 1, self.hidden, 1, DV.pack_bf16(self.router), None)
        block.gate_up_s = self.gate_up.matrix(self.e + 1).packed
        block.down_s = self.down.matrix(self.e + 1).packed
        return block

    def expert(self, x, i):
        n = 2 * self.inter
        y = (x @ self.gate_up.rows64(i * n, (i + 1) * n).T).view(-1, n // 16, 2, 8)
        act = (_silu64(y[:, :, 0]) * y[:, :, 1]).reshape(-1, self.inter)
        return act @ self.down.rows64(i * self.hidden, (i + 1) * self.hidden).T

    def exact(self, h):
        x = _rms64(h, self.norm)
        # the choice is defined on the BF16 logits of the BF16 input; ties go to the lower index
        logits = (x.to(BF16).double() @ self.router.double().T).to(BF16).double()
        p = torch.softmax(logits[:, : self.e], -1)
        y = h.clone()
        for t in range(h.shape[0]):
            ids = torch.sort(p[t], descending=True, stable=True).indices[: self.top_k]
            wts = p[t][ids] / p[t][ids].sum()
            for i, wt in zip(ids.tolist(), wts):
                y[t] += wt * self.expert(x[t: t + 1], i)[0]
        return y + torch.sigmoid(logits[:, self.e:]) * self.expert(x, self.e)


def _moe_inputs(c, seed):
    g = _gen(seed)
    return _Moe(g, c), _rows_bf16(g, c["m"], c["hidden"])


def _moe_prepare(c, seed):
    w, h = _moe_inputs(c, seed)
    block = w.block(c, seed)
    out = torch.empty_like(h)

    def call():
        block(h, out=out)
    _eager(call)
    return State(out, graphs=[_record(call)], keep=(block, h))


def _moe_work(c):
    e, k, hidden, inter, m = c["experts"], c["top_k"], c["hidden"], c["inter"], c["m"]
    chosen = e * (1 - (1 - k / e) ** m) + 1              # distinct experts that m tokens meet, and the shared one
    return (chosen * _weight_bytes("nvfp4", 3 * inter, hidden) + 2 * (e + 1) * hidden + 4 * hidden + m * 4 * hidden,
            2 * m * hidden * (e + 1 + 3 * inter * (k + 1)))


def _moe_exact(c, seed):
    w, h = _moe_inputs(c, seed)
    return w.exact(h.double())


# ---- drawing a token ------------------------------------------------------------------------------------------------
def _sample_inputs(c, seed):
    g = _gen(seed)
    # logits of a trained head: a broad bulk and a few dozen likely tokens
    x = 2.5 * _randn(g, c["rows"], c["vocab"])
    at = torch.randint(0, c["vocab"], (c["rows"], 40), generator=g, device=DEV)
    return x.scatter_add_(1, at, 6.0 + 3.0 * _randn(g, c["rows"], 40)).to(BF16)


def _sample_prepare(c, seed):
    logits = _sample_inputs(c, seed)
    ids = torch.empty(c["rows"], dtype=torch.int32, device=DEV)

    def call():
        kernels.sample(logits, temperature=c["temperature"], top_k=c["top_k"], top_p=c["top_p"], min_p=c["min_p"],
                       seed=seed, step=7, out=ids)
    return State(ids, call=call, keep=(logits,))


def _sample_work(c):
    return 2 * c["rows"] * c["vocab"] + 4 * c["rows"], 4 * c["rows"] * c["vocab"]


# ---- a whole step ---------------------------------------------------------------------------------------------------
class _Model:
    def __init__(self, g, c):
        self.c = c
        self.table = (0.5 * _randn(g, c["vocab"], c["hidden"])).to(BF16)
        self.gdn, self.attn = _Gdn(g, c), _Attn(g, c)
        self.norm = _norm_weight(g, c["hidden"])
        self.head = Bf16(g, c["vocab"], c["hidden"])
        self.ids = torch.randint(0, c["vocab"], (c["m"],), generator=g, device=DEV).to(torch.int32)


def _model_prepare(c, seed):
    w = _Model(_gen(seed), c)
    m, gdn, attn, head = c["m"], w.gdn.layer(c, seed), w.attn.layer(c, seed), w.head.packed()
    h = [torch.empty(m, c["hidden"], dtype=BF16, device=DEV) for _ in range(3)]
    logits = torch.empty(m, c["vocab"], dtype=BF16, device=DEV)
    w.head = None

    def call():
        kernels.embed(w.table, w.ids, t=m, out=h[0])
        gdn.step(h[0], out=h[1])
        attn.step(h[1], c["pos"], out=h[2])
        kernels.gemv(head, h[2], norm_w=w.norm, eps=EPS, out=logits)
    _eager(call)
    w.gdn.restore(gdn)
    graphs = [_record(call), _record(call)]
    gdn.parity = 0
    return State({"logits": logits, "rec": gdn.rec}, graphs=graphs, keep=(w, gdn, attn, head, h))


def _model_work(c):
    nbytes, flops = _gdn_bytes(c) + _attn_bytes(c), _gdn_flops(c) + _attn_flops(c)
    return (nbytes + c["vocab"] * c["hidden"] * 2 + 4 * c["hidden"] + c["m"] * 2 * (c["hidden"] + c["vocab"]),
            flops + 2 * c["m"] * c["vocab"] * c["hidden"])


def _model_exact(c, seed):
    w = _Model(_gen(seed), c)
    y, rec, _ = w.gdn.exact(w.table[w.ids.long()].double())
    y = w.attn.exact(y)
    return {"logits": _matmul64(_rms64(y, w.norm), w.head), "rec": rec}


KINDS = {
    "gemv": (_gemv_prepare, _gemv_work, _gemv_exact, _gemv_tolerance),
    "mlp": (_mlp_prepare, _mlp_work, _mlp_exact, _layer_tolerance),
    "gdn": (_gdn_prepare, _gdn_work, _gdn_exact, _layer_tolerance),
    "attn": (_attn_prepare, _attn_work, _attn_exact, _attn_tolerance),
    "moe": (_moe_prepare, _moe_work, _moe_exact, _layer_tolerance),
    "sample": (_sample_prepare, _sample_work, lambda c, s: None, lambda c: "exact"),
    "model": (_model_prepare, _model_work, _model_exact, _layer_tolerance),
}
