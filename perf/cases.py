"""The workloads whose speed is measured: the quantized FFN, projection, MoE
and weight-loading calls that an engine built on moty_amd makes, through
moty_amd.ops, from one-token decode to whole prefill chunks.

A case names a path ("kind"), a token count S and a layer shape.  Decode-sized
cases run several layers with weights of their own per pass, as a model does,
so that the weights stream from memory and not from a cache.  Weights are
N(0, 0.02) and activations N(0, 1), quantized here in plain torch into the
layouts of include/moty_hw_hip.h."""
import math

import torch

from moty_amd import ORDER_EXPERT, ORDER_TOPK, ops

DEV = "cuda:0"

# (hidden, FFN width) of dense layers: the two the benchmark runs (0.6B and 8B
# class) and generic ones between and beside them, 14336 being the widest row
# that the tests go to and 1088 x 3008 multiples of 64 but not of 128
DENSE = [(1024, 3072), (4096, 12288), (896, 4864), (2048, 5632), (2560, 9728), (3072, 8192), (4096, 14336),
         (1088, 3008)]
# (experts, routed, expert width, hidden) of MoE layers
MOE = [(64, 8, 1024, 2048), (128, 8, 768, 2048), (32, 4, 1408, 1024), (16, 2, 896, 1536)]
# GGUF block types (io/st.h:74): elements and bytes of a block
GGUF = {"q8_0": (4, 32, 34), "q4_0": (5, 32, 18), "q4_k": (6, 256, 144), "q6_k": (8, 256, 210)}

BIG = 4096 * 12288  # elements of the 8B FFN's matrices


def listed():
    return [
        # one token of a 0.6B-class model through its 28 FFNs: the smallest
        # calls, where launches and latency count
        dict(name="q8_decode", kind="q8", S=1, D=1024, I=3072, layers=28),
        # a decode step of 24 concurrent sequences through 8B FFNs
        dict(name="q8_batch24", kind="q8", S=24, D=4096, I=12288, layers=2),
        # a long prompt (ragged, not a multiple of any tile) through an 8B FFN
        dict(name="q8_prefill2000", kind="q8", S=2000, D=4096, I=12288, layers=1),
        # a 512-token chunk through the seven projections of a 0.6B-class
        # layer (q/k/v/gate/up fused by rows, o, down)
        dict(name="q8_proj512", kind="q8_proj", S=512, D=1024, I=3072, layers=8),
        # one token through 8B FFNs in grouped int4, int8 activations
        dict(name="i4g_decode", kind="i4g", S=1, D=4096, I=12288, layers=4),
        # a ragged prefill chunk through the same
        dict(name="i4g_prefill500", kind="i4g", S=500, D=4096, I=12288, layers=1),
        # a prefill chunk with exact f32 activations, the engines' default
        # when IDOT4 is unset
        dict(name="i4g_f32_prefill250", kind="i4g_f32", S=250, D=4096, I=12288, layers=1),
        # a ragged prefill chunk in the 4-row-block format
        dict(name="q4r4_prefill301", kind="q4r4", S=301, D=4096, I=12288, layers=1),
        # one token through 128-expert MoE layers
        dict(name="moe_decode", kind="moe", S=1, E=128, K=8, D=2048, I=768, layers=4, order="topk", skew=0),
        # OLMoE-shaped layer over a 256-token chunk
        dict(name="moe_t256", kind="moe", S=256, E=64, K=8, D=2048, I=1024, layers=1, order="topk", skew=0),
        # 48 decode sequences and a 1024-token chunk in one ragged batch, the
        # routing skewed towards 8 hot experts
        dict(name="moe_t1072_skew", kind="moe", S=1072, E=128, K=8, D=2048, I=768, layers=1, order="expert", skew=1),
        # loading one 8B FFN matrix of a GGUF file into the Q8 layout
        dict(name="load_q4k_q8", kind="load", src="q4_k", dst="q8", O=12288, I=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _stack(S, wbytes):
    """Layers per pass: small calls run a stack of them, to about 300 MB of weights."""
    return max(1, min(28, round(3e8 / wbytes))) if S <= 32 else 1


def draw(rng):
    kind = rng.choice(["q8", "q8", "q8_proj", "i4g", "i4g", "i4g_f32", "q4r4", "q8r4", "moe", "moe", "load"])
    if kind == "load":
        src = rng.choice(sorted(GGUF))
        dst = rng.choice(["q8", "i4g", "q4r4"])
        return dict(kind=kind, src=src, dst=dst, O=_log_int(rng, 256, 12288), I=256 * rng.choice([4, 8, 12, 16]))
    if kind == "moe":
        E, K, I, D = rng.choice(MOE)
        S = _log_int(rng, 1, 1072)
        layers = max(1, min(4, round(3e8 / (min(E, S * K) * 3 * I * D)))) if S <= 32 else 1
        return dict(kind=kind, S=S, E=E, K=K, D=D, I=I, layers=layers, order=rng.choice(["topk", "expert"]),
                    skew=rng.choice([0, 1]))
    D, I = rng.choice(DENSE)
    # the largest listed case of the kind bounds S * D * I
    most = {"q8": 2000, "q8_proj": 2000, "i4g": 500, "i4g_f32": 250, "q4r4": 301, "q8r4": 301}[kind] * BIG
    S = _log_int(rng, 1, min(4096, most // (D * I)))
    if kind == "q8_proj":
        S = max(S, 5)
    per = {"q8": 1, "q8_proj": 1, "i4g": 0.625, "i4g_f32": 0.625, "q4r4": 0.5625, "q8r4": 1.0625}[kind]
    return dict(kind=kind, S=S, D=D, I=I, layers=_stack(S, 3 * D * I * per))


# ---------------------------------------------------------------- weights
def _gen(seed, *path):
    k = seed & 0xFFFFFFFF
    for p in path:
        k = (k * 1000003 + p + 0x9E3779B9) & 0x7FFFFFFFFFFF
    return torch.Generator(device=DEV).manual_seed(k)


def _randn(shape, g, std=1.0):
    return torch.randn(shape, generator=g, device=DEV) * std


def _rows8(w):
    """Per-row int8 (nn/quant.c:12-33): codes [O][I], scales [O]."""
    s = (w.abs().amax(1) / 127).clamp_min(1e-8)
    return torch.round(w / s[:, None]).clamp_(-128, 127).to(torch.int8), s


def _group4(w):
    """Grouped int4 (nn/quant.c:57-83): codes -8..7 [O][I], scales [O][I/32]."""
    g = w.view(w.shape[0], -1, 32)
    s = (g.abs().amax(2) / 7).clamp_min(1e-8)
    return torch.round(g / s[:, :, None]).clamp_(-8, 7).to(torch.int8).view(w.shape), s


def _nibbles(c):
    n = (c + 8).to(torch.uint8)
    return n[:, 0::2] | (n[:, 1::2] << 4)


def _r4(w, q8):
    """4-row blocks (nn/quant.c:135-177): codes [O][I] and f16 scales
    [O][I/32], the scale signed so that the largest weight meets the longer
    end of the code range."""
    g = w.view(w.shape[0], -1, 32)
    lo, hi = (128, 127) if q8 else (8, 7)
    mx = g.gather(2, g.abs().argmax(2, keepdim=True))[:, :, 0]
    opp = torch.where((g > 0) != (mx > 0)[:, :, None], g.abs(), torch.zeros_like(g)).amax(2)
    d = torch.maximum(mx.abs() / lo, opp / hi)
    d = torch.where(mx > 0, -d, d).half()
    inv = torch.where(d != 0, 1 / d.float(), torch.zeros_like(mx))
    return torch.round(g * inv[:, :, None]).clamp_(-lo, hi).to(torch.int8).view(w.shape), d


def _r4_layout(c, d, q8):
    O, I = c.shape  # O % 4 == 0
    c = c.view(O // 4, 4, I // 32, 32).permute(0, 2, 1, 3)
    if not q8:
        n = (c + 8).to(torch.uint8)
        c = n[..., :16] | (n[..., 16:] << 4)
    d = d.view(O // 4, 4, I // 32).permute(0, 2, 1).contiguous().view(torch.int16)
    return c.contiguous().view(-1), d.view(-1)


def _shapes(case):
    D, I = case["D"], case["I"]
    if case["kind"] == "q8_proj":  # q, k, v, gate, up by rows; o; down
        return [(4 * D + 2 * I, D), (D, 2 * D), (D, I)]
    return [(I, D), (I, D), (D, I)]


def _codes(case, seed, layer):
    """[(codes, scales)] of one layer's matrices, in row order."""
    kind = case["kind"]
    out = []
    for j, shape in enumerate(_shapes(case)):
        w = _randn(shape, _gen(seed, layer, j), 0.02)
        out.append(_rows8(w) if kind in ("q8", "q8_proj") else _r4(w, kind == "q8r4") if kind in ("q4r4", "q8r4")
                   else _group4(w))
    return out


def _experts(case, seed, layer):
    E, D, I = case["E"], case["D"], case["I"]
    out = []
    for j, shape in enumerate([(E * I, D), (E * I, D), (E * D, I)]):
        c, s = _rows8(_randn(shape, _gen(seed, layer, j), 0.02))
        out.append((c.view(E, shape[0] // E, shape[1]), s.view(E, -1)))
    router = _randn((E, D), _gen(seed, layer, 3), 0.02)
    bias = None
    if case["skew"]:
        bias = torch.zeros(E, device=DEV)
        bias[::max(1, E // 8)] = 2.0
    return router, bias, out


def _inputs(case, seed, layer):
    widths = {"q8_proj": lambda: (case["D"], 2 * case["D"], case["I"])}.get(case["kind"], lambda: (case["D"],))()
    return [_randn((case["S"], w), _gen(seed, layer, 10 + j)) for j, w in enumerate(widths)]


def _raw(case, seed):
    """GGUF blocks of an [O][I] matrix: random codes and sub-scales, the f16
    scales such that weights come out at about 0.02."""
    _, E, B = GGUF[case["src"]]
    n = case["O"] * case["I"] // E
    raw = torch.randint(0, 256, (n, B), generator=_gen(seed, 0), device=DEV, dtype=torch.uint8)
    unit = {"q8_0": 3e-4, "q4_0": 5e-3, "q4_k": 1e-4, "q6_k": 2e-5}[case["src"]]

    def half(k, scale):
        v = ((torch.rand(n, generator=_gen(seed, k), device=DEV) + 0.5) * scale).half()
        return v.view(torch.int16).view(n, 1).view(torch.uint8)
    if case["src"] == "q6_k":
        raw[:, 208:210] = half(1, unit)
    else:
        raw[:, 0:2] = half(1, unit)
    if case["src"] == "q4_k":
        raw[:, 2:4] = half(2, unit * 7)
    return raw.view(-1)


# ---------------------------------------------------------------- the calls
def prepare(case, seed):
    kind = case["kind"]
    if kind == "load":
        return {"case": case, "raw": _raw(case, seed)}
    S, D = case["S"], case["D"]
    layers = []
    for k in range(case["layers"]):
        xs = _inputs(case, seed, k)
        if kind == "moe":
            router, bias, ex = _experts(case, seed, k)
            (g, gs), (u, us), (d, ds) = ex
            order = ORDER_TOPK if case["order"] == "topk" else ORDER_EXPERT
            w = ops.MoeLayer(router, g, gs, u, us, d, ds, case["K"], norm_topk=int(order == ORDER_EXPERT), order=order,
                             logit_bias=bias)
        else:
            w = _codes(case, seed, k)
            if kind in ("q8", "q8_proj"):
                w = [t for m in w for t in m]
            elif kind in ("i4g", "i4g_f32"):
                w = [t for c, s in w for t in (_nibbles(c), s)]
            else:
                q8 = kind == "q8r4"
                (g, gd), (u, ud), (d, dd) = w
                w = [*_r4_layout(torch.cat([g, u]), torch.cat([gd, ud]), q8), *_r4_layout(d, dd, q8)]
        widths = [m[0] for m in _shapes(case)] if kind == "q8_proj" else [D]
        layers.append((xs, w, [torch.empty((S, n), device=DEV) for n in widths]))
    return {"case": case, "layers": layers}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "load":
        w = ops.gguf_dequant(GGUF[case["src"]][0], state["raw"], case["O"] * case["I"]).view(case["O"], case["I"])
        return ops.quantize_rows(w) if case["dst"] == "q8" else (
            ops.pack_int4_grouped(w) if case["dst"] == "i4g" else ops.pack_r4(w))
    for xs, w, outs in state["layers"]:
        if kind == "q8":
            ops.dense_ffn_q8(xs[0], *w, out=outs[0])
        elif kind == "q8_proj":
            for (xq, sx), q, s, y in zip(ops.qrow_i8_multi(xs), w[0::2], w[1::2], outs):
                ops.matmul_q8_preq(xq, sx, q, s, out=y)
        elif kind == "moe":
            w(xs[0], out=outs[0])
        elif kind in ("i4g", "i4g_f32"):
            ops.dense_ffn_i4g(xs[0], *w, idot4=kind == "i4g", out=outs[0])
        else:
            ops.dense_ffn_r4(xs[0], *w, case["I"], q8=kind == "q8r4", out=outs[0])
    return [y for _, _, outs in state["layers"] for y in outs]


def work(case):
    kind = case["kind"]
    if kind == "load":
        n = case["O"] * case["I"]
        _, E, B = GGUF[case["src"]]
        out = {"q8": n + 4 * case["O"], "i4g": n * 0.625, "q4r4": n * 0.5625}[case["dst"]]
        return {"bytes": n // E * B + out, "flops": 2 * n}
    S, D, I, L = case["S"], case["D"], case["I"], case["layers"]
    if kind == "moe":
        E, K = case["E"], case["K"]
        active = E * (1 - (1 - K / E) ** S)  # expected, routing uniform
        nbytes = active * (3 * I * D + (2 * I + D) * 4) + E * D * 4 + 2 * S * D * 4
        return {"bytes": L * nbytes, "flops": L * S * (6 * K * I * D + 2 * E * D)}
    n = sum(a * b for a, b in _shapes(case))
    rows = sum(a for a, _ in _shapes(case))
    scales = {"q8": rows * 4, "q8_proj": rows * 4, "i4g": n / 8, "i4g_f32": n / 8, "q4r4": n / 16, "q8r4": n / 16}[kind]
    codes = n if kind in ("q8", "q8_proj", "q8r4") else n / 2
    acts = 4 * S * (rows + 3 * D + I if kind == "q8_proj" else 2 * D)
    return {"bytes": L * (codes + scales + acts), "flops": L * 2 * S * n}


def tolerance(case):
    # every entry point gives the reference's bits: integer sums are exact in
    # any order, and the order of every float step is part of the contract
    # (include/moty_hw_hip.h), so a correct implementation differs in no bit
    return "exact"


# ---------------------------------------------------------------- 64 bits
def _q127(x, least):
    s = (x.abs().amax(-1, keepdim=True) / 127).clamp_min(least)
    return torch.round(x / s) * s


def _act(x, kind):
    """The activations as the path quantizes them, in 64 bits."""
    if kind == "i4g_f32":
        return x
    if kind in ("q4r4", "q8r4"):
        return _q127(x.view(x.shape[0], -1, 32), 1e-30).view(x.shape)
    return _q127(x, 1e-12)


def _dense(c, s):
    """Codes [O][I] times their row or group scales, in 64 bits."""
    s = s.double()
    return c.double() * s[:, None] if s.dim() == 1 else (c.double().view(*s.shape, 32) * s[:, :, None]).view(c.shape)


def _matmul(x, m, kind):
    return _act(x, kind) @ _dense(*m).t().contiguous()


def _ffn(x, g, u, d, kind):
    return _matmul(torch.nn.functional.silu(_matmul(x, g, kind)) * _matmul(x, u, kind), d, kind)


def _dequant(case, raw):
    """io/gguf.h:231-330 in 64 bits: [O][I]."""
    src = case["src"]
    b = raw.view(-1, GGUF[src][2])

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()
    if src == "q8_0":
        w = half(0) * b[:, 2:].contiguous().view(torch.int8).double()
    elif src == "q4_0":
        q = b[:, 2:].int()
        w = half(0) * (torch.cat([q & 15, q >> 4], 1) - 8).double()
    elif src == "q4_k":
        s, q = b[:, 4:16].int(), b[:, 16:].int().view(-1, 4, 32)
        a, m, top = s[:, 0:4], s[:, 4:8], s[:, 8:12]
        sc = torch.cat([a & 63, (top & 15) | ((a >> 6) << 4)], 1).double()
        mn = torch.cat([m & 63, (top >> 4) | ((m >> 6) << 4)], 1).double()
        v = torch.stack([q & 15, q >> 4], 2).view(-1, 8, 32).double()
        w = (half(0) * sc)[:, :, None] * v - (half(2) * mn)[:, :, None]
    else:
        ql, qh = b[:, :128].int().view(-1, 2, 2, 32), b[:, 128:192].int().view(-1, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)
        hi = torch.cat([(qh >> (2 * r)) & 3 for r in range(4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double().view(-1, 2, 4, 2, 1)
        w = (half(208) * sc.view(-1, 16)).view(sc.shape) * ((lo | (hi << 4)) - 32).double().view(-1, 2, 4, 2, 16)
    return w.reshape(case["O"], case["I"])


def exact(case, seed):
    kind = case["kind"]
    if kind == "load":
        w = _dequant(case, _raw(case, seed))
        g = w.view(case["O"], -1, 32)
        # the codes are whole numbers, and so have no value in 64 bits; nor
        # has an f16 scale returned as its 16 bits
        return (None, (w.abs().amax(1) / 127).clamp_min(1e-8) if case["dst"] == "q8"
                else (g.abs().amax(2) / 7).clamp_min(1e-8) if case["dst"] == "i4g" else None)
    outs = []
    for k in range(case["layers"]):
        xs = [x.double() for x in _inputs(case, seed, k)]
        if kind == "q8_proj":
            outs += [_matmul(x, m, kind) for x, m in zip(xs, _codes(case, seed, k))]
        elif kind != "moe":
            outs.append(_ffn(xs[0], *_codes(case, seed, k), kind))
        else:
            router, bias, ((g, gs), (u, us), (d, ds)) = _experts(case, seed, k)
            logits = xs[0] @ router.double().t().contiguous()
            p = torch.softmax(logits if bias is None else logits + bias.double(), 1)
            w, idx = p.topk(case["K"], 1)
            if case["order"] == "expert":
                w = w / w.sum(1, keepdim=True)
            y = torch.zeros_like(xs[0])
            for e in range(case["E"]):
                t, j = (idx == e).nonzero(as_tuple=True)
                if t.numel():
                    y.index_add_(0, t, _ffn(xs[0][t], (g[e], gs[e]), (u[e], us[e]), (d[e], ds[e]), kind) *
                                 w[t, j][:, None])
            outs.append(y)
    return outs
