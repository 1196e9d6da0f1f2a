"""The work that the K-quant matmuls, expert gathers and decode attention are measured on.

Five kinds of work, each through the ops a program calls:

  linear   one weight matrix (ops.quantized_matmul), any codec, a decode row up to a prompt chunk
  layer    the linear projections of a transformer layer in the Q4_K_M mix: q|k|v, o, gate|up and down; decode
           batches are replayed from a HIP graph, as a serving loop keeps them, prompt chunks run eagerly
  mlp      a whole MLP (ops.fused_mlp) over a prompt chunk
  moe      a mixture-of-experts layer: router, fused GLU gather, down gather with the routing mix
  attn     one query token per row over a left-padded cache, per-row slabs or an 8-bit cache, and the shared-prefix
           (cascade) form, at decode and verify widths

Weights are GGUF blocks, quantised here from N(0, 0.02) by a plain min / max rule (the IQ2_XXS ones are random grid
picks of the same spread); activations are N(0, 1) with a few large channels, K / V and queries N(0, 1).  exact()
dequantises and multiplies the same bytes in 64 bits with torch alone.
"""
import math

import numpy as np
import torch

from gmlx_amd import ops

QK = 256
BLOCK = {"q4_k": 144, "q6_k": 210, "iq2_xxs": 66}
DTYPE = {"f16": torch.float16, "bf16": torch.bfloat16}


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # a small model's MLP-up row at batch 1: launch latency and the call itself
        dict(name="linear_b1_small", kind="linear", codec="q4_k", N=3072, K=1024, M=1, dtype="f16"),
        # the default decode width of a server on an 8B model: four launches a layer, weights streamed once
        dict(name="layers_decode_b8", kind="layer", hidden=4096, qrows=4096, kvrows=1024, inter=12288, M=8,
             dtype="f16", layers=4, graph=True),
        # a busy server: more rows than a decode batch usually has, bf16, an odd count
        dict(name="layers_decode_b37_bf16", kind="layer", hidden=4096, qrows=4096, kvrows=1024, inter=12288, M=37,
             dtype="bf16", layers=2, graph=True),
        # a short prompt, ragged row count
        dict(name="layer_prompt_333", kind="layer", hidden=4096, qrows=4096, kvrows=1024, inter=12288, M=333,
             dtype="f16", layers=1, graph=False),
        # a full prefill chunk through the MLP, the largest work here
        dict(name="mlp_prompt_2048_bf16", kind="mlp", hidden=4096, inter=12288, down="q6_k", codec="q4_k", M=2048,
             dtype="bf16"),
        # an MoE layer at a decode batch of 32
        dict(name="moe_decode_t32", kind="moe", E=128, D=2048, I=768, k=8, T=32, gu="q4_k", down="q6_k",
             dtype="f16", graph=True),
        # a large 2-bit MoE layer at a decode batch of 8
        dict(name="moe_decode_iq2_t8", kind="moe", E=256, D=7168, I=2048, k=8, T=8, gu="iq2_xxs", down="iq2_xxs",
             dtype="f16", graph=True),
        # the same kind of layer over a prompt chunk: every expert gets a few tens of rows
        dict(name="moe_prompt_t500_bf16", kind="moe", E=128, D=2048, I=768, k=8, T=500, gu="q4_k", down="q6_k",
             dtype="bf16", graph=False),
        # chat decode: few rows, short left-padded caches, one call per layer
        dict(name="attn_padded_b3_short", kind="attn", form="padded", layers=8, B=3, Hq=32, Hkv=8, D=128, lo=300,
             hi=1900, qL=1, dtype="bf16", lens=1, graph=True),
        # a long-context batch with very different row lengths
        dict(name="attn_slabs_b16_long", kind="attn", form="slabs", layers=1, B=16, Hq=32, Hkv=8, D=128, lo=1024,
             hi=131072, qL=1, dtype="f16", lens=0, graph=False),
        # an 8-bit KV cache at moderate depth
        dict(name="attn_q8_b6_mid", kind="attn", form="q8", layers=2, B=6, Hq=32, Hkv=8, D=128, lo=6000, hi=12000,
             qL=1, dtype="bf16", lens=2, graph=True),
        # sequences that share a long system prompt
        dict(name="attn_cascade_b8", kind="attn", form="cascade", layers=2, B=8, Hq=32, Hkv=8, D=128, P=16384, S=512,
             lo=384, hi=512, qL=1, dtype="f16", lens=3, graph=True),
    ]


def _log(rng, lo, hi, step=1):
    return max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)) * step)


def draw(rng):
    kind = rng.choice(["linear", "linear", "layer", "layer", "mlp", "moe", "moe", "attn", "attn", "attn"])
    dtype = rng.choice(["f16", "bf16"])
    if kind == "linear":
        return dict(kind=kind, codec=rng.choice(["q4_k", "q6_k", "iq2_xxs"]), N=_log(rng, 250, 32000),
                    K=_log(rng, 256, 14336, QK), M=_log(rng, 1, 1024), dtype=dtype)
    if kind == "layer":
        hidden, qrows, kvrows, inter = rng.choice([(1024, 2048, 1024, 3072), (2048, 4096, 512, 6144),
                                                   (2560, 4096, 1024, 9728), (4096, 4096, 1024, 12288),
                                                   (4096, 4096, 1024, 14336), (5120, 8192, 1024, 17408)])
        M = _log(rng, 1, 1024)
        return dict(kind=kind, hidden=hidden, qrows=qrows, kvrows=kvrows, inter=inter, M=M, dtype=dtype,
                    layers=2 if M <= 64 else 1, graph=M <= 64)
    if kind == "mlp":
        hidden, inter = rng.choice([(1024, 3072), (2048, 6144), (4096, 12288), (4096, 14336)])
        return dict(kind=kind, hidden=hidden, inter=inter, codec="q4_k", down=rng.choice(["q4_k", "q6_k"]),
                    M=_log(rng, 65, 1600), dtype=dtype)
    if kind == "moe":
        E, D, I, gu, down = rng.choice([(128, 2048, 768, "q4_k", "q6_k"), (128, 2048, 768, "q4_k", "q4_k"),
                                        (64, 2048, 1024, "q4_k", "q6_k"), (8, 4096, 6144, "q4_k", "q6_k"),
                                        (256, 7168, 2048, "iq2_xxs", "iq2_xxs")])
        T = _log(rng, 1, 512 if E > 8 else 128)
        return dict(kind=kind, E=E, D=D, I=I, k=min(8, E // 4), T=T, gu=gu, down=down, dtype=dtype, graph=T <= 64)
    form = rng.choice(["padded", "padded", "slabs", "q8", "cascade"])
    D = rng.choice([64, 128, 128, 256])
    Hkv = rng.choice([2, 4, 8, 8])
    B = _log(rng, 1, 32)
    Hq = Hkv * rng.choice([1, 4, 4, 5, 8])
    lens = rng.randrange(1 << 20)
    if form == "cascade":
        B = max(2, min(B, 8))
        S = _log(rng, 32, 2048)
        return dict(kind=kind, form=form, layers=2, B=B, Hq=Hq, Hkv=Hkv, D=D, P=_log(rng, 1024, 32768), S=S,
                    lo=max(8, S - 128), hi=S, qL=rng.choice([1, 1, 2, 4]), dtype=dtype, lens=lens, graph=True)
    hi = _log(rng, 64, min(65536, 2000000 // (B * Hkv)))
    return dict(kind=kind, form=form, layers=1 if hi * B > 100000 else 4, B=B, Hq=Hq, Hkv=Hkv, D=D,
                lo=max(1, hi // rng.choice([1, 3, 20])), hi=hi, qL=1, dtype=dtype, lens=lens, graph=form != "slabs")


# ------------------------------------------------------------- GGUF wire bytes

# The IQ2_XXS grid: code i holds eight 2-bit digits that pick a magnitude of {8, 25, 43}.
_GRID = (
    0, 2, 5, 8, 10, 17, 20, 32, 34, 40, 42, 65, 68, 80, 88, 97, 100, 128, 130, 138, 162, 257, 260, 272, 277, 320, 388,
    408, 512, 514, 546, 642, 1025, 1028, 1040, 1057, 1060, 1088, 1090, 1096, 1120, 1153, 1156, 1168, 1188, 1280, 1282,
    1288, 1312, 1350, 1385, 1408, 1425, 1545, 1552, 1600, 1668, 1700, 2048, 2053, 2056, 2068, 2088, 2113, 2116, 2128,
    2130, 2184, 2308, 2368, 2562, 2580, 4097, 4100, 4112, 4129, 4160, 4192, 4228, 4240, 4245, 4352, 4360, 4384, 4432,
    4442, 4480, 4644, 4677, 5120, 5128, 5152, 5157, 5193, 5248, 5400, 5474, 5632, 5654, 6145, 6148, 6160, 6208, 6273,
    6400, 6405, 6560, 6737, 8192, 8194, 8202, 8260, 8289, 8320, 8322, 8489, 8520, 8704, 8706, 9217, 9220, 9232, 9280,
    9302, 9472, 9537, 9572, 9872, 10248, 10272, 10388, 10820, 16385, 16388, 16400, 16408, 16417, 16420, 16448, 16456,
    16470, 16480, 16513, 16516, 16528, 16640, 16672, 16737, 16768, 16773, 16897, 16912, 16968, 16982, 17000, 17408,
    17416, 17440, 17536, 17561, 17682, 17700, 17920, 18433, 18436, 18448, 18496, 18501, 18688, 18776, 18785, 18818,
    19013, 19088, 20480, 20488, 20497, 20505, 20512, 20608, 20616, 20740, 20802, 20900, 21137, 21648, 21650, 21770,
    22017, 22100, 22528, 22545, 22553, 22628, 22848, 23048, 24580, 24592, 24640, 24680, 24832, 24917, 25112, 25184,
    25600, 25605, 25872, 25874, 25988, 26690, 32768, 32770, 32778, 32833, 32898, 33028, 33048, 33088, 33297, 33793,
    33796, 33808, 33813, 33856, 33888, 34048, 34118, 34196, 34313, 34368, 34400, 34818, 35076, 35345, 36868, 36880,
    36900, 36928, 37025, 37142, 37248, 37445, 37888, 37922, 37956, 38225, 39041, 39200, 40962, 41040, 41093, 41225,
    41472, 42008, 43088, 43268)


def _bytes(t):
    return t.contiguous().view(torch.uint8)


def _wire_q4(w):
    nb = w.shape[0]
    w = w.view(nb, 8, 32)
    low = w.amin(2).clamp(max=0).neg()
    step = (w.amax(2) + low) / 15
    d = (step.amax(1) / 63).half()
    dm = (low.amax(1) / 63).half()
    ls = (step / d.float().clamp(min=1e-7)[:, None]).round().clamp(0, 63)
    lm = (low / dm.float().clamp(min=1e-7)[:, None]).round().clamp(0, 63)
    unit = (d.float()[:, None] * ls).clamp(min=1e-9)[:, :, None]
    q = ((w + (dm.float()[:, None] * lm)[:, :, None]) / unit).round_().clamp_(0, 15).to(torch.uint8)
    ls, lm = ls.to(torch.uint8), lm.to(torch.uint8)
    sc = torch.cat([ls[:, :4] | (ls[:, 4:] >> 4 << 6), lm[:, :4] | (lm[:, 4:] >> 4 << 6),
                    (ls[:, 4:] & 15) | ((lm[:, 4:] & 15) << 4)], 1)
    q = q.view(nb, 4, 2, 32)
    qs = (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(nb, 128)
    return torch.cat([_bytes(d[:, None]), _bytes(dm[:, None]), sc, qs], 1)


def _wire_q6(w):
    nb = w.shape[0]
    w = w.view(nb, 16, 16)
    step = w.abs().amax(2) / 31
    d = (step.amax(1) / 127).half()
    sc = (step / d.float().clamp(min=1e-7)[:, None]).round().clamp(1, 127)
    q = (w / (d.float()[:, None] * sc).clamp(min=1e-9)[:, :, None]).round_().clamp_(-32, 31).add_(32).to(torch.uint8)
    q = q.view(nb, 2, 4, 32)  # half, quarter, position
    ql = torch.stack([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
    qh = (q[:, :, 0] >> 4) | (q[:, :, 1] >> 4 << 2) | (q[:, :, 2] >> 4 << 4) | (q[:, :, 3] >> 4 << 6)
    return torch.cat([ql.reshape(nb, 128), qh.reshape(nb, 64), sc.to(torch.uint8), _bytes(d[:, None])], 1)


def _wire(gen, codec, *shape):
    """Wire bytes [..., K / 256 * block] of a matrix or expert stack [..., K] of N(0, 0.02) values."""
    nb = math.prod(shape) // QK
    cols = shape[-1] // QK * BLOCK[codec]
    if codec == "iq2_xxs":
        out = torch.randint(0, 256, (nb, 66), dtype=torch.uint8, device="cuda", generator=gen)
        d = 4.0e-4 * (1 + 0.3 * torch.rand(nb, 1, device="cuda", generator=gen))
        out[:, :2] = _bytes(d.half())
        return out.view(*shape[:-1], cols)
    make = _wire_q4 if codec == "q4_k" else _wire_q6
    out = torch.empty(nb, BLOCK[codec], dtype=torch.uint8, device="cuda")
    part = 1 << 18  # blocks at a time: 64 M values
    for i in range(0, nb, part):
        n = min(part, nb - i)
        out[i:i + n] = make(torch.randn(n, QK, device="cuda", generator=gen).mul_(0.02))
    return out.view(*shape[:-1], cols)


def _half(b):
    return b.contiguous().view(torch.float16).double()


def _values(wire, codec):
    """The weights of wire rows [N, cols] in 64 bits, [N, K]."""
    N = wire.shape[0]
    b = wire.reshape(-1, BLOCK[codec])
    nb = b.shape[0]
    if codec == "q4_k":
        d, dm = _half(b[:, 0:2]), _half(b[:, 2:4])
        s = b[:, 4:16]
        ls = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6 << 4)], 1).double()
        lm = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6 << 4)], 1).double()
        qs = b[:, 16:].view(nb, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(nb, 8, 32).double()
        v = (d * ls)[:, :, None] * q - (dm * lm)[:, :, None]
    elif codec == "q6_k":
        ql, qh = b[:, :128].view(nb, 2, 2, 32), b[:, 128:192].view(nb, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)
        hi = torch.cat([qh & 3, (qh >> 2) & 3, (qh >> 4) & 3, qh >> 6], 2)
        q = (lo | (hi << 4)).double() - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        v = (_half(b[:, 208:210]) * sc)[:, :, None] * q.view(nb, 16, 16)
    else:
        grid = torch.tensor([[(8, 25, 43)[(c >> (2 * j)) & 3] for j in range(8)] for c in _GRID], dtype=torch.float64)
        sign = torch.tensor([[-1.0 if ((i | ((bin(i).count("1") & 1) << 7)) >> j) & 1 else 1.0 for j in range(8)]
                             for i in range(128)], dtype=torch.float64)
        grid, sign = grid.to(b.device), sign.to(b.device)
        aux = b[:, 2:].contiguous().view(nb, 8, 8)
        word = aux[:, :, 4:].contiguous().view(torch.int32).view(nb, 8).long() & 0xFFFFFFFF
        s = torch.stack([(word >> (7 * l)) & 127 for l in range(4)], 2)
        scale = _half(b[:, :2])[:, :, None] * (0.5 + (word >> 28).double()[:, :, None]) * 0.25
        v = scale[..., None] * grid[aux[:, :, :4].long()] * sign[s]
    return v.reshape(N, -1)


# --------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _rows(gen, M, K, dtype):
    x = torch.randn(M, K, device="cuda", generator=gen)
    big = torch.rand(K, device="cuda", generator=gen) < 0.004
    return (x * torch.where(big, 8.0, 1.0)).to(dtype)


def _lens(case):
    r = np.random.default_rng(case["lens"])
    return [int(v) for v in np.exp(r.uniform(math.log(case["lo"]), math.log(case["hi"]), case["B"]))]


def _affine8(x, dt):
    """x [..., D] as an 8-bit affine cache: values, scales and biases per 64."""
    g = x.view(*x.shape[:-1], -1, 64)
    lo, hi = g.amin(-1, keepdim=True), g.amax(-1, keepdim=True)
    s = ((hi - lo) / 255).to(dt)
    b = lo.to(dt)
    q = ((g - b.float()) / s.float()).round_().clamp_(0, 255).to(torch.uint8)
    return q.view(x.shape), s.squeeze(-1), b.squeeze(-1)


def _normal(gen, dt, *shape):
    return torch.randn(*shape, device="cuda", generator=gen).to(dt)


def _attn_inputs(case, gen):
    dt, B, Hq, Hkv, D, qL = DTYPE[case["dtype"]], case["B"], case["Hq"], case["Hkv"], case["D"], case["qL"]
    lens = _lens(case)
    q = _normal(gen, dt, B, Hq, qL, D)
    if case["form"] == "slabs":
        n = sum(lens) * Hkv * D
        offs = [0]
        for n_row in lens[:-1]:
            offs.append(offs[-1] + n_row * Hkv * D)
        return dict(q=q[:, :, 0].contiguous(), k=_normal(gen, dt, n), v=_normal(gen, dt, n), lens=lens, offs=offs)
    if case["form"] == "cascade":
        P, S = case["P"], case["S"]
        # a left-padded cache as the engine holds it: the prefix is row 0's copy, the rest of each row follows it
        keys, values = (_normal(gen, dt, B, Hkv, P + S, D) for _ in range(2))
        starts = torch.tensor([S - n for n in lens], dtype=torch.int32, device="cuda")
        return dict(q=q, k0=keys[0:1, :, :P], v0=values[0:1, :, :P], k=keys[:, :, P:], v=values[:, :, P:],
                    starts=starts, lens=lens)
    L = max(lens)
    starts = torch.tensor([L - n for n in lens], dtype=torch.int32, device="cuda")
    if case["form"] == "padded":
        return dict(q=q, k=_normal(gen, dt, B, Hkv, L, D), v=_normal(gen, dt, B, Hkv, L, D), starts=starts, lens=lens)
    k, v = (_affine8(torch.randn(B, Hkv, L, D, device="cuda", generator=gen), dt) for _ in range(2))
    return dict(q=q, k=k, v=v, starts=starts, lens=lens)


def _inputs(case, seed):
    """What a program has in hand: weights and activations, a list of one dict per layer."""
    gen, kind = _gen(seed), case["kind"]
    dt = DTYPE[case["dtype"]]
    if kind == "linear":
        return [dict(w=_wire(gen, case["codec"], case["N"], case["K"]), x=_rows(gen, case["M"], case["K"], dt))]
    if kind == "layer":
        H, Q, KV, I, M = case["hidden"], case["qrows"], case["kvrows"], case["inter"], case["M"]
        return [dict(q=_wire(gen, "q4_k", Q, H), k=_wire(gen, "q4_k", KV, H), v=_wire(gen, "q6_k", KV, H),
                     o=_wire(gen, "q4_k", H, Q), gate=_wire(gen, "q4_k", I, H), up=_wire(gen, "q4_k", I, H),
                     down=_wire(gen, "q6_k", H, I), x=_rows(gen, M, H, dt), a=_rows(gen, M, Q, dt),
                     y=_rows(gen, M, H, dt), h=_rows(gen, M, I, dt)) for _ in range(case["layers"])]
    if kind == "mlp":
        H, I = case["hidden"], case["inter"]
        return [dict(gate=_wire(gen, case["codec"], I, H), up=_wire(gen, case["codec"], I, H),
                     down=_wire(gen, case["down"], H, I), x=_rows(gen, case["M"], H, dt))]
    if kind == "moe":
        E, D, I, T = case["E"], case["D"], case["I"], case["T"]
        return [dict(gate=_wire(gen, case["gu"], E, I, D), up=_wire(gen, case["gu"], E, I, D),
                     down=_wire(gen, case["down"], E, D, I), x=_rows(gen, T, D, dt),
                     logits=torch.randn(T, E, device="cuda", generator=gen))]
    return [_attn_inputs(case, gen) for _ in range(case["layers"])]


# ----------------------------------------------------------------- one pass

def _one(case, s):
    kind = case["kind"]
    if kind == "linear":
        return [ops.quantized_matmul(s["x"], s["w"], None, case["codec"])]
    if kind == "layer":
        q, k, v = ops.quantized_matmul_grouped([(s["x"], s["q"], "q4_k"), (s["x"], s["k"], "q4_k"),
                                                (s["x"], s["v"], "q6_k")])
        o = ops.quantized_matmul(s["a"], s["o"], None, "q4_k")
        gate, up = ops.quantized_matmul_grouped([(s["y"], s["gate"], "q4_k"), (s["y"], s["up"], "q4_k")])
        return [q, k, v, o, gate, up, ops.quantized_matmul(s["h"], s["down"], None, "q6_k")]
    if kind == "mlp":
        return [ops.fused_mlp(s["x"], s["gate"], s["up"], s["down"], codec=case["codec"], down_codec=case["down"])]
    if kind == "moe":
        idx, scores = ops.moe_router_topk(s["logits"], case["k"], shared_gate=False)
        h = ops.moe_glu_gather_kq(s["x"], s["gate"], s["up"], case["gu"], idx, out_dtype=s["x"].dtype)
        return [idx, scores, ops.gather_qmv_mix_ns_kq(h, s["down"], case["down"], idx, scores)]
    scale = case["D"] ** -0.5
    if case["form"] == "slabs":
        return [ops.sdpa_decode_slabs(s["q"], s["k"], s["v"], s["offs"], s["lens"], case["Hkv"], scale)]
    if case["form"] == "cascade":
        return [ops.sdpa_decode_gqa_cascade(s["q"], s["k0"], s["v0"], s["k"], s["v"], scale, starts=s["starts"])]
    if case["form"] == "q8":
        (k, ks, kb), (v, vs, vb) = s["k"], s["v"]
        return [ops.sdpa_decode_gqa(s["q"], k, v, scale, starts=s["starts"], k_scales=ks, k_biases=kb, v_scales=vs,
                                    v_biases=vb)]
    return [ops.sdpa_decode_gqa(s["q"], s["k"], s["v"], scale, starts=s["starts"])]


def _all(case, inputs):
    return [out for s in inputs for out in _one(case, s)]


_STREAM = []


def prepare(case, seed):
    inputs = _inputs(case, seed)
    if not case.get("graph"):
        return dict(case=case, inputs=inputs)
    # a serving loop captures its decode step once and replays it
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    stream = _STREAM[0]
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        _all(case, inputs)
    torch.cuda.current_stream().wait_stream(stream)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        outs = _all(case, inputs)
    return dict(graph=graph, outs=outs, inputs=inputs)


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["outs"]
    return _all(state["case"], state["inputs"])


# ------------------------------------------------------------ work, tolerance

def _matmul(codec, N, K):
    return N * K // QK * BLOCK[codec]


def work(case):
    kind = case["kind"]
    if kind in ("linear", "layer", "mlp"):
        M = case["M"]
        if kind == "linear":
            mats = [(case["codec"], case["N"], case["K"])]
            rows = case["N"] + case["K"]
        elif kind == "layer":
            H, Q, KV, I = case["hidden"], case["qrows"], case["kvrows"], case["inter"]
            mats = [("q4_k", Q, H), ("q4_k", KV, H), ("q6_k", KV, H), ("q4_k", H, Q), ("q4_k", 2 * I, H),
                    ("q6_k", H, I)]
            rows = 4 * H + 2 * Q + 2 * KV + 3 * I
        else:
            H, I = case["hidden"], case["inter"]
            mats = [(case["codec"], 2 * I, H), (case["down"], H, I)]
            rows = 2 * H
        n = case.get("layers", 1)
        return {"bytes": n * (sum(_matmul(*m) for m in mats) + 2 * M * rows),
                "flops": n * sum(2 * M * N * K for _, N, K in mats)}
    if kind == "moe":
        E, D, I, k, T = case["E"], case["D"], case["I"], case["k"], case["T"]
        touched = E * (1 - (1 - k / E) ** T)
        return {"bytes": touched * (2 * _matmul(case["gu"], I, D) + _matmul(case["down"], D, I)) + T * (D * 6 + E * 4),
                "flops": 6 * T * k * D * I}
    B, Hq, Hkv, D, qL = case["B"], case["Hq"], case["Hkv"], case["D"], case["qL"]
    keys = sum(_lens(case))
    shared = case["P"] if case["form"] == "cascade" else 0
    token = Hkv * 2 * (D + D // 64 * 4 if case["form"] == "q8" else 2 * D)
    return {"bytes": case["layers"] * ((keys + shared) * token + 4 * B * Hq * qL * D),
            "flops": case["layers"] * 4 * Hq * D * qL * (keys + B * shared)}


def tolerance(case):
    # the outputs' own rounding is what shows: 16-bit outputs, and in the MLP and MoE forms a 16-bit h between
    rel = 1.2e-3 if case["dtype"] == "f16" else 8e-3
    if case["kind"] in ("mlp", "moe"):
        return {"rel": 1.5 * rel, "max": 0.05 if case["dtype"] == "f16" else 0.2, "differ": 0.002}
    return {"rel": rel, "max": 0.02 if case["dtype"] == "f16" else 0.1}


# --------------------------------------------------------------------- exact

def _times(x, wire, codec):
    """x . values(wire)^T in 64 bits, a part of the rows at a time."""
    part = max(1, (1 << 27) // (wire.shape[1] // BLOCK[codec] * QK))
    x = x.double()
    return torch.cat([x @ _values(wire[i:i + part], codec).T for i in range(0, wire.shape[0], part)], 1)


def _silu(g):
    return g * torch.sigmoid(g)


def _attend(q, k, v, scale):
    """q [Hq, D] over k, v [Hkv, n, D], in 64 bits."""
    Hkv = k.shape[0]
    s = torch.einsum("hgd,hnd->hgn", q.double().view(Hkv, -1, q.shape[-1]) * scale, k.double())
    return torch.einsum("hgn,hnd->hgd", torch.softmax(s, -1), v.double()).reshape(q.shape)


def _attn_exact(case, s):
    scale, Hkv, D, rows = case["D"] ** -0.5, case["Hkv"], case["D"], []
    for b, n in enumerate(s["lens"]):
        if case["form"] == "slabs":
            k, v = (s[x][s["offs"][b]:s["offs"][b] + n * Hkv * D].view(Hkv, n, D) for x in "kv")
            rows.append(_attend(s["q"][b], k, v, scale))
            continue
        if case["form"] == "cascade":
            own, qL = s["k"].shape[2] - n, case["qL"]
            k, v = (torch.cat([s[x + "0"][0], s[x][b, :, own:]], 1) for x in "kv")
            rows.append(torch.stack([_attend(s["q"][b, :, i], k[:, :k.shape[1] - qL + i + 1],
                                             v[:, :k.shape[1] - qL + i + 1], scale) for i in range(qL)], 1))
            continue
        if case["form"] == "q8":
            k, v = ((w[b].double().view(Hkv, -1, D // 64, 64) * sc[b].double()[..., None] + bi[b].double()[..., None])
                    .view(Hkv, -1, D)[:, -n:] for w, sc, bi in (s["k"], s["v"]))
        else:
            k, v = (s[x][b, :, -n:] for x in "kv")
        rows.append(_attend(s["q"][b, :, 0], k, v, scale)[:, None])
    return torch.stack(rows)


def _moe_exact(case, s):
    p = torch.softmax(s["logits"].double(), -1)
    scores, idx = torch.sort(p, dim=-1, descending=True, stable=True)
    scores, idx = scores[:, :case["k"]], idx[:, :case["k"]]
    scores = scores / (scores.sum(-1, keepdim=True) + 1e-20)
    y = torch.zeros(case["T"], case["D"], dtype=torch.float64, device="cuda")
    for e in torch.unique(idx).tolist():
        t, slot = torch.where(idx == e)
        h = _silu(_times(s["x"][t], s["gate"][e], case["gu"])) * _times(s["x"][t], s["up"][e], case["gu"])
        y.index_add_(0, t, _times(h, s["down"][e], case["down"]) * scores[t, slot][:, None])
    return [idx.int(), scores, y]


def exact(case, seed):
    outs = []
    for s in _inputs(case, seed):
        if case["kind"] == "linear":
            outs.append(_times(s["x"], s["w"], case["codec"]))
        elif case["kind"] == "layer":
            outs += [_times(s["x"], s[n], c) for n, c in (("q", "q4_k"), ("k", "q4_k"), ("v", "q6_k"))]
            outs.append(_times(s["a"], s["o"], "q4_k"))
            outs += [_times(s["y"], s[n], "q4_k") for n in ("gate", "up")]
            outs.append(_times(s["h"], s["down"], "q6_k"))
        elif case["kind"] == "mlp":
            h = _silu(_times(s["x"], s["gate"], case["codec"])) * _times(s["x"], s["up"], case["codec"])
            outs.append(_times(h, s["down"], case["down"]))
        elif case["kind"] == "moe":
            outs += _moe_exact(case, s)
        else:
            outs.append(_attn_exact(case, s))
    return outs
