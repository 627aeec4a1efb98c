"""The work that a user of this library has it do, as cases that can be timed
and checked: projections, the SwiGLU feed-forward, attention, whole blocks
(through the block driver and op by op), the language encoder's layer input,
the pack quantizer and the whole forward, each through its public entry point.

A case is a dict of plain values. prepare() makes its inputs from a seed and
the handles a program keeps (context, resident weights, output planes), run()
is one pass, exact() the same function in 64-bit torch arithmetic.

The widths are the model's: hidden 3840 (30 heads of 128), feed-forward 10240,
adaLN width 256, caption features 2560. Rows are tokens: an image of p x q
pixels is (p / 16) * (q / 16) rows, joined by its caption's rows.
"""
import math
import os
import sys
import zlib

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "vpipe-ming-image_amd"))
import ming_dit_amd as m  # noqa: E402

HID, FFN, HEADS, HD, ADA, CAP = 3840, 10240, 30, 128, 256, 2560
EPS = 1e-5
BLOCK_SHAPES = {"q": (HID, HID), "k": (HID, HID), "v": (HID, HID), "o": (HID, HID),
                "w1": (FFN, HID), "w3": (FFN, HID), "w2": (HID, FFN)}
# What is bound on a projection: nothing (the plain model), one adapter (a
# style or a distillation adapter), the benchmark's eight slots with two of
# them switched off, or eight wide ones.
ADAPTERS = {
    "none": ((), ()),
    "one": ((16,), (0.8,)),
    "eight": ((4, 8, 16, 16, 32, 32, 64, 128), (1.0, 0.5, 0.0, -0.3, 0.8, 0.0, 1.2, 0.25)),
    "wide": ((64,) * 8, (1.4, -0.8, 0.3, 0.9, -0.2, 1.1, 0.6, -0.5)),
}


# ---- the cases ---------------------------------------------------------------
def listed():
    return [
        # one row: a block's adaLN projection when its modulation is made alone
        {"name": "ada_w4_1row", "kind": "lin", "bits": 4, "M": 1, "N": 4 * HID, "K": ADA,
         "adapters": "none"},
        # the language encoder's layer input over a prompt of odd length:
        # norm, biased dense qkv, per-head norm and rotate-half rotation
        {"name": "encoder_231", "kind": "encoder", "M": 231, "n_q": 20, "n_k": 4},
        # a caption (odd length) through a context-refiner block, eight slots
        {"name": "block_caption_w4_203", "kind": "block", "bits": 4, "M": 203, "modulated": False,
         "adapters": "eight"},
        # one projection of a w8 pack with one adapter, 1024 x 1024 pixels
        {"name": "to_q_w8_4096_one", "kind": "lin", "bits": 8, "M": 4096, "N": HID, "K": HID,
         "adapters": "one"},
        # the feed-forward at 1024 x 1024 with its caption, eight slots
        {"name": "ffn_w4_4352_eight", "kind": "ffn", "bits": 4, "M": 4352, "adapters": "eight"},
        # a main block at 512 x 512 with its caption, w8, the plain model
        {"name": "block_w8_1280", "kind": "block", "bits": 8, "M": 1280, "modulated": True,
         "adapters": "none"},
        # a main block of an unquantized checkpoint at 768 x 768, one adapter
        {"name": "block_dense_2560_one", "kind": "block", "bits": 16, "M": 2560,
         "modulated": True, "adapters": "one"},
        # a main block at 1024 x 1024, w4, eight slots
        {"name": "block_w4_4352_eight", "kind": "block", "bits": 4, "M": 4352, "modulated": True,
         "adapters": "eight"},
        # a block's ops called one by one (a host that binds the ops itself)
        # over an odd number of rows
        {"name": "ops_w4_1493_one", "kind": "ops", "bits": 4, "M": 1493, "adapters": "one"},
        # attention at 2048 x 2048
        {"name": "attention_16640", "kind": "attention", "M": 16640, "heads": HEADS},
        # making a pack: the feed-forward's largest matrix to w4
        {"name": "quantize_w4_10240", "kind": "quantize", "bits": 4, "N": FFN, "K": HID},
        # one whole step of the sampler at 1024 x 1024, w4, eight slots
        {"name": "forward_w4_1024", "kind": "forward", "bits": 4, "gh": 64, "gw": 64, "cap": 256,
         "layers": 30, "refiner": 2, "adapters": "eight"},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["lin", "lin", "ffn", "block", "block", "ops", "attention", "encoder",
                       "quantize", "forward"])
    adapters = rng.choice(["none", "none", "one", "eight", "wide"])
    bits = rng.choice([4, 4, 8, 16])
    if kind == "lin":
        N, K = rng.choice([(HID, HID), (FFN, HID), (HID, FFN), (8 * _log(rng, 8, 1920),
                                                                64 * _log(rng, 1, 160))])
        return {"kind": kind, "bits": bits, "M": _log(rng, 1, 16640), "N": N, "K": K,
                "adapters": adapters}
    if kind == "ffn":
        return {"kind": kind, "bits": bits, "M": _log(rng, 16, 16640), "adapters": adapters}
    if kind == "block":
        return {"kind": kind, "bits": bits, "M": _log(rng, 32, 8704),
                "modulated": rng.random() < 0.7, "adapters": adapters}
    if kind == "ops":
        return {"kind": kind, "bits": bits, "M": _log(rng, 32, 8704), "adapters": adapters}
    if kind == "attention":
        return {"kind": kind, "M": _log(rng, 40, 16640), "heads": rng.choice([6, 16, HEADS])}
    if kind == "encoder":
        n_q, n_k = rng.choice([(20, 4), (16, 4), (14, 2), (8, 8)])
        return {"kind": kind, "M": _log(rng, 9, 2048), "n_q": n_q, "n_k": n_k}
    if kind == "quantize":
        return {"kind": kind, "bits": rng.choice([4, 8]), "N": 8 * _log(rng, 32, 1920),
                "K": 64 * _log(rng, 4, 160)}
    return {"kind": "forward", "bits": bits, "gh": rng.randint(16, 64), "gw": rng.randint(16, 64),
            "cap": rng.randint(24, 512), "layers": rng.randint(1, 5), "refiner": 1,
            "adapters": adapters}


# ---- inputs, from the seed alone -----------------------------------------------
def _gen(seed, tag):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + zlib.crc32(tag.encode())) % (1 << 62))
    return g


def _randn(g, shape, std=1.0, mean=0.0):
    t = torch.randn(shape, generator=g, device="cuda")
    return (t * std + mean if (std != 1.0 or mean) else t).to(torch.bfloat16)


def _pack_words(q, bits):
    """Unsigned codes [N, K] -> LSB-first 32-bit words."""
    per = 32 // bits
    q = q.to(torch.int32).reshape(q.shape[0], -1, per)
    w = torch.zeros(q.shape[:2], dtype=torch.int32, device=q.device)
    for i in range(per):
        w |= q[:, :, i] << (bits * i)
    return w


def _weight(seed, tag, N, K, bits):
    """A projection as a checkpoint holds it: dense bf16, or group-64 codes
    with bf16 scales and biases (w4 affine, w8 symmetric)."""
    g = _gen(seed, tag)
    if bits == 16:
        return {"N": N, "K": K, "w": _randn(g, (N, K), 1.0 / math.sqrt(K))}
    w = torch.randn((N, K // 64, 64), generator=g, device="cuda") * 0.02
    if bits == 4:
        lo = w.amin(-1)
        s = ((w.amax(-1) - lo) / 15.0).to(torch.bfloat16)
        b = lo.to(torch.bfloat16)
        q = torch.round((w - b.float()[..., None]) / s.float()[..., None]).clamp_(0, 15)
    else:
        s = (w.abs().amax(-1) / 127.0).to(torch.bfloat16)
        b = (s.float() * -128.0).to(torch.bfloat16)
        q = torch.round(w / s.float()[..., None]).clamp_(-127, 127) + 128
    return {"N": N, "K": K, "bits": bits, "codes": _pack_words(q.reshape(N, K), bits),
            "scales": s.contiguous(), "biases": b.contiguous()}


def _loras(seed, tag, N, K, adapters):
    g = _gen(seed, tag + "/lora")
    return [(_randn(g, (r, K), 1.0 / math.sqrt(K)), _randn(g, (N, r), 0.01))
            for r in ADAPTERS[adapters][0]]


def _positions(gh, gw, cap):
    """Joint positions: image rows at t = cap + 1 on a gh x gw grid, then the
    caption rows at (1 + i, 0, 0)."""
    n = gh * gw
    i = np.arange(n)
    z = np.zeros(cap, np.int64)
    return (np.concatenate([np.full(n, cap + 1), 1 + np.arange(cap)]).astype(np.int32),
            np.concatenate([i // gw, z]).astype(np.int32),
            np.concatenate([i % gw, z]).astype(np.int32))


def _angles(pos):
    """Rotary angles [rows, 64] in 64 bits: 16, 24 and 24 pairs of the axes."""
    out = []
    for p, n in zip(pos, (32, 48, 48)):
        f = 256.0 ** (-np.arange(0, n, 2, dtype=np.float64) / n)
        out.append(np.asarray(p, np.float64)[:, None] * f[None])
    return torch.from_numpy(np.concatenate(out, 1)).cuda()


def _row_positions(rows):
    """Positions of `rows` rows: a nearly square image over a short caption."""
    cap = min(256, max(1, rows // 8))
    n = rows - cap
    gw = max(1, int(round(math.sqrt(n))))
    pt, ph, pw = _positions((n + gw - 1) // gw, gw, cap)
    full = len(pt) - cap
    keep = np.concatenate([np.arange(n), full + np.arange(cap)])
    return pt[keep], ph[keep], pw[keep]


def _block_inputs(seed, tag, bits, modulated, adapters):
    b = {"proj": {}, "lora": {}}
    for name, (N, K) in BLOCK_SHAPES.items():
        b["proj"][name] = _weight(seed, tag + name, N, K, bits)
        b["lora"][name] = _loras(seed, tag + name, N, K, adapters)
    g = _gen(seed, tag + "vec")
    if modulated:
        b["ada"] = _weight(seed, tag + "ada", 4 * HID, ADA, bits)
        b["ada_b"] = _randn(g, (4 * HID,), 0.1)
    for n in ("an1", "an2", "fn1", "fn2"):
        b[n] = _randn(g, (HID,), 0.1, 1.0)
    for n in ("nq", "nk"):
        b[n] = _randn(g, (HD,), 0.1, 1.0)
    return b


def _model_vecs(seed):
    def dense(tag, N, K):
        return _weight(seed, tag, N, K, 16)

    g = _gen(seed, "model")
    return {"time_1": dense("time_1", 1024, 256), "time_1b": _randn(g, (1024,), 0.05),
            "time_2": dense("time_2", ADA, 1024), "time_2b": _randn(g, (ADA,), 0.05),
            "x_in": dense("x_in", HID, 64), "x_in_b": _randn(g, (HID,), 0.05),
            "cap_norm": _randn(g, (CAP,), 0.1, 1.0), "cap_in": dense("cap_in", HID, CAP),
            "cap_in_b": _randn(g, (HID,), 0.05), "final_ada": dense("final_ada", HID, ADA),
            "final_ada_b": _randn(g, (HID,), 0.05), "final_lin": dense("final_lin", 64, HID),
            "final_lin_b": _randn(g, (64,), 0.05)}


def _inputs(c, seed):
    kind, g = c["kind"], _gen(seed, "x")
    if kind == "lin":
        return {"x": _randn(g, (c["M"], c["K"])), "w": _weight(seed, "w", c["N"], c["K"], c["bits"]),
                "lora": _loras(seed, "w", c["N"], c["K"], c["adapters"])}
    if kind == "ffn":
        out = {"x": _randn(g, (c["M"], HID))}
        for n in ("w1", "w3", "w2"):
            out[n] = _weight(seed, n, *BLOCK_SHAPES[n], c["bits"])
            out[n + "_lora"] = _loras(seed, n, *BLOCK_SHAPES[n], c["adapters"])
        return out
    if kind in ("block", "ops"):
        # ops: the gates of the two residuals are given, nothing is modulated
        mod = kind == "block" and c["modulated"]
        b = _block_inputs(seed, "", c["bits"], mod, c["adapters"])
        a = _angles(_row_positions(c["M"]))
        return {"x": _randn(g, (c["M"], HID)), "b": b, "temb": _randn(g, (ADA,)),
                "gates": _randn(g, (2, HID), 0.5), "cos": a.cos().float(), "sin": a.sin().float()}
    if kind == "attention":
        return {"qkv": _randn(g, (c["M"], 3 * c["heads"] * HD))}
    if kind == "encoder":
        D, width = CAP, (c["n_q"] + 2 * c["n_k"]) * HD
        inv = 10000.0 ** (-np.arange(64, dtype=np.float64) / 64)
        a = torch.from_numpy(np.arange(c["M"], dtype=np.float64)[:, None] * inv[None]).cuda()
        return {"x": _randn(g, (c["M"], D)), "norm": _randn(g, (D,), 0.1, 1.0),
                "w": _weight(seed, "qkv", width, D, 16), "b": _randn(g, (width,), 0.2),
                "nq": _randn(g, (HD,), 0.1, 1.0), "nk": _randn(g, (HD,), 0.1, 1.0),
                "cos": a.cos().float().contiguous(), "sin": a.sin().float().contiguous()}
    if kind == "quantize":
        return {"w": torch.randn((c["N"], c["K"]), generator=g, device="cuda") * 0.02}
    n = c["gh"] * c["gw"]
    return {"lat": _randn(g, (n, 64)), "cap": _randn(g, (c["cap"], CAP)),
            "sigma": 0.05 + 0.9 * ((seed * 37) % 101) / 101.0, "m": _model_vecs(seed)}


# ---- what a program keeps -------------------------------------------------------
class State:
    pass


_streams = []


def _stream():
    """The one stream of the program: every pass is queued behind the last."""
    if not _streams:
        _streams.append(torch.cuda.Stream())
    return _streams[0]


def _handle(st, w, loras=()):
    """A resident weight with its adapters bound (device sources)."""
    if "w" in w:
        q = m.QWeight.dense(st.ctx, w["w"], on_device=True)
    else:
        q = m.QWeight.quantized(st.ctx, w["codes"], w["scales"], w["biases"], w["bits"],
                                on_device=True)
    for slot, (A, B) in enumerate(loras):
        q.bind_lora(slot, A, B, on_device=True)
    return q


def _block_handles(st, b):
    parts = {n: _handle(st, b["proj"][n], b["lora"][n]) for n in BLOCK_SHAPES}
    if "ada" in b:
        parts["ada"] = _handle(st, b["ada"])
        parts["ada_b"] = b["ada_b"]
    for n in ("an1", "an2", "fn1", "fn2", "nq", "nk"):
        parts[n] = b[n]
    return parts


def _scales(c):
    return list(ADAPTERS[c["adapters"]][1]) if c["adapters"] != "none" else None


def _empty(*shape, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=dtype, device="cuda")


def prepare(case, seed):
    c, st = case, State()
    st.case, st.stream = c, _stream()
    st.ctx = m.Ctx(0, st.stream.cuda_stream)
    kind = c["kind"]
    d = _inputs(c, seed)
    torch.cuda.synchronize()      # the library reads them on its own stream
    if kind == "lin":
        st.x, st.w = d["x"], _handle(st, d["w"], d["lora"])
        st.y = _empty(c["M"], c["N"])
    elif kind == "ffn":
        st.x = d["x"]
        st.w = [_handle(st, d[n], d[n + "_lora"]) for n in ("w1", "w3", "w2")]
        st.h, st.y = _empty(c["M"], FFN), _empty(c["M"], HID)
    elif kind == "block":
        st.x, st.cos, st.sin, st.temb = d["x"], d["cos"], d["sin"], d["temb"]
        st.desc = m.block_desc(**_block_handles(st, d["b"]))
        st.dims = m.BlockDims(hidden=HID, n_heads=HEADS, ffn=FFN, adaln_dim=ADA, eps=EPS)
        st.y = _empty(c["M"], HID)
        st.ws = _empty(st.ctx.block_workspace_bytes(st.dims, c["M"]), dtype=torch.uint8)
    elif kind == "ops":
        st.x, st.cos, st.sin, st.gates = d["x"], d["cos"], d["sin"], d["gates"]
        st.p = _block_handles(st, d["b"])
        M = c["M"]
        st.y, st.nrm, st.qkv = _empty(M, HID), _empty(M, HID), _empty(M, 3 * HID)
        st.sub, st.g, st.u = _empty(M, HID), _empty(M, FFN), _empty(M, FFN)
    elif kind == "attention":
        st.qkv, st.y = d["qkv"], _empty(c["M"], c["heads"] * HD)
    elif kind == "encoder":
        st.d, st.w = d, _handle(st, d["w"])
        st.nrm, st.y = _empty(c["M"], CAP), _empty(c["M"], st.w.N)
    elif kind == "quantize":
        st.w = d["w"]
        N, K = c["N"], c["K"]
        st.codes = _empty(N, K * c["bits"] // 32, dtype=torch.int32)
        st.s, st.b = (_empty(N, K // 64, dtype=torch.int16) for _ in range(2))
    else:
        st.lat, st.cap, st.sigma = d["lat"], d["cap"], d["sigma"]
        st.pos = _positions(c["gh"], c["gw"], c["cap"])
        blocks = []
        for i in range(2 * c["refiner"] + c["layers"]):
            b = _block_inputs(seed, "block%d/" % i, c["bits"], i >= c["refiner"], c["adapters"])
            torch.cuda.synchronize()
            blocks.append(m.block_desc(**_block_handles(st, b)))
        md = m.ModelDesc()
        md.hidden, md.n_heads, md.ffn = HID, HEADS, FFN
        md.n_layers, md.n_refiner, md.adaln_dim = c["layers"], c["refiner"], ADA
        md.time_freq, md.time_mid, md.patch_dim, md.cap_dim = 256, 1024, 64, CAP
        md.eps, md.rope_theta, md.t_scale = EPS, 256.0, 1000.0
        md.axes[:], md.axes_lens[:] = [32, 48, 48], [1536, 512, 512]
        parts = {k: _handle(st, v) if isinstance(v, dict) else v for k, v in d["m"].items()}
        for k, v in parts.items():
            setattr(md, k, m._h(v))
        r = c["refiner"]
        st.model = m.Model(st.ctx, md, blocks[:r], blocks[r:], keep=[parts, blocks])
        # each pass stands for a step with a caption of its own
        st.model.set_caption_cache(False)
        for slot, s in enumerate(_scales(c) or ()):
            st.model.set_lora_scale(slot, s)
        st.y = _empty(c["gh"] * c["gw"], 64)
    st.ctx.synchronize()
    return st


def run(st):
    c, x = st.case, st.ctx
    kind, M = c["kind"], c.get("M")
    if kind == "lin":
        x.lin(st.w, st.x, st.y, M, _scales(c))
        return st.y
    if kind == "ffn":
        x.ffn(*st.w, st.x, st.y, M, _scales(c), h=st.h)
        return [st.h, st.y]
    if kind == "block":
        with torch.cuda.stream(st.stream):
            st.y.copy_(st.x)          # the block works in place on the stream's rows
        x.block_forward(st.desc, st.dims, st.y, M, st.cos, st.sin,
                        st.temb if c["modulated"] else None, _scales(c), st.ws)
        return st.y
    if kind == "ops":
        p, sc = st.p, _scales(c)
        with torch.cuda.stream(st.stream):
            st.y.copy_(st.x)
        x.rmsnorm(st.x, p["an1"], st.nrm, M, HID, EPS)
        for i, n in enumerate("qkv"):
            x.lin(p[n], st.nrm, st.qkv.data_ptr() + 2 * HID * i, M, sc, ldy=3 * HID)
        x.qk_norm_rope(st.qkv, 3 * HID, 0, HID, M, HEADS, p["nq"], p["nk"], st.cos, st.sin, EPS)
        x.attention(st.qkv, 3 * HID, 0, HID, 2 * HID, st.nrm, HID, M, HEADS)
        x.lin(p["o"], st.nrm, st.sub, M, sc)
        x.rmsnorm(st.sub, p["an2"], st.sub, M, HID, EPS)
        x.gated_residual(st.y, st.gates[0], st.sub, M, HID)
        x.rmsnorm(st.y, p["fn1"], st.nrm, M, HID, EPS)
        x.lin(p["w1"], st.nrm, st.g, M, sc)
        x.lin(p["w3"], st.nrm, st.u, M, sc)
        x.swiglu(st.g, st.u, st.g, M, FFN)
        x.lin(p["w2"], st.g, st.sub, M, sc)
        x.rmsnorm(st.sub, p["fn2"], st.sub, M, HID, EPS)
        x.gated_residual(st.y, st.gates[1], st.sub, M, HID)
        return [st.qkv, st.g, st.y]
    if kind == "attention":
        w = c["heads"] * HD
        x.attention(st.qkv, 3 * w, 0, w, 2 * w, st.y, w, M, c["heads"])
        return st.y
    if kind == "encoder":
        d = st.d
        x.rmsnorm(d["x"], d["norm"], st.nrm, M, CAP, 1e-6)
        x.lin_bias(st.w, st.nrm, st.y, M, d["b"])
        x.llm_qk_norm_rope(st.y, d["nq"], d["nk"], d["cos"], d["sin"], M, st.w.N, c["n_q"],
                           c["n_k"], 64, 1e-6)
        return st.y
    if kind == "quantize":
        x.quantize_pack(st.w, c["N"], c["K"], c["bits"], st.codes, st.s, st.b)
        return [st.codes, st.s, st.b]
    n = c["gh"] * c["gw"]
    st.model.forward(st.lat, st.cap, CAP, n, c["cap"], c["cap"], *st.pos, st.sigma, st.y)
    return st.y


# ---- the work a pass cannot do without -------------------------------------------
def _lin_work(M, N, K, bits, adapters):
    """(weight and adapter bytes, flops) of one projection over M rows."""
    r = sum(a for a, s in zip(*ADAPTERS[adapters]) if s)
    wb = 2.0 * N * K if bits == 16 else N * K * bits / 8.0 + 4.0 * N * K / 64
    return wb + 2.0 * r * (N + K), 2.0 * M * N * K + 2.0 * M * r * (N + K)


def _block_work(M, bits, modulated, adapters):
    b, f = 0.0, 4.0 * HEADS * HD * M * M
    for N, K in BLOCK_SHAPES.values():
        wb, wf = _lin_work(M, N, K, bits, adapters)
        b, f = b + wb, f + wf
    if modulated:
        wb, wf = _lin_work(1, 4 * HID, ADA, bits, "none")
        b, f = b + wb, f + wf
    return b, f


def work(case):
    c, kind, M = case, case["kind"], case.get("M")
    if kind == "lin":
        wb, f = _lin_work(M, c["N"], c["K"], c["bits"], c["adapters"])
        return {"bytes": wb + 2.0 * M * (c["K"] + c["N"]), "flops": f}
    if kind == "ffn":
        b, f = 2.0 * M * (2 * HID + FFN), 0.0      # x in, h and y out
        for n in ("w1", "w3", "w2"):
            wb, wf = _lin_work(M, *BLOCK_SHAPES[n], c["bits"], c["adapters"])
            b, f = b + wb, f + wf
        return {"bytes": b, "flops": f}
    if kind == "block":
        b, f = _block_work(M, c["bits"], c["modulated"], c["adapters"])
        return {"bytes": b + M * (4.0 * HID + 512), "flops": f}
    if kind == "ops":
        # every op reads its rows once and writes them once
        b, f = _block_work(M, c["bits"], False, c["adapters"])
        planes = 8 + (3 + 3) + 4 + 4 + 2 + 6       # norms, qkv, rope, attention, o, residuals
        return {"bytes": b + 2.0 * M * (HID * (planes + 3) + FFN * 6) + 512.0 * M, "flops": f}
    if kind == "attention":
        w = c["heads"] * HD
        return {"bytes": 8.0 * M * w, "flops": 4.0 * w * M * M}
    if kind == "encoder":
        N = (c["n_q"] + 2 * c["n_k"]) * HD
        rope = 4.0 * M * (c["n_q"] + c["n_k"]) * HD + 512.0 * M
        return {"bytes": 6.0 * M * CAP + 2.0 * N * CAP + 2.0 * M * N + rope,
                "flops": 2.0 * M * N * CAP}
    if kind == "quantize":
        n = float(c["N"]) * c["K"]
        return {"bytes": 4.0 * n + n * c["bits"] / 8 + n / 16, "flops": 4.0 * n}
    n, cap = c["gh"] * c["gw"], c["cap"]
    b = 4.0 * n * 64 + 2.0 * cap * CAP + 2.0 * (HID * (64 + CAP + ADA + 64) + 1024 * 512)
    f = 2.0 * n * HID * 128 + 2.0 * cap * HID * CAP
    for i in range(2 * c["refiner"] + c["layers"]):
        rows = cap if i < c["refiner"] else n if i < 2 * c["refiner"] else n + cap
        wb, wf = _block_work(rows, c["bits"], i >= c["refiner"], c["adapters"])
        b, f = b + wb, f + wf
    return {"bytes": b, "flops": f}


def tolerance(case):
    """About four times the distance from the 64-bit result that one bf16
    rounding per op gives (measured: a projection 1.7e-3, the feed-forward
    3.5e-3, attention 2.3e-3, a block 3.6e-3 to 6.3e-3, the forward 1.7e-2)."""
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    rel = {"lin": 6.6e-3, "encoder": 1e-2, "attention": 1e-2, "ffn": 1.4e-2, "block": 2.2e-2,
           "ops": 2.2e-2, "forward": 7e-2}[kind]
    return {"rel": rel}


# ---- the same functions in 64 bits -------------------------------------------------
def _f(t):
    return t.double()


def _w64(w):
    if "w" in w:
        return _f(w["w"])
    bits, per = w["bits"], 32 // w["bits"]
    shifts = torch.arange(per, device="cuda", dtype=torch.int32) * bits
    q = ((w["codes"][:, :, None] >> shifts) & ((1 << bits) - 1)).reshape(w["N"], -1, 64)
    return (_f(q) * _f(w["scales"])[..., None] + _f(w["biases"])[..., None]).reshape(w["N"], w["K"])


def _lin64(x, w, loras=(), adapters="none"):
    y = x @ _w64(w).t()
    for (A, B), s in zip(loras, ADAPTERS[adapters][1]):
        if s:
            y += float(np.float32(s)) * ((x @ _f(A).t()) @ _f(B).t())
    return y


def _rms64(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope64(x, cos, sin):
    """Interleaved pairs of [rows, heads, 128] rotated by cos / sin [rows, 64]."""
    a, b = x[..., 0::2], x[..., 1::2]
    cs, sn = cos[:, None, :], sin[:, None, :]
    return torch.stack((a * cs - b * sn, a * sn + b * cs), -1).flatten(-2)


def _attn64(q, k, v, heads):
    out = torch.empty_like(q)
    for h in range(heads):
        s = slice(HD * h, HD * (h + 1))
        for r in range(0, q.shape[0], 4096):
            p = torch.softmax((q[r:r + 4096, s] / math.sqrt(HD)) @ k[:, s].t(), -1)
            out[r:r + 4096, s] = p @ v[:, s]
    return out


def _block64(x, b, cos, sin, adapters, temb=None, gates=None, keep=None):
    L, rows = b["lora"], x.shape[0]

    def P(n, t):
        return _lin64(t, b["proj"][n], L[n], adapters)

    g1, g3 = _f(b["an1"]), _f(b["fn1"])
    ga = gf = None
    if temb is not None:
        mods = _lin64(temb[None], b["ada"])[0] + _f(b["ada_b"])
        g1, g3 = g1 * (1 + mods[:HID]), g3 * (1 + mods[2 * HID:3 * HID])
        ga, gf = torch.tanh(mods[HID:2 * HID]), torch.tanh(mods[3 * HID:])
    if gates is not None:
        ga, gf = torch.tanh(_f(gates[0])), torch.tanh(_f(gates[1]))
    nrm = _rms64(x, g1, EPS)
    q, k, v = P("q", nrm), P("k", nrm), P("v", nrm)
    q = _rope64(_rms64(q.view(rows, HEADS, HD), _f(b["nq"]), EPS), cos, sin).reshape(rows, HID)
    k = _rope64(_rms64(k.view(rows, HEADS, HD), _f(b["nk"]), EPS), cos, sin).reshape(rows, HID)
    if keep is not None:
        keep.append(torch.cat((q, k, v), 1))
    sub = _rms64(P("o", _attn64(q, k, v, HEADS)), _f(b["an2"]), EPS)
    x = x + (sub if ga is None else ga * sub)
    nrm = _rms64(x, g3, EPS)
    h = torch.nn.functional.silu(P("w1", nrm)) * P("w3", nrm)
    if keep is not None:
        keep.append(h)
    sub = _rms64(P("w2", h), _f(b["fn2"]), EPS)
    return x + (sub if gf is None else gf * sub)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "quantize":
        return None                     # whole numbers, compared as they are
    d = _inputs(c, seed)
    if kind == "lin":
        return _lin64(_f(d["x"]), d["w"], d["lora"], c["adapters"])
    if kind == "ffn":
        x, ad = _f(d["x"]), c["adapters"]
        h = (torch.nn.functional.silu(_lin64(x, d["w1"], d["w1_lora"], ad))
             * _lin64(x, d["w3"], d["w3_lora"], ad))
        return [h, _lin64(h, d["w2"], d["w2_lora"], ad)]
    if kind == "block":
        return _block64(_f(d["x"]), d["b"], _f(d["cos"]), _f(d["sin"]), c["adapters"],
                        _f(d["temb"]) if c["modulated"] else None)
    if kind == "ops":
        keep = []
        y = _block64(_f(d["x"]), d["b"], _f(d["cos"]), _f(d["sin"]), c["adapters"],
                     gates=d["gates"], keep=keep)
        return keep + [y]
    if kind == "attention":
        w = c["heads"] * HD
        q = _f(d["qkv"])
        return _attn64(q[:, :w], q[:, w:2 * w], q[:, 2 * w:], c["heads"])
    if kind == "encoder":
        y = _lin64(_rms64(_f(d["x"]), _f(d["norm"]), 1e-6), d["w"]) + _f(d["b"])
        n = c["n_q"] + c["n_k"]
        t = y[:, :n * HD].reshape(c["M"], n, HD)
        gain = torch.cat((_f(d["nq"]).expand(c["n_q"], HD), _f(d["nk"]).expand(c["n_k"], HD)))
        t = _rms64(t, gain, 1e-6)
        a, b = t[..., :64], t[..., 64:]
        cs, sn = _f(d["cos"])[:, None], _f(d["sin"])[:, None]
        t = torch.cat((a * cs - b * sn, b * cs + a * sn), -1)
        return torch.cat((t.reshape(c["M"], n * HD), y[:, n * HD:]), 1)
    # the whole forward: timestep, embeddings, refiners, layers, final layer
    md, n, r = d["m"], c["gh"] * c["gw"], c["refiner"]
    ang = _angles(_positions(c["gh"], c["gw"], c["cap"]))
    cos, sin = ang.cos(), ang.sin()
    silu = torch.nn.functional.silu
    t = 1000.0 * (1.0 - float(np.float32(d["sigma"])))
    f = torch.exp(-math.log(10000.0) * torch.arange(128, device="cuda", dtype=torch.float64) / 128)
    tin = _f(torch.cat(((t * f).cos(), (t * f).sin())).float().to(torch.bfloat16))
    te = silu(_lin64(tin[None], md["time_1"]) + _f(md["time_1b"]))
    temb = (_lin64(te, md["time_2"]) + _f(md["time_2b"]))[0]
    img = _lin64(_f(d["lat"]), md["x_in"]) + _f(md["x_in_b"])
    cap = _lin64(_rms64(_f(d["cap"]), _f(md["cap_norm"]), EPS), md["cap_in"]) + _f(md["cap_in_b"])
    joint = None
    for i in range(2 * r + c["layers"]):
        b = _block_inputs(seed, "block%d/" % i, c["bits"], i >= r, c["adapters"])
        if i < r:
            cap = _block64(cap, b, cos[n:], sin[n:], c["adapters"])
        elif i < 2 * r:
            img = _block64(img, b, cos[:n], sin[:n], c["adapters"], temb)
        else:
            joint = torch.cat((img, cap)) if joint is None else joint
            joint = _block64(joint, b, cos, sin, c["adapters"], temb)
    x = (img if joint is None else joint)[:n]
    scale = (_lin64(silu(temb)[None], md["final_ada"]) + _f(md["final_ada_b"]))[0]
    x = torch.nn.functional.layer_norm(x, (HID,), eps=1e-6) * (1 + scale)
    return _lin64(x, md["final_lin"]) + _f(md["final_lin_b"])
