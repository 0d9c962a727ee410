"""The measured work of the decode path, as a user's program calls it.

Shapes are the three models the benchmark and the tests run -- MiniMind3-64M
(dim 768, FFN 2432, 8 query / 4 KV heads of 96), the LFM2.5-230M-shaped hybrid
(1024, 4608, 16 / 8 heads of 64) and the 0.5B Llama-shaped ternary body (1024,
4096, 16 / 2 heads of 64) -- over every weight format (q8, q4, t3), both KV
widths and every batch the engine forms: one token, a prompt of up to 512
positions, sequences in lockstep.

Outputs are integers on the q16 grid and every path must reproduce them bit
for bit (the integer sums are exact, the fp32 epilogues fixed), so the
tolerance is "exact" wherever a case returns integers.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "vc4-gles2-inference_amd"))

from vgx import gpu as vgpu  # noqa: E402
from vgx import mmcf, synth  # noqa: E402
from vgx.engine import Engine  # noqa: E402

EPS = 1e-5
MODELS = {
    "minimind3": dict(dim=768, hidden=2432, heads=8, kv_heads=4, qk_norm=1, theta=1e6),
    "lfm2": dict(dim=1024, hidden=4608, heads=16, kv_heads=8, qk_norm=1, theta=1e6),
    "bitcpm": dict(dim=1024, hidden=4096, heads=16, kv_heads=2, qk_norm=0, theta=10000.0),
}


def listed():
    return [
        # the smallest call: the norm and FFN gate of one decoded token (the 0.5B model's)
        dict(name="gate_t3", op="gate", kind="t3", rows=4096, cols=1024),
        # one layer's attention of one decoded token near the end of a 768-position q8 cache
        dict(name="attn_token_768", op="attn", model="minimind3", kv_bits=8, pos=767),
        # the final norm, LM head and greedy token of the hybrid's 64,402-row vocabulary
        dict(name="head_64402", op="head", rows=64402, cols=1024),
        # weights streamed from HBM: the benchmark's fp32-in, fp32-out sweep of
        # the LM-head shape over copies that exceed every cache
        dict(name="stream_q8", op="stream", kind="q8", rows=6400, cols=768, mb=512),
        # prompt processing, one layer: MiniMind3's q4 body and q8 cache at the
        # benchmark's 256-token prompt
        dict(name="prompt_q4_256", op="layer", model="minimind3", kind="q4", kv_bits=8, n=256, pos0=0),
        # the engine's largest prompt batch through an attention layer of the hybrid
        dict(name="prompt_q8_512", op="layer", model="lfm2", kind="q8", kv_bits=16, n=512, pos0=0),
        # a ragged prompt of the ternary body
        dict(name="prompt_t3_117", op="layer", model="bitcpm", kind="t3", kv_bits=16, n=117, pos0=0),
        # a short turn appended to a conversation: few rows, a long cached prefix
        dict(name="turn_q8_17", op="layer", model="minimind3", kind="q8", kv_bits=16, n=17, pos0=460),
        # a ragged prompt through a gated short-conv layer of the hybrid
        dict(name="conv_q8_200", op="conv", kind="q8", n=200),
        # one layer of 32 sequences decoding in lockstep (the 0.5B ternary model)
        dict(name="lockstep_t3_32", op="lockstep", model="bitcpm", kind="t3", kv_bits=16, n=32, pos=255),
        # a whole chat turn at the headline shape: MiniMind3 q8, 32 prompt + 64 greedy
        # tokens, then the logits of the position after them
        dict(name="chat_q8", op="engine", kind="q8", kv_bits=16, seq=256, prompt=32, gen=64),
        # a long prompt and a short answer: MiniMind3 q4 over the q8 cache, 256 + 16
        dict(name="chat_q4", op="engine", kind="q4", kv_bits=8, seq=768, prompt=256, gen=16),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["gate", "attn", "head", "stream", "layer", "layer", "layer", "layer", "conv", "lockstep",
                     "lockstep", "engine"])
    kind = rng.choice(["q8", "q4", "t3"])
    kv_bits = rng.choice([16, 8])
    model = rng.choice(sorted(MODELS))
    if op == "gate":
        return dict(op=op, kind=kind, rows=2 * _logint(rng, 512, 4096), cols=32 * _logint(rng, 16, 64))
    if op == "attn":
        return dict(op=op, model=model, kv_bits=kv_bits, pos=_logint(rng, 1, 768) - 1)
    if op == "head":
        return dict(op=op, rows=_logint(rng, 6400, 73448), cols=rng.choice([768, 1024]))
    if op == "stream":
        return dict(op=op, kind=kind, rows=_logint(rng, 384, 6400), cols=rng.choice([768, 1024, 2432]), mb=512)
    if op == "conv":
        return dict(op=op, kind=kind, n=_logint(rng, 2, 512))
    if op == "lockstep":
        return dict(op=op, model=model, kind=kind, kv_bits=kv_bits, n=_logint(rng, 2, 32), pos=rng.randrange(8, 384))
    if op == "engine":
        return dict(op=op, kind=rng.choice(["q8", "q4"]), kv_bits=kv_bits, seq=768, prompt=_logint(rng, 1, 400),
                    gen=_logint(rng, 2, 64))
    n = _logint(rng, 2, 512)
    return dict(op=op, model=model, kind=kind, kv_bits=kv_bits, n=n, pos0=rng.choice([0, rng.randrange(0, 769 - n)]))


# ---- inputs ------------------------------------------------------------------

_GPU = []


def _gpu():
    """The program's one context."""
    if not _GPU:
        _GPU.append(vgpu.GPU(0))
    return _GPU[0]


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _matrix(rng, kind, rows, cols, std=0.02):
    """(the packed matrix, its integer levels rows x cols, the value of one level: a row vector or a number).
    Projections are N(0, std) (ternary: per-row {0, +-s}), packed as a container holds them."""
    if kind == "t3":
        w = synth.ternary_matrix(rng, rows, cols)
        body, unit, plane = mmcf.t3mat(w)
        m = mmcf.Matrix("t3", rows, cols, np.frombuffer(body, np.uint8).copy(), unit, True, plane)
        return m, lambda: np.sign(w).astype(np.float64), _row_value(unit * 127.0, plane)
    w = rng.standard_normal((rows, cols), dtype=np.float32) * np.float32(std)
    if kind == "q8":
        q, unit, plane = mmcf.q8_per_row(w)
        m = mmcf.Matrix("q8", rows, cols, (q.view(np.uint8) ^ 0x80).ravel(), unit, True, plane)
        return m, lambda: q.astype(np.float64), _row_value(unit, plane)
    nib, s16, m16, ps, g = mmcf.q4mat(w)
    m = mmcf.Matrix("q4", rows, cols, nib.ravel(), ps, s16=s16.ravel(), m16=m16.ravel())

    def levels():
        n = np.stack([nib & 15, nib >> 4], axis=2).reshape(rows, g, 32).astype(np.float64)
        return (n * s16[:, :, None].astype(np.float64) + m16[:, :, None].astype(np.float64)).reshape(rows, cols)
    return m, levels, float(ps)


def _row_value(unit, plane):
    # the container's row scales travel as 16-bit fractions of the unit
    return np.clip(np.rint(plane.astype(np.float64) * 65536.0), 0, 65535) * float(unit) / 65536.0


def _act(rng, *shape):
    """q16 activations: N(0, 1) hidden states on the 1/256 grid."""
    v = rng.standard_normal(shape, dtype=np.float32) * np.float32(256.0)
    return np.clip(np.rint(v), -32768, 32767).astype(np.int16)


def _norm_w(rng, n):
    return np.clip(np.rint(rng.uniform(0.5, 1.5, n) * 256.0), 1, 32767).astype(np.int16)


def _rope(theta, hd, seq):
    f = 1.0 / theta ** (np.arange(0, hd, 2, dtype=np.float64) / hd)
    a = np.arange(seq, dtype=np.float64)[:, None] * f[None, :]
    return np.cos(a).astype(np.float32), np.sin(a).astype(np.float32)


def _attention(g, cfg, kv_bits, seq, qn, kn, nseq=1):
    hd = cfg["dim"] // cfg["heads"]
    rc, rs = _rope(cfg["theta"], hd, seq)
    return g.attention(dim=cfg["dim"], heads=cfg["heads"], kv_heads=cfg["kv_heads"], head_dim=hd, seq=seq, layers=1,
                       kv_bits=kv_bits, rope_half=1, qk_norm=cfg["qk_norm"], rope_cos=rc, rope_sin=rs,
                       q_norm=qn, k_norm=kn, nseq=nseq)


def _layer_inputs(case, seed):
    """Everything a layer case draws, in one order, for prepare and exact alike."""
    rng = np.random.default_rng(seed)
    if case["op"] == "conv":
        cfg = MODELS["lfm2"]
    else:
        cfg = MODELS[case["model"]]
    D, H = cfg["dim"], cfg["hidden"]
    hd = D // cfg["heads"]
    qkv_rows = D + 2 * cfg["kv_heads"] * hd
    kind = case.get("kind", "q8")
    d = dict(cfg=cfg, hd=hd)
    if case["op"] == "conv":
        d["w_in"], d["w_out"] = _matrix(rng, kind, 3 * D, D), _matrix(rng, kind, D, D)
        d["taps"] = rng.standard_normal((1, D, 3), dtype=np.float32) * np.float32(0.3)
        d["norm"] = _norm_w(rng, D)
        d["x"] = _act(rng, case["n"], D)
        return d
    d["qn"] = rng.uniform(0.5, 1.5, (1, hd)).astype(np.float32) if cfg["qk_norm"] else None
    d["kn"] = rng.uniform(0.5, 1.5, (1, hd)).astype(np.float32) if cfg["qk_norm"] else None
    if case["op"] == "attn":
        d["hist"] = _act(rng, case["pos"], qkv_rows)
        d["qkv"] = _act(rng, qkv_rows)
        return d
    d["qkv"], d["wo"] = _matrix(rng, kind, qkv_rows, D), _matrix(rng, kind, D, D)
    d["w1"], d["w3"] = _matrix(rng, kind, H, D), _matrix(rng, kind, H, D)
    d["w2"] = _matrix(rng, kind, D, H)
    d["norm1"], d["norm2"], d["norm3"] = _norm_w(rng, D), _norm_w(rng, D), _norm_w(rng, D)
    d["x"] = _act(rng, case["n"], D)
    if case["op"] == "lockstep":
        d["hist"] = _act(rng, case["n"], case["pos"], qkv_rows)
    else:
        d["hist"] = _act(rng, case["pos0"], qkv_rows)
    return d


def _fill(att, hist):
    """Cached positions 0 .. len(hist)-1, as earlier turns left them."""
    if len(hist):
        att.block_batch(0, 0, _dev(hist))


def prepare(case, seed):
    g = _gpu()
    op = case["op"]
    s = dict(op=op, g=g)
    if op == "engine":
        spec = synth.minimind3_spec(case["seq"])
        blob = synth.container(spec, case["kind"], seed=seed)
        s["eng"] = Engine(blob, seq=case["seq"], kv_bits=case["kv_bits"])
        s["prompt"] = synth.prompt(case["prompt"], spec.vocab, seed=seed)
        s["gen"] = case["gen"]
        return s
    if op in ("gate", "head", "stream"):
        rng = np.random.default_rng(seed)
        rows, cols = case["rows"], case["cols"]
        if op == "gate":
            s["w1"], s["w3"] = (g.upload(_matrix(rng, case["kind"], rows, cols)[0]) for _ in range(2))
            s["w"], s["x"] = _dev(_norm_w(rng, cols)), _dev(_act(rng, cols))
            s["y"] = torch.empty(rows, dtype=torch.int16, device="cuda")
        elif op == "head":
            m = _matrix(rng, "q8", rows, cols)[0]
            s["m"] = g.group([g.upload(m.slice_rows(r, min(r + mmcf.LOGITS_GRID, rows)))
                              for r in range(0, rows, mmcf.LOGITS_GRID)])
            s["w"], s["x"] = _dev(_norm_w(rng, cols)), _dev(_act(rng, cols))
            s["y"] = torch.empty(rows, dtype=torch.int16, device="cuda")
            s["tok"] = torch.empty(1, dtype=torch.int32, device="cuda")
        else:
            first = g.upload(_matrix(rng, case["kind"], rows, cols)[0])
            n = _copies(case)
            s["m"] = g.group([first] + [g.clone(first) for _ in range(n - 1)])
            s["x"] = _dev(rng.standard_normal(cols, dtype=np.float32))
            s["y"] = torch.empty(rows * n, dtype=torch.float32, device="cuda")
        return s
    d = _layer_inputs(case, seed)
    cfg, D = d["cfg"], d["cfg"]["dim"]

    def buf(*shape):
        return torch.empty(shape, dtype=torch.int16, device="cuda")

    if op == "conv":
        n = case["n"]
        s["w_in"], s["w_out"] = g.upload(d["w_in"][0]), g.upload(d["w_out"][0])
        s["conv"] = g.conv(d["taps"])
        s["norm"], s["x"] = _dev(d["norm"]), _dev(d["x"])
        s["xn"], s["bcx"], s["y"], s["h"] = buf(n, D), buf(n, 3 * D), buf(n, D), buf(n, D)
        return s
    if op == "attn":
        s["att"] = _attention(g, cfg, case["kv_bits"], 768, d["qn"], d["kn"])
        _fill(s["att"], d["hist"])
        s["qkv"], s["pos"], s["out"] = _dev(d["qkv"]), case["pos"], buf(D)
        return s
    n = case["n"]
    for k in ("qkv", "wo", "w1", "w3", "w2"):
        s[k] = g.upload(d[k][0])
    for k in ("norm1", "norm2", "norm3", "x"):
        s[k] = _dev(d[k])
    s["split"] = (cfg["hidden"] + 1) // 2
    s["bq"], s["ba"], s["bx1"], s["bh"], s["by"] = (buf(n, s["qkv"].rows), buf(n, D), buf(n, D),
                                                    buf(n, cfg["hidden"]), buf(n, D))
    s["bn"] = buf(n, D)
    if op == "lockstep":
        s["pos"] = case["pos"]
        s["att"] = _attention(g, cfg, case["kv_bits"], 512, d["qn"], d["kn"], nseq=n)
        for q in range(n):
            _fill(s["att"].view(q), d["hist"][q])
    else:
        s["pos0"] = case["pos0"]
        s["att"] = _attention(g, cfg, case["kv_bits"], 768, d["qn"], d["kn"])
        _fill(s["att"], d["hist"])
    return s


# ---- one pass ----------------------------------------------------------------

def run(s):
    g, op = s["g"], s["op"]
    if op == "gate":
        return g.ffn_gate_rms(s["w1"], s["w3"], s["x"], s["w"], EPS, out=s["y"])
    if op == "stream":
        return s["m"].gemv_f32(s["x"], out=s["y"])
    if op == "head":
        return s["m"].logits_argmax_rms(s["x"], s["w"], EPS, s["y"], s["tok"])
    if op == "attn":
        return s["att"].block(0, s["pos"], s["qkv"], out=s["out"])
    if op == "engine":
        toks, _, _ = s["eng"].generate(s["prompt"], s["gen"])
        logits, nxt = s["eng"].step(toks[-1], len(s["prompt"]) + s["gen"] - 1)
        return toks, logits, nxt
    if op == "conv":
        s["conv"].reset()
        g.rmsnorm_batch(s["x"], s["norm"], EPS, out=s["xn"])
        g.gemm(s["w_in"], s["xn"], out=s["bcx"])
        s["conv"].step(0, s["bcx"], out=s["y"])
        g.gemm(s["w_out"], s["y"], s["x"], out=s["h"])
        return s["bcx"], s["y"], s["h"]
    if op == "lockstep":
        # the engine's lockstep layer: rows arrive normalised by the GEMM before
        g.rmsnorm_batch(s["x"], s["norm1"], EPS, out=s["bn"])
        g.gemm(s["qkv"], s["bn"], out=s["bq"])
        s["att"].block_seqs(0, s["pos"], s["bq"], out=s["ba"])
        x1, xn = g.gemm_norm(s["wo"], s["ba"], s["x"], s["norm2"], EPS)
        g.ffn_gate_batch(s["w1"], s["w3"], xn, out=s["bh"])
        h, hn = g.gemm_norm(s["w2"], s["bh"], x1, s["norm3"], EPS, split=s["split"])
        return s["bq"], s["ba"], x1, s["bh"], h, hn
    # a prompt's layer as the engine runs it: the norms inside the GEMMs up to 32 rows
    if s["x"].shape[0] <= 32:
        g.gemm_rms(s["qkv"], s["x"], s["norm1"], EPS, out=s["bq"])
    else:
        g.rmsnorm_batch(s["x"], s["norm1"], EPS, out=s["bn"])
        g.gemm(s["qkv"], s["bn"], out=s["bq"])
    s["att"].block_batch(0, s["pos0"], s["bq"], out=s["ba"])
    g.gemm(s["wo"], s["ba"], s["x"], out=s["bx1"])
    if s["x"].shape[0] <= 32:
        g.ffn_gate_batch_rms(s["w1"], s["w3"], s["bx1"], s["norm2"], EPS, out=s["bh"])
    else:
        g.rmsnorm_batch(s["bx1"], s["norm2"], EPS, out=s["bn"])
        g.ffn_gate_batch(s["w1"], s["w3"], s["bn"], out=s["bh"])
    g.gemm_add_split(s["w2"], s["split"], s["bh"], s["bx1"], out=s["by"])
    return s["bq"], s["ba"], s["bx1"], s["bh"], s["by"]


# ---- what a pass cannot do without ---------------------------------------------

def _wbytes(kind, rows, cols):
    if kind == "q8":
        return rows * cols + 4 * rows
    if kind == "q4":
        return rows * cols // 2 + 4 * rows * (cols // 32)
    return rows * cols // 4 + 4 * rows


def _copies(case):
    return max(2, -(-case["mb"] * (1 << 20) // _wbytes(case["kind"], case["rows"], case["cols"])))


def _layer_shapes(cfg):
    D, H = cfg["dim"], cfg["hidden"]
    kvd = cfg["kv_heads"] * (D // cfg["heads"])
    return [(D + 2 * kvd, D), (D, D), (H, D), (H, D), (D, H)], kvd


def work(case):
    op = case["op"]
    if op == "gate":
        r, c = case["rows"], case["cols"]
        return dict(bytes=2 * _wbytes(case["kind"], r, c) + 4 * c + 2 * r, flops=4 * r * c)
    if op == "head":
        r, c = case["rows"], case["cols"]
        return dict(bytes=_wbytes("q8", r, c) + 4 * c + 2 * r + 4, flops=2 * r * c)
    if op == "stream":
        r, c, n = case["rows"], case["cols"], _copies(case)
        return dict(bytes=n * (_wbytes(case["kind"], r, c) + 4 * r) + 4 * c, flops=2 * r * c * n)
    if op == "conv":
        D, n = MODELS["lfm2"]["dim"], case["n"]
        shapes = [(3 * D, D), (D, D)]
        b = sum(_wbytes(case["kind"], r, c) for r, c in shapes) + 2 * n * D * 6
        return dict(bytes=b, flops=sum(2 * n * r * c for r, c in shapes))
    if op == "attn":
        cfg = MODELS[case["model"]]
        D = cfg["dim"]
        kvd = cfg["kv_heads"] * (D // cfg["heads"])
        ctx = case["pos"] + 1
        return dict(bytes=2 * kvd * ctx * case["kv_bits"] // 8 + 2 * (2 * D + 2 * kvd), flops=4 * D * ctx)
    if op == "engine":
        spec = synth.minimind3_spec(case["seq"])
        cfg = MODELS["minimind3"]
        shapes, kvd = _layer_shapes(cfg)
        body = spec.layers * sum(_wbytes(case["kind"], r, c) for r, c in shapes)
        head = _wbytes("q8", spec.vocab, spec.dim)
        params = spec.layers * sum(r * c for r, c in shapes)
        steps, total = case["gen"], case["prompt"] + case["gen"]
        kv = spec.layers * 2 * kvd * case["kv_bits"] // 8
        # the prompt pass, then `gen` single-token passes (the last for its logits)
        b = body * (1 + steps) + head * (1 + steps) + kv * (total + sum(range(case["prompt"], total)))
        att = 4 * spec.dim * spec.layers * total * (total + 1) // 2
        return dict(bytes=b, flops=2 * params * total + 2 * spec.vocab * spec.dim * (1 + steps) + att)
    cfg = MODELS[case["model"]]
    shapes, kvd = _layer_shapes(cfg)
    n, D = case["n"], cfg["dim"]
    b = sum(_wbytes(case["kind"], r, c) for r, c in shapes) + 2 * n * 2 * D
    f = sum(2 * n * r * c for r, c in shapes)
    kv = 2 * kvd * case["kv_bits"] // 8
    if op == "lockstep":
        b += n * kv * (case["pos"] + 1)
        f += 4 * D * n * (case["pos"] + 1)
    else:
        b += kv * (case["pos0"] + n)
        f += 4 * D * (n * case["pos0"] + n * (n + 1) // 2)
    return dict(bytes=b, flops=f)


def tolerance(case):
    if case["op"] == "stream":
        # an exact integer times one fp32 scale, rounded twice: 2^-23 relative an element
        return dict(rel=5e-7)
    return "exact"


# ---- the same numbers in 64 bits ------------------------------------------------

def _r16(v):
    return torch.clamp(torch.floor(v + 0.5), -32768, 32767)


def _t64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(torch.float64)


def _lin(w, x):
    """Row values (q16 units) of rows x: the exact integer sums times the row value."""
    _, levels, value = w
    v = x @ _t64(levels()).T
    return v * (_t64(value) if isinstance(value, np.ndarray) else value)


def _norm(x, w):
    n = x.shape[-1]
    per = -(-n // 32)
    sq = torch.nn.functional.pad(x * x, (0, 32 * per - n)).reshape(*x.shape[:-1], 32, per).sum(-1)
    ss = torch.floor(sq / 16.0 + 0.5).sum(-1, keepdim=True) / 4096.0
    return _r16(x / torch.sqrt(ss / n + EPS) * (_t64(w) / 256.0))


def _gate(v1, v3):
    a, u = _r16(v1) / 256.0, _r16(v3) / 256.0
    return _r16(a / (1.0 + torch.exp(-a)) * u * 256.0)


def _rot(x, pos, cfg, hd, nw, query):
    """Head vectors (..., hd) in units of 1: q/k norm, then the rotation at `pos` (per row)."""
    if cfg["qk_norm"]:
        r = 1.0 / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)
        if query:
            r = torch.floor(torch.clamp(r, max=127.0) * 65536.0 + 0.5) / 65536.0
        x = x * r * torch.round(_t64(nw[0]) * 256.0) / 256.0
    rc, rs = _rope(cfg["theta"], hd, 768)
    c = (torch.round(_t64(rc) * 4096.0) / 4096.0)[pos][:, None, :]
    s = (torch.round(_t64(rs) * 4096.0) / 4096.0)[pos][:, None, :]
    a, b = x[..., :hd // 2], x[..., hd // 2:]
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _attend(qkv, pos0, nq, cfg, hd, kv_bits, d):
    """The last nq rows of qkv (positions 0..) attend to their prefixes: q16 rows."""
    D, kvh = cfg["dim"], cfg["kv_heads"]
    grp = cfg["heads"] // kvh
    n = qkv.shape[0]
    pos = torch.arange(n)
    x = qkv / 256.0
    grid, lim = (2048.0, 32768) if kv_bits == 16 else (16.0, 128)

    def kvq(v):
        return torch.clamp(torch.floor(v * grid + 0.5), -lim, lim - 1) / grid

    k = kvq(_rot(x[:, D:D + kvh * hd].reshape(n, kvh, hd), pos, cfg, hd, d["kn"], False))
    v = kvq(x[:, D + kvh * hd:].reshape(n, kvh, hd))
    q = _r16(_rot(x[n - nq:, :D].reshape(nq, kvh * grp, hd), pos[n - nq:], cfg, hd, d["qn"], True) * 256.0) / 256.0
    out = torch.empty(nq, kvh * grp, hd, dtype=torch.float64)
    mask = torch.arange(n)[None, :] > pos[n - nq:][:, None]
    for h in range(kvh * grp):
        sc = _r16(q[:, h] @ k[:, h // grp].T / math.sqrt(hd) * 1024.0) / 1024.0
        sc = sc.masked_fill(mask, -math.inf)
        e = torch.exp(sc - sc.max(-1, keepdim=True).values)
        den = torch.clamp(torch.floor(e.sum(-1, keepdim=True) * 32.0 + 0.5), -32768, 32767) / 32.0
        out[:, h] = (e / den) @ v[:, h // grp]
    return _r16(out.reshape(nq, D) * 256.0)


def exact(case, seed):
    op = case["op"]
    if op == "engine":
        return None
    if op in ("gate", "head", "stream"):
        rng = np.random.default_rng(seed)
        rows, cols = case["rows"], case["cols"]
        if op == "gate":
            w1, w3 = _matrix(rng, case["kind"], rows, cols), _matrix(rng, case["kind"], rows, cols)
            nw, x = _norm_w(rng, cols), _t64(_act(rng, cols))
            xn = _norm(x[None], nw)
            return _gate(_lin(w1, xn), _lin(w3, xn))[0]
        if op == "head":
            w = _matrix(rng, "q8", rows, cols)
            nw, x = _norm_w(rng, cols), _t64(_act(rng, cols))
            y = _r16(_lin(w, _norm(x[None], nw))[0])
            return y, torch.argmax(y).reshape(1)
        w = _matrix(rng, case["kind"], rows, cols)
        x = _t64(rng.standard_normal(cols, dtype=np.float32))
        xq = torch.clamp(torch.round(x * 256.0), -32768, 32767)
        return (_lin(w, xq[None])[0] / 256.0).repeat(_copies(case))
    d = _layer_inputs(case, seed)
    cfg, hd = d["cfg"], d["hd"]
    if op == "conv":
        x = _t64(d["x"])
        D = cfg["dim"]
        bcx = _r16(_lin(d["w_in"], _norm(x, d["norm"])))
        taps = torch.clamp(torch.round(_t64(d["taps"][0]) * 256.0), -32768, 32767)
        gt = _r16(bcx[:, :D] * bcx[:, 2 * D:] / 256.0)
        p = torch.nn.functional.pad(gt, (0, 0, 2, 0))
        cv = _r16((taps[:, 0] * p[:-2] + taps[:, 1] * p[1:-1] + taps[:, 2] * gt) / 256.0)
        y = _r16(bcx[:, D:2 * D] * cv / 256.0)
        return bcx, y, _r16(_lin(d["w_out"], y) + x)
    if op == "attn":
        qkv = _t64(np.concatenate([d["hist"], d["qkv"][None]]))
        return _attend(qkv, case["pos"], 1, cfg, hd, case["kv_bits"], d)[0]
    x = _t64(d["x"])
    qkv = _r16(_lin(d["qkv"], _norm(x, d["norm1"])))
    if op == "lockstep":
        att = torch.cat([_attend(torch.cat([_t64(d["hist"][q]), qkv[q:q + 1]]), case["pos"], 1, cfg, hd,
                                 case["kv_bits"], d) for q in range(case["n"])])
    else:
        att = _attend(torch.cat([_t64(d["hist"]), qkv]), case["pos0"], case["n"], cfg, hd, case["kv_bits"], d)
    x1 = _r16(_lin(d["wo"], att) + x)
    xn = _norm(x1, d["norm2"])
    hid = _gate(_lin(d["w1"], xn), _lin(d["w3"], xn))
    m, levels, value = d["w2"]
    lv, sp = _t64(levels()), (cfg["hidden"] + 1) // 2
    val = _t64(value) if isinstance(value, np.ndarray) else value
    h = _r16(hid[:, sp:] @ lv[:, sp:].T * val + _r16(hid[:, :sp] @ lv[:, :sp].T * val + x1))
    if op == "lockstep":
        return qkv, att, x1, hid, h, _norm(h, d["norm3"])
    return qkv, att, x1, hid, h
