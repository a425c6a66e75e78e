"""The work whose speed this framework is measured by, through its public entry points.

Single kernels (lokal_amd.kernels) run on device buffers that the caller owns;
here those are torch tensors on the null stream.  The engine calls (Session,
Batcher) take host ids and hand host logits back, as a serving program uses
them.  Shapes are those of the three model families in lokal_amd/config.py:
SmolLM2-135M (F16), Qwen2.5-0.5B (Q8_0) and TinyLlama-1.1B (Q4_K, and the
Q4_K / Q6_K mix of *_K_M files); draw() also takes widths between them.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from lokal_amd import BatchRow, Engine, config, kernels, synth

TYPES = {"f16": synth.F16, "q8_0": synth.Q8_0, "q4_k": synth.Q4_K, "q6_k": synth.Q6_K}
FAMILIES = {"smollm2": (config.SMOLLM2_135M, "f16"), "qwen": (config.QWEN25_05B, "q8_0"),
            "tinyllama": (config.TINYLLAMA_11B, "q4_k"), "tinyllama_km": (config.TINYLLAMA_11B, "mix")}
MAX_SEQ = 1024  # positions of a session or a Batcher slot here


def listed():
    return [
        # What a decode step of 8 rows does besides its matrices: embedding rows, norm, RoPE, SwiGLU,
        # called one by one.  The smallest work there is; launches are all of it.
        {"name": "elementwise-qwen-8", "op": "elementwise", "family": "qwen", "n": 8},
        # One token through the Q6_K down matrix of a *_K_M file: mixed models decode matrix by matrix.
        {"name": "matvec-q6k-2048x5632", "op": "matvec", "type": "q6_k", "rows": 2048, "cols": 5632},
        # The gate matrix of the smallest family for a batch of 16 sequences.
        {"name": "matmul-f16-1536x576-16", "op": "matmul", "type": "f16", "rows": 1536, "cols": 576, "n": 16,
         "bias": False},
        # The gate matrix over a whole 512-token prefill chunk.
        {"name": "matmul-q8-4864x896-512", "op": "matmul", "type": "q8_0", "rows": 4864, "cols": 896, "n": 512,
         "bias": False},
        # The down matrix over a ragged prompt, deep in K.
        {"name": "matmul-q4k-2048x5632-203", "op": "matmul", "type": "q4_k", "rows": 2048, "cols": 5632, "n": 203,
         "bias": False},
        # A matrix of a *_K_M file's Q6_K share over a 256-token prompt.
        {"name": "matmul-q6k-5632x2048-256", "op": "matmul", "type": "q6_k", "rows": 5632, "cols": 2048, "n": 256,
         "bias": False},
        # The lm_head of a full Batcher step.
        {"name": "matmul-q8-151936x896-64", "op": "matmul", "type": "q8_0", "rows": 151936, "cols": 896, "n": 64,
         "bias": False},
        # Decode attention of a few long conversations, of different lengths.
        {"name": "attn-4x32768", "op": "attn", "n_seq": 4, "heads": 14, "kv_heads": 2, "max_seq": 32768},
        # Decode attention of a serving batch with short contexts.
        {"name": "attn-40x1000", "op": "attn", "n_seq": 40, "heads": 32, "kv_heads": 4, "max_seq": 1000},
        # One decode step of a batch of 24 sequences through a block of 4 layers and the lm_head.
        {"name": "batch-tinyllama-4l-24", "op": "batch", "family": "tinyllama", "layers": 4, "n": 24},
        # Whole calls: one token of one conversation, and a prompt.
        {"name": "forward-qwen-700", "op": "forward", "family": "qwen", "layers": 24, "pos": 700},
        {"name": "prefill-qwen-512", "op": "prefill", "family": "qwen", "layers": 24, "n": 512},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["elementwise", "matvec", "matmul", "matmul", "matmul", "attn", "attn", "batch", "forward",
                     "prefill"])
    family = rng.choice(sorted(FAMILIES))
    if op == "elementwise":
        return {"op": op, "family": family, "n": _log(rng, 1, 64)}
    if op in ("matvec", "matmul"):
        t = rng.choice(sorted(TYPES))
        cols = 256 * rng.randint(1, 22) if t in ("q4_k", "q6_k") else 32 * rng.randint(8, 176)
        most = 30_000_000 // cols
        c = {"op": op, "type": t, "rows": _log(rng, 64 if op == "matmul" else 2_000_000 // cols, most), "cols": cols}
        if op == "matmul":
            # at most about the flops and the outputs of the listed matrices
            c["n"] = max(2, min(_log(rng, 2, 512), 8_000_000_000 // (2 * c["rows"] * cols), 8_000_000 // c["rows"]))
            c["bias"] = rng.random() < 0.3
        return c
    if op == "attn":
        heads, kv = rng.choice([(9, 3), (14, 2), (32, 4)])
        max_seq = _log(rng, 64, 32768)
        return {"op": op, "n_seq": max(1, min(_log(rng, 1, 64), 262144 // (kv * max_seq))), "heads": heads,
                "kv_heads": kv, "max_seq": max_seq}
    layers = rng.randint(1, 4)
    if op == "batch":
        return {"op": op, "family": family, "layers": layers, "n": _log(rng, 1, 64)}
    if op == "forward":
        return {"op": op, "family": family, "layers": layers, "pos": _log(rng, 1, 1000)}
    return {"op": op, "family": family, "layers": layers, "n": _log(rng, 1, 512)}


# ------------------------------------------------------------------ inputs

class _Dev:
    """A torch tensor as the device buffer the kernel-level calls take."""

    def __init__(self, t):
        self.t = t
        self.ptr = ctypes.c_void_p(t.data_ptr())


class _Gen:
    """Seeded inputs, made on the GPU."""

    def __init__(self, seed, tag=0):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) * 1009 + tag)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.g, device="cuda")

    def whole(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda")

    def uniform(self, lo, hi, *shape):
        return torch.rand(shape, generator=self.g, device="cuda") * (hi - lo) + lo

    def activations(self, n, cols):
        """What a norm or a SwiGLU hands to a matrix: about unit scale, with a few large channels."""
        x = self.normal(n, cols)
        big = self.whole(0, cols, max(1, cols // 128))
        x[:, big] *= 12.0
        return x

    def weight(self, name, t, rows, cols):
        """GGUF bytes of a rows x cols matrix (on the GPU, flat uint8), its values of about 0.02."""
        nb = rows * cols // synth.BLK[t][0]
        if t == synth.F16:
            return (self.normal(rows * cols) * 0.02).half().view(torch.uint8)
        b = torch.randint(0, 256, (nb, synth.BLK[t][1]), generator=self.g, device="cuda", dtype=torch.uint8)
        if t == synth.Q8_0:
            b[:, 0:2] = (self.normal(nb).abs() * 0.0003).half().view(torch.uint8).view(nb, 2)
        elif t == synth.Q4_K:
            d = self.uniform(5e-5, 2e-4, nb)  # the mins offset the nibbles' mean, so the values' mean is 0
            b[:, 0:2], b[:, 2:4] = (v.half().view(torch.uint8).view(nb, 2) for v in (d, 7.5 * d))
        else:  # Q6_K: signed 8-bit sub-block scales
            b[:, 208:210] = self.uniform(1e-5, 3e-5, nb).half().view(torch.uint8).view(nb, 2)
        return b.view(-1)


def _tensors(case, seed):
    """[(name, GGUF type, dims, bytes on the GPU)] of the case's model."""
    cfg, kind = FAMILIES[case["family"]]
    cfg = cfg.with_(num_hidden_layers=case["layers"])
    base = synth.Q4_K if kind == "mix" else TYPES[kind]
    mix = synth.k_mix(synth.Q4_K, cfg) if kind == "mix" else lambda layer, proj: base
    g = _Gen(seed, 1)
    h, inter, kvd, qd = cfg.hidden_size, cfg.intermediate_size, cfg.kv_dim(), cfg.q_dim()
    out = []

    def vec(name, n, mean, std):
        out.append((name, synth.F32, (n,), (g.normal(n) * std + mean).view(torch.uint8)))

    def mat(name, t, rows, cols):
        out.append((name, t, (rows, cols), g.weight(name, t, rows, cols)))
    for i in range(cfg.num_hidden_layers):
        p = f"model.layers.{i}."
        vec(p + "input_layernorm.weight", h, 1.0, 0.1)
        vec(p + "post_attention_layernorm.weight", h, 1.0, 0.1)
        for proj, rows, cols in (("q_proj", qd, h), ("k_proj", kvd, h), ("v_proj", kvd, h), ("o_proj", h, qd)):
            mat(p + f"self_attn.{proj}.weight", mix(i, proj), rows, cols)
            if case["family"] == "qwen" and proj != "o_proj":
                vec(p + f"self_attn.{proj}.bias", rows, 0.0, 0.02)
        for proj, rows, cols in (("gate_proj", inter, h), ("up_proj", inter, h), ("down_proj", h, inter)):
            mat(p + f"mlp.{proj}.weight", mix(i, proj), rows, cols)
    mat("model.embed_tokens.weight", base, cfg.vocab_size, h)
    vec("model.norm.weight", h, 1.0, 0.1)
    if kind in ("q4_k", "mix"):
        mat("lm_head.weight", mix(None, "lm_head"), cfg.vocab_size, h)
    return cfg, out


def _tokens(case, seed, cfg):
    """The prompts: one list of ids per sequence, the last id being the one a decode step feeds."""
    rng = np.random.default_rng(int(seed) + 7)
    if case["op"] == "prefill":
        lengths = [case["n"]]
    elif case["op"] == "forward":
        lengths = [case["pos"] + 1]
    else:
        lengths = [int(v) for v in rng.integers(2, 601, case["n"])]
    return [rng.integers(0, cfg.vocab_size, m).astype(np.uint32) for m in lengths]


def _inputs(case, seed):
    """The tensors of a single-kernel case, by name."""
    g = _Gen(seed)
    op = case["op"]
    if op == "elementwise":
        cfg, kind = FAMILIES[case["family"]]
        t = TYPES["q4_k" if kind == "mix" else kind]
        n, h, inter = case["n"], cfg.hidden_size, cfg.intermediate_size
        return {"table": g.weight("", t, cfg.vocab_size, h), "ids": g.whole(0, cfg.vocab_size, n).int(),
                "gain": g.normal(h) * 0.1 + 1, "pos": g.whole(0, 4096, n).int(), "gate": g.normal(n, inter),
                "up": g.normal(n, inter)}
    if op == "attn":
        s, m, kv = case["n_seq"], case["max_seq"], case["kv_heads"]
        return {"q": g.normal(s, case["heads"] * 64) * 2, "k": g.normal(s, kv, m, 64).half(),
                "v": g.normal(s, kv, m, 64).half(), "ctx": g.whole(max(1, m // 4), m + 1, s).int()}
    n = case.get("n", 1)
    d = {"w": g.weight("", TYPES[case["type"]], case["rows"], case["cols"]), "x": g.activations(n, case["cols"])}
    if case.get("bias"):
        d["bias"] = g.normal(case["rows"]) * 0.1
    return d


class _State:
    """Keeps what a program holds between calls; frees the engine's buffers with it."""

    def __init__(self, **kw):
        self.__dict__.update(kw)

    def __del__(self):
        for name in ("session", "batcher", "engine"):
            h = self.__dict__.get(name)
            if h is not None:
                h.close()


def prepare(case, seed):
    op = case["op"]
    if op in ("forward", "prefill", "batch"):
        cfg, tensors = _tensors(case, seed)
        engine = Engine.from_tensors(cfg, [synth.Tensor(n, t, d, b.cpu().numpy()) for n, t, d, b in tensors])
        ids = _tokens(case, seed, cfg)
        if op == "batch":
            batcher = engine.batcher(len(ids), MAX_SEQ)
            for slot, p in enumerate(ids):
                batcher.prefill(slot, p[:-1])
            rows = [BatchRow(int(p[-1]), len(p) - 1, slot) for slot, p in enumerate(ids)]
            return _State(op=op, engine=engine, batcher=batcher, rows=rows)
        session = engine.session(MAX_SEQ)
        if op == "forward":
            session.prefill(ids[0][:-1])
        return _State(op=op, engine=engine, session=session, ids=ids[0])
    d = _inputs(case, seed)
    s = _State(op=op, case=case, t=d)
    if op == "elementwise":
        cfg, kind = FAMILIES[case["family"]]
        s.cfg = cfg
        s.w = kernels.Weight(TYPES["q4_k" if kind == "mix" else kind], cfg.vocab_size, cfg.hidden_size,
                             d["table"].cpu().numpy())
        s.out = [torch.empty(case["n"], cfg.hidden_size, device="cuda") for _ in range(2)]
        s.out.append(torch.empty(case["n"], cfg.intermediate_size, device="cuda"))
    elif op == "attn":
        s.out = [torch.empty_like(d["q"])]
    else:
        s.w = kernels.Weight(TYPES[case["type"]], case["rows"], case["cols"], d.pop("w").cpu().numpy())
        s.out = [torch.empty(case.get("n", 1), case["rows"], device="cuda")]
    s.dev = {k: _Dev(v) for k, v in d.items()}
    s.dout = [_Dev(v) for v in s.out]
    torch.cuda.synchronize()  # torch made the inputs; the handles above were uploaded by the framework
    return s


def run(s):
    op = s.op
    if op == "prefill":
        return s.session.prefill(s.ids)
    if op == "forward":
        return s.session.forward(int(s.ids[-1]), len(s.ids) - 1)
    if op == "batch":
        return s.batcher.decode_step(s.rows)
    c, d, o = s.case, s.dev, s.dout
    if op == "elementwise":
        n, h = c["n"], s.cfg.hidden_size
        kernels.embed_gather(s.w, d["ids"], n, o[0])
        kernels.rmsnorm(o[0], d["gain"], n, h, s.cfg.rms_norm_eps, o[1])
        kernels.rope_pairs(o[1], n, h, 64, d["pos"], s.cfg.rope_theta)
        kernels.swiglu(d["gate"], d["up"], n * s.cfg.intermediate_size, o[2])
    elif op == "attn":
        kernels.attn_decode(d["q"], d["k"], d["v"], d["ctx"], c["n_seq"], c["heads"], c["kv_heads"], 64,
                            c["max_seq"], o[0])
    elif op == "matvec":
        kernels.matvec(s.w, d["x"], o[0])
    else:
        kernels.matmul(s.w, d["x"], c["n"], o[0], bias=d.get("bias"))
    return s.out


# ------------------------------------------------------ what a pass has to do

def _model_work(case):
    """(weight bytes, weight values, embedding bytes of a row) of the layers, then of the lm_head."""
    cfg, kind = FAMILIES[case["family"]]
    cfg = cfg.with_(num_hidden_layers=case["layers"])
    mix = synth.k_mix(synth.Q4_K, cfg) if kind == "mix" else lambda layer, proj: TYPES[kind]
    h, inter, kvd, qd = cfg.hidden_size, cfg.intermediate_size, cfg.kv_dim(), cfg.q_dim()
    nbytes = values = 0
    for i in range(cfg.num_hidden_layers):
        for proj, rows, cols in (("q_proj", qd, h), ("k_proj", kvd, h), ("v_proj", kvd, h), ("o_proj", h, qd),
                                 ("gate_proj", inter, h), ("up_proj", inter, h), ("down_proj", h, inter)):
            nbytes += rows * synth.row_bytes(mix(i, proj), cols)
            values += rows * cols
    return cfg, nbytes, values, cfg.vocab_size * synth.row_bytes(mix(None, "lm_head"), h)


def work(case):
    op = case["op"]
    if op in ("forward", "prefill", "batch"):
        cfg, nbytes, values, head = _model_work(case)
        # the mean length of a drawn batch's sequences is 300
        rows, ctx = {"forward": (1, case.get("pos", 0) + 1), "prefill": (case.get("n"), (case.get("n", 0) + 1) / 2),
                     "batch": (case.get("n"), 300)}[op]
        heads = 1 if op != "batch" else case["n"]
        kv_rows = case["n"] if op == "prefill" else rows * ctx
        kv = kv_rows * 2 * cfg.kv_dim() * 2 * cfg.num_hidden_layers
        attn = 4 * rows * ctx * cfg.q_dim() * cfg.num_hidden_layers
        return {"bytes": nbytes + head + kv + heads * cfg.vocab_size * 4,
                "flops": 2 * values * rows + 2 * heads * cfg.vocab_size * cfg.hidden_size + attn}
    if op == "elementwise":
        cfg, kind = FAMILIES[case["family"]]
        row = synth.row_bytes(TYPES["q4_k" if kind == "mix" else kind], cfg.hidden_size)
        n, h, inter = case["n"], cfg.hidden_size, cfg.intermediate_size
        return {"bytes": n * (row + 12 * h + 12 * inter) + 4 * h, "flops": n * (12 * h + 6 * inter)}
    if op == "attn":
        ctx = case["n_seq"] * case["max_seq"] * 5 / 8
        return {"bytes": ctx * case["kv_heads"] * 256 + case["n_seq"] * case["heads"] * 512,
                "flops": ctx * case["heads"] * 256}
    n = case.get("n", 1)
    return {"bytes": case["rows"] * synth.row_bytes(TYPES[case["type"]], case["cols"])
            + 4 * n * (case["rows"] + case["cols"]), "flops": 2 * n * case["rows"] * case["cols"]}


def tolerance(case):
    if case["op"] in ("forward", "prefill", "batch"):
        # f32 sums, and an f16 K / V cache: a last-bit difference before it moves a cached value by 2^-11, which
        # weighs most after a short prompt.  Measured against 64 bits with K and V rounded so: 3e-5 for the
        # 24-layer calls, up to 3.7e-4 for a row of a batch
        return {"rel": 1.5e-3, "max": 0.03}
    # f32 sums; measured against 64 bits: up to 8e-7 (Q6_K, 5632 deep)
    return {"rel": 3e-6, "max": 1.2e-4}


# ----------------------------------------------------------- in 64 bits, plainly

def _f64(t, b, rows, cols):
    """GGUF bytes (on the GPU) as rows x cols doubles."""
    if t == synth.F32:
        return b.view(torch.float32).double()
    if t == synth.F16:
        return b.view(torch.float16).double().view(rows, cols)
    b = b.view(-1, synth.BLK[t][1])

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()
    if t == synth.Q8_0:
        return (half(0) * b[:, 2:].contiguous().view(torch.int8).double()).view(rows, cols)
    if t == synth.Q4_K:
        s = b[:, 4:16].int()
        lo, mid, hi = s[:, 0:4], s[:, 4:8], s[:, 8:12]
        sc = torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1).double()
        mn = torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1).double()
        q = b[:, 16:].view(-1, 4, 32)
        q = torch.stack([q & 15, q >> 4], 2).view(-1, 8, 32).double()
        return (half(0)[:, :, None] * sc[:, :, None] * q - half(2)[:, :, None] * mn[:, :, None]).view(rows, cols)
    # Q6_K: two halves of 128 values; 4 low bits in ql, 2 high bits in qh
    ql, qh = b[:, 0:128].int().view(-1, 2, 2, 32), b[:, 128:192].int().view(-1, 2, 32)
    q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                     (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | (((qh >> 6) & 3) << 4)], 2)
    sc = b[:, 192:208].contiguous().view(torch.int8).double()
    return (half(208)[:, :, None] * sc[:, :, None] * (q - 32).double().view(-1, 16, 16)).view(rows, cols)


def _rope64(x, pos, theta):
    """x [n, heads, 64] turned at positions pos."""
    f = theta ** (-torch.arange(0, 64, 2, device="cuda", dtype=torch.float64) / 64)
    a = pos.double()[:, None, None] * f
    u, v = x[..., :32], x[..., 32:]
    return torch.cat([u * a.cos() - v * a.sin(), u * a.sin() + v * a.cos()], -1)


def _norm64(x, w, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w


def _model64(cfg, tensors, prompts):
    """The last position's logits of each prompt."""
    w = {n: _f64(t, b, *(d if len(d) == 2 else (1, d[0]))) for n, t, d, b in tensors if not n.startswith("model.layers")}
    embed = w["model.embed_tokens.weight"]
    xs = [embed[torch.from_numpy(p.astype(np.int64)).cuda()] for p in prompts]
    nh, nkv, kvd = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.kv_dim()
    for i in range(cfg.num_hidden_layers):
        p = f"model.layers.{i}."
        lw = {n[len(p):]: _f64(t, b, *(d if len(d) == 2 else (1, d[0]))) for n, t, d, b in tensors if n.startswith(p)}
        for k, x in enumerate(xs):
            n = x.shape[0]
            y = _norm64(x, lw["input_layernorm.weight"], cfg.rms_norm_eps)
            q, kk, v = (y @ lw[f"self_attn.{m}.weight"].T + lw.get(f"self_attn.{m}.bias", 0.0)
                        for m in ("q_proj", "k_proj", "v_proj"))
            pos = torch.arange(n, device="cuda")
            q = _rope64(q.view(n, nh, 64), pos, cfg.rope_theta)
            kk, v = _rope64(kk.view(n, nkv, 64), pos, cfg.rope_theta), v.view(n, nkv, 64)
            kk, v = (t.repeat_interleave(nh // nkv, 1).transpose(0, 1).contiguous() for t in (kk, v))
            sc = torch.matmul(q.transpose(0, 1).contiguous(), kk.transpose(1, 2).contiguous()) / 8
            sc = sc.masked_fill(torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1), -torch.inf)
            a = torch.matmul(sc.softmax(-1), v).transpose(0, 1).reshape(n, nh * 64)
            x = x + a @ lw["self_attn.o_proj.weight"].T
            y = _norm64(x, lw["post_attention_layernorm.weight"], cfg.rms_norm_eps)
            g = y @ lw["mlp.gate_proj.weight"].T
            xs[k] = x + (g * torch.sigmoid(g) * (y @ lw["mlp.up_proj.weight"].T)) @ lw["mlp.down_proj.weight"].T
    last = _norm64(torch.stack([x[-1] for x in xs]), w["model.norm.weight"], cfg.rms_norm_eps)
    return last @ w.get("lm_head.weight", embed).T


def exact(case, seed):
    op = case["op"]
    if op in ("forward", "prefill", "batch"):
        cfg, tensors = _tensors(case, seed)
        out = _model64(cfg, tensors, _tokens(case, seed, cfg))
        return list(out) if op == "batch" else out[0]
    d = _inputs(case, seed)
    if op == "elementwise":
        cfg, kind = FAMILIES[case["family"]]
        table = _f64(TYPES["q4_k" if kind == "mix" else kind], d["table"], cfg.vocab_size, cfg.hidden_size)
        h = table[d["ids"].long()]
        x = _norm64(h, d["gain"].double(), cfg.rms_norm_eps)
        x = _rope64(x.view(case["n"], -1, 64), d["pos"], cfg.rope_theta).view(case["n"], -1)
        g = d["gate"].double()
        return [h, x, g * torch.sigmoid(g) * d["up"].double()]
    if op == "attn":
        out = torch.empty(d["q"].shape, dtype=torch.float64, device="cuda")
        kv = case["kv_heads"]
        for s, c in enumerate(d["ctx"].tolist()):
            q = d["q"][s].double().view(kv, -1, 64)
            p = torch.softmax(torch.matmul(q, d["k"][s, :, :c].double().transpose(1, 2).contiguous()) / 8, -1)
            out[s] = torch.matmul(p, d["v"][s, :, :c].double()).reshape(-1)
        return [out]
    y = d["x"].double() @ _f64(TYPES[case["type"]], d["w"], case["rows"], case["cols"]).T
    return [y + d["bias"].double() if case.get("bias") else y]
