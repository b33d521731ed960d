"""Performance cases of the framework, through its public entry points.

A case is a dict of plain values; `prepare` makes what a program holds before
the call (weights uploaded, an engine, inputs), `run` is one pass.  Kinds:

  generate  Engine.reset + Engine.generate (prompt and decode rounds) and the
            forward of the last token: one request of one sequence
  prefill   a prompt forwarded into an empty cache and the logits of its
            last tokens: what comes before every long-context answer
  batch     BatchEngine.generate_batch: many requests decoded together
  linear    pf_gemv_q: int8 activations x a block-quantized matrix, 1 row
            (decode), 2-8 (verify) and up to 512 (prompts, many sequences)
  int8      pf_matmul_quantized: fp32 activations x a plain int8 matrix
  unembed   pf_gemv_f32: hidden rows x the tied table
  heads     MTPHeads.forward: the draft heads with an fp32 tied table

Weights are N(0, 0.02^2), as the repository's models are; every matrix draws
its 32-element blocks (codes with their scale) from a quantized pool, which
keeps the values' distribution and makes a 1B model in seconds.
"""
import ctypes as C
import math

import numpy as np
import torch

import pocketforge_amd as pf

FMTS = {"q4": pf.FMT_Q4, "q2": pf.FMT_Q2, "q15": pf.FMT_Q15, "q8": pf.FMT_Q8}
# widths of the repository's models: (hidden, heads, head_dim, ff)
WIDTHS = {256: (256, 4, 64, 512), 768: (768, 12, 64, 2048), 2048: (2048, 16, 128, 5632)}
SAMPLERS = {"greedy": (0.8, 0.95, 40, 1), "top_p": (0.8, 0.95, 40, 0), "temperature": (0.8, 1.0, 0, 0)}
POOL_BLOCKS = 32768
N_MTP = 4
TAIL = 8   # last prompt tokens of a prefill case, forwarded with outputs

_ctx = []


def _context():
    """One context per process, as the library's programs keep it."""
    if not _ctx:
        _ctx.append(pf.Context(0))
    return _ctx[0]


def listed():
    return [
        # the smallest call: a two-layer model, where launches and host time are all there is
        dict(name="tiny_generate", kind="generate", width=256, layers=2, vocab=1024, fmts="q4", prompt=16, new=24,
             window=64, pool=6, sampler="greedy"),
        # a 150M assistant: short prompt, greedy, drafts partly accepted
        dict(name="small_generate", kind="generate", width=768, layers=12, vocab=16384, fmts="q4", prompt=64, new=128,
             window=8192, pool=64, sampler="greedy"),
        # 1B-width layers in the mixed formats (attention Q4, gate/up Q2, down Q1.5), top-p
        # sampling, and a prompt longer than the window: eviction and pooled rows
        dict(name="mixed_generate", kind="generate", width=2048, layers=4, vocab=16384, fmts="mixed", prompt=700,
             new=64, window=512, pool=16, sampler="top_p"),
        # the headline model whole: 24 layers, 2048-token prompt, greedy decode
        dict(name="one_b_generate", kind="generate", width=2048, layers=24, vocab=16384, fmts="q4", prompt=2048,
             new=64, window=8192, pool=64, sampler="greedy"),
        # two of its layers over a long prompt of ragged length
        dict(name="long_prefill", kind="prefill", width=2048, layers=2, vocab=16384, fmts="q4", prompt=6000,
             window=8192, pool=64),
        # a serving batch: 64 requests of different lengths through two of its layers
        dict(name="batch_generate", kind="batch", width=2048, layers=2, vocab=16384, fmts="q4", seqs=64, prompt=768,
             new=24, window=8192, pool=64, sampler="greedy"),
        # the gate|up product of one decode row
        dict(name="linear_decode", kind="linear", m=1, rows=11264, cols=2048, fmt="q4"),
        # the down product of a five-row verify pass, in the .squeeze default format
        dict(name="linear_verify", kind="linear", m=5, rows=2048, cols=5632, fmt="q8"),
        # the QKV product of a prompt pass
        dict(name="linear_prefill", kind="linear", m=256, rows=6144, cols=2048, fmt="q4"),
        # the plain int8 matmul API, ragged in every dimension
        dict(name="int8_matmul", kind="int8", m=100, n=3000, k=1100, given=False),
        # the tied unembedding of a verify pass
        dict(name="unembed_verify", kind="unembed", m=5, vocab=16384, cols=2048, fmt="q4"),
        # four draft heads of the 1B model with an fp32 tied table
        dict(name="draft_heads", kind="heads", heads=4, cols=2048, vocab=16384),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["generate", "generate", "prefill", "prefill", "batch", "linear", "linear", "linear", "int8",
                       "int8", "unembed", "heads"])
    if kind in ("generate", "prefill", "batch"):
        width = rng.choice([256, 768, 2048])
        case = dict(kind=kind, width=width, layers=rng.randint(1, 2 if kind == "batch" else 4),
                    vocab=64 * rng.randint(16, 256), fmts=rng.choice(["q4", "q4", "mixed"]))
        if kind == "generate":
            case.update(prompt=_log(rng, 8, 1500), new=_log(rng, 8, 64), window=rng.choice([64, 500, 8192]),
                        pool=rng.choice([6, 16, 64]), sampler=rng.choice(["greedy", "top_p", "temperature"]))
        elif kind == "prefill":
            case.update(layers=rng.randint(1, 2), prompt=_log(rng, 64, 6000), window=8192, pool=64)
        else:
            case.update(seqs=_log(rng, 3, 64), prompt=_log(rng, 64, 768), new=_log(rng, 8, 24), window=8192, pool=64,
                        sampler=rng.choice(["greedy", "top_p"]))
        return case
    if kind == "linear":
        return dict(kind=kind, m=_log(rng, 1, 512), rows=64 * _log(rng, 4, 176), cols=256 * rng.randint(1, 22),
                    fmt=rng.choice(["q4", "q4", "q2", "q15", "q8"]))
    if kind == "int8":
        return dict(kind=kind, m=_log(rng, 1, 256), n=_log(rng, 16, 4096), k=_log(rng, 32, 4096),
                    given=rng.random() < 0.5)
    if kind == "unembed":
        return dict(kind=kind, m=rng.randint(1, 8), vocab=64 * _log(rng, 16, 256), cols=256 * rng.randint(1, 8),
                    fmt=rng.choice(["q4", "q8"]))
    return dict(kind=kind, heads=rng.randint(1, 4), cols=256 * rng.randint(1, 8), vocab=_log(rng, 512, 16384))


# ---------------------------------------------------------------- weights

class _Blocks:
    """Quantized N(0, 0.02^2) blocks per format, and matrices drawn from them."""

    def __init__(self, seed):
        self.seed, self.rng, self.pools = seed, np.random.default_rng(seed), {}

    def matrix(self, rows, cols, fmt):
        if fmt not in self.pools:
            c, s = pf.gen_matrix(self.seed + 1, fmt, 0.02, POOL_BLOCKS // 32, 1024, fmt)
            self.pools[fmt] = c.reshape(POOL_BLOCKS, -1).view(np.dtype((np.void, c.shape[-1]))).reshape(-1), s.reshape(-1)
        pc, ps = self.pools[fmt]
        at = self.rng.integers(0, POOL_BLOCKS, (rows, cols // 32), dtype=np.int32)
        return fmt, np.ascontiguousarray(pc[at]).view(np.uint8).reshape(rows, cols // 32, -1), ps[at]


def _model_cfg(case):
    d, heads, hd, ff = WIDTHS[case["width"]]
    return dict(n_layers=case["layers"], n_embd=d, n_heads=heads, head_dim=hd, n_ff=ff, n_vocab=case["vocab"],
                n_mtp=N_MTP)


def _model_weights(case, seed):
    cfg, blocks = _model_cfg(case), _Blocks(seed)
    mixed = case["fmts"] == "mixed"
    gate, down = (pf.FMT_Q2, pf.FMT_Q15) if mixed else (pf.FMT_Q4, pf.FMT_Q4)
    d, ff = cfg["n_embd"], cfg["n_ff"]
    layers = []
    for _ in range(cfg["n_layers"]):
        lw = {n: blocks.matrix(d, d, pf.FMT_Q4) for n in ("wq", "wk", "wv", "wo")}
        lw.update(wgate=blocks.matrix(ff, d, gate), wup=blocks.matrix(ff, d, gate), wdown=blocks.matrix(d, ff, down))
        layers.append(lw)
    ones = np.ones((cfg["n_layers"], d), np.float32)
    return dict(layers=layers, emb=blocks.matrix(cfg["n_vocab"], d, pf.FMT_Q4),
                mtp=[{n: blocks.matrix(d, d, pf.FMT_Q4) for n in ("gate", "up", "down")} for _ in range(N_MTP)],
                attn_norm=ones, ffn_norm=ones)


def _tokens(case, seed):
    """The prompt (batch: one per sequence, of 1/8 to all of `prompt` tokens)."""
    rng = np.random.default_rng(seed + 77)
    if case["kind"] == "batch":
        lens = rng.integers(max(1, case["prompt"] // 8), case["prompt"] + 1, case["seqs"])
        return [rng.integers(0, case["vocab"], n, dtype=np.int32) for n in lens]
    return rng.integers(0, case["vocab"], case["prompt"], dtype=np.int32)


def _activations(seed, rows, cols):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(rows, cols, generator=g, dtype=torch.float32)


def _int8_inputs(case, seed):
    a = _activations(seed, case["m"], case["k"])
    g = torch.Generator().manual_seed(seed + 1)
    b = torch.randint(-127, 128, (case["n"], case["k"]), generator=g, dtype=torch.int8)
    ws = torch.rand(case["n"], generator=g) * 0.02 + 0.001
    # given scales: the caller's own calibration, which covers the rows' range
    act = a.abs().amax(1) / 120.0 if case["given"] else None
    return a, b, ws, act


def _dequantized(w):
    """A matrix of interchange codes as float64 values."""
    fmt, codes, scales = w
    c = torch.from_numpy(codes).cuda()
    if fmt == pf.FMT_Q8:
        v = c.view(torch.int8).double()
    elif fmt == pf.FMT_Q4:
        v = torch.stack([c & 15, c >> 4], -1).flatten(-2).double() - 8
    else:
        v = torch.stack([(c >> s) & 3 for s in (0, 2, 4, 6)], -1).flatten(-2).double() - (2 if fmt == pf.FMT_Q2 else 1)
    s = torch.from_numpy(scales.view(np.float16).astype(np.float64)).cuda()
    return (v * s[..., None]).flatten(-2)


# ------------------------------------------------------- prepare and run

def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    state = dict(kind=kind, ctx=ctx)
    if kind in ("generate", "prefill", "batch"):
        cfg = _model_cfg(case)
        model = pf.Model(ctx, cfg, _model_weights(case, seed))
        kv = dict(sink_size=4, window_size=case["window"], pool_block=case["pool"],
                  max_context=case["prompt"] + case.get("new", TAIL) + 64)
        state.update(model=model, prompt=_tokens(case, seed))
        if kind == "generate":
            state.update(eng=pf.Engine(model, **kv))
        else:
            state.update(eng=pf.BatchEngine(model, case.get("seqs", 1), **kv))
        if "sampler" in case:
            state.update(new=case["new"], cap=case["prompt"] + case["new"] + 8, sampling=pf.Sampling(*SAMPLERS[case["sampler"]]),
                         seeds=np.arange(case.get("seqs", 1), dtype=np.uint64) + 7)
    elif kind == "linear":
        fmt, codes, scales = _Blocks(seed).matrix(case["rows"], case["cols"], FMTS[case["fmt"]])
        state.update(m=case["m"], w=ctx.upload_matrix(fmt, codes, scales),
                     x=_activations(seed, case["m"], case["cols"]).cuda(),
                     y=torch.empty(case["m"], case["rows"], device="cuda"))
    elif kind == "unembed":
        fmt, codes, scales = _Blocks(seed).matrix(case["vocab"], case["cols"], FMTS[case["fmt"]])
        state.update(m=case["m"], w=ctx.upload_matrix(fmt, codes, scales, rowmajor=True),
                     x=_activations(seed, case["m"], case["cols"]).cuda(),
                     y=torch.empty(case["m"], case["vocab"], device="cuda"))
    elif kind == "int8":
        a, b, ws, act = _int8_inputs(case, seed)
        state.update(shape=(case["m"], case["n"], case["k"]), a=a.cuda(), b=b.cuda(), ws=ws.cuda(),
                     act=None if act is None else act.cuda(), y=torch.empty(case["m"], case["n"], device="cuda"))
    else:
        heads = pf.MTPHeads(ctx, case["heads"], case["cols"], case["vocab"])
        ws, table = _heads_weights(case, seed)
        for k, hw in enumerate(ws):
            for which, (_, codes, scales) in enumerate(hw):
                heads.set_head(k, which, codes, scales)
        heads.set_table(table)
        state.update(heads=heads, hidden=_activations(seed, 1, case["cols"]).numpy()[0])
    torch.cuda.synchronize()
    return state


def _heads_weights(case, seed):
    blocks = _Blocks(seed)
    ws = [[blocks.matrix(case["cols"], case["cols"], pf.FMT_Q4) for _ in range(3)] for _ in range(case["heads"])]
    table = np.random.default_rng(seed + 5).standard_normal((case["vocab"], case["cols"]), dtype=np.float32)
    table *= np.float32(0.02)
    return ws, table


def _padded(tokens, cap):
    """Token rows of different lengths as one array, -1 past their ends."""
    out = np.full((len(tokens), cap), -1, np.int32)
    for row, t in zip(out, tokens):
        row[: len(t)] = t
    return out


def _ptr(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def run(state):
    kind = state["kind"]
    if kind == "generate":
        eng = state["eng"]
        eng.reset()
        tokens, res = eng.generate(state["prompt"], state["new"], state["sampling"], 7)
        logits, hidden = eng.forward(tokens[-1:])
        return dict(tokens=_padded([tokens], state["cap"]), accepted=res.mtp_accepted, rejected=res.mtp_rejected,
                    logits=logits, hidden=hidden)
    if kind == "prefill":
        eng, prompt = state["eng"], state["prompt"]
        eng.reset()
        eng.prefill_seq(0, prompt[:-TAIL])
        logits, hidden = eng.forward_batch([0], prompt[None, -TAIL:])
        return dict(logits=logits, hidden=hidden)
    if kind == "batch":
        eng = state["eng"]
        eng.reset()
        tokens, res = eng.generate_batch(state["prompt"], state["new"], state["sampling"], state["seeds"])
        logits, hidden = eng.forward_batch(np.arange(eng.n_seq), np.array([t[-1] for t in tokens])[:, None])
        return dict(tokens=_padded(tokens, state["cap"]), accepted=np.array([r.mtp_accepted for r in res]),
                    logits=logits, hidden=hidden)
    ctx, lib = state["ctx"], pf.lib()
    if kind == "linear":
        ctx.check(lib.pf_gemv_q(ctx.h, state["w"].h, _ptr(state["x"]), _ptr(state["y"]), state["m"]), "pf_gemv_q")
        return state["y"]
    if kind == "unembed":
        ctx.check(lib.pf_gemv_f32(ctx.h, state["w"].h, _ptr(state["x"]), _ptr(state["y"]), state["m"]), "pf_gemv_f32")
        return state["y"]
    if kind == "int8":
        m, n, k = state["shape"]
        ctx.check(lib.pf_matmul_quantized(ctx.h, _ptr(state["a"]), _ptr(state["b"]), _ptr(state["y"]), m, n, k,
                                          _ptr(state["ws"]), _ptr(state["act"])), "pf_matmul_quantized")
        return state["y"]
    return state["heads"].forward(state["hidden"])


# ------------------------------------------------------ work and accuracy

def work(case):
    kind = case["kind"]
    if kind in ("generate", "prefill", "batch"):
        d, heads, hd, ff = WIDTHS[case["width"]]
        block = {"q4": 18 / 32, "mixed": 10 / 32}
        attn_w, ffn_w = 4 * d * d, 3 * d * ff
        layer = attn_w * block["q4"] + ffn_w * block[case["fmts"]]
        table = case["vocab"] * d * block["q4"]
        seqs, new = case.get("seqs", 1), case.get("new", TAIL)
        prompt = case["prompt"] if kind != "batch" else int(case["prompt"] * 9 / 16)
        # the weights once for the prompts and once per generated token of a
        # sequence (TAIL outputs: once); K/V rows written once, and read once
        # per generated token
        reads = 1 + (0 if kind == "prefill" else new)
        entry = 2 * heads * (hd + 4)
        seen = min(prompt, case["window"])
        kv = case["layers"] * entry * seqs * (prompt + new + (reads - 1) * seen)
        rows = seqs * (prompt + new)
        attn = 4.0 * seqs * d * sum(min(p, case["window"]) for p in range(prompt + new))
        flops = case["layers"] * (2.0 * rows * (attn_w + ffn_w) + attn) + 2.0 * seqs * new * case["vocab"] * d
        return dict(bytes=case["layers"] * layer * reads + table * max(1, reads - 1) + kv, flops=flops)
    if kind == "linear":
        m, n, k = case["m"], case["rows"], case["cols"]
        per = {"q4": 18, "q2": 10, "q15": 10, "q8": 34}[case["fmt"]]
        return dict(bytes=n * k // 32 * per + 4 * m * (n + k), flops=2.0 * m * n * k)
    if kind == "unembed":
        m, n, k = case["m"], case["vocab"], case["cols"]
        return dict(bytes=n * k // 32 * {"q4": 18, "q8": 34}[case["fmt"]] + 4 * m * (n + k), flops=2.0 * m * n * k)
    if kind == "int8":
        m, n, k = case["m"], case["n"], case["k"]
        return dict(bytes=n * k + 4 * m * (n + k) + 4 * n, flops=2.0 * m * n * k)
    h, d, v = case["heads"], case["cols"], case["vocab"]
    return dict(bytes=h * 3 * d * d * 18 // 32 + 4 * v * d + 4 * (d + h * v), flops=2.0 * h * (3 * d * d + v * d))


def tolerance(case):
    kind = case["kind"]
    if kind in ("generate", "prefill", "batch"):
        # every reduction of the engine has one fixed order (the GPU's token
        # streams and logits equal the CPU oracle's bit for bit).  There is
        # no smaller tolerance to state: a changed last bit flips an int8
        # activation code somewhere, and the flips spread to the size of the
        # int8 rounding itself (0.04 between this path and 64 bits over a
        # 6000-token prompt)
        return "exact"
    if kind in ("linear", "int8"):
        return dict(rel=2e-7)                # exact sums, then the roundings of the scales and the result
    return dict(rel=1e-6)                    # fp32 chains of 32, a tree over the blocks


def _act_codes(x):
    """quantize_activation_row: codes round(x * (127 / max|x|)), scale max|x| / 127."""
    amax = x.abs().amax(-1, keepdim=True)
    full = torch.full_like(amax, 127.0)   # tensors: a division by or of a number may be a product
    inv = torch.where(amax == 0, torch.ones_like(amax), full / amax)
    v = (x * inv).double()
    codes = torch.sign(v) * torch.floor(v.abs() + 0.5)
    return codes, torch.where(amax == 0, torch.ones_like(amax), amax / full).double()


def _q(x):
    codes, scale = _act_codes(x)
    return codes * scale


def _exact_prefill(case, seed):
    cfg, w = _model_cfg(case), _model_weights(case, seed)
    d, heads, hd = cfg["n_embd"], cfg["n_heads"], cfg["head_dim"]
    tokens = torch.from_numpy(_tokens(case, seed)).long().cuda()
    n = len(tokens)
    emb = _dequantized(w["emb"])
    x = emb[tokens]
    freq = torch.tensor([1.0 / np.float32(np.float32(5000000.0) ** np.float32(2 * t / hd)) for t in range(hd // 2)],
                        dtype=torch.float32)
    ang = (torch.arange(n, dtype=torch.float32)[:, None] * freq).double().cuda()
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rope(t):
        a, b = t[..., 0::2], t[..., 1::2]
        return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).flatten(-2)

    def norm(t):
        return t / torch.sqrt((t * t).mean(-1, keepdim=True) + 1e-6)

    before = torch.ones(n, n, dtype=torch.bool, device="cuda").tril(-1)
    for lw in w["layers"]:
        a = _q(norm(x))
        q, k, v = ((a @ _dequantized(lw[m]).T).view(n, heads, hd) for m in ("wq", "wk", "wv"))
        q, k = rope(q), rope(k)
        kq, vq = _q(k), _q(v)
        out = torch.empty(n, heads, hd, dtype=torch.float64, device="cuda")
        for h in range(heads):
            s = q[:, h] @ kq[:, h].T / math.sqrt(hd)
            own = (q[:, h] * k[:, h]).sum(-1) / math.sqrt(hd)
            s = s.masked_fill(~before, -math.inf)
            s[range(n), range(n)] = own
            p = torch.softmax(s, -1)
            self_p = p.diagonal().clone()
            out[:, h] = (p - torch.diag(self_p)) @ vq[:, h] + self_p[:, None] * v[:, h]
        x = x + _q(out.reshape(n, d)) @ _dequantized(lw["wo"]).T
        a = _q(norm(x))
        g = a @ _dequantized(lw["wgate"]).T
        f = g * torch.sigmoid(g) * (a @ _dequantized(lw["wup"]).T)
        x = x + _q(f) @ _dequantized(lw["wdown"]).T
    hidden = x[-TAIL:]
    return dict(logits=(hidden @ emb.T)[None].cpu(), hidden=hidden[None].cpu())


def exact(case, seed):
    kind = case["kind"]
    if kind in ("generate", "batch"):
        return None      # tokens and the logits behind them follow from every rounding before
    if kind == "prefill":
        return _exact_prefill(case, seed)
    if kind == "linear":
        w = _dequantized(_Blocks(seed).matrix(case["rows"], case["cols"], FMTS[case["fmt"]]))
        codes, scale = _act_codes(_activations(seed, case["m"], case["cols"]).cuda())
        return (codes @ w.T) * scale
    if kind == "unembed":
        w = _dequantized(_Blocks(seed).matrix(case["vocab"], case["cols"], FMTS[case["fmt"]]))
        return _activations(seed, case["m"], case["cols"]).cuda().double() @ w.T
    if kind == "int8":
        a, b, ws, act = (None if t is None else t.cuda() for t in _int8_inputs(case, seed))
        if act is None:
            codes, scale = _act_codes(a)
        else:
            v = (a / act[:, None]).double()
            codes, scale = torch.sign(v) * torch.floor(v.abs() + 0.5), act[:, None].double()
        return (codes @ b.double().T) * scale * ws.double()
    ws, table = _heads_weights(case, seed)
    h = _activations(seed, 1, case["cols"]).cuda().double()[0]
    t = torch.from_numpy(table).cuda().double()
    out = []
    for hw in ws:
        gate, up, down = (_dequantized(m) for m in hw)
        g = gate @ h
        h = h + down @ (g * torch.sigmoid(g) * (up @ h))
        out.append(t @ h)
    return torch.stack(out).cpu().numpy()
