"""The work that a user of this framework has it do, as cases that can be timed and compared.

A case is a dict of plain values; its "kind" says which public entry points one pass calls:

  linears  the four DetLinear calls of one decoder layer (qkv, o, gate_up, down) on fp32 rows:
           decode steps, small batches and prefill of the deterministic runtime
  layer    detgpu.layer_fused: one whole decoder layer of B sequences of T tokens
  stage    detgpu.forward_stage_roots: embedding, several layers, every layer's stage-output root
           (the unit of work that a job of the runtime commits to)
  logits   detgpu.final_logits and the row roots of the integer logits: the head of a forward
  sweep    MinedWeight.forward_many and sweep_winners: a miner's sweep of nonces with useful output
  attempt  MinedWeight.noise_mine and winners: a pure miner's attempt, tiles only
  hf       the four MinedLinear modules of one layer of a Hugging Face model on bf16 rows, mined
           (with their winners read back) or integer only

Every result is consensus: the int32 sums, the requantized bytes, the fp32 steps (each one IEEE
operation in a fixed order), the digests and the winners are the same bits in every correct
implementation, so every case is compared exactly. exact() gives the fp32 and bf16 outputs in
float64 from the same inputs.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "useful-work-coin_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

DEV = "cuda"
EPS = 1e-6
THETA = 1e6
MAX_WINS = 64

# hidden, query heads, kv heads, head_dim, intermediate; qknorm: per-head RMSNorm of q and k
QWEN3_1P7B = dict(D=2048, H=16, Hkv=8, hd=128, I=6144, qknorm=True)
LLAMA_8B = dict(D=4096, H=32, Hkv=8, hd=128, I=14336, qknorm=False)
VOCAB = 151936


def listed():
    return [
        # one token of a decode step: eight small launches, weights read once
        dict(name="linears_decode_1", kind="linears", m=1, hb=512, **QWEN3_1P7B),
        # a decode batch of an odd size on the larger model: weight streaming
        dict(name="linears_batch_33", kind="linears", m=33, hb=512, **LLAMA_8B),
        # a prompt as it comes: a ragged number of rows
        dict(name="linears_prompt_777", kind="linears", m=777, hb=512, **QWEN3_1P7B),
        # prefill of a whole chunk
        dict(name="linears_prefill_2048", kind="linears", m=2048, hb=512, **QWEN3_1P7B),
        # the longest prefill of the larger model
        dict(name="linears_prefill_8192", kind="linears", m=8192, hb=512, **LLAMA_8B),
        # a verifier's layer over a short prompt: launches and small grids
        dict(name="layer_prompt_200", kind="layer", B=1, T=200, **QWEN3_1P7B),
        # two ragged prompts through a layer without q/k norms
        dict(name="layer_batch_2x1000", kind="layer", B=2, T=1000, **LLAMA_8B),
        # a stage of a long job with its commitments
        dict(name="stage_8192", kind="stage", T=8192, L=4, V=VOCAB, **QWEN3_1P7B),
        # the logits of a verified continuation, committed row by row
        dict(name="logits_300", kind="logits", rows=300, V=VOCAB, **QWEN3_1P7B),
        # the mining shape, nonces in one sweep, exact int32 products kept
        dict(name="sweep_4096", kind="sweep", m=4096, n=4096, k=4096, r=64, nonces=20),
        # one attempt of a pure miner at its own shape
        dict(name="attempt_8192x16384", kind="attempt", m=8192, n=16384, k=4096, r=128),
        # a provider's mined layer over a prompt, bf16 in and out
        dict(name="hf_mined_1000", kind="hf", tokens=1000, mode="mined", hb=512, **QWEN3_1P7B),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _model(rng):
    """Qwen3-1.7B's or Llama-3.1-8B's layer, or a generic one of widths in between."""
    pick = rng.random()
    if pick < 0.4:
        return dict(QWEN3_1P7B)
    if pick < 0.6:
        return dict(LLAMA_8B)
    hd = rng.choice([64, 128, 128])
    Hkv = rng.choice([2, 4, 8])
    H = Hkv * rng.choice([1, 2, 4])
    return dict(D=128 * rng.randint(8, 32), H=H, Hkv=Hkv, hd=hd, I=128 * rng.randint(16, 96), qknorm=rng.random() < 0.5)


def draw(rng):
    kind = rng.choice(["linears", "linears", "linears", "linears", "layer", "layer", "layer", "stage", "logits", "sweep",
                       "sweep", "attempt", "hf", "hf"])
    if kind == "linears":
        return dict(kind=kind, m=_log_int(rng, 1, 6000), hb=rng.choice([128, 512, 512]), **_model(rng))
    if kind == "layer":
        B = rng.choice([1, 1, 2, 4])
        return dict(kind=kind, B=B, T=_log_int(rng, 8, 4096 // B), **_model(rng))
    if kind == "stage":
        return dict(kind=kind, T=_log_int(rng, 256, 4096), L=rng.randint(1, 4), V=VOCAB, **QWEN3_1P7B)
    if kind == "logits":
        return dict(kind=kind, rows=_log_int(rng, 1, 1024), V=VOCAB, **QWEN3_1P7B)
    if kind == "hf":
        mode = rng.choice(["mined", "int"])
        return dict(kind=kind, tokens=_log_int(rng, 1, 4096), mode=mode, hb=512, **QWEN3_1P7B)
    # the rank rule: k between max(1024, 16 r) and 4 r^2
    r = rng.choice([64, 64, 128])
    k = 128 * rng.randint(max(1024, 16 * r) // 128, 4096 // 128)
    if kind == "sweep":
        return dict(kind=kind, m=128 * rng.randint(8, 32), n=128 * rng.randint(8, 32), k=k, r=r, nonces=rng.randint(1, 20))
    return dict(kind=kind, m=256 * rng.randint(4, 32), n=256 * rng.randint(8, 64), k=k, r=r)


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEV)


def _hidden(g, rows, k):
    """Normed hidden rows: unit variance with a few loud channels, as a transformer's are."""
    return _randn(g, rows, k) * torch.exp(0.5 * _randn(g, k))


def _gated(g, rows, k):
    """silu(g) * u of a gated MLP: many values near zero, heavy tails."""
    return torch.nn.functional.silu(_randn(g, rows, k)) * _randn(g, rows, k)


def _linear_shapes(c):
    D, H, Hkv, hd, I = c["D"], c["H"], c["Hkv"], c["hd"], c["I"]
    return {"qkv": ((H + 2 * Hkv) * hd, D), "o": (D, H * hd), "gu": (2 * I, D), "down": (D, I)}


def _linear_inputs(g, c, rows):
    x = _hidden(g, rows, c["D"])
    return {"qkv": x, "o": 0.3 * _randn(g, rows, c["H"] * c["hd"]), "gu": _hidden(g, rows, c["D"]),
            "down": _gated(g, rows, c["I"])}


def _weights(g, n, k):
    return 0.02 * _randn(g, n, k)


def _layer_weights(g, c):
    """One layer's fp32 parameters."""
    near1 = lambda k: 1.0 + 0.05 * _randn(g, k)  # noqa: E731
    return dict(in_norm=near1(c["D"]), post_norm=near1(c["D"]), q_norm=near1(c["hd"]), k_norm=near1(c["hd"]),
                **{nm: _weights(g, n, k) for nm, (n, k) in _linear_shapes(c).items()})


def _det_model(g, c, layers, positions, vocab=None, head=False):
    """A detgpu.DetModel of `layers` layers from freshly drawn fp32 parameters."""
    from uwc_amd import detgpu
    from uwc_amd.detrt import DetLinear
    Ls = []
    for _ in range(layers):
        w = _layer_weights(g, c)
        Ls.append({nm: DetLinear(t, DEV, 512) if nm in ("qkv", "o", "gu", "down") else t for nm, t in w.items()})
        del w
    cos, sin = (torch.from_numpy(t).to(DEV) for t in detgpu.rope_table(THETA, c["hd"], positions))
    embed = _randn(g, vocab or 8, c["D"])
    norm = 1.0 + 0.05 * _randn(g, c["D"])
    lm = DetLinear(_weights(g, vocab, c["D"]), DEV, 512) if head else None
    cfg = dict(D=c["D"], H=c["H"], Hkv=c["Hkv"], hd=c["hd"], eps=EPS, Bs=512, arch=0 if c["qknorm"] else 1)
    return detgpu.DetModel(cfg, embed, Ls, cos, sin, norm, lm)


def _bytes(g, n):
    return bytes(torch.randint(0, 256, (n,), generator=g, device=DEV).tolist())


def _target(tiles, wins):
    """Little-endian target words met by about `wins` of `tiles` random digests."""
    v = min((1 << 256) - 1, ((1 << 256) // tiles) * wins)
    return np.array([(v >> (32 * i)) & 0xFFFFFFFF for i in range(8)], dtype=np.uint32)


def _tiles(m, n):
    return (m // 64) * (n // 64) * 32


def _int8(g, *shape):
    return torch.randint(-64, 64, shape, generator=g, device=DEV, dtype=torch.int8)


def prepare(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    if kind == "linears":
        from uwc_amd.detrt import DetLinear
        lins = {nm: DetLinear(_weights(g, n, k), DEV, c["hb"]) for nm, (n, k) in _linear_shapes(c).items()}
        return dict(kind=kind, lins=lins, x=_linear_inputs(g, c, c["m"]))
    if kind == "layer":
        m = _det_model(g, c, 1, c["T"])
        return dict(kind=kind, model=m, x=_hidden(g, c["B"] * c["T"], c["D"]), B=c["B"], T=c["T"])
    if kind == "stage":
        m = _det_model(g, c, c["L"], c["T"], vocab=c["V"])
        tokens = torch.randint(0, c["V"], (1, c["T"]), generator=g, device=DEV)
        return dict(kind=kind, model=m, tokens=tokens)
    if kind == "logits":
        m = _det_model(g, c, 0, 8, vocab=c["V"], head=True)
        return dict(kind=kind, model=m, x=_hidden(g, c["rows"], c["D"]))
    if kind in ("sweep", "attempt"):
        from uwc_amd import ops
        m, n, k, r = c["m"], c["n"], c["k"], c["r"]
        w = ops.MinedWeight(Bt=_int8(g, n, k), b_scale=torch.ones(n, device=DEV), r=r, max_wins=MAX_WINS)
        w.setup_block(_bytes(g, 32), _target(_tiles(m, n), 8))
        if kind == "attempt":
            return dict(kind=kind, w=w, A=_int8(g, m, k))
        N = c["nonces"]
        out = torch.empty((N, m, n), dtype=torch.int32, device=DEV)
        w.reserve_sweep(m, N)
        return dict(kind=kind, w=w, As=[_int8(g, m, k) for _ in range(N)], scale=torch.ones(m, device=DEV), out=out)
    from uwc_amd import model
    mls = {}
    for nm, (n, k) in _linear_shapes(c).items():
        lin = torch.nn.Linear(k, n, bias=False, device=DEV)
        with torch.no_grad():
            lin.weight.copy_(_weights(g, n, k))
        ml = mls[nm] = model.MinedLinear([lin], DEV, mode=c["mode"], hadamard_block=c["hb"], r=128)
        key, tiles = _bytes(g, 32), _tiles(-(-c["tokens"] // 128) * 128, n)
        ml.setup_block(lambda k: key, lambda k: _target(tiles, 8))
    x = {nm: t.to(torch.bfloat16) for nm, t in _linear_inputs(g, c, c["tokens"]).items()}
    return dict(kind=kind, mls=mls, x=x, mined=c["mode"] == "mined", m=-(-c["tokens"] // 128) * 128)


# ------------------------------------------------------------------ one pass
def _wins(lists):
    """Win lists, whose records come in no order, as an array: per list the count, then the sorted
    records (row, column, eight digest words), zero past the count."""
    a = np.zeros((len(lists), 1 + MAX_WINS, 10), dtype=np.int64)
    a[:, 0, 0] = [len(wins) for wins in lists]
    found = [(i, 1 + j, row, col, digest) for i, wins in enumerate(lists) for j, (row, col, digest) in enumerate(sorted(wins))]
    if found:
        i, j, row, col, digest = zip(*found)
        a[i, j, 0], a[i, j, 1] = row, col
        a[i, j, 2:] = np.frombuffer(b"".join(digest), dtype=np.uint32).reshape(-1, 8)
    return a


def run(state):
    s, kind = state, state["kind"]
    if kind == "linears":
        return {nm: lin(s["x"][nm]) for nm, lin in s["lins"].items()}
    if kind == "sweep":
        from uwc_amd import ops
        s["w"].forward_many(s["As"], s["scale"], outs=list(s["out"].unbind(0)), out_mode=ops.OUT_I32)
        return {"out": s["out"], "wins": _wins(s["w"].sweep_winners())}
    if kind == "attempt":
        s["w"].noise_mine(s["A"])
        return {"wins": _wins([s["w"].winners(s["A"].shape[0])])}
    if kind == "hf":
        with torch.no_grad():
            y = {nm: ml(s["x"][nm]) for nm, ml in s["mls"].items()}
        if s["mined"]:
            y["wins"] = _wins([ml.mw.winners(s["m"]) for ml in s["mls"].values()])
        return y
    from uwc_amd import detgpu
    if kind == "layer":
        return detgpu.layer_fused(s["model"], s["model"].layers[0], s["x"], s["B"], s["T"])
    if kind == "stage":
        x, roots = detgpu.forward_stage_roots(s["model"], s["tokens"])
        return {"out": x, "roots": roots}
    acc, logits = detgpu.final_logits(s["model"], s["x"])
    return {"acc": acc, "logits": logits, "roots": detgpu.row_roots(acc)}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    c, kind = case, case["kind"]
    shapes = _linear_shapes(c) if "D" in c else {}
    wbytes = sum(n * k + 4 * n for n, k in shapes.values())
    macs = sum(n * k for n, k in shapes.values())
    if kind == "linears":
        rows = c["m"]
        return dict(bytes=wbytes + rows * sum(4 * k + 4 * n for n, k in shapes.values()), flops=2 * rows * macs)
    if kind == "hf":
        rows = c["tokens"]
        return dict(bytes=wbytes + rows * sum(2 * k + 2 * n for n, k in shapes.values()), flops=2 * rows * macs)
    if kind in ("layer", "stage"):
        B, T, L = c.get("B", 1), c["T"], c.get("L", 1)
        attn = 2 * B * c["H"] * c["hd"] * T * (T + 1)  # q.k and p.v over the causal half
        return dict(bytes=L * wbytes + (L + 1) * 4 * B * T * c["D"], flops=L * (2 * B * T * macs + attn))
    if kind == "logits":
        rows, D, V = c["rows"], c["D"], c["V"]
        return dict(bytes=V * D + 4 * V + 4 * rows * D + 8 * rows * V, flops=2 * rows * D * V)
    m, n, k, r = c["m"], c["n"], c["k"], c["r"]
    N = c.get("nonces", 1)
    denoise = 2 * m * n * 2 * r if kind == "sweep" else 0
    out = 4 * m * n if kind == "sweep" else 0
    return dict(bytes=n * k + N * (m * k + out), flops=N * (2 * m * n * k + denoise))


def tolerance(case):
    return "exact"


# ------------------------------------------------------------------ the same in float64
F64 = torch.float64


def _rotated(x, hb):
    """x (rows, k) rotated by the orthonormal Walsh-Hadamard matrix in blocks of min(hb, k & -k)."""
    k = x.shape[1]
    bs = min(hb, k & -k) if hb else 1
    y = x.to(F64)
    h = 1
    while h < bs:
        y = y.view(-1, 2, h)
        y = torch.stack([y[:, 0] + y[:, 1], y[:, 0] - y[:, 1]], dim=1)
        h *= 2
    return y.reshape(x.shape) / math.sqrt(bs)


def _quantized(y, qmax):
    """(integer-valued q, scale) of symmetric quantization along the last axis, half to even."""
    s = y.abs().amax(-1, keepdim=True).clamp(min=1e-8) / qmax
    return torch.round(y / s).clamp(-qmax, qmax), s


def _linear64(x, W, hb):
    """x W^T with both sides rotated and quantized to [-64, 64], the weight a slab at a time."""
    q, s = _quantized(_rotated(x, hb), 64)
    out = torch.empty((x.shape[0], W.shape[0]), dtype=F64, device=x.device)
    for i in range(0, W.shape[0], 8192):
        wq, ws = _quantized(_rotated(W[i:i + 8192], hb), 64)
        out[:, i:i + 8192] = (q @ wq.t()) * s * ws.t()
    return out


def _rmsnorm64(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.to(F64)


def _layer64(c, w, x, B, T):
    D, H, Hkv, hd, I = c["D"], c["H"], c["Hkv"], c["hd"], c["I"]
    qkv = _linear64(_rmsnorm64(x, w["in_norm"]), w["qkv"], 512).view(B, T, H + 2 * Hkv, hd)
    q, k, v = qkv.split([H, Hkv, Hkv], dim=2)
    if c["qknorm"]:
        q, k = _rmsnorm64(q, w["q_norm"]), _rmsnorm64(k, w["k_norm"])
    freq = THETA ** (-torch.arange(0, hd, 2, dtype=F64, device=x.device) / hd)
    ang = torch.arange(T, dtype=F64, device=x.device)[:, None] * freq.repeat(2)[None]
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    turn = lambda z: z * cos + torch.cat([-z[..., hd // 2:], z[..., :hd // 2]], -1) * sin  # noqa: E731
    q, k = turn(q), turn(k)
    o = torch.empty((B, T, H, hd), dtype=F64, device=x.device)
    mask = torch.ones((T, T), dtype=torch.bool, device=x.device).tril()
    for b in range(B):
        for h in range(H):
            (qq, qs), (kq, ks), (vq, vs) = (_quantized(z, 127) for z in (q[b, :, h], k[b, :, h * Hkv // H], v[b, :, h * Hkv // H]))
            sc = (qq @ kq.t()) * qs * ks.t() / math.sqrt(hd)
            p = torch.softmax(sc.masked_fill_(~mask, -math.inf), -1) * vs.t()
            sp = p.amax(-1, keepdim=True).clamp(min=1e-30) / 16383
            o[b, :, h] = (torch.round(p / sp) @ vq) * sp
    x = x + _linear64(o.view(B * T, H * hd), w["o"], 512)
    gu = _linear64(_rmsnorm64(x, w["post_norm"]), w["gu"], 512)
    return x + _linear64(torch.nn.functional.silu(gu[:, :I]) * gu[:, I:], w["down"], 512)


def exact(case, seed):
    c, g, kind = case, _gen(seed), case["kind"]
    if kind in ("linears", "hf"):
        W = {}
        for nm, (n, k) in _linear_shapes(c).items():
            W[nm] = _weights(g, n, k)
            if kind == "hf":
                _bytes(g, 32)
        x = _linear_inputs(g, c, c.get("m") or c["tokens"])
        if kind == "hf":
            x = {nm: t.to(torch.bfloat16) for nm, t in x.items()}
        y = {nm: _linear64(x[nm], W[nm], c["hb"]) for nm in W}
        if c.get("mode") == "mined":
            y["wins"] = None
        return y
    if kind == "layer":
        w = _layer_weights(g, c)
        _randn(g, 8, c["D"]), _randn(g, c["D"])  # the model's embedding and final norm
        return _layer64(c, w, _hidden(g, c["B"] * c["T"], c["D"]).to(F64), c["B"], c["T"])
    if kind == "stage":
        ws = [_layer_weights(g, c) for _ in range(c["L"])]
        embed, _ = _randn(g, c["V"], c["D"]), _randn(g, c["D"])
        x = embed[torch.randint(0, c["V"], (1, c["T"]), generator=g, device=DEV)[0]].to(F64)
        for w in ws:
            x = _layer64(c, w, x, 1, c["T"])
        return {"out": x, "roots": None}
    if kind == "logits":
        _randn(g, c["V"], c["D"])  # the model's embedding
        norm = 1.0 + 0.05 * _randn(g, c["D"])
        W = _weights(g, c["V"], c["D"])
        x = _hidden(g, c["rows"], c["D"]).to(F64)
        return {"acc": None, "logits": _linear64(_rmsnorm64(x, norm), W, 512), "roots": None}
    return None  # integers and digests only
