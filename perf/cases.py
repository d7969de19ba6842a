"""The work that a user of this library has it do, as timed cases.

Five kinds, each through the library's public entry points:

  chain   the memory-bound ops of one layer on their own: token-embedding gather (F32 or
          quantized table) -> residual add + RMSNorm -> RoPE on Q and K -> SwiGLU
  layer   the embedding gather and one whole transformer layer over a batch of tokens: a decode
          step (tokens at given positions of the cache, weights with their planar copies) or a
          prompt chunk at consecutive positions
  linear  one projection over quantized (blocks or planar copy) or fp32 weights
  head    the final RMSNorm and the vocabulary projection of some rows (the logits)
  model   a whole small model, tokens to logits on the host (DeviceModel.forward)

Sizes are the Llama-3-8B and Llama-3-70B shapes and the tiny configurations of
cpp-minilamma_amd/workloads.py, bench.py and tests/.  Inputs are made with torch on the GPU from
the seed; quantized weights are made here by a plain torch quantizer, so `exact` needs nothing of
the library.
"""
from __future__ import annotations

import importlib
import math

import numpy as np
import torch

from __graft_entry__ import load_package

DEV = "cuda"
QK = 32  # elements of a quantization block
VOCAB = 128256
SHAPES = {  # dim, hidden_dim, n_heads, n_kv_heads, head_dim, theta, vocab
    "tiny": dict(dim=64, hidden_dim=172, n_heads=4, n_kv_heads=2, head_dim=16, theta=10000.0,
                 vocab=131),
    "8b": dict(dim=4096, hidden_dim=14336, n_heads=32, n_kv_heads=8, head_dim=128,
               theta=500000.0, vocab=VOCAB),
    "70b": dict(dim=8192, hidden_dim=28672, n_heads=64, n_kv_heads=8, head_dim=128,
                theta=500000.0, vocab=VOCAB),
}
EPS = 1e-5
BLOCK_BYTES = {"q8_0": 34, "q4_0": 18, "q4_1": 20}
MAX_SEQ = 8192  # cache length of the decode and chunk cases

_mods = {}


def lib():
    """The package and its forward module."""
    if not _mods:
        _mods["mlk"] = load_package()
        _mods["fwd"] = importlib.import_module(_mods["mlk"].__name__ + ".forward")
        _mods["mlk"].set_device(0)
    return _mods["mlk"], _mods["fwd"]


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # the tiny model's op chain on a 6-token prompt: launches and their latency
        dict(name="chain_tiny_6", kind="chain", shape="tiny", tokens=6, table="f32"),
        # the library's headline: the op chain of a 4096-token prompt at the 8B shape
        dict(name="chain_8b_4096", kind="chain", shape="8b", tokens=4096, table="f32"),
        # the op chain at the 70B shape over an odd-sized prompt, rows from a quantized table
        dict(name="chain_70b_q4_0_1001", kind="chain", shape="70b", tokens=1001, table="q4_0"),
        # one decode step of one sequence at the end of an 8192-token context
        dict(name="layer_8b_q8_0_decode_1", kind="layer", shape="8b", type="q8_0", tokens=1,
             decode=True, pos0=8191),
        # decode steps of small and larger batches, positions spread over the context
        dict(name="layer_8b_q4_0_decode_16", kind="layer", shape="8b", type="q4_0", tokens=16,
             decode=True, pos0=8191),
        dict(name="layer_8b_q8_0_decode_64", kind="layer", shape="8b", type="q8_0", tokens=64,
             decode=True, pos0=8191),
        # a later, ragged chunk of a chat's prompt
        dict(name="layer_8b_q4_0_chunk_389", kind="layer", shape="8b", type="q4_0", tokens=389,
             decode=False, pos0=1500),
        # a long prompt over unquantized weights
        dict(name="layer_8b_f32_prefill_1024", kind="layer", shape="8b", type="f32", tokens=1024,
             decode=False, pos0=0),
        # a full prompt
        dict(name="layer_8b_q8_0_prefill_4096", kind="layer", shape="8b", type="q8_0",
             tokens=4096, decode=False, pos0=0),
        # a short prompt's down projection at the 70B shape, the third block format
        dict(name="linear_70b_q4_1_down_100", kind="linear", shape="70b", proj="w_down",
             type="q4_1", layout="blocks", tokens=100),
        # the logits of one decode step
        dict(name="head_8b_q8_0_1", kind="head", shape="8b", type="q8_0", tokens=1),
        # a whole tiny model on a 9-token prompt, logits of every token on the host
        dict(name="model_tiny_9", kind="model", dim=32, hidden_dim=86, layers=2, n_heads=4,
             n_kv_heads=2, head_dim=8, type="f32", tokens=9),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["chain", "chain", "layer", "layer", "layer", "layer", "linear", "linear",
                       "head", "model"])
    types = ["q8_0", "q8_0", "q4_0", "q4_0", "q4_1", "f32"]
    if kind == "chain":
        shape = rng.choice(["tiny", "8b", "8b", "70b"])
        return dict(kind=kind, shape=shape, tokens=_log_int(rng, 1, 2048 if shape == "70b" else 4096),
                    table=rng.choice(["f32", "q8_0", "q4_0", "q4_1"]))
    if kind == "layer":
        shape = rng.choice(["8b", "8b", "8b", "70b"])
        wt = rng.choice(types)
        if shape == "70b" and wt == "f32":
            wt = "q8_0"
        if rng.random() < 0.5:
            tokens = _log_int(rng, 1, 64)
            return dict(kind=kind, shape=shape, type=wt, tokens=tokens, decode=True,
                        pos0=rng.randint(max(tokens, 200), MAX_SEQ - 1))
        most = {"8b": 3000, "70b": 700}[shape]
        if wt in ("q4_1", "f32"):
            most //= 3
        tokens = _log_int(rng, 8, most)
        return dict(kind=kind, shape=shape, type=wt, tokens=tokens, decode=False,
                    pos0=rng.choice([0, rng.randint(1, MAX_SEQ - tokens)]))
    if kind == "linear":
        wt = rng.choice(types)
        return dict(kind=kind, shape=rng.choice(["8b", "70b"]),
                    proj=rng.choice(["wq", "wk", "wo", "w_gate", "w_down"]), type=wt,
                    layout=rng.choice(["blocks", "planar"]) if wt in ("q8_0", "q4_0") else "blocks",
                    tokens=_log_int(rng, 1, 2500 if wt in ("q8_0", "q4_0") else 800))
    if kind == "head":
        return dict(kind=kind, shape="8b", type=rng.choice(types), tokens=_log_int(rng, 1, 100))
    n_heads = rng.choice([4, 8])
    hd = rng.choice([8, 32, 64])
    return dict(kind=kind, dim=n_heads * hd, hidden_dim=rng.choice([86, 172, 384, 512, 1024]),
                layers=rng.choice([2, 3]), n_heads=n_heads, n_kv_heads=rng.choice([1, 2, 4]),
                head_dim=hd, type=rng.choice(["f32", "q8_0", "q4_0"]), tokens=rng.randint(1, 64))


# ------------------------------------------------------------------ inputs

def _gen(seed):
    g = torch.Generator(DEV)
    g.manual_seed(int(seed))
    return g


def _normal(g, shape, std=1.0, mean=0.0):
    x = torch.empty(shape, device=DEV, dtype=torch.float32)
    return x.normal_(mean, std, generator=g)


def _zipf_ids(g, n, vocab, s=1.1):
    """n token ids, id r with probability proportional to (r + 1)^-s."""
    cdf = torch.arange(1, vocab + 1, device=DEV, dtype=torch.float64).pow(-s).cumsum(0)
    u = torch.rand(n, device=DEV, dtype=torch.float64, generator=g) * cdf[-1]
    return torch.searchsorted(cdf, u).clamp_max(vocab - 1).to(torch.int32)


def _quantize(w, qtype):
    """[rows, cols] fp32 -> the packed blocks [rows, bytes] of the three GGUF formats."""
    rows, cols = w.shape
    nb = -(-cols // QK)
    if cols % QK:
        w = torch.nn.functional.pad(w, (0, nb * QK - cols))
    out = torch.empty((rows, nb, BLOCK_BYTES[qtype]), device=w.device, dtype=torch.uint8)
    step = max(1, (1 << 26) // (nb * QK))
    for r in range(0, rows, step):
        b = w[r:r + step].reshape(-1, nb, QK)
        n = b.shape[0]
        if qtype == "q8_0":
            d = (b.abs().amax(-1) / 127).half()
            head = d.view(torch.uint8).reshape(n, nb, 2)
            q = (b / d.float().clamp_min(1e-12)[..., None]).round().clamp(-127, 127)
            codes = q.to(torch.int8).view(torch.uint8)
        else:
            if qtype == "q4_0":
                d = (b.abs().amax(-1) / 7).half()
                head = d.view(torch.uint8).reshape(n, nb, 2)
                q = (b / d.float().clamp_min(1e-12)[..., None]).round().clamp(-8, 7) + 8
            else:
                lo, hi = b.amin(-1), b.amax(-1)
                d, m = ((hi - lo) / 15).half(), lo.half()
                head = torch.stack([d, m], -1).view(torch.uint8).reshape(n, nb, 4)
                q = ((b - m.float()[..., None]) / d.float().clamp_min(1e-12)[..., None])
                q = q.round().clamp(0, 15)
            q = q.to(torch.uint8)
            codes = q[..., :QK // 2] | (q[..., QK // 2:] << 4)
        out[r:r + step, :, :head.shape[-1]] = head
        out[r:r + step, :, head.shape[-1]:] = codes
    return out.reshape(rows, -1)


def _dequantize(blocks, qtype, cols):
    """The packed blocks [rows, bytes] as float64 [rows, cols]."""
    rows = blocks.shape[0]
    b = blocks.reshape(rows, -1, BLOCK_BYTES[qtype])
    half = lambda at: b[..., at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if qtype == "q8_0":
        w = b[..., 2:].contiguous().view(torch.int8).double() * half(0)
    else:
        at = 2 if qtype == "q4_0" else 4
        codes = torch.cat([b[..., at:] & 15, b[..., at:] >> 4], -1).double()
        w = (codes - 8) * half(0) if qtype == "q4_0" else codes * half(0) + half(2)
    return w.reshape(rows, -1)[:, :cols]


def _weight(g, rows, cols, wt, std=0.02):
    w = _normal(g, (rows, cols), std)
    return w if wt == "f32" else _quantize(w, wt)


def _weight64(w, wt, cols):
    return w.double() if wt == "f32" else _dequantize(w, wt, cols)


def _projections(s):
    D, F = s["dim"], s["hidden_dim"]
    QD, KD = s["n_heads"] * s["head_dim"], s["n_kv_heads"] * s["head_dim"]
    return {"wq": (QD, D), "wk": (KD, D), "wv": (KD, D), "wo": (D, QD), "w_gate": (F, D),
            "w_up": (F, D), "w_down": (D, F)}


def _positions(g, case):
    """A decode batch's cache positions: distinct, increasing, the last at pos0; the cases with
    one token pass pos0 itself."""
    T, top = case["tokens"], case["pos0"]
    p = torch.randperm(top, device=DEV, generator=g)[:T - 1].sort().values
    return torch.cat([p, torch.tensor([top], device=DEV)]).to(torch.int32)


def _layer_inputs(case, seed):
    s, wt, T = SHAPES[case["shape"]], case["type"], case["tokens"]
    g = _gen(seed)
    D = s["dim"]
    slots = MAX_SEQ if case["decode"] else case["pos0"] + T
    d = {"g1": _normal(g, (D,), 0.1, 1.0), "g2": _normal(g, (D,), 0.1, 1.0)}
    d["w"] = {n: _weight(g, o, i, wt) for n, (o, i) in _projections(s).items()}
    d["table"] = _weight(g, s["vocab"], D, wt)
    d["ids"] = _zipf_ids(g, T, s["vocab"])
    d["k"] = _normal(g, (1, slots, s["n_kv_heads"], s["head_dim"]))
    d["v"] = _normal(g, (1, slots, s["n_kv_heads"], s["head_dim"]))
    d["pos"] = _positions(g, case) if case["decode"] and T > 1 else None
    return d


def _chain_inputs(case, seed):
    s, T = SHAPES[case["shape"]], case["tokens"]
    g = _gen(seed)
    D, F, hd = s["dim"], s["hidden_dim"], s["head_dim"]
    return {"table": _weight(g, s["vocab"], D, case["table"]), "ids": _zipf_ids(g, T, s["vocab"]),
            "delta": _normal(g, (T, D), 0.02), "w": _normal(g, (D,), 0.1, 1.0),
            "q": _normal(g, (T, s["n_heads"], hd)), "k": _normal(g, (T, s["n_kv_heads"], hd)),
            "gate": _normal(g, (T, F)), "up": _normal(g, (T, F))}


def _linear_inputs(case, seed):
    s = SHAPES[case["shape"]]
    g = _gen(seed)
    out, inner = (s["vocab"], s["dim"]) if case["kind"] == "head" else \
        _projections(s)[case["proj"]]
    return {"x": _normal(g, (case["tokens"], inner)), "w": _weight(g, out, inner, case["type"]),
            "g": _normal(g, (inner,), 0.1, 1.0)}


def _model_inputs(case, seed):
    """A small model in DeviceModel's layout (numpy), and its tokens."""
    c = dict(vocab=131, max_seq=128, rope_type=0, theta=10000.0, eps=EPS,
             **{k: case[k] for k in ("dim", "hidden_dim", "layers", "n_heads", "n_kv_heads",
                                     "head_dim")})
    r = np.random.default_rng(seed)
    wt = case["type"]

    def mat(o, i):
        w = (r.standard_normal((o, i)) / math.sqrt(i)).astype(np.float32)
        return ("f32", w) if wt == "f32" else (wt, _quantize(torch.from_numpy(w), wt).numpy())

    def norm():
        return (1 + 0.1 * r.standard_normal(c["dim"])).astype(np.float32)

    layers = []
    for _ in range(c["layers"]):
        lw = {n: mat(o, i) for n, (o, i) in _projections(c).items()}
        lw.update(attention_norm=norm(), ffn_norm=norm())
        layers.append(lw)
    model = {"config": c, "embedding": r.standard_normal((c["vocab"], c["dim"])).astype(np.float32),
             "layers": layers, "final_norm": norm(), "lm_head": mat(c["vocab"], c["dim"])}
    return model, r.integers(0, c["vocab"], case["tokens"]).astype(np.int32)


def prepare(case, seed):
    mlk, fwd = lib()
    kind = case["kind"]
    if kind == "model":
        model, tokens = _model_inputs(case, seed)
        return dict(case=case, model=fwd.DeviceModel(model), tokens=tokens)
    if kind == "chain":
        d = _chain_inputs(case, seed)
        d["x"], d["y"] = torch.empty_like(d["delta"]), torch.empty_like(d["delta"])
        d["ffn"] = torch.empty_like(d["gate"])
        return dict(d, case=case, s=SHAPES[case["shape"]])
    if kind in ("linear", "head"):
        d = _linear_inputs(case, seed)
        T, K, O = case["tokens"], d["x"].shape[1], d["w"].shape[0]
        d["y"] = torch.empty((T, O), device=DEV)
        if kind == "head":
            d["h"] = torch.empty((T, K), device=DEV)
        elif case["layout"] == "planar":
            d["planar"] = torch.empty(mlk.quant_planar_bytes(case["type"], O, K), device=DEV,
                                      dtype=torch.uint8)
            mlk.quant_to_planar(case["type"], d["w"].data_ptr(), O, K, d["planar"].data_ptr())
        return dict(d, case=case)
    d = _layer_inputs(case, seed)
    s, T, wt = SHAPES[case["shape"]], case["tokens"], case["type"]
    cfg = dict(s, rope_type=0, eps=EPS)
    lw, planars = fwd.LayerWeights(), []
    lw.attention_norm, lw.ffn_norm = d["g1"].data_ptr(), d["g2"].data_ptr()
    for n, (o, i) in _projections(s).items():
        w = fwd.LinearWeight()
        w.type = fwd.WEIGHT_F32 if wt == "f32" else mlk.QUANT[wt]
        w.data = d["w"][n].data_ptr()
        # a serving program keeps planar copies for its decode steps
        if case["decode"] and wt in ("q8_0", "q4_0"):
            p = torch.empty(mlk.quant_planar_bytes(wt, o, i), device=DEV, dtype=torch.uint8)
            mlk.quant_to_planar(wt, w.data, o, i, p.data_ptr())
            w.planar = p.data_ptr()
            planars.append(p)
        setattr(lw, n, w)
    max_ctx = case["pos0"] + (1 if case["decode"] else T)
    ws = mlk.DeviceBuffer(fwd.layer_workspace_bytes(cfg, T, max_ctx, d["pos"] is None), np.uint8)
    x = torch.empty((T, s["dim"]), device=DEV)
    return dict(d, case=case, cfg=cfg, lw=lw, planars=planars, ws=ws, x=x, max_ctx=max_ctx)


# ------------------------------------------------------------------ one pass

def _gather(mlk, wt, table, vocab, D, ids, T, out):
    if wt == "f32":
        mlk.gather_f32(table.data_ptr(), vocab, D, ids.data_ptr(), T, out.data_ptr())
    else:
        mlk.gather_quant(wt, table.data_ptr(), vocab, D, ids.data_ptr(), T, out.data_ptr())


def _linear(mlk, wt, x, w, y):
    T, K, O = x.shape[0], x.shape[1], y.shape[1]
    if wt == "f32":
        mlk.linear_f32(x.data_ptr(), w.data_ptr(), y.data_ptr(), T, K, O)
    else:
        mlk.linear_quant(wt, x.data_ptr(), w.data_ptr(), y.data_ptr(), T, K, O)


def run(st):
    mlk, fwd = lib()
    case = st["case"]
    kind, T = case["kind"], case["tokens"]
    if kind == "chain":
        s = st["s"]
        D = s["dim"]
        _gather(mlk, case["table"], st["table"], s["vocab"], D, st["ids"], T, st["x"])
        mlk.add_rmsnorm(st["x"].data_ptr(), st["delta"].data_ptr(), st["w"].data_ptr(),
                        st["y"].data_ptr(), T, D, EPS)
        mlk.rope(st["q"].data_ptr(), st["k"].data_ptr(), T, s["n_heads"], s["n_kv_heads"],
                 s["head_dim"], theta=s["theta"])
        mlk.swiglu(st["gate"].data_ptr(), st["up"].data_ptr(), st["ffn"].data_ptr(),
                   T * s["hidden_dim"])
        return st["x"], st["y"], st["q"], st["k"], st["ffn"]
    if kind == "layer":
        cfg, pos = st["cfg"], st["pos"]
        _gather(mlk, case["type"], st["table"], cfg["vocab"], cfg["dim"], st["ids"], T, st["x"])
        fwd.forward_layer_batch(cfg, st["lw"], st["x"].data_ptr(), T, st["k"].data_ptr(),
                                st["v"].data_ptr(), 1, st["k"].shape[1], 0, st["max_ctx"],
                                st["ws"], positions=None if pos is None else pos.data_ptr(),
                                pos0=case["pos0"] if pos is None else 0)
        return st["x"], st["k"], st["v"]
    if kind == "linear":
        if case["layout"] == "planar":
            mlk.linear_planar(case["type"], st["x"].data_ptr(), st["planar"].data_ptr(),
                              st["y"].data_ptr(), T, st["x"].shape[1], st["y"].shape[1])
        else:
            _linear(mlk, case["type"], st["x"], st["w"], st["y"])
        return st["y"]
    if kind == "head":
        K = st["x"].shape[1]
        mlk.rmsnorm(st["x"].data_ptr(), st["g"].data_ptr(), st["h"].data_ptr(), T, K, EPS)
        _linear(mlk, case["type"], st["h"], st["w"], st["y"])
        return st["y"]
    return st["model"].forward(st["tokens"], all_logits=True)


# ------------------------------------------------------------------ what it cannot do without

def _weight_bytes(wt, o, i):
    return 4 * o * i if wt == "f32" else o * -(-i // QK) * BLOCK_BYTES[wt]


def _layer_work(s, wt, T, ctx, pairs):
    """Bytes and flops of one layer on T tokens, `ctx` cache rows read or written, `pairs` (token,
    attended position) pairs."""
    mats = _projections(s).values()
    rows = s["n_kv_heads"] * s["head_dim"]
    return (sum(_weight_bytes(wt, o, i) for o, i in mats) + 8 * s["dim"] + 8 * ctx * rows
            + 4 * T * s["dim"] + 8 * T * rows,
            sum(2 * T * o * i for o, i in mats) + 4 * s["head_dim"] * s["n_heads"] * pairs)


def work(case):
    kind, T = case["kind"], case["tokens"]
    if kind == "chain":
        s, wt = SHAPES[case["shape"]], case["table"]
        D, F = s["dim"], s["hidden_dim"]
        qk = (s["n_heads"] + s["n_kv_heads"]) * s["head_dim"]
        # table rows, ids; delta; x and y written; q and k in place; gate, up, ffn
        return {"bytes": T * (_weight_bytes(wt, 1, D) + 4) + 12 * T * D + 4 * D + 8 * T * qk
                + 12 * T * F, "flops": T * (6 * D + 3 * qk + 6 * F)}
    if kind == "layer":
        s, wt = SHAPES[case["shape"]], case["type"]
        if case["decode"]:  # positions spread evenly below the last
            ctx, pairs = case["pos0"] + 1, int((T + 1) / 2 * (case["pos0"] + 1)) if T > 1 else \
                case["pos0"] + 1
        else:
            ctx, pairs = case["pos0"] + T, T * case["pos0"] + T * (T + 1) // 2
        b, f = _layer_work(s, wt, T, ctx, pairs)
        return {"bytes": b + T * (_weight_bytes(wt, 1, s["dim"]) + 4), "flops": f}
    if kind in ("linear", "head"):
        s = SHAPES[case["shape"]]
        o, i = (s["vocab"], s["dim"]) if kind == "head" else _projections(s)[case["proj"]]
        return {"bytes": _weight_bytes(case["type"], o, i) + 4 * T * (o + i),
                "flops": 2 * T * o * i}
    b, f = _layer_work(case, case["type"], T, T, T * (T + 1) // 2)
    D = case["dim"]
    return {"bytes": case["layers"] * b + _weight_bytes(case["type"], 131, D) + 4 * T * (D + 131),
            "flops": case["layers"] * f + 2 * T * 131 * D}


def tolerance(case):
    # fp32 everywhere, four times the error measured against `exact`: the chain's ops round once or
    # twice (5e-8); a projection's sums over 4096..28672 fp32 products are up to 2.1e-6 off, the
    # logits' 1.1e-6, a small model's 6e-7, a layer's output (attention and seven projections)
    # 0.8e-6 to 3.3e-6.
    return {"rel": {"chain": 2e-7, "linear": 8e-6, "head": 4.5e-6, "model": 2.5e-6,
                    "layer": 1.3e-5}[case["kind"]]}


# ------------------------------------------------------------------ 64 bits, plain torch

def _rms64(x, g):
    return x * g.double() / torch.sqrt(x.square().mean(-1, keepdim=True) + EPS)


def _rope64(x, pos, theta):
    """x [T, heads, hd], pairs (2i, 2i + 1)."""
    hd = x.shape[-1]
    f = theta ** (-torch.arange(0, hd, 2, device=x.device, dtype=torch.float64) / hd)
    a = pos.double()[:, None, None] * f
    c, s = torch.cos(a), torch.sin(a)
    e, o = x[..., 0::2], x[..., 1::2]
    return torch.stack([e * c - o * s, e * s + o * c], -1).flatten(-2)


def _matmul64(x, w, wt):
    """x [T, in] (float64) with the weight [out, in], a part of the rows at a time."""
    o, step = w.shape[0], max(1, (1 << 28) // x.shape[1])
    return torch.cat([x @ _weight64(w[r:r + step], wt, x.shape[1]).T for r in range(0, o, step)],
                     1)


def _layer64(s, wt, w, g1, g2, x, k, v, pos, eps=EPS):
    """One layer over x [T, dim] (float64) at positions pos; k and v are the caches [slots, KV, hd]
    (float64, updated in place)."""
    T, H, KV, hd = x.shape[0], s["n_heads"], s["n_kv_heads"], s["head_dim"]
    h = _rms64(x, g1)
    q = _rope64(_matmul64(h, w["wq"], wt).view(T, H, hd), pos, s["theta"])
    k[pos] = _rope64(_matmul64(h, w["wk"], wt).view(T, KV, hd), pos, s["theta"])
    v[pos] = _matmul64(h, w["wv"], wt).view(T, KV, hd)
    ctx = int(pos.max()) + 1
    future = torch.arange(ctx, device=x.device)[None, :] > pos[:, None]
    a = torch.empty_like(q)
    for i in range(H):
        kv = i // (H // KV)
        sc = (q[:, i] @ k[:ctx, kv].T.contiguous()) / math.sqrt(hd)
        a[:, i] = torch.softmax(sc.masked_fill(future, -math.inf), -1) @ v[:ctx, kv].contiguous()
    x = x + _matmul64(a.reshape(T, H * hd), w["wo"], wt)
    h = _rms64(x, g2)
    gate = _matmul64(h, w["w_gate"], wt)
    f = gate * torch.sigmoid(gate) * _matmul64(h, w["w_up"], wt)
    return x + _matmul64(f, w["w_down"], wt)


def exact(case, seed):
    kind, T = case["kind"], case["tokens"]
    if kind == "chain":
        d, s = _chain_inputs(case, seed), SHAPES[case["shape"]]
        pos = torch.arange(T, device=DEV)
        x = _weight64(d["table"][d["ids"].long()], case["table"], s["dim"]) + d["delta"].double()
        g = d["gate"].double()
        return (x, _rms64(x, d["w"]), _rope64(d["q"].double(), pos, s["theta"]),
                _rope64(d["k"].double(), pos, s["theta"]), g * torch.sigmoid(g) * d["up"].double())
    if kind == "layer":
        d, s, wt = _layer_inputs(case, seed), SHAPES[case["shape"]], case["type"]
        pos = d["pos"].long() if d["pos"] is not None else \
            case["pos0"] + torch.arange(T, device=DEV)
        x = _weight64(d["table"][d["ids"].long()], wt, s["dim"])
        k, v = d["k"][0].double(), d["v"][0].double()
        x = _layer64(s, wt, d["w"], d["g1"], d["g2"], x, k, v, pos)
        return x, k[None], v[None]
    if kind in ("linear", "head"):
        d = _linear_inputs(case, seed)
        x = d["x"].double()
        return _matmul64(_rms64(x, d["g"]) if kind == "head" else x, d["w"], case["type"])
    model, tokens = _model_inputs(case, seed)
    c, wt = model["config"], case["type"]
    t = torch.from_numpy
    pos = torch.arange(T)
    x = t(model["embedding"])[t(tokens).long()].double()
    for lw in model["layers"]:
        k = torch.zeros((T, c["n_kv_heads"], c["head_dim"]), dtype=torch.float64)
        v = torch.zeros_like(k)
        w = {n: t(lw[n][1]) for n in _projections(c)}
        x = _layer64(c, wt, w, t(lw["attention_norm"]), t(lw["ffn_norm"]), x, k, v, pos)
    return _matmul64(_rms64(x, t(model["final_norm"])), t(model["lm_head"][1]), wt)
