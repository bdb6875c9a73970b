"""What this engine is measured on: the calls a serving program makes, through the public entry
points of qwen35 (include/q35.h), from one request on an idle GPU to full batches.

Sizes come from the benchmark configurations: the 24-layer text tower (hidden 1024, intermediate
3584, vocabulary 248320), decode attention over 1,024 .. 32,768 slots at 1 .. 256 lanes, the
GatedDeltaNet step at 1 .. 1,024 lanes, the projections at 1 .. 2,048 rows, prompts of up to
4,096 tokens. Weights are the seeded random-init ones (N(0, 0.02)), activations N(0, 1),
recurrent states N(0, 0.1) and K/V caches N(0, 1), as in bench.py.

One engine (weights, scratch, stream) serves every case, as one does in a server.
"""
import functools
import math
import sys
from pathlib import Path

import numpy as np
import torch

PKG = str(Path(__file__).resolve().parents[1] / "qwen3.5-0.8b_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

from qwen35 import Engine, State  # noqa: E402

HIDDEN, FF, VOCAB = 1024, 3584, 248320
LAYERS, GDN_LAYERS = 24, 18
GDN_IN, ATTN_IN = 8224, 5120          # columns of the fused input projections
MAX_ROWS, MAX_CTX = 2048, 33024       # rows of one body pass; largest cache of any state
WEIGHT_BYTES = 1_504_793_280          # bf16 weights of the text tower, the tied embedding once
LM = "model.language_model."
DEV = "cuda"


# ------------------------------------------------------------------------------ the cases
def listed():
    return [
        # One user chatting: a greedy step of one lane whose host samples from the logits.
        {"name": "decode_1x4096", "kind": "decode", "lanes": 1, "ctx": 4096},
        # Time to first token of a long document: two full waves of the engine's rows.
        {"name": "prefill_4096", "kind": "prefill", "tokens": 4096},
        # One attention layer of a decode step: one long conversation; a server's mixed
        # conversations of many lengths; the headline batch; the 3 rows a lane's speculative
        # round verifies at once.
        {"name": "attn_1x8192", "kind": "attn", "lanes": 1, "ctx": 8192, "rows": 1, "ragged": False},
        {"name": "attn_32x8192_ragged", "kind": "attn", "lanes": 32, "ctx": 8192, "rows": 1, "ragged": True},
        {"name": "attn_256x4096", "kind": "attn", "lanes": 256, "ctx": 4096, "rows": 1, "ragged": False},
        {"name": "verify_128x2000_ragged", "kind": "attn", "lanes": 128, "ctx": 2000, "rows": 3, "ragged": True},
        # One GatedDeltaNet layer's step (conv, gates, delta rule, gated norm) of one request and
        # of the largest batch of the configurations.
        {"name": "gdn_1", "kind": "gdn", "lanes": 1},
        {"name": "gdn_1024", "kind": "gdn", "lanes": 1024},
        # One SwiGLU MLP: one request's step, the headline batch, a prompt wave of odd length.
        {"name": "mlp_1", "kind": "mlp", "rows": 1},
        {"name": "mlp_256", "kind": "mlp", "rows": 256},
        {"name": "mlp_1999", "kind": "mlp", "rows": 1999},
        # The tied head with its greedy ids and logits for the headline batch.
        {"name": "head_256", "kind": "head", "rows": 256},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "prefill", "attn", "attn", "verify", "gdn", "mlp", "mlp", "head"])
    if kind == "decode":
        return {"kind": kind, "lanes": _log_int(rng, 1, 8), "ctx": _log_int(rng, 64, 8192)}
    if kind == "prefill":
        return {"kind": kind, "tokens": _log_int(rng, 16, 4095)}
    if kind in ("attn", "verify"):
        lanes = _log_int(rng, 1, 256)
        rows = 1 if kind == "attn" else rng.choice([2, 3])
        ctx = _log_int(rng, 64, min(32768, (1 << 20) // (lanes * rows)))
        return {"kind": "attn", "lanes": lanes, "ctx": ctx, "rows": rows, "ragged": rng.random() < 0.5}
    if kind == "gdn":
        return {"kind": kind, "lanes": _log_int(rng, 2, 1023)}
    if kind == "mlp":
        return {"kind": kind, "rows": _log_int(rng, 2, 2048)}
    return {"kind": kind, "rows": _log_int(rng, 1, 512)}


# ------------------------------------------------------------------------------ inputs
@functools.lru_cache(maxsize=None)
def engine():
    torch.zeros(1, device=DEV)        # torch's runtime first: it makes the buffers
    return Engine(max_rows=MAX_ROWS, max_ctx=MAX_CTX, seed=0, use_graph=True)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _bf16(g, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(torch.bfloat16)


def _tiled(eng, w):
    t = torch.empty_like(w)
    torch.cuda.synchronize()
    eng.op_tile_weight(w.data_ptr(), w.shape[0], w.shape[1], t.data_ptr())
    eng.sync()
    return t


def _positions(case):
    """The lanes' context lengths: all the same, or spread evenly from an eighth of it up."""
    n, c = case["lanes"], case["ctx"]
    if not case["ragged"]:
        return np.full(n, c, np.int32)
    return np.array([c - (i * (c - c // 8)) // n for i in range(n)], np.int32)


def prepare(case, seed):
    eng, kind = engine(), case["kind"]
    s = {"case": case, "eng": eng}
    g = _gen(seed)
    if kind == "decode":
        # room for the steps of a long answer; a lane that fills up starts over (run)
        s["st"] = State(eng, case["lanes"], case["ctx"] + 4096)
        s["st"].seed(seed, case["ctx"])
        s["seed"], s["left"] = seed, 4096
        s["tok"] = np.random.default_rng(seed).integers(0, VOCAB, case["lanes"]).astype(np.int32)
    elif kind == "prefill":
        s["st"] = State(eng, 1, case["tokens"] + 64)
        s["ids"] = np.random.default_rng(seed).integers(0, VOCAB, case["tokens"]).astype(np.int32)
    elif kind == "attn":
        n, T = case["lanes"], case["rows"]
        s["st"] = State(eng, n, case["ctx"] + 16)
        s["st"].seed(seed, case["ctx"])
        s["lanes"] = np.arange(n, dtype=np.int32)
        s["pos"] = np.random.default_rng(seed).permutation(_positions(case)).astype(np.int32)
        s["layer"] = int(seed) % 6
        s["proj"] = _bf16(g, n * T, ATTN_IN)
        s["qn"], s["kn"] = _bf16(g, 256, scale=0.1), _bf16(g, 256, scale=0.1)
        s["out"] = torch.empty(n * T, 2048, dtype=torch.bfloat16, device=DEV)
    elif kind == "gdn":
        n = case["lanes"]
        s["proj"] = _bf16(g, n, GDN_IN)
        s["conv"] = _bf16(g, 6144, 4, scale=0.3)
        s["A"] = (1 + 15 * torch.rand(16, generator=g, device=DEV)).log().to(torch.bfloat16)
        s["dt"] = (2 * torch.rand(16, generator=g, device=DEV) - 1).to(torch.bfloat16)
        s["gn"] = (1 + 0.25 * torch.randn(128, generator=g, device=DEV)).to(torch.bfloat16)
        # two state slots per lane: 0 the state before the step, 1 the state after it
        s["S"] = torch.empty(n, 2, 16, 128, 128, device=DEV)
        s["S"].normal_(0, 0.1, generator=g)
        s["W"] = _bf16(g, n, 2, 3, 6144).float()
        s["o"] = torch.empty(n, 2048, device=DEV)
        s["y"] = torch.empty(n, 2048, dtype=torch.bfloat16, device=DEV)
    elif kind == "mlp":
        m = case["rows"]
        s["gu_w"], s["down_w"] = _bf16(g, 2 * FF, HIDDEN, scale=0.02), _bf16(g, HIDDEN, FF, scale=0.02)
        s["gu_t"], s["down_t"] = _tiled(eng, s["gu_w"]), _tiled(eng, s["down_w"])
        s["x"] = _bf16(g, m, HIDDEN)
        s["mid"] = torch.empty(m, 2 * FF if m <= 16 else FF, dtype=torch.bfloat16, device=DEV)
        s["y"] = torch.empty(m, HIDDEN, dtype=torch.bfloat16, device=DEV)
    else:
        m = case["rows"]
        s["x"] = _bf16(g, m, HIDDEN)
        s["tok"] = torch.empty(m, dtype=torch.int32, device=DEV)
        s["logits"] = torch.empty(m, VOCAB, device=DEV)
    torch.cuda.synchronize()          # the engine's stream reads what torch's stream has made
    return s


# ------------------------------------------------------------------------------ one pass
def run(s):
    case, eng = s["case"], s["eng"]
    kind = case["kind"]
    if kind == "decode":
        if s["left"] == 0:
            s["st"].seed(s["seed"], case["ctx"])
            s["left"] = 4096
        s["left"] -= 1
        s["tok"], logits = s["st"].decode_step(s["tok"], logits=True)
        return logits
    if kind == "prefill":
        s["st"].reset()
        return s["st"].prefill(0, s["ids"], logits=True)[1]
    if kind == "attn":
        eng.op_attn_decode(s["st"], s["layer"], s["lanes"], s["pos"], case["rows"], s["proj"].data_ptr(),
                           s["qn"].data_ptr(), s["kn"].data_ptr(), s["out"].data_ptr())
        return s["out"]
    if kind == "gdn":
        eng.op_gdn_step_norm(*[s[k].data_ptr() for k in ("proj", "conv", "A", "dt", "gn", "S", "W", "o", "y")],
                             case["lanes"])
        return {"y": s["y"], "o": s["o"], "state": s["S"], "window": s["W"]}
    m = case["rows"]
    if kind == "mlp":
        x, mid, y = s["x"].data_ptr(), s["mid"].data_ptr(), s["y"].data_ptr()
        if m <= 16:      # gate | up stored, SwiGLU in the down projection's A operand
            eng.op_gemm(s["gu_t"].data_ptr(), 2 * FF, HIDDEN, x, m, mid)
            eng.op_gemm_a(s["down_t"].data_ptr(), HIDDEN, FF, 1, mid, 2 * FF, mid + 2 * FF, 2 * FF, 0, m, y)
        else:            # SwiGLU in the gate | up epilogue (6: the many-row kernel), then down
            eng.op_gemm_a(s["gu_t"].data_ptr(), 2 * FF, HIDDEN, 5 if m < 512 else 6, x, HIDDEN, 0, 0, 0, m, mid)
            eng.op_gemm(s["down_t"].data_ptr(), HIDDEN, FF, mid, m, y)
        return {"y": s["y"], "mid": s["mid"]}
    eng.op_lm_head_argmax(s["x"].data_ptr(), m, s["tok"].data_ptr(), s["logits"].data_ptr())
    return {"logits": s["logits"], "tok": s["tok"]}


# ------------------------------------------------------------------------------ floors, tolerances
def work(case):
    """Bytes and operations of one pass: inputs read once, outputs written once."""
    kind = case["kind"]
    if kind == "decode":
        n, c = case["lanes"], case["ctx"]
        state = GDN_LAYERS * 2 * (16 * 128 * 128 * 4 + 3 * 6144 * 4) + 12288 * c
        return {"bytes": WEIGHT_BYTES + n * (state + 4 * VOCAB),
                "flops": n * (WEIGHT_BYTES + 6 * 4 * 8 * 256 * c + GDN_LAYERS * 16 * 8 * 128 * 128)}
    if kind == "prefill":
        t = case["tokens"]
        tower = WEIGHT_BYTES - 2 * VOCAB * HIDDEN
        return {"bytes": WEIGHT_BYTES + 12288 * t + 4 * VOCAB + GDN_LAYERS * (1 << 20),
                "flops": t * tower + 2 * VOCAB * HIDDEN + 6 * 2 * 8 * 256 * t * t + t * GDN_LAYERS * 16 * 8 * 128 * 128}
    if kind == "attn":
        T, pos = case["rows"], _positions(case).astype(np.float64)
        return {"bytes": float((pos * 2048).sum()) + len(pos) * T * (2 * ATTN_IN + 2 * 2048 + 2048),
                "flops": float(((pos + T) * T * 4 * 8 * 256).sum())}
    if kind == "gdn":
        n = case["lanes"]
        return {"bytes": n * (2 * 16 * 128 * 128 * 4 + 2 * 3 * 6144 * 4 + 2 * GDN_IN + 4 * 2048 + 2 * 2048),
                "flops": n * 16 * 8 * 128 * 128}
    m = case["rows"]
    if kind == "mlp":
        return {"bytes": 2 * 3 * FF * HIDDEN + 2 * m * (2 * HIDDEN + (2 * FF if m <= 16 else FF)),
                "flops": 2 * m * 3 * FF * HIDDEN}
    return {"bytes": 2 * VOCAB * HIDDEN + m * (2 * HIDDEN + 4 * VOCAB + 4), "flops": 2 * m * VOCAB * HIDDEN}


def tolerance(case):
    """Whole calls: the prompt's exact form against its default one (the same sums in another
    order, measured) moves the logits by 0.025 .. 0.043, every rounding to bf16 in 24 layers
    shifting a little; less is stated. Layers: four times and less what bf16 results (1.7e-3 from
    64 bits; sums in another order flip few of them) and the attention's bf16 weights (3.3e-3)
    give; the delta rule's state and output are 32-bit and within 6e-7, but travel with y."""
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        return {"rel": 0.03}
    if kind == "attn":
        return {"rel": 8e-3}
    return {"rel": 1e-3, "max": 0.02} if kind == "gdn" else {"rel": 2e-3, "max": 0.03, "differ": 0.01}


# ------------------------------------------------------------------------------ the same in 64 bits
def _f64(a):
    """bf16 bits (uint16) or any array -> float64 on the GPU."""
    if a.dtype == np.uint16:
        return torch.from_numpy(a.view(np.int16)).to(DEV).view(torch.bfloat16).double()
    return torch.from_numpy(a).to(DEV).double()


def _round(x):
    return x.to(torch.bfloat16).double()


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * w


def _silu(x):
    return x * torch.sigmoid(x)


def _rope(x, pos):
    """The first 64 of 256 dims in pairs (i, i + 32), angles pos * f32(1e7 ** (-i / 32)) in f32."""
    inv = 1.0 / (1e7 ** (2 * torch.arange(32, dtype=torch.float32, device=DEV) / 64))
    ang = (pos.float()[:, None] * inv).double()
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., :32], x[..., 32:64]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., 64:]], -1)


def _attend(qg, k, v, qw, kw, K, V, pos, stored=lambda x: x):
    """T rows at pos .. pos + T - 1 over the cache K, V [2][pos][256] and themselves; stored:
    the rounding of what the layer keeps in bf16 (the normed q and k, the cached k)."""
    T = qg.shape[0]
    at = pos + torch.arange(T, device=DEV)
    q, gate = qg.view(T, 8, 512).split(256, -1)
    q = _rope(stored(_rms(q, 1 + qw)), at)
    k = stored(_rope(stored(_rms(k.view(T, 2, 256), 1 + kw)), at))
    K, V = torch.cat([K, k.transpose(0, 1)], 1), torch.cat([V, v.view(T, 2, 256).transpose(0, 1)], 1)
    hide = torch.arange(K.shape[1], device=DEV)[None] > at[:, None]
    out = torch.empty(T, 8, 256, dtype=torch.float64, device=DEV)
    for h in range(8):
        sc = (q[:, h] @ K[h // 4].t() / 16).masked_fill_(hide, -math.inf)
        out[:, h] = sc.softmax(-1) @ V[h // 4]
    return (out * torch.sigmoid(gate)).reshape(T, 2048)


def _gates(a, b, A, dt):
    return torch.exp(-A.exp() * torch.nn.functional.softplus(a + dt)), torch.sigmoid(b)


def _unit(x):
    return x * torch.rsqrt(x.square().sum(-1, keepdim=True) + 1e-6)


def _delta(S, q, k, v, decay, beta):
    """One row per entry of the leading dims: S [..., 16, 128, 128] <- the delta rule; o = S^T q."""
    S = S * decay[..., None, None]
    dv = beta[..., None] * (v - (S * k[..., None]).sum(-2))
    S = S + k[..., None] * dv[..., None, :]
    return S, (S * q[..., None]).sum(-2)


@functools.lru_cache(maxsize=1)
def _weights():
    """The engine's weights, read back in checkpoint layout."""
    eng, w = engine(), {}

    def rd(name, *shape):
        w[name] = _f64(eng.read_tensor(LM + name, int(np.prod(shape)))).view(*shape)

    rd("embed_tokens.weight", VOCAB, HIDDEN)
    rd("norm.weight", HIDDEN)
    for l in range(LAYERS):
        p = f"layers.{l}."
        rd(p + "input_layernorm.weight", HIDDEN)
        rd(p + "post_attention_layernorm.weight", HIDDEN)
        if l % 4 == 3:
            p += "self_attn."
            for n, r in (("q_proj", 4096), ("k_proj", 512), ("v_proj", 512)):
                rd(p + n + ".weight", r, HIDDEN)
            rd(p + "q_norm.weight", 256)
            rd(p + "k_norm.weight", 256)
            rd(p + "o_proj.weight", HIDDEN, 2048)
        else:
            p += "linear_attn."
            for n, r in (("qkv", 6144), ("z", 2048), ("b", 16), ("a", 16)):
                rd(p + f"in_proj_{n}.weight", r, HIDDEN)
            rd(p + "conv1d.weight", 6144, 4)
            rd(p + "A_log", 16)
            rd(p + "dt_bias", 16)
            rd(p + "norm.weight", 128)
            rd(p + "out_proj.weight", HIDDEN, 2048)
        for n, r, c in (("gate", FF, HIDDEN), ("up", FF, HIDDEN), ("down", HIDDEN, FF)):
            rd(f"layers.{l}.mlp.{n}_proj.weight", r, c)
    return w


def _tower(ids, S, win, K, V, pos):
    """Logits after the last of `ids`, from S [18][16][128][128], win [18][3][6144] and the
    caches K, V [6][2][pos][256] of one lane."""
    w = _weights()
    T = len(ids)
    x = w["embed_tokens.weight"][torch.from_numpy(np.asarray(ids, np.int64)).to(DEV)]
    for l in range(LAYERS):
        p = f"layers.{l}."
        h = _rms(x, 1 + w[p + "input_layernorm.weight"])
        if l % 4 == 3:
            a = p + "self_attn."
            h = _attend(*[h @ w[a + n + "_proj.weight"].t() for n in "qkv"], w[a + "q_norm.weight"],
                        w[a + "k_norm.weight"], K[l // 4], V[l // 4], pos) @ w[a + "o_proj.weight"].t()
        else:
            a, j = p + "linear_attn.", l - (l + 1) // 4
            raw, z, b, aa = (h @ w[a + f"in_proj_{n}.weight"].t() for n in ("qkv", "z", "b", "a"))
            ext = torch.cat([win[j], raw])
            u = _silu(sum(ext[i:i + T] * w[a + "conv1d.weight"][:, i] for i in range(4)))
            q, k, v = (t.reshape(T, 16, 128) for t in u.split(2048, -1))
            q, k = _unit(q) / math.sqrt(128), _unit(k)
            decay, beta = _gates(aa, b, w[a + "A_log"], w[a + "dt_bias"])
            st, o = S[j], torch.empty_like(v)
            for t in range(T):
                st, o[t] = _delta(st, q[t], k[t], v[t], decay[t], beta[t])
            y = _rms(o, w[a + "norm.weight"]) * _silu(z.view(T, 16, 128))
            h = y.reshape(T, 2048) @ w[a + "out_proj.weight"].t()
        x = x + h
        h = _rms(x, 1 + w[p + "post_attention_layernorm.weight"])
        m = p + "mlp."
        x = x + (_silu(h @ w[m + "gate_proj.weight"].t()) * (h @ w[m + "up_proj.weight"].t())) @ w[m + "down_proj.weight"].t()
    return _rms(x[-1], 1 + w["norm.weight"]) @ w["embed_tokens.weight"].t()


def exact(case, seed):
    kind = case["kind"]
    if kind == "attn" and case["lanes"] * case["ctx"] > 1 << 18:
        return None                   # reading the caches back alone takes over 20 seconds
    s = prepare(case, seed)
    if kind == "decode":
        rows = []
        for l in range(case["lanes"]):
            K, V = (_f64(s["st"].read(l, n, case["ctx"])) for n in "kv")
            rows.append(_tower(s["tok"][l:l + 1], _f64(s["st"].read(l, "S")), _f64(s["st"].read(l, "win")), K, V,
                               case["ctx"]))
        return torch.stack(rows)
    if kind == "prefill":
        z = functools.partial(torch.zeros, dtype=torch.float64, device=DEV)
        return _tower(s["ids"], z(GDN_LAYERS, 16, 128, 128), z(GDN_LAYERS, 3, 6144), z(6, 2, 0, 256), z(6, 2, 0, 256), 0)
    if kind == "attn":
        T, rows = case["rows"], []
        for i, p in enumerate(s["pos"]):
            K, V = (_f64(s["st"].read(i, n, int(p))[s["layer"]]) for n in "kv")
            x = s["proj"][i * T:(i + 1) * T].double()
            rows.append(_attend(x[:, :4096], x[:, 4096:4608], x[:, 4608:], s["qn"].double(), s["kn"].double(), K, V,
                                int(p), _round))
        return torch.cat(rows)
    if kind == "gdn":
        n = case["lanes"]
        W, proj = s["W"].double(), s["proj"].double()
        ext = torch.cat([W[:, 0], proj[:, None, :6144]], 1)
        u = _round(_silu(_round((ext * s["conv"].double().t()).sum(1))))     # the conv and its SiLU are kept in bf16
        q, k, v = (t.reshape(n, 16, 128) for t in u.split(2048, -1))
        decay, beta = _gates(proj[:, 8208:], proj[:, 8192:8208], s["A"].double(), s["dt"].double())
        W[:, 1] = ext[:, 1:]
        S, o, y = s["S"].double(), [], []
        for b in range(0, n, 64):
            e = min(n, b + 64)
            S[b:e, 1], ob = _delta(S[b:e, 0], _unit(q[b:e]) / math.sqrt(128), _unit(k[b:e]), v[b:e], decay[b:e], beta[b:e])
            o.append(ob.reshape(e - b, 2048))
            y.append((_rms(ob, s["gn"].double()) * _silu(proj[b:e, 6144:8192].view(-1, 16, 128))).reshape(e - b, 2048))
        return {"y": torch.cat(y), "o": torch.cat(o), "state": S, "window": W}
    x = s["x"].double()
    if kind == "mlp":
        gu = x @ s["gu_w"].double().t()
        act = _round(_round(_silu(_round(gu[:, :FF]))) * _round(gu[:, FF:]))  # silu and the product are kept in bf16
        return {"y": act @ s["down_w"].double().t(), "mid": gu if case["rows"] <= 16 else act}
    return {"logits": x @ _f64(engine().read_tensor(LM + "embed_tokens.weight", VOCAB * HIDDEN)).view(VOCAB, HIDDEN).t(),
            "tok": None}
