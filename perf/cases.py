"""The work that programs have this framework do, as cases that can be timed
and compared: the blocks of a quantized Qwen3 layer at decode, verify and
prefill sizes through the package's operators (MLP, attention over a KV
cache, vocabulary head with greedy argmax), a routed-expert MLP, and whole
forwards and decode steps of a small-depth model loaded from an MLX
checkpoint.

Weights are MLX affine 4-bit (group size 64) quantizations of N(0, 0.02)
matrices, activations bf16.  `exact` repeats each case in float64 with plain
torch.
"""
import json
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "base-mlx_amd"))
import bmx  # noqa: E402

HEAD_DIM = 128
EPS, THETA = 1e-6, 1e6
VOCAB = 151936
MODEL_VOCAB = 4096  # the whole-model cases: the head has cases of its own
WS_TOKENS = 16      # widest decode / verify call a program sizes its attention workspace for
# the shapes the package names (dims of one layer)
SHAPES = {"0.6b": bmx.QWEN3_0_6B, "4b": bmx.QWEN3_4B, "8b": bmx.QWEN3_8B, "32b": bmx.QWEN3_32B}
# routed experts of the benchmark: 128 experts, top 8, gate|up concatenated
MOE_E, MOE_TOPK, MOE_HIDDEN, MOE_INTER = 128, 8, 2048, 768
MOST_FLOPS = 3.4e11  # of a drawn case: the largest listed ones


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------
def listed():
    return [
        {"name": "head_verify5", "kind": "head", "shape": "4b", "M": 5},
        {"name": "mlp_32b_verify5", "kind": "mlp", "shape": "32b", "M": 5},
        {"name": "mlp_4b_prompt37", "kind": "mlp", "shape": "4b", "M": 37},
        {"name": "mlp_8b_prompt200", "kind": "mlp", "shape": "8b", "M": 200},
        {"name": "mlp_4b_prefill2048", "kind": "mlp", "shape": "4b", "M": 2048},
        {"name": "attn_4b_decode", "kind": "attn", "shape": "4b", "M": 1, "past": 4096},
        {"name": "attn_8b_chunk203", "kind": "attn", "shape": "8b", "M": 203, "past": 3000},
        {"name": "attn_4b_prefill4096", "kind": "attn", "shape": "4b", "M": 4096, "past": 0},
        {"name": "moe_decode", "kind": "moe", "T": 1},
        {"name": "moe_prefill333", "kind": "moe", "T": 333},
        {"name": "model_prompt77", "kind": "forward", "shape": "4b", "M": 77, "past": 0, "all_logits": False},
        {"name": "model_decode", "kind": "decode", "shape": "4b", "past": 4096},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["head", "mlp", "mlp", "mlp", "attn", "attn", "moe", "forward", "decode"])
    if kind == "moe":
        return {"kind": kind, "T": _log_int(rng, 1, 333)}
    if kind == "head":
        return {"kind": kind, "shape": rng.choice(["0.6b", "4b", "8b"]), "M": _log_int(rng, 1, 64)}
    if kind == "mlp":
        s = rng.choice(sorted(SHAPES))
        per_row = 6.0 * SHAPES[s]["hidden"] * SHAPES[s]["inter"]
        return {"kind": kind, "shape": s, "M": _log_int(rng, 1, min(4096, int(MOST_FLOPS / per_row)))}
    if kind == "attn":
        s = rng.choice(sorted(SHAPES))
        c = {"kind": kind, "shape": s, "M": _log_int(rng, 1, 4096), "past": rng.choice([0, _log_int(rng, 64, 4096)])}
        while work(c)["flops"] > MOST_FLOPS:
            c["M"] -= c["M"] // 4
        return c
    s = rng.choice(["0.6b", "4b"])
    if kind == "forward":
        verify = rng.random() < 0.3
        return {"kind": kind, "shape": s, "M": rng.randint(2, 8) if verify else _log_int(rng, 9, 1024),
                "past": _log_int(rng, 64, 2048) if verify else 0, "all_logits": verify}
    return {"kind": kind, "shape": s, "past": _log_int(rng, 64, 4096)}


def _model_dims(shape):
    return dict(SHAPES[shape], layers=2, vocab=MODEL_VOCAB, tied=1)


def _qbytes(n, k):
    return 0.5625 * n * k


def _attn_work(d, M, past):
    """(weights, flops, KV and activation bytes) of one attention block"""
    H, hq, hkv = d["hidden"], d["n_heads"] * HEAD_DIM, d["n_kv_heads"] * HEAD_DIM
    n = H * (2 * hq + 2 * hkv)
    keys = M * past + M * (M + 1) / 2.0  # visible (query, key) pairs
    return n, 2.0 * M * n + 4.0 * keys * hq, 4.0 * (past + M) * hkv


def work(case):
    k = case["kind"]
    if k == "moe":
        T = case["T"]
        used = MOE_E * (1.0 - (1.0 - MOE_TOPK / MOE_E) ** T)
        per = 3 * MOE_HIDDEN * MOE_INTER
        return {"bytes": used * _qbytes(1, per) + 2.0 * T * MOE_HIDDEN * (1 + MOE_TOPK),
                "flops": 2.0 * T * MOE_TOPK * per}
    d = SHAPES[case["shape"]]
    H, I = d["hidden"], d["inter"]
    if k == "head":
        return {"bytes": _qbytes(VOCAB, H) + 2.0 * case["M"] * (H + VOCAB), "flops": 2.0 * case["M"] * VOCAB * H}
    if k == "mlp":
        return {"bytes": _qbytes(3 * I, H) + 4.0 * case["M"] * H, "flops": 6.0 * case["M"] * I * H}
    if k == "attn":
        n, fl, kv = _attn_work(d, case["M"], case["past"])
        return {"bytes": _qbytes(1, n) + kv + 4.0 * case["M"] * H, "flops": fl}
    M = case.get("M", 1)
    n, fl, kv = _attn_work(d, M, case["past"])
    rows = M if case.get("all_logits") else 1
    return {"bytes": 2 * (_qbytes(1, n) + _qbytes(3 * I, H) + kv) + _qbytes(MODEL_VOCAB, H) + 2.0 * rows * MODEL_VOCAB,
            "flops": 2 * (fl + 6.0 * M * I * H) + 2.0 * rows * MODEL_VOCAB * H}


# About four times the error against float64 that bf16 results and
# intermediates leave: 0.0029 (head), 0.0042-0.0056 (expert and plain MLP),
# up to 0.0048 (attention: its K / V rows and the residual sum), 0.013-0.015
# (two whole layers and the head, where each rounding travels on; at most 0.03)
_REL = {"head": 0.012, "mlp": 0.02, "moe": 0.016, "attn": 0.016, "forward": 0.03, "decode": 0.03}


def tolerance(case):
    return {"rel": _REL[case["kind"]]}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class Inputs:
    """Seeded tensors on the GPU; the same calls give the same values."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0):
        return (torch.randn(*shape, generator=self.g, device="cuda") * std + mean).to(torch.bfloat16)

    def norm_weight(self, n):
        return self.normal(n, std=0.1, mean=1.0)

    def ints(self, high, n):
        return torch.randint(0, high, (n,), generator=self.g, device="cuda", dtype=torch.int64)

    def qlinear(self, N, K, std=0.02):
        """MLX affine 4-bit quantization of an [N, K] normal matrix."""
        w = torch.empty(N, K // 8, dtype=torch.int32, device="cuda")
        s = torch.empty(N, K // 64, dtype=torch.bfloat16, device="cuda")
        b = torch.empty_like(s)
        shift = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
        step = max(1, (1 << 26) // K)
        for i in range(0, N, step):
            n = min(step, N - i)
            v = torch.randn(n, K // 64, 64, generator=self.g, device="cuda") * std
            lo, hi = v.amin(-1), v.amax(-1)
            s[i:i + n] = ((hi - lo) / 15).to(torch.bfloat16)
            b[i:i + n] = lo.to(torch.bfloat16)
            q = ((v - b[i:i + n, :, None].float()) / s[i:i + n, :, None].float()).round().clamp(0, 15).to(torch.int32)
            w[i:i + n] = (q.view(n, K // 8, 8) << shift).sum(-1, dtype=torch.int32)
        return w, s, b


def _experts(inp, N, K):
    w, s, b = inp.qlinear(MOE_E * N, K)
    return w.view(MOE_E, N, K // 8), s.view(MOE_E, N, K // 64), b.view(MOE_E, N, K // 64)


def _inputs(case, seed):
    """The tensors of an operator-level case."""
    inp, k = Inputs(seed), case["kind"]
    if k == "moe":
        T = case["T"]
        scores = torch.rand(T, MOE_E, generator=inp.g, device="cuda")
        return {"x": inp.normal(T, 1, MOE_HIDDEN),
                "routes": scores.topk(MOE_TOPK, dim=-1).indices.to(torch.int32).reshape(-1).contiguous(),
                "gate_up": _experts(inp, 2 * MOE_INTER, MOE_HIDDEN), "down": _experts(inp, MOE_HIDDEN, MOE_INTER)}
    d, M = SHAPES[case["shape"]], case["M"]
    H, I = d["hidden"], d["inter"]
    t = {"norm": inp.norm_weight(H)}
    if k == "head":
        t["head"] = inp.qlinear(VOCAB, H)
        # a trained tied head: the hidden state points at the next token's row
        ids = inp.ints(VOCAB, M)
        rows = _dequant(*(v[ids] for v in t["head"]), torch.float32)
        t["x"] = (torch.randn(M, H, generator=inp.g, device="cuda") + 25.0 * rows).to(torch.bfloat16)
        return t
    t["x"] = inp.normal(M, H)
    if k == "mlp":
        t.update(gate=inp.qlinear(I, H), up=inp.qlinear(I, H), down=inp.qlinear(H, I))
        return t
    hq, hkv = d["n_heads"] * HEAD_DIM, d["n_kv_heads"] * HEAD_DIM
    cap = _capacity(case["past"] + M)
    t.update(q=inp.qlinear(hq, H), k=inp.qlinear(hkv, H), v=inp.qlinear(hkv, H), o=inp.qlinear(H, hq),
             q_norm=inp.norm_weight(HEAD_DIM), k_norm=inp.norm_weight(HEAD_DIM),
             k_cache=torch.zeros(d["n_kv_heads"], cap, HEAD_DIM, dtype=torch.bfloat16, device="cuda"),
             v_cache=torch.zeros(d["n_kv_heads"], cap, HEAD_DIM, dtype=torch.bfloat16, device="cuda"))
    if case["past"]:
        t["k_cache"][:, :case["past"]] = inp.normal(d["n_kv_heads"], case["past"], HEAD_DIM)
        t["v_cache"][:, :case["past"]] = inp.normal(d["n_kv_heads"], case["past"], HEAD_DIM, std=0.7)
    return t


def _capacity(n):
    return (n + 8 + 255) // 256 * 256


_PROJ = [("self_attn.q_proj", "q"), ("self_attn.k_proj", "k"), ("self_attn.v_proj", "v"), ("self_attn.o_proj", "o"),
         ("mlp.gate_proj", "gate"), ("mlp.up_proj", "up"), ("mlp.down_proj", "down")]


def _model_inputs(case, seed):
    """Weights of a whole model, the cached tokens and the new ones."""
    inp, d = Inputs(seed), _model_dims(case["shape"])
    H, I, hq, hkv = d["hidden"], d["inter"], d["n_heads"] * HEAD_DIM, d["n_kv_heads"] * HEAD_DIM
    t = {"embed": inp.qlinear(MODEL_VOCAB, H, std=0.05), "final": inp.norm_weight(H), "layers": []}
    for _ in range(d["layers"]):
        t["layers"].append({
            "in_norm": inp.norm_weight(H), "post_norm": inp.norm_weight(H),
            "q_norm": inp.norm_weight(HEAD_DIM), "k_norm": inp.norm_weight(HEAD_DIM),
            "q": inp.qlinear(hq, H), "k": inp.qlinear(hkv, H), "v": inp.qlinear(hkv, H), "o": inp.qlinear(H, hq),
            "gate": inp.qlinear(I, H), "up": inp.qlinear(I, H), "down": inp.qlinear(H, I)})
    t["past"] = inp.ints(MODEL_VOCAB, case["past"]).cpu().numpy()
    t["tokens"] = inp.ints(MODEL_VOCAB, case.get("M", 1)).cpu().numpy()
    return t


def _write_checkpoint(path, d, t):
    """config.json and one safetensors shard under the MLX tensor names."""
    with open(os.path.join(path, "config.json"), "w") as f:
        json.dump({"model_type": "qwen3", "hidden_size": d["hidden"], "intermediate_size": d["inter"],
                   "num_hidden_layers": d["layers"], "num_attention_heads": d["n_heads"],
                   "num_key_value_heads": d["n_kv_heads"], "head_dim": HEAD_DIM, "vocab_size": d["vocab"],
                   "rms_norm_eps": EPS, "rope_theta": THETA, "tie_word_embeddings": True,
                   "quantization": {"group_size": 64, "bits": 4}}, f)
    named = []

    def qlinear(prefix, q):
        named.extend([(prefix + ".weight", "U32", q[0]), (prefix + ".scales", "BF16", q[1]),
                      (prefix + ".biases", "BF16", q[2])])

    qlinear("model.embed_tokens", t["embed"])
    for i, L in enumerate(t["layers"]):
        p = "model.layers.%d." % i
        for name, key in _PROJ:
            qlinear(p + name, L[key])
        for name, key in (("input_layernorm", "in_norm"), ("post_attention_layernorm", "post_norm"),
                          ("self_attn.q_norm", "q_norm"), ("self_attn.k_norm", "k_norm")):
            named.append((p + name + ".weight", "BF16", L[key]))
    named.append(("model.norm.weight", "BF16", t["final"]))
    header, at = {}, 0
    for name, kind, v in named:
        n = v.numel() * v.element_size()
        header[name] = {"dtype": kind, "shape": list(v.shape), "data_offsets": [at, at + n]}
        at += n
    text = json.dumps(header).encode()
    text += b" " * (-len(text) % 8)
    with open(os.path.join(path, "model.safetensors"), "wb") as f:
        f.write(struct.pack("<Q", len(text)))
        f.write(text)
        for _, _, v in named:
            f.write((v.view(torch.int16) if v.dtype == torch.bfloat16 else v).cpu().numpy().tobytes())


def prepare(case, seed):
    if case["kind"] in ("forward", "decode"):
        t, d = _model_inputs(case, seed), _model_dims(case["shape"])
        most = max(len(t["past"]), len(t["tokens"]), WS_TOKENS)
        with tempfile.TemporaryDirectory() as path:
            _write_checkpoint(path, d, t)
            model = bmx.Qwen3.load(path, max_tokens=most)
        cache = model.new_cache(_capacity(case["past"] + len(t["tokens"])))
        if case["past"]:
            model.forward(cache, t["past"])
        return {"case": case, "model": model, "cache": cache, "tokens": t["tokens"].astype(np.uint32)}
    t = _inputs(case, seed)
    t["case"] = case
    if case["kind"] == "attn":
        # one workspace for every call, as wide as the widest decode / verify
        t["ws"] = bmx.attention_workspace(SHAPES[case["shape"]]["n_heads"], WS_TOKENS)
    return t


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _run_mlp(t):
    h = bmx.rms_norm(t["x"], t["norm"], EPS)
    a = bmx.silu_mul(bmx.quantized_matmul(h, *t["gate"]), bmx.quantized_matmul(h, *t["up"]))
    return bmx.add(t["x"], bmx.quantized_matmul(a, *t["down"]))


def _run_attn(t):
    case = t["case"]
    M, past, rep = case["M"], case["past"], SHAPES[case["shape"]]["n_heads"] // SHAPES[case["shape"]]["n_kv_heads"]
    h = bmx.rms_norm(t["x"], t["norm"], EPS)
    q, k, v = (bmx.quantized_matmul(h, *t[n]) for n in ("q", "k", "v"))
    if M <= WS_TOKENS and M * rep <= 64:
        att = bmx.qk_norm_rope_kv_attention(q, k, v, t["q_norm"], t["k_norm"], t["k_cache"], t["v_cache"], past, EPS,
                                            THETA, workspace=t["ws"])
    else:
        qr = bmx.qk_norm_rope_kv(q, k, v, t["q_norm"], t["k_norm"], t["k_cache"], t["v_cache"], past, EPS, THETA)
        att = bmx.attention(qr, t["k_cache"], t["v_cache"], past, workspace=t["ws"])
    return {"y": bmx.add(t["x"], bmx.quantized_matmul(att, *t["o"])), "k": t["k_cache"], "v": t["v_cache"]}


def _run_moe(t):
    gu = bmx.gather_qmm(t["x"], *t["gate_up"], t["routes"], MOE_TOPK)
    a = bmx.silu_mul(gu[..., :MOE_INTER].contiguous(), gu[..., MOE_INTER:].contiguous())
    return bmx.gather_qmm(a, *t["down"], t["routes"], 1)


def run(state):
    kind = state["case"]["kind"]
    if kind == "mlp":
        return _run_mlp(state)
    if kind == "attn":
        return _run_attn(state)
    if kind == "moe":
        return _run_moe(state)
    if kind == "head":
        logits = bmx.quantized_matmul(bmx.rms_norm(state["x"], state["norm"], EPS), *state["head"])
        return {"logits": logits, "tokens": bmx.argmax_rows(logits)}
    state["cache"].truncate(state["case"]["past"])
    if kind == "forward":
        return state["model"].forward(state["cache"], state["tokens"], all_logits=state["case"]["all_logits"])
    _, logits = state["model"].decode_step(state["cache"], state["tokens"][0], want_logits=True)
    return logits


# ---------------------------------------------------------------------------
# the same in float64
# ---------------------------------------------------------------------------
def _dequant(w, s, b, dtype=torch.float64):
    shift = torch.arange(0, 32, 4, device=w.device, dtype=torch.int32)
    q = ((w[..., None] >> shift) & 15).reshape(*s.shape, 64).to(dtype)
    return (q * s.to(dtype)[..., None] + b.to(dtype)[..., None]).reshape(*w.shape[:-1], w.shape[-1] * 8)


def _linear64(x, q):
    step = max(1, (1 << 28) // x.shape[-1])
    return torch.cat([x @ _dequant(*(v[i:i + step] for v in q)).t() for i in range(0, q[0].shape[0], step)], -1)


def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, offset):
    """x [T, heads, 128] rotated at positions offset .. offset + T - 1"""
    half = HEAD_DIM // 2
    f = THETA ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    ang = (offset + torch.arange(x.shape[0], device=x.device, dtype=torch.float64))[:, None, None] * f
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], -1)


def _sdpa64(q, k, v, past):
    """q [M, Hq, 128], k / v [Hkv, L, 128] -> [M, Hq * 128]; query t sees keys <= past + t"""
    M, hq = q.shape[:2]
    rep = hq // k.shape[0]
    see = torch.arange(k.shape[1], device=q.device)[None, :] <= past + torch.arange(M, device=q.device)[:, None]
    out = []
    for h in range(hq):
        p = (q[:, h] @ k[h // rep].t() / math.sqrt(HEAD_DIM)).masked_fill(~see, -math.inf).softmax(-1)
        out.append(p @ v[h // rep])
    return torch.cat(out, -1)


def _attn64(x, t, kc, vc, past):
    """the attention block with its residual; kc / vc [Hkv, past, 128] -> y, all keys, all values"""
    M = x.shape[0]
    h = _norm64(x, t["in_norm"] if "in_norm" in t else t["norm"])
    q, k, v = (_linear64(h, t[n]).view(M, -1, HEAD_DIM) for n in ("q", "k", "v"))
    q, k = _rope64(_norm64(q, t["q_norm"]), past), _rope64(_norm64(k, t["k_norm"]), past)
    kc, vc = torch.cat([kc, k.transpose(0, 1)], 1), torch.cat([vc, v.transpose(0, 1)], 1)
    return x + _linear64(_sdpa64(q, kc, vc, past), t["o"]), kc, vc


def _mlp64(x, norm, t):
    h = _norm64(x, norm)
    g = _linear64(h, t["gate"])
    return x + _linear64(g * torch.sigmoid(g) * _linear64(h, t["up"]), t["down"])


def _moe64(t):
    x, routes = t["x"].double()[:, 0], t["routes"].long()
    out = torch.empty(routes.numel(), 1, MOE_HIDDEN, dtype=torch.float64, device="cuda")
    token = torch.arange(routes.numel(), device="cuda") // MOE_TOPK
    for e in routes.unique().tolist():
        at = (routes == e).nonzero()[:, 0]
        gu = x[token[at]] @ _dequant(*(v[e] for v in t["gate_up"])).t()
        g, u = gu[:, :MOE_INTER], gu[:, MOE_INTER:]
        out[at, 0] = (g * torch.sigmoid(g) * u) @ _dequant(*(v[e] for v in t["down"])).t()
    return out


def _model64(case, t):
    d = _model_dims(case["shape"])
    tokens = torch.from_numpy(np.concatenate([t["past"], t["tokens"]])).cuda()
    x = _dequant(*(v[tokens] for v in t["embed"]))
    none = torch.empty(d["n_kv_heads"], 0, HEAD_DIM, dtype=torch.float64, device="cuda")
    for L in t["layers"]:
        x = _mlp64(_attn64(x, L, none, none, 0)[0], L["post_norm"], L)
    rows = len(t["tokens"]) if case.get("all_logits") else 1
    out = _linear64(_norm64(x[-rows:], t["final"]), t["embed"])
    return out if case.get("all_logits") else out[0]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("forward", "decode"):
        return _model64(case, _model_inputs(case, seed))
    t = _inputs(case, seed)
    if kind == "moe":
        return _moe64(t)
    x = t["x"].double()
    if kind == "mlp":
        return _mlp64(x, t["norm"], t)
    if kind == "head":
        return {"logits": _linear64(_norm64(x, t["norm"]), t["head"]), "tokens": None}
    past, M = case["past"], case["M"]
    y, kc, vc = _attn64(x, t, t["k_cache"][:, :past].double(), t["v_cache"][:, :past].double(), past)
    k, v = t["k_cache"].double(), t["v_cache"].double()
    k[:, past:past + M], v[:, past:past + M] = kc[:, past:], vc[:, past:]
    return {"y": y, "k": k, "v": v}
