"""The work this library does for its users, as cases that can be timed and
checked: one MoE layer at every batch size from one decoded token to a long
prompt, the whole batch-1 token, the FP8 attention projections, the BF16
lm_head and the per-matmul calls of an engine that knows the six drop-in
symbols only.  Shapes are the ones the benchmark and the tests use.

Weights are drawn N(0, 0.02) and quantised per 128x128 block to E4M3 (scale =
amax / 448); activations are N(0, 1) f32.  Inputs live in HBM except for the
drop-in calls, which take host arrays by their contract.

The streaming tier is not among the cases: what one of its passes costs
depends on what the passes before it left in the pool.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from colizig_amd import _lib, moe

BLOCK = 128

# model: hidden, experts, top-k, expert width, shared-expert width
MODELS = {
    "qwen3": (2048, 128, 8, 768, 0),         # Qwen3-30B-A3B
    "qwen4": (4096, 512, 10, 512, 4096),     # Qwen4-Exp
    "small": (512, 16, 4, 256, 256),         # the smallest layer the fast kernels serve
}
# attention projections of Qwen3-30B-A3B: rows of q, k, v (width 2048) and o (width 4096)
QD, KVD, HIDDEN = 4096, 512, 2048
VOCAB = 151936
EPS = 1e-6
TOKEN_SETS = 4  # distinct expert sets of a whole model's layers (layer l holds its own copy of set l % 4)


def listed() -> list[dict]:
    return [
        # one decoded token through a whole model's MoE stack, replayed as a graph
        dict(name="token_qwen3", kind="token", layers=48),
        # an engine that runs its layers one by one: a single decoded token
        dict(name="layer_qwen3_1", kind="layer", model="qwen3", tokens=1, zipf=0.0),
        # a handful of requests decoded together, or a short speculative draft
        dict(name="layer_qwen3_6", kind="layer", model="qwen3", tokens=6, zipf=0.0),
        # a prompt (or prompt chunk) of 512 tokens, experts as skewed as real routers make them
        dict(name="layer_qwen3_512", kind="layer", model="qwen3", tokens=512, zipf=1.1),
        # a long prompt in one call, not a power of two
        dict(name="layer_qwen3_2000", kind="layer", model="qwen3", tokens=2000, zipf=1.1),
        # the larger model with a shared expert: one token, and a server's decode batch
        dict(name="layer_qwen4_1", kind="layer", model="qwen4", tokens=1, zipf=0.0),
        dict(name="layer_qwen4_32", kind="layer", model="qwen4", tokens=32, zipf=0.0),
        # a layer's q, k, v and o projections: one token, and a prompt chunk
        dict(name="attn_1", kind="attn", tokens=1),
        dict(name="attn_385", kind="attn", tokens=385),
        # next-token logits of one sequence, and of a decode batch
        dict(name="lm_head_1", kind="lm_head", tokens=1, rows=VOCAB),
        dict(name="lm_head_8", kind="lm_head", tokens=8, rows=VOCAB),
        # an unchanged engine: one expert's three matmuls on host buffers
        dict(name="dropin_expert_1", kind="dropin", tokens=1, hidden=2048, inter=768),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["layer"] * 6 + ["attn"] * 2 + ["lm_head", "dropin", "token"])
    if kind == "layer":
        model = rng.choice(["qwen3", "qwen3", "qwen4", "small"])
        tokens = _log_int(rng, 2, {"qwen3": 1999, "qwen4": 200, "small": 1999}[model])
        return dict(kind=kind, model=model, tokens=tokens, zipf=rng.choice([0.0, 1.1]) if tokens >= 16 else 0.0)
    if kind == "attn":
        return dict(kind=kind, tokens=_log_int(rng, 2, 1500))
    if kind == "lm_head":
        return dict(kind=kind, tokens=_log_int(rng, 1, 16), rows=rng.randrange(30000, VOCAB))
    if kind == "dropin":
        return dict(kind=kind, tokens=_log_int(rng, 1, 64), hidden=rng.choice([512, 1024, 2048, 4096]),
                    inter=64 * rng.randrange(4, 25))
    return dict(kind=kind, layers=rng.randrange(4, 48))


# ---- inputs ----------------------------------------------------------------
def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape) -> torch.Tensor:
    return torch.randn(*shape, generator=g, device="cuda")


def _fp8(g, n: int, rows: int, cols: int):
    """n matrices [rows, cols] as E4M3 bytes and scales [n, nblk(rows), nblk(cols)]."""
    ws, ss = [], []
    nr, nc = moe.nblk(rows), moe.nblk(cols)
    for i in range(0, n, 64):  # bounds the f32 copy
        m = min(64, n - i)
        w = (_randn(g, m, nr * BLOCK, nc * BLOCK) * 0.02).view(m, nr, BLOCK, nc, BLOCK)
        s = w.abs().amax(dim=(2, 4)) / 448.0
        q = (w / s[:, :, None, :, None]).to(torch.float8_e4m3fn).view(torch.uint8)
        ws.append(q.view(m, nr * BLOCK, nc * BLOCK)[:, :rows, :cols].contiguous())
        ss.append(s)
    return torch.cat(ws), torch.cat(ss)


def _layer_weights(case: dict, seed: int) -> dict:
    H, E, K, I, SI = MODELS[case["model"]]
    g = _gen(seed)
    w = dict(router=_randn(g, E, H) * 0.02, x=_randn(g, case["tokens"], H))
    w["gate"], w["up"], w["down"] = _fp8(g, E, I, H), _fp8(g, E, I, H), _fp8(g, E, H, I)
    if SI:
        w["shared"] = [_fp8(g, 1, SI, H), _fp8(g, 1, SI, H), _fp8(g, 1, H, SI)]
        w["sh_gate"] = _randn(g, H) * 0.02
    if case["zipf"]:
        # expert popularity ~ rank^-s: the log of it, centred, on every logit
        rank = 1 + torch.randperm(E, generator=g, device="cuda").double()
        lp = -case["zipf"] * rank.log()
        w["bias"] = (lp - lp.mean()).float()
    return w


def _token_weights(case: dict, seed: int) -> dict:
    H, E, _, I, _ = MODELS["qwen3"]
    g = _gen(seed)
    w = dict(x=_randn(g, 1, H), router=_randn(g, case["layers"], E, H) * 0.02)
    w["sets"] = [dict(gate=_fp8(g, E, I, H), up=_fp8(g, E, I, H), down=_fp8(g, E, H, I))
                 for _ in range(min(TOKEN_SETS, case["layers"]))]
    return w


def _attn_weights(case: dict, seed: int) -> dict:
    g = _gen(seed)
    w = dict(x=_randn(g, case["tokens"], HIDDEN), a=_randn(g, case["tokens"], QD))
    w["mats"] = [_fp8(g, 1, QD, HIDDEN), _fp8(g, 1, KVD, HIDDEN), _fp8(g, 1, KVD, HIDDEN), _fp8(g, 1, HIDDEN, QD)]
    return w


def _lm_head_weights(case: dict, seed: int):
    g = _gen(seed)
    return _randn(g, case["tokens"], HIDDEN), (_randn(g, case["rows"], HIDDEN) * 0.02).to(torch.bfloat16)


def _dropin_weights(case: dict, seed: int):
    H, I = case["hidden"], case["inter"]
    g = _gen(seed)
    mats = [_fp8(g, 1, I, H), _fp8(g, 1, I, H), _fp8(g, 1, H, I)]
    return _randn(g, case["tokens"], H), _randn(g, case["tokens"], I), mats


# ---- what a program keeps ----------------------------------------------------
_stream = None
_layer_ids: list[int] = []   # given back by states that are gone
_next_layer = 0
_keys: dict = {}             # (type, rows, columns) -> keys given back
_next_key = 1


def _start():
    """The library, and the stream this program puts its work on."""
    global _stream
    if _stream is None:
        moe.init()
        moe.set_vram_budget(16 << 30)
        _stream = torch.cuda.Stream()
    return _lib.hip(), ctypes.c_void_p(_stream.cuda_stream)


class _Layers:
    """Consecutive layer ids, whose memory goes back with the object."""

    def __init__(self, n: int):
        global _next_layer
        if n == 1 and _layer_ids:
            self.first = _layer_ids.pop()
        else:
            self.first, _next_layer = _next_layer, _next_layer + n
        self.n = n

    def __del__(self):
        torch.cuda.synchronize()
        d = moe.dims(256, 1, 1, 128)
        for l in range(self.first, self.first + self.n):
            moe.Layer.load(l, d, np.zeros((1, 256), np.float32))  # frees the layer's weights
            _layer_ids.append(l)


class _Keys:
    """Keys of the HBM matrix cache for matrices of the given types and shapes."""

    def __init__(self, shapes):
        global _next_key
        self.shapes, self.keys = shapes, []
        for s in shapes:
            if _keys.get(s):
                self.keys.append(_keys[s].pop())
            else:
                self.keys.append(_next_key)
                _next_key += 1

    def __del__(self):
        torch.cuda.synchronize()
        for s, k in zip(self.shapes, self.keys):
            _keys.setdefault(s, []).append(k)


def _on_host(t: torch.Tensor) -> np.ndarray:
    return torch.empty(t.shape, dtype=t.dtype, pin_memory=True).copy_(t).numpy()


def _load_experts(L: moe.Layer, host: dict) -> None:
    for e in range(L.d.experts):
        L.load_expert(e, *(host[m][j][e] for m in ("gate", "up", "down") for j in (0, 1)))


def _load_layer(ids: _Layers, case: dict, w: dict) -> moe.Layer:
    H, E, K, I, SI = MODELS[case["model"]]
    L = moe.Layer.load(ids.first, moe.dims(H, E, K, I, SI), w["router"].cpu().numpy())
    _load_experts(L, {m: [_on_host(t) for t in w[m]] for m in ("gate", "up", "down")})
    if SI:
        L.set_shared(*(t[0].cpu().numpy() for pair in w["shared"] for t in pair), w["sh_gate"].cpu().numpy())
    if "bias" in w:
        L.set_router_bias(w["bias"].cpu().numpy())
    return L


def prepare(case: dict, seed: int) -> dict:
    hip, st = _start()
    kind = case["kind"]
    s = dict(kind=kind, hip=hip, stream=st)
    if kind == "token":
        H, E, K, I, _ = MODELS["qwen3"]
        w = _token_weights(case, seed)
        s["ids"] = _Layers(case["layers"])
        routers = _on_host(w["router"])
        for i, experts in enumerate(w["sets"]):
            host = {m: [_on_host(t) for t in experts[m]] for m in ("gate", "up", "down")}
            for l in range(i, case["layers"], TOKEN_SETS):
                _load_experts(moe.Layer.load(s["ids"].first + l, moe.dims(H, E, K, I), routers[l]), host)
        s["x0"] = w["x"]
        s["x"] = s["x0"].clone()
        torch.cuda.synchronize()
        s["graph"] = _Graph(hip, hip.colizig_hip_chain_graph_create(s["ids"].first, case["layers"], s["x"].data_ptr(),
                                                                  1, EPS))
    elif kind == "layer":
        H, E, K, I, SI = MODELS[case["model"]]
        w = _layer_weights(case, seed)
        s["ids"] = _Layers(1)
        s["layer"] = _load_layer(s["ids"], case, w)
        s["x"] = w["x"]
        s["out"] = torch.empty_like(w["x"])
        s["idx"] = torch.zeros(case["tokens"], K, dtype=torch.int32, device="cuda")
        s["gates"] = torch.zeros(case["tokens"], K, device="cuda")
    elif kind == "attn":
        w = _attn_weights(case, seed)
        s["keys"] = _Keys([("fp8",) + tuple(q.shape) for q, _ in w["mats"]])
        for k, (q, sc) in zip(s["keys"].keys, w["mats"]):
            moe.matrix_load(k, q[0].cpu().numpy(), sc[0].cpu().numpy())
        s["x"], s["a"], s["S"] = w["x"], w["a"], case["tokens"]
        s["y"] = [torch.empty(case["tokens"], o, device="cuda") for o in (QD, KVD, KVD, HIDDEN)]
    elif kind == "lm_head":
        x, w = _lm_head_weights(case, seed)
        s["keys"] = _Keys([("bf16",) + tuple(w.shape)])
        moe.matrix_load_bf16(s["keys"].keys[0], w.view(torch.int16).cpu().numpy().view(np.uint16))
        s["x"], s["S"], s["rows"] = x, case["tokens"], case["rows"]
        s["y"] = torch.empty(case["tokens"], case["rows"], device="cuda")
    else:
        # a key names one matrix for good: an engine never reuses it
        global _next_key
        x, h, mats = _dropin_weights(case, seed)
        s["x"], s["h"], s["S"] = x.cpu().numpy(), h.cpu().numpy(), case["tokens"]
        s["mats"] = []
        for q, sc in mats:
            s["mats"].append((q[0].cpu().numpy(), sc[0].cpu().numpy(), _next_key))
            _next_key += 1
    torch.cuda.synchronize()
    return s


class _Graph:
    def __init__(self, hip, handle: int):
        if handle <= 0:
            raise RuntimeError(f"graph capture failed: {_lib.last_error()}")
        self.hip, self.handle = hip, handle

    def __del__(self):
        torch.cuda.synchronize()
        self.hip.colizig_hip_graph_destroy(self.handle)


def _ok(rc: int) -> None:
    if rc != 0:
        raise RuntimeError(f"rc={rc}: {_lib.last_error()}")


def run(s: dict):
    kind, hip, st = s["kind"], s["hip"], s["stream"]
    if kind == "layer":
        x = s["x"]
        _ok(hip.colizig_hip_moe_forward_dev(s["layer"].layer, x.data_ptr(), x.shape[0], s["out"].data_ptr(),
                                            s["idx"].data_ptr(), s["gates"].data_ptr(), st))
        return dict(out=s["out"], idx=s["idx"], gates=s["gates"])
    if kind == "token":
        with torch.cuda.stream(_stream):
            s["x"].copy_(s["x0"])  # the token's embedding
        _ok(hip.colizig_hip_graph_launch(s["graph"].handle, st))
        return s["x"]
    if kind == "attn":
        y, k, S = s["y"], s["keys"].keys, s["S"]
        moe.matmul_fp8_dev_multi([t.data_ptr() for t in y[:3]], s["x"].data_ptr(), S, HIDDEN, [QD, KVD, KVD], k[:3], st)
        moe.matmul_fp8_dev(y[3].data_ptr(), s["a"].data_ptr(), S, QD, HIDDEN, k[3], st)
        return y
    if kind == "lm_head":
        moe.matmul_bf16_dev(s["y"].data_ptr(), s["x"].data_ptr(), s["S"], HIDDEN, s["rows"], s["keys"].keys[0], st)
        return s["y"]
    outs = []
    for a, (q, sc, key) in zip((s["x"], s["x"], s["h"]), s["mats"]):
        outs.append(moe.matmul_fp8(a, q, sc, s["S"], q.shape[1], q.shape[0], key))
    return outs


# ---- what a pass cannot do without ------------------------------------------
def _experts_touched(E: int, K: int, tokens: int, zipf: float) -> float:
    """Expected distinct experts of `tokens` tokens (each picks K of E, evenly
    or with popularity ~ rank^-zipf)."""
    p = [(r + 1.0) ** -zipf for r in range(E)]
    lo, hi = 0.0, 1e9
    for _ in range(100):  # pick probabilities 1 - exp(-c p) that add up to K
        c = 0.5 * (lo + hi)
        lo, hi = (c, hi) if sum(1 - math.exp(-c * v) for v in p) < K * sum(p) / sum(p) else (lo, c)
    return sum(1 - math.exp(-lo * v * tokens) for v in p)


def work(case: dict) -> dict:
    kind = case["kind"]

    def fp8_bytes(o, i):
        return o * i + 4 * moe.nblk(o) * moe.nblk(i)

    if kind in ("layer", "token"):
        H, E, K, I, SI = MODELS[case.get("model", "qwen3")]
        S, n = case.get("tokens", 1), case.get("layers", 1)
        expert = 2 * fp8_bytes(I, H) + fp8_bytes(H, I)
        b = 4 * E * H + _experts_touched(E, K, S, case.get("zipf", 0.0)) * expert
        f = 2 * S * (E * H + K * 3 * H * I)
        if SI:
            b += 2 * fp8_bytes(SI, H) + fp8_bytes(H, SI) + 4 * H
            f += 2 * S * 3 * H * SI
        return dict(bytes=n * b + 8 * S * H, flops=n * f)
    S = case["tokens"]
    if kind == "attn":
        o = QD + 2 * KVD
        return dict(bytes=fp8_bytes(o, HIDDEN) + fp8_bytes(HIDDEN, QD) + 4 * S * (2 * HIDDEN + o + QD),
                    flops=2 * S * (o * HIDDEN + HIDDEN * QD))
    if kind == "lm_head":
        return dict(bytes=2 * case["rows"] * HIDDEN + 4 * S * (HIDDEN + case["rows"]),
                    flops=2 * S * case["rows"] * HIDDEN)
    H, I = case["hidden"], case["inter"]
    return dict(bytes=3 * fp8_bytes(I, H) + 4 * S * (3 * H + 3 * I), flops=6 * S * H * I)


def tolerance(case: dict):
    kind = case["kind"]
    if kind == "lm_head":
        return "exact"  # every dot in dotBf16's order, bit for bit
    if kind == "layer" and case["tokens"] >= 16 and case["tokens"] * MODELS[case["model"]][2] <= 8192:
        # the grouped GEMMs split activations into three E4M3 terms (about 12
        # bits): 4.5e-5 measured.  Routing is exact.
        return dict(rel=2e-4, max=2e-3)
    if kind == "token":
        return dict(rel=4e-6, max=4e-5)  # 48 chained layers of f32 sums: 4.4e-7 measured
    return dict(rel=2e-6, max=2e-5)      # f32 sums: 3e-7 measured


# ---- the same in 64 bits -----------------------------------------------------
def _wide(pair, i: int) -> torch.Tensor:
    q, s = pair
    r, c = q.shape[1:]
    scale = s[i].double().repeat_interleave(BLOCK, 0).repeat_interleave(BLOCK, 1)
    return q[i].view(torch.float8_e4m3fn).double() * scale[:r, :c]


def _swiglu(x, g, u, d):
    a = x @ g.T.contiguous()
    return (a * torch.sigmoid(a) * (x @ u.T.contiguous())) @ d.T.contiguous()


def _routed(x, router, bias, w, K: int):
    """The routed experts' sum for rows x, and the gates."""
    logits = x @ router.double().T.contiguous()
    if bias is not None:
        logits = logits + bias.double()
    gates, idx = torch.topk(torch.softmax(logits, dim=1), K, dim=1)
    gates = gates / gates.sum(dim=1, keepdim=True)
    out = torch.zeros_like(x)
    for e in torch.unique(idx).tolist():
        t, z = torch.nonzero(idx == e, as_tuple=True)
        y = _swiglu(x[t], _wide(w["gate"], e), _wide(w["up"], e), _wide(w["down"], e))
        out.index_add_(0, t, y * gates[t, z][:, None])
    return out, gates


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "token":
        w = _token_weights(case, seed)
        x = w["x"].double()
        for l in range(case["layers"]):
            n = x / torch.sqrt((x * x).mean(dim=1, keepdim=True) + EPS)
            x = x + _routed(n, w["router"][l], None, w["sets"][l % TOKEN_SETS], MODELS["qwen3"][2])[0]
        return x
    if kind == "layer":
        H, E, K, I, SI = MODELS[case["model"]]
        w = _layer_weights(case, seed)
        x = w["x"].double()
        out, gates = _routed(x, w["router"], w.get("bias"), w, K)
        if SI:
            y = _swiglu(x, *(_wide(m, 0) for m in w["shared"]))
            out += torch.sigmoid(x @ w["sh_gate"].double())[:, None] * y
        return dict(out=out, idx=None, gates=gates)
    if kind == "attn":
        w = _attn_weights(case, seed)
        x, a = w["x"].double(), w["a"].double()
        return [v @ _wide(m, 0).T.contiguous() for v, m in zip((x, x, x, a), w["mats"])]
    if kind == "lm_head":
        x, w = _lm_head_weights(case, seed)
        return x.double() @ w.double().T.contiguous()
    x, h, mats = _dropin_weights(case, seed)
    return [(v.double() @ _wide(m, 0).T.contiguous()).cpu().numpy() for v, m in zip((x, x, h), mats)]
