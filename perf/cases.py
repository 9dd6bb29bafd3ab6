"""Performance cases of the library: what a host program has it do, through its
public entry points.

A case is one of five kinds:

* ``linear``   -- the isolated matrix product ``linear`` (bf16 W [N, K] times
  f32 X [M, K], f32 out) on device buffers, as a program with its own loop
  calls it: one row (a decode step), a few rows (a small batch or draft
  verification), a prompt's rows.
* ``prefill``  -- ``Runner.prefill``: a prompt, or a later turn of one after
  ``start`` cached positions, through the whole model; the last row's logits
  and their argmax.
* ``generate`` -- ``Runner.generate_greedy_measured`` / ``Runner.generate``:
  a prompt and the tokens after it. The logits of one more step right behind
  the prompt come beside the tokens (they depend on the prompt alone).
* ``step``     -- ``Runner.forward_token`` token by token at a cached context,
  as a host that owns the loop drives it.

Shapes are the named decoders of ``vvli_amd.config``. ``layers`` cuts a model
to that many decoder layers, and ``vocab`` its vocabulary, where the case
stands for the layers and not for the whole model (so that the states stay
small); widths, heads and experts are always the named model's. Weights are
N(0, 0.02) with norm weights around 1, tokens uniform.
"""
from __future__ import annotations

import dataclasses
import math

import numpy as np
import torch

from vvli_amd import config as C
from vvli_amd import runtime as R

DEV = "cuda"


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------
def listed() -> list:
    return [
        # One activation row through a 2048 x 2048 projection (Llama-3.2-1B q or
        # o): the smallest product of a decode step, where the launch counts.
        dict(name="proj-1row", kind="linear", M=1, N=2048, K=2048, bias=False),
        # A small batch through the down projection: long K, few rows of W.
        dict(name="down-16rows", kind="linear", M=16, N=2048, K=8192, bias=False),
        # Odd rows through Qwen2.5-0.5B's stacked q|k|v with its bias.
        dict(name="qkv-33rows", kind="linear", M=33, N=1152, K=896, bias=True),
        # A small batch's logits: the largest weight of the 1B model, read once.
        dict(name="head-16rows", kind="linear", M=16, N=128256, K=2048, bias=False),
        # A prompt's rows through gate or up: matrix-core work.
        dict(name="gate-512rows", kind="linear", M=512, N=8192, K=2048, bias=False),
        # A short user turn behind a cached system prompt, the whole model:
        # time to first token of a chat.
        dict(name="llama1b-turn-45", kind="prefill", model="llama-3.2-1b", layers=16, vocab=128256, rows=45,
             start=200, f32=False),
        # A long document: the largest prompt (two chunks of 2048 rows).
        dict(name="llama1b-prompt-4096", kind="prefill", model="llama-3.2-1b", layers=16, vocab=128256, rows=4096,
             start=0, f32=False),
        # The benchmark's request: a 512-token prompt, then greedy decoding.
        dict(name="llama1b-greedy-512+32", kind="generate", model="llama-3.2-1b", layers=16, vocab=128256, prompt=512,
             new=32, sampled=False),
        # A chat answer with the generator's default sampling options.
        dict(name="qwen05b-sampled-32+24", kind="generate", model="qwen2.5-0.5b", layers=24, vocab=151936, prompt=32,
             new=24, sampled=True),
        # Decode steps of the 7B layers at a long context, the host owning the
        # loop (four of the layers, a small head: the layers are what counts).
        dict(name="qwen7b-layers-step", kind="step", model="qwen2.5-7b", layers=4, vocab=4096, ctx=4000, steps=4),
        # The mixture-of-experts layers over a 64-token prompt (two of them).
        dict(name="olmoe-layers-64", kind="prefill", model="olmoe-1b-7b", layers=2, vocab=4096, rows=64, start=0,
             f32=False),
        # f32 weights, as a checkpoint stored in f32 is loaded: a short prompt
        # through Qwen2.5-0.5B's layers (four of them).
        dict(name="qwen05b-f32-48", kind="prefill", model="qwen2.5-0.5b", layers=4, vocab=4096, rows=48, start=0,
             f32=True),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["linear", "linear", "linear", "prefill", "prefill", "prefill_layers", "generate", "step"])
    if kind == "linear":
        # Any rows up to a prompt's, any width of W up to a model's (K in whole
        # 16-byte units, N any), the head only with the rows a batch has.
        if rng.random() < 0.15:
            return dict(kind="linear", M=_log_int(rng, 1, 64), N=rng.choice([128256, 50304]), K=2048, bias=False)
        if rng.random() < 0.5:
            n, k = rng.choice([(2048, 2048), (512, 2048), (8192, 2048), (2048, 8192), (896, 896), (4864, 896),
                               (896, 4864), (3584, 3584), (1152, 896)])
        else:
            n, k = _log_int(rng, 256, 19000), 8 * _log_int(rng, 64, 1100)
        return dict(kind="linear", M=_log_int(rng, 1, 700), N=n, K=k, bias=rng.random() < 0.5)
    if kind == "prefill":
        model = rng.choice(["llama-3.2-1b", "qwen2.5-0.5b"])
        cfg = C.NAMED[model]()
        return dict(kind="prefill", model=model, layers=cfg.num_hidden_layers, vocab=cfg.vocab_size,
                    rows=_log_int(rng, 4, 3000), start=rng.choice([0, 0, _log_int(rng, 8, 1000)]), f32=False)
    if kind == "prefill_layers":
        model = rng.choice(["qwen2.5-7b", "olmoe-1b-7b", "qwen2.5-0.5b"])
        f32 = model == "qwen2.5-0.5b"
        return dict(kind="prefill", model=model, layers=rng.randint(1, 3), vocab=4096,
                    rows=_log_int(rng, 8, 100 if f32 else 1500), start=rng.choice([0, _log_int(rng, 8, 300)]), f32=f32)
    if kind == "generate":
        model = rng.choice(["llama-3.2-1b", "qwen2.5-0.5b"])
        cfg = C.NAMED[model]()
        return dict(kind="generate", model=model, layers=cfg.num_hidden_layers, vocab=cfg.vocab_size,
                    prompt=_log_int(rng, 8, 500), new=rng.randint(4, 24), sampled=rng.random() < 0.5)
    model = rng.choice(["qwen2.5-7b", "olmoe-1b-7b", "llama-3.2-1b"])
    return dict(kind="step", model=model, layers=rng.randint(2, 4), vocab=4096, ctx=_log_int(rng, 16, 3900),
                steps=rng.randint(2, 4))


# ---------------------------------------------------------------------------
# Models
# ---------------------------------------------------------------------------
def _config(case) -> C.Config:
    return dataclasses.replace(C.NAMED[case["model"]](), num_hidden_layers=case["layers"], vocab_size=case["vocab"])


def _slices(cfg: C.Config, f32: bool) -> dict:
    """(slot, layer) -> (element offset, count) of the model's blob."""
    ea = 16 if f32 else 32
    H, kv, I, E = cfg.hidden_size, cfg.kv_dim(), cfg.intermediate_size, cfg.num_experts
    if not E:
        return {(s, l): (o, n) for s, l, o, n in R.dense_slices(cfg, C.WEIGHT_F32 if f32 else C.WEIGHT_BF16)}
    out = {("embed", None): (0, cfg.vocab_size * H)}
    sizes = dict(input_norm=H, q=H * H, k=kv * H, v=kv * H, q_norm=H, k_norm=kv, o=H * H, post_norm=H, router=E * H,
                 gate_up=2 * E * I * H, down=E * H * I)
    end = 0
    for l in range(cfg.num_hidden_layers):
        for s, n in sizes.items():
            o = R.moe_slice_offset(cfg, l, s)
            out[(s, l)] = (o, n)
            end = o + n
    end = -(-end // ea) * ea
    out[("final_norm", None)] = (end, H)
    out[("lm_head", None)] = (-(-(end + H) // ea) * ea, cfg.vocab_size * H)
    return out


def _blob(cfg: C.Config, f32: bool, seed: int) -> torch.Tensor:
    """The blob on the GPU, bf16 or f32, from the seed alone."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    n = cfg.storage_element_count(C.WEIGHT_F32 if f32 else C.WEIGHT_BF16)
    out = torch.empty(n, device=DEV, dtype=torch.float32 if f32 else torch.bfloat16)
    step = 1 << 28
    for i in range(0, n, step):
        m = min(step, n - i)
        out[i:i + m] = torch.randn(m, device=DEV, generator=g) * 0.02
    for (slot, _), (o, m) in _slices(cfg, f32).items():
        if slot.endswith("norm"):
            out[o:o + m] = 1 + 0.1 * torch.randn(m, device=DEV, generator=g)
    return out


def _runner(case, seed: int, max_seq: int) -> R.Runner:
    cfg, f32 = _config(case), bool(case.get("f32"))
    blob = _blob(cfg, f32, seed)
    host = blob.cpu()
    del blob
    host = host.numpy() if f32 else host.view(torch.int16).numpy().view(np.uint16)
    return (R.MoeRunner if cfg.num_experts else R.Runner)(cfg, host, max_seq)


def _tokens(case, seed: int, n: int) -> np.ndarray:
    return np.random.RandomState(seed + 1).randint(0, case["vocab"], n).astype(np.uint32)


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def _linear_inputs(case, seed: int):
    M, N, K = case["M"], case["N"], case["K"]
    g = torch.Generator(device=DEV).manual_seed(seed)
    w = (torch.randn(N, K, device=DEV, generator=g) * 0.02).bfloat16()
    x = torch.randn(M, K, device=DEV, generator=g)
    b = (torch.randn(N, device=DEV, generator=g) * 0.02).bfloat16() if case["bias"] else None
    return w, x, b


def prepare(case, seed: int) -> dict:
    kind = case["kind"]
    st = {"kind": kind}
    if kind == "linear":
        st["w"], st["x"], st["b"] = _linear_inputs(case, seed)
        st["y"] = torch.empty(case["M"], case["N"], device=DEV)
        st["dims"] = (case["M"], case["N"], case["K"])
        st["stream"] = torch.cuda.current_stream().cuda_stream
    elif kind == "prefill":
        n = case["start"] + case["rows"]
        toks = _tokens(case, seed, n)
        st["r"] = _runner(case, seed, n + 64)
        if case["start"]:
            st["r"].prefill(toks[: case["start"]], 0)
        st["tokens"], st["start"] = toks[case["start"]:], case["start"]
    elif kind == "generate":
        st["r"] = _runner(case, seed, case["prompt"] + case["new"] + 64)
        st["tokens"], st["new"] = _tokens(case, seed, case["prompt"]), case["new"]
        st["next"] = int(_tokens(case, seed + 7, 1)[0])
        st["sampling"] = R.Sampling(seed=seed + 3) if case["sampled"] else None
    else:
        n = case["ctx"] + case["steps"]
        toks = _tokens(case, seed, n)
        st["r"] = _runner(case, seed, n + 64)
        st["r"].prefill(toks[: case["ctx"]], 0)
        st["tokens"], st["ctx"] = [int(t) for t in toks[case["ctx"]:]], case["ctx"]
    return st


def run(st):
    kind = st["kind"]
    if kind == "linear":
        M, N, K = st["dims"]
        R.linear(st["w"].data_ptr(), st["x"].data_ptr(), st["y"].data_ptr(), M, N, K,
                 None if st["b"] is None else st["b"].data_ptr(), st["stream"])
        return st["y"]
    r = st["r"]
    if kind == "prefill":
        logits, top = r.prefill(st["tokens"], st["start"])
        return {"logits": logits, "argmax": top}
    if kind == "generate":
        if st["sampling"] is None:
            toks, _ = r.generate_greedy_measured(st["tokens"], st["new"], batched_prefill=True)
        else:
            toks, _ = r.generate(st["tokens"], st["new"], st["sampling"], batched_prefill=True)
        return {"tokens": toks.astype(np.int64), "logits": r.forward_token(st["next"], len(st["tokens"]))}
    out = []
    for i, t in enumerate(st["tokens"]):
        out.append(r.forward_token(t, st["ctx"] + i).copy())  # the host keeps each step's scores
    return {"logits": out}


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------
def _layer_weights(cfg: C.Config, rows: int) -> tuple:
    """(weight elements read, weight elements multiplied per row) of a layer."""
    H, kv, I = cfg.hidden_size, cfg.kv_dim(), cfg.intermediate_size
    attn = 2 * H * H + 2 * kv * H
    if not cfg.num_experts:
        return attn + 3 * H * I, attn + 3 * H * I
    E, k = cfg.num_experts, cfg.num_experts_per_token
    hit = E * (1 - (1 - k / E) ** rows)  # experts that some row takes
    return attn + E * H + int(hit * 3 * H * I), attn + E * H + k * 3 * H * I


def _pass_work(cfg: C.Config, rows: int, start: int, heads: int, eb: int) -> tuple:
    """(bytes, flops) of `rows` positions in one pass behind `start` cached ones, `heads` rows of logits."""
    read, mult = _layer_weights(cfg, rows)
    kv, H, V, L = cfg.kv_dim(), cfg.hidden_size, cfg.vocab_size, cfg.num_hidden_layers
    pairs = rows * start + rows * (rows + 1) // 2
    flops = L * (2 * rows * mult + 4 * pairs * H) + 2 * heads * V * H
    byts = L * (read * eb + 2 * 4 * kv * (start + rows)) + V * H * eb + rows * H * eb + heads * V * 4
    return byts, flops


def work(case) -> dict:
    if case["kind"] == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 2 * N * K + 4 * M * K + 4 * M * N + (2 * N if case["bias"] else 0), "flops": 2 * M * N * K}
    cfg = _config(case)
    eb = 4 if case.get("f32") else 2
    if case["kind"] == "prefill":
        b, f = _pass_work(cfg, case["rows"], case["start"], 1, eb)
        return {"bytes": b, "flops": f}
    if case["kind"] == "generate":
        b, f = _pass_work(cfg, case["prompt"], 0, 1, eb)
        steps = [case["prompt"] + i for i in range(case["new"])] + [case["prompt"]]
    else:
        b = f = 0
        steps = [case["ctx"] + i for i in range(case["steps"])]
    for p in steps:
        pb, pf = _pass_work(cfg, 1, p, 1, eb)
        b, f = b + pb, f + pf
    return {"bytes": b, "flops": f}


def tolerance(case):
    if case["kind"] == "linear":
        # One row: f32 sums (1.3e-7 off the 64-bit result). More rows: f32
        # activations held as two bf16 halves, f32 sums (2.5e-6 off).
        return {"rel": 1e-6 if case["M"] == 1 else 1e-5}
    # Whole passes, off the 64-bit result: 2.6e-5 through 16 bf16 layers (two
    # passes with other sum orders 1.2e-5 apart, their largest 5.6e-5 of the
    # root mean square), 5e-7 through f32 ones. "differ": a token at a near
    # tie, and those after it.
    tol = {"rel": 4e-6, "max": 4e-5} if case.get("f32") else {"rel": 1e-4, "max": 6e-4}
    if case["kind"] in ("prefill", "generate"):
        tol["differ"] = 0.5
    return tol


# ---------------------------------------------------------------------------
# exact: the same passes in 64 bits
# ---------------------------------------------------------------------------
class _Exact:
    """The decoder in f64: RMSNorm, RoPE (angles are f32, as the model defines
    them), causal GQA attention, SwiGLU or routed experts."""

    def __init__(self, case, seed: int):
        self.cfg, self.f32 = _config(case), bool(case.get("f32"))
        self.blob = _blob(self.cfg, self.f32, seed)
        self.at = _slices(self.cfg, self.f32)

    def w(self, slot, layer=None):
        if (slot, layer) not in self.at:
            return None
        o, n = self.at[(slot, layer)]
        return self.blob[o:o + n].double()

    def norm(self, x, w):
        return x * w / torch.sqrt((x * x).mean(-1, keepdim=True) + self.cfg.rms_norm_eps)

    def rope(self, x):  # [rows, heads, hd]
        hd, n = x.shape[-1], x.shape[0]
        half = hd // 2
        ex = (2 * np.arange(half, dtype=np.float32)) / np.float32(hd)
        inv = (1 / np.power(float(self.cfg.rope_theta), ex.astype(np.float64)).astype(np.float32)).astype(np.float32)
        ang = (np.arange(n, dtype=np.float32)[:, None] * inv[None]).astype(np.float64)
        c = torch.from_numpy(np.cos(ang)).to(DEV)[:, None]
        s = torch.from_numpy(np.sin(ang)).to(DEV)[:, None]
        if self.cfg.rope_layout == C.ROPE_INTERLEAVED:
            a, b = x[..., 0::2], x[..., 1::2]
            return torch.stack([a * c - b * s, a * s + b * c], -1).reshape(x.shape)
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * c - b * s, a * s + b * c], -1)

    def attention(self, h, l):
        cfg = self.cfg
        H, kv, hd, n = cfg.hidden_size, cfg.kv_dim(), cfg.head_dim(), h.shape[0]
        q, k, v = (h @ self.w(s, l).view(m, H).t() for s, m in (("q", H), ("k", kv), ("v", kv)))
        if cfg.qkv_bias:
            q, k, v = q + self.w("q_bias", l), k + self.w("k_bias", l), v + self.w("v_bias", l)
        if cfg.qk_norm:
            q, k = self.norm(q, self.w("q_norm", l)), self.norm(k, self.w("k_norm", l))
        q, k = self.rope(q.view(n, -1, hd)), self.rope(k.view(n, -1, hd))
        v = v.view(n, -1, hd)
        mask = torch.ones(n, n, device=DEV, dtype=torch.bool).triu(1)
        out = torch.empty_like(q)
        for j in range(q.shape[1]):
            kj = j // cfg.kv_group_size()
            sc = (q[:, j] @ k[:, kj].t() / math.sqrt(hd)).masked_fill_(mask, -math.inf)
            out[:, j] = torch.softmax(sc, -1) @ v[:, kj]
        return out.reshape(n, H) @ self.w("o", l).view(H, H).t()

    def mlp(self, h, l):
        cfg = self.cfg
        H, I = cfg.hidden_size, cfg.intermediate_size
        if not cfg.num_experts:
            g, u = h @ self.w("gate", l).view(I, H).t(), h @ self.w("up", l).view(I, H).t()
            return (torch.nn.functional.silu(g) * u) @ self.w("down", l).view(H, I).t()
        E = cfg.num_experts
        p = torch.softmax(h @ self.w("router", l).view(E, H).t(), -1)
        top, idx = p.topk(cfg.num_experts_per_token, -1)
        wt = torch.zeros_like(p).scatter_(1, idx, top)
        gu, dn = self.w("gate_up", l).view(E, 2 * I, H), self.w("down", l).view(E, H, I)
        out = torch.zeros_like(h)
        for e in range(E):
            r = wt[:, e].nonzero()[:, 0]
            if r.numel():
                y = h[r] @ gu[e].t()
                y = (torch.nn.functional.silu(y[:, :I]) * y[:, I:]) @ dn[e].t()
                out.index_add_(0, r, y * wt[r, e, None])
        return out

    def logits(self, tokens, rows: int):
        """Logits of the last `rows` positions of `tokens` (from position 0)."""
        cfg = self.cfg
        H = cfg.hidden_size
        x = self.w("embed").view(-1, H)[torch.from_numpy(np.asarray(tokens, np.int64)).to(DEV)]
        for l in range(cfg.num_hidden_layers):
            x = x + self.attention(self.norm(x, self.w("input_norm", l)), l)
            x = x + self.mlp(self.norm(x, self.w("post_norm", l)), l)
        x = self.norm(x[-rows:], self.w("final_norm"))
        return x @ self.w("embed" if cfg.tie_word_embeddings else "lm_head").view(-1, H).t()


def exact(case, seed: int):
    kind = case["kind"]
    if kind == "linear":
        w, x, b = _linear_inputs(case, seed)
        y = x.double() @ w.double().t()
        return y if b is None else y + b.double()
    m = _Exact(case, seed)
    if kind == "prefill":
        lg = m.logits(_tokens(case, seed, case["start"] + case["rows"]), 1)[0]
        return {"logits": lg, "argmax": int(lg.argmax())}
    if kind == "generate":
        toks = np.concatenate([_tokens(case, seed, case["prompt"]), _tokens(case, seed + 7, 1)])
        return {"tokens": None, "logits": m.logits(toks, 1)[0]}
    lg = m.logits(_tokens(case, seed, case["ctx"] + case["steps"]), case["steps"])
    return {"logits": list(lg)}
