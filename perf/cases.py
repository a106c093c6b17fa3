"""The calls whose speed this library answers for, as a user's program makes them.

Every case runs one pass through public entry points: a decode tick of the
engine (`engine.LoopedModel.run_passes`), a prompt (`prefill_seq`), the
attention module (`attention.attn_dense` / `attn_varlen` / `compute_qkv`) and
the row-wise ops a program composes a block from (`ops`). Sizes are those of
the configurations in model.CONFIGS and of the ranges the tests and the
benchmark use: rows of a wave from one to a few hundred, prefixes from a
hundred keys to 32k, prompts from a few dozen tokens to 16k.

  listed()          the fixed cases
  draw(rng)         one more case of the same ranges
  prepare(case, s)  inputs, weights and engine, from the seed
  run(state)        one pass
  work(case)        bytes and operations a pass cannot do without
  tolerance(case)   how far two correct implementations may differ
  exact(case, s)    run()'s outputs in 64-bit torch
"""
from __future__ import annotations

import math
from types import SimpleNamespace

import torch

import __graft_entry__

__graft_entry__.load_package()

from wavefront_decoding_amd import attention, ops  # noqa: E402
from wavefront_decoding_amd.engine import LoopedModel  # noqa: E402
from wavefront_decoding_amd.model import CONFIGS  # noqa: E402

DEV = "cuda"
EPS = 1e-6
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed() -> list[dict]:
    return [
        # one token of the tiny fp32 model through its whole depth (P, 4 x R, C
        # as one replay): the smallest call, all launches and latency
        dict(name="tick_tiny_f32", kind="tick", model="tiny", batch=1, width=1, loops=4, lo=150, hi=150),
        # single-user decoding: an 8-row wave of one sequence on the 2048-d
        # model, depths spread over the loop, with its prelude and coda
        dict(name="tick_wave8", kind="tick", model="looped-2048", batch=1, width=8, loops=1, lo=512, hi=760),
        # served batch: 28 sequences x 4 wave rows, ragged prefixes
        dict(name="tick_batch112", kind="tick", model="looped-2048", batch=28, width=4, loops=1, lo=128, hi=1200),
        # the prompt of a single-user request, through the 2048-d model's layers
        # with its core run once (a deeper loop repeats the same launches, and
        # its bf16 rounding grows from loop to loop until nothing can be compared)
        dict(name="prefill_512", kind="prefill", model="looped-2048", loops=1, length=512),
        # one layer's attention of the single-user wave, called by itself
        dict(name="attn_wave8", kind="decode", rows=8, H=16, Hkv=16, Dh=128, lo=512, hi=778, dtype="bf16"),
        # long-context GQA decoding: 4 sequences x 16 wave rows over 32k keys
        dict(name="attn_gqa_32k", kind="decode", rows=64, H=16, Hkv=4, Dh=128, lo=32700, hi=32768, dtype="bf16"),
        # a packed varlen call over mixed segments: single rows beside short
        # causal runs (a coda's verifies, re-entered tokens, chunked prompts)
        dict(name="varlen_mixed", kind="varlen", segs=48, max_q=64, lo=100, hi=2048, H=16, Hkv=16, Dh=128,
             causal=True, dtype="bf16"),
        # prompt attention, an ordinary batch of two and a long GQA prompt
        dict(name="dense_2k", kind="dense", B=2, Tq=2000, Tk=2000, H=16, Hkv=16, Dh=128, causal=True, dtype="bf16"),
        dict(name="dense_gqa_16k", kind="dense", B=1, Tq=16384, Tk=16384, H=16, Hkv=4, Dh=128, causal=True,
             dtype="bf16"),
        # the fused projection + RoPE of a prompt chunk through compute_qkv
        dict(name="qkv_1500", kind="qkv", B=1, T=1500, C=2048, H=16, Hkv=16, Dh=128, dtype="bf16"),
        # gated MLP + residual norms over the rows of a served batch's union
        dict(name="mlp_192", kind="mlp", rows=192, D=2048, F=5632, dtype="bf16"),
        # the head over a served batch's coda rows: logits and greedy ids
        dict(name="head_100", kind="head", rows=100, D=2048, V=32000, dtype="bf16"),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["tick", "tick", "prefill", "decode", "decode", "varlen", "varlen", "dense", "dense", "qkv",
                       "mlp", "mlp", "head"])
    H, Hkv, Dh = rng.choice([(16, 16, 128), (16, 16, 128), (16, 4, 128), (4, 4, 64), (4, 2, 64)])
    dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
    if kind == "tick":
        model = rng.choice(["tiny", "looped-2048", "looped-2048"])
        T = CONFIGS[model].T_total
        loops = rng.choice([1, T]) if model == "tiny" else 1
        width = rng.randint(1, min(8, T - loops + 1))
        batch = _log_int(rng, 1, 28)
        while batch * width > 112:
            width -= 1
        hi = _log_int(rng, 140, 1200)
        return dict(kind="tick", model=model, batch=batch, width=width, loops=loops, lo=rng.randint(100, hi), hi=hi)
    if kind == "prefill":
        return dict(kind="prefill", model=rng.choice(["tiny", "looped-2048"]), loops=1, length=_log_int(rng, 24, 700))
    if kind == "decode":
        hi = _log_int(rng, 64, 32768)
        rows = _log_int(rng, 1, min(256, max(8, 64 * 32768 // hi)))
        if H == Hkv == 16:
            rows = max(1, min(rows, 16 * 32768 // hi))
        return dict(kind="decode", rows=rows, H=H, Hkv=Hkv, Dh=Dh, lo=rng.randint(max(1, hi // 4), hi), hi=hi,
                    dtype="bf16" if hi > 4096 else dtype)
    if kind == "varlen":
        hi = _log_int(rng, 64, 2048)
        return dict(kind="varlen", segs=_log_int(rng, 1, 48), max_q=_log_int(rng, 1, 64), lo=rng.randint(1, hi), hi=hi,
                    H=H, Hkv=Hkv, Dh=Dh, causal=rng.random() < 0.7, dtype=dtype)
    if kind == "dense":
        if dtype == "f32":
            Tk = _log_int(rng, 20, 500)
            B = rng.randint(1, 2)
        else:
            Tk = _log_int(rng, 20, 8192)
            B = rng.randint(1, 3)
        causal = rng.random() < 0.8
        if not causal:
            Tk = min(Tk, 1000)
        Tq = Tk if rng.random() < 0.7 else rng.randint(1, Tk)
        return dict(kind="dense", B=B, Tq=Tq, Tk=Tk, H=H, Hkv=Hkv, Dh=Dh, causal=causal, dtype=dtype)
    if kind == "qkv":
        return dict(kind="qkv", B=rng.randint(1, 2), T=_log_int(rng, 1, 1500), C=1024 if dtype == "f32" else 2048,
                    H=H, Hkv=Hkv, Dh=Dh, dtype=dtype)
    if kind == "mlp":
        rows = _log_int(rng, 1, 300 if dtype == "f32" else 1500)
        D, F = (256, 1024) if dtype == "f32" else rng.choice([(2048, 5632), (2048, 5632), (512, 1536)])
        return dict(kind="mlp", rows=rows, D=D, F=F, dtype=dtype)
    D, V = (256, 4096) if dtype == "f32" else (2048, 32000)
    return dict(kind="head", rows=_log_int(rng, 1, 112), D=D, V=V, dtype=dtype)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed: int, device=DEV) -> torch.Generator:
    return torch.Generator(device=device).manual_seed(seed)


def _randn(g, *shape, dtype, std: float = 1.0) -> torch.Tensor:
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=g)


def _norm_weight(g, D: int, dtype) -> torch.Tensor:
    return _randn(g, D, dtype=torch.float32, std=0.1).add_(1.0).to(dtype)


def _lengths(case: dict, n: int, seed: int) -> list[int]:
    g = torch.Generator().manual_seed(seed + 77)
    return torch.randint(case["lo"], case["hi"] + 1, (n,), generator=g).tolist()


def _config(case: dict):
    """The case's model; a prompt pass runs its core `loops` times."""
    cfg = CONFIGS[case["model"]]
    return cfg.with_(T_total=case["loops"]) if case["kind"] == "prefill" else cfg


def _model_weights(cfg, g) -> dict[str, torch.Tensor]:
    """N(0, init_std) linears, norm weights around 1, in the run dtype."""
    D, F, dt = cfg.d_model, cfg.ffn, cfg.torch_dtype
    w = {"wte": _randn(g, cfg.vocab_size, D, dtype=dt, std=cfg.init_std)}
    for part, count in (("prelude", cfg.n_prelude), ("core", cfg.n_core), ("coda", cfg.n_coda)):
        for i in range(count):
            p = f"{part}.{i}."
            for leaf, N, K in (("Wqkv", cfg.qkv_dim, D), ("proj", D, cfg.n_heads * cfg.head_dim), ("fc", 2 * F, D),
                               ("mlp_proj", D, F)):
                w[p + leaf] = _randn(g, N, K, dtype=dt, std=cfg.init_std)
            for j in (1, 2, 3, 4):
                w[p + f"norm_{j}"] = _norm_weight(g, D, dt)
    w["adapter"] = _randn(g, D, 2 * D, dtype=dt, std=cfg.init_std)
    w["ln_f"] = _norm_weight(g, D, dt)
    w["lm_head"] = _randn(g, cfg.vocab_size, D, dtype=dt, std=cfg.init_std)
    return w


def _tick_rows(case: dict, cfg, seed: int):
    """(seqs, positions, first steps) of the wave: `width` rows per sequence at
    consecutive positions after its prefix, the oldest deepest in the loop."""
    w, T, r = case["width"], cfg.T_total, case["loops"]
    stride = (T - r) // (w - 1) if w > 1 else 0
    seqs, pos, steps = [], [], []
    for b, L in enumerate(_lengths(case, case["batch"], seed)):
        for j in range(w):
            seqs.append(b)
            pos.append(L + j)
            steps.append((w - 1 - j) * stride)
    return seqs, pos, steps


def _tick_cache_len(case: dict) -> int:
    return case["hi"] + case["width"] + 1


def _token_ids(cfg, n: int, seed: int) -> list[int]:
    return torch.randint(0, cfg.vocab_size, (n,), generator=torch.Generator().manual_seed(seed + 5)).tolist()


def _fill_std(cfg) -> float:
    """Spread of K / V values of a normalized row through N(0, init_std) weights."""
    return cfg.init_std * math.sqrt(cfg.d_model)


def _segments(case: dict):
    """(q lengths, k lengths): every third segment a single row, the rest up to max_q rows."""
    g = torch.Generator().manual_seed(78)
    k = _lengths(case, case["segs"], 0)
    q = torch.randint(1, case["max_q"] + 1, (case["segs"],), generator=g).tolist()
    return [1 if i % 3 == 0 else min(a, b) for i, (a, b) in enumerate(zip(q, k))], k


def _offsets(lens: list[int]) -> torch.Tensor:
    return torch.tensor([0] + lens).cumsum(0).to(torch.int32).to(DEV)


def prepare(case: dict, seed: int) -> dict:
    g, kind = _gen(seed), case["kind"]
    st = {"kind": kind, "case": case}
    if kind in ("tick", "prefill"):
        cfg = _config(case)
        w = _model_weights(cfg, g)
        if kind == "prefill":
            m = LoopedModel(cfg, w, DEV, max_seq_len=case["length"], max_batch=1)
            return st | dict(model=m, cache=m.create_cache(), ids=_token_ids(cfg, case["length"], seed))
        m = LoopedModel(cfg, w, DEV, max_seq_len=_tick_cache_len(case), max_batch=case["batch"], use_graphs=True)
        cache = m.create_cache()
        for t in (cache.flat_k, cache.flat_v):
            t.normal_(0.0, _fill_std(cfg), generator=g)
        seqs, pos, steps = _tick_rows(case, cfg, seed)
        passes = [("P", seqs, pos, _token_ids(cfg, len(seqs), seed))]
        passes += [("R", seqs, pos, [s + r for s in steps]) for r in range(case["loops"])]
        passes += [("C", seqs, pos, None)]
        st |= dict(model=m, cache=cache, passes=passes)
        run(st)  # a serving program has captured its tick before this request's
        return st
    dt = DTYPES[case["dtype"]]
    if kind == "decode":
        n, S, Hkv, Dh = case["rows"], case["hi"], case["Hkv"], case["Dh"]
        q = _randn(g, n, case["H"], Dh, dtype=dt)
        kc, vc = _randn(g, n, Hkv, S, Dh, dtype=dt), _randn(g, n, Hkv, S, Dh, dtype=dt)
        return st | dict(q=q, k=kc, v=vc, base=torch.arange(n, dtype=torch.int64, device=DEV) * S,
                         lens=torch.tensor(_lengths(case, n, seed), dtype=torch.int32, device=DEV))
    if kind == "varlen":
        ql, kl = _segments(case)
        q = _randn(g, sum(ql), case["H"], case["Dh"], dtype=dt)
        k = _randn(g, sum(kl), case["Hkv"], case["Dh"], dtype=dt)
        v = _randn(g, sum(kl), case["Hkv"], case["Dh"], dtype=dt)
        return st | dict(q=q, k=k, v=v, cu_q=_offsets(ql), cu_k=_offsets(kl), max_q=max(ql), max_k=max(kl))
    if kind == "dense":
        B, Dh = case["B"], case["Dh"]
        return st | dict(q=_randn(g, B, case["Tq"], case["H"], Dh, dtype=dt),
                         k=_randn(g, B, case["Tk"], case["Hkv"], Dh, dtype=dt),
                         v=_randn(g, B, case["Tk"], case["Hkv"], Dh, dtype=dt))
    if kind == "qkv":
        H, Hkv, Dh, C = case["H"], case["Hkv"], case["Dh"], case["C"]
        x = _randn(g, case["B"], case["T"], C, dtype=dt)
        W = _randn(g, (H + 2 * Hkv) * Dh, C, dtype=dt, std=0.02)
        cos, sin = _rope(case["T"], Dh)
        attn = SimpleNamespace(Wqkv=ops.pack_linear(W), n_head=H, n_kv_head=Hkv, head_dim=Dh)
        return st | dict(x=x, W=W, attn=attn, freqs=torch.complex(cos, sin).to(torch.complex64))
    if kind == "mlp":
        n, D, F = case["rows"], case["D"], case["F"]
        x, h = _randn(g, n, D, dtype=dt), _randn(g, n, D, dtype=dt)
        fc, down = _randn(g, 2 * F, D, dtype=dt, std=0.02), _randn(g, D, F, dtype=dt, std=0.02)
        return st | dict(x=x, h=h, fc=fc, down=down, fcp=ops.pack_linear(fc, swiglu=True),
                         downp=ops.pack_linear(down), w1=_norm_weight(g, D, dt), w2=_norm_weight(g, D, dt))
    assert kind == "head"
    h, W = _randn(g, case["rows"], case["D"], dtype=dt), _randn(g, case["V"], case["D"], dtype=dt, std=0.02)
    return st | dict(h=h, W=W, Wp=ops.pack_linear(W))


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st: dict):
    kind = st["kind"]
    if kind == "tick":
        m = st["model"]
        logits, _ = m.run_passes(st["cache"], st["passes"])
        # every row's logits, and the loop and static state of every token (the
        # last pool row only absorbs padding rows)
        return {"logits": logits, "state": m.pool[: m.trash_pool_row]}
    if kind == "prefill":
        logits = st["model"].prefill_seq(st["cache"], 0, st["ids"])
        return {"logits": logits, "k": st["cache"].flat_k, "v": st["cache"].flat_v}
    if kind == "decode":
        return ops.attn_decode(st["q"], st["k"], st["v"], st["base"], st["lens"], kv_len_max=st["case"]["hi"])
    if kind == "varlen":
        return attention.attn_varlen(st["q"], st["k"], st["v"], st["cu_q"], st["cu_k"], st["max_q"], st["max_k"],
                                     causal=st["case"]["causal"])
    if kind == "dense":
        return attention.attn_dense(st["q"], st["k"], st["v"], causal=st["case"]["causal"])
    if kind == "qkv":
        return attention.compute_qkv(st["attn"], st["x"], st["freqs"])
    if kind == "mlp":
        u = ops.linear(st["h"], st["fcp"], swiglu=True)
        m = ops.linear(u, st["downp"])
        return ops.add_rmsnorm(m, st["w1"], EPS, res=st["x"], w2=st["w2"])
    logits = ops.linear(st["h"], st["Wp"], out_dtype=torch.float32)
    return logits, ops.argmax(logits)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _block_work(cfg, n: int, keys: int, el: int) -> tuple[float, float]:
    """(bytes, flops) of one block over n rows that read `keys` keys in all: its
    weights once, the rows' keys and values, their append, the rows in and out."""
    D, F, Hd, Kd = cfg.d_model, cfg.ffn, cfg.n_heads * cfg.head_dim, cfg.n_kv_heads * cfg.head_dim
    weights = cfg.qkv_dim * D + D * Hd + 3 * F * D + 4 * D
    return ((weights + 2 * Kd * (keys + n) + 2 * n * D) * el,
            2.0 * n * (cfg.qkv_dim * D + D * Hd + 3 * F * D) + 4.0 * keys * Hd)


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind in ("tick", "prefill"):
        cfg = _config(case)
        el, D = (2 if cfg.torch_dtype == torch.bfloat16 else 4), cfg.d_model
        if kind == "tick":
            n = case["batch"] * case["width"]
            # mean prefix of the drawn range (rows of one sequence share a slot's keys in P and C)
            mean = (case["lo"] + case["hi"]) / 2 + (case["width"] + 1) / 2
            shared = case["batch"] * (mean + (case["width"] - 1) / 2)
            loops, head_rows = case["loops"], n
            pre = _block_work(cfg, n, shared, el)
            core = _block_work(cfg, n, n * mean, el)
            flops_extra = 4.0 * (n * mean - shared) * cfg.n_heads * cfg.head_dim * (cfg.n_prelude + cfg.n_coda)
        else:
            n = case["length"]
            loops, head_rows = cfg.T_total, 1
            pre = core = _block_work(cfg, n, 0, el)
            flops_extra = (4.0 * n * (n + 1) / 2 * cfg.n_heads * cfg.head_dim) * cfg.n_slots
        outer = cfg.n_prelude + cfg.n_coda
        b = outer * pre[0] + loops * (cfg.n_core * core[0] + (2 * D * D + 3 * n * D) * el)
        f = outer * pre[1] + loops * (cfg.n_core * core[1] + 4.0 * n * D * D) + flops_extra
        b += cfg.vocab_size * D * el + head_rows * cfg.vocab_size * 4 + n * D * el
        return {"bytes": b, "flops": f + 2.0 * head_rows * D * cfg.vocab_size}
    el = 2 if case["dtype"] == "bf16" else 4
    if kind == "decode":
        n, mean = case["rows"], (case["lo"] + case["hi"]) / 2
        return {"bytes": (2 * n * mean * case["Hkv"] + 2 * n * case["H"]) * case["Dh"] * el,
                "flops": 4.0 * n * mean * case["H"] * case["Dh"]}
    if kind == "varlen":
        ql, kl = _segments(case)
        pairs = sum(q * k - (q * (q - 1) / 2 if case["causal"] else 0) for q, k in zip(ql, kl))
        return {"bytes": (2 * sum(ql) * case["H"] + 2 * sum(kl) * case["Hkv"]) * case["Dh"] * el,
                "flops": 4.0 * pairs * case["H"] * case["Dh"]}
    if kind == "dense":
        B, q, k = case["B"], case["Tq"], case["Tk"]
        pairs = B * (q * k - (q * (q - 1) / 2 if case["causal"] else 0))
        return {"bytes": B * (2 * q * case["H"] + 2 * k * case["Hkv"]) * case["Dh"] * el,
                "flops": 4.0 * pairs * case["H"] * case["Dh"]}
    if kind == "qkv":
        n, N = case["B"] * case["T"], (case["H"] + 2 * case["Hkv"]) * case["Dh"]
        return {"bytes": (n * case["C"] + N * case["C"] + n * N) * el, "flops": 2.0 * n * N * case["C"]}
    n, D = case["rows"], case["D"]
    if kind == "mlp":
        return {"bytes": (3 * D * case["F"] + 4 * n * D) * el, "flops": 6.0 * n * D * case["F"]}
    return {"bytes": (n * D + case["V"] * D) * el + n * case["V"] * 4 + n * 8, "flops": 2.0 * n * D * case["V"]}


def tolerance(case: dict):
    """About four times what the same path differs by from 64-bit arithmetic
    (or, for whole passes, from itself with a norm's rounding moved)."""
    kind = case["kind"]
    if kind in ("tick", "prefill"):
        # bf16 rounding of every layer's rows carries through the layers after it
        return {"rel": 2e-5} if case["model"] == "tiny" else {"rel": 3e-2}
    if kind == "head":
        # ids of near-equal logits may swap; logits are 32-bit sums
        return {"rel": 2e-6, "differ": 0.01}
    if case["dtype"] == "f32":
        return {"rel": 1e-5}
    return {"rel": 1e-2}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------
def _rope(T: int, Dh: int, base: float = 10000.0) -> tuple[torch.Tensor, torch.Tensor]:
    """(T, Dh / 2) float32 cos / sin of pos * base^(-2j / Dh)."""
    theta = base ** (-2.0 * torch.arange(Dh // 2, dtype=torch.float64) / Dh)
    ang = torch.arange(T, dtype=torch.float64)[:, None] * theta[None]
    return ang.cos().float().to(DEV), ang.sin().float().to(DEV)


def _rotate(x: torch.Tensor, cos: torch.Tensor, sin: torch.Tensor) -> torch.Tensor:
    """Interleaved-pair rotation of x (n, heads, Dh) by cos / sin (n, Dh / 2)."""
    c, s = cos.double()[:, None], sin.double()[:, None]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * c - b * s, a * s + b * c], dim=-1).flatten(-2)


def _rms(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, causal: bool) -> torch.Tensor:
    """q (Tq, H, Dh) over k / v (Tk, Hkv, Dh), bottom-right causal, in float64."""
    Tq, H, Dh = q.shape
    Tk, Hkv, _ = k.shape
    out = torch.zeros(Tq, H, Dh, dtype=torch.float64, device=q.device)
    last = torch.arange(Tq, device=q.device)[:, None] + (Tk - Tq)
    for h in range(H):
        kh, vh = k[:, h // (H // Hkv)].double(), v[:, h // (H // Hkv)].double()
        for i in range(0, Tq, 4096):
            s = q[i: i + 4096, h].double() @ kh.t() / math.sqrt(Dh)
            if causal:
                s.masked_fill_(torch.arange(Tk, device=q.device)[None] > last[i: i + 4096], -math.inf)
            out[i: i + 4096, h] = torch.nan_to_num(torch.softmax(s, -1), nan=0.0) @ vh
    return out


def _mlp(h: torch.Tensor, fc: torch.Tensor, down: torch.Tensor) -> torch.Tensor:
    gu = h @ fc.double().t()
    F = fc.shape[0] // 2
    return (torch.nn.functional.silu(gu[:, :F]) * gu[:, F:]) @ down.double().t()


def _block(w: dict, p: str, cfg, x: torch.Tensor, cos, sin, attend) -> torch.Tensor:
    """One sandwich block; attend(q, k, v) appends the rows' k / v and reads the slots."""
    n, H, Hkv, Dh = x.shape[0], cfg.n_heads, cfg.n_kv_heads, cfg.head_dim
    qkv = _rms(x, w[p + "norm_1"]) @ w[p + "Wqkv"].double().t()
    q, k, v = qkv.view(n, -1, Dh).split([H, Hkv, Hkv], dim=1)
    o = attend(_rotate(q, cos, sin), _rotate(k, cos, sin), v)
    x = _rms(o.reshape(n, -1) @ w[p + "proj"].double().t() + x, w[p + "norm_2"])
    return _rms(_mlp(_rms(x, w[p + "norm_3"]), w[p + "fc"], w[p + "mlp_proj"]) + x, w[p + "norm_4"])


def _s0(cfg, seed: int, shape) -> torch.Tensor:
    out = torch.zeros(shape)
    torch.nn.init.trunc_normal_(out, std=cfg.state_std, a=-3 * cfg.state_std, b=3 * cfg.state_std,
                                generator=torch.Generator().manual_seed(seed))
    return (out * cfg.emb_scale).to(cfg.torch_dtype).to(DEV).double()


def _exact_tick(case: dict, seed: int):
    cfg, g = _config(case), _gen(seed)
    w = _model_weights(cfg, g)
    S, B = _tick_cache_len(case), case["batch"]
    cache = [_randn(g, cfg.n_slots * B + 1, cfg.n_kv_heads, S, cfg.head_dim, dtype=cfg.torch_dtype,
                    std=_fill_std(cfg)) for _ in range(2)]
    seqs, pos, steps = _tick_rows(case, cfg, seed)
    ids, n = _token_ids(cfg, len(seqs), seed), len(seqs)
    cos, sin = (t[pos] for t in _rope(S, cfg.head_dim, cfg.rope_base))
    written: dict = {}  # (block of the cache) -> {position: (k, v)}

    def attend_at(slots):
        def attend(q, k, v):
            for i in range(n):
                written.setdefault(slots[i] * B + seqs[i], {})[pos[i]] = (k[i], v[i])
            out = []
            for i in range(n):
                blk = slots[i] * B + seqs[i]
                kk, vv = (t[blk, :, : pos[i] + 1].double() for t in cache)
                for p, (kp, vp) in written[blk].items():
                    if p <= pos[i]:
                        kk[:, p], vv[:, p] = kp, vp
                out.append(_attend(q[i: i + 1], kk.transpose(0, 1), vv.transpose(0, 1), False))
            return torch.cat(out)
        return attend

    e = w["wte"][ids].double() * cfg.emb_scale
    for i in range(cfg.n_prelude):
        e = _block(w, f"prelude.{i}.", cfg, e, cos, sin, attend_at([i] * n))
    s = torch.stack([_s0(cfg, p + 1, (cfg.d_model,)) for p in pos])
    for r in range(case["loops"]):
        x = torch.cat([s, e], 1) @ w["adapter"].double().t()
        for i in range(cfg.n_core):
            slots = [cfg.n_prelude + (t + r) * cfg.n_core + i for t in steps]
            x = _block(w, f"core.{i}.", cfg, x, cos, sin, attend_at(slots))
        s = x
    x = _rms(s, w["ln_f"])
    for i in range(cfg.n_coda):
        x = _block(w, f"coda.{i}.", cfg, x, cos, sin, attend_at([cfg.n_prelude + cfg.T_total * cfg.n_core + i] * n))
    logits = _rms(x, w["ln_f"]) @ w["lm_head"].double().t()
    # the pool keeps T_total + 2 rows per sequence, a position's row by its remainder
    state = torch.zeros(B * (cfg.T_total + 2), 2 * cfg.d_model, dtype=torch.float64, device=DEV)
    rows = [b * (cfg.T_total + 2) + p % (cfg.T_total + 2) for b, p in zip(seqs, pos)]
    state[rows] = torch.cat([s, e], 1)
    return {"logits": logits, "state": state}


def _exact_prefill(case: dict, seed: int):
    cfg, g, L = _config(case), _gen(seed), case["length"]
    w = _model_weights(cfg, g)
    cos, sin = _rope(L, cfg.head_dim, cfg.rope_base)
    shape = (cfg.n_slots + 1, cfg.n_kv_heads, L, cfg.head_dim)
    K, V = (torch.zeros(shape, dtype=torch.float64, device=DEV) for _ in range(2))

    def attend_at(slot):
        def attend(q, k, v):
            K[slot], V[slot] = k.transpose(0, 1), v.transpose(0, 1)
            return _attend(q, k, v, True)
        return attend

    e = w["wte"][_token_ids(cfg, L, seed)].double() * cfg.emb_scale
    for i in range(cfg.n_prelude):
        e = _block(w, f"prelude.{i}.", cfg, e, cos, sin, attend_at(i))
    s = _s0(cfg, 0, (1, L, cfg.d_model))[0]
    for r in range(cfg.T_total):
        s = torch.cat([s, e], 1) @ w["adapter"].double().t()
        for i in range(cfg.n_core):
            s = _block(w, f"core.{i}.", cfg, s, cos, sin, attend_at(cfg.n_prelude + r * cfg.n_core + i))
    x = _rms(s, w["ln_f"])
    for i in range(cfg.n_coda):
        x = _block(w, f"coda.{i}.", cfg, x, cos, sin, attend_at(cfg.n_prelude + cfg.T_total * cfg.n_core + i))
    logits = _rms(x[-1:], w["ln_f"]) @ w["lm_head"].double().t()
    return {"logits": logits[0], "k": K, "v": V}


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind == "tick":
        return _exact_tick(case, seed)
    if kind == "prefill":
        return _exact_prefill(case, seed)
    st = prepare(case, seed)
    if kind == "decode":
        lens = st["lens"].tolist()
        return torch.cat([_attend(st["q"][i: i + 1], st["k"][i, :, :L].transpose(0, 1),
                                  st["v"][i, :, :L].transpose(0, 1), False) for i, L in enumerate(lens)])
    if kind == "varlen":
        cq, ck = st["cu_q"].tolist(), st["cu_k"].tolist()
        return torch.cat([_attend(st["q"][cq[i]: cq[i + 1]], st["k"][ck[i]: ck[i + 1]], st["v"][ck[i]: ck[i + 1]],
                                  case["causal"]) for i in range(len(cq) - 1)])
    if kind == "dense":
        # a lone query attends the whole prefix either way
        return torch.stack([_attend(st["q"][b], st["k"][b], st["v"][b], case["causal"]) for b in range(case["B"])])
    if kind == "qkv":
        B, T, H, Hkv, Dh = (case[k] for k in ("B", "T", "H", "Hkv", "Dh"))
        qkv = (st["x"].reshape(B * T, -1).double() @ st["W"].double().t()).view(B * T, -1, Dh)
        q, k, v = qkv.split([H, Hkv, Hkv], dim=1)
        cos, sin = (t.repeat(B, 1) for t in _rope(T, Dh))
        return (_rotate(q, cos, sin).view(B, T, H, Dh), _rotate(k, cos, sin).view(B, T, Hkv, Dh),
                v.reshape(B, T, Hkv, Dh))
    if kind == "mlp":
        x = _rms(_mlp(st["h"].double(), st["fc"], st["down"]) + st["x"].double(), st["w1"])
        return x, _rms(x, st["w2"])
    return st["h"].double() @ st["W"].double().t(), None
