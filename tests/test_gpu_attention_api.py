"""The reference's attention-backend API (wavefront_decoding_amd.attention)
against the oracle (GPU).

Each entry point is called with the argument layout the reference's callers
use (src/decoding/fa4_attention.py:191-342): packed varlen segments with
cu_seqlens, dense (B, T, H, Dh) batches, the coda's per-query cutoff, and the
q1 padded form. Tolerance: max relative error 2e-2 (bf16) / 1e-4 (fp32).
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import kernels as ok
from tests.conftest import rel_err
from wavefront_decoding_amd import attention as A
from wavefront_decoding_amd import ops

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 2e-2, torch.float32: 1e-4}


def _np(t):
    return t.detach().float().cpu().numpy().astype(np.float64)


def _varlen_ref(q, k, v, cu_q, cu_k, causal):
    """Oracle: each segment's rows over the segment's keys, bottom-right causal
    per segment when asked (rows with no keys are zero)."""
    qn, kn, vn = _np(q), _np(k), _np(v)
    out = np.zeros_like(qn)
    for s in range(len(cu_q) - 1):
        q0, q1, k0, k1 = cu_q[s], cu_q[s + 1], cu_k[s], cu_k[s + 1]
        ql, kl = q1 - q0, k1 - k0
        for r in range(ql):
            n = max(kl - ql + r + 1, 0) if causal else kl
            out[q0 + r] = ok.attention(qn[q0 + r], kn[k0:k1], vn[k0:k1], n)
    return out


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("H,Hkv,Dh", [(16, 16, 128), (16, 4, 128), (4, 4, 64)])
def test_attn_varlen_matches_oracle(gpu, dtype, causal, H, Hkv, Dh):
    """Packed segments of ragged query and key lengths, including one with
    fewer keys than queries (its first rows have no keys under causal) and a
    long one that spans several key splits."""
    seg = [(1, 700), (5, 5), (3, 1), (8, 2500), (1, 1), (4, 33)]  # (q_len, k_len)
    cu_q = np.concatenate([[0], np.cumsum([a for a, _ in seg])]).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum([b for _, b in seg])]).astype(np.int32)
    g = torch.Generator().manual_seed(H * 7 + Dh + causal)
    q = torch.randn(int(cu_q[-1]), H, Dh, generator=g).to(dtype)
    k = torch.randn(int(cu_k[-1]), Hkv, Dh, generator=g).to(dtype)
    v = torch.randn(int(cu_k[-1]), Hkv, Dh, generator=g).to(dtype)
    print(f"[attn_varlen] dtype={dtype} causal={causal} H={H} Hkv={Hkv} Dh={Dh}", flush=True)
    out = A.attn_varlen(q.to(gpu), k.to(gpu), v.to(gpu), torch.from_numpy(cu_q).to(gpu),
                        torch.from_numpy(cu_k).to(gpu), max(a for a, _ in seg), max(b for _, b in seg), causal=causal)
    ref = _varlen_ref(q, k, v, cu_q, cu_k, causal)
    assert rel_err(_np(out), ref) <= TOL[dtype]
    if causal:  # rows with no keys come back as zeros
        assert torch.count_nonzero(out[cu_q[2]: cu_q[2] + 2].float()) == 0


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("H,Hkv,Dh", [(4, 4, 128), (8, 2, 128), (4, 2, 64), (2, 2, 64)])
def test_attn_varlen_shared_rows(gpu, causal, H, Hkv, Dh):
    """The kernel that reads a key once for the rows of a segment, at the edges
    of its row tiles (32 / G rows), key tiles (32) and splits (1024), with rows
    outside every segment, an empty segment, segments with fewer keys than rows
    and none, and more segments than its table workgroup has threads. Error
    against float64 relative to the result's norm: at most the bf16 output
    rounding (2^-9) plus that of the probabilities' two bf16 terms (2^-17),
    three times over for rows whose values cancel. A row alone in its segment
    (bottom-right causal: its last row) has the same bits as in the full one."""
    T = 32 // (H // Hkv)
    seg = [(T, 31), (1, 32), (T + 1, 33), (0, 5), (2 * T - 1, 1024), (3, 1025), (2, 2100), (5, 2), (4, 0), (1, 1)]
    seg += [(1 + i % 2, 1 + i % 40) for i in range(300)]
    lead, tail = 3, 2
    cu_q = lead + np.concatenate([[0], np.cumsum([a for a, _ in seg])]).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum([b for _, b in seg])]).astype(np.int32)
    n = int(cu_q[-1]) + tail
    g = torch.Generator().manual_seed(H + Dh + causal)
    mk = lambda r, h: torch.randn(r, h, Dh, generator=g).to(torch.bfloat16)  # noqa: E731
    q, k, v = mk(n, H), mk(int(cu_k[-1]), Hkv), mk(int(cu_k[-1]), Hkv)
    print(f"[attn_varlen shared rows] causal={causal} H={H} Hkv={Hkv} Dh={Dh}", flush=True)
    dev = [t.to(gpu) for t in (q, k, v)]
    cq, ck = torch.from_numpy(cu_q).to(gpu), torch.from_numpy(cu_k).to(gpu)
    shared = lambda q_, k_, v_, a, b, mk_: ops.attn_varlen(q_, k_, v_, a, b, max_k=mk_, causal=causal)  # noqa: E731
    out = shared(*dev, cq, ck, max(b for _, b in seg))
    ref = np.zeros((n, H, Dh))
    ref[lead: int(cu_q[-1])] = _varlen_ref(q[lead:], k, v, cu_q - lead, cu_k, causal)[: int(cu_q[-1]) - lead]
    got = _np(out)
    assert np.linalg.norm(got - ref) <= 3 * 2.0 ** -9 * np.linalg.norm(ref)
    assert rel_err(got, ref) <= TOL[torch.bfloat16]
    assert not got[:lead].any() and not got[n - tail:].any()  # outside every segment
    # the last row of each of the first segments, among one-row segments and a two-row one
    last = [i for i, (a, _) in enumerate(seg[:10]) if a > 0]
    rows = torch.tensor([int(cu_q[i + 1]) - 1 for i in last], device=gpu)
    qs = torch.cat([dev[0][rows], dev[0][:2]])
    ks = torch.cat([dev[1][cu_k[i]: cu_k[i + 1]] for i in last] + [dev[1][:7]])
    vs = torch.cat([dev[2][cu_k[i]: cu_k[i + 1]] for i in last] + [dev[2][:7]])
    kl = [seg[i][1] for i in last] + [7]
    off = lambda x: torch.tensor(np.concatenate([[0], np.cumsum(x)]), dtype=torch.int32, device=gpu)  # noqa: E731
    alone = shared(qs, ks, vs, off([1] * len(last) + [2]), off(kl), max(kl))
    assert torch.equal(alone[: len(last)], out[rows])


@pytest.mark.parametrize("rows,causal", [(3, True), (70, True), (70, False)])
def test_attn_varlen_routes_agree(gpu, rows, causal):
    """attn_varlen and non-causal attn_dense on both sides of the choice of
    kernel (three rows a segment: the decode kernel; 70: the shared-rows one)
    against the decode kernel's rows: each is within bf16 rounding of float64."""
    H, Hkv, Dh, segs, Tk = 4, 4, 128, 5, 130
    g = torch.Generator().manual_seed(rows)
    q, k, v = (torch.randn(segs * r, h, Dh, generator=g).to(torch.bfloat16).to(gpu)
               for r, h in ((rows, H), (Tk, Hkv), (Tk, Hkv)))
    cq, ck = (torch.arange(segs + 1, dtype=torch.int32, device=gpu) * t for t in (rows, Tk))
    assert A._shared_rows(segs * rows, segs, Tk, H, Hkv, Dh) == (rows == 70)
    rb, kl = ops.attn_varlen_rows(cq, ck, segs * rows, causal=causal)
    ref = ops.attn_decode(q, k, v, rb, kl, kv_len_max=Tk).float()
    outs = [A.attn_varlen(q, k, v, cq, ck, rows, Tk, causal=causal)]
    if not causal:
        outs.append(A.attn_dense(q.view(segs, rows, H, Dh), k.view(segs, Tk, Hkv, Dh), v.view(segs, Tk, Hkv, Dh),
                                 causal=False).view_as(q))
    for out in outs:  # two bf16 roundings of the same value
        assert (out.float() - ref).norm() <= 2.0 ** -8 * ref.norm()


def test_attn_varlen_shared_rows_special_values(gpu):
    """Infinities and NaN stay with the rows that attend them: a causal segment
    whose last keys' V hold them leaves the rows before those keys finite (and,
    before the 32-key tile that holds them, bit for bit the same), and the rows
    that attend an infinity get it."""
    g = torch.Generator().manual_seed(3)
    n, H, Dh = 60, 2, 128
    q, k, v = (torch.randn(n, H, Dh, generator=g).to(torch.bfloat16).to(gpu) for _ in range(3))
    cu = torch.tensor([0, n], dtype=torch.int32, device=gpu)
    plain = ops.attn_varlen(q, k, v, cu, cu, max_k=n, causal=True)
    v[40, 0, 5] = float("inf")
    v[50, 1, 7] = float("nan")
    got = ops.attn_varlen(q, k, v, cu, cu, max_k=n, causal=True)
    assert torch.equal(got[:32], plain[:32])
    assert torch.isinf(got[40:, 0, 5]).all() and torch.isnan(got[50:, 1, 7]).all()
    clean = torch.ones_like(got, dtype=torch.bool)
    clean[40:, 0, 5] = clean[50:, 1, 7] = False
    assert torch.isfinite(got[clean].float()).all()
    # the tile that holds them was summed key by key in fp32: the other values agree to bf16 rounding
    d = (got.float() - plain.float())[clean].norm() / plain.float()[clean].norm()
    assert d <= 2.0 ** -8


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("H,Hkv,Dh", [(16, 16, 128), (16, 8, 128), (16, 4, 128), (4, 4, 64), (4, 2, 64), (8, 2, 64)])
def test_attn_varlen_rows_keep_their_bits(gpu, causal, H, Hkv, Dh):
    """A row of a packed call has the bits of that row decoded alone, whatever
    else the call holds: short calls, calls of many rows, other segments around
    it, at the edges of row tiles (16 / G rows), key tiles and splits, with
    scores from flat to so steep that probabilities underflow."""
    T = 16 // (H // Hkv)
    probe = [(T, 31), (T + 1, 33), (1, 64), (2, 1), (2 * T - 1, 1024), (3, 1025), (T, 2100), (5, 2), (3, 65)]
    many = probe + [(40, 50 + i) for i in range(1400 // (40 * Hkv) + 12)]
    nq, nk = (sum(x[i] for x in many) for i in (0, 1))
    g = torch.Generator().manual_seed(H + Hkv + Dh + causal)
    mk = lambda r, h: torch.randn(r, h, Dh, generator=g).to(torch.bfloat16).to(gpu)  # noqa: E731
    q, k, v = mk(nq, H), mk(nk, Hkv), mk(nk, Hkv)
    q *= torch.logspace(-2, 1.3, nq, device=gpu)[torch.randperm(nq, generator=g).to(gpu), None, None].to(q.dtype)
    off = lambda x: torch.tensor(np.concatenate([[0], np.cumsum(x)]), dtype=torch.int32, device=gpu)  # noqa: E731
    print(f"[attn_varlen bits] causal={causal} H={H} Hkv={Hkv} Dh={Dh}", flush=True)

    def call(segs, q_, k_, v_, fn):
        cq, ck, mk_ = off([a for a, _ in segs]), off([b for _, b in segs]), max(b for _, b in segs)
        return fn(q_, k_, v_, cq, ck, max(a for a, _ in segs), mk_)

    def rows(q_, k_, v_, cq, ck, mq, mk_):
        rb, kl = ops.attn_varlen_rows(cq, ck, q_.shape[0], causal=causal)
        return ops.attn_decode(q_, k_, v_, rb, kl, kv_len_max=mk_)

    api = lambda *a: A.attn_varlen(*a, causal=causal)  # noqa: E731
    shared = lambda q_, k_, v_, cq, ck, mq, mk_: ops.attn_varlen(q_, k_, v_, cq, ck, max_k=mk_, causal=causal)  # noqa: E731
    assert A._shared_rows(nq, len(many), 2100, H, Hkv, Dh)
    want = call(many, q, k, v, rows)
    assert torch.equal(call(many, q, k, v, shared), want)
    assert torch.equal(call(many, q, k, v, api), want)
    q0 = k0 = 0
    for a, b in probe:
        args = q[q0: q0 + a], k[k0: k0 + b], v[k0: k0 + b]
        for fn in (api, shared):
            assert torch.equal(call([(a, b)], *args, fn), want[q0: q0 + a]), (a, b)
        last = call([(1, b)], args[0][-1:], *args[1:], api)  # bottom-right: the segment's last row by itself
        assert torch.equal(last, want[q0 + a - 1: q0 + a]), (a, b)
        q0, k0 = q0 + a, k0 + b
    if not causal:  # a dense call of many rows: one segment per batch row
        B, Tq, Tk = 3, 1600 // Hkv, 70
        d = [x[: B * t].view(B, t, -1, Dh) for x, t in ((mk(B * Tq, H), Tq), (k, Tk), (v, Tk))]
        assert A._shared_rows(B * Tq, B, Tk, H, Hkv, Dh)
        out = A.attn_dense(*d, causal=False)
        for i in (0, 7, Tq - 1):
            assert torch.equal(A.attn_dense(d[0][:, i: i + 1], *d[1:], causal=False), out[:, i: i + 1])


@pytest.mark.parametrize("Hkv,Dh", [(2, 128), (1, 128), (2, 64)])
def test_attn_varlen_special_values_stay_with_their_rows(gpu, Hkv, Dh):
    """Infinities and NaN in V change no bit of a row that does not attend them,
    in the key tile that holds them too, nor another column of one that does."""
    g = torch.Generator().manual_seed(4)
    n, H = 90, 2
    q, k, v = (torch.randn(n, h, Dh, generator=g).to(torch.bfloat16).to(gpu) for h in (H, Hkv, Hkv))
    cu = torch.tensor([0, n], dtype=torch.int32, device=gpu)
    plain = ops.attn_varlen(q, k, v, cu, cu, max_k=n, causal=True)
    v[40, 0, 5] = float("inf")
    v[70, Hkv - 1, 7] = float("nan")
    v[71, Hkv - 1, 8] = float("-inf")
    got = ops.attn_varlen(q, k, v, cu, cu, max_k=n, causal=True)
    inf_heads, last_heads = slice(0, H // Hkv), slice(H - H // Hkv, H)
    assert (got[40:, inf_heads, 5] == float("inf")).all()
    assert torch.isnan(got[70:, last_heads, 7]).all() and (got[71:, last_heads, 8] == float("-inf")).all()
    clean = torch.ones_like(got, dtype=torch.bool)
    clean[40:, inf_heads, 5] = clean[70:, last_heads, 7] = clean[71:, last_heads, 8] = False
    assert torch.equal(got[clean], plain[clean])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_attn_varlen_q1_padded_matches_oracle(gpu, dtype):
    lens = [1, 64, 300, 1025, 7]
    cu_k = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    g = torch.Generator().manual_seed(5)
    q = torch.randn(len(lens), 16, 128, generator=g).to(dtype)
    k = torch.randn(int(cu_k[-1]), 16, 128, generator=g).to(dtype)
    v = torch.randn(int(cu_k[-1]), 16, 128, generator=g).to(dtype)
    out = A.attn_varlen_q1_padded(q.to(gpu), k.to(gpu), v.to(gpu), torch.from_numpy(cu_k).to(gpu), max(lens))
    ref = _varlen_ref(q, k, v, np.arange(len(lens) + 1), cu_k, False)
    assert rel_err(_np(out), ref) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("B,Tq,Tk,H,Hkv,Dh", [(2, 200, 200, 16, 4, 128), (3, 7, 150, 4, 4, 64),
                                             (1, 1, 300, 16, 16, 128), (2, 40, 20, 4, 2, 64), (1, 9, 60, 4, 2, 64)])
def test_attn_dense_matches_oracle(gpu, dtype, causal, B, Tq, Tk, H, Hkv, Dh):
    """Bottom-right causal (or full) dense attention over (B, T, H, Dh)
    batches: bf16 prompts go through the MFMA prefill kernel, the rest through
    the decode kernel; Tq > Tk leaves the first rows without keys (zeros)."""
    g = torch.Generator().manual_seed(B * 100 + Tq + Tk)
    q = torch.randn(B, Tq, H, Dh, generator=g).to(dtype)
    k = torch.randn(B, Tk, Hkv, Dh, generator=g).to(dtype)
    v = torch.randn(B, Tk, Hkv, Dh, generator=g).to(dtype)
    out = A.attn_dense(q.to(gpu), k.to(gpu), v.to(gpu), causal=causal)
    qn, kn, vn = _np(q), _np(k), _np(v)
    ref = np.zeros_like(qn)
    for b in range(B):
        for j in range(Tq):
            n = max(Tk - Tq + j + 1, 0) if (causal and Tq > 1) else Tk
            ref[b, j] = ok.attention(qn[b, j], kn[b], vn[b], n)
    assert out.shape == q.shape
    assert rel_err(_np(out), ref) <= TOL[dtype]


def test_attn_cutoff_multi_matches_oracle(gpu):
    """The coda's verify + draft rows at disjoint positions on one slot."""
    g = torch.Generator().manual_seed(9)
    qpos = [510, 517, 600]
    Tk = max(qpos) + 1
    q = torch.randn(1, 3, 16, 128, generator=g).to(torch.bfloat16)
    k = torch.randn(1, Tk, 16, 128, generator=g).to(torch.bfloat16)
    v = torch.randn(1, Tk, 16, 128, generator=g).to(torch.bfloat16)
    for pos in (qpos, torch.tensor(qpos, device=gpu)):
        out = A.attn_cutoff_multi(q.to(gpu), k.to(gpu), v.to(gpu), pos)
        ref = np.stack([ok.attention(_np(q)[0, j], _np(k)[0], _np(v)[0], p + 1) for j, p in enumerate(qpos)])
        assert rel_err(_np(out)[0], ref) <= 2e-2


def test_compute_qkv_matches_oracle(gpu):
    """Fused Wqkv projection + interleaved-pair RoPE at given positions."""
    from wavefront_decoding_amd.model import rope_tables

    class Attn:
        n_head, n_kv_head, head_dim = 4, 2, 64

    g = torch.Generator().manual_seed(2)
    B, T, C = 2, 5, 256
    N = (4 + 2 * 2) * 64
    Attn.Wqkv = (0.05 * torch.randn(N, C, generator=g)).to(gpu)
    x = torch.randn(B, T, C, generator=g).to(gpu)
    cos, sin = rope_tables(64, 64, 10000.0)
    pos = torch.tensor([3, 4, 9, 10, 40], dtype=torch.int32)
    q, k, v = A.compute_qkv(Attn, x, (cos.to(gpu), sin.to(gpu), pos.to(gpu)))
    qkv = _np(x).reshape(B * T, C) @ _np(Attn.Wqkv).T
    oc, os_ = ok.rope_tables(64, 64)
    for r in range(B * T):
        p = int(pos[r % T])
        qr = ok.rope(qkv[r, :256].reshape(4, 64), p, oc, os_)
        kr = ok.rope(qkv[r, 256:384].reshape(2, 64), p, oc, os_)
        assert rel_err(_np(q).reshape(B * T, 4, 64)[r], qr) <= 1e-4
        assert rel_err(_np(k).reshape(B * T, 2, 64)[r], kr) <= 1e-4
        assert rel_err(_np(v).reshape(B * T, 2, 64)[r], qkv[r, 384:].reshape(2, 64)) <= 1e-4


@pytest.mark.parametrize("dtype,H,Hkv,Dh", [(torch.bfloat16, 16, 16, 128), (torch.bfloat16, 16, 4, 128),
                                            (torch.float32, 4, 2, 64)])
def test_compute_qkv_reference_form(gpu, dtype, H, Hkv, Dh):
    """The reference's call form (src/decoding/fa4_attention.py:128-152):
    separate bias-free c_q / c_k / c_v nn.Linear projections and complex
    freqs_cis shaped (1, T, 1, Dh/2). q and k are the projections rotated as
    complex numbers (x[2j] + i x[2j+1]) * freqs[t, j], v the plain projection
    (numpy, float64); the fused-Wqkv form gives the same bits; use_rope =
    False returns the plain projections; a weight changed in place is seen."""
    g = torch.Generator().manual_seed(H + Hkv + Dh)
    B, T, C = 2, 7, 512

    class Attn(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.n_head, self.n_kv_head, self.head_dim = H, Hkv, Dh
            self.c_q = torch.nn.Linear(C, H * Dh, bias=False)
            self.c_k = torch.nn.Linear(C, Hkv * Dh, bias=False)
            self.c_v = torch.nn.Linear(C, Hkv * Dh, bias=False)

    attn = Attn()
    with torch.no_grad():
        for m in (attn.c_q, attn.c_k, attn.c_v):
            m.weight.copy_(0.05 * torch.randn(m.weight.shape, generator=g))
    attn = attn.to(device=gpu, dtype=dtype)
    x = torch.randn(B, T, C, generator=g).to(device=gpu, dtype=dtype)
    ang = torch.rand(T, Dh // 2, generator=g, dtype=torch.float64) * 6.0
    freqs = torch.polar(torch.ones_like(ang), ang).to(torch.complex64).view(1, T, 1, Dh // 2)

    def reference(x, attn):
        xs = _np(x).reshape(B * T, C)
        qs = xs @ _np(attn.c_q.weight).T
        ks = xs @ _np(attn.c_k.weight).T
        vs = xs @ _np(attn.c_v.weight).T
        f = freqs.view(T, Dh // 2).to(torch.complex128).numpy()

        def rot(a, heads):
            a = a.reshape(B, T, heads, Dh // 2, 2)
            z = (a[..., 0] + 1j * a[..., 1]) * f[None, :, None, :]
            return np.stack([z.real, z.imag], axis=-1).reshape(B, T, heads, Dh)

        return rot(qs, H), rot(ks, Hkv), vs.reshape(B, T, Hkv, Dh)

    q, k, v = A.compute_qkv(attn, x, freqs, None, None)
    rq, rk, rv = reference(x, attn)
    tol = TOL[dtype]
    assert rel_err(_np(q), rq) <= tol and rel_err(_np(k), rk) <= tol and rel_err(_np(v), rv) <= tol

    class Fused:
        n_head, n_kv_head, head_dim = H, Hkv, Dh
        Wqkv = torch.cat([attn.c_q.weight, attn.c_k.weight, attn.c_v.weight]).detach().contiguous()

    q2, k2, v2 = A.compute_qkv(Fused, x, freqs)
    assert torch.equal(q2, q) and torch.equal(k2, k) and torch.equal(v2, v)

    class NoRope:
        class rope_settings:
            use_rope = False
        clip_qkv = None
        qk_bias = False
        qk_norm = False

    q3, k3, v3 = A.compute_qkv(attn, x, freqs, None, NoRope)
    xs = _np(x).reshape(B * T, C)
    assert rel_err(_np(q3).reshape(B * T, -1), xs @ _np(attn.c_q.weight).T) <= tol
    assert rel_err(_np(k3).reshape(B * T, -1), xs @ _np(attn.c_k.weight).T) <= tol
    assert torch.equal(v3, v)

    with torch.no_grad():
        attn.c_k.weight.mul_(-1)  # in place: the packed copy must be rebuilt
    q4, k4, v4 = A.compute_qkv(attn, x, freqs)
    assert torch.equal(q4, q) and torch.equal(v4, v) and torch.equal(k4, -k)


def _capture(fn):
    """fn() as a graph, captured on torch's own capture stream after one call
    on the current one: (graph, the outputs it writes)."""
    fn()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    torch.cuda.synchronize()
    return graph, out if isinstance(out, tuple) else (out,)


@pytest.mark.parametrize("form", ["prompt", "whole", "short keys", "one row", "fp32 rows", "q1", "qkv"])
def test_captured_calls_replay_after_other_shapes(gpu, form):
    """Each entry point that uses index tables, captured after a warm-up on
    another stream, then replayed on new inputs after 300 other shapes have
    gone through the module (more than it keeps) and their memory has been
    reused: the eager call's bits every time."""
    H, Hkv, Dh, B = 4, 4, 64, 2
    Tq, Tk = {"prompt": (70, 90), "whole": (90, 70), "short keys": (90, 70), "one row": (1, 70),
              "fp32 rows": (5, 70)}.get(form, (1, 1))
    dt = torch.float32 if form == "fp32 rows" else torch.bfloat16
    g = torch.Generator().manual_seed(len(form))
    mk = lambda *s: torch.randn(*s, generator=g).to(dt).to(gpu)  # noqa: E731
    if form == "qkv":
        attn = type("Attn", (), dict(Wqkv=ops.pack_linear(0.05 * mk((H + 2 * Hkv) * Dh, 256)), n_head=H,
                                     n_kv_head=Hkv, head_dim=Dh))
        ang = torch.rand(33, Dh // 2, generator=g)
        freqs = torch.polar(torch.ones_like(ang), ang).to(gpu)
        ins = [mk(B, 33, 256)]
        fn = lambda: A.compute_qkv(attn, ins[0], freqs)  # noqa: E731
    elif form == "q1":
        cu = torch.tensor([0, 40, 41, 200], dtype=torch.int32, device=gpu)
        ins = [mk(3, H, Dh), mk(200, Hkv, Dh), mk(200, Hkv, Dh)]
        fn = lambda: A.attn_varlen_q1_padded(*ins, cu, 159)  # noqa: E731
    else:
        ins = [mk(B, Tq, H, Dh), mk(B, Tk, Hkv, Dh), mk(B, Tk, Hkv, Dh)]
        fn = lambda: A.attn_dense(*ins, causal=form != "whole")  # noqa: E731
    print(f"[captured {form}]", flush=True)
    graph, outs = _capture(fn)
    x = torch.zeros(1, 400, 256, dtype=torch.bfloat16, device=gpu)
    small = type("Small", (), dict(Wqkv=ops.pack_linear(torch.zeros(48, 256, dtype=torch.bfloat16, device=gpu)),
                                   n_head=1, n_kv_head=1, head_dim=16))
    ones = torch.ones(400, 8, dtype=torch.complex64, device=gpu)
    for T in range(1, 301):
        A.compute_qkv(small, x[:, :T], ones[:T])
    junk = [torch.full((2048,), 0x7f7f7f7f, dtype=torch.int32, device=gpu) for _ in range(600)]
    for _ in range(3):
        for t in ins:
            t.copy_(mk(*t.shape))
        graph.replay()
        torch.cuda.synchronize()
        want = fn()
        for a, b in zip(outs, want if isinstance(want, tuple) else (want,), strict=True):
            assert torch.equal(a, b)
    assert len(junk) == 600
