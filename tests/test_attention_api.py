"""Host behaviour of the attention-backend API (CPU): backend selection and
argument errors that are raised before anything is launched."""
from __future__ import annotations

import pytest
import torch

from wavefront_decoding_amd import _lib
from wavefront_decoding_amd import attention as A


def test_backend_names():
    assert A.backend() == "hip"
    for name in ("torch", "fa4", "hip"):  # the reference's fused backends map to the HIP kernels
        A.set_backend(name)
        assert A.backend() == "hip"
    with pytest.raises(ValueError, match="parity reference"):
        A.set_backend("sdpa")
    with pytest.raises(ValueError, match="unknown"):
        A.set_backend("triton")
    assert A.backend() == "hip"


def test_reference_entry_points_exist():
    for name in ("attn_dense", "attn_cutoff_multi", "attn_varlen", "attn_varlen_q1_padded", "set_backend",
                 "backend", "compute_qkv"):
        assert callable(getattr(A, name)), name


def test_shape_errors_before_launch():
    q = torch.empty(1, 3, 4, 64, device="meta")
    with pytest.raises(_lib.WfdError):
        A.attn_dense(q, torch.empty(2, 5, 4, 64, device="meta"), torch.empty(2, 5, 4, 64, device="meta"), causal=True)
    with pytest.raises(AssertionError, match="max\\(qpos\\)\\+1"):
        A.attn_cutoff_multi(q, torch.empty(1, 9, 4, 64, device="meta"), torch.empty(1, 9, 4, 64, device="meta"),
                            [2, 3, 5])
    with pytest.raises(_lib.WfdError, match="not supported"):
        A.compute_qkv(object(), torch.empty(1, 2, 8, device="meta"), (None, None, 0), ve=torch.empty(1))


def test_host_tensors_are_refused():
    q, cu = torch.zeros(1, 3, 2, 64), torch.tensor([0, 1, 2, 3], dtype=torch.int32)
    for call in (lambda: A.attn_dense(q, q, q, causal=True), lambda: A.attn_dense(q[:, :1], q, q, causal=False),
                 lambda: A.attn_varlen_q1_padded(q[0], q[0], q[0], cu, 1)):
        with pytest.raises(_lib.WfdError, match="GPU tensors"):
            call()


def _table_calls(device):
    """Every index table the module keeps: (call, the tables it must return)."""
    t = lambda *v: torch.tensor(v, dtype=torch.int32)  # noqa: E731
    return {
        "rows": (lambda: A._dense_rows(2, 3, 2, True, device), (t(0, 0, 0, 2, 2, 2).long(), t(0, 1, 2, 0, 1, 2))),
        "rows, whole": (lambda: A._dense_rows(2, 1, 5, False, device), (t(0, 5).long(), t(5, 5))),
        "no keys": (lambda: A._dense_rows(2, 2, 0, True, device), (t(0, 0, 0, 0).long(), t(0, 0, 0, 0))),
        "prefill": (lambda: A._prefill_segments(3, 4, 7, device), (t(0, 7, 14).long(), t(0, 4, 8, 12), t(3, 3, 3))),
        "offsets": (lambda: A._dense_offsets(2, 4, 7, device), (t(0, 4, 8), t(0, 7, 14))),
        "tokens": (lambda: A._token_tables(2, 3, device), (t(0, 1, 2, 0, 1, 2), t(0, 1, 2, 3, 4, 5).long())),
    }


def test_tables_under_capture_belong_to_the_graph(monkeypatch):
    """A capturing stream neither reads nor leaves a kept table, whether or not
    the shape was seen before the capture: what a graph replays over lies in
    its own memory. (torch's calls that need a GPU are stood in for.)"""
    stream, capturing = [7], [False]
    monkeypatch.setattr(A, "_raw_stream", lambda device: stream[0])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    monkeypatch.setattr(A, "_TABLES", type(A._TABLES)())
    for name, (call, want) in _table_calls(torch.device("cpu")).items():
        kept = call()
        assert all(torch.equal(a, b) and a.dtype == b.dtype for a, b in zip(kept, want, strict=True)), name
        assert all(a is b for a, b in zip(call(), kept)), name
        before = set(A._TABLES)
        for s in (7, 8):  # the warmed-up stream, and the one torch.cuda.graph captures on
            stream[0], capturing[0] = s, True
            own = call()
            assert all(torch.equal(a, b) and a.data_ptr() != c.data_ptr() for a, b, c in zip(own, want, kept)), name
            assert set(A._TABLES) == before, name
        stream[0], capturing[0] = 7, False
