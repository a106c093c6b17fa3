"""Host behaviour of the attention-backend API (CPU): backend selection and
argument errors that are raised before anything is launched."""
from __future__ import annotations

import pytest
import torch

from wavefront_decoding_amd import _lib
from wavefront_decoding_amd import attention as A
from wavefront_decoding_amd import ops


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
        "one batch row": (lambda: A._dense_rows(1, 3, 5, True, device), (t(0, 0, 0).long(), t(3, 4, 5))),
        "one batch row, whole": (lambda: A._dense_rows(1, 2, 5, False, device), (t(0, 0).long(), t(5, 5))),
        "lone rows": (lambda: A._dense_rows(3, 1, 4, True, device), (t(0, 4, 8).long(), t(4, 4, 4))),
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
    monkeypatch.setattr(A, "_TABLES", A._TableCache())
    for name, (call, want) in _table_calls(torch.device("cpu")).items():
        kept = call()
        assert all(torch.equal(a, b) and a.dtype == b.dtype for a, b in zip(kept, want, strict=True)), name
        assert all(a.is_contiguous() for a in kept), name  # the kernels read them by their address
        assert all(a is b for a, b in zip(call(), kept)), name
        before = set(A._TABLES.held)
        for s in (7, 8):  # the warmed-up stream, and the one torch.cuda.graph captures on
            stream[0], capturing[0] = s, True
            own = call()
            assert all(torch.equal(a, b) and a.data_ptr() != c.data_ptr() for a, b, c in zip(own, want, kept)), name
            assert set(A._TABLES.held) == before, name
        stream[0], capturing[0] = 7, False


def test_tables_stay_with_their_stream_and_shape(monkeypatch):
    """A table is handed to the stream that built it only, and other shapes --
    of any entry point, on any stream -- push out the least recently used
    tables one by one, never one in use; few or huge ones, within the bytes."""
    stream = [7]
    monkeypatch.setattr(A, "_raw_stream", lambda device: stream[0])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(A, "_TABLES", A._TableCache())
    dev = torch.device("cpu")
    for name, (call, _) in _table_calls(dev).items():
        mine = call()
        stream[0] = 8
        assert not {t.data_ptr() for t in call()} & {t.data_ptr() for t in mine}, name
        stream[0] = 7
    for first, (call, _) in _table_calls(dev).items():
        A._TABLES = A._TableCache()
        kept = call()
        for T in range(1, 400):  # more shapes than are kept; this one is used all along
            stream[0] = 7 + T % 3
            A._token_tables(5, T + 10, dev)
            stream[0] = 7
            assert all(a is b for a, b in zip(call(), kept, strict=True)), (first, T)
        held = A._TABLES.held
        assert len(held) == A._TABLES.max_tables
        assert A._TABLES.bytes == sum(t.nbytes for ts, _ in held.values() for t in ts)
    A._TABLES = A._TableCache(max_bytes=5000)
    for T in (100, 300, 10, 20, 2000, 30):
        assert A._token_tables(1, T, dev)[1].numel() == T
        assert A._TABLES.bytes <= 5000 or len(A._TABLES.held) == 1
    assert [k[-1] for k in A._TABLES.held] == [30]


def test_tables_of_two_threads_on_one_stream(monkeypatch):
    """Two threads that miss together each get whole tables; one pair is kept
    and its bytes are counted once."""
    import threading

    monkeypatch.setattr(A, "_raw_stream", lambda device: 7)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(A, "_TABLES", A._TableCache())
    gate, got = threading.Barrier(2), []

    def build():
        gate.wait(timeout=30)
        return (torch.arange(4),)

    def call():
        got.append(A._cached(torch.device("cpu"), ("x", 1), build))

    ts = [threading.Thread(target=call) for _ in range(2)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(timeout=30)
    assert len(got) == 2 and all(torch.equal(g[0], torch.arange(4)) for g in got)
    assert len(A._TABLES.held) == 1 and A._TABLES.bytes == 32


def test_split_workspace_belongs_to_its_stream(monkeypatch):
    """The workspace attn_decode takes when none is passed: one per stream and
    thread, replaced only when a launch needs more; a capturing stream's is its own."""
    import threading

    stream, capturing = [7], [False]
    monkeypatch.setattr(ops, "_raw_stream", lambda device: stream[0])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: capturing[0])
    monkeypatch.setattr(ops, "_WS", type(ops._WS)())
    ws = lambda n: ops.attn_workspace(n, 16, 128, 4096, "cpu")  # noqa: E731
    a = ws(8)
    assert a.numel() >= ops.attn_workspace_bytes(8, 16, 128, 4096) and ws(4) is a
    other = []
    t = threading.Thread(target=lambda: other.append(ws(8)))
    t.start()
    t.join(30)
    assert other[0] is not a and ws(8) is a
    stream[0] = 8
    b = ws(8)
    assert b is not a and ws(8) is b
    capturing[0] = True
    own = ws(8)
    assert own is not b and own.numel() >= ops.attn_workspace_bytes(8, 16, 128, 4096) and ws(8) is not own
    capturing[0] = False
    assert ws(16).numel() >= ops.attn_workspace_bytes(16, 16, 128, 4096)
    for s in range(100):
        stream[0] = s
        ws(1)
    assert len(ops._WS) == ops._MAX_WORKSPACES
