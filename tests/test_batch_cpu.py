"""What the Python layer hands to the library, without a GPU: a JunqiBatch whose
library calls are recorded instead of run."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from junqi_amd import _lib as jl  # noqa: E402
from junqi_amd import batch as jb  # noqa: E402


class _Recorder:
    """Stands for the library: every call succeeds and is kept with its arguments;
    `seats` are the int8 values behind a seat pointer at the time of the call."""

    def __init__(self, n, seat_arg):
        self.n, self.seat_arg, self.calls = n, seat_arg, []

    def __getattr__(self, name):
        def call(*args):
            ptr = args[self.seat_arg.get(name, 0)] if name in self.seat_arg else None
            seats = None if ptr is None else np.frombuffer(C.string_at(ptr, self.n), np.int8).copy()
            self.calls.append((name, seats))
            return 0
        return call


class _HostBatch(jb.JunqiBatch):
    stream = 0

    def __init__(self, n):
        self.n, self.device, self._h = n, torch.device("cpu"), None
        self.counts = torch.zeros(n, dtype=torch.int32)
        self.offsets = torch.zeros(n + 1, dtype=torch.int32)
        self.values = torch.zeros(n * jl.MAX_LEGAL, dtype=torch.int32)
        self.mask_words = torch.zeros((n, jl.MASK_WORDS), dtype=torch.int32)
        self._turn_view = torch.zeros(n, dtype=torch.int8)


@pytest.fixture
def recorded(monkeypatch):
    n = 6
    rec = _Recorder(n, {"jq_legal_dense_host": 1})
    monkeypatch.setattr(jb, "lib", rec)
    return _HostBatch(n), rec


@pytest.mark.parametrize("seats", [
    np.array([0, 1, 2, 3, 0, 1], np.int64), np.array([0, 1, 2, 3, 0, 1], np.int32),
    np.arange(12, dtype=np.int8)[::2] % 4, [3, 2, 1, 0, 3, 2],
], ids=["int64", "int32", "strided", "list"])
def test_dense_legal_seats_are_read_by_value(recorded, seats):
    b, rec = recorded
    b.legal_dense_numpy(seats, 8)
    (name, got), = rec.calls
    assert name == "jq_legal_dense_host" and np.array_equal(got, np.asarray(seats).astype(np.int8))


@pytest.mark.parametrize("shape", [(0,), (5,), (7,), (6, 1), (1, 6), ()])
def test_dense_legal_refuses_other_shapes(recorded, shape):
    b, rec = recorded
    with pytest.raises(ValueError, match="acting"):
        b.legal_dense_numpy(np.zeros(shape, np.int8), 8)
    assert not rec.calls


def test_a_closed_batch_hands_out_no_view():
    from junqi_amd.gpu_rollout import GpuRollout

    r = GpuRollout.__new__(GpuRollout)
    r._b = b = _HostBatch(6)
    live = r.turn_torch()
    assert b._seats(live) is None, "the live view stands for the current turn"
    r.close()
    for view in (r.turn_torch, r.terminated_torch, r.winner_team_torch, r.draw_torch):
        with pytest.raises(jl.ArgumentError):
            view()
    assert b._seats(live) is not None, "the view of a closed batch is not the current turn"
    with pytest.raises(jl.JunqiError):
        b.legal_slots(torch.zeros(6, dtype=torch.int8), out=torch.empty((6, 120, 80), dtype=torch.bool))


@pytest.mark.parametrize("call", ["step_device_torch", "build_acting_seat_observation_torch"])
def test_collector_calls_need_their_seats(recorded, monkeypatch, call):
    from junqi_amd.gpu_rollout import GpuRollout

    b, rec = recorded
    monkeypatch.setattr(jl, "lib", rec)
    r = GpuRollout.__new__(GpuRollout)
    r._b, r.device, r.num_envs = b, b.device, b.n
    r._step_out = {k: torch.zeros(b.n) for k in ("event", "terminated", "winner_team", "draw", "rewards")}
    r._sp1 = torch.zeros((b.n, 317, 17, 17))
    r._gl1 = torch.zeros((b.n, 28))
    seats = torch.zeros(b.n, dtype=torch.int8)
    args = (torch.zeros(b.n, dtype=torch.int32),) if call == "step_device_torch" else ()
    getattr(r, call)(*args, seats)
    assert len(rec.calls) == 1
    with pytest.raises((ValueError, AttributeError)):
        getattr(r, call)(*args, None)
    assert len(rec.calls) == 1


def test_short_device_seats_are_refused(recorded):
    """The kernels read n seats (4n for all-seat observations)."""
    b, rec = recorded
    n = b.n
    seat_calls = {
        "legal": lambda s: b.legal(s), "legal_slots": lambda s: b.legal_slots(s, out=torch.empty((n, 120, 80), dtype=torch.bool)),
        "sample_logits": lambda s: b.sample_logits(1, 2, acting=s), "observe": lambda s: b.observe(s, fmt="u8"),
    }
    for name, call in seat_calls.items():
        for ok in (torch.zeros(n, dtype=torch.int64), torch.zeros((n, 1), dtype=torch.int8), torch.zeros(n + 3, dtype=torch.int8)):
            call(ok)
        done = len(rec.calls)
        for short in (torch.zeros(0, dtype=torch.int8), torch.zeros(n - 1, dtype=torch.int8)):
            with pytest.raises(ValueError, match="seats"):
                call(short)
        assert len(rec.calls) == done, name
    b.observe(torch.zeros((n, 4), dtype=torch.int8), fmt="u8", all_seats=True)
    done = len(rec.calls)
    with pytest.raises(ValueError, match="seats"):
        b.observe(torch.zeros(n, dtype=torch.int8), fmt="u8", all_seats=True)
    assert len(rec.calls) == done
