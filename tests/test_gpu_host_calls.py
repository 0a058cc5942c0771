"""The calls that take and fill host arrays, and the live turn view as acting
seats, against the device calls they stand for: batch sizes on both sides of the
staging limits, id rows longer than the first copy's share and than the row
width."""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from tests.test_gpu import _engineer_positions, _import_positions  # noqa: E402


@pytest.fixture(scope="module")
def jq():
    if not torch.cuda.is_available():
        pytest.fail("GPU test collected on a machine without a visible GPU")
    import junqi_amd
    return junqi_amd


def _dense(offs, vals, n, width):
    ids = np.full((n, width), -1, np.int32)
    for i in range(n):
        row = vals[offs[i]:offs[i + 1]][:width]
        ids[i, :len(row)] = row
    return ids


@pytest.mark.parametrize("n", [1, 67, 4096, 4097, 16385])
def test_host_ply_and_flags(jq, n):
    print(f"[host] n={n}", flush=True)
    a, b = (jq.JunqiBatch(n, show_mode=2, pool_size=64, max_num_moves=90) for _ in range(2))
    for x in (a, b):
        x.reset_terminated(5)
        x.legal()
        for k in range(85):
            x.env_step(sampler="uniform", sample_seed=1, ply=k, reset_seed=k)
    for k in range(6):   # past the cap: draws, then skipped games
        acts = a.sample_uniform(9, k).cpu().numpy()
        acts[::5] = 12345   # illegal
        want = a.step(torch.from_numpy(acts).cuda())
        got = b.step_numpy(acts)
        for key, v in got.items():
            assert v.dtype == want[key].cpu().numpy().dtype and np.array_equal(v, want[key].cpu().numpy()), (k, key)
        assert np.array_equal(b.copy_turn_to_host(), a.get_field("turn")[:, 0])
        t = b.termination()
        for key, f in (("terminated", "terminated"), ("winner_team", "winner"), ("draw", "draw")):
            assert np.array_equal(t[key], a.get_field(f)[:, 0].astype(t[key].dtype)), (k, key)
        seats = (np.arange(n) % 4).astype(np.int8)
        offs, vals = a.legal_csr_numpy(torch.from_numpy(seats))
        ids, counts = b.legal_dense_numpy(seats, 17)
        assert np.array_equal(counts, np.diff(offs)) and np.array_equal(ids, _dense(offs, vals, n, 17))
        a.legal()
        b.legal()
    a.close()
    b.close()


def test_host_rows_beyond_the_first_copy(jq):
    positions = _engineer_positions(33, 7)
    b = jq.JunqiBatch(len(positions), show_mode=2, pool_size=16)
    _import_positions(jq, b, positions)
    for seat in range(4):
        acting = np.full(b.n, seat, np.int8)
        offs, vals = b.legal_csr_numpy(torch.from_numpy(acting))
        # the share copied first is 64 ids a game; the richest games alone exceed it
        ids, counts = b.legal_dense_numpy(acting, 512)
        assert np.array_equal(counts, np.diff(offs)) and np.array_equal(ids, _dense(offs, vals, b.n, 512))
    rich = [p for _, p in sorted(zip(np.diff(offs), range(b.n)))][-4:]
    c = jq.JunqiBatch(4, show_mode=2, pool_size=16)
    _import_positions(jq, c, [positions[i] for i in rich])
    acting = np.full(4, 3, np.int8)
    offs, vals = c.legal_csr_numpy(torch.from_numpy(acting))
    assert offs[-1] > 64 * 4
    ids, counts = c.legal_dense_numpy(acting, 512)
    assert np.array_equal(counts, np.diff(offs)) and np.array_equal(ids, _dense(offs, vals, 4, 512))
    b.close()
    c.close()


def test_live_turn_view_is_the_copied_seats(jq):
    n = 130
    a, b = (jq.GpuRollout(n, show_mode=1, max_num_moves=60) for _ in range(2))
    for x in (a, b):
        x.reset(3)
        x.batch.legal()
    for k in range(70):
        out = []
        for x, seats in ((a, a.turn_torch()), (b, b.turn_torch().clone())):
            canon = torch.empty(n, dtype=torch.int32, device=x.device)
            world = x.batch.sample_logits(4, k, acting=seats, canonical_out=canon)
            sp, gl = x.build_acting_seat_observation_torch(seats)
            mask = x.legal_mask_canonical_torch_device(seats).clone()
            slots = x.batch.legal_slots(seats)
            step = {q: v.clone() for q, v in x.step_device_torch(canon, seats).items()}
            x.reset_terminated_device(seed=k)
            legal = {q: v.clone() for q, v in x.batch.legal(x.turn_torch() if x is a else x.turn_torch().clone()).items()}
            out.append([world, canon, sp, gl, mask, slots, *step.values(), legal["counts"], legal["offsets"],
                        legal["mask_words"]])
        for p, q in zip(*out):
            assert torch.equal(p, q), k
    a.close()
    b.close()
