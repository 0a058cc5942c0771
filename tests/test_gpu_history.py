"""Compact rollout history (GpuRolloutHistory over jq_history_*) on an MI355X.

Games are played with a snapshot of the pre-action state at every step, as the
reference collector does (junqi_rl/training/gpu_collector.py:872); rows chosen
beforehand are then rebuilt from the history and compared bit-exactly with the
oracle's observation, globals and canonical legal mask at that step, for the
acting seat and for other seats (junqi_rl/gpu_rollout.py:164-217).
"""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from oracle import oracle as O  # noqa: E402
from tests import gpu_compare as G  # noqa: E402
from tests.test_gpu import _bf16_rne  # noqa: E402
from tests.test_gpu_api import _canonical_ids  # noqa: E402

ROW_BYTES = 35972


@pytest.fixture(scope="module")
def jq():
    if not torch.cuda.is_available():
        pytest.fail("GPU test collected on a machine without a visible GPU")
    import junqi_amd
    return junqi_amd


def test_history_reconstructs_observations_and_masks(jq):
    n, steps, show = 20, 16, 2
    print(f"[history] n={n} steps={steps} show={show}", flush=True)
    ro = jq.GpuRollout(n, show_mode=show, max_num_moves=400)
    ro.reset(31)
    games = G.oracle_games_from_lineups(jq.generate_lineups(31, n), show, 400)
    hist = ro.create_rollout_history(steps)
    assert hist.history_bytes == steps * n * ROW_BYTES
    rng = np.random.default_rng(4)
    # rows to rebuild: (step, env, seat offset from the acting seat)
    picks = [(int(t), int(i), int(k)) for t, i, k in zip(rng.integers(steps, size=40), rng.integers(n, size=40),
                                                         rng.integers(4, size=40))]
    want = {}
    seats = {}
    for t in range(steps):
        acting = ro.turn_torch().clone()
        hist.snapshot(ro.state, acting, t)
        for (pt, i, k) in picks:
            if pt == t:
                seat = (int(games[i].turn) + k) & 3
                sp, gl = games[i].observe(seat)
                want[(pt, i, k)] = (sp, gl, _canonical_ids(games[i].legal_ids(seat), seat))
                seats[(pt, i, k)] = seat
        acts = np.full(n, -1, np.int32)
        for i, g in enumerate(games):
            ids = g.legal_ids()
            if len(ids) and not g.terminated:
                acts[i] = ids[rng.integers(len(ids))]
        out = ro.step(acts)
        for i, g in enumerate(games):
            if acts[i] >= 0:
                rc, o = g.step_id(int(acts[i]))
                assert rc == 0 and bool(out["valid"][i])
    flat = torch.tensor([t * n + i for (t, i, k) in picks], dtype=torch.int64, device=ro.device)
    obs = torch.tensor([seats[p] for p in picks], dtype=torch.int8, device=ro.device)
    sp, gl, mask = hist.reconstruct(flat, obs, dtype=torch.float32)
    assert sp.shape == (len(picks), 317, 17, 17) and gl.shape == (len(picks), 28) and mask.dtype == torch.bool
    sp, gl, mask = sp.cpu().numpy(), gl.cpu().numpy(), mask.cpu().numpy()
    for b, p in enumerate(picks):
        wsp, wgl, wids = want[p]
        assert np.array_equal(sp[b].view(np.uint32), wsp.view(np.uint32)), (p, "obs")
        assert np.array_equal(gl[b], wgl), (p, "globals")
        wm = np.zeros(16641, bool)
        wm[wids] = True
        assert np.array_equal(mask[b], wm), (p, "mask")
    # bf16 storage dtype: round-to-nearest-even of the f32 observation
    sb, gb, mb = hist.reconstruct(flat, obs, dtype=torch.bfloat16)
    assert sb.dtype == torch.bfloat16 and gb.dtype == torch.bfloat16
    for b, p in enumerate(picks):
        assert np.array_equal(sb[b].view(torch.int16).cpu().numpy().view(np.uint16), _bf16_rne(want[p][0])), p
    assert np.array_equal(mb.cpu().numpy(), mask)
    # a smaller batch after a larger one
    s2, g2, m2 = hist.reconstruct(flat[:3].flip(0), obs[:3].flip(0), dtype=torch.float32)
    for b, p in enumerate(reversed(picks[:3])):
        assert np.array_equal(s2[b].cpu().numpy().view(np.uint32), want[p][0].view(np.uint32)), p
    # rows outside the history rebuild the empty terminated state: no legal action
    bad = torch.tensor([-1, steps * n], dtype=torch.int64, device=ro.device)
    _, _, mbad = hist.reconstruct(bad, torch.zeros(2, dtype=torch.int8, device=ro.device), dtype=torch.float32)
    assert not mbad.any()
    with pytest.raises(ValueError):
        hist.reconstruct(flat[:0], obs[:0], dtype=torch.float32)
    with pytest.raises(ValueError):
        hist.reconstruct(flat, obs[:2], dtype=torch.float32)
    with pytest.raises(IndexError):
        hist.snapshot(ro.state, ro.turn_torch().clone(), steps)
    hist.close()
    ro.close()


def test_history_rejects_a_mismatched_state(jq):
    ro = jq.GpuRollout(8, show_mode=2)
    ro.reset(1)
    hist = jq.GpuRolloutHistory(num_steps=2, num_envs=9, show_mode=2)
    with pytest.raises(jq.JunqiError):
        hist.snapshot(ro.state, torch.zeros(9, dtype=torch.int8, device=ro.device), 0)
    other = jq.GpuRolloutHistory(num_steps=2, num_envs=8, show_mode=0)
    with pytest.raises(jq.JunqiError):
        other.snapshot(ro.state, ro.turn_torch().clone(), 0)
    hist.close()
    other.close()
    ro.close()


@pytest.mark.parametrize("n,show", [(1, 0), (67, 1), (256, 2)])
def test_history_rows_equal_the_live_state(jq, n, show):
    """Rows rebuilt in place equal the live games' own observations and masks
    (which read the derived views, not the records) for every seat and format,
    after enough play for combat memory, deaths and restarts; rows outside the
    history equal an empty batch's."""
    from junqi_amd import _lib as L
    print(f"[history] live n={n} show={show}", flush=True)
    b = jq.JunqiBatch(n, show_mode=show, max_num_moves=500)
    b.reset(9)
    b.legal()
    for k in range(420):
        b.env_step(sampler="logits", sample_seed=3, ply=k, reset_seed=k)
    dev, steps = b.device, 3
    hist = jq.GpuRolloutHistory(num_steps=steps, num_envs=n, show_mode=show)
    for t in (2, 0, 1):   # the last snapshot is the live state
        hist.snapshot(b, torch.zeros(n, dtype=torch.int8, device=dev), t)
        if t != 1:
            b.env_step(sampler="logits", sample_seed=3, ply=1000 + t, reset_seed=t)
    empty = jq.JunqiBatch(1, show_mode=show)
    for fmt, dt in (("f32", torch.float32), ("bf16", torch.bfloat16), ("u8", torch.uint8)):
        code = {"f32": L.OBS_F32, "bf16": L.OBS_BF16, "u8": L.OBS_U8}[fmt]
        for seat in range(4):
            seats = torch.full((n,), seat, dtype=torch.int8, device=dev)
            live = b.observe(seats, fmt=fmt)
            legal = b.legal(seats, mask_bool=True)
            none = empty.observe(seats[:1], fmt=fmt)
            flat = torch.cat([torch.arange(n, device=dev) + n, torch.tensor([-1, steps * n, 1 << 40], device=dev)])
            rows, obs = n + 3, torch.full((n + 3,), seat, dtype=torch.int8, device=dev)
            sp = torch.empty((rows, 317, 17, 17), dtype=dt, device=dev)
            gl = torch.empty((rows, 28), dtype=torch.float32, device=dev)
            aux = torch.empty((rows, L.AUX_BYTES), dtype=torch.uint8, device=dev) if fmt == "u8" else None
            words = torch.empty((rows, 521), dtype=torch.int32, device=dev)
            mask = torch.empty((rows, 16641), dtype=torch.bool, device=dev)
            L.check(L.lib.jq_history_reconstruct(hist._h, flat.data_ptr(), obs.data_ptr(), rows, code, sp.data_ptr(),
                                                 None if aux is None else aux.data_ptr(), gl.data_ptr(),
                                                 words.data_ptr(), mask.data_ptr(),
                                                 torch.cuda.current_stream().cuda_stream))
            got = [sp, gl] + ([aux] if fmt == "u8" else [])
            for g, w, e in zip(got, live, none):
                assert torch.equal(g[:n], w) and torch.equal(g[n:], e.expand_as(g[n:])), (fmt, seat)
            assert torch.equal(words[:n], legal["mask_words"]) and torch.equal(mask[:n], legal["mask_bool"])
            assert not words[n:].any() and not mask[n:].any()
    hist.close()
    b.close()
    empty.close()
