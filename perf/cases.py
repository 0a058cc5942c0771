"""Performance cases of the batched Junqi environment on one GPU.

Every case is one pass of something a training or evaluation program does in a
loop, through the package's public entry points. All results are whole numbers,
table values or correctly rounded quotients, so two correct implementations
agree bit for bit.

Kinds of cases (`kind`):
  env_step   JunqiBatch.env_step: sample, ply, restart, legal CSR + packed mask
             and (unless fmt is "none") the acting seat's observation
  rollout    one step of a PPO collector over GpuRollout: sampled canonical
             actions, step, device reset, bool legal mask + CSR, f32 observation
  rebuild    rollout history: snapshot of every game, then one PPO minibatch of
             observations and masks rebuilt from the stored steps
  masks      legal-support storage: dense bool masks -> id lists, then a
             shuffled minibatch of id lists -> dense masks
  legal      legal sets of a seat per game on engineer-dense positions
  all_seats  observations of all four seats of every game
  host       the numpy-facing loop: acting seats and legal ids on the host,
             step from numpy actions, termination flags, device reset
"""

from __future__ import annotations

import numpy as np
import torch

import junqi_amd
from junqi_amd import masks

FLAT = 16641            # canonical action ids, 129 * 129
OBS_ELEMS = 317 * 289   # elements of one observation
GLOBALS = 28
STAGGER = 480           # games are at plies 0 .. STAGGER when a pass first sees them
ELEM_BYTES = {"u8": 1, "bf16": 2, "f32": 4}
DTYPE = {"u8": torch.uint8, "bf16": torch.bfloat16, "f32": torch.float32}
AUX_BYTES = 2320


def listed():
    return [
        # the rollout loop at the batch size the environment is built for
        {"name": "step_u8_32768", "kind": "env_step", "games": 32768, "fmt": "u8", "sampler": "logits", "show": 2},
        # half that batch with bf16 planes, fed to a bf16 network without decoding
        {"name": "step_bf16_16384", "kind": "env_step", "games": 16384, "fmt": "bf16", "sampler": "uniform", "show": 2},
        # search and data generation without a network: state and legal sets only
        {"name": "step_only_4096", "kind": "env_step", "games": 4096, "fmt": "none", "sampler": "uniform", "show": 2},
        # a debugging or evaluation batch: launches and latency
        {"name": "step_u8_64", "kind": "env_step", "games": 64, "fmt": "u8", "sampler": "uniform", "show": 0},
        # the PPO collector's step with float32 observations; an odd batch
        {"name": "rollout_4099", "kind": "rollout", "games": 4099, "show": 1},
        # an evaluation match of a few dozen games
        {"name": "rollout_24", "kind": "rollout", "games": 24, "show": 2},
        # PPO epoch: a bf16 minibatch out of an 8-step rollout of 1,024 games
        {"name": "rebuild_bf16_4096", "kind": "rebuild", "games": 1024, "steps": 8, "rows": 4096, "fmt": "bf16",
         "show": 1},
        # the last, ragged float32 minibatch of a small rollout
        {"name": "rebuild_f32_333", "kind": "rebuild", "games": 96, "steps": 5, "rows": 333, "fmt": "f32", "show": 2},
        # rollout buffer that keeps legal supports as id lists
        {"name": "masks_8192", "kind": "masks", "rows": 8192, "k_max": 256},
        # legal queries where engineers reach far along the rails
        {"name": "legal_8192", "kind": "legal", "games": 8192},
        # belief and value targets of every seat of a collector's batch
        {"name": "all_seats_f32_1000", "kind": "all_seats", "games": 1000, "fmt": "f32", "show": 1},
        # an agent driven from numpy
        {"name": "host_256", "kind": "host", "games": 256, "show": 2},
    ]


def _size(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]; odd ones as likely as even."""
    v = int(round(lo * (hi / lo) ** rng.random()))
    return max(lo, min(hi, v + rng.randrange(2)))


def draw(rng):
    kind = rng.choice(["env_step", "env_step", "rollout", "rebuild", "masks", "legal", "all_seats", "host"])
    show = rng.randrange(3)
    if kind == "env_step":
        fmt = rng.choice(["u8", "u8", "bf16", "f32", "none"])
        top = {"u8": 32000, "bf16": 16000, "f32": 8000, "none": 32000}[fmt]
        return {"kind": kind, "games": _size(rng, 16, top), "fmt": fmt, "sampler": rng.choice(["logits", "uniform"]),
                "show": show}
    if kind == "rollout":
        return {"kind": kind, "games": _size(rng, 16, 8000), "show": show}
    if kind == "rebuild":
        fmt = rng.choice(["bf16", "f32"])
        return {"kind": kind, "games": _size(rng, 16, 4096), "steps": rng.randrange(2, 13),
                "rows": _size(rng, 32, 12000 if fmt == "bf16" else 6000), "fmt": fmt, "show": show}
    if kind == "masks":
        return {"kind": kind, "rows": _size(rng, 16, 16000), "k_max": rng.choice([256, 333, 512])}
    if kind == "legal":
        return {"kind": kind, "games": _size(rng, 16, 16000)}
    if kind == "all_seats":
        fmt = rng.choice(["u8", "bf16", "f32"])
        return {"kind": kind, "games": _size(rng, 2, {"u8": 8000, "bf16": 4000, "f32": 2000}[fmt]), "fmt": fmt,
                "show": show}
    return {"kind": "host", "games": _size(rng, 8, 1024), "show": show}


# ------------------------------------------------------------------ inputs
def _play_into_mixed_stages(b, seed):
    """Play b's freshly reset games so that game i has taken up to STAGGER - S_i
    plies, S_i uniform: openings, middle games, endgames and restarted games."""
    n, dev = b.n, b.device
    start = torch.from_numpy(np.random.default_rng(seed).integers(0, STAGGER, n)).to(dev)
    idle = torch.full((n,), -1, dtype=torch.int32, device=dev)
    acts = torch.empty(n, dtype=torch.int32, device=dev)
    b.legal()
    for k in range(STAGGER):
        b.sample_logits(seed, k, out=acts)
        b.env_step(actions=torch.where(start > k, idle, acts), ply=k, reset_seed=seed + k)


def _batch(n, show, seed):
    """A batch of n games at mixed stages; the first games come from its setup pool."""
    b = junqi_amd.JunqiBatch(n, show_mode=show)
    b.reset_terminated(seed)   # a new batch holds finished games only
    _play_into_mixed_stages(b, seed)
    return b


def _rail_cells():
    """Flat cells of the 73 rail nodes: the outer ring of rows 0-4 of each seat's
    5 x 6 block and the nine-grid."""
    cells = []
    for seat in range(4):
        for slot in range(25):
            col, row = slot % 5, slot // 5
            if row in (0, 4) or col in (0, 4):
                x, y = ((10 - col, 11 + row), (5 - row, 10 - col), (6 + col, 5 - row), (11 + row, 6 + col))[seat]
                cells.append(y * 17 + x)
    cells += [(6 + 2 * gy) * 17 + 6 + 2 * gx for gx in range(3) for gy in range(3)]
    return np.array(sorted(cells), np.int16)


def _engineer_batch(n, seed):
    """n positions with three engineers and up to six other pieces per seat on
    random rail cells."""
    rng = np.random.default_rng(seed)
    rail = _rail_cells()
    order = rng.random((n, rail.size)).argsort(axis=1)[:, :36]
    cells = rail[order].reshape(n, 4, 9)
    ptype = np.full((n, 4, 32), -1, np.int8)
    pos = np.full((n, 4, 32), -1, np.int16)
    ptype[:, :, :3] = 13
    ptype[:, :, 3:9] = rng.integers(4, 13, (n, 4, 6))
    alive = np.arange(9) < rng.integers(3, 10, (n, 4, 1))
    pos[:, :, :9] = np.where(alive, cells, -1)
    ptype[:, :, :9] = np.where(alive, ptype[:, :, :9], -1)
    pos, ptype = pos[:, :, :30].reshape(n, 120), ptype[:, :, :30].reshape(n, 120)
    cell = np.full((n, 292), -1, np.int8)
    game, pid = np.nonzero(pos >= 0)
    cell[game, pos[game, pid]] = pid
    pad = lambda a: np.concatenate([a, np.full((n, 8), -1, a.dtype)], axis=1)  # noqa: E731
    b = junqi_amd.JunqiBatch(n, show_mode=2, pool_size=64)
    b.set_field("cell", cell)
    b.set_field("ptype", pad(ptype))
    b.set_field("pos", pad(pos))
    b.set_field("zero", pad(pos))
    b.set_termination(np.zeros(n, bool), np.full(n, -1, np.int8), np.zeros(n, bool), finalize=False)
    b.finalize_import()
    return b


def prepare(case, seed):
    kind = case["kind"]
    if kind == "env_step":
        n, fmt = case["games"], case["fmt"]
        b = _batch(n, case["show"], seed)
        dev = b.device
        s = {"kind": kind, "b": b, "ply": STAGGER, "seed": seed,
             "out": {"terminated": torch.empty(n, dtype=torch.uint8, device=dev),
                     "reward": torch.empty(n, dtype=torch.float32, device=dev),
                     "hash_out": torch.empty(n, dtype=torch.int64, device=dev),
                     "actions_out": torch.empty(n, dtype=torch.int32, device=dev)},
             "obs": {}, "sampler": case["sampler"], "fmt": "u8" if fmt == "none" else fmt}
        if fmt != "none":
            s["obs"] = {"spatial": torch.empty((n, 317, 17, 17), dtype=DTYPE[fmt], device=dev),
                        "glob": torch.empty((n, GLOBALS), dtype=torch.float32, device=dev)}
            if fmt == "u8":
                s["obs"]["aux"] = torch.empty((n, AUX_BYTES), dtype=torch.uint8, device=dev)
        return s
    if kind == "rollout":
        r = junqi_amd.GpuRollout(case["games"], show_mode=case["show"], max_num_moves=1200)
        r.reset(seed)
        b = r.batch
        _play_into_mixed_stages(b, seed)
        return {"kind": kind, "r": r, "ply": STAGGER, "seed": seed,
                "world": torch.empty(b.n, dtype=torch.int32, device=b.device),
                "canon": torch.empty(b.n, dtype=torch.int32, device=b.device)}
    if kind == "rebuild":
        n, steps, rows = case["games"], case["steps"], case["rows"]
        r = junqi_amd.GpuRollout(n, show_mode=case["show"], max_num_moves=1200)
        r.reset(seed)
        b = r.batch
        _play_into_mixed_stages(b, seed)
        hist = r.create_rollout_history(steps)
        turns = torch.empty((steps, n), dtype=torch.int8, device=b.device)
        for k in range(steps):
            turns[k] = r.turn_torch()
            hist.snapshot(r.state, turns[k], k)
            b.env_step(sampler="logits", sample_seed=seed, ply=STAGGER + k, reset_seed=seed + k)
        turns[steps - 1] = r.turn_torch()   # the pass stores the last step again, from the current state
        flat = torch.from_numpy(np.random.default_rng(seed).integers(0, steps * n, rows)).to(b.device)
        return {"kind": kind, "r": r, "hist": hist, "turn": turns[steps - 1], "step": steps - 1, "flat": flat,
                "seats": turns.reshape(-1)[flat].contiguous(), "dtype": DTYPE[case["fmt"]]}
    if kind == "masks":
        rows = case["rows"]
        b = _batch(rows, 2, seed)
        mask = b.legal(mask_words=False, mask_bool=True)["mask_bool"].clone()
        dev = mask.device
        b.close()
        idx = torch.from_numpy(np.random.default_rng(seed).permutation(rows)[:max(1, rows // 2)]).to(dev)
        return {"kind": kind, "mask": mask, "idx": idx,
                "ids": torch.empty((rows, case["k_max"]), dtype=torch.int32, device=dev),
                "counts": torch.empty(rows, dtype=torch.int32, device=dev)}
    if kind == "legal":
        b = _engineer_batch(case["games"], seed)
        acting = torch.from_numpy(np.random.default_rng(seed + 1).integers(0, 4, case["games"]).astype(np.int8))
        return {"kind": kind, "b": b, "acting": acting.to(b.device)}
    if kind == "all_seats":
        n, fmt = case["games"], case["fmt"]
        b = _batch(n, case["show"], seed)
        dev = b.device
        s = {"kind": kind, "b": b, "fmt": fmt,
             "out": {"out_spatial": torch.empty((n, 4, 317, 17, 17), dtype=DTYPE[fmt], device=dev),
                     "out_global": torch.empty((n, 4, GLOBALS), dtype=torch.float32, device=dev)}}
        if fmt == "u8":
            s["out"]["out_aux"] = torch.empty((n, 4, AUX_BYTES), dtype=torch.uint8, device=dev)
        return s
    r = junqi_amd.GpuRollout(case["games"], show_mode=case["show"], max_num_moves=1200)
    r.reset(seed)
    _play_into_mixed_stages(r.batch, seed)
    return {"kind": "host", "r": r, "rng": np.random.default_rng(seed), "ply": STAGGER, "seed": seed}


# ------------------------------------------------------------------ one pass
def run(state):
    s = state
    kind = s["kind"]
    if kind == "env_step":
        b, ply = s["b"], s["ply"]
        s["ply"] = ply + 1
        b.env_step(sampler=s["sampler"], sample_seed=s["seed"], ply=ply, reset_seed=s["seed"] + ply, obs_fmt=s["fmt"],
                   **s["obs"], **s["out"])
        return {**s["out"], **s["obs"], "counts": b.counts, "offsets": b.offsets, "values": b.values,
                "mask_words": b.mask_words}
    if kind == "rollout":
        r, ply = s["r"], s["ply"]
        s["ply"] = ply + 1
        turn = r.turn_torch()
        r.batch.sample_logits(s["seed"], ply, acting=turn, out=s["world"], canonical_out=s["canon"])
        step = r.step_device_torch(s["canon"], turn)
        r.update_beliefs_device(step, turn)
        r.reset_terminated_device(seed=s["seed"] + ply)
        legal = r.batch.legal(mask_words=False, mask_bool=True)
        spatial, glob = r.build_acting_seat_observation_torch(r.turn_torch())
        return {**step, "actions": s["canon"], "mask": legal["mask_bool"], "counts": legal["counts"],
                "spatial": spatial, "glob": glob}
    if kind == "rebuild":
        s["hist"].snapshot(s["r"].state, s["turn"], s["step"])
        spatial, glob, mask = s["hist"].reconstruct(s["flat"], s["seats"], dtype=s["dtype"])
        return {"spatial": spatial, "glob": glob, "mask": mask}
    if kind == "masks":
        masks.dense_mask_to_csr(s["mask"], s["ids"], s["counts"])
        dense = masks.csr_to_dense_selected(s["ids"], s["counts"], s["idx"], FLAT)
        return {"ids": s["ids"], "counts": s["counts"], "dense": dense}
    if kind == "legal":
        return s["b"].legal(s["acting"])
    if kind == "all_seats":
        out = s["b"].observe(fmt=s["fmt"], all_seats=True, **s["out"])
        return list(out)
    r, ply = s["r"], s["ply"]
    s["ply"] = ply + 1
    acting = r.state.copy_turn_to_host()
    ids, counts = r.legal_actions_dense(acting)
    pick = (s["rng"].random(r.num_envs) * counts).astype(np.int64)
    actions = ids[np.arange(r.num_envs), pick]
    step = r.step(actions)
    ended = r.read_termination()
    r.reset_terminated_device(seed=s["seed"] + ply)
    return {"ids": ids, "counts": counts, "actions": actions, "step": step, "ended": ended}


# ------------------------------------------------------------------ what a pass cannot do without
# Per game: the board (289 B), the 120 piece records (16 B), the env record (32 B)
# and the move ring (128 B) of a ply; the observer's view of a row (60 enemy
# pieces of 16 B, 30 own pieces of 16 B, 120 belief codes, 48 counts).
STATE_BYTES = 289 + 120 * 16 + 32 + 128
VIEW_BYTES = 60 * 16 + 30 * 16 + 120 + 48
MEAN_LEGAL = 42
CSR_BYTES = 8 + 4 * MEAN_LEGAL
MASK_WORD_BYTES = 521 * 4
HISTORY_ROW_BYTES = 35972


def _obs_bytes(fmt):
    return OBS_ELEMS * ELEM_BYTES[fmt] + GLOBALS * 4 + (AUX_BYTES if fmt == "u8" else 0)


def work(case):
    kind = case["kind"]
    if kind == "env_step":
        per = STATE_BYTES + 4 * MEAN_LEGAL + 17 + CSR_BYTES + MASK_WORD_BYTES
        if case["fmt"] != "none":
            per += VIEW_BYTES + _obs_bytes(case["fmt"])
        return {"bytes": per * case["games"], "flops": 0}
    if kind == "rollout":
        per = STATE_BYTES + VIEW_BYTES + 4 * MEAN_LEGAL + 16 + CSR_BYTES + FLAT + _obs_bytes("f32")
        return {"bytes": per * case["games"], "flops": 0}
    if kind == "rebuild":
        per_row = STATE_BYTES + VIEW_BYTES + FLAT + _obs_bytes(case["fmt"])
        return {"bytes": per_row * case["rows"] + 2 * HISTORY_ROW_BYTES * case["games"], "flops": 0}
    if kind == "masks":
        rows = case["rows"]
        batch = max(1, rows // 2)
        return {"bytes": rows * (FLAT + 4 * case["k_max"] + 4) + batch * (FLAT + 4 * MEAN_LEGAL + 12), "flops": 0}
    if kind == "legal":
        return {"bytes": case["games"] * (289 + 120 + 32 + CSR_BYTES + MASK_WORD_BYTES), "flops": 0}
    if kind == "all_seats":
        return {"bytes": case["games"] * (STATE_BYTES + 4 * (VIEW_BYTES + _obs_bytes(case["fmt"]))), "flops": 0}
    return {"bytes": case["games"] * (STATE_BYTES + 512 * 4 + 4 + 30), "flops": 0}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """The id lists and dense rows of a masks case in plain numpy; None for the
    kinds whose results are the game's rules (they hold no rounded sums)."""
    if case["kind"] != "masks":
        return None
    s = prepare(case, seed)
    mask, idx = s["mask"].cpu().numpy(), s["idx"].cpu().numpy()
    ids = np.zeros((case["rows"], case["k_max"]), np.int32)
    row, col = np.nonzero(mask)
    counts = mask.sum(axis=1).astype(np.int32)
    ids[row, np.arange(row.size) - (np.cumsum(counts) - counts)[row]] = col
    return {"ids": ids, "counts": counts, "dense": mask[idx]}
