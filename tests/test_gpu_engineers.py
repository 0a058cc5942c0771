"""Engineers' legal sets against the oracle where their closures differ in kind:
an almost empty railway (one region), crowded ones (many small regions, sources
between several), no neighbour free, and more engineers than one group of three."""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from tests.test_gpu import _import_positions  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def jq():
    if not torch.cuda.is_available():
        pytest.fail("GPU test collected on a machine without a visible GPU")
    import junqi_amd
    return junqi_amd


def _positions(n, engineers, others, seed):
    """n positions with `engineers` engineers and `others` other pieces per seat on
    random rail cells (73 in all)."""
    rng = np.random.default_rng(seed)
    rail = np.flatnonzero(O.tables()["rail"])
    out = []
    for _ in range(n):
        cells = rng.permutation(rail)[:4 * (engineers + others)].reshape(4, -1)
        pieces = [(s * 30 + j, 13 if j < engineers else int(rng.integers(4, 13)), int(f) % 17, int(f) // 17)
                  for s in range(4) for j, f in enumerate(cells[s])]
        out.append(dict(pieces=pieces, turn=int(rng.integers(4)), mc=0, mslc=0, dead=[0] * 4, flag=[0] * 4))
    return out


@pytest.mark.parametrize("engineers,others", [(1, 0), (3, 0), (3, 5), (3, 11), (3, 15), (5, 9), (7, 1)])
def test_legal_sets_and_moves_equal_oracle(jq, engineers, others):
    print(f"[engineers] {engineers} engineers, {others} others per seat", flush=True)
    positions = _positions(160, engineers, others, 10 * engineers + others)
    b = jq.JunqiBatch(len(positions), show_mode=2, pool_size=64)
    _import_positions(jq, b, positions)
    games = [O.Game.from_pieces(p["pieces"], turn=p["turn"]) for p in positions]
    for seat in range(4):
        acting = torch.full((b.n,), seat, dtype=torch.int8, device=b.device)
        offs, vals = b.legal_csr_numpy(acting)
        for i, g in enumerate(games):
            assert np.array_equal(vals[offs[i]:offs[i + 1]], g.legal_ids(seat)), (i, seat)
    # one ply: engineer moves that only an engineer can make leave their mark
    offs, vals = b.legal_csr_numpy()
    rng = np.random.default_rng(1)
    acts = np.array([vals[rng.integers(offs[i], offs[i + 1])] if offs[i + 1] > offs[i] else -1 for i in range(b.n)],
                    np.int32)
    b.step(torch.from_numpy(acts).cuda())
    for i, g in enumerate(games):
        if acts[i] >= 0:
            g.step_id(int(acts[i]))
    from tests import gpu_compare as G
    G.compare_state(G.device_fields(b), G.oracle_fields(games), ctx=f"{engineers} engineers, {others} others")
    b.close()
