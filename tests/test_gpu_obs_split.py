"""Observations at the row counts where the kernel's work split changes: one to
sixteen blocks per row, ordinary and streaming stores, and row starts at every
16-byte phase. Every row of every game against the oracle, bit for bit (bf16 =
round to nearest even of the float32; u8 through the decode table)."""

from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from oracle import oracle as O  # noqa: E402
from tests.test_gpu import _bf16_rne  # noqa: E402


@pytest.fixture(scope="module")
def jq():
    if not torch.cuda.is_available():
        pytest.fail("GPU test collected on a machine without a visible GPU")
    import junqi_amd
    return junqi_amd


def _offset(n_elems, dt, shift, dev):
    """A contiguous tensor of n_elems whose first element sits `shift` elements
    past a 16-byte boundary, and guard elements around it."""
    es = torch.empty((), dtype=dt).element_size()
    base = torch.full((n_elems + 64 // es + shift,), 7, dtype=dt, device=dev)
    pad = 32 // es + shift
    return base, base[pad:pad + n_elems]


# 733 f32, 1,466 bf16 and 2,931 u8 rows are the first past the 256 MiB of ordinary stores
@pytest.mark.parametrize("n", [1, 3, 24, 63, 100, 257, 333, 513, 704, 733, 1466, 2931])
def test_split_rows_equal_the_oracle(jq, n):
    print(f"[split] n={n}", flush=True)
    steps, seed = 40, 11
    b = jq.JunqiBatch(n, show_mode=n % 3, pool_size=64)
    b.reset(seed)
    b.legal()
    ob = O.Batch(jq.generate_lineups(seed, n), show_mode=n % 3)
    O.rollout(ob, b.pool, sampler=0, seed=seed, ply0=0, reset_seed0=0, steps=steps, active_from=None)
    for k in range(steps):
        b.env_step(sampler="uniform", sample_seed=seed, ply=k, reset_seed=k)
    for fmt, dt in (("f32", torch.float32), ("bf16", torch.bfloat16), ("u8", torch.uint8)):
        per16 = 16 // torch.empty((), dtype=dt).element_size()
        base, flat = _offset(n * 317 * 289, dt, n % per16, b.device)
        sp = flat.view(n, 317, 17, 17)
        out = b.observe(fmt=fmt, out_spatial=sp)
        torch.cuda.synchronize()
        pad = base.numel() - n * 317 * 289
        lead = flat.storage_offset()
        assert (base[:lead] == 7).all() and (base[lead + flat.numel():] == 7).all() and pad > 0, "guards written"
        for lo in range(0, n, 512):
            hi = min(n, lo + 512)
            osp, ogl = O.batch_observe(ob, lo, hi)
            osp = osp.reshape(hi - lo, 317, 17, 17)
            got = out[0][lo:hi]
            if fmt == "f32":
                assert np.array_equal(got.cpu().numpy().view(np.uint32), osp.view(np.uint32)), (n, lo, fmt)
            elif fmt == "bf16":
                assert np.array_equal(got.view(torch.int16).cpu().numpy().view(np.uint16), _bf16_rne(osp)), (n, lo, fmt)
            else:
                dec = jq.decode_u8(got.cpu().numpy(), out[2][lo:hi].cpu().numpy())
                assert np.array_equal(dec.view(np.uint32), osp.view(np.uint32)), (n, lo, fmt)
            assert np.array_equal(out[1][lo:hi].cpu().numpy(), ogl.reshape(hi - lo, 28)), (n, lo, fmt, "globals")
        del base, flat, sp, out
    b.close()
