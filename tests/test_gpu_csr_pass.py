"""The one-pass CSR (offsets and ids written together) against the two-kernel
route that buffers below the always-fits bound take, over batch sizes around
the pass's block and wave edges, with the count buffer at every 4-byte phase."""

from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def jq():
    if not torch.cuda.is_available():
        pytest.fail("GPU test collected on a machine without a visible GPU")
    import junqi_amd
    return junqi_amd


@pytest.mark.parametrize("n", [1, 7, 8, 9, 31, 65, 1000, 8192, 8193, 24576, 24577, 32768, 32769])
def test_one_pass_equals_scan_and_emit(jq, n):
    from junqi_amd import _lib as L
    print(f"[csr] n={n}", flush=True)
    b = jq.JunqiBatch(n, show_mode=2, pool_size=256)
    b.reset_terminated(n)
    b.legal()
    for k in range(60):
        b.env_step(sampler="uniform", sample_seed=n, ply=k, reset_seed=k)
    dev = b.device
    s = torch.cuda.current_stream().cuda_stream
    bound = n * L.MAX_LEGAL
    acting = torch.arange(n, device=dev).to(torch.int8) % 5 - 1   # seats 0-3 and seats without a move
    want_v = torch.full((bound,), -7, dtype=torch.int32, device=dev)
    want_c = torch.empty(n, dtype=torch.int32, device=dev)
    want_o = torch.empty(n + 1, dtype=torch.int32, device=dev)
    L.check(L.lib.jq_legal(b._h, acting.data_ptr(), want_c.data_ptr(), want_o.data_ptr(), want_v.data_ptr(),
                           bound - 1, None, None, s))
    for phase in range(4):
        got_v = torch.full((bound,), -7, dtype=torch.int32, device=dev)
        got_c = torch.full((n + 8,), -7, dtype=torch.int32, device=dev)
        got_o = torch.full((n + 9,), -7, dtype=torch.int32, device=dev)
        c, o = got_c[phase:phase + n], got_o[phase:phase + n + 1]
        L.check(L.lib.jq_legal(b._h, acting.data_ptr(), c.data_ptr(), o.data_ptr(), got_v.data_ptr(), bound, None,
                               None, s))
        assert torch.equal(c, want_c) and torch.equal(o, want_o) and torch.equal(got_v, want_v), phase
        assert (got_o[:phase] == -7).all() and (got_o[phase + n + 1:] == -7).all()
    b.close()
