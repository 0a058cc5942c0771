"""The move generator's records (struct jq::MoveTables) on the CPU: the runs a
piece gets from them by bit scans, over random occupancies, are those of walking
the board tables cell by cell."""

import numpy as np
import pytest

from junqi_amd import _lib as jl
from tests.test_lib_cpu import _product_tables, _struct

_REC = _struct([("adj", "<u8", (2,), 16), ("run", "<u8", (2, 2)), ("meta", "<u4", ()), ("adj2", "<u4", ()), ("pad", "<u4", (2,))])
_LANE = _struct([("pre", "<u8", (2,), 16), ("cells", "<i2", (3,)), ("track", "<i2", ()), ("pad", "<u4", (2,))])


def _word(w):
    return int(w[0]) | (int(w[1]) << 64)


@pytest.fixture(scope="module")
def tables():
    raw = np.zeros(289 * 2 * 64 + 64 * 32, np.uint8)
    assert jl.lib.jq_move_tables(raw.ctypes.data, raw.nbytes) == 0, jl.lib.jq_last_error()
    assert _REC.itemsize == 64 and _LANE.itemsize == 32
    rec = raw[:289 * 2 * 64].view(_REC).reshape(289, 2)
    return _product_tables(jl), rec, raw[289 * 2 * 64:].view(_LANE)


def test_lane_records(tables):
    t, _, lane = tables
    pre = 0
    for i in range(64):
        assert [int(v) for v in lane["cells"][i]] == [t["c2f"][i], t["c2f"][i + 64], t["c2f"][128]]
        assert _word(lane["pre"][i]) == pre
        if lane["track"][i] >= 0:
            pre |= 1 << int(t["f2c"][lane["track"][i]])
    assert lane["track"][63] == -1 and bin(pre).count("1") == int((t["craylen"].sum(1) > 0).sum())


def _walk(cells, occ, att):
    out = set()
    for f in cells:
        if f not in occ:
            out.add(f)
            continue
        if f in att:
            out.add(f)
        break
    return out


@pytest.mark.parametrize("density", [0.0, 0.15, 0.5, 1.0])
def test_runs_equal_the_walk(tables, density):
    t, rec, lane = tables
    rng = np.random.default_rng(int(density * 100))
    f2c, c2f = t["f2c"], t["c2f"]
    for _ in range(4):
        occ = {int(f) for f in c2f if rng.random() < density}
        att = {f for f in occ if rng.random() < 0.5 and not (int(t["cflags"][f]) & 4)}
        ob = sum(1 << int(f2c[f]) for f in occ)
        land = ~ob | sum(1 << int(f2c[f]) for f in att)
        tocc = sum(1 << i for i in range(64) if lane["track"][i] < 0 or int(lane["track"][i]) in occ)
        tea = sum(1 << i for i in range(64) if int(lane["track"][i]) in att)
        for f in map(int, c2f):
            r = int(t["railidx"][f])
            want = {int(v) for v in list(t["adj"][f]) + list(t["diag"][f]) if v >= 0 and (v not in occ or v in att)}
            for k in range(4 if r >= 0 else 0):
                want |= _walk([int(v) for v in t["rays"][r][k][:t["raylen"][r][k]]], occ, att)
            for d in range(2 if r >= 0 else 0):
                want |= _walk([int(v) for v in t["crays"][r][d][:t["craylen"][r][d]]], occ, att)
            got = 0
            for h in range(2):
                m = rec[f][h]
                meta = int(m["meta"])
                assert meta & 0xFF == f2c[f] and ((meta >> 8) & 0xFF) - 1 == r
                assert (meta >> 16) & 0xFF == int(t["cflags"][f]) & 0xFF
                got |= (_word(m["adj"]) | int(m["adj2"]) << 128) & land
                up, down = _word(m["run"][0]), _word(m["run"][1])
                b = up & ob
                got |= up & land & (b ^ (b - 1) if b else ~0)
                b = down & ob
                got |= down & land & (~0 << (b.bit_length() - 1) if b else ~0)
                s = (meta >> 24) - 1
                if s < 0:
                    continue
                if h == 0:
                    x = tocc >> (s + 1)
                    e = s + 1 + ((x & -x).bit_length() - 1)
                    lo, hi = s + 1, e + ((tea >> e) & 1)
                else:
                    e = (tocc & ((1 << s) - 1)).bit_length() - 1
                    lo, hi = (e + 1 - ((tea >> e) & 1) if e >= 0 else 0), s
                got |= _word(lane["pre"][hi]) ^ _word(lane["pre"][lo])
            assert {int(c2f[i]) for i in range(129) if (got >> i) & 1} == want, (density, f)


def test_off_board_records_are_empty(tables):
    t, rec, _ = tables
    off = t["f2c"] < 0
    assert off[0] and not rec[off].view(np.uint8).any()
