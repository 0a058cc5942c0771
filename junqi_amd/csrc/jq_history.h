// Compact rollout history: every per-env state block of a handle, one copy per
// rollout step. Observations and legal masks of a batch of (step, env) rows are
// produced from these arrays in place (k_observe and k_legal with HIST;
// src/env/cuda/src/rollout_history.cu:160-525 keeps the same pre-action state
// per step and rebuilds PPO minibatches from it).
//
// Included into jq_lib.hip's translation unit.
#pragma once

namespace jq {

// Per-env bytes of one history row: board, piece records, all four observers'
// combat memory (records and eaten-by sets; the views and summary bytes are derived when
// a row is rebuilt) and belief codes, remaining counts, env record, move ring.
constexpr size_t HIST_ROW_BYTES = CELL_STRIDE + PID_STRIDE * sizeof(PieceRec) +
                                  4 * PID_STRIDE * (sizeof(CmRec) + sizeof(CmEat)) + 4 * PID_STRIDE + 4 * 48 +
                                  sizeof(EnvRec) + HIST_LEN * sizeof(int32_t);

// History arrays, row r = step * n + env, each laid out like the State array
// of the same name.
struct HistState {
    int32_t steps, n;
    int8_t *cell;
    PieceRec *piece;
    CmRec *cm;
    CmEat *cme;
    uint8_t *bcode;
    int8_t *rem;
    EnvRec *env;
    int32_t *hist;
};

// The history's rows as a state: row r is env r. It has no views, summary bytes
// or legal records, so only kernels built for it (HIST) take it.
inline State history_state(const HistState &H, const float *rlut, int32_t show_mode)
{
    State S{};
    S.n = H.steps * H.n;
    S.show_mode = show_mode;
    S.cell = H.cell; S.piece = H.piece; S.cm = H.cm; S.cme = H.cme; S.bcode = H.bcode; S.rem = H.rem;
    S.env = H.env; S.hist = H.hist;
    S.rlut = rlut;
    return S;
}

// Rows step * n .. step * n + n - 1 <- the state's envs, one 256-thread block
// per env. Bound: HBM copy, 2 x 35,972 bytes per env. All of a thread's loads
// (nine 16-byte words and one word of the 292-byte board, which keeps only
// 4-byte alignment) go out before its first store. One launch in place of a
// device copy per array: those took 4-5 us each however small (1,024 envs: 48 us
// for the eight, 96 envs: 40 us).
__global__ __launch_bounds__(256) void k_history_snapshot(State S, HistState H, int32_t step)
{
    constexpr int CM_Q = 4 * PID_STRIDE * (int)(sizeof(CmRec) / 16), CME_Q = 4 * PID_STRIDE;
    static_assert(CM_Q == 6 * 256 && CME_Q == 512 && PID_STRIDE == 128, "the block's passes below");
    const int i = blockIdx.x, t = threadIdx.x;
    if (i >= H.n) return;
    const size_t e = (size_t)i, r = (size_t)step * H.n + i;
    auto q16 = [](const void *p) { return const_cast<uint4 *>(static_cast<const uint4 *>(p)); };
    const uint4 *cs = q16(S.cm) + e * CM_Q + t, *es = q16(S.cme) + e * CME_Q;
    uint4 *cd = q16(H.cm) + r * CM_Q + t, *ed = q16(H.cme) + r * CME_Q;
    // the last pass: half the block on the eaten-by sets' end, the other half on
    // the small arrays (the threads past them repeat the move ring's last word)
    const uint4 *xs = q16(S.piece) + e * PID_STRIDE + t, *ys;
    uint4 *xd = q16(H.piece) + r * PID_STRIDE + t, *yd;
    if (t >= 128) { xs = es + (t - 128); xd = ed + (t - 128); }
    const int k = t - 128;
    if (k < 0) { ys = es + 384 + t; yd = ed + 384 + t; }
    else if (k < 32) { ys = q16(S.bcode) + e * 32 + k; yd = q16(H.bcode) + r * 32 + k; }
    else if (k < 44) { ys = q16(S.rem) + e * 12 + (k - 32); yd = q16(H.rem) + r * 12 + (k - 32); }
    else if (k < 46) { ys = q16(S.env) + e * 2 + (k - 44); yd = q16(H.env) + r * 2 + (k - 44); }
    else { const int j = min(k - 46, 7); ys = q16(S.hist) + e * 8 + j; yd = q16(H.hist) + r * 8 + j; }
    const uint32_t *bs = reinterpret_cast<const uint32_t *>(S.cell) + e * (CELL_STRIDE / 4) + min(t, CELL_STRIDE / 4 - 1);
    uint32_t *bd = reinterpret_cast<uint32_t *>(H.cell) + r * (CELL_STRIDE / 4) + min(t, CELL_STRIDE / 4 - 1);
    const uint4 c0 = cs[0], c1 = cs[256], c2 = cs[512], c3 = cs[768], c4 = cs[1024], c5 = cs[1280];
    const uint4 x = *xs, m = es[128 + t], y = *ys;
    const uint32_t w = *bs;
    cd[0] = c0; cd[256] = c1; cd[512] = c2; cd[768] = c3; cd[1024] = c4; cd[1280] = c5;
    *xd = x;
    ed[128 + t] = m;
    *yd = y;
    *bd = w;
}

}  // namespace jq
