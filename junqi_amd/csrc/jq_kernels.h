// HIP kernels for the batched Junqi environment (gfx950, wave64); included by jq_lib.hip.
//
// Execution model: one wavefront owns one env. Its cell map and piece rows are
// staged in LDS; rules logic that is serial by nature (one ply) runs uniformly on
// all 64 lanes, and the wide parts are spread over lanes: the 30 pieces of a seat
// for move generation, the 73 rail nodes for the engineer's reachability closure
// (two 64-bit ballots per hop), the 120 pids for purges and Zobrist folds, and the
// four observers for combat memory and beliefs.
//
// Reference semantics: junqi_core/state.py::GameState.step_inplace (638-998),
// move_gen.py (SoA generator 1052-1199, legacy predicates 127-376),
// combat_memory.py (339-569), info_model.py (218-429).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "junqi_amd.h"
#include "jq_device.h"
#include "jq_topology.h"

namespace jq {

__constant__ Tables cT;
__constant__ MoveTables cM;
constexpr int JQ_MASK_WORDS_PAD = 528;
constexpr int LSCR_WORDS = 12;   // legal_body's per-wave LDS scratch (u64 words)

// ------------------------------------------------------------------ helpers
__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

__device__ __forceinline__ uint32_t nib_to_bytes(uint32_t nib)
{   // 4 bits -> 4 bytes of 0/1: the shifted copies land on disjoint bit positions
    return __umul24(nib & 0xFu, 0x00204081u) & 0x01010101u;
}

// Entry i of a byte or halfword table in cT, read through the aligned 32-bit
// word that holds it. At a wave-uniform index this is a scalar load (there are
// none for bytes or halfwords), which neither waits for nor is waited for by
// the wave's vector stores; at a per-lane index it is an ordinary vector load.
template <typename T>
__device__ __forceinline__ T tab(const T *table, int i)
{
    static_assert(sizeof(T) <= 2, "byte and halfword tables only");
    typedef const __attribute__((address_space(4))) uint32_t *const_word;   // constant memory
    const uintptr_t a = reinterpret_cast<uintptr_t>(table + i);
    const uint32_t w = *reinterpret_cast<const_word>(a & ~uintptr_t(3));
    return (T)(w >> (8 * (a & 3)));
}

__device__ __forceinline__ uint16_t cflags(int f) { return tab(cT.cflags, f); }

// A 32-bit word of global memory at a wave-uniform address, read as a scalar
// load. Only for a word no wave writes before this read in the same kernel
// (an env's CSR count and offset are rewritten only by that env's own wave,
// after it has read them): the scalar cache is not coherent with vector stores.
// Loads through the constant address space count as invariant to the compiler,
// which may then re-issue one at a later use instead of keeping its register;
// after the wave's own store to the word that would read the new value. The
// empty asm takes the loaded word as its output, which the compiler can only
// keep (or spill), never recompute: every later use sees the value read here.
__device__ __forceinline__ int32_t uniform_word_raw(const int32_t *p)
{
    typedef const __attribute__((address_space(4))) int32_t *const_i32;
    return *reinterpret_cast<const_i32>(reinterpret_cast<uintptr_t>(p));
}
__device__ __forceinline__ void pin_word(int32_t &v) { asm volatile("" : "+s"(v)); }
__device__ __forceinline__ int32_t uniform_word(const int32_t *p)
{
    int32_t v = uniform_word_raw(p);
    pin_word(v);
    return v;
}

// An env's 32-byte record as one scalar load: only the env's own wave writes it,
// after reading it (at the end of its ply or restart); every field keeps the
// value read here (uniform_word).
__device__ __forceinline__ EnvRec env_record(const State &S, int env)
{
    const int32_t *w = reinterpret_cast<const int32_t *>(S.env + env);
    int32_t v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = uniform_word_raw(w + k);
#pragma unroll
    for (int k = 0; k < 8; ++k) pin_word(v[k]);
    EnvRec E;
    __builtin_memcpy(&E, v, sizeof E);
    return E;
}
__device__ __forceinline__ bool is_rail(int f) { return cflags(f) & CF_RAIL; }
__device__ __forceinline__ bool is_camp(int f) { return cflags(f) & CF_CAMP; }
__device__ __forceinline__ bool is_sh(int f) { return cflags(f) & CF_SH; }
__device__ __forceinline__ int team_of(int pid) { return (pid / 30) & 1; }

// Bits [base, base + 30) of the 120-bit pid set (hi:lo), i.e. the 30 pids of one seat.
__device__ __forceinline__ uint32_t seat_bits(uint64_t lo, uint64_t hi, int base)
{
    const uint64_t w = base == 0 ? lo : base < 64 ? ((lo >> base) | (hi << (64 - base))) : (hi >> (base - 64));
    return (uint32_t)w & 0x3FFFFFFFu;
}

__device__ __forceinline__ bool enemy_att(const int8_t *cell, int f, int team)
{   // enemy piece on a non-camp cell (move_gen.py:822-867)
    const int p = cell[f];
    return p >= 0 && team_of(p) != team && !is_camp(f);
}
__device__ __forceinline__ bool landable(const int8_t *cell, int f, int team)
{
    return cell[f] < 0 || enemy_att(cell, f, team);
}

__device__ __forceinline__ void setbit3(uint64_t &m0, uint64_t &m1, uint64_t &m2, int c)
{
    const uint64_t b = 1ull << (c & 63);
    const int w = c >> 6;
    m0 |= (w == 0) ? b : 0ull;
    m1 |= (w == 1) ? b : 0ull;
    m2 |= (w == 2) ? b : 0ull;
}

// Whole-wave reductions (every lane active), from the ROCm device library's
// wavefront reductions (DPP / lane permutes instead of six LDS shuffles).
extern "C" __device__ __attribute__((const)) unsigned long long __ockl_wfred_or_u64(unsigned long long);
extern "C" __device__ __attribute__((const)) unsigned long long __ockl_wfred_xor_u64(unsigned long long);
extern "C" __device__ __attribute__((const)) unsigned long long __ockl_wfred_max_u64(unsigned long long);
extern "C" __device__ __attribute__((const)) int __ockl_wfred_add_i32(int);
__device__ __forceinline__ uint64_t wave_or(uint64_t v) { return __ockl_wfred_or_u64(v); }
__device__ __forceinline__ uint64_t wave_xor(uint64_t v) { return __ockl_wfred_xor_u64(v); }
__device__ __forceinline__ uint64_t wave_max(uint64_t v) { return __ockl_wfred_max_u64(v); }
__device__ __forceinline__ int wave_sum(int v) { return __ockl_wfred_add_i32(v); }

// Reachability closure of an engineer standing on rail index `src_r`: the source
// plus every rail node joined to it through empty rail cells. Lane l evaluates
// nodes l and l+64 each hop; the frontier grows until a hop adds nothing, or
// until it touches a node of the target set (t0, t1) when one is given. A node
// already in the closure may be reported again by its lane: growth is what the
// ballot adds beyond the closure.
__device__ void rail_closure(const int8_t *cell, int src_r, uint64_t &r0, uint64_t &r1, uint64_t t0 = 0,
                             uint64_t t1 = 0)
{
    const int l = lane_id();
    const int v1 = l + 64;
    const bool e0 = cell[cT.railcell[l]] < 0;
    const bool e1 = v1 < NRAIL && cell[cT.railcell[v1 < NRAIL ? v1 : 0]] < 0;
    const uint64_t a0 = cT.rnbr[l][0], a1 = cT.rnbr[l][1];
    const uint64_t b0 = v1 < NRAIL ? cT.rnbr[v1][0] : 0ull, b1 = v1 < NRAIL ? cT.rnbr[v1][1] : 0ull;
    r0 = src_r < 64 ? (1ull << src_r) : 0ull;
    r1 = src_r >= 64 ? (1ull << (src_r - 64)) : 0ull;
    for (int hop = 0; hop < NRAIL; ++hop) {
        if ((r0 & t0) | (r1 & t1)) break;
        const uint64_t g0 = __ballot(e0 && ((a0 & r0) | (a1 & r1)) != 0);
        const uint64_t g1 = __ballot(e1 && ((b0 & r0) | (b1 & r1)) != 0) & 0x1FFull;
        if (!((g0 & ~r0) | (g1 & ~r1))) break;
        r0 |= g0;
        r1 |= g1;
    }
}

// Engineer destinations (move_gen.py:870-895) as a compact-index mask (uniform).
__device__ void engineer_mask(const int8_t *cell, int src, int team, uint64_t &m0, uint64_t &m1, uint64_t &m2)
{
    const int l = lane_id();
    const int sr = cT.railidx[src];
    uint64_t r0, r1;
    rail_closure(cell, sr, r0, r1);
    uint64_t p0 = 0, p1 = 0, p2 = 0;
    for (int v = l; v < NRAIL; v += 64) {
        const bool adj = ((cT.rnbr[v][0] & r0) | (cT.rnbr[v][1] & r1)) != 0;
        const int f = cT.railcell[v];
        if (v != sr && adj && landable(cell, f, team)) setbit3(p0, p1, p2, cT.f2c[f]);
    }
    m0 = wave_or(p0); m1 = wave_or(p1); m2 = wave_or(p2);
}

// ------------------------------------------------------------------ bitboards
// 129-bit sets over compact cells (bit c = compact cell c), three words.
struct BB {
    uint64_t w0, w1, w2;
};
__device__ __forceinline__ bool bb_has(const BB &b, int c)
{
    const uint64_t w = c < 64 ? b.w0 : c < 128 ? b.w1 : b.w2;
    return (w >> (c & 63)) & 1ull;
}

// The board of an env as uniform sets: occupied cells, cells holding an enemy of
// `team` that may be attacked (not in a camp), and the same of the track slots
// (MoveTables; slots without a cell count as occupied, so every curve run ends
// inside its own path). `cell` is the board (flat, LDS), T lane l's cells.
struct Boards {
    BB occ, ea;
    uint64_t tocc, tea;
};
__device__ __forceinline__ void env_boards(const int8_t *cell, int team, const LaneRec &T, Boards &B)
{
    const int l = lane_id();
    const int p0 = cell[T.c0], p1 = cell[T.c1], p2 = l == 0 ? cell[T.c2] : -1;
    const int pt = T.track >= 0 ? cell[T.track] : -1;
    B.occ = {__ballot(p0 >= 0), __ballot(p1 >= 0), __ballot(p2 >= 0)};
    const BB en = {__ballot(p0 >= 0 && team_of(p0) != team), __ballot(p1 >= 0 && team_of(p1) != team),
                   __ballot(p2 >= 0 && team_of(p2) != team)};
    B.ea = {en.w0 & ~cT.campm[0], en.w1 & ~cT.campm[1], en.w2 & ~cT.campm[2]};
    B.tocc = __ballot(T.track < 0 || pt >= 0);
    B.tea = __ballot(pt >= 0 && team_of(pt) != team);   // no rail cell is a camp
}

// Track slots [a, b) that the piece on track slot s reaches along its curve
// rail: up the path (half 0) or down it (half 1), to the first occupied slot,
// that one included if attackable.
__device__ __forceinline__ void track_run(int s, int h, const Boards &B, int &a, int &b)
{
    const uint64_t up = B.tocc >> (s + 1), down = B.tocc & ((1ull << s) - 1);
    const int eu = s + 1 + __builtin_ctzll(up | (1ull << 63)), ed = down ? 63 - __builtin_clzll(down) : -1;
    const int e = h ? ed : eu, hit = e >= 0 ? (int)((B.tea >> (e & 63)) & 1) : 0;
    a = h ? e + 1 - hit : s + 1;
    b = h ? s : e + hit;
}

// The moves of a piece's half (MoveRec M, non-engineers' rail runs included),
// the curve run excepted: road steps and straight runs to the first occupied
// cell, that one included if attackable (move_gen.py:1052-1199 parts a, b, c).
// blk ^ (blk - 1) is the lowest occupied cell and all below it.
__device__ __forceinline__ BB straight_moves_half(const MoveRec &M, bool engineer, const Boards &B)
{
    const uint64_t n0 = ~B.occ.w0 | B.ea.w0, n1 = ~B.occ.w1 | B.ea.w1;   // empty or attackable
    BB m = {M.adj[0] & n0, M.adj[1] & n1, (uint64_t)M.adj2 & (~B.occ.w2 | B.ea.w2)};
    if (engineer) return m;   // off the rails both runs are empty
    {
        const uint64_t b0 = M.run[0][0] & B.occ.w0, b1 = M.run[0][1] & B.occ.w1;
        const uint64_t v0 = b0 ^ (b0 - 1), v1 = b0 ? 0ull : b1 ^ (b1 - 1);
        m.w0 |= M.run[0][0] & n0 & v0;
        m.w1 |= M.run[0][1] & n1 & v1;
    }
    {   // the highest occupied cell and all above it
        const uint64_t b0 = M.run[1][0] & B.occ.w0, b1 = M.run[1][1] & B.occ.w1;
        const uint64_t v1 = ~0ull << (63 - __builtin_clzll(b1 | 1)), v0 = b1 ? 0ull : ~0ull << (63 - __builtin_clzll(b0 | 1));
        m.w0 |= M.run[1][0] & n0 & v0;
        m.w1 |= M.run[1][1] & n1 & v1;
    }
    return m;
}

// Rail destinations of up to three engineers (move_gen.py:870-895): the
// landable rail nodes adjacent to the closure of engineer j's source (rail index
// sr[j]) through empty rail nodes, OR-ed into the wave's LDS words
// dst[3j .. 3j + 2] (compact cells; zero on entry). Lane v evaluates rail nodes
// v and v + 64. A closure is its source and the connected regions of empty nodes
// next to it; a region is grown hop by hop (two ballots) from one node, and the
// largest one is kept for the next engineers, who mostly stand next to the same
// one. 8,192 positions with three engineers a seat: 39.4 -> 32.8 us for the legal
// sets, against one closure grown per engineer.
__device__ __forceinline__ void engineers_bb(int ne, const int sr[3], const BB &occ, const BB &ea, uint64_t *dst)
{
    const int l = lane_id(), v1 = l + 64;
    const bool has1 = v1 < NRAIL;
    const int c0 = cT.railc[l], c1 = has1 ? cT.railc[v1] : 0;
    const bool e0 = !bb_has(occ, c0), e1 = has1 && !bb_has(occ, c1);
    const bool l0 = e0 || bb_has(ea, c0), l1 = has1 && (e1 || bb_has(ea, c1));   // landable (empty or attackable)
    const uint64_t a0 = cT.rnbr[l][0], a1 = cT.rnbr[l][1];
    const uint64_t b0 = has1 ? cT.rnbr[v1][0] : 0ull, b1 = has1 ? cT.rnbr[v1][1] : 0ull;
    uint64_t k0 = 0, k1 = 0;   // the largest region so far
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        if (j >= ne) break;
        uint64_t r0 = sr[j] < 64 ? 1ull << sr[j] : 0ull, r1 = sr[j] >= 64 ? 1ull << (sr[j] - 64) : 0ull;
        // empty neighbours of the source whose region is not in the closure yet
        uint64_t t0 = __ballot(e0 && ((a0 & r0) | (a1 & r1)) != 0);
        uint64_t t1 = __ballot(e1 && ((b0 & r0) | (b1 & r1)) != 0);
        if ((t0 & k0) | (t1 & k1)) {
            r0 |= k0; r1 |= k1;
            t0 &= ~k0; t1 &= ~k1;
        }
        while (t0 | t1) {   // at most four rounds: each takes at least its own node out
            uint64_t q0 = t0 ? t0 & (0 - t0) : 0ull, q1 = t0 ? 0ull : t1 & (0 - t1);
            for (int hop = 0; hop < NRAIL; ++hop) {
                const uint64_t g0 = __ballot(e0 && ((a0 & q0) | (a1 & q1)) != 0);
                const uint64_t g1 = __ballot(e1 && ((b0 & q0) | (b1 & q1)) != 0);
                if (!((g0 & ~q0) | (g1 & ~q1))) break;
                q0 |= g0;
                q1 |= g1;
            }
            r0 |= q0; r1 |= q1;
            t0 &= ~q0; t1 &= ~q1;
            if (__popcll(q0) + __popcll(q1) > __popcll(k0) + __popcll(k1)) { k0 = q0; k1 = q1; }
        }
        if (l != sr[j] && l0 && ((a0 & r0) | (a1 & r1)) != 0)
            atomicOr(reinterpret_cast<unsigned long long *>(&dst[3 * j + (c0 >> 6)]), 1ull << (c0 & 63));
        if (has1 && v1 != sr[j] && l1 && ((b0 & r0) | (b1 & r1)) != 0)
            atomicOr(reinterpret_cast<unsigned long long *>(&dst[3 * j + (c1 >> 6)]), 1ull << (c1 & 63));
    }
}

// Road steps and (for non-engineers) straight rays and curve runs of one piece,
// computed by the calling lane alone (move_gen.py:1052-1199 parts a, b, c, e).
__device__ void piece_mask_lane(const int8_t *cell, int src, int team, bool engineer,
                                uint64_t &m0, uint64_t &m1, uint64_t &m2)
{
    m0 = m1 = m2 = 0;
    for (int k = 0; k < 4; ++k) {
        const int nb = cT.adj[src][k];
        if (nb >= 0 && landable(cell, nb, team)) setbit3(m0, m1, m2, cT.f2c[nb]);
    }
    for (int k = 0; k < 4; ++k) {
        const int nb = cT.diag[src][k];
        if (nb >= 0 && landable(cell, nb, team)) setbit3(m0, m1, m2, cT.f2c[nb]);
    }
    if (engineer) return;
    const int r = cT.railidx[src];
    if (r < 0) return;
    for (int k = 0; k < 4; ++k) {
        const int len = cT.raylen[r][k];
        for (int i = 0; i < len; ++i) {
            const int nb = cT.rays[r][k][i];
            if (cell[nb] < 0) { setbit3(m0, m1, m2, cT.f2c[nb]); continue; }
            if (enemy_att(cell, nb, team)) setbit3(m0, m1, m2, cT.f2c[nb]);
            break;
        }
    }
    for (int d = 0; d < 2; ++d) {
        const int len = cT.craylen[r][d];
        for (int i = 0; i < len; ++i) {
            const int nb = cT.crays[r][d][i];
            if (cell[nb] < 0) { setbit3(m0, m1, m2, cT.f2c[nb]); continue; }
            if (enemy_att(cell, nb, team)) setbit3(m0, m1, m2, cT.f2c[nb]);
            break;
        }
    }
}

// dst on a straight run (k < 4) or curve run of src with every earlier cell empty
// (move_gen.py:127-171 and 384-423). Uniform; every lane active. A straight move
// stays on src's row or column, so only the run toward dst is looked at; lane i
// takes the run's cell i (curve runs: lanes 0-10 and 16-26), all cells at once.
__device__ __forceinline__ bool run_clear(const int8_t *cell, int src, int dst, bool curve)
{
    const int r = tab(cT.railidx, src), l = lane_id();
    if (r < 0) return false;
    int nb = -1;   // the runs are padded with -1
    if (!curve) {
        const int sx = src % 17, sy = src / 17, dx = dst % 17, dy = dst / 17;
        const int k = sy == dy ? (dx > sx ? 0 : 1) : (dy > sy ? 2 : 3);   // +x, -x, +y, -y
        if (l < 12) nb = cT.rays[r][k][l];
    } else if (l < 32 && (l & 15) < 11) {
        nb = cT.crays[r][l >> 4][l & 15];
    }
    const uint64_t hit = __ballot(nb == dst), occ = __ballot(nb >= 0 && cell[nb >= 0 ? nb : 0] >= 0);
    if (!hit) return false;
    const int at = __builtin_ctzll(hit);   // a cell is on one of the two curve runs only
    return (occ & ((1ull << at) - (1ull << (at & 48)))) == 0;
}

__device__ __forceinline__ bool engineer_reaches(const int8_t *cell, int src, int dst)
{   // move_gen.py:186-224: dst is adjacent to the closure of src
    if (!is_rail(src) || !is_rail(dst) || src == dst) return false;
    uint64_t r0, r1;
    const int dr = tab(cT.railidx, dst);
    const uint64_t t0 = cT.rnbr[dr][0], t1 = cT.rnbr[dr][1];
    rail_closure(cell, tab(cT.railidx, src), r0, r1, t0, t1);
    return ((t0 & r0) | (t1 & r1)) != 0;
}

// is_legal_move (move_gen.py:299-376) of the piece sp of type st on src to dst,
// where dp stands (-1 none), and move_requires_gongb (move_gen.py:245-296) of a
// legal engineer move. Uniform; src and dst are cells of the 17 x 17 board. A
// straight or curve run that is clear is also a path of the engineer's closure,
// so an engineer's closure is grown only where no run reaches dst.
__device__ __forceinline__ bool legal_pair(const int8_t *cell, int seat, int src, int dst, int sp, int st, int dp,
                                           bool &engineer_only)
{
    engineer_only = false;
    const uint16_t fs = cflags(src), fd = cflags(dst);
    if (src == dst || !(fs & CF_ON) || !(fd & CF_ON)) return false;
    if (sp < 0 || sp / 30 != seat) return false;
    if (st < T_ZHADAN || st > T_GONGB) return false;   // JUNQI / DILEI never move (no other value is a piece)
    if (fs & CF_SH) return false;
    if (dp >= 0 && (team_of(dp) == (seat & 1) || (fd & CF_CAMP))) return false;   // landable: empty, or an enemy outside a camp
    const int sx = src % 17, sy = src / 17, dx = dst % 17, dy = dst / 17;
    const int adx = abs(sx - dx), ady = abs(sy - dy);
    if (adx <= 1 && ady <= 1 && (adx + ady == 1 || ((fs | fd) & CF_CAMP))) return true;
    if (!(fs & fd & CF_RAIL)) return false;
    const bool straight = sx == dx || sy == dy, curve = (fs >> 8) > 0 && (fs >> 8) == (fd >> 8);
    if ((straight || curve) && run_clear(cell, src, dst, !straight)) return true;
    engineer_only = st == T_GONGB && engineer_reaches(cell, src, dst);
    return engineer_only;
}

// Does `seat` have a legal move (the Q12 test, state.py:1139-1165)?
__device__ __forceinline__ bool seat_has_move(const int8_t *cell, const int16_t *pos, const int8_t *ptype, int seat)
{
    const int l = lane_id(), team = seat & 1;
    bool mov = false, quick = false, eng = false;
    int src = -1;
    if (l < 30) {
        const int pid = seat * 30 + l;
        src = pos[pid];
        const int t = ptype[pid];
        // one round of independent table loads (flags and the four road
        // neighbours), then the LDS reads: no load waits on another
        const int s = src >= 0 ? src : 0;
        const uint16_t fl = cT.cflags[s];
        const int n0 = cT.adj[s][0], n1 = cT.adj[s][1], n2 = cT.adj[s][2], n3 = cT.adj[s][3];
        mov = src >= 0 && t != T_JUNQI && t != T_DILEI && !(fl & CF_SH);
        eng = t == T_GONGB;
        const bool e0 = (n0 >= 0) & (cell[n0 >= 0 ? n0 : 0] < 0), e1 = (n1 >= 0) & (cell[n1 >= 0 ? n1 : 0] < 0);
        const bool e2 = (n2 >= 0) & (cell[n2 >= 0 ? n2 : 0] < 0), e3 = (n3 >= 0) & (cell[n3 >= 0 ? n3 : 0] < 0);
        quick = mov & (e0 | e1 | e2 | e3);
    }
    if (__ballot(mov && quick)) return true;
    uint64_t m0 = 0, m1 = 0, m2 = 0;
    if (mov) piece_mask_lane(cell, src, team, eng, m0, m1, m2);
    if (__ballot((m0 | m1 | m2) != 0)) return true;
    uint64_t engs = __ballot(mov && eng && is_rail(src < 0 ? 0 : src));
    while (engs) {
        const int e = __builtin_ctzll(engs);
        engs &= engs - 1;
        const int esrc = __builtin_amdgcn_readlane(src, e);   // e is wave-uniform
        uint64_t e0, e1, e2;
        engineer_mask(cell, esrc, team, e0, e1, e2);
        if (e0 | e1 | e2) return true;
    }
    return false;
}

__device__ __forceinline__ int resolve_combat(int a, int d)
{   // rules.py:466-516, rows in order
    if (a == T_ZHADAN || d == T_ZHADAN) return EV_BOMB;
    if (d == T_JUNQI) return EV_EAT;
    if (d == T_DILEI) return a == T_GONGB ? EV_EAT : EV_KILLED;
    if (a == d) return EV_BOMB;
    return a < d ? EV_EAT : EV_KILLED;
}

// The Zobrist key table is written only by its upload, never by a kernel, so
// kernels read it as constant memory: a wave-uniform key is then a scalar load,
// which does not wait behind the wave's vector stores.
typedef const __attribute__((address_space(4))) uint64_t *KeyTable;
__device__ __forceinline__ KeyTable keys(const uint64_t *z) { return reinterpret_cast<KeyTable>(reinterpret_cast<uintptr_t>(z)); }

__device__ __forceinline__ int zp_index(int pid, int t, int f)
{   // indexes come from state rows; out-of-range values read entry 0 instead of faulting
    pid = (unsigned)pid < 120u ? pid : 0;
    t = (unsigned)t < 14u ? t : 0;
    f = (unsigned)f < 289u ? f : 0;
    return (pid * 14 + t) * 289 + f;
}
__device__ __forceinline__ uint64_t zp(const uint64_t *z, int pid, int t, int f) { return keys(z)[zp_index(pid, t, f)]; }

__device__ __forceinline__ int tracked(int t) { return (t >= 2 && t <= 13) ? t - 2 : -1; }
__device__ __forceinline__ bool code_onehot(int c) { return c >= 1 && c <= 12; }
__device__ __forceinline__ int rank_floor_next(int t)
{   // combat_memory.py:163-173: ordinary rank GONGB=1..SILING=9, floor = min(rank+1, 9)
    if (t < T_SILING || t > T_GONGB) return 0;
    const int r = T_GONGB - t + 1;
    return r + 1 < 9 ? r + 1 : 9;
}
__device__ __forceinline__ bool sees_truth(int o, int owner, int mode)
{   // info_model.py:568-577
    if (mode == SM_BRIGHT || o == owner) return true;
    return mode == SM_HALF_DARK && ((o & 1) == (owner & 1));
}

// ------------------------------------------------------------------ step
struct StepOut {
    uint8_t *valid; int8_t *event; uint8_t *term; int8_t *winner; uint8_t *draw;
    uint8_t *fcap; uint8_t *died; float *reward; int32_t *world;
    uint64_t *hash;   // Zobrist hash after the ply (unchanged when none was applied)
};

// The values a ply reports (wave-uniform). The caller stores them once its
// own loads are issued: a load issued after a store waits for that store too.
struct StepRes {
    int valid, event, term, winner, draw, fcap, died, world;
    float reward;
    uint64_t hash;
};

__device__ __forceinline__ void write_step_res(const StepOut &O, int env, const StepRes &r)
{
    if (O.valid) O.valid[env] = (uint8_t)r.valid;
    if (O.event) O.event[env] = (int8_t)r.event;
    if (O.term) O.term[env] = (uint8_t)r.term;
    if (O.winner) O.winner[env] = (int8_t)r.winner;
    if (O.draw) O.draw[env] = (uint8_t)r.draw;
    if (O.fcap) O.fcap[env] = (uint8_t)r.fcap;
    if (O.died) O.died[env] = (uint8_t)r.died;
    if (O.reward) O.reward[env] = r.reward;
    if (O.world) O.world[env] = r.world;
    if (O.hash) O.hash[env] = r.hash;
}

// Remove every live piece of `seat` (state.py:1639-1692): KILLED_BY_ENEMY at the
// piece's current cell. Lanes 0..29 take one pid each and fold its key into
// their share zacc of the Zobrist change.
__device__ void purge_seat(const State &S, int env, int8_t *cell, int16_t *pos, const int8_t *ptype, int seat,
                           int step, uint64_t &zacc)
{
    const int l = lane_id();
    wave_sync();
    if (l < 30) {
        const int pid = seat * 30 + l;
        const int cur = pos[pid];
        if ((unsigned)cur < (unsigned)NC) {
            zacc ^= zp(S.ztab, pid, ptype[pid], cur);
            cell[cur] = -1; pos[pid] = -1;
            PieceRec &r = S.piece[pc_idx(env, pid)];
            r.pos = -1; r.dreason = 0; r.dstep = (int16_t)step; r.dloc = (int16_t)cur;
            S.cell[(size_t)env * CELL_STRIDE + cur] = -1;
        }
    }
    wave_sync();
}

// The Zobrist keys a ply may XOR in, one per lane, loaded together as soon as
// the moving pieces are known: the ply collects the lanes that count in a
// uniform set and folds them once at its end. (As scalar loads each was waited
// for at the wave's next LDS fence, which shares their counter.) With the kills
// and the move in one block, one legality walk, counters from the records
// already loaded and boards moved as words, a wave's ply went from 8,112 to
// 6,545 lines of assembly and 23.6 k to 20.8 k cycles alone on its SIMD (us per
// fused step: u8 32,768 games 723 -> 713, bf16 16,384 658 -> 652, state only
// 4,096 32.1 -> 29.6, u8 64 25.2 -> 23.8).
enum : int {
    ZL_TURN = 0, ZL_MC0 = 4, ZL_MC1 = 5, ZL_MSLC0 = 6, ZL_MSLC1 = 7, ZL_MSLC_RESET = 8, ZL_SRC = 9, ZL_DST = 10,
    ZL_KILL_D = 11, ZL_KILL_S = 12, ZL_TERM = 16, ZL_WIN = ZL_TERM + (ZOFF_WIN - ZOFF_TERM),
    ZL_DRAW = ZL_TERM + (ZOFF_DRAW - ZOFF_TERM), ZL_SDEAD = ZL_TERM + (ZOFF_SDEAD - ZOFF_TERM),
    ZL_SFLAG = ZL_TERM + (ZOFF_SFLAG - ZOFF_TERM), ZL_END = ZL_SFLAG + 4
};
static_assert(ZL_END <= 32, "one bit of a 32-bit set per key");

// CombatMemory update for EAT / KILLED (combat_memory.py:354-569). Lane o < 4
// handles observer o; observers never touch each other's records. K is the
// surviving piece, V the killed one; V's own kills cannot include K (K is alive).
__device__ __forceinline__ void cm_apply(const State &S, int env, bool is_eat, int apid, int dpid, int aseat, int dseat,
                         int atype, int dtype, int step)
{
    const int o = lane_id();
    if (o >= 4) return;
    int K, V, Vs, Vt;
    if (is_eat) { K = apid; V = dpid; Vs = dseat; Vt = dtype; }
    else        { K = dpid; V = apid; Vs = aseat; Vt = atype; }
    const size_t kI = cm_idx(env, o, K), vI = cm_idx(env, o, V);
    CmRec k = S.cm[kI];
    const CmRec v = S.cm[vI];
    if (!is_eat) {
        const bool known = (v.flags & CMF_IS_GONGB) || (atype == T_GONGB && o == Vs);
        if (known) k.flags |= CMF_ATK_GONGB;
    }
    k.clo |= v.dlo | v.clo;
    k.chi |= v.dhi | v.chi;
    if (V < 64) k.clo |= 1ull << V; else k.chi |= 1ull << (V - 64);
    k.ctype = (uint16_t)(k.ctype | v.dtype | v.ctype);
    if (v.floor > 0) {
        const int prop = v.floor + 1 < 9 ? v.floor + 1 : 9;
        if (prop > k.floor) { k.floor = (int8_t)prop; k.fstep = (int16_t)step; }
        k.flags |= CMF_NOT_GONGB;
    }
    // v6 reverse projection: observer's own pids V had eaten (directly or by chain),
    // plus V itself when V belongs to the observer, are now eaten by K too.
    {
        // pids 30o .. 30o + 29 as a 128-bit set (o = 0..3: bit offsets 0, 30, 60, 90)
        constexpr uint64_t SEAT30 = 0x3FFFFFFFull;
        const int b0 = o * 30;
        const uint64_t mlo = b0 < 64 ? SEAT30 << b0 : 0ull;
        const uint64_t mhi = b0 == 0 ? 0ull : b0 < 64 ? SEAT30 >> (64 - b0) : SEAT30 << (b0 - 64);
        uint64_t vlo = (v.dlo | v.clo) & mlo, vhi = (v.dhi | v.chi) & mhi;
        if (Vs == o) { if (V < 64) vlo |= 1ull << V; else vhi |= 1ull << (V - 64); }
        const uint64_t klo = K < 64 ? (1ull << K) : 0ull, khi = K >= 64 ? (1ull << (K - 64)) : 0ull;
        while (vlo) { const int b = __builtin_ctzll(vlo); vlo &= vlo - 1; CmEat &t = S.cme[cm_idx(env, o, b)]; t.elo |= klo; t.ehi |= khi; }
        while (vhi) { const int b = __builtin_ctzll(vhi) + 64; vhi &= vhi - 1; CmEat &t = S.cme[cm_idx(env, o, b)]; t.elo |= klo; t.ehi |= khi; }
    }
    if (Vs != o) {
        const int c = k.ocnt + 1;
        k.ocnt = (int16_t)(c < 32767 ? c : 32767);
    } else {
        if (V < 64) k.dlo |= 1ull << V; else k.dhi |= 1ull << (V - 64);
        const int vi = tracked(Vt);
        if (vi >= 0) {
            k.dtype = (uint16_t)(k.dtype | (1u << vi));
            k.ctype = (uint16_t)(k.ctype | (1u << vi));
        }
        if (is_eat) k.flags |= (Vt == T_DILEI) ? CMF_IS_GONGB : CMF_NOT_GONGB;
        if (Vt >= T_SILING && Vt <= T_GONGB) {
            const int pr = rank_floor_next(Vt);
            if (pr > k.floor) { k.floor = (int8_t)pr; k.fstep = (int16_t)step; }
        }
    }
    k.ldir = (int16_t)step;
    k.lchain = (int16_t)step;
    S.cm[kI] = k;
    S.cmk[kI] = cm_summary(k);
    S.cmv[kI] = cm_view(k, o);
}

// BeliefTensor.update for the four observers (info_model.py:271-429). Entries are
// keyed by pid so R1 migration is implicit; lane o < 4 handles observer o, whose
// tracked seats (trk) and codes of the two pieces are loaded by the caller.
__device__ __forceinline__ void belief_update(const State &S, int env, const int8_t *cell, int sp, int dp, int ss, int ds,
                              int dt, int dst, int ev, bool rsrc, bool rdst, bool fcap, int died, uint8_t trk,
                              int acode, const int dcode)
{
    const int o = lane_id();
    if (o >= 4) return;
    uint8_t *bc = S.bcode + ((size_t)env * 4 + o) * PID_STRIDE;
    int8_t *rem = S.rem + ((size_t)env * 4 + o) * 48;
    auto dec = [&](int seat, int ti) {
        if ((trk >> seat) & 1) { int8_t &c = rem[seat * 12 + ti]; if (c > 0) --c; }
    };
    if (rsrc) dec(ss, T_SILING - 2);
    if (rdst) dec(ds, T_SILING - 2);
    if (ev == EV_EAT && dp >= 0 && dt == T_DILEI && !code_onehot(acode)) {
        acode = 1 + (T_GONGB - 2);
        bc[sp] = (uint8_t)acode;
        dec(ss, T_GONGB - 2);
    }
    if (fcap) {
        trk &= (uint8_t)~(1u << ds);
    } else if (ev == EV_EAT && dp >= 0 && is_sh(dst) && tab(cT.owner, dst) == ds) {
        const int other = tab(cT.sh_other, dst);
        const int op = cell[other];
        if (op >= 0 && !code_onehot(bc[op])) bc[op] = (uint8_t)(1 + (T_JUNQI - 2));
    }
    auto removed = [&](int seat, int code) { if (((trk >> seat) & 1) && code_onehot(code)) dec(seat, code - 1); };
    if (ev == EV_EAT) { if (dp >= 0) removed(ds, dcode); }
    else if (ev == EV_KILLED) removed(ss, acode);
    else if (ev == EV_BOMB) { removed(ss, acode); if (dp >= 0) removed(ds, dcode); }
    trk &= (uint8_t)~died;
    S.env[env].remtrk[o] = trk;
}

// What the env record says after a step (wave-uniform), for work that follows
// the step in the same kernel.
struct TurnAfter {
    int turn;
    bool term;
    uint8_t sdead;
};

// One ply of env `env` by its wave (GameState.step_inplace, state.py:700-1167).
// cell / pos / ptype are the wave's LDS arrays; on return they hold the board
// after the step (unchanged if the action was not applied).
// The board and piece records of one env, lane l's share: the loads of a ply's
// first memory round trip, which a caller can issue early.
struct StepLoad {
    uint32_t c0, c1;   // board words l and l + 64 (l < 9)
    uint4 r0, r1;      // records of pids l and l + 64
};

// A board is 73 words in global memory and in LDS, the three bytes past its last
// cell -1. Lane l moves words l and l + 64.
__device__ __forceinline__ void board_load(const State &S, int env, int l, uint32_t &c0, uint32_t &c1)
{
    const uint32_t *w = reinterpret_cast<const uint32_t *>(S.cell + (size_t)env * CELL_STRIDE);
    c0 = w[l];
    c1 = w[min(l + 64, CELL_STRIDE / 4 - 1)];
}
__device__ __forceinline__ void board_stage(int8_t *cell, int l, uint32_t c0, uint32_t c1)
{
    static_assert(CELL_STRIDE / 4 == 73 && NC == 289, "the last word holds one cell");
    uint32_t *w = reinterpret_cast<uint32_t *>(cell);
    w[l] = c0;
    if (l < CELL_STRIDE / 4 - 64) w[l + 64] = l == CELL_STRIDE / 4 - 65 ? c1 | 0xFFFFFF00u : c1;
}

__device__ __forceinline__ void step_load(const State &S, int env, int l, StepLoad &P)
{
    board_load(S, env, l, P.c0, P.c1);
    P.r0 = *reinterpret_cast<const uint4 *>(&S.piece[pc_idx(env, l)]);
    P.r1 = *reinterpret_cast<const uint4 *>(&S.piece[pc_idx(env, l + 64)]);
}
__device__ __forceinline__ PieceRec piece_rec(const uint4 &v)
{
    PieceRec r;
    __builtin_memcpy(&r, &v, sizeof r);
    return r;
}

__device__ void step_env(const State &S, int env, int l, int32_t a, const int8_t *__restrict__ acting, int act_fmt,
                         StepRes &res, int8_t *cell, int16_t *pos, int8_t *ptype, TurnAfter &nx,
                         const StepLoad *pre = nullptr, const EnvRec *pre_rec = nullptr)
{

    // the board, the piece records, the env record and the action are all
    // loaded into registers first (one memory round trip, or `pre` issued
    // earlier by the caller), then staged in LDS; the checks below only decide
    // whether the board is used
    StepLoad ld;
    if (pre) ld = *pre;
    else step_load(S, env, l, ld);
    const PieceRec r0 = piece_rec(ld.r0), r1 = piece_rec(ld.r1);
    // the env record, read once into scalar registers before any store of the
    // ply (only this wave writes it, at the end), or handed in by the caller
    const EnvRec E = pre_rec ? *pre_rec : env_record(S, env);
    board_stage(cell, l, ld.c0, ld.c1);
    pos[l] = r0.pos; ptype[l] = r0.ptype;
    pos[l + 64] = r1.pos; ptype[l + 64] = r1.ptype;
    const bool was_term = E.term != 0;
    const int seat = E.turn;
    nx.turn = seat; nx.term = was_term; nx.sdead = E.sdead;
    res = {0, 0, was_term ? 1 : 0, (int)E.winner, (int)E.draw, 0, 0, -1, 0.f, E.zob};
    if (was_term) return;

    a = __builtin_amdgcn_readfirstlane(a);   // wave-uniform: the ply's scalar work stays on the SALU
    int src = -1, dst = -1;
    if (act_fmt == 1) {
        const int as = __builtin_amdgcn_readfirstlane(acting ? (int)acting[env] : seat);
        if (a >= 0 && a < NONB * NONB && as >= 0 && as < 4) {
            src = tab(cT.unrot[as], tab(cT.c2f, a / NONB));
            dst = tab(cT.unrot[as], tab(cT.c2f, a % NONB));
        }
    } else if (a >= 0 && a < NC * NC) {
        src = a / NC; dst = a % NC;
    }
    if (src >= 0) res.world = src * NC + dst;
    if (src < 0) return;
    if (acting && acting[env] != seat) return;
    const uint8_t sdead0 = E.sdead;
    if ((sdead0 >> seat) & 1) return;
    wave_sync();
    // the pieces on both cells, their types and cells: two rounds of LDS reads
    const int sp = __builtin_amdgcn_readfirstlane(cell[src]), dp = __builtin_amdgcn_readfirstlane(cell[dst]);
    int st = -1, dt = -1, spos = -1, dpos = -1;
    {
        const int a = sp >= 0 ? sp : 0, d = dp >= 0 ? dp : 0;
        const int v0 = ptype[a], v1 = ptype[d], v2 = pos[a], v3 = pos[d];
        st = __builtin_amdgcn_readfirstlane(v0);
        spos = __builtin_amdgcn_readfirstlane(v2);
        if (dp >= 0) { dt = __builtin_amdgcn_readfirstlane(v1); dpos = __builtin_amdgcn_readfirstlane(v3); }
    }
    bool gongb_only;
    if (!legal_pair(cell, seat, src, dst, sp, st, dp, gongb_only)) return;

    const int mc0 = E.mc, mslc0 = E.mslc;
    const int step = mc0 + 1;
    int died = 0;
    uint8_t sdead = sdead0, sflag = E.sflag;
    const int ss = sp / 30, ds = dp >= 0 ? dp / 30 : -1;

    // loads whose values are only needed at the ply's end: the Zobrist keys
    // (lane ZL_*) and the four observers' belief codes of the two pieces
    int zi = l < 4 ? ZOFF_TURN + l : ZOFF_TERM + (l < ZL_END ? l - ZL_TERM : 0);
    // the value is fixed as a scalar first, so that this is a select and not a branch
    auto put = [&](int lane, int v) { v = __builtin_amdgcn_readfirstlane(v); zi = l == lane ? v : zi; };
    put(ZL_MC0, ZOFF_MC + (mc0 & 0xFFF));
    put(ZL_MC1, ZOFF_MC + ((mc0 + 1) & 0xFFF));
    put(ZL_MSLC0, ZOFF_MSLC + (mslc0 & 0x1FF));
    put(ZL_MSLC1, ZOFF_MSLC + ((mslc0 + 1) & 0x1FF));
    put(ZL_MSLC_RESET, ZOFF_MSLC);
    put(ZL_SRC, zp_index(sp, st, src));
    put(ZL_DST, zp_index(sp, st, dst));
    put(ZL_KILL_D, zp_index(dp, dt, dpos));
    put(ZL_KILL_S, zp_index(sp, st, spos));
    const uint64_t zkey = S.ztab[zi];
    const uint8_t *bc = S.bcode + ((size_t)env * 4 + (l & 3)) * PID_STRIDE;   // every lane loads, lanes 0-3 use it
    const int acode = bc[sp], dcode = bc[dp >= 0 ? dp : sp];                  // dcode: only with a piece on dst
    uint64_t zm = 1u << (ZL_TURN + seat) | 1u << ZL_MC0 | 1u << ZL_MSLC0;   // the lanes whose keys count
    uint64_t zacc = 0;                                                      // this lane's purged pieces

    if (gongb_only) {
        if (l < 4) {
            S.cm[cm_idx(env, l, sp)].flags |= CMF_IS_GONGB;
            S.cmk[cm_idx(env, l, sp)] |= (uint8_t)(CMF_IS_GONGB << 2);
            S.cmv[cm_idx(env, l, sp)].types |= (uint32_t)CMF_IS_GONGB << 28;
        }
    }
    // move history (state.py:673-678)
    const int hcnt = E.hmeta & 0xFF, hhead = (E.hmeta >> 8) & 31;
    if (l == 0) S.hist[(size_t)env * HIST_LEN + hhead] = src | (dst << 16);
    int ev;
    bool rsrc = false, rdst = false, fcap = false;
    auto set_flag = [&](int s) { if (!((sflag >> s) & 1)) { sflag |= (uint8_t)(1u << s); zm ^= 1u << (ZL_SFLAG + s); } };
    auto set_dead = [&](int s) { if (!((sdead >> s) & 1)) { sdead |= (uint8_t)(1u << s); zm ^= 1u << (ZL_SDEAD + s); } };
    ev = dp < 0 ? EV_MOVE : resolve_combat(st, dt);
    const bool moved = ev == EV_MOVE || ev == EV_EAT;
    const bool kill_s = (ev == EV_KILLED || ev == EV_BOMB) && (unsigned)spos < (unsigned)NC;   // a piece on no cell stays as it is
    const bool kill_d = (ev == EV_EAT || ev == EV_BOMB) && (unsigned)dpos < (unsigned)NC;
    if (dp >= 0) {
        rsrc = st == T_SILING && (ev == EV_KILLED || ev == EV_BOMB);
        rdst = dt == T_SILING && (ev == EV_EAT || ev == EV_BOMB);
        fcap = dt == T_JUNQI;
        if (rsrc) set_flag(ss);
        if (rdst) set_flag(ds);
    }
    if (kill_s) zm ^= 1u << ZL_KILL_S;
    if (kill_d) zm ^= 1u << ZL_KILL_D;
    if (moved) zm ^= 1u << ZL_SRC | 1u << ZL_DST;
    // the counter of a move, a capture or a survived attack, by the lane that
    // loaded the piece's record
    const int cp = ev == EV_KILLED ? dp : sp;
    if (ev != EV_BOMB && l == (cp & 63)) {
        const int16_t m = cp < 64 ? r0.mcount : r1.mcount, e = cp < 64 ? r0.aeat : r1.aeat, v = cp < 64 ? r0.psurv : r1.psurv;
        int16_t *c = &S.piece[pc_idx(env, cp)].mcount;   // mcount, aeat, psurv in a row
        c[ev == EV_MOVE ? 0 : ev == EV_EAT ? 1 : 2] = (int16_t)((ev == EV_MOVE ? m : ev == EV_EAT ? e : v) + 1);
    }
    wave_sync();
    // kills (state.py:1027-1049): lane 0 the piece on dst, lane 1 the mover
    if (l < 2 && (l ? kill_s : kill_d)) {
        const int pid = l ? sp : dp, cur = l ? spos : dpos;
        const int why = ev == EV_BOMB ? 2 : (l && (dt == T_DILEI || dt == T_ZHADAN)) ? 1 : 0;
        cell[cur] = -1; pos[pid] = -1;
        PieceRec &r = S.piece[pc_idx(env, pid)];
        r.pos = -1; r.dreason = (int8_t)why; r.dstep = (int16_t)step; r.dloc = (int16_t)dst;
        S.cell[(size_t)env * CELL_STRIDE + cur] = -1;
    }
    if (moved && l == 0) {   // state.py:1005-1025; after lane 0's own kill on dst
        cell[src] = -1; cell[dst] = (int8_t)sp; pos[sp] = (int16_t)dst;
        S.cell[(size_t)env * CELL_STRIDE + src] = -1;
        S.cell[(size_t)env * CELL_STRIDE + dst] = (int8_t)sp;
        S.piece[pc_idx(env, sp)].pos = (int16_t)dst;
    }
    wave_sync();
    if (ev == EV_EAT || ev == EV_KILLED) cm_apply(S, env, ev == EV_EAT, sp, dp, ss, ds, st, dt, step);
    if (fcap && !((sdead >> ds) & 1)) {   // state.py:864-890
        set_dead(ds); set_flag(ds);
        purge_seat(S, env, cell, pos, ptype, ds, step, zacc);
        died |= 1 << ds;
    }
    {   // dead sweep (state.py:895-901)
        const uint64_t a0 = __ballot(pos[l] >= 0), a1 = __ballot(l + 64 < NP && pos[l + 64] >= 0);   // pids on the board
        for (int s = 0; s < 4; ++s)
            if (!((sdead >> s) & 1) && !seat_bits(a0, a1, s * 30)) { set_dead(s); died |= 1 << s; }
    }
    const int nmc = mc0 + 1, nmslc = ev == EV_MOVE ? mslc0 + 1 : 0;
    auto victory = [&](int &term, int &win, int &drw) {   // state.py:1695-1726
        const bool red = !(((sdead >> 0) & 1) && ((sdead >> 2) & 1));
        const bool blue = !(((sdead >> 1) & 1) && ((sdead >> 3) & 1));
        term = 0; win = -1; drw = 0;
        if (!red && !blue) { term = 1; win = seat & 1; return; }
        if (!red) { term = 1; win = 1; return; }
        if (!blue) { term = 1; win = 0; return; }
        if (nmc >= 4000 || nmslc >= 200) { term = 1; drw = 1; }
    };
    int term, win, drw, nturn;
    victory(term, win, drw);
    if (!term) {   // state.py:1109-1167
        int cand = (seat + 1) & 3;
        for (int it = 0; it < 4; ++it) {
            if ((sdead >> cand) & 1) { cand = (cand + 1) & 3; continue; }
            if (seat_has_move(cell, pos, ptype, cand)) break;
            set_dead(cand);
            purge_seat(S, env, cell, pos, ptype, cand, step, zacc);
            died |= 1 << cand;
            cand = (cand + 1) & 3;
        }
        nturn = cand;
        victory(term, win, drw);
    } else {
        nturn = seat;
    }
    if (!term && nmc >= S.max_moves) { term = 1; drw = 1; }   // env move cap
    zm ^= 1u << (ZL_TURN + nturn) | 1u << ZL_MC1;
    zm ^= 1u << (ev == EV_MOVE ? ZL_MSLC1 : ZL_MSLC_RESET);
    if (term) zm ^= 1u << ZL_TERM;
    if (drw) zm ^= 1u << ZL_DRAW;
    if (win >= 0) zm ^= 1u << ZL_WIN | 1u << (ZL_WIN + win + 1);
    const uint64_t zob = E.zob ^ wave_xor(zacc ^ ((zm >> l) & 1 ? zkey : 0ull));

    const uint8_t trk = l == 0 ? E.remtrk[0] : l == 1 ? E.remtrk[1] : l == 2 ? E.remtrk[2] : E.remtrk[3];
    belief_update(S, env, cell, sp, dp, ss, ds, dt, dst, ev, rsrc, rdst, fcap, died, trk, acode, dcode);

    nx.turn = nturn; nx.term = term != 0; nx.sdead = sdead;
    if (l == 0) {
        EnvRec &W = S.env[env];   // remtrk belongs to belief_update's lanes
        W.zob = zob; W.mc = nmc; W.mslc = nmslc;
        W.hmeta = (hcnt < 32 ? hcnt + 1 : 32) | (((hhead + 1) & 31) << 8);
        W.turn = (int8_t)nturn; W.term = (uint8_t)term; W.winner = (int8_t)win; W.draw = (uint8_t)drw;
        W.sdead = sdead; W.sflag = sflag;
    }
    res.valid = 1; res.event = ev; res.term = term; res.winner = win; res.draw = drw; res.fcap = fcap;
    res.died = died; res.hash = zob;
    res.reward = (term && !drw && win >= 0) ? (((seat & 1) == win) ? 1.f : -1.f) : 0.f;
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(8, 8))) void k_step(State S, const int32_t *__restrict__ actions,
                                             const int8_t *__restrict__ acting, int act_fmt, StepOut O)
{
    const int env = blockIdx.x, l = threadIdx.x;
    if (env >= S.n) return;
    __shared__ alignas(4) int8_t cell[CELL_STRIDE];
    __shared__ int16_t pos[PID_STRIDE];
    __shared__ int8_t ptype[PID_STRIDE];
    TurnAfter nx;
    StepRes res;
    step_env(S, env, l, actions[env], acting, act_fmt, res, cell, pos, ptype, nx);
    if (l == 0) write_step_res(O, env, res);
}

// ------------------------------------------------------------------ reset
// Empty, terminated state of every env (no pieces, empty board, zero beliefs),
// before the first reset.
__global__ __launch_bounds__(64) void k_clear(State S)
{
    const int env = blockIdx.x, t = threadIdx.x, nt = 64;
    if (env >= S.n) return;
    for (int f = t; f < CELL_STRIDE; f += nt) S.cell[(size_t)env * CELL_STRIDE + f] = -1;
    PieceRec r;
    r.pos = r.zero = r.dstep = r.dloc = -1;
    r.mcount = r.aeat = r.psurv = 0;
    r.ptype = r.dreason = -1;
    CmRec c = {};
    c.ldir = c.lchain = c.fstep = -1;
    const CmEat ce = {};
    const CmView cv = cm_view(c, 0);
    for (int p = t; p < PID_STRIDE; p += nt) {
        S.piece[pc_idx(env, p)] = r;
        for (int o = 0; o < 4; ++o) {
            S.cm[cm_idx(env, o, p)] = c;
            S.cme[cm_idx(env, o, p)] = ce;
            S.cmk[cm_idx(env, o, p)] = 0;
            S.cmv[cm_idx(env, o, p)] = cv;
            S.bcode[((size_t)env * 4 + o) * PID_STRIDE + p] = 0;
        }
    }
    for (int k = t; k < 4 * 48; k += nt) S.rem[(size_t)env * 4 * 48 + k] = 0;
    for (int k = t; k < HIST_LEN; k += nt) S.hist[(size_t)env * HIST_LEN + k] = 0;
    if (t == 0) {
        EnvRec E = {};
        E.winner = -1;
        E.term = 1;
        S.env[env] = E;
        S.lg[env].n = 0;
        S.lg[env].seat = 0;
    }
}

// Start an env from a lineup (GameState.new_game, state.py:490-620; beliefs,
// info_model.py:218-265). Zobrist includes every term new_game XORs in. If
// lcell is given, the new board is also staged in the wave's LDS arrays
// lcell / lpos / ltype (as step_env leaves them).
__device__ void init_env(const State &S, int env, const int8_t *types, int8_t *lcell = nullptr,
                         int16_t *lpos = nullptr, int8_t *ltype = nullptr)
{
    const int l = lane_id();
    int8_t *cell = S.cell + (size_t)env * CELL_STRIDE;
    for (int f = l; f < CELL_STRIDE; f += 64) {
        cell[f] = -1;
        if (lcell) lcell[f] = -1;
    }
    wave_sync();
    uint64_t z = 0;
    for (int p = l; p < PID_STRIDE; p += 64) {
        const size_t pi = (size_t)env * PID_STRIDE + p;
        const int t = p < NP ? types[p] : 0;
        const bool alive = t != T_NONE && cT.home[p < NP ? p : 0] >= 0 && p < NP;
        const int h = alive ? cT.home[p] : -1;
        PieceRec r;
        r.ptype = alive ? (int8_t)t : (int8_t)-1;
        r.pos = (int16_t)h; r.zero = (int16_t)h;
        r.mcount = 0; r.aeat = 0; r.psurv = 0;
        r.dreason = -1; r.dstep = -1; r.dloc = -1;
        S.piece[pi] = r;
        if (alive) { cell[h] = (int8_t)p; z ^= zp(S.ztab, p, t, h); }
        if (lcell) {
            if (alive) lcell[h] = (int8_t)p;
            lpos[p] = (int16_t)h;
            ltype[p] = r.ptype;
        }
        for (int o = 0; o < 4; ++o) {
            uint8_t code = 0;
            if (alive) code = sees_truth(o, p / 30, S.show_mode) ? (uint8_t)(1 + t - 2) : (uint8_t)(BC_PRIOR0 + p % 30);
            S.bcode[((size_t)env * 4 + o) * PID_STRIDE + p] = code;
            CmRec c = {};
            c.ldir = -1; c.lchain = -1; c.fstep = -1;
            S.cm[cm_idx(env, o, p)] = c;
            S.cme[cm_idx(env, o, p)] = CmEat{};
            S.cmk[cm_idx(env, o, p)] = 0;
            S.cmv[cm_idx(env, o, p)] = cm_view(c, o);
        }
    }
    z = wave_xor(z);
    static constexpr int8_t kCounts[12] = {1, 3, 2, 1, 1, 2, 2, 2, 2, 3, 3, 3};
    for (int i = l; i < 4 * 48; i += 64) {
        const int o = i / 48, s = (i / 12) % 4, t = i % 12;
        const bool tracked_seat = s != o && ((s & 1) != (o & 1));
        S.rem[(size_t)env * 4 * 48 + i] = tracked_seat ? kCounts[t] : 0;
    }
    if (l < 4) {
        uint8_t trk = 0;
        for (int s = 0; s < 4; ++s) if (s != l && ((s & 1) != (l & 1))) trk |= (uint8_t)(1u << s);
        S.env[env].remtrk[l] = trk;
    }
    if (l == 0) {
        const KeyTable Z = keys(S.ztab);
        z ^= Z[ZOFF_TURN + 0] ^ Z[ZOFF_MC + 0] ^ Z[ZOFF_MSLC + 0] ^ Z[ZOFF_WIN + 0] ^ Z[ZOFF_SHOW + S.show_mode];
        EnvRec &W = S.env[env];
        W.zob = z; W.mc = 0; W.mslc = 0; W.hmeta = 0;
        W.turn = 0; W.term = 0; W.winner = -1; W.draw = 0; W.sdead = 0; W.sflag = 0;
    }
}

__global__ __launch_bounds__(64) void k_reset_lineups(State S, const int8_t *__restrict__ lineups)
{
    const int env = blockIdx.x;
    if (env >= S.n) return;
    init_env(S, env, lineups + (size_t)env * NP);
}

// Pool entry a finished env restarts from: the reference reset kernel's hash
// (game_state.cu:2986-2991).
__device__ __forceinline__ int reset_pool_index(int env, int64_t seed, int pool_size)
{
    uint64_t h = (uint64_t)env * 2654435761ull + (uint64_t)seed;
    h ^= h >> 17;
    h *= 0xbf58476d1ce4e5b9ull;
    h ^= h >> 31;
    return (int)(h % (uint64_t)pool_size);
}

__global__ __launch_bounds__(64) void k_reset_terminated(State S, int64_t seed)
{
    const int env = blockIdx.x;
    if (env >= S.n || !S.env[env].term) return;
    init_env(S, env, S.pool + (size_t)reset_pool_index(env, seed, S.pool_size) * NP);
}

// Recompute Zobrist and (if `beliefs`) re-seed beliefs from the current board
// (hand-built states); only envs whose `mask` entry is nonzero when a mask is given.
__global__ __launch_bounds__(64) void k_finalize(State S, int beliefs, const uint8_t *__restrict__ mask)
{
    const int env = blockIdx.x, l = threadIdx.x;
    if (env >= S.n || (mask && !mask[env])) return;
    uint64_t z = 0;
    for (int p = l; p < NP; p += 64) {
        const size_t pi = (size_t)env * PID_STRIDE + p;
        const PieceRec r = S.piece[pi];
        const int f = r.pos, t = r.ptype;
        if (f >= 0 && t >= 0) z ^= zp(S.ztab, p, t, f);
        for (int o = 0; o < 4; ++o) {
            const CmRec c = S.cm[cm_idx(env, o, p)];
            S.cmk[cm_idx(env, o, p)] = cm_summary(c);
            S.cmv[cm_idx(env, o, p)] = cm_view(c, o);
        }
        for (int o = 0; o < 4 && beliefs; ++o) {
            uint8_t code = 0;
            if (f >= 0 && t >= 2) {
                if (sees_truth(o, p / 30, S.show_mode)) code = (uint8_t)(1 + t - 2);
                else code = (cT.owner[f] == p / 30) ? (uint8_t)(BC_PRIOR0 + cT.localidx[f]) : (uint8_t)BC_UNIFORM;
            }
            S.bcode[((size_t)env * 4 + o) * PID_STRIDE + p] = code;
        }
    }
    z = wave_xor(z);
    static constexpr int8_t kCounts[12] = {1, 3, 2, 1, 1, 2, 2, 2, 2, 3, 3, 3};
    if (beliefs && l < 48) {
        for (int o = 0; o < 4; ++o) {
            const int s = l / 12, t = l % 12;
            const bool tracked_seat = s != o && ((s & 1) != (o & 1));
            S.rem[((size_t)env * 4 + o) * 48 + l] = tracked_seat ? kCounts[t] : 0;
        }
    }
    if (beliefs && l < 4) {
        uint8_t trk = 0;
        for (int s = 0; s < 4; ++s) if (s != l && ((s & 1) != (l & 1))) trk |= (uint8_t)(1u << s);
        S.env[env].remtrk[l] = trk;
    }
    if (l == 0) {
        const KeyTable Z = keys(S.ztab);
        const EnvRec &E = S.env[env];
        const int w = E.winner;
        z ^= Z[ZOFF_TURN + (E.turn & 3)] ^ Z[ZOFF_MC + (E.mc & 0xFFF)] ^ Z[ZOFF_MSLC + (E.mslc & 0x1FF)];
        z ^= Z[ZOFF_WIN + (w < 0 ? 0 : (w & 1) + 1)] ^ Z[ZOFF_SHOW + S.show_mode];
        if (E.term) z ^= Z[ZOFF_TERM];
        if (E.draw) z ^= Z[ZOFF_DRAW];
        for (int s = 0; s < 4; ++s) {
            if ((E.sdead >> s) & 1) z ^= Z[ZOFF_SDEAD + s];
            if ((E.sflag >> s) & 1) z ^= Z[ZOFF_SFLAG + s];
        }
        S.env[env].zob = z;
    }
}

// ------------------------------------------------------------------ legal
// Per env: masks of the acting seat's movable pieces (lanes = pieces), engineer
// closures, counts, the packed canonical mask and the CSR scratch in ascending
// source order (move_gen.py:1199 sorts the ids).
// Legal sets of env `env` for `seat` by its wave (off: none): the board in LDS
// (cell, padded to CELL_STRIDE with -1) and, for the canonical mask, bits
// cleared; rotl is filled here. src / t: cell and type of piece l & 31 of the seat (lanes p
// and p + 32 share piece p < 30, one half of its moves each).
// lscr: LSCR_WORDS words of the wave's LDS, the compact source cells of the
// movable pieces (words 0-2) and the engineers' rail destinations (3-11).
// The masks go to row `row` (the env's own index, or the row of a minibatch
// rebuilt from a history); REC: the legal record of the CSR pass is written.
//
// Bound: one wave's chain of dependent loads and VALU work, so what a piece
// needs of its source cell is one record, asked for before the board is
// scanned, and its curve run is two bit scans of the track slots (MoveTables).
// From dependent table loads and a cell-by-cell walk of the curves this part went
// from 5,400 to 1,130 cycles of a wave alone on its SIMD (us per fused step:
// u8 32,768 games 738 -> 722, bf16 16,384 666 -> 658, state only 4,096 33.4 -> 32.1).
template <bool REC = true>
__device__ __forceinline__ void legal_body(const State &S, int env, int row, int l, int seat, bool off, const int8_t *cell, uint32_t *bits,
                           uint8_t *rotl, int src, int t, uint64_t *lscr,
                           int32_t *__restrict__ counts, int32_t *__restrict__ mask_words, uint8_t *__restrict__ mask_bool)
{
    const int team = seat & 1;
    uint64_t *srcset = lscr, *edst = lscr + 3;
    const LaneRec T = cM.lane[l];
    const int h = l >> 5, p = l & 31;
    const bool own = !off && p < 30 && (unsigned)src < (unsigned)NC;
    const MoveRec M = cM.rec[own ? src : 0][h];   // cell 0 is off the board: an empty record
    const uint8_t *rot = cT.rotc[seat & 3];   // world compact -> canonical compact of the seat
    const uint8_t q0 = rot[l], q1 = rot[l + 64], q2 = rot[NONB - 1];
    if (l < 3) srcset[l] = 0;
    Boards B;
    env_boards(cell, team, T, B);
    const int sc = (int)(M.meta & 0xFF), ridx = (int)((M.meta >> 8) & 0xFF) - 1, slot = (int)(M.meta >> 24) - 1;
    const bool mov = own && t != T_JUNQI && t != T_DILEI && ((M.meta >> 16) & (CF_ON | CF_SH)) == CF_ON;
    const bool eng = mov && t == T_GONGB;
    uint64_t m0 = 0, m1 = 0, m2 = 0;
    if (mov) {
        const BB m = straight_moves_half(M, eng, B);
        m0 = m.w0; m1 = m.w1; m2 = m.w2;
    }
    {   // curve runs: cells of track slots [ta, tb), from the lanes' prefix sets
        int ta = 0, tb = 0;
        if (mov && !eng && slot >= 0) track_run(slot, h, B, ta, tb);
        m0 |= (uint64_t)(__shfl((long long)T.pre[0], tb) ^ __shfl((long long)T.pre[0], ta));
        m1 |= (uint64_t)(__shfl((long long)T.pre[1], tb) ^ __shfl((long long)T.pre[1], ta));
    }
    m0 |= (uint64_t)__shfl_xor((long long)m0, 32);
    m1 |= (uint64_t)__shfl_xor((long long)m1, 32);
    m2 |= (uint64_t)__shfl_xor((long long)m2, 32);
    // engineers on a rail, three at a time (a seat has at most three)
    uint64_t engs = __ballot(mov && eng && ridx >= 0 && h == 0);
    while (engs) {
        int lanes[3], sr[3], ne = 0;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            lanes[j] = engs ? __builtin_ctzll(engs) : 64;
            ne += engs ? 1 : 0;
            engs &= engs - 1;
            sr[j] = lanes[j] < 64 ? __builtin_amdgcn_readlane(ridx, lanes[j]) : -1;   // uniform lane
        }
        if (l < 9) edst[l] = 0;
        engineers_bb(ne, sr, B.occ, B.ea, edst);
        wave_sync();
#pragma unroll
        for (int j = 0; j < 3; ++j)
            if (p == lanes[j]) { m0 |= edst[3 * j]; m1 |= edst[3 * j + 1]; m2 |= edst[3 * j + 2]; }
        wave_sync();
    }
    const bool lead = mov && h == 0;   // the lane that reports piece p
    const int cnt = __popcll(m0) + __popcll(m1) + __popcll(m2);
    // rank of this piece's source cell among the movable pieces: the movable
    // sources below it in a 129-bit set (compact order is flat order)
    if (lead) atomicOr(reinterpret_cast<unsigned long long *>(&srcset[sc >> 6]), 1ull << (sc & 63));
    rotl[l] = q0; rotl[l + 64] = q1; rotl[NONB - 1] = q2;
    wave_sync();
    int rank = 0;
    if (lead) {
        const int w = sc >> 6;
        rank = __popcll(srcset[w] & ((1ull << (sc & 63)) - 1)) + (w > 0 ? __popcll(srcset[0]) : 0) +
               (w > 1 ? __popcll(srcset[1]) : 0);
    }
    const int nmov = __popcll(__ballot(lead));
    const int total = wave_sum(lead ? cnt : 0);
    if (REC && lead) {
        LegalRec &G = S.lg[env];
        G.src[rank] = (int16_t)src;
        G.mask[rank][0] = m0; G.mask[rank][1] = m1; G.mask[rank][2] = m2;
    }
    // canonical compact mask bits (gpu_rollout.py:1220-1238 layout): the two
    // lanes of a piece take alternate destination bits
    if (mov && (mask_words || mask_bool)) {
        const int cs = rotl[sc] * NONB;
        const uint64_t half = h ? 0xAAAAAAAAAAAAAAAAull : 0x5555555555555555ull;
        const uint64_t w[3] = {m0 & half, m1 & half, m2 & half};
        for (int q = 0; q < 3; ++q) {   // a loop over two words at once, two lookups in flight, took 2,500 cycles for 1,900
            uint64_t x = w[q];
            while (x) {
                const int b = __builtin_ctzll(x) + 64 * q;
                x &= x - 1;
                const int bit = cs + rotl[b];
                atomicOr(&bits[bit >> 5], 1u << (bit & 31));
            }
        }
    }
    if (REC && l == 0) {
        S.lg[env].n = nmov;
        S.lg[env].seat = seat;
        if (counts) counts[env] = total;
    }
    wave_sync();
    if (mask_words)
        for (int w = l; w < JQ_MASK_WORDS; w += 64) mask_words[(size_t)row * JQ_MASK_WORDS + w] = (int32_t)bits[w];
    if (mask_bool) {
        __builtin_amdgcn_s_setprio(0);
        uint8_t *out = mask_bool + (size_t)row * JQ_ACTION_DIM;
        // bytes until the first 16-byte boundary, then whole 16-byte chunks, then the tail
        const int mis = (int)((uintptr_t)out & 15);
        const int head = mis ? 16 - mis : 0;
        for (int i = l; i < head; i += 64) out[i] = (bits[i >> 5] >> (i & 31)) & 1;
        const int nchunks = (JQ_ACTION_DIM - head) / 16;
        for (int q = l; q < nchunks; q += 64) {
            const int i0 = head + q * 16;   // bits i0 .. i0 + 15 (word (i0 >> 5) + 1 <= 520)
            const uint32_t v = __builtin_amdgcn_alignbit(bits[(i0 >> 5) + 1], bits[i0 >> 5], i0 & 31);
            *reinterpret_cast<uint4 *>(out + i0) =
                make_uint4(nib_to_bytes(v), nib_to_bytes(v >> 4), nib_to_bytes(v >> 8), nib_to_bytes(v >> 12));
        }
        for (int i = head + nchunks * 16 + l; i < JQ_ACTION_DIM; i += 64) out[i] = (bits[i >> 5] >> (i & 31)) & 1;
    }
}

// One wave's LDS for the legal sets of a row.
struct LegalLds {
    uint64_t lscr[LSCR_WORDS];
    uint32_t bits[JQ_MASK_WORDS_PAD];
    alignas(4) int8_t cell[CELL_STRIDE];
    uint8_t rotl[NONB + 3];   // world compact -> canonical compact of the acting seat
};

// Legal sets of row `row` by one wave (lane l). HIST: history row flat[row]
// (S = history_state) for seat acting[row], its masks as row `row` of the
// minibatch; flat values outside [0, S.n) have no legal action. No counts or
// legal records then.
template <bool HIST>
__device__ __forceinline__ void legal_row(const State &S, int row, int l, LegalLds &L, const int8_t *__restrict__ acting,
                                          int32_t *__restrict__ counts, int32_t *__restrict__ mask_words,
                                          uint8_t *__restrict__ mask_bool, const int64_t *__restrict__ flat)
{
    int env = row;
    bool stored = true;
    if constexpr (HIST) {
        const int64_t f = flat[row];
        stored = f >= 0 && f < (int64_t)S.n;
        env = stored ? (int)f : 0;
    }
    const EnvRec &E = S.env[env];
    const int seat = acting ? acting[row] : E.turn;
    const bool off = !stored || E.term || seat < 0 || seat > 3 || ((E.sdead >> (seat & 3)) & 1);
    uint32_t c0, c1;
    board_load(S, env, l, c0, c1);
    int src = -1, t = -1;   // the seat's piece l & 31
    if (!off && (l & 31) < 30) {
        const PieceRec r = piece_rec(*reinterpret_cast<const uint4 *>(&S.piece[pc_idx(env, seat * 30 + (l & 31))]));
        src = r.pos;
        t = r.ptype;
    }
    // wave issue priority 2 through the legal pass, 0 for the bool rows'
    // stores (legal_body lowers it): a wave still computing gets issue slots
    // ahead of the waves that are storing rows (drop-in step at 32,768 games:
    // 2.486 -> 2.474 ms)
    __builtin_amdgcn_s_setprio(2);
    for (int w = l; w < JQ_MASK_WORDS_PAD; w += 64) L.bits[w] = 0;
    board_stage(L.cell, l, c0, c1);
    wave_sync();
    legal_body<!HIST>(S, env, row, l, seat, off, L.cell, L.bits, L.rotl, src, t, L.lscr, counts, mask_words, mask_bool);
}

template <bool HIST = false>
__global__ __launch_bounds__(64) void k_legal(State S, const int8_t *__restrict__ acting,
                                              int32_t *__restrict__ counts, int32_t *__restrict__ mask_words,
                                              uint8_t *__restrict__ mask_bool,
                                              const int64_t *__restrict__ flat = nullptr)
{
    __shared__ LegalLds L;
    if (!HIST && (int)blockIdx.x >= S.n) return;
    legal_row<HIST>(S, blockIdx.x, threadIdx.x, L, acting, counts, mask_words, mask_bool, flat);
}

// Exclusive scan of counts into offsets (N+1); one 1024-thread block walks the
// array in tiles of 32768 (one tile at the usual batch sizes). Wave w scans the
// tile's 2048 counts from 2048 w on: lane l holds the four counts at 4 (64 k + l)
// for k < 8, so every 16-byte load and store of the wave covers one contiguous
// 1 KB; eight wave scans give the running sums, the 16 wave totals are scanned
// through LDS, and a carry runs between tiles. The carry is 64-bit: a total
// beyond INT32_MAX (offsets are int32, as the reference's) writes offsets[n] =
// -1, which the host reads as "does not fit" before any id is emitted.
constexpr int SCAN_THREADS = 1024, SCAN_CHUNKS = 8, SCAN_TILE = SCAN_THREADS * 4 * SCAN_CHUNKS;
__global__ __launch_bounds__(SCAN_THREADS) void k_scan(const int32_t *__restrict__ counts, int32_t *__restrict__ offsets,
                                                      int n)
{
    __shared__ int32_t wsum[SCAN_THREADS / 64];
    __shared__ int32_t tile_total;
    const int t = threadIdx.x, lane = t & 63, w = t >> 6;
    const bool vec = ((reinterpret_cast<uintptr_t>(counts) | reinterpret_cast<uintptr_t>(offsets)) & 15) == 0;
    int64_t carry = 0;
    for (int base = 0; base < n; base += SCAN_TILE) {
        const int seg = base + w * 64 * 4 * SCAN_CHUNKS;
        int4 v[SCAN_CHUNKS];
        int excl[SCAN_CHUNKS];
        int segsum = 0;
#pragma unroll
        for (int k = 0; k < SCAN_CHUNKS; ++k) {
            const int i = seg + 4 * (64 * k + lane);
            if (vec && i + 4 <= n) {
                v[k] = *reinterpret_cast<const int4 *>(counts + i);
            } else {
                v[k].x = i < n ? counts[i] : 0;
                v[k].y = i + 1 < n ? counts[i + 1] : 0;
                v[k].z = i + 2 < n ? counts[i + 2] : 0;
                v[k].w = i + 3 < n ? counts[i + 3] : 0;
            }
        }
#pragma unroll
        for (int k = 0; k < SCAN_CHUNKS; ++k) {
            const int s4 = v[k].x + v[k].y + v[k].z + v[k].w;
            int incl = s4;
            for (int o = 1; o < 64; o <<= 1) { const int u = __shfl_up(incl, o); if (lane >= o) incl += u; }
            excl[k] = segsum + incl - s4;
            segsum += __builtin_amdgcn_readlane(incl, 63);
        }
        if (lane == 0) wsum[w] = segsum;
        __syncthreads();
        if (w == 0) {
            const int x = lane < SCAN_THREADS / 64 ? wsum[lane] : 0;
            int y = x;
            for (int o = 1; o < SCAN_THREADS / 64; o <<= 1) { const int u = __shfl_up(y, o); if (lane >= o) y += u; }
            if (lane < SCAN_THREADS / 64) wsum[lane] = y - x;   // exclusive wave prefix
            if (lane == SCAN_THREADS / 64 - 1) tile_total = y;
        }
        __syncthreads();
        const int64_t wbase = carry + wsum[w];   // a tile's sums fit int: 32,768 x JQ_MAX_LEGAL < 2^31
#pragma unroll
        for (int k = 0; k < SCAN_CHUNKS; ++k) {
            const int i = seg + 4 * (64 * k + lane);
            int4 o;
            o.x = (int)(wbase + excl[k]);
            o.y = o.x + v[k].x;
            o.z = o.y + v[k].y;
            o.w = o.z + v[k].z;
            if (vec && i + 4 <= n) {
                *reinterpret_cast<int4 *>(offsets + i) = o;
            } else {
                if (i < n) offsets[i] = o.x;
                if (i + 1 < n) offsets[i + 1] = o.y;
                if (i + 2 < n) offsets[i + 2] = o.z;
                if (i + 3 < n) offsets[i + 3] = o.w;
            }
        }
        carry += tile_total;
        __syncthreads();
    }
    if (t == 0) offsets[n] = carry > (int64_t)INT32_MAX ? -1 : (int)carry;
}

// Position of the k-th set bit (k < popcount) of a 64-bit word.
__device__ __forceinline__ int select64(uint64_t x, int k)
{
    int pos = 0;
#pragma unroll
    for (int width = 32; width >= 1; width >>= 1) {
        const int c = __popcll(x & ((1ull << width) - 1ull));
        if (k >= c) { k -= c; x >>= width; pos += width; }
    }
    return pos;
}

// One env's piece of the CSR for its group of W = 32 or 64 lanes: pieces in
// ascending source order, each piece's destinations ascending (compact order =
// flat order). A seat has at most 30 movable pieces, so lane p of the group
// holds piece p.
struct EmitPiece {
    uint64_t m0, m1, m2;   // destinations (none past the last piece)
    int src, cnt, seat, n;
};

// Lane p's piece of env (none when !live). The record's fields do not wait for
// its piece count: what lies past it is dropped.
__device__ __forceinline__ EmitPiece emit_load(const State &S, int env, int p, bool live)
{
    EmitPiece e = {};
    if (!live) return e;
    const LegalRec &G = S.lg[env];
    const int q = p < 30 ? p : 0;
    const int src = G.src[q];
    const uint64_t m0 = G.mask[q][0], m1 = G.mask[q][1], m2 = G.mask[q][2];
    e.n = min((int)G.n, 30);
    e.seat = G.seat & 3;
    if (p < e.n) {
        e.src = src;
        e.m0 = m0; e.m1 = m1; e.m2 = m2;
        e.cnt = __popcll(m0) + __popcll(m1) + __popcll(m2);
    }
    return e;
}

// Write the ids of each group's env at base + 0, 1, ...: lane j of a group of W
// produces ids j, j + W, ...: it finds its piece from the running counts (start,
// the group's 33 LDS words), the destination by selecting a bit of that piece's
// mask, and maps it to a flat cell through an LDS copy of the compact table.
// MASK: each id also sets its canonical bit in the group's LDS mask words (csrc:
// the piece's canonical source, rot: world -> canonical compact).
template <int W, bool MASK>
__device__ __forceinline__ void emit_ids(const EmitPiece &e, int p, const int16_t *c2f, int32_t *start, int64_t base,
                                         int32_t *__restrict__ values, int64_t cap, int csrc = 0,
                                         const uint8_t *rot = nullptr, uint32_t *mbits = nullptr)
{
    int incl = e.cnt;
    for (int o = 1; o < 32; o <<= 1) { const int v = __shfl_up(incl, o, W); if (p >= o) incl += v; }
    if (p < e.n) start[p] = incl - e.cnt;
    const int total = __shfl(incl, 31, W);
    if (p == 0) start[e.n] = total;
    wave_sync();
    // uniform trip count (the larger group's total): every lane takes the shuffles
    const int trips = max(__builtin_amdgcn_readlane(total, 0), __builtin_amdgcn_readlane(total, W == 32 ? 32 : 0));
    for (int b = 0; b < trips; b += W) {
        const int i = b + p;
        int j = 0;   // piece of id i: the last piece whose start is <= i
        for (int step = 16; step >= 1; step >>= 1)
            if (j + step < e.n && start[j + step] <= i) j += step;
        const uint64_t w0 = __shfl(e.m0, j, W), w1 = __shfl(e.m1, j, W), w2 = __shfl(e.m2, j, W);
        const int s = __shfl(e.src, j, W), cs = MASK ? __shfl(csrc, j, W) : 0;
        if (i < total) {
            const int k = i - start[j];
            const int c0 = __popcll(w0), c1 = __popcll(w1);
            const int c = k < c0 ? select64(w0, k)
                                 : k < c0 + c1 ? 64 + select64(w1, k - c0) : 128 + select64(w2, k - c0 - c1);
            if (base >= 0 && base + i < cap) values[base + i] = s * NC + c2f[c];
            if (MASK) {   // canonical bit (rotated source) * 129 + (rotated destination)
                const int bit = cs * NONB + rot[c];
                atomicOr(&mbits[bit >> 5], 1u << (bit & 31));
            }
        }
    }
}

// The ids of every env at its scanned offset (k_scan), two envs per wave: half h
// (lanes 32h .. 32h + 31) takes env 2 * block + h. With mask_words the canonical
// mask of each env is built too, in LDS.
__global__ __launch_bounds__(64) void k_emit(State S, const int32_t *__restrict__ offsets, int32_t *__restrict__ values,
                                             int64_t cap, int32_t *__restrict__ mask_words)
{
    const int l = threadIdx.x, h = l >> 5, p = l & 31;
    const int env = 2 * (int)blockIdx.x + h;
    const bool live = env < S.n;
    __shared__ int16_t c2f[NONB + 3];
    __shared__ int32_t start[2][33];   // per half: first id of each piece, start[n] = total
    __shared__ uint32_t mbits[2][JQ_MASK_WORDS_PAD];
    __shared__ uint8_t rot[2][NONB + 3];   // world compact -> canonical compact of the env's acting seat
    for (int c = l; c < NONB; c += 64) c2f[c] = cT.c2f[c];
    const EmitPiece e = emit_load(S, env, p, live);
    const int64_t base = live ? offsets[env] : 0;
    if (!mask_words) {
        emit_ids<32, false>(e, p, c2f, start[h], base, values, cap);
        return;
    }
    for (int w = p; w < JQ_MASK_WORDS_PAD; w += 32) mbits[h][w] = 0;
    for (int c = p; c < NONB; c += 32) rot[h][c] = cT.rotc[e.seat][c];
    const int csrc = cT.canc[e.seat][e.src];
    emit_ids<32, true>(e, p, c2f, start[h], base, values, cap, csrc, rot[h], mbits[h]);
    wave_sync();
    if (live)
        for (int w = p; w < JQ_MASK_WORDS; w += 32)
            stream_store(mask_words + (size_t)env * JQ_MASK_WORDS + w, (int32_t)mbits[h][w]);
}

// Scan and emit in one pass of CSR_THREADS-thread blocks: a block sums the
// counts of all envs before its own, writes its envs' offsets and then their
// ids, one env per wave and pass. For batches whose ids always fit the buffer
// (no total to read back).
// Why: k_scan is one block, 6.2 us however few the envs, and k_emit waits for
// it. The blocks read the counts again and again (n * n / (16 * passes) words in
// all, from L2), so larger batches take more envs per block.
constexpr int CSR_THREADS = 512, CSR_WAVES = CSR_THREADS / 64, CSR_MOST_PASSES = 4;
struct CsrArgs {
    const int32_t *counts;
    int32_t *offsets, *values;
    int64_t cap;
    int passes;   // envs per wave
    int blocks;   // of a launch: 0 = no CSR pass in it
};

// The legal masks of a minibatch of history rows, as blocks of the launch that
// observes them (either output may be null).
struct MaskArgs {
    int32_t *words;
    uint8_t *bytes;
    int blocks;   // 0 = no masks in the launch
};

struct CsrLds {
    int32_t start[CSR_WAVES][33];
    int32_t wsum[CSR_WAVES];
    int16_t c2f[NONB + 3];
};

__device__ __forceinline__ void csr_block(const State &S, const CsrArgs &A, int block, CsrLds &L)
{
    const int t = threadIdx.x, l = t & 63, w = __builtin_amdgcn_readfirstlane(t >> 6);
    const int envs = CSR_WAVES * A.passes, e0 = block * envs;   // wave w: envs e0 + w, e0 + w + 8, ...
    EmitPiece e = emit_load(S, e0 + w, l, e0 + w < S.n);
    const int own = l < envs && e0 + l < S.n ? A.counts[e0 + l] : 0;   // the block's counts, in every wave
    int sum = 0;
    if ((reinterpret_cast<uintptr_t>(A.counts) & 15) == 0) {
        const int4 *c4 = reinterpret_cast<const int4 *>(A.counts);
        for (int i = t; i < e0 / 4; i += CSR_THREADS) {
            const int4 v = c4[i];
            sum += (v.x + v.y) + (v.z + v.w);
        }
    } else {
        for (int i = t; i < e0; i += CSR_THREADS) sum += A.counts[i];
    }
    sum = wave_sum(sum);
    if (l == 0) L.wsum[w] = sum;
    if (t < NONB) L.c2f[t] = cT.c2f[t];
    lds_barrier();
    int before = 0;
#pragma unroll
    for (int k = 0; k < CSR_WAVES; ++k) before += L.wsum[k];
    int incl = own;
    for (int o = 1; o < CSR_WAVES * CSR_MOST_PASSES; o <<= 1) { const int v = __shfl_up(incl, o); if (l >= o) incl += v; }
    const int first = before + incl - own;   // lane j: offset of env e0 + j
    if (w == 0 && l < envs && e0 + l < S.n) {
        A.offsets[e0 + l] = first;
        if (e0 + l == S.n - 1) A.offsets[S.n] = first + own;
    }
    for (int k = 0; k < A.passes; ++k) {
        if (k) {
            const int env = e0 + w + CSR_WAVES * k;
            e = emit_load(S, env, l, env < S.n);
            wave_sync();   // the last pass's reads of `start` are done
        }
        const int base = __builtin_amdgcn_readlane(first, w + CSR_WAVES * k);
        emit_ids<64, false>(e, l, L.c2f, L.start[w], base, A.values, A.cap);
    }
}

__global__ __launch_bounds__(CSR_THREADS) void k_csr(State S, CsrArgs A)
{
    __shared__ CsrLds L;
    csr_block(S, A, blockIdx.x, L);
}

// ------------------------------------------------------------------ slot mask
// Per-piece 80-slot legal mask (game_state.cu:1964-2197) from the legal sets
// k_legal left in S.lg. Slots 0-3 are the road steps in table order, 4-7 the
// camp diagonals, 8 + dir*12 + k the k-th cell of a non-engineer's straight
// rail run (road neighbours of the source excepted, they sit in 0-3). The
// reference packs curve-rail destinations (56..67) and an engineer's rail
// destinations (8..79) contiguously in its BFS order, so those sections are a
// run of ones as long as the destinations the earlier slots leave over.
constexpr int JQ_SLOTS = 80;
constexpr int JQ_SLOT_ROW = NP * JQ_SLOTS;   // bytes per env

__device__ __forceinline__ void set_run(uint64_t &lo, uint32_t &hi, int a, int len)
{   // bits [a, a + len) of the 80-bit slot set, a + len <= 80
    if (len <= 0) return;
    const int e = a + len;
    if (a < 64) {
        const int n = (e < 64 ? e : 64) - a;
        lo |= (n == 64 ? ~0ull : ((1ull << n) - 1)) << a;
    }
    if (e > 64) {
        const int ha = a > 64 ? a - 64 : 0;
        hi |= ((1u << (e - 64 - ha)) - 1) << ha;
    }
}

__device__ __forceinline__ uint32_t nibble_bytes(uint32_t nib)
{   // 4 bits -> 4 bytes of 0 / 1
    return (nib * 0x00204081u) & 0x01010101u;
}

__global__ __launch_bounds__(64) void k_slots(State S, uint8_t *__restrict__ out)
{
    const int env = blockIdx.x, l = threadIdx.x;
    if (env >= S.n) return;
    __shared__ uint4 rows[30][JQ_SLOTS / 16];   // the acting seat's 30 piece rows
    const LegalRec &G = S.lg[env];
    const int n = G.n, seat = G.seat;
    for (int q = l; q < 30 * (JQ_SLOTS / 16); q += 64) rows[q / 5][q % 5] = make_uint4(0, 0, 0, 0);
    __syncthreads();
    const int src = l < n ? G.src[l] : -1;
    const int pid = (unsigned)src < (unsigned)NC ? S.cell[(size_t)env * CELL_STRIDE + src] : -1;
    if (l < n && (unsigned)(pid - seat * 30) < 30u) {   // a consistent state always passes
        const BB M{G.mask[l][0], G.mask[l][1], G.mask[l][2]};
        const bool eng = S.piece[pc_idx(env, pid)].ptype == T_GONGB;
        uint64_t lo = 0;
        uint32_t hi = 0;
        int a[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            a[k] = cT.adj[src][k];
            if (a[k] >= 0 && bb_has(M, cT.f2c[a[k]])) lo |= 1ull << k;
            const int d = cT.diag[src][k];
            if (d >= 0 && bb_has(M, cT.f2c[d])) lo |= 1ull << (4 + k);
        }
        const int total = __popcll(M.w0) + __popcll(M.w1) + __popcll(M.w2);
        const int r = cT.railidx[src];
        if (r >= 0 && !eng) {
            for (int d = 0; d < 4; ++d)
                for (int k = 0; k < cT.raylen[r][d]; ++k) {
                    const int f = cT.rays[r][d][k];
                    if (f != a[0] && f != a[1] && f != a[2] && f != a[3] && bb_has(M, cT.f2c[f]))
                        lo |= 1ull << (8 + d * 12 + k);
                }
            const int rest = total - __popcll(lo);
            set_run(lo, hi, 56, rest < 12 ? rest : 12);
        } else if (r >= 0) {
            const int rest = total - __popcll(lo);
            set_run(lo, hi, 8, rest < 72 ? rest : 72);
        }
        uint4 *row = rows[pid - seat * 30];
#pragma unroll
        for (int j = 0; j < JQ_SLOTS / 16; ++j) {
            const uint32_t b = j < 4 ? (uint32_t)(lo >> (16 * j)) & 0xFFFFu : hi & 0xFFFFu;
            row[j] = make_uint4(nibble_bytes(b & 0xF), nibble_bytes((b >> 4) & 0xF),
                                nibble_bytes((b >> 8) & 0xF), nibble_bytes(b >> 12));
        }
    }
    __syncthreads();
    uint4 *dst = reinterpret_cast<uint4 *>(out + (size_t)env * JQ_SLOT_ROW);
    for (int q = l; q < JQ_SLOT_ROW / 16; q += 64) {
        const int p = q / 5 - seat * 30;
        dst[q] = (n > 0 && (unsigned)p < 30u) ? rows[p][q % 5] : make_uint4(0, 0, 0, 0);
    }
}

// ------------------------------------------------------------------ sampler
__device__ __forceinline__ uint32_t philox4x32_10(uint32_t c0, uint32_t c1, uint32_t c2, uint32_t c3,
                                                 uint32_t k0, uint32_t k1)
{   // Philox4x32-10 (Salmon et al., SC'11); returns the first output word
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint64_t p0 = (uint64_t)0xD2511F53u * c0, p1 = (uint64_t)0xCD9E8D57u * c2;
        const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0, hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
        c0 = hi1 ^ c1 ^ k0; c1 = lo1; c2 = hi0 ^ c3 ^ k1; c3 = lo0;
        k0 += 0x9E3779B9u; k1 += 0xBB67AE85u;
    }
    return c0;
}

// Uniform pick from env's CSR row of c ids at offset off: Philox4x32-10 word 0
// of counter (env, ply lo, ply hi, 0) under key (seed lo, seed hi), scaled to
// the count; -1 for an empty row or one that does not lie inside the values
// buffer.
__device__ __forceinline__ int32_t uniform_pick(int env, int c, int64_t off, const int32_t *__restrict__ values,
                                                int64_t cap, uint64_t seed, uint64_t ply)
{
    if (c <= 0 || off < 0 || off + c > cap) return -1;
    const uint32_t u = philox4x32_10((uint32_t)env, (uint32_t)ply, (uint32_t)(ply >> 32), 0u,
                                     (uint32_t)seed, (uint32_t)(seed >> 32));
    return values[off + (int)(((uint64_t)u * (uint64_t)c) >> 32)];
}

// One env per thread.
__global__ void k_sample(int n, const int32_t *__restrict__ counts, const int32_t *__restrict__ offsets,
                         const int32_t *__restrict__ values, int64_t cap, uint64_t seed, uint64_t ply,
                         int32_t *__restrict__ out)
{
    const int env = blockIdx.x * blockDim.x + threadIdx.x;
    if (env >= n) return;
    out[env] = uniform_pick(env, counts[env], offsets[env], values, cap, seed, ply);
}

// Masked-logit pick by env's wave (lane l): the legal ids of the CSR row, lane
// j taking ids j, j + 64, ...; each id's canonical id c under `seat` draws
// u_c = Philox word 0 of counter (env, ply lo, ply hi, 1 + c). The N(0,1) logit
// Phi^-1((u_c + 1/2) / 2^32) is increasing in u_c, so the argmax over the row is
// the largest u_c, ties to the smallest c: one 64-bit key (u_c, ~c) per lane,
// maximised across the wave. Returns the world id (wave-uniform, -1 for an
// empty or out-of-buffer row) and its canonical id in `canon`.
// `c` and `off` are the env's CSR count and offset (wave-uniform).
__device__ __forceinline__ int32_t sample_logits_wave(int env, int l, int seat, int c, int64_t off,
                                                      const int32_t *__restrict__ values, int64_t cap, uint64_t seed,
                                                      uint64_t ply, int &canon)
{
    canon = -1;
    if (c <= 0 || seat < 0 || seat > 3) return -1;
    if (off < 0 || off + c > cap) return -1;
    uint64_t best = 0;
    int32_t bw = -1;
    for (int j = l; j < c; j += 64) {
        const int32_t w = values[off + j];
        const int src = w / NC, dst = w - src * NC;
        const int cc = (int)cT.canc[seat][src] * NONB + (int)cT.canc[seat][dst];
        const uint32_t u = philox4x32_10((uint32_t)env, (uint32_t)ply, (uint32_t)(ply >> 32), (uint32_t)(1 + cc),
                                         (uint32_t)seed, (uint32_t)(seed >> 32));
        const uint64_t key = ((uint64_t)u << 32) | (uint32_t)~(uint32_t)cc;   // > 0 for every real id
        if (key > best) { best = key; bw = w; }
    }
    const uint64_t m = wave_max(best);
    const uint64_t who = __ballot(best == m && bw >= 0);
    const int src_lane = who ? __builtin_ctzll(who) : 0;
    canon = (int)~(uint32_t)(m & 0xFFFFFFFFu);
    return __builtin_amdgcn_readlane(bw, src_lane);   // src_lane is wave-uniform
}

__global__ __launch_bounds__(64) void k_sample_logits(State S, const int8_t *__restrict__ acting,
                                                      const int32_t *__restrict__ counts,
                                                      const int32_t *__restrict__ offsets,
                                                      const int32_t *__restrict__ values, int64_t cap, uint64_t seed,
                                                      uint64_t ply, int32_t *__restrict__ out,
                                                      int32_t *__restrict__ canon_out)
{
    const int env = blockIdx.x, l = threadIdx.x;
    if (env >= S.n) return;
    const int seat = acting ? acting[env] : S.env[env].turn;
    int32_t c = uniform_word_raw(counts + env), o = uniform_word_raw(offsets + env);
    pin_word(c);
    pin_word(o);
    int cc;
    const int32_t a = sample_logits_wave(env, l, seat, c, o, values, cap, seed, ply, cc);
    if (l == 0) {
        out[env] = a;
        if (canon_out) canon_out[env] = a >= 0 ? cc : -1;
    }
}

// One env-step's state work by one wave per env: the action (given, or the
// Philox pick of k_sample from the env's previous CSR row, read before this
// wave overwrites the env's count), the ply (k_step), the restart
// of a finished game from the setup pool (k_reset_terminated, if do_reset) and
// the legal sets of the next acting seat (k_legal with the current
// turn), on the board the wave keeps in LDS, with no global round trip between
// the three.
// One wave's board while it steps its env: the LDS that step_env, init_env and
// legal_body work on.
struct EnvLds {
    alignas(16) uint32_t bits[JQ_MASK_WORDS_PAD];
    StepRes res;   // the step's reports, parked here across the legal pass
    uint64_t lscr[LSCR_WORDS];
    int16_t pos[PID_STRIDE];
    int8_t ptype[PID_STRIDE];
    alignas(4) int8_t cell[CELL_STRIDE];
    uint8_t rotl[NONB + 3];
};

// Inputs of one env-step beyond the state: the action source (`actions`, else a
// Philox pick from the env's previous CSR row `offsets` / `values` with
// `counts`), the pool restart and the outputs.
struct EnvStepArgs {
    const int32_t *actions; int sampler; uint64_t sample_seed, ply; const int32_t *offsets, *values;
    int64_t values_cap; int32_t *actions_out; StepOut O; int do_reset; int64_t reset_seed;
    int32_t *counts, *mask_words;
};

// The env-step of `env` by one wave (lane l): sample its action, apply the ply,
// restart the env from the setup pool if it ended, then the next seat's legal
// sets and canonical mask, all on the board the wave keeps in E. It synchronises
// only its own wave (wave_sync), so it never waits on other waves of a block.
__device__ __forceinline__ void env_step_wave(const State &S, int env, int l, const EnvStepArgs &A, EnvLds &E)
{
    StepLoad ld;   // the ply's first loads go out before the sampler's
    step_load(S, env, l, ld);
    // the env record and the CSR count and offset in one batch of scalar loads:
    // one wait, then the sampler's only dependent load is its row of ids
    const int32_t *ew = reinterpret_cast<const int32_t *>(S.env + env);
    int32_t v[10];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = uniform_word_raw(ew + k);
    const bool sampled = !A.actions;
    v[8] = sampled ? uniform_word_raw(A.counts + env) : 0;
    v[9] = sampled ? uniform_word_raw(A.offsets + env) : 0;
#pragma unroll
    for (int k = 0; k < 10; ++k) pin_word(v[k]);
    EnvRec E0;
    __builtin_memcpy(&E0, v, sizeof E0);
    int32_t a;
    if (A.actions) {
        a = A.actions[env];
    } else if (A.sampler == 1) {
        int cc;
        a = sample_logits_wave(env, l, E0.turn, v[8], v[9], A.values, A.values_cap, A.sample_seed, A.ply, cc);
    } else {
        a = uniform_pick(env, v[8], v[9], A.values, A.values_cap, A.sample_seed, A.ply);
    }
    if (A.actions_out && l == 0) A.actions_out[env] = a;
    TurnAfter nx;
    {
        StepRes res;
        step_env(S, env, l, a, nullptr, 0, res, E.cell, E.pos, E.ptype, nx, &ld, &E0);
        if (l == 0) E.res = res;
    }
    wave_sync();
    if (A.do_reset && S.pool_size > 0 && nx.term) {
        init_env(S, env, S.pool + (size_t)reset_pool_index(env, A.reset_seed, S.pool_size) * NP, E.cell, E.pos,
                 E.ptype);
        nx.turn = 0; nx.term = false; nx.sdead = 0;
    }
    const int seat = nx.turn;
    const bool off = nx.term || seat < 0 || seat > 3 || ((nx.sdead >> (seat & 3)) & 1);
    if (A.mask_words)
        for (int w = l; w < JQ_MASK_WORDS_PAD; w += 64) E.bits[w] = 0;
    wave_sync();
    const int mine = !off && (l & 31) < 30 ? seat * 30 + (l & 31) : -1;   // the next seat's piece of this lane
    legal_body(S, env, env, l, seat, off, E.cell, E.bits, E.rotl, mine >= 0 ? E.pos[mine] : -1,
               mine >= 0 ? E.ptype[mine] : -1, E.lscr, A.counts, A.mask_words, nullptr);
    if (l == 0) write_step_res(A.O, env, E.res);   // the step's reports go out last
}

__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(7, 8))) void k_env_step(State S, EnvStepArgs A)
{
    const int env = blockIdx.x;
    if (env >= S.n) return;
    __shared__ EnvLds E;
    env_step_wave(S, env, threadIdx.x, A, E);
}


}  // namespace jq
