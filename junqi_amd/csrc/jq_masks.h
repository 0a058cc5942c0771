// Dense bool masks <-> per-row id lists, for rollout buffers that keep the
// legal support as ids (junqi_rl/training/rollout_gpu.py:119-198).
//
// Included into jq_lib.hip's translation unit.
#pragma once

namespace jq {

// Nonzero-byte bits of a 16-byte word (bit k = byte k != 0).
__device__ __forceinline__ uint32_t nz_bytes(uint4 v)
{
    uint32_t m = 0;
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        // bit 7 of each nonzero byte (no carry leaves a byte), then the four
        // bits side by side: the multiply puts byte k's bit at 21 + k
        const uint32_t t = (((w[i] & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | w[i]) & 0x80808080u;
        m |= (((t >> 7) * 0x00204081u >> 21) & 0xFu) << (4 * i);
    }
    return m;
}

// Walk one mask row [base, base + d) in column order, one wave: the bytes up
// to the first 16-byte boundary, whole 16-byte words (64 per step, MASK_AHEAD
// steps' loads in flight), then the tail bytes. f(col, nzbits, lane_byte) is
// called by every lane for its piece of each step in which any lane has a
// nonzero byte; lane_byte >= 0 marks a piece of one byte.
constexpr int MASK_AHEAD = 9;   // two rounds for the 1,040 words of a 16,641-byte row
template <class F>
__device__ __forceinline__ void mask_row_walk(const uint8_t *base, int d, F &&f)
{
    const int l = threadIdx.x & 63;
    const uintptr_t b0 = reinterpret_cast<uintptr_t>(base);
    const int head = (int)(min((uintptr_t)d, ((b0 + 15) & ~(uintptr_t)15) - b0));
    const int body = (d - head) / 16;
    const int t0 = head + 16 * body, tail = d - t0;
    // the row's ends (at most 15 bytes each), one lane per byte
    const bool h_on = l < head && base[l] != 0, t_on = l < tail && base[t0 + l] != 0;
    if (__ballot(h_on)) f(0, h_on ? 1u << l : 0u, l);
    const uint4 *w = reinterpret_cast<const uint4 *>(base + head);
    for (int q0 = 0; q0 < body; q0 += 64 * MASK_AHEAD) {
        uint4 v[MASK_AHEAD];
#pragma unroll
        for (int k = 0; k < MASK_AHEAD; ++k) {
            const int q = q0 + 64 * k + l;
            v[k] = q < body ? w[q] : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int k = 0; k < MASK_AHEAD; ++k) {
            if (!__ballot((v[k].x | v[k].y | v[k].z | v[k].w) != 0)) continue;   // most steps of a legal mask
            f(head + 16 * (q0 + 64 * k + l), nz_bytes(v[k]), -1);
        }
    }
    if (__ballot(t_on)) f(t0, t_on ? 1u << l : 0u, l);
}

__device__ __forceinline__ int wave_excl(int v, int &total)
{
    const int l = threadIdx.x & 63;
    int incl = v;
    for (int o = 1; o < 64; o <<= 1) { const int u = __shfl_up(incl, o); if (l >= o) incl += u; }
    total = __builtin_amdgcn_readlane(incl, 63);
    return incl - v;
}

// counts[r] = nonzero bytes of row r. One wave per row.
__global__ __launch_bounds__(64) void k_mask_count(const uint8_t *__restrict__ mask, int n, int d,
                                                   int32_t *__restrict__ counts)
{
    const int r = blockIdx.x;
    if (r >= n) return;
    int c = 0;
    mask_row_walk(mask + (size_t)r * d, d, [&](int, uint32_t m, int) { c += __popc(m); });
    c = wave_sum(c);
    if ((threadIdx.x & 63) == 0) counts[r] = c;
}

// The nonzero columns of one row in order into out[0 .. k_max) (those past k_max
// are dropped), the rest of it 0; returns how many the row has. One wave.
__device__ __forceinline__ int row_to_ids(const uint8_t *row, int d, int k_max, int32_t *__restrict__ out)
{
    int run = 0;
    mask_row_walk(row, d, [&](int col0, uint32_t m, int lane_byte) {
        int tot;
        int at = run + wave_excl(__popc(m), tot);
        for (uint32_t x = m; x; x &= x - 1, ++at)
            // single-byte pieces put the lane's bit at its lane index
            if (at < k_max) out[at] = col0 + (lane_byte >= 0 ? lane_byte : __builtin_ctz(x));
        run += tot;
    });
    for (int j = run + (int)(threadIdx.x & 63); j < k_max; j += 64) out[j] = 0;
    return run;
}

// ids[r] = the nonzero columns of row r (row_to_ids), counts[r] (may be null)
// how many there are. One wave per row. Bound: HBM read of the masks (8,192 rows
// of 16,641 bytes in 28 us, 4.9 TB/s): a row's words are asked for in two
// rounds, and a step of 1 KB without a nonzero byte costs one ballot. Rounds of
// 5 or 17 steps, or 4 or 8 rows per block: all within 1 us.
__global__ __launch_bounds__(64) void k_mask_to_ids(const uint8_t *__restrict__ mask, int n, int d, int k_max,
                                                    int32_t *__restrict__ ids, int32_t *__restrict__ counts)
{
    const int r = blockIdx.x;
    if (r >= n) return;
    const int run = row_to_ids(mask + (size_t)r * d, d, k_max, ids + (size_t)r * k_max);
    if (counts && (threadIdx.x & 63) == 0) counts[r] = run;
}

// Publish encoded rows if every count fits: most[0] = the largest of wc[0 .. n);
// when it is at most k_max, ids <- wids (n * k_max) and counts <- wc, else both
// stay as they are. Each block finds the largest count itself (4 n bytes from
// L2, 32 KB at 8,192 rows), so the masks are read once and the host is asked
// nothing in between: an
// encode was a count of the masks (23 us at 8,192 rows), a test on the host and
// a second pass over them (27 us); it is now 28 + 6 us.
constexpr int MASK_COMMIT_BLOCKS = 512, MASK_COMMIT_THREADS = 512;
__global__ __launch_bounds__(MASK_COMMIT_THREADS) void k_mask_commit(const int32_t *__restrict__ wids, const int32_t *__restrict__ wc,
                                                     int n, int k_max, int32_t *__restrict__ ids,
                                                     int32_t *__restrict__ counts, int32_t *__restrict__ most)
{
    __shared__ int32_t part[MASK_COMMIT_THREADS / 64];
    const int t = threadIdx.x;
    int m = 0;
    const int4 *w4 = reinterpret_cast<const int4 *>(wc);   // 16-byte aligned scratch
    for (int i = t; i < n / 4; i += MASK_COMMIT_THREADS) {
        const int4 v = w4[i];
        m = max(max(m, max(v.x, v.y)), max(v.z, v.w));
    }
    for (int i = n / 4 * 4 + t; i < n; i += MASK_COMMIT_THREADS) m = max(m, wc[i]);
    for (int o = 32; o >= 1; o >>= 1) m = max(m, __shfl_xor(m, o));
    if ((t & 63) == 0) part[t >> 6] = m;
    __syncthreads();
    for (int k = 0; k < MASK_COMMIT_THREADS / 64; ++k) m = max(m, part[k]);
    const int64_t i0 = (int64_t)blockIdx.x * MASK_COMMIT_THREADS + t, step = (int64_t)gridDim.x * MASK_COMMIT_THREADS;
    if (i0 == 0) most[0] = m;
    if (m > k_max) return;
    const int64_t total = (int64_t)n * k_max;
    if (((reinterpret_cast<uintptr_t>(wids) | reinterpret_cast<uintptr_t>(ids)) & 15) == 0) {
        for (int64_t i = i0; i < total / 4; i += step)
            reinterpret_cast<int4 *>(ids)[i] = reinterpret_cast<const int4 *>(wids)[i];
        for (int64_t i = total / 4 * 4 + i0; i < total; i += step) ids[i] = wids[i];
    } else {
        for (int64_t i = i0; i < total; i += step) ids[i] = wids[i];
    }
    for (int64_t i = i0; i < n; i += step) counts[i] = wc[i];
}

// out[b] = dense bool row of the id list of row idx[b] (counts[idx[b]] ids of
// ids[idx[b]]); ids outside [0, d) and rows outside [0, rows) contribute
// nothing. One 256-thread block per output row.
__global__ __launch_bounds__(256) void k_ids_to_mask(const int32_t *__restrict__ ids, const int32_t *__restrict__ counts,
                                                     int64_t rows, int k_max, const int64_t *__restrict__ idx, int batch,
                                                     int d, uint8_t *__restrict__ out)
{
    const int b = blockIdx.x, t = threadIdx.x;
    if (b >= batch) return;
    uint8_t *row = out + (size_t)b * d;
    const uintptr_t b0 = reinterpret_cast<uintptr_t>(row);
    const int head = (int)(min((uintptr_t)d, ((b0 + 15) & ~(uintptr_t)15) - b0));
    const int body = (d - head) / 16;
    for (int i = t; i < head; i += 256) row[i] = 0;
    uint4 *w = reinterpret_cast<uint4 *>(row + head);
    for (int q = t; q < body; q += 256) w[q] = make_uint4(0, 0, 0, 0);
    for (int i = head + 16 * body + t; i < d; i += 256) row[i] = 0;
    __syncthreads();
    const int64_t src = idx[b];
    if (src < 0 || src >= rows) return;
    const int cnt = min(counts[src], k_max);
    for (int j = t; j < cnt; j += 256) {
        const int c = ids[(size_t)src * k_max + j];
        if (c >= 0 && c < d) row[c] = 1;
    }
}

}  // namespace jq
