// cells_device.hpp -- the cells of two or more atoms among a wave's share of
// the sorted slots, for the collide kernels of both numerical forms.
#pragma once

#include "dsmc_device.hpp"

namespace dsmc {

constexpr uint32_t kNoKey = 0xFFFFFFFFu;             // no slot there (keys are below 2^31)

// Cells of two or more atoms that start in a wave's chunk of 64 ITEMS slots,
// in slot order.
template <int ITEMS>
struct WaveCells {
    static constexpr int kMax = kWave * ITEMS / 2;
    uint32_t key[kMax];
    int      end[kMax];     // slot after the cell's last
    short    start[kMax];   // first slot, from the chunk's
    short    heavy[kMax];   // (the collide's) cells run by the whole wave
};

// A chunk's keys: lane l holds slots chunk0 + ITEMS l .. + ITEMS - 1; the key
// before the chunk, and the l-th slot after it (for the end of the last cell).
template <int ITEMS>
struct ChunkKeys {
    static_assert(ITEMS == 2 || ITEMS == 4 || ITEMS == 8, "a lane's keys are whole loads");
    uint32_t k[ITEMS];
    uint32_t before, after;
};

// Orders a wave's LDS writes before its later reads.
__device__ __forceinline__ void wave_lds_fence()
{
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Issues the chunk's loads (those below the capacity n_cap; the buffer is
// 16-byte aligned).  Which slots are alive is not needed yet.
template <int ITEMS>
__device__ __forceinline__ void chunk_load(const uint32_t *__restrict__ key, int n_cap, int chunk0,
                                           ChunkKeys<ITEMS> &c)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int b = chunk0 + lane * ITEMS;
    if (b + ITEMS <= n_cap) {
        if constexpr (ITEMS == 8) {
            const uint4 x = *(const uint4 *)(key + b), y = *(const uint4 *)(key + b + 4);
            c.k[0] = x.x; c.k[1] = x.y; c.k[2] = x.z; c.k[3] = x.w;
            c.k[4] = y.x; c.k[5] = y.y; c.k[6] = y.z; c.k[7] = y.w;
        } else if constexpr (ITEMS == 4) {
            const uint4 x = *(const uint4 *)(key + b);
            c.k[0] = x.x; c.k[1] = x.y; c.k[2] = x.z; c.k[3] = x.w;
        } else {
            const uint2 x = *(const uint2 *)(key + b);
            c.k[0] = x.x; c.k[1] = x.y;
        }
    } else {
#pragma unroll
        for (int j = 0; j < ITEMS; ++j) c.k[j] = b + j < n_cap ? key[b + j] : kNoKey;
    }
    const int a = chunk0 + kWave * ITEMS + lane;
    c.after = a < n_cap ? key[a] : kNoKey;
    c.before = chunk0 > 0 && chunk0 <= n_cap ? key[chunk0 - 1] : kNoKey;
}

// Lists the cells of two or more atoms that start in the chunk (n alive
// slots); returns their number.  k_first: key of the chunk's first slot,
// k_last: of the last cell that starts in it.  Every lane of the wave calls
// it.  A lane's slots are consecutive, so a cell's head, and mostly its
// end, are found in the lane's own registers: five exchanges per wave where
// slots dealt out 64 apart needed five for every eighth of the chunk.  That
// was 40 % of a wave's time in the collide (N = 1e6 in one trap: collide
// 16.3 -> 14.4 us, a group of 128 traps: 21.2 -> 19.6 us).
template <int ITEMS>
__device__ __forceinline__ int wave_list_cells(const uint32_t *__restrict__ key, int n, int chunk0,
                                               ChunkKeys<ITEMS> &c, WaveCells<ITEMS> &L, uint32_t &k_first,
                                               uint32_t &k_last)
{
    const int lane = threadIdx.x & (kWave - 1);
    const int b = chunk0 + lane * ITEMS;
    const int chunk1 = min(n, chunk0 + kWave * ITEMS);
#pragma unroll
    for (int j = 0; j < ITEMS; ++j)
        if (b + j >= n) c.k[j] = kNoKey;
    if (chunk0 + kWave * ITEMS + lane >= n) c.after = kNoKey;
    uint32_t kp = __shfl_up(c.k[ITEMS - 1], 1, kWave), kn = __shfl_down(c.k[0], 1, kWave);
    const uint32_t k_after = __builtin_amdgcn_readfirstlane(c.after);
    if (lane == 0) kp = chunk0 <= n ? c.before : kNoKey;
    if (lane == kWave - 1) kn = k_after;
    // heads of all cells, and of those of two or more atoms, one bit per slot
    uint32_t hm = 0, mm = 0, kl = 0;
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        const uint32_t k = c.k[j], p = j > 0 ? c.k[j > 0 ? j - 1 : 0] : kp,
                       x = j + 1 < ITEMS ? c.k[j + 1 < ITEMS ? j + 1 : j] : kn;
        const bool head = k != kNoKey && (k != p || b + j == 0);
        hm |= (uint32_t)head << j;
        mm |= (uint32_t)(head && x == k) << j;
        if (head) kl = k;   // the lane's last head
    }
    k_first = __builtin_amdgcn_readfirstlane(c.k[0]);
    const uint64_t any = __ballot(hm != 0);
    if (!any) return 0;   // no cell starts here
    k_last = __builtin_amdgcn_readlane(kl, 63 - __clzll((long long)any));
    // end of the last cell: the first later slot with another key.  The wave
    // holds the next 64 slots; a longer cell (e.g. the overflow cell of atoms
    // outside the grid) is searched by galloping.
    int end;
    {
        const uint64_t bd = __ballot(chunk1 == chunk0 + kWave * ITEMS && c.after != kNoKey && c.after != k_last);
        end = chunk1 + kWave;
        if (bd) end = chunk1 + __ffsll((unsigned long long)bd) - 1;
        if (chunk1 + kWave >= n) end = min(end, n);
        if (!bd && end < n) {
            int lo = end, stp = 1;
            while (lo + stp - 1 < n && key[lo + stp - 1] == k_last) { lo += stp; stp <<= 1; }
            int hi = min(n, lo + stp - 1);  // the first other key is in [lo, hi]
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (key[mid] == k_last) lo = mid + 1; else hi = mid;
            }
            end = lo;
        }
    }
    // the first head in a later lane ends this lane's last cell
    const uint64_t later = lane < kWave - 1 ? any & (~0ull << (lane + 1)) : 0ull;
    const int m = later ? __ffsll((unsigned long long)later) - 1 : lane;
    const int first = __shfl(b + __ffs((int)hm) - 1, m, kWave);
    if (later) end = first;
    // places in the list: lanes list up to four cells each, counted bit by bit
    const uint32_t cnt = (uint32_t)__popc(mm);
    const uint64_t lt = lanemask_lt();
    const uint64_t c0 = __ballot(cnt & 1u), c1 = ITEMS > 2 ? __ballot(cnt & 2u) : 0ull,
                   c2 = ITEMS > 4 ? __ballot(cnt & 4u) : 0ull;
    int pos = __popcll(c0 & lt) + 2 * __popcll(c1 & lt) + 4 * __popcll(c2 & lt);
    const int nm = __popcll(c0) + 2 * __popcll(c1) + 4 * __popcll(c2);
#pragma unroll
    for (int j = 0; j < ITEMS; ++j) {
        if ((mm >> j) & 1u) {
            const uint32_t rest = hm >> (j + 1);
            L.key[pos] = c.k[j];
            L.end[pos] = rest ? b + j + __ffs((int)rest) : end;
            L.start[pos] = (short)(lane * ITEMS + j);
            ++pos;
        }
    }
    wave_lds_fence();
    return nm;
}

}  // namespace dsmc
