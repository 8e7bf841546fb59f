// resort_device.hpp -- device side of the incremental re-sort: its first phase
// (run by the finalize kernels of both forms beside their sums) and the merge
// of one tile.  The scheme is described in primitives.hip.
#pragma once

#include "dsmc_device.hpp"
#include "dsmc_internal.hpp"

namespace dsmc {

constexpr int kStayTile = kResortTile;         // slots per tile (and bucket)
constexpr int kStayShift = 11;
constexpr int kTileWords = kStayTile / 64;     // mask words per tile
constexpr int kBucketLds = 512;                // movers a bucket ranks in LDS
constexpr int kBucketCap = 1024;               // fixed room of a bucket (>= kBucketLds)
static_assert((1 << kStayShift) == kStayTile, "stay tile");
static_assert(kTileWords == 32, "a tile's mask words are half a wave");

// Exclusive prefix of v over the 32 lanes of this lane's half-wave.
__device__ __forceinline__ uint32_t halfwave_exclusive_scan(uint32_t v)
{
    return halfwave_inclusive_scan(v) - v;
}

// (key, slot) order; slots are distinct.
__device__ __forceinline__ bool kv_less(uint32_t ka, uint32_t va, uint32_t kb, uint32_t vb)
{
    return ka < kb || (ka == kb && va < vb);
}

// Block j (256 threads) of the re-sort's first phase, on the move's masks of
// mask words [64 j, 64 j + 64) (two tiles of the n slots): the tiles' movers
// and removed atoms counted, and every mover (new key k, slot v) put into the
// bucket of its tile, the last one whose first (key, slot) lies below (k, v),
// or the first tile.  The tiles' first keys (left by the merge) are searched
// in LDS; lanes of a wave with the same bucket share one atomic (nearby
// movers mostly do): 30000 movers' own returning atomics took the move that
// issued them from 26 to 98 us at N = 1e6, and to 44 us with every counter in
// a line of its own.  A bucket has a fixed room of kBucketCap movers; those
// beyond it go to an overflow list.  Bound by its chain of dependent loads
// (masks, keys, atomic), which runs beside the finalize's sums: the step lost
// the launch that located every mover's exact slot (six more dependent loads;
// the merge now finds it in LDS), N = 2e4 30.5 -> 26.5 us, N = 1e6 61.3 ->
// 55.5 us, 256 traps in two groups 155 -> 150 us.
constexpr int kListWords = 64;               // mask words per block
constexpr int kListSlots = kListWords * 64;
constexpr int kBucketBits = 13;
constexpr int kMaxTiles = 1 << kBucketBits;  // tiles the LDS sample table holds
static_assert(kListSlots == 2 * kStayTile, "two tiles per block");

__host__ __device__ inline int resort_list_blocks(int n_cap)
{
    return n_cap > 0 ? (n_cap + kListSlots - 1) / kListSlots : 1;
}

// LDS of the tiles' first keys (dynamic).
inline size_t resort_list_lds(const ResortList &rl)
{
    return rl.blocks > 0 ? (((size_t)rl.tiles + 3) & ~(size_t)3) * sizeof(uint32_t) : 0;
}

// Dynamic LDS of a finalize with that work.
inline size_t resort_work_lds(const ResortWork &w)
{
    return w.merge.tiles > 0 ? (((size_t)w.merge.n_cap + 7) & ~(size_t)7) * sizeof(unsigned short)
                             : resort_list_lds(w.list);
}

// first: the dynamic LDS above; slot: the block's movers, from its first slot.
__device__ __forceinline__ void resort_list_block(const ResortList &rl, int j, uint32_t *first,
                                                  unsigned short *slot)
{
    const ResortBuckets &rb = rl.b;
    const int tid = (int)threadIdx.x, lane = tid & (kWave - 1);
    const int w = j * kListWords + lane;   // every wave reads the block's 64 words
    const uint64_t mm = rl.mask_m[w];
    const uint64_t md = rl.may_remove ? rl.mask_d[w] : 0ull;
    {
        const uint4 *t4 = (const uint4 *)rb.tsamp;
        uint4 *l4 = (uint4 *)first;
        const int nv = (rl.tiles + 3) >> 2;
        for (int v0 = tid; v0 < nv; v0 += 4 * 256) {
            uint4 c[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) c[u] = v0 + u * 256 < nv ? t4[v0 + u * 256] : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (v0 + u * 256 < nv) l4[v0 + u * 256] = c[u];
        }
    }
    const int n = *rl.n_dev;
    if (j > 0 && j * kListSlots >= n) {         // whole block leaves together
        if (tid < 2) rb.tile_moved[2 * j + tid] = rb.tile_dead[2 * j + tid] = 0u;   // (all tiles are summed)
        return;
    }
    // the words' movers and removed atoms (bits past the slots are zero)
    const uint32_t cnt = (uint32_t)__popcll(mm) << 16 | (uint32_t)__popcll(md);
    const uint32_t inc = wave_inclusive_scan(cnt);
    const uint32_t half = __shfl(inc, kTileWords - 1, kWave);   // the first tile's: words 0 .. 31
    if (tid == kTileWords - 1 || tid == kWave - 1) {
        const int t = 2 * j + (tid == kWave - 1);
        const uint32_t c = t > 0 && t * kStayTile >= n ? 0u : tid == kWave - 1 ? inc - half : inc;
        rb.tile_moved[t] = c >> 16;
        rb.tile_dead[t] = c & 0xFFFFu;
    }
    const int m = (int)(__builtin_amdgcn_readlane(inc, kWave - 1) >> 16);
    if (m == 0) return;
    // list the movers: wave q lists the words 16 q .. 16 q + 15, four lanes a
    // word, a quarter of its bits each
    {
        const int q = tid / kWave, wl = 16 * q + (lane >> 2), part = lane & 3;
        const uint64_t word = __shfl(mm, wl, kWave);
        const uint32_t excl = __shfl((inc >> 16) - (uint32_t)__popcll(mm), wl, kWave);
        const uint64_t below = part ? word & (~0ull >> (64 - 16 * part)) : 0ull;
        int o = (int)excl + __popcll(below);
        for (uint32_t bits = (uint32_t)(word >> (16 * part)) & 0xFFFFu; bits; bits &= bits - 1)
            slot[o++] = (unsigned short)(wl * 64 + 16 * part + __ffs((int)bits) - 1);
    }
    __syncthreads();   // (m is the same in every wave)
    const int nt = (n + kStayTile - 1) >> kStayShift;
    for (int e0 = 0; e0 < m; e0 += 256) {
        const int e = e0 + tid;
        const bool valid = e < m;
        const uint32_t v = valid ? (uint32_t)(j * kListSlots) + slot[e] : 0u;
        const uint32_t k = valid ? rl.key_new[v] : 0u;
        int lo = 0;   // tiles after the first that lie below (k, v): a prefix
        if (valid) {
            int hi = nt - 1;
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if (kv_less(first[mid], (uint32_t)mid << kStayShift, k, v)) lo = mid; else hi = mid - 1;
            }
        }
        const uint64_t peers = match_bits<kBucketBits>((uint32_t)lo, __ballot(valid));
        const int leader = __ffsll((unsigned long long)peers) - 1;
        uint32_t base = 0;
        if (valid && lane == leader) base = atomicAdd(&rb.bcnt[lo], (uint32_t)__popcll(peers));
        base = __shfl(base, leader < 0 ? 0 : leader, kWave);
        if (valid) {
            const uint32_t r = base + (uint32_t)__popcll(peers & lanemask_lt());
            const uint64_t kv = (uint64_t)k << 32 | v;
            if (r < (uint32_t)kBucketCap) rb.room[(size_t)lo * kBucketCap + r] = kv;
            else rb.over[atomicAdd(rb.n_over, 1u)] = kv;
        }
    }
}

// Clears the buckets' counts (by the collide, which runs between the merge
// that reads them and the next first phase): thread g of `threads`.
__device__ __forceinline__ void resort_clear(const ResortBuckets &rb, int g, int threads)
{
    for (int i = g; i < rb.n_counts; i += threads) rb.bcnt[i] = 0u;
}

// LDS of a merge block (256 threads): 16.3 KB, so that nine blocks fit a CU.
struct MergeLds {
    __align__(16) uint64_t kv[kBucketLds];      // the bucket's movers, key << 32 | slot, by insertion point
    uint32_t K[kStayTile];                      // the tile's keys of the last sort
    // movers inserted at each slot, then the scan E (below 2048 + kBucketLds)
    __align__(16) unsigned short H[kStayTile];
    uint64_t stay[kTileWords];                  // stay bits of the tile's words
    uint32_t wst[kTileWords];                   // stays of the tile before each word
    uint32_t sum[3][256 / kWave];
    uint32_t at_end;                            // movers inserted after the tile's last slot
    int n_big;                                  // movers gathered for a big bucket
};

// Insertion point in the tile: the first p in [0, ns] with (K[p], g0 + p) >= (k, v).
__device__ __forceinline__ uint32_t merge_point(const uint32_t *K, int ns, uint32_t g0, uint32_t k, uint32_t v)
{
    int lo = 0, hi = ns;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (kv_less(K[mid], g0 + (uint32_t)mid, k, v)) lo = mid + 1; else hi = mid;
    }
    return (uint32_t)lo;
}

// Sort of one bucket that does not fit the LDS table, by one block, in
// global scratch: chunks of kBucketLds sorted in LDS (bitonic network), then
// pairwise merges of runs (merge path per thread).  Used only when a great
// many atoms land in the same tile (e.g. nearly all atoms change cell in one
// step); O(b log b) work for one block.  Leaves the sorted bucket in a0 or
// a1; returns the one that holds it.
__device__ inline uint64_t *big_bucket_sort(uint64_t *a0, uint64_t *a1, int b, uint64_t *lds)
{
    const int tid = threadIdx.x;
    for (int c0 = 0; c0 < b; c0 += kBucketLds) {
        const int c = min(kBucketLds, b - c0);
        for (int e = tid; e < kBucketLds; e += 256) lds[e] = e < c ? a0[c0 + e] : ~0ull;
        __syncthreads();
        for (int size = 2; size <= kBucketLds; size <<= 1) {
            for (int stride = size >> 1; stride > 0; stride >>= 1) {
                for (int pr = tid; pr < kBucketLds / 2; pr += 256) {
                    const int i = 2 * pr - (pr & (stride - 1));   // lower index of the pair
                    const int j = i + stride;
                    const uint64_t x = lds[i], y = lds[j];
                    if ((y < x) == ((i & size) == 0)) { lds[i] = y; lds[j] = x; }
                }
                __syncthreads();
            }
        }
        for (int e = tid; e < c; e += 256) a0[c0 + e] = lds[e];
        __syncthreads();
    }
    uint64_t *s = a0, *d = a1;
    for (int wdt = kBucketLds; wdt < b; wdt <<= 1) {
        for (int lo = 0; lo < b; lo += 2 * wdt) {
            const int na = min(wdt, b - lo), nb = max(0, min(wdt, b - lo - wdt));
            const int len = na + nb;
            const int per = (len + 255) / 256;
            const int d0 = min(tid * per, len), d1 = min(d0 + per, len);
            // merge path split of output d0 between run a = [lo, lo+na), b = [lo+na, ...)
            int l = max(0, d0 - nb), h = min(d0, na);
            while (l < h) {
                const int mid = (l + h) >> 1;
                if (s[lo + mid] < s[lo + na + d0 - 1 - mid]) l = mid + 1; else h = mid;
            }
            int ia = l, ib = d0 - l;
            for (int o = d0; o < d1; ++o) {
                const bool ta = ia < na && (ib >= nb || s[lo + ia] < s[lo + na + ib]);
                d[lo + o] = ta ? s[lo + ia] : s[lo + na + ib];
                ia += ta; ib += !ta;
            }
        }
        __syncthreads();   // this pass's writes are visible to the whole block
        uint64_t *x = s; s = d; d = x;
    }
    return s;
}

// The sum of the elements of c, elements i0 .. i0 + 3 of an array, below n.
__device__ __forceinline__ uint32_t sum_below_n(uint4 c, int i0, int n)
{
    return (i0 < n ? c.x : 0u) + (i0 + 1 < n ? c.y : 0u) + (i0 + 2 < n ? c.z : 0u) + (i0 + 3 < n ? c.w : 0u);
}

// Sum of v[0 .. n), this thread's share (256 threads; v is 16-byte aligned
// and ends on a multiple of four elements).
__device__ __forceinline__ uint32_t sum_share(const uint32_t *__restrict__ v, int n)
{
    const uint4 *v4 = (const uint4 *)v;
    uint32_t s = 0;
    for (int i = (int)threadIdx.x; 4 * i < n; i += 256) s += sum_below_n(v4[i], 4 * i, n);
    return s;
}

// This thread's shares of the sums over the tiles (256 threads): movers
// inserted before tile t less the movers and removed atoms that left its
// earlier slots; removed atoms before it; and all.  The three arrays'
// loads go out together, two words of each: one round of latency up to 4 M
// slots (a loop per array, each waiting for its own, took four).
__device__ __forceinline__ void tile_sums(const ResortBuckets &rb, bool may_remove, int t, int tiles,
                                          uint32_t (&part)[3])
{
    const uint4 *ins = (const uint4 *)rb.bcnt, *mv = (const uint4 *)rb.tile_moved, *dd = (const uint4 *)rb.tile_dead;
    const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
    part[0] = part[1] = part[2] = 0u;
    const int end = may_remove ? tiles : t;
    for (int i = (int)threadIdx.x; 4 * i < end; i += 2 * 256) {
        uint4 a[2], b[2], c[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = 4 * (i + 256 * u);
            a[u] = e < t ? ins[i + 256 * u] : zero;
            b[u] = e < t ? mv[i + 256 * u] : zero;
            c[u] = may_remove && e < end ? dd[i + 256 * u] : zero;
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = 4 * (i + 256 * u);
            const uint32_t d = sum_below_n(c[u], e, t);
            part[0] += sum_below_n(a[u], e, t) - sum_below_n(b[u], e, t) - d;
            part[1] += d;
            part[2] += sum_below_n(c[u], e, end);
        }
    }
}

// Of tile t's bucket: above the tile's first (key, slot) (or the first tile)
// and not above the next tile's (if it has one).
__device__ __forceinline__ bool in_bucket(int t, uint32_t f0, bool has1, uint32_t f1, uint64_t kv)
{
    const uint32_t k = (uint32_t)(kv >> 32), v = (uint32_t)kv;
    const bool ge = t == 0 || kv_less(f0, (uint32_t)(t * kStayTile), k, v);
    const bool lt = !has1 || !kv_less(f1, (uint32_t)((t + 1) * kStayTile), k, v);
    return ge && lt;
}

constexpr int kMergePer = kStayTile / 256;   // slots per thread

// What a merge block starts from.
struct MergeTile {
    uint32_t kk[kMergePer];   // keys of the last sort at positions tid + 256 u
    uint64_t wm, wd;          // mask words (threads 0 .. 31)
    uint32_t part[3];         // this thread's shares: movers inserted before the tile less the movers and
                              // removed atoms that left its earlier slots; removed atoms before it; all
    int n, b;                 // slots, and movers of the bucket
};

// Block of 256 threads for tile t (2048 slots).  The tile's output is a
// contiguous window from w0: position p of the tile (slot g0 + p) is preceded
// there by E(p) = the stays below p plus the bucket movers inserted below p,
// so a stay at p goes to w0 + E(p) + h(p), h(p) = movers inserted at p, and a
// mover inserted at p to w0 + E(p) + (its rank among the movers inserted at
// p).  E is an exclusive scan of st(p) + h(p) over the tile, h a histogram of
// the bucket in LDS; p may also be the tile's end.  A stay's key is its key of
// the last sort and a mover's comes with it, so the new keys are not read.
// Buckets larger than the LDS table are sorted in global scratch by the
// block; movers then go to w0 + (stays below p) + (rank in the bucket), stays
// after the movers below them.  Bound by its chain of loads and barriers at
// small N and by the O(b) work of the movers at large: the histogram's atomics
// number the movers of a point, so that each is ranked among those alone
// (comparing it with all b of the bucket, and the sums one after the other:
// 11.2 us at N = 1e6, now 8.0).
// mover(e): the bucket's e-th mover, for e = tid, tid + 256 below kBucketLds;
// gather(): all of a larger bucket's movers, in ra.big.
template <class Mover, class Gather>
__device__ __forceinline__ void merge_window(const ResortMerge &ra, int t, MergeLds &L, const MergeTile &mt,
                                             Mover mover, Gather gather)
{
    const int tid = threadIdx.x;
    const int g0 = t * kStayTile;
    const int p0 = tid * kMergePer;   // positions p0 .. p0 + 7 in the scan
    const int n = mt.n, b = mt.b;
    const uint32_t(&kk)[kMergePer] = mt.kk;
    const uint64_t wm = mt.wm, wd = mt.wd;
    uint32_t part[3] = { mt.part[0], mt.part[1], mt.part[2] };
    const int ns = min(kStayTile, n - g0);   // slots of the tile
#pragma unroll
    for (int u = 0; u < kMergePer; ++u) L.K[tid + 256 * u] = kk[u];
    ((uint4 *)L.H)[tid] = make_uint4(0u, 0u, 0u, 0u);
    if (tid == 0) L.at_end = 0u;
    uint64_t dd = 0ull;
    if (tid < kTileWords) {
        const int l0 = tid * 64;
        uint64_t st = 0ull;
        if (l0 < ns) {
            const uint64_t in = ns - l0 >= 64 ? ~0ull : (1ull << (ns - l0)) - 1ull;
            st = ~(wm | wd) & in;
            dd = wd & in;
        }
        L.stay[tid] = st;
        L.wst[tid] = halfwave_exclusive_scan((uint32_t)__popcll(st));
    }
    const int lane = tid & (kWave - 1), w = tid / kWave;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        if (k > 0 && !ra.may_remove) break;
        part[k] = wave_sum(part[k]);
        if (lane == 0) L.sum[k][w] = part[k];
    }
    __syncthreads();   // H cleared, keys, stay words and sums in place
    auto total_of = [&](int k) { return L.sum[k][0] + L.sum[k][1] + L.sum[k][2] + L.sum[k][3]; };
    const uint32_t w0 = (uint32_t)g0 + total_of(0);   // first output slot of the tile
    if (ra.may_remove && tid < kTileWords) {
        // removed atoms: to the end of the output, in slot order
        uint32_t od = (uint32_t)n - total_of(2) + total_of(1) + halfwave_exclusive_scan((uint32_t)__popcll(dd));
        for (uint64_t bb = dd; bb; bb &= bb - 1) {
            ra.out_k[od] = ra.dead_key;
            ra.out_v[od++] = (uint32_t)(g0 + tid * 64) + (uint32_t)(__ffsll((unsigned long long)bb) - 1);
        }
    }
    auto put = [&](uint32_t o, uint32_t k, uint32_t v) {
        ra.out_k[o] = k;
        ra.out_v[o] = v;
        if ((o & (kStayTile - 1)) == 0) ra.tsamp_out[o >> kStayShift] = k;
    };
    auto stays_below = [&](uint32_t p) {
        if (p >= (uint32_t)kStayTile) return L.wst[kTileWords - 1] + (uint32_t)__popcll(L.stay[kTileWords - 1]);
        const uint64_t m = (p & 63) ? L.stay[p >> 6] & (~0ull >> (64 - (p & 63))) : 0ull;
        return L.wst[p >> 6] + (uint32_t)__popcll(m);
    };
    if (b > kBucketLds) {
        // the bucket gathered in scratch, at the earlier buckets' movers, and
        // sorted there
        __syncthreads();   // the sums are read
        uint64_t *const a = gather(), *const c = ra.big_alt + (a - ra.big);
        __syncthreads();
        const uint64_t *g = big_bucket_sort(a, c, b, L.kv);
        // a stay goes after the movers below it, found in the sorted bucket
        for (int u = 0; u < kMergePer; ++u) {
            const int p = tid + 256 * u;
            if (p >= ns || !((L.stay[p >> 6] >> (p & 63)) & 1ull)) continue;
            const uint64_t key = (uint64_t)kk[u] << 32 | (uint32_t)(g0 + p);
            int lo = 0, hi = b;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (g[mid] < key) lo = mid + 1; else hi = mid;
            }
            put(w0 + stays_below((uint32_t)p) + (uint32_t)lo, kk[u], (uint32_t)(g0 + p));
        }
        for (int r = tid; r < b; r += 256) {
            const uint32_t k = (uint32_t)(g[r] >> 32), v = (uint32_t)g[r];
            put(w0 + stays_below(merge_point(L.K, ns, (uint32_t)g0, k, v)) + (uint32_t)r, k, v);
        }
        return;
    }
    // the movers stay in registers until their points' windows are known;
    // `claim` numbers the movers of one point
    constexpr int kMv = kBucketLds / 256;
    uint64_t kv[kMv];
    uint32_t q[kMv], claim[kMv];
#pragma unroll
    for (int u = 0; u < kMv; ++u) {
        const int e = tid + 256 * u;
        if (e >= b) continue;
        kv[u] = mover(e);
        q[u] = merge_point(L.K, ns, (uint32_t)g0, (uint32_t)(kv[u] >> 32), (uint32_t)kv[u]);
        if (q[u] < (uint32_t)kStayTile) {
            const int sh = 16 * (q[u] & 1);
            claim[u] = (atomicAdd((uint32_t *)L.H + (q[u] >> 1), 1u << sh) >> sh) & 0xFFFFu;
        } else {
            claim[u] = atomicAdd(&L.at_end, 1u);
        }
    }
    __syncthreads();
    // E: exclusive scan of st(p) + h(p) over the tile, 8 consecutive
    // positions per thread (16 bytes of H)
    {
        const uint4 h4 = ((const uint4 *)L.H)[tid];
        const uint32_t h[4] = { h4.x, h4.y, h4.z, h4.w };
        const uint32_t st8 = (uint32_t)(L.stay[p0 >> 6] >> (p0 & 63)) & 0xFFu;
        uint32_t e[kMergePer], run = 0;
#pragma unroll
        for (int u = 0; u < kMergePer; ++u) {
            e[u] = run;
            run += ((st8 >> u) & 1u) + ((h[u >> 1] >> (16 * (u & 1))) & 0xFFFFu);
        }
        const uint32_t inc = wave_inclusive_scan(run);
        if (lane == kWave - 1) L.sum[1][w] = inc;
        __syncthreads();
        uint32_t base = inc - run;
        for (int ww = 0; ww < w; ++ww) base += L.sum[1][ww];
        uint4 o;
        o.x = (base + e[0]) | (base + e[1]) << 16;
        o.y = (base + e[2]) | (base + e[3]) << 16;
        o.z = (base + e[4]) | (base + e[5]) << 16;
        o.w = (base + e[6]) | (base + e[7]) << 16;
        ((uint4 *)L.H)[tid] = o;
    }
    __syncthreads();   // E complete
    const uint32_t total = total_of(1), at_end = L.at_end;
    // stays, at positions tid + 256 u (coalesced stores): E(p) + h(p) =
    // E(p + 1) - st(p) = E(p + 1) - 1
#pragma unroll
    for (int u = 0; u < kMergePer; ++u) {
        const int p = tid + 256 * u;
        if (p >= ns || !((L.stay[p >> 6] >> (p & 63)) & 1ull)) continue;
        put(w0 + (p + 1 < kStayTile ? L.H[p + 1] : total) - 1u, kk[u], (uint32_t)(g0 + p));
    }
    // movers: those of one point beside each other in LDS, then each one's
    // rank among them
    uint32_t ep[kMv], at[kMv], hp[kMv];
#pragma unroll
    for (int u = 0; u < kMv; ++u) {
        if (tid + 256 * u >= b) continue;
        const uint32_t p = q[u];
        ep[u] = total; hp[u] = at_end;
        if (p < (uint32_t)kStayTile) {
            ep[u] = L.H[p];
            hp[u] = (p + 1 < (uint32_t)kStayTile ? L.H[p + 1] : total) - ep[u] -
                    ((uint32_t)(L.stay[p >> 6] >> (p & 63)) & 1u);
        }
        at[u] = ep[u] - stays_below(p);   // movers inserted below p
        L.kv[at[u] + claim[u]] = kv[u];
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < kMv; ++u) {
        if (tid + 256 * u >= b) continue;
        uint32_t r = 0;   // (key, slot) order is the order of key << 32 | slot
        for (uint32_t f = 0; hp[u] > 1 && f < hp[u]; ++f) r += (uint32_t)(L.kv[at[u] + f] < kv[u]);
        put(w0 + ep[u] + r, (uint32_t)(kv[u] >> 32), (uint32_t)kv[u]);
    }
}

// After the first phase.
__device__ __forceinline__ void resort_merge_block(const ResortMerge &ra, int t, MergeLds &L)
{
    const ResortBuckets &rb = ra.b;
    const int tid = threadIdx.x;
    const int g0 = t * kStayTile;
    // Every load that does not need the slot count is issued together with
    // it, in one round: the tile's keys at positions tid + 256 u (coalesced;
    // up to the capacity, those past the slots are never used), its mask
    // words, the counts of the earlier tiles, its bucket's size, and this
    // thread's first mover of the bucket's room (used when the bucket holds it).
    MergeTile mt;
#pragma unroll
    for (int u = 0; u < kMergePer; ++u) {
        const int p = tid + 256 * u;
        mt.kk[u] = g0 + p < ra.n_cap ? ra.key_old[g0 + p] : 0u;
    }
    mt.n = *ra.n_dev;
    mt.b = (int)rb.bcnt[t];
    mt.wm = mt.wd = 0ull;   // (in bounds up to the last tile + 1)
    if (tid < kTileWords) {
        mt.wm = ra.mask_m[(g0 >> 6) + tid];
        mt.wd = ra.mask_d[(g0 >> 6) + tid];
    }
    const size_t fb0 = (size_t)t * kBucketCap;   // the bucket's fixed room
    constexpr int kFirst = 128;                  // movers loaded before the count is known
    const uint64_t mkv = tid < kFirst ? rb.room[fb0 + tid] : 0ull;
    tile_sums(rb, ra.may_remove, t, ra.tiles, mt.part);
    if (t > 0 && g0 >= mt.n) return;   // whole block leaves together
    auto mover = [&](int e) { return e < kFirst ? mkv : rb.room[fb0 + e]; };
    // the bucket's room, then its movers in the overflow list
    auto gather = [&]() {
        const int lane = tid & (kWave - 1), w = tid / kWave;
        const uint32_t fs = wave_sum(sum_share(rb.bcnt, t));
        if (lane == 0) L.sum[0][w] = fs;
        if (tid == 0) L.n_big = min(mt.b, kBucketCap);
        __syncthreads();
        uint64_t *const a = ra.big + (L.sum[0][0] + L.sum[0][1] + L.sum[0][2] + L.sum[0][3]);
        for (int e = tid; e < min(mt.b, kBucketCap); e += 256) a[e] = rb.room[fb0 + e];
        if (mt.b > kBucketCap) {
            const int no = (int)*rb.n_over;
            const bool has1 = g0 + kStayTile < mt.n;   // (tsamp is being replaced by the merge)
            const uint32_t f1 = has1 ? ra.key_old[g0 + kStayTile] : 0u;
            for (int e = tid; e < no; e += 256) {
                const uint64_t kv = rb.over[e];
                if (in_bucket(t, L.K[0], has1, f1, kv)) a[atomicAdd(&L.n_big, 1)] = kv;
            }
        }
        return a;
    };
    merge_window(ra, t, L, mt, mover, gather);
}

// Without a first phase, for up to kScanSlots slots: every tile's block reads
// the masks and the movers' new keys of all slots and keeps those of its
// bucket.  list: the movers' slots (n_cap of them at most).  Bound by its
// chain of loads (masks, new keys) and barriers: 7.9 us beside the finalize at
// N = 2e4, where the first phase took 4.7 and the merge 6.8.
__device__ __forceinline__ void resort_scan_merge_block(const ResortMerge &ra, int t, MergeLds &L,
                                                        unsigned short *list)
{
    const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
    const int g0 = t * kStayTile, g1 = g0 + kStayTile;
    MergeTile mt;
#pragma unroll
    for (int u = 0; u < kMergePer; ++u) {
        const int p = tid + 256 * u;
        mt.kk[u] = g0 + p < ra.n_cap ? ra.key_old[g0 + p] : 0u;
    }
    const int n = *ra.n_dev;
    const uint32_t f0 = g0 < ra.n_cap ? ra.key_old[g0] : 0u, f1 = g1 < ra.n_cap ? ra.key_old[g1] : 0u;
    mt.wm = mt.wd = 0ull;
    if (tid < kTileWords) {
        mt.wm = ra.mask_m[(g0 >> 6) + tid];
        mt.wd = ra.mask_d[(g0 >> 6) + tid];
    }
    // two words of the masks per thread
    static_assert(kScanSlots == 2 * 256 * 64, "two words per thread");
    uint64_t m[2], d[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int wl = 2 * tid + u;
        m[u] = 64 * wl < ra.n_cap ? ra.mask_m[wl] : 0ull;
        d[u] = 64 * wl < ra.n_cap && ra.may_remove ? ra.mask_d[wl] : 0ull;
    }
    if (t > 0 && g0 >= n) return;   // whole block leaves together
    mt.n = n;
    uint32_t moved = 0, gone_before = 0, gone = 0, moved_before = 0;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int s0 = 64 * (2 * tid + u);
        const uint64_t in = n - s0 >= 64 ? ~0ull : n > s0 ? (1ull << (n - s0)) - 1ull : 0ull;
        m[u] &= in; d[u] &= in;
        const uint32_t cm = (uint32_t)__popcll(m[u]), cd = (uint32_t)__popcll(d[u]);
        moved += cm; gone += cd;
        if (s0 < g0) { moved_before += cm; gone_before += cd; }
    }
    const uint32_t inc = wave_inclusive_scan(moved);
    if (lane == kWave - 1) L.sum[0][w] = inc;
    if (tid == 0) L.n_big = 0;
    __syncthreads();
    uint32_t at = inc - moved;
    for (int ww = 0; ww < w; ++ww) at += L.sum[0][ww];
    const int total = (int)(L.sum[0][0] + L.sum[0][1] + L.sum[0][2] + L.sum[0][3]);
#pragma unroll
    for (int u = 0; u < 2; ++u)
        for (uint64_t bits = m[u]; bits; bits &= bits - 1)
            list[at++] = (unsigned short)(64 * (2 * tid + u) + __ffsll((unsigned long long)bits) - 1);
    __syncthreads();
    const bool has1 = g1 < n;
    constexpr int kAhead = 8;   // movers whose keys a thread loads together
    uint32_t below = 0;         // movers inserted before the tile (this thread's)
    for (int e0 = tid; e0 < total; e0 += kAhead * 256) {
        uint32_t v[kAhead], k[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int e = e0 + 256 * u;
            v[u] = e < total ? list[e] : 0u;
            k[u] = e < total ? ra.key_new[v[u]] : 0u;
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            if (e0 + 256 * u >= total) continue;
            const uint64_t kv = (uint64_t)k[u] << 32 | v[u];
            if (in_bucket(t, f0, has1, f1, kv)) {
                const int x = atomicAdd(&L.n_big, 1);
                if (x < kBucketLds) L.kv[x] = kv;
            } else if (t > 0 && !kv_less(f0, (uint32_t)g0, k[u], v[u])) {
                ++below;
            }
        }
    }
    mt.part[0] = below - moved_before - gone_before;
    mt.part[1] = gone_before;
    mt.part[2] = gone;
    __syncthreads();
    mt.b = L.n_big;
    uint64_t mine[kBucketLds / 256];
#pragma unroll
    for (int u = 0; u < kBucketLds / 256; ++u) mine[u] = tid + 256 * u < mt.b ? L.kv[tid + 256 * u] : 0ull;
    auto mover = [&](int e) { return e < 256 ? mine[0] : mine[1]; };
    auto gather = [&]() {
        const uint32_t s = wave_sum(below);
        if (lane == 0) L.sum[0][w] = s;
        if (tid == 0) L.n_big = 0;
        __syncthreads();
        uint64_t *const a = ra.big + (L.sum[0][0] + L.sum[0][1] + L.sum[0][2] + L.sum[0][3]);
        for (int e = tid; e < total; e += 256) {
            const uint32_t v = list[e];
            const uint64_t kv = (uint64_t)ra.key_new[v] << 32 | v;
            if (in_bucket(t, f0, has1, f1, kv)) a[atomicAdd(&L.n_big, 1)] = kv;
        }
        return a;
    };
    merge_window(ra, t, L, mt, mover, gather);
}

}  // namespace dsmc
