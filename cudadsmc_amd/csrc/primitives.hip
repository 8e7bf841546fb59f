// primitives.hip -- data-movement primitives of the DSMC step written for
// wave64 / LDS on gfx950:
//   * stable LSD radix sort of (uint32 key, uint32 value) pairs, digits of 8 or
//     10 bits, reduce-then-scan per pass (upsweep histogram, per-digit scan, downsweep
//     scatter).  Within a tile the rank of each key among equal digits comes
//     from one wave ballot per bit (lanes whose digit matches) plus a per-wave running
//     count in LDS, so the order of equal keys is the input order (stable);
//     the scatter is staged through LDS so global writes are digit runs.
//     Replaces thrust::sort_by_key (collisions.cu:282-284).
//   * exclusive scan of int32 (thrust::exclusive_scan, main.cu:440-442).
//   * stable stream compaction map from a stencil (thrust::remove_if,
//     main.cu:493-498), ballot + popcount ranks.
//   * fills and a Philox block generator (for known-answer tests).
// None of these kernels waits on another block, so none can hang.
#include "dsmc_device.hpp"
#include "dsmc_internal.hpp"
#include "resort_device.hpp"

#include <algorithm>

namespace dsmc {

// ---------------------------------------------------------------------------
// Radix sort
// ---------------------------------------------------------------------------
// One pass over digits of B bits: BLOCK threads take a tile of BLOCK * ITEMS
// pairs.  n_dev: the pair count on the device, or null (then n).  FEW: the
// counts go out tile by tile, for a downsweep that adds them up itself.
template <int B, int BLOCK, int ITEMS, bool FEW>
__global__ __launch_bounds__(BLOCK) void k_radix_upsweep(const uint32_t *__restrict__ keys,
                                                         const int *__restrict__ n_dev, int n_host, int shift,
                                                         uint32_t *__restrict__ hist, int nb)
{
    constexpr int R = 1 << B, TILE = BLOCK * ITEMS;
    __shared__ uint32_t h[R];
    const int tid = threadIdx.x;
    for (int i = tid; i < R; i += BLOCK) h[i] = 0;
    __syncthreads();
    const int n = n_dev ? *n_dev : n_host;
    const long long tile0 = (long long)blockIdx.x * TILE;
    if (tile0 < n) {
        const int lane = tid & (kWave - 1), w = tid / kWave;
        const long long base = tile0 + w * (kWave * ITEMS) + lane;
        uint32_t k[ITEMS];
#pragma unroll
        for (int u = 0; u < ITEMS; ++u) k[u] = base + u * kWave < n ? keys[base + u * kWave] : 0u;
#pragma unroll
        for (int u = 0; u < ITEMS; ++u)
            if (base + u * kWave < n) atomicAdd(&h[(k[u] >> shift) & (R - 1)], 1u);
    }
    // tiles past the end are not scanned (block 0 always writes: n may be 0)
    if (tile0 >= n && blockIdx.x > 0) return;
    __syncthreads();
    for (int d = tid; d < R; d += BLOCK) {
        if constexpr (FEW) hist[(size_t)blockIdx.x * R + d] = h[d];
        else hist[(size_t)d * nb + blockIdx.x] = h[d];
    }
}

// One block per digit: exclusive scan of that digit's per-block counts.
__global__ __launch_bounds__(256) void k_radix_scan(uint32_t *__restrict__ hist, uint32_t *__restrict__ totals,
                                                    const int *__restrict__ n_dev, int n_host, int tile, int nb)
{
    __shared__ uint32_t tmp[256 / kWave + 1];
    const int n = n_dev ? *n_dev : n_host;
    const int nb_used = min(nb, ((n > 0 ? n : 1) + tile - 1) / tile);  // tiles with data
    uint32_t *row = hist + (size_t)blockIdx.x * nb;
    const int per = (nb_used + 255) / 256;
    const int b0 = threadIdx.x * per;
    uint32_t s = 0;
    for (int i = 0; i < per; ++i) {
        const int j = b0 + i;
        if (j < nb_used) s += row[j];
    }
    uint32_t total;
    uint32_t ex = block_exclusive_scan<256>(s, tmp, &total);
    for (int i = 0; i < per; ++i) {
        const int j = b0 + i;
        if (j < nb_used) { const uint32_t c = row[j]; row[j] = ex; ex += c; }
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = total;
}

template <int B, int BLOCK, int ITEMS, bool FEW>
__global__ __launch_bounds__(BLOCK) void k_radix_downsweep(
    const uint32_t *__restrict__ keys_in, const uint32_t *__restrict__ vals_in,
    uint32_t *__restrict__ keys_out, uint32_t *__restrict__ vals_out,
    const int *__restrict__ n_dev, int n_host, int shift, const uint32_t *__restrict__ hist,
    const uint32_t *__restrict__ totals, int nb)
{
    constexpr int R = 1 << B, TILE = BLOCK * ITEMS, W = BLOCK / kWave, D = (R + BLOCK - 1) / BLOCK;
    __shared__ uint32_t wcnt[W][R];
    __shared__ uint32_t lstart[R];
    __shared__ int delta[R];
    __shared__ uint32_t skey[TILE];
    __shared__ uint32_t sval[TILE];
    __shared__ uint32_t tmp[W + 1];

    const int n = n_dev ? *n_dev : n_host;
    const long long tile0 = (long long)blockIdx.x * TILE;
    if (tile0 >= n) return;  // whole block leaves together

    const int tid = threadIdx.x, lane = tid & (kWave - 1), w = tid / kWave;
    // the digits' places are loaded with the keys: thread t holds digits t D ..
    uint32_t tot[D], before[D];
#pragma unroll
    for (int u = 0; u < D; ++u) {
        const int d = tid * D + u;
        if constexpr (FEW) {
            tot[u] = before[u] = 0u;
            continue;
        }
        tot[u] = d < R ? totals[d] : 0u;
        before[u] = d < R ? hist[(size_t)d * nb + blockIdx.x] : 0u;
    }
    if constexpr (FEW) {   // every tile's counts of this thread's digits
        const int used = (int)((n + (long long)TILE - 1) / TILE);   // tiles with data
        for (int b0 = 0; b0 < used; b0 += 8) {
            uint32_t c[8][D];
#pragma unroll
            for (int x = 0; x < 8; ++x)
#pragma unroll
                for (int u = 0; u < D; ++u) {
                    const int d = tid * D + u;
                    c[x][u] = b0 + x < used && d < R ? hist[(size_t)(b0 + x) * R + d] : 0u;
                }
#pragma unroll
            for (int x = 0; x < 8; ++x)
#pragma unroll
                for (int u = 0; u < D; ++u) {
                    tot[u] += c[x][u];
                    before[u] += b0 + x < (int)blockIdx.x ? c[x][u] : 0u;
                }
        }
    }
    for (int i = tid; i < W * R; i += BLOCK) (&wcnt[0][0])[i] = 0;

    uint32_t key[ITEMS], val[ITEMS], rank[ITEMS];
    const long long base = tile0 + w * (kWave * ITEMS) + lane;
    const uint64_t lt = lanemask_lt();
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const long long idx = base + k * kWave;
        const bool valid = idx < n;
        key[k] = valid ? keys_in[idx] : 0xFFFFFFFFu;
        val[k] = valid ? (vals_in ? vals_in[idx] : (uint32_t)idx) : 0u;
    }
    __syncthreads();   // counts cleared
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        const bool valid = base + k * kWave < n;
        const uint32_t d = (key[k] >> shift) & (R - 1);
        const uint64_t peers = match_bits<B>(d, __ballot(valid));
        const uint32_t prev = wcnt[w][d];
        // Lanes of one wave issue the read above before the leader's write below
        // (in-order LDS per wave; the write depends on the read).
        if (valid && (peers & lt) == 0) wcnt[w][d] = prev + (uint32_t)__popcll(peers);
        rank[k] = prev + (uint32_t)__popcll(peers & lt);
    }
    __syncthreads();

    // exclusive offsets across waves, per digit; the digits' first places in
    // the tile and in the output
    uint32_t cnt[D], csum = 0, tsum = 0;
#pragma unroll
    for (int u = 0; u < D; ++u) {
        const int d = tid * D + u;
        uint32_t run = 0;
        if (d < R) {
#pragma unroll
            for (int ww = 0; ww < W; ++ww) { const uint32_t c = wcnt[ww][d]; wcnt[ww][d] = run; run += c; }
        }
        cnt[u] = run;
        csum += run;
        tsum += tot[u];
    }
    uint32_t all;
    uint32_t lex = block_exclusive_scan<BLOCK>(csum, tmp, &all);
    uint32_t gex = block_exclusive_scan<BLOCK>(tsum, tmp, &all);
#pragma unroll
    for (int u = 0; u < D; ++u) {
        const int d = tid * D + u;
        if (d < R) {
            lstart[d] = lex;
            delta[d] = (int)(gex + before[u] - lex);
        }
        lex += cnt[u];
        gex += tot[u];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < ITEMS; ++k) {
        if (base + k * kWave < n) {
            const uint32_t d = (key[k] >> shift) & (R - 1);
            const uint32_t p = lstart[d] + wcnt[w][d] + rank[k];
            skey[p] = key[k];
            sval[p] = val[k];
        }
    }
    __syncthreads();
    const int m = (int)min((long long)TILE, n - tile0);
    for (int p = tid; p < m; p += BLOCK) {
        const uint32_t k = skey[p];
        const uint32_t g = (uint32_t)(p + delta[(k >> shift) & (R - 1)]);
        keys_out[g] = k;
        vals_out[g] = sval[p];
    }
}

// Digits of 10 bits where they save a pass and the pairs are few enough: a
// tile's runs of equal digits, which its writes are made of, are four times
// shorter than with 8 bits (2^20 keys of 20 bits 63 us against 72, of 26 bits
// 90 against 83; 4e6 of 24 bits 198 against 125; 1e5 of 20 bits 48 against 53).
// Tiles of 4096 pairs from 2^18 pairs on: runs twice as long (1.6e7 pairs of
// 31 bits 474 us against 644 with 2048), below that too few blocks.
constexpr int kWideBits = 10;
RadixPlan radix_plan(int n, int key_bits, int widest)
{
    RadixPlan p;
    const int p8 = std::max(1, div_up(key_bits, kRadixBits)), p10 = std::max(1, div_up(key_bits, kWideBits));
    const bool wide = widest >= kWideBits && p10 < p8 && n <= (p10 == 2 ? 3 << 19 : 1 << 18);
    p.bits = wide ? kWideBits : kRadixBits;
    p.passes = wide ? p10 : p8;
    p.block = wide || n >= 1 << 18 ? 512 : 256;
    return p;
}

size_t sort_scratch_bytes(int n_cap)
{
    const int n = n_cap > 0 ? n_cap : 1;
    const size_t wide = (size_t)kRadixMax * div_up(n, 512 * kSortItems), narrow = (size_t)kRadix * div_up(n, kSortTile);
    return (std::max(wide, narrow) + kRadixMax) * sizeof(uint32_t) + 256;
}

void sort_scratch_bind(SortScratch &s, int n_cap, void *mem, int digits)
{
    s.n_cap = n_cap;
    s.totals = (uint32_t *)mem;
    s.hist = s.totals + digits;
}

// Up to kFewTiles tiles a pass is two launches: every block of the downsweep
// adds up the tiles' counts itself (two passes: 1e3 pairs 60 -> 36 us, 3e4
// 60 -> 44, 1e5 62 -> 52; 2e5, 49 tiles, 60 to 64 either way).
constexpr int kFewTiles = 32;

template <int B, int BLOCK, int ITEMS>
static void radix_pass(const uint32_t *sk, const uint32_t *sv, uint32_t *dk, uint32_t *dv, const int *n_dev, int n,
                       int shift, const SortScratch &s, hipStream_t stream, Profiler *prof)
{
    const int nb = div_up(n > 0 ? n : 1, BLOCK * ITEMS), digits = 1 << B;
    if (nb <= kFewTiles) {
        DSMC_LAUNCH(prof, "radix_upsweep", (double)n * 4.0, (k_radix_upsweep<B, BLOCK, ITEMS, true>), nb, BLOCK,
                    stream, sk, n_dev, n, shift, s.hist, nb);
        DSMC_LAUNCH(prof, "radix_downsweep", (double)n * 16.0, (k_radix_downsweep<B, BLOCK, ITEMS, true>), nb, BLOCK,
                    stream, sk, sv, dk, dv, n_dev, n, shift, s.hist, s.totals, nb);
        return;
    }
    DSMC_LAUNCH(prof, "radix_upsweep", (double)n * 4.0, (k_radix_upsweep<B, BLOCK, ITEMS, false>), nb, BLOCK, stream,
                sk, n_dev, n, shift, s.hist, nb);
    DSMC_LAUNCH(prof, "radix_scan", (double)digits * nb * 8.0, k_radix_scan, digits, 256, stream, s.hist, s.totals,
                n_dev, n, BLOCK * ITEMS, nb);
    DSMC_LAUNCH(prof, "radix_downsweep", (double)n * 16.0, (k_radix_downsweep<B, BLOCK, ITEMS, false>), nb, BLOCK, stream,
                sk, sv, dk, dv, n_dev, n, shift, s.hist, s.totals, nb);
}

void radix_sort(const uint32_t *keys, const uint32_t *vals, uint32_t *keys_alt, uint32_t *vals_alt,
                uint32_t *keys_out, uint32_t *vals_out, const int *n_dev, const RadixPlan &plan,
                const SortScratch &s, hipStream_t stream, Profiler *prof)
{
    const uint32_t *sk = keys;
    const uint32_t *sv = vals;
    for (int p = 0; p < plan.passes; ++p) {
        const int q = plan.passes - 1 - p;  // passes still to go after this one
        uint32_t *dk = (q % 2 == 0) ? keys_out : keys_alt;
        uint32_t *dv = (q % 2 == 0) ? vals_out : vals_alt;
        const int shift = p * plan.bits;
        auto pass = plan.bits == kWideBits ? radix_pass<kWideBits, 512, kSortItems>
                    : plan.block == 512    ? radix_pass<kRadixBits, 512, kSortItems>
                                           : radix_pass<kRadixBits, 256, kSortItems>;
        pass(sk, sv, dk, dv, n_dev, s.n_cap, shift, s, stream, prof);
        sk = dk;
        sv = dv;
    }
}

// ---------------------------------------------------------------------------
// Incremental re-sort.  Input: slots that were in stable sorted order of
// key_old[0..n) (the previous sort's keys), their new keys, and what the move
// kernel left: per 64 slots a mask of the atoms whose key changed ("movers")
// and one of the removed atoms (dead key, which sorts last).  Output: the
// stable sort of the new keys by (key, slot) -- the same permutation a full
// radix sort gives -- in a buffer other than key_old.  Between time steps only
// the atoms that crossed a cell face change key (a few percent); the others
// ("stays") keep their order, so nothing is sorted but the movers, and the
// stays are never copied out of slot order:
//   * first phase (resort_list_block, in the finalize's launch): the movers and
//     removed atoms of every 2048-slot tile are counted, and every mover goes
//     to the bucket of its tile, the last one whose first (key, slot) lies
//     below its own: the next place of the bucket's fixed room of kBucketCap
//     entries or, beyond it, of an overflow list;
//   * merge (resort_merge_block): one block per tile adds up the counts of the
//     earlier tiles, finds its bucket's insertion points by binary search of
//     the tile's keys in LDS and ranks movers at the same point by counting
//     (buckets hold a few dozen; one beyond the LDS table of kBucketLds movers
//     is gathered and sorted in scratch), and writes the tile's stays and
//     movers to their final positions: with S = stays before the tile plus
//     movers in earlier buckets, a stay goes to S + (stays of the tile before
//     it) + (bucket movers inserted up to it), a mover of rank r to S + (stays
//     of the tile below its point) + r.  The tile's removed atoms go to the
//     end of the output, in slot order.  It also leaves the first key of
//     every tile of the new order, for the next move.
// Up to kScanSlots slots both run in the finalize's launch
// (resort_scan_merge_block): a tile's block reads the masks and the movers'
// new keys of all slots and keeps those of its bucket, so that nothing has to
// be finished by other blocks first.
// No kernel waits on another block.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_ins_merge(ResortMerge m)
{
    __shared__ MergeLds lds;
    resort_merge_block(m, (int)blockIdx.x, lds);
}

__global__ __launch_bounds__(256) void k_tile_samples(const uint32_t *__restrict__ sorted, int tiles,
                                                      uint32_t *__restrict__ tsamp)
{
    const int t = blockIdx.x * 256 + threadIdx.x;
    if (t < tiles) tsamp[t] = sorted[(size_t)t * kStayTile];   // past the slots: never used
}

// The buckets' fixed rooms (kBucketCap movers for each of the tiles), the
// overflow list, scratch for large buckets, and the counts.
size_t resort_scratch_bytes(int n_cap)
{
    const size_t n = (size_t)(n_cap > 0 ? n_cap : 1);
    const size_t tiles = (size_t)div_up((long long)n, kStayTile);
    return (3 * n + tiles * (size_t)kBucketCap) * sizeof(uint64_t) + (4 * (tiles + 8) + 4) * sizeof(uint32_t) +
           16 * 256;
}

void resort_scratch_bind(ResortScratch &r, int n_cap, void *mem)
{
    auto align = [](char *p) { return (char *)(((uintptr_t)p + 255) & ~(uintptr_t)255); };
    const size_t n = (size_t)(n_cap > 0 ? n_cap : 1);
    r.n_cap = (int)n;
    r.tiles = div_up((long long)n, kStayTile);
    const size_t row = ((size_t)r.tiles + 1 + 3) & ~(size_t)3;   // rows 16-byte aligned, an even number of tiles
    char *p = align((char *)mem);
    r.b.room = (uint64_t *)p; p = align(p + (size_t)r.tiles * kBucketCap * sizeof(uint64_t));
    r.b.over = (uint64_t *)p; p = align(p + n * sizeof(uint64_t));
    r.big = (uint64_t *)p; p = align(p + n * sizeof(uint64_t));
    r.big_alt = (uint64_t *)p; p = align(p + n * sizeof(uint64_t));
    r.alt_k = (uint32_t *)r.big_alt;
    r.alt_v = r.alt_k + n;
    r.tsamp = (uint32_t *)p; p = align(p + row * sizeof(uint32_t));
    r.b.tile_moved = (uint32_t *)p;
    r.b.tile_dead = r.b.tile_moved + row;
    r.b.bcnt = r.b.tile_dead + row;
    r.b.n_over = r.b.bcnt + row;
    r.b.n_counts = (int)row + 1;
    r.b.tsamp = r.tsamp;
}

bool resort_supported(int n_cap) { return (n_cap > 0 ? n_cap : 1) / kStayTile + 1 <= kMaxTiles; }

size_t resort_mask_words(int n_cap)
{
    // whole tiles and whole first-phase blocks, so that every word of a move
    // grid of blocks up to 2048 slots is inside
    return (size_t)resort_list_blocks(n_cap) * kListWords + kTileWords;
}

ResortList resort_list_args(const ResortScratch &r, const uint32_t *key_new, const int *n_dev,
                            const uint64_t *mask_m, const uint64_t *mask_d, bool may_remove)
{
    ResortList l;
    l.blocks = resort_list_blocks(r.n_cap);
    l.tiles = r.tiles; l.may_remove = may_remove ? 1 : 0;
    l.n_dev = n_dev;
    l.key_new = key_new;
    l.mask_m = mask_m; l.mask_d = mask_d;
    l.b = r.b;
    return l;
}

ResortMerge resort_merge_args(const ResortScratch &r, const uint32_t *key_old, const int *n_dev,
                              uint32_t dead_key, const uint64_t *mask_m, const uint64_t *mask_d,
                              bool may_remove, uint32_t *out_k, uint32_t *out_v)
{
    ResortMerge m;
    m.b = r.b;
    m.key_old = key_old;
    m.mask_m = mask_m; m.mask_d = mask_d;
    m.n_dev = n_dev;
    m.n_cap = r.n_cap; m.tiles = r.tiles; m.may_remove = may_remove ? 1 : 0;
    m.dead_key = dead_key;
    m.big = r.big; m.big_alt = r.big_alt;
    m.out_k = out_k; m.out_v = out_v;
    m.tsamp_out = r.tsamp;
    return m;
}

void resort_merge(const ResortMerge &m, hipStream_t stream, Profiler *prof)
{
    DSMC_LAUNCH(prof, "resort_merge", (double)m.n_cap * 12.0, k_ins_merge, m.tiles, 256, stream, m);
}

void resort_samples(const ResortScratch &r, const uint32_t *sorted, hipStream_t stream, Profiler *prof)
{
    DSMC_LAUNCH(prof, "resort_samples", (double)r.tiles * 8.0, k_tile_samples, div_up(r.tiles, 256), 256, stream,
                sorted, r.tiles, r.tsamp);
}

void resort_clear_counts(const ResortScratch &r, hipStream_t stream, Profiler *prof)
{
    fill_u32(r.b.bcnt, 0u, r.b.n_counts, stream, prof);
}

// ---------------------------------------------------------------------------
// Exclusive scan (int32)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kScanBlock) void k_scan_reduce(const int *__restrict__ in, int n,
                                                            int *__restrict__ partial)
{
    __shared__ int tmp[kScanBlock / kWave + 1];
    const int tile0 = blockIdx.x * kScanTile;
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const int i = tile0 + k * kScanBlock + threadIdx.x;
        if (i < n) s += in[i];
    }
    int total;
    (void)block_exclusive_scan<kScanBlock>(s, tmp, &total);
    if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

// Sum of partial[0 .. b) over the block's threads (every thread returns it).
__device__ __forceinline__ int sum_below(const int *__restrict__ partial, int b, int *tmp)
{
    int s = 0;
    for (int i0 = threadIdx.x; i0 < b; i0 += 4 * kScanBlock) {
        int c[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) c[u] = i0 + u * kScanBlock < b ? partial[i0 + u * kScanBlock] : 0;
#pragma unroll
        for (int u = 0; u < 4; ++u) s += c[u];
    }
    int total;
    (void)block_exclusive_scan<kScanBlock>(s, tmp, &total);
    return total;
}

// Sum of the tiles before tile b: partial holds the tiles' own sums, or
// (scanned) the sums before them.
__device__ __forceinline__ int tiles_before(const int *__restrict__ partial, int b, bool scanned, int *tmp)
{
    return scanned ? partial[b] : sum_below(partial, b, tmp);
}

// in and out may be the same array.
__global__ __launch_bounds__(kScanBlock) void k_scan_final(const int *in, int *out, int n,
                                                           const int *__restrict__ partial, bool scanned)
{
    __shared__ int tmp[kScanBlock / kWave + 1];
    const int t0 = blockIdx.x * kScanTile + threadIdx.x * kScanItems;
    int v[kScanItems];
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        v[k] = (t0 + k < n) ? in[t0 + k] : 0;
        s += v[k];
    }
    const int before = tiles_before(partial, (int)blockIdx.x, scanned, tmp);
    int total;
    int run = block_exclusive_scan<kScanBlock>(s, tmp, &total) + before;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        if (t0 + k < n) out[t0 + k] = run;
        run += v[k];
    }
}

// Scans the sums of more than kSumTiles tiles in place (partial's nb words and
// `extra` behind them); returns whether it did.
static bool scan_tiles(int *partial, int nb, int extra, hipStream_t stream, Profiler *prof);

int scan_partials(int n)
{
    const int nb = div_up(n > 0 ? n : 1, kScanTile);
    return nb + 1 + (nb > kSumTiles ? scan_partials(nb + 1) : 0);
}

void exclusive_scan(const int *in, int *out, int n, int *partial, hipStream_t stream,
                    Profiler *prof)
{
    if (n <= 0) return;
    const int nb = div_up(n, kScanTile);
    DSMC_LAUNCH(prof, "scan_reduce", (double)n * 4.0, k_scan_reduce, nb, kScanBlock, stream,
                in, n, partial);
    const bool scanned = scan_tiles(partial, nb, 0, stream, prof);
    DSMC_LAUNCH(prof, "scan_final", (double)n * 8.0, k_scan_final, nb, kScanBlock, stream, in,
                out, n, (const int *)partial, scanned);
}

static bool scan_tiles(int *partial, int nb, int extra, hipStream_t stream, Profiler *prof)
{
    if (nb <= kSumTiles) return false;
    exclusive_scan(partial, partial, nb + extra, partial + nb + 1, stream, prof);
    return true;
}

// ---------------------------------------------------------------------------
// Removal in place (thrust::remove_if): every block compacts its tile's kept
// values into tmp, then moves them to their place behind the earlier tiles'.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kScanBlock) void k_remove_tile(const int *__restrict__ values,
                                                            const int *__restrict__ stencil, int n,
                                                            int *__restrict__ tmp_out, int *__restrict__ partial)
{
    constexpr int W = kScanBlock / kWave;
    __shared__ int wtot[W];
    __shared__ int kept[kScanTile];
    const int tile0 = blockIdx.x * kScanTile;
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int base = tile0 + w * (kWave * kScanItems) + lane;
    const uint64_t lt = lanemask_lt();
    int v[kScanItems], rank[kScanItems];
    bool keep[kScanItems];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const int i = base + k * kWave;
        v[k] = i < n ? values[i] : 0;
        keep[k] = i < n && stencil[i] == 0;
    }
    int run = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const uint64_t b = __ballot(keep[k]);
        rank[k] = run + __popcll(b & lt);
        run += __popcll(b);
    }
    if (lane == 0) wtot[w] = run;
    __syncthreads();
    int off = 0, all = 0;
#pragma unroll
    for (int ww = 0; ww < W; ++ww) {
        if (ww < w) off += wtot[ww];
        all += wtot[ww];
    }
#pragma unroll
    for (int k = 0; k < kScanItems; ++k)
        if (keep[k]) kept[off + rank[k]] = v[k];
    __syncthreads();
    for (int i = threadIdx.x; i < all; i += kScanBlock) tmp_out[tile0 + i] = kept[i];
    if (threadIdx.x == 0) partial[blockIdx.x] = all;
    if (threadIdx.x == 0 && blockIdx.x == 0) partial[gridDim.x] = 0;   // (scanned, the total)
}

__global__ __launch_bounds__(kScanBlock) void k_remove_place(const int *__restrict__ tmp_in,
                                                             const int *__restrict__ partial, int nb, bool scanned,
                                                             int *__restrict__ values, int *__restrict__ kept)
{
    __shared__ int tmp[kScanBlock / kWave + 1];
    const int before = tiles_before(partial, (int)blockIdx.x, scanned, tmp);
    const int m = scanned ? partial[blockIdx.x + 1] - before : partial[blockIdx.x];
    const int *src = tmp_in + (size_t)blockIdx.x * kScanTile;
    for (int i = threadIdx.x; i < m; i += kScanBlock) values[before + i] = src[i];
    if ((int)blockIdx.x == nb - 1 && threadIdx.x == 0) *kept = before + m;
}

void remove_if(int *values, const int *stencil, int n, int *tmp, int *partial, int *kept, hipStream_t stream)
{
    const int nb = div_up(n > 0 ? n : 1, kScanTile);
    hipLaunchKernelGGL(k_remove_tile, dim3(nb), dim3(kScanBlock), 0, stream, values, stencil, n, tmp, partial);
    DSMC_HIP(hipGetLastError());
    const bool scanned = scan_tiles(partial, nb, 1, stream, nullptr);
    hipLaunchKernelGGL(k_remove_place, dim3(nb), dim3(kScanBlock), 0, stream, tmp, partial, nb, scanned,
                       values, kept);
    DSMC_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Stable compaction map
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kScanBlock) void k_compact_count(const int *__restrict__ stencil,
                                                              const int *__restrict__ n_dev,
                                                              int *__restrict__ partial)
{
    __shared__ int tmp[kScanBlock / kWave + 1];
    const int n = *n_dev;
    const int tile0 = blockIdx.x * kScanTile;
    int s = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const int i = tile0 + k * kScanBlock + threadIdx.x;
        if (i < n) s += stencil[i] == 0;
    }
    int total;
    (void)block_exclusive_scan<kScanBlock>(s, tmp, &total);
    if (threadIdx.x == 0) partial[blockIdx.x] = total;
    if (threadIdx.x == 0 && blockIdx.x == 0) partial[gridDim.x] = 0;   // (scanned, the total)
}

__global__ __launch_bounds__(kScanBlock) void k_compact_scatter(
    const int *__restrict__ stencil, const int *__restrict__ n_dev,
    const int *__restrict__ partial, bool scanned, uint32_t *__restrict__ map, int *__restrict__ n_out,
    int nb)
{
    constexpr int W = kScanBlock / kWave;
    __shared__ int wtot[W];
    __shared__ int tmp[W + 1];
    const int n = *n_dev;
    const int tile0 = blockIdx.x * kScanTile;
    const bool last = (int)blockIdx.x == nb - 1;
    if (tile0 >= n && !last) return;
    const int before = tiles_before(partial, (int)blockIdx.x, scanned, tmp);
    if (last && threadIdx.x == 0) *n_out = scanned ? partial[nb] : before + partial[blockIdx.x];
    if (tile0 >= n) return;
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int base = tile0 + w * (kWave * kScanItems);
    const uint64_t lt = lanemask_lt();
    uint32_t rank[kScanItems];
    bool keep[kScanItems];
    int run = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k) {
        const int i = base + k * kWave + lane;
        keep[k] = i < n && stencil[i] == 0;
        const uint64_t b = __ballot(keep[k]);
        rank[k] = run + __popcll(b & lt);
        run += __popcll(b);
    }
    if (lane == 0) wtot[w] = run;
    __syncthreads();
    int off = before;
    for (int ww = 0; ww < w; ++ww) off += wtot[ww];
#pragma unroll
    for (int k = 0; k < kScanItems; ++k)
        if (keep[k]) map[off + rank[k]] = (uint32_t)(base + k * kWave + lane);
}

void compaction_map(const int *stencil, const int *n_dev, int n_cap, uint32_t *map,
                    int *n_out_dev, int *partial, hipStream_t stream, Profiler *prof)
{
    const int nb = div_up(n_cap > 0 ? n_cap : 1, kScanTile);
    DSMC_LAUNCH(prof, "compact_count", (double)n_cap * 4.0, k_compact_count, nb, kScanBlock,
                stream, stencil, n_dev, partial);
    const bool scanned = scan_tiles(partial, nb, 1, stream, prof);
    DSMC_LAUNCH(prof, "compact_scatter", (double)n_cap * 8.0, k_compact_scatter, nb, kScanBlock,
                stream, stencil, n_dev, (const int *)partial, scanned, map, n_out_dev, nb);
}

__global__ __launch_bounds__(256) void k_gather_u32(uint32_t *__restrict__ dst,
                                                    const uint32_t *__restrict__ src,
                                                    const uint32_t *__restrict__ map,
                                                    const int *__restrict__ n_dev, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < (n_dev ? *n_dev : n)) dst[i] = src[map[i]];
}

void gather_u32(uint32_t *dst, const uint32_t *src, const uint32_t *map, const int *n_dev,
                int n_cap, hipStream_t stream, Profiler *prof)
{
    DSMC_LAUNCH(prof, "gather_u32", (double)n_cap * 12.0, k_gather_u32, div_up(n_cap > 0 ? n_cap : 1, 256),
                256, stream, dst, src, map, n_dev, n_cap);
}

// ---------------------------------------------------------------------------
// Fills and Philox
// ---------------------------------------------------------------------------
__global__ void k_fill_u32(uint32_t *p, uint32_t v, long long n)
{
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n;
         i += (long long)gridDim.x * blockDim.x)
        p[i] = v;
}

static int fill_grid(long long n) { return (int)std::min<long long>(4096, (n + 255) / 256 + 1); }

void fill_u32(uint32_t *p, uint32_t v, long long n, hipStream_t stream, Profiler *prof)
{
    if (n <= 0) return;
    DSMC_LAUNCH(prof, "fill", (double)n * 4.0, k_fill_u32, fill_grid(n), 256, stream, p, v, n);
}

// Streaming copy for counter calibration: four 16-byte vectors per thread
// and round, loads issued together, non-temporal loads and stores (each byte
// is touched once), grid-stride over whole rounds.
constexpr int kCopyUnroll = 4;
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(256) void k_stream_copy(const u32x4 *__restrict__ src,
                                                     u32x4 *__restrict__ dst, long long n16)
{
    const long long stride = (long long)gridDim.x * 256 * kCopyUnroll;
    for (long long i0 = (long long)blockIdx.x * 256 * kCopyUnroll + threadIdx.x; i0 < n16; i0 += stride) {
        u32x4 v[kCopyUnroll];
#pragma unroll
        for (int u = 0; u < kCopyUnroll; ++u) {
            const long long i = i0 + (long long)u * 256;
            if (i < n16) v[u] = __builtin_nontemporal_load(src + i);
        }
#pragma unroll
        for (int u = 0; u < kCopyUnroll; ++u) {
            const long long i = i0 + (long long)u * 256;
            if (i < n16) __builtin_nontemporal_store(v[u], dst + i);
        }
    }
}

void stream_copy(void *dst, const void *src, size_t bytes, hipStream_t stream)
{
    const long long n16 = (long long)(bytes / 16);
    if (n16 <= 0) return;
    const int grid = (int)std::min<long long>((n16 + 256 * kCopyUnroll - 1) / (256 * kCopyUnroll), 8192LL);
    hipLaunchKernelGGL(k_stream_copy, dim3(grid), dim3(256), 0, stream, (const u32x4 *)src,
                       (u32x4 *)dst, n16);
    DSMC_HIP(hipGetLastError());
}

// Gather of the FP32 state's tiled 16-byte records (three planes of 64
// records per 64-slot tile) through a slot map: record planes of slot i of
// dst = those of slot map[i] of src.  The access pattern of the fused move's
// state gather, for calibrating the traffic counters on it: 4 bytes of map
// and 48 bytes of records read, 48 bytes written per slot.
__global__ __launch_bounds__(256) void k_gather_copy(const u32x4 *__restrict__ src,
                                                     u32x4 *__restrict__ dst,
                                                     const uint32_t *__restrict__ map, int n)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint32_t j = __builtin_nontemporal_load(map + i);
    const size_t qs = (size_t)(j / 64) * 192 + (j % 64), qd = (size_t)(i / 64) * 192 + (i % 64);
    const u32x4 a = __builtin_nontemporal_load(src + qs), b = __builtin_nontemporal_load(src + qs + 64),
                c = __builtin_nontemporal_load(src + qs + 128);
    __builtin_nontemporal_store(a, dst + qd);
    __builtin_nontemporal_store(b, dst + qd + 64);
    __builtin_nontemporal_store(c, dst + qd + 128);
}

void gather_copy(void *dst, const void *src, const uint32_t *map, int n, hipStream_t stream)
{
    if (n <= 0) return;
    hipLaunchKernelGGL(k_gather_copy, dim3(div_up(n, 256)), dim3(256), 0, stream, (const u32x4 *)src,
                       (u32x4 *)dst, map, n);
    DSMC_HIP(hipGetLastError());
}

__global__ void k_philox_fill(uint32_t *out, int n, U32x4 ctr, uint32_t k0, uint32_t k1)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    U32x4 c = { ctr.x + (uint32_t)i, ctr.y, ctr.z, ctr.w };
    U32x4 o = philox(c, k0, k1);
    out[4 * i + 0] = o.x;
    out[4 * i + 1] = o.y;
    out[4 * i + 2] = o.z;
    out[4 * i + 3] = o.w;
}

void philox_fill(uint32_t *out, int n, const uint32_t ctr[4], const uint32_t key[2],
                 hipStream_t stream)
{
    if (n <= 0) return;
    U32x4 c = { ctr[0], ctr[1], ctr[2], ctr[3] };
    hipLaunchKernelGGL(k_philox_fill, dim3(div_up(n, 256)), dim3(256), 0, stream, out, n, c,
                       key[0], key[1]);
    DSMC_HIP(hipGetLastError());
}

}  // namespace dsmc
