// dsmc_internal.hpp -- host-side internals shared by the library's
// translation units: launch bookkeeping (optional per-kernel hipEvent timing),
// error propagation, and the device-primitive launchers (radix sort, scan,
// compaction) that both numerical forms use.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <map>
#include <stdexcept>
#include <string>
#include <vector>

namespace dsmc {

// Thrown inside the library only; every extern "C" entry point catches it and
// converts it into a dsmc_status plus a message.
struct Error : std::runtime_error {
    int status;
    Error(int s, const std::string &m) : std::runtime_error(m), status(s) {}
};

void hip_check(hipError_t e, const char *what, const char *file, int line);
#define DSMC_HIP(call) ::dsmc::hip_check((call), #call, __FILE__, __LINE__)

// Per-kernel timing with hipEvents on the launch stream.
class Profiler {
public:
    bool enabled = false;
    void begin(hipStream_t s, const char *name, double bytes);
    void end(hipStream_t s);
    // Resolve pending events (synchronises) and fold them into the totals.
    void collect();
    void reset();
    struct Stat { long long launches = 0; double total_ms = 0.0; double bytes = 0.0; };
    const std::map<std::string, Stat> &stats() const { return stats_; }
    ~Profiler();

private:
    struct Rec { std::string name; double bytes; hipEvent_t b, e; };
    std::vector<Rec> pending_;
    std::vector<hipEvent_t> pool_;
    std::map<std::string, Stat> stats_;
    hipEvent_t take();
};

// Launch `kernel` with optional profiling.  `bytes` is the algorithmic byte
// count of this launch (used only for reporting).
#define DSMC_LAUNCH(prof, name, bytes, kernel, grid, block, stream, ...)            \
    do {                                                                            \
        ::dsmc::Profiler *p_ = (prof);                                              \
        if (p_ && p_->enabled) p_->begin((stream), (name), (double)(bytes));        \
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), 0, (stream), __VA_ARGS__); \
        DSMC_HIP(hipGetLastError());                                                \
        if (p_ && p_->enabled) p_->end((stream));                                   \
    } while (0)

// ---------------------------------------------------------------------------
// Device primitives (primitives.hip).
// ---------------------------------------------------------------------------
constexpr int kRadixBits = 8;
constexpr int kRadix = 1 << kRadixBits;
constexpr int kSortBlock = 256;
constexpr int kSortItems = 8;
constexpr int kSortTile = kSortBlock * kSortItems;
constexpr int kScanBlock = 256;
constexpr int kScanItems = 8;
constexpr int kScanTile = kScanBlock * kScanItems;

inline int div_up(long long a, long long b) { return (int)((a + b - 1) / b); }

// How a radix sort goes over its keys: `passes` passes over digits of `bits`
// bits, in tiles of block * kSortItems pairs.
struct RadixPlan { int bits, passes, block; };
constexpr int kRadixMax = 1 << 10;
// The plan for n pairs with keys in [0, 2^key_bits); digits of at most
// `widest` bits.
RadixPlan radix_plan(int n, int key_bits, int widest = 10);

// Scratch for a radix sort of up to n_cap pairs with at most `digits` digits.
struct SortScratch {
    int n_cap = 0;
    uint32_t *totals = nullptr;   // digits
    uint32_t *hist = nullptr;     // digits * tiles
};
size_t sort_scratch_bytes(int n_cap);
void sort_scratch_bind(SortScratch &s, int n_cap, void *mem, int digits = kRadixMax);

// Stable LSD radix sort of keys[0..n) with values (identity slot indices when
// vals == nullptr).  n is read from device memory (n_dev null: s.n_cap).  The
// sorted result lands in (keys_out, vals_out); ping-pong through (keys_alt,
// vals_alt) for the intermediate passes.
void radix_sort(const uint32_t *keys, const uint32_t *vals, uint32_t *keys_alt,
                uint32_t *vals_alt, uint32_t *keys_out, uint32_t *vals_out,
                const int *n_dev, const RadixPlan &plan, const SortScratch &s,
                hipStream_t stream, Profiler *prof);

// Incremental re-sort (see primitives.hip): the stable sort of a state's new
// keys by (key, slot), for slots in stable sorted order of key_old, into out
// (which must not alias key_old).  dead_key sorts last.  Slots are grouped in
// tiles of kResortTile.
constexpr int kResortTile = 2048;
// What the first phase leaves for the merge: the movers in buckets and the
// movers and removed atoms per tile.  tsamp: first key of every tile of the
// order that the slots are in.
struct ResortBuckets {
    const uint32_t *tsamp = nullptr;
    uint32_t *tile_moved = nullptr;
    uint32_t *tile_dead = nullptr;
    uint32_t *bcnt = nullptr;         // movers per bucket; cleared with n_over: n_counts words from here
    uint32_t *n_over = nullptr;       // movers in the overflow list
    uint64_t *room = nullptr;         // the buckets' fixed rooms (key << 32 | slot)
    uint64_t *over = nullptr;
    int n_counts = 0;
};
// One first phase: the n_dev slots' new keys and the move's masks of the atoms
// whose key changed and of the removed ones.  blocks = 0: none.
struct ResortList {
    int blocks = 0;
    int tiles = 0, may_remove = 1;
    const int *n_dev = nullptr;
    const uint32_t *key_new = nullptr;
    const uint64_t *mask_m = nullptr, *mask_d = nullptr;
    ResortBuckets b;
};
struct ResortScratch {
    int n_cap = 0, tiles = 0;
    ResortBuckets b;
    uint32_t *tsamp = nullptr;        // b.tsamp, for its writers
    uint64_t *big = nullptr, *big_alt = nullptr;        // buckets larger than the merge's LDS table
    uint32_t *alt_k = nullptr, *alt_v = nullptr;        // the radix sort's alternates (share big_alt)
};
// One merge: n_dev slots in sorted order of key_old, the move's masks of the
// movers and removed atoms; may_remove = 0: no atom can have been removed.
struct ResortMerge {
    ResortBuckets b;
    const uint32_t *key_old = nullptr;
    const uint64_t *mask_m = nullptr, *mask_d = nullptr;
    const int *n_dev = nullptr;
    int n_cap = 0, tiles = 0, may_remove = 1;
    uint32_t dead_key = 0;
    const uint32_t *key_new = nullptr;   // (without a first phase) the new keys
    uint64_t *big = nullptr, *big_alt = nullptr;
    uint32_t *out_k = nullptr, *out_v = nullptr;
    uint32_t *tsamp_out = nullptr;
};
size_t resort_scratch_bytes(int n_cap);
void resort_scratch_bind(ResortScratch &r, int n_cap, void *mem);
bool resort_supported(int n_cap);
// 64-bit words of each of the mover and removal masks for n_cap slots.
size_t resort_mask_words(int n_cap);
ResortList resort_list_args(const ResortScratch &r, const uint32_t *key_new, const int *n_dev,
                            const uint64_t *mask_m, const uint64_t *mask_d, bool may_remove);
ResortMerge resort_merge_args(const ResortScratch &r, const uint32_t *key_old, const int *n_dev,
                              uint32_t dead_key, const uint64_t *mask_m, const uint64_t *mask_d,
                              bool may_remove, uint32_t *out_k, uint32_t *out_v);
void resort_merge(const ResortMerge &m, hipStream_t stream, Profiler *prof);
// Largest capacity whose merge needs no first phase (its blocks read all the
// masks and all the movers' new keys) and runs in the finalize's launch: three
// launches a step instead of four, N = 2e3 21.1 -> 19.2 us, 1e4 23.2 -> 20.8,
// 2e4 24.0 -> 22.1 (FP64 21.9 -> 20.2) when it was taken.  The gain shrinks
// with the movers that every block reads, and two mask words per thread end
// here.
constexpr int kScanSlots = 32768;
// What a finalize launch runs beside its sums: the first phase of a re-sort,
// a whole one (merge.tiles > 0), or neither.
struct ResortWork {
    ResortList list;
    ResortMerge merge;
    int blocks() const { return merge.tiles > 0 ? merge.tiles : list.blocks; }
};
// After a full sort: the first keys of the tiles of the sorted order.
void resort_samples(const ResortScratch &r, const uint32_t *sorted, hipStream_t stream, Profiler *prof);
// Clears the buckets' counts (a collide after the merge does it otherwise).
void resort_clear_counts(const ResortScratch &r, hipStream_t stream, Profiler *prof);

// Exclusive scan of n ints (n known on the host; in and out may be the same);
// partial holds scan_partials(n).
void exclusive_scan(const int *in, int *out, int n, int *partial, hipStream_t stream,
                    Profiler *prof);
// Up to kSumTiles tiles every block of a scan, a removal or a compaction map
// adds up the tiles before its own itself; beyond, where that grows with the
// square of the tiles, their sums are scanned first, in two more launches
// (added up / scanned first, us: scan of 1e6 elements 20 / 24, 1.6e7 87 / 93,
// 3.2e7 163 / 162, 6.4e7 384 / 323, 2.56e8 2230 / 1190, 1e9 18500 / 4500;
// removal of 1.6e7 58 / 60, 3.2e7 123 / 114, 2.56e8 2350 / 1160).
constexpr int kSumTiles = 12288;
int scan_partials(int n);

// Stable compaction map: for stencil[i] == 0 (kept), map[j] = i for the j-th
// kept element; *n_out (device) = number kept.  n read from device memory;
// n_cap bounds the grid.  partial holds scan_partials(n_cap).
void compaction_map(const int *stencil, const int *n_dev, int n_cap, uint32_t *map,
                    int *n_out_dev, int *partial, hipStream_t stream, Profiler *prof);

// Stable in-place removal of the values with a non-zero stencil; *kept (device
// or pinned host memory) receives how many stay.  tmp holds n ints, partial
// scan_partials(n).
void remove_if(int *values, const int *stencil, int n, int *tmp, int *partial, int *kept, hipStream_t stream);

// dst[i] = src[map[i]] for i < *n_dev (i < n_cap when n_dev is null).
void gather_u32(uint32_t *dst, const uint32_t *src, const uint32_t *map, const int *n_dev,
                int n_cap, hipStream_t stream, Profiler *prof);

void fill_u32(uint32_t *p, uint32_t v, long long n, hipStream_t stream, Profiler *prof);

// Streaming device-to-device copy of bytes (multiple of 16) for counter
// calibration.
void stream_copy(void *dst, const void *src, size_t bytes, hipStream_t stream);
// Gather of n slots of the FP32 state's tiled records (48 bytes a slot, in
// whole 64-slot tiles) through map, for counter calibration.
void gather_copy(void *dst, const void *src, const uint32_t *map, int n, hipStream_t stream);

void philox_fill(uint32_t *out, int n, const uint32_t ctr[4], const uint32_t key[2],
                 hipStream_t stream);

}  // namespace dsmc
