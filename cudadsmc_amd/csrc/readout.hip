// readout.hip -- see readout.hpp.  Every kernel here touches each byte once and
// is bound by the memory it streams; the copy over the host link that
// follows takes some forty times longer (24 bytes per atom and field at 39
// GB/s into pageable memory against 72 bytes at 5 TB/s here).  Before these
// kernels the host unpacked the records itself, one strided read per
// component: N = 4e6, position, velocity and labels took 292 ms, now 6.7 ms.
#include "readout.hpp"

namespace dsmc {

constexpr int kRBlock = 256;

static int rgrid(long long n) { return div_up(n > 0 ? n : 1, kRBlock); }

#define DSMC_READOUT(kernel, n, st, ...)                                                             \
    do {                                                                                             \
        if ((n) > 0) {                                                                               \
            hipLaunchKernelGGL(kernel, dim3(rgrid(n)), dim3(kRBlock), 0, (st), __VA_ARGS__);         \
            DSMC_HIP(hipGetLastError());                                                             \
        }                                                                                            \
    } while (0)

template <RecVec W>
__global__ __launch_bounds__(kRBlock) void k_pack_records(const f4 *__restrict__ r,
                                                          const uint32_t *__restrict__ map, int n,
                                                          double *__restrict__ out)
{
    const int i = blockIdx.x * kRBlock + threadIdx.x;
    if (i >= n) return;
    constexpr bool pos = W == RecVec::Pos || W == RecVec::PosRem;
    constexpr bool rem = W == RecVec::PosRem || W == RecVec::VelRem;
    const f4 *q = r + rec_index(map ? map[i] : (uint32_t)i);
    const f4 hi = q[pos ? 0 : kRecTile], p2 = q[2 * kRecTile];
    const float l[3] = { pos ? rem_value(hi.w) : hi.w, pos ? rem_value(p2.x) : p2.z,
                         pos ? rem_value(p2.y) : p2.w };
    double *o = out + 3 * (size_t)i;
#pragma unroll
    for (int c = 0; c < 3; ++c) o[c] = rem ? (double)l[c] : (double)hi[c] + (double)l[c];
}

void launch_pack_records(RecVec what, const FusedPtrs &s, const uint32_t *map, int n, double *out,
                         hipStream_t st)
{
    switch (what) {
    case RecVec::Pos: DSMC_READOUT(k_pack_records<RecVec::Pos>, n, st, s.r, map, n, out); break;
    case RecVec::Vel: DSMC_READOUT(k_pack_records<RecVec::Vel>, n, st, s.r, map, n, out); break;
    case RecVec::PosRem: DSMC_READOUT(k_pack_records<RecVec::PosRem>, n, st, s.r, map, n, out); break;
    case RecVec::VelRem: DSMC_READOUT(k_pack_records<RecVec::VelRem>, n, st, s.r, map, n, out); break;
    }
}

__global__ __launch_bounds__(kRBlock) void k_pack_labels(const f4 *__restrict__ r,
                                                         const uint32_t *__restrict__ map, int n,
                                                         int *__restrict__ out)
{
    const int i = blockIdx.x * kRBlock + threadIdx.x;
    if (i >= n) return;
    const f4 *q = r + rec_index(map ? map[i] : (uint32_t)i);
    const f4 p2 = q[2 * kRecTile];
    out[i] = rec_label(q[0].w, p2.x, p2.y);
}

void launch_pack_labels(const FusedPtrs &s, const uint32_t *map, int n, int *out, hipStream_t st)
{
    DSMC_READOUT(k_pack_labels, n, st, s.r, map, n, out);
}

__global__ __launch_bounds__(kRBlock) void k_unpack_records(const double *__restrict__ pos,
                                                            const double *__restrict__ vel, int n,
                                                            f4 *__restrict__ r)
{
    const int i = blockIdx.x * kRBlock + threadIdx.x;
    if (i >= n) return;
    float ph[3], pl[3], vh[3], vl[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const double p = pos[3 * (size_t)i + c], v = vel[3 * (size_t)i + c];
        ph[c] = (float)p; pl[c] = (float)(p - (double)ph[c]);
        vh[c] = (float)v; vl[c] = (float)(v - (double)vh[c]);
    }
    const FState a = { ph[0], ph[1], ph[2], pl[0], vh[0], vh[1], vh[2], vl[0], pl[1], pl[2], vl[1], vl[2] };
    rec_store(r, (uint32_t)i, a, i);
}

void launch_unpack_records(const double *pos, const double *vel, int n, const FusedPtrs &s, hipStream_t st)
{
    DSMC_READOUT(k_unpack_records, n, st, pos, vel, n, s.r);
}

// Up to four columns between AoS rows of doubles and SoA arrays of T.
template <typename T>
struct Columns { T *c[4]; };

template <typename T>
__global__ __launch_bounds__(kRBlock) void k_pack_columns(Columns<const T> cols, int ncols,
                                                          const uint32_t *__restrict__ map, int n,
                                                          double *__restrict__ out)
{
    const int i = blockIdx.x * kRBlock + threadIdx.x;
    if (i >= n) return;
    const uint32_t j = map ? map[i] : (uint32_t)i;
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (c < ncols) out[(size_t)i * ncols + c] = (double)cols.c[c][j];
}

template <typename T>
__global__ __launch_bounds__(kRBlock) void k_unpack_columns(const double *__restrict__ in, int ncols,
                                                            const uint32_t *__restrict__ map, int n,
                                                            Columns<T> cols)
{
    const int i = blockIdx.x * kRBlock + threadIdx.x;
    if (i >= n) return;
    const uint32_t j = map ? map[i] : (uint32_t)i;
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (c < ncols) cols.c[c][j] = (T)in[(size_t)i * ncols + c];
}

template <typename T, typename P>
static Columns<T> columns(P *const *cols, int ncols)
{
    Columns<T> k = {};
    for (int c = 0; c < ncols; ++c) k.c[c] = cols[c];
    return k;
}

void launch_pack_columns(const double *const *cols, int ncols, int n, double *out, hipStream_t st)
{
    DSMC_READOUT(k_pack_columns<double>, n, st, columns<const double>(cols, ncols), ncols,
                 (const uint32_t *)nullptr, n, out);
}

void launch_pack_columns(const float *const *cols, int ncols, const uint32_t *map, int n, double *out,
                         hipStream_t st)
{
    DSMC_READOUT(k_pack_columns<float>, n, st, columns<const float>(cols, ncols), ncols, map, n, out);
}

void launch_unpack_columns(const double *in, int ncols, int n, double *const *cols, hipStream_t st)
{
    DSMC_READOUT(k_unpack_columns<double>, n, st, in, ncols, (const uint32_t *)nullptr, n,
                 columns<double>(cols, ncols));
}

void launch_unpack_columns(const double *in, int ncols, const uint32_t *map, int n, float *const *cols,
                           hipStream_t st)
{
    DSMC_READOUT(k_unpack_columns<float>, n, st, in, ncols, map, n, columns<float>(cols, ncols));
}

__global__ __launch_bounds__(kRBlock) void k_widen_f(const float *__restrict__ in, long long n,
                                                     double *__restrict__ out)
{
    const long long i = (long long)blockIdx.x * kRBlock + threadIdx.x;
    if (i < n) out[i] = (double)in[i];
}

void launch_widen(const float *in, long long n, double *out, hipStream_t st)
{
    DSMC_READOUT(k_widen_f, n, st, in, n, out);
}

__global__ __launch_bounds__(kRBlock) void k_iota(int *__restrict__ out, int n)
{
    const int i = blockIdx.x * kRBlock + threadIdx.x;
    if (i < n) out[i] = i;
}

void launch_iota(int *out, int n, hipStream_t st) { DSMC_READOUT(k_iota, n, st, out, n); }

__global__ __launch_bounds__(kRBlock) void k_dead_stencil(const uint32_t *__restrict__ key,
                                                          const int *__restrict__ n_dev,
                                                          uint32_t dead_key, int *__restrict__ stencil)
{
    const int i = blockIdx.x * kRBlock + threadIdx.x;
    if (i < *n_dev) stencil[i] = key[i] == dead_key ? 1 : 0;
}

void launch_dead_stencil(const uint32_t *key, const int *n_dev, int n_cap, uint32_t dead_key, int *stencil,
                         hipStream_t st)
{
    DSMC_READOUT(k_dead_stencil, n_cap, st, key, n_dev, dead_key, stencil);
}

// One thread per key; its trap by a binary search of the key bases (a block's
// 256 keys share the search's cache lines).
template <typename T>
__global__ __launch_bounds__(kRBlock) void k_init_sigvrmax(const TrapDev *__restrict__ traps,
                                                           const int *__restrict__ key_base, int n_traps,
                                                           int n_keys, T *__restrict__ out)
{
    const int k = blockIdx.x * kRBlock + threadIdx.x;
    if (k >= n_keys) return;
    if (k >= key_base[n_traps]) { out[k] = (T)0; return; }
    int lo = 0, hi = n_traps - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (key_base[mid] <= k) lo = mid; else hi = mid - 1;
    }
    out[k] = (T)traps[lo].sigvrmax0;
}

void launch_init_sigvrmax(const TrapDev *traps, const int *key_base, int n_traps, int n_keys, double *out,
                          hipStream_t st)
{
    DSMC_READOUT(k_init_sigvrmax<double>, n_keys, st, traps, key_base, n_traps, n_keys, out);
}

void launch_init_sigvrmax(const TrapDev *traps, const int *key_base, int n_traps, int n_keys, float *out,
                          hipStream_t st)
{
    DSMC_READOUT(k_init_sigvrmax<float>, n_keys, st, traps, key_base, n_traps, n_keys, out);
}

}  // namespace dsmc
