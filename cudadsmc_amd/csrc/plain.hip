// plain.hip -- FP64 drop-in form of the DSMC step, one kernel per reference
// call, structure-of-arrays state kept physically in cell order.
//
// The reference keeps AoS double3 state fixed in memory and permutes an atomID
// indirection list (main.cu:88-140), so after the first sort every per-atom
// kernel gathers through atomID.  Here the state itself is gathered into sorted
// order after each sort (k_gather_plain), so every per-atom kernel streams
// contiguous SoA arrays and collide reads each cell's atoms contiguously; the
// slot -> atom label map is carried along as `id`.
#include "dsmc_device.hpp"
#include "dsmc_internal.hpp"
#include "plain_device.hpp"

namespace dsmc {

constexpr int kBlock = 256;

// ---------------------------------------------------------------------------
// indexAtoms -> findAtomIndex (collisions.cu:163-185): key[slot].
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_index_plain(TrapDev t, const double *__restrict__ x,
                                                        const double *__restrict__ y,
                                                        const double *__restrict__ z,
                                                        uint32_t *__restrict__ key,
                                                        const int *__restrict__ n_dev)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < *n_dev) key[i] = (uint32_t)(t.key_base + cell_of(t, x[i], y[i], z[i]));
}

// Gather every state array through `map` (dst[i] = src[map[i]]).  n_out,
// n_host (pinned; when not null) receive the count.
__global__ __launch_bounds__(kBlock) void k_gather_plain(PlainPtrs dst, PlainPtrs src,
                                                         const uint32_t *__restrict__ map,
                                                         const int *__restrict__ n_dev, int spin,
                                                         int *__restrict__ n_out, int *__restrict__ n_host)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const int n = *n_dev;
    if (i == 0) {
        if (n_out) *n_out = n;
        if (n_host) *n_host = n;
    }
    if (i >= n) return;
    const uint32_t j = map[i];
#pragma unroll
    for (int c = 0; c < 9; ++c) dst.d[c][i] = src.d[c][j];
    dst.id[i] = src.id[j];
    dst.up[i] = src.up[j];
    if (spin) {
#pragma unroll
        for (int c = 0; c < 4; ++c) dst.psi[c][i] = src.psi[c][j];
    }
}

// ---------------------------------------------------------------------------
// Cell table (main.cu:426-442; collisions.cu:228-271).
// ---------------------------------------------------------------------------
// First slot with a key of at least c, of n slots with ascending keys: the wave
// probes 64 places at a time (four rounds of loads for 2^24 slots).
__device__ __forceinline__ int wave_lower_bound(const uint32_t *__restrict__ key, int n, uint32_t c)
{
    const int lane = threadIdx.x & (kWave - 1);
    int lo = 0, hi = n;   // the answer is in [lo, hi]
    while (hi > lo) {
        const int s = (hi - lo + kWave - 1) / kWave;   // probes at lo + (lane + 1) s - 1
        const long long p = (long long)lo + (long long)(lane + 1) * s - 1;
        const bool below = p < hi && key[p] < c;
        const int k = __popcll(__ballot(below));   // a prefix of the lanes
        const int first = lo + k * s;
        hi = (int)min((long long)hi, (long long)lo + (long long)(k + 1) * s - 1);
        lo = first;
        if (hi < lo) hi = lo;
    }
    return lo;
}

// The whole table in one launch: a block finds where the keys of its 256 cells
// lie (two searches by waves), takes them into LDS when they fit, and every
// cell finds its first slot there.  Bound by that chain of loads; it replaces a
// fill, a pass over the keys, a pass over the cells and a scan, five launches
// (the loop of single calls at N = 3e4 in 41^3 cells, with the move leaving its
// own sums and the compaction in three launches: 145 -> 111 us).
constexpr int kTableKeys = 4096;

__global__ __launch_bounds__(kBlock) void k_cell_table(const uint32_t *__restrict__ key,
                                                       const int *__restrict__ n_dev, int cells,
                                                       int2 *__restrict__ se, int *__restrict__ count,
                                                       int *__restrict__ prefix)
{
    __shared__ uint32_t k[kTableKeys];
    __shared__ int bound[2];
    __shared__ int first[kBlock + 1];
    const int n = *n_dev;
    const int c0 = blockIdx.x * kBlock, tid = threadIdx.x;
    const int w = tid / kWave;
    if (w < 2) {
        const int b = wave_lower_bound(key, n, (uint32_t)(c0 + w * kBlock));
        if ((tid & (kWave - 1)) == 0) bound[w] = b;
    }
    __syncthreads();
    const int a = bound[0], m = bound[1] - a;
    const bool in_lds = m <= kTableKeys;
    if (in_lds)
        for (int i = tid; i < m; i += kBlock) k[i] = key[a + i];
    __syncthreads();
    int lo = 0, hi = m;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if ((in_lds ? k[mid] : key[a + mid]) < (uint32_t)(c0 + tid)) lo = mid + 1; else hi = mid;
    }
    first[tid] = a + lo;
    if (tid == 0) first[kBlock] = a + m;
    __syncthreads();
    const int c = c0 + tid;
    if (c >= cells) return;
    const int f = first[tid], cnt = first[tid + 1] - f;
    prefix[c] = f;
    count[c] = cnt;
    se[c] = cnt > 0 ? make_int2(f, f + cnt - 1) : make_int2(-1, -1);
}

// ---------------------------------------------------------------------------
// collide (collisions.cu:291-445): one thread per cell, trials in sequence.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_collide_plain(
    TrapDev t, CollideParams cp, double *__restrict__ vx, double *__restrict__ vy,
    double *__restrict__ vz, double *__restrict__ sigvrmax, const int *__restrict__ prefix,
    int *__restrict__ coll_count, unsigned long long *__restrict__ coll_total, int ncells,
    uint32_t step)
{
    const double cellVolume = t.cell_vol;
    const double crossSection = cp.sigma;
    const double lpc = cp.lpc;
    unsigned long long mine = 0;
    for (int cell = blockIdx.x * kBlock + threadIdx.x; cell < ncells;
         cell += gridDim.x * kBlock) {
        const int n = prefix[cell + 1] - prefix[cell];
        // every cell's count is that of this call: collisions.cu:308,335
        // reset it only in cells of two or more atoms (a cell that empties
        // keeps a stale count there)
        if (n <= 1) { coll_count[cell] = 0; continue; }
        double lambda;
        const int Ncol = plain_trials(t, cp, n, sigvrmax[cell], lambda);
        const int base = prefix[cell];
        int count = 0;
        double smax = sigvrmax[cell];
        for (int tr = 0; tr < Ncol; ++tr) {
            int i, j;
            double u_acc;
            plain_trial(cp, t.stream, (uint32_t)cell, step, tr, n, i, j, u_acc);
            const int a = base + i, b = base + j;
            D3 va = { vx[a], vy[a], vz[a] }, vb = { vx[b], vy[b], vz[b] };
            const double dx = va.x - vb.x, dy = va.y - vb.y, dz = va.z - vb.z;
            const double magVrel = sqrt(dx * dx + dy * dy + dz * dz);
            if (magVrel * crossSection > smax) smax = magVrel * crossSection;
            const double ProbCol =
                t.alpha * lpc * cp.dt / cellVolume * magVrel * crossSection / lambda;
            if (ProbCol > u_acc) {
                plain_scatter(t, cp, (uint32_t)cell, step, tr, magVrel, va, vb);
                vx[a] = va.x; vy[a] = va.y; vz[a] = va.z;
                vx[b] = vb.x; vy[b] = vb.y; vz[b] = vb.z;
                ++count;
            }
        }
        sigvrmax[cell] = smax;
        coll_count[cell] = count;
        mine += (unsigned long long)count;
    }
    mine = wave_sum(mine);
    if ((threadIdx.x & (kWave - 1)) == 0 && mine) atomicAdd(coll_total, mine);
}

// ---------------------------------------------------------------------------
// moveAtoms (moveAtoms.cu:23-91): velocity Verlet with stored acceleration.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void move_atom(const TrapDev &t, double dt, const PlainPtrs &s, int i, D3 &p, D3 &v,
                                          bool &up)
{
    p = D3{ s.d[0][i], s.d[1][i], s.d[2][i] };
    v = D3{ s.d[3][i], s.d[4][i], s.d[5][i] };
    D3 a = { s.d[6][i], s.d[7][i], s.d[8][i] };
    up = s.up[i] != 0;
    plain_verlet(t, dt, up, p, v, a);
    s.d[0][i] = p.x; s.d[1][i] = p.y; s.d[2][i] = p.z;
    s.d[3][i] = v.x; s.d[4][i] = v.y; s.d[5][i] = v.z;
    s.d[6][i] = a.x; s.d[7][i] = a.y; s.d[8][i] = a.z;
}

// The observables of the moved state (calculateTemp, evaporation.cu:108-189,
// and the energy of energyChecker.py:117-122): a block's sums, in a fixed
// order (reproducible); k_observe_finalize_plain adds the blocks.
constexpr int kObsK = 5;  // ek, ep, vx^2, vy^2, vz^2

__device__ __forceinline__ void observe_block(const TrapDev &t, double mass, bool in, bool up, const D3 &p,
                                              const D3 &w, double *__restrict__ partials)
{
    __shared__ double tmp[(kBlock / kWave) * kObsK];
    double v[kObsK] = { 0.0, 0.0, 0.0, 0.0, 0.0 };
    if (in) {
        v[0] = 0.5 * mass * (w.x * w.x + w.y * w.y + w.z * w.z);
        // U_up = mu (|B| - B0); a spin-down atom (after a flip) has
        // U_down = -mu (|B| + B0), so that a flip conserves E_k + U
        const double u = potential_energy(t, p.x, p.y, p.z);
        v[1] = up ? u : -u - 2.0 * t.mu * t.B0;
        v[2] = w.x * w.x; v[3] = w.y * w.y; v[4] = w.z * w.z;
    }
    block_sum<kBlock, kObsK>(v, tmp);
    if (threadIdx.x == 0) {
#pragma unroll
        for (int k = 0; k < kObsK; ++k) partials[(size_t)blockIdx.x * kObsK + k] = v[k];
    }
}

// The move leaves the block sums of the moved state as it goes (the state was
// read a second time for them).
__global__ __launch_bounds__(kBlock) void k_move_plain(TrapDev t, double dt, double mass, PlainPtrs s,
                                                       const int *__restrict__ n_dev,
                                                       double *__restrict__ partials)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const bool in = i < *n_dev;
    D3 p = { 0.0, 0.0, 0.0 }, v = p;
    bool up = true;
    if (in) move_atom(t, dt, s, i, p, v, up);
    observe_block(t, mass, in, up, p, v, partials);
}

// ---------------------------------------------------------------------------
// evolveWavefunction (wavefunction.cu:11-73) and normalise (:279-299).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_spin_plain(TrapDev t, SpinParams sp, PlainPtrs s,
                                                       const int *__restrict__ n_dev)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= *n_dev) return;
    const D3 p = { s.d[0][i], s.d[1][i], s.d[2][i] };
    D3 v = { 0.0, 0.0, 0.0 }, a = v;
    if (sp.interp) {
        v = D3{ s.d[3][i], s.d[4][i], s.d[5][i] };
        a = D3{ s.d[6][i], s.d[7][i], s.d[8][i] };
    }
    Spinor q = { s.psi[0][i], s.psi[1][i], s.psi[2][i], s.psi[3][i] };
    plain_spin(t, sp, p, v, a, q);
    s.psi[0][i] = q.ur; s.psi[1][i] = q.ui; s.psi[2][i] = q.dr; s.psi[3][i] = q.di;
}

__global__ __launch_bounds__(kBlock) void k_normalise_plain(PlainPtrs s,
                                                            const int *__restrict__ n_dev)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= *n_dev) return;
    Spinor q = { s.psi[0][i], s.psi[1][i], s.psi[2][i], s.psi[3][i] };
    plain_normalise(q);
    s.psi[0][i] = q.ur; s.psi[1][i] = q.ui; s.psi[2][i] = q.dr; s.psi[3][i] = q.di;
}

// Majorana spin-flip model, one call each (plain_device.hpp).
__global__ __launch_bounds__(kBlock) void k_local_pops_plain(TrapDev t, PlainPtrs s,
                                                             double *__restrict__ pops,
                                                             const int *__restrict__ n_dev)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= *n_dev) return;
    double pu, pd;
    local_pops(t, D3{ s.d[0][i], s.d[1][i], s.d[2][i] },
               Spinor{ s.psi[0][i], s.psi[1][i], s.psi[2][i], s.psi[3][i] }, pu, pd);
    const size_t id = (size_t)s.id[i];
    pops[2 * id] = pu;
    pops[2 * id + 1] = pd;
}

__global__ __launch_bounds__(kBlock) void k_flip_plain(TrapDev t, FlipParams fp, PlainPtrs s,
                                                       const double *__restrict__ pops,
                                                       unsigned long long *__restrict__ flips,
                                                       const int *__restrict__ n_dev)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    unsigned long long cnt = 0ull;
    if (i < *n_dev) {
        const D3 p = { s.d[0][i], s.d[1][i], s.d[2][i] };
        D3 v = { s.d[3][i], s.d[4][i], s.d[5][i] };
        const uint32_t id = (uint32_t)s.id[i];
        bool up = s.up[i] != 0;
        if (plain_flip(t, fp, id, pops[2 * (size_t)id], pops[2 * (size_t)id + 1], p,
                       Spinor{ s.psi[0][i], s.psi[1][i], s.psi[2][i], s.psi[3][i] }, v, up)) {
            s.up[i] = up ? 1 : 0;
            s.d[3][i] = v.x; s.d[4][i] = v.y; s.d[5][i] = v.z;
            cnt = 1ull;
        }
    }
    cnt = wave_sum(cnt);
    if ((threadIdx.x & (kWave - 1)) == 0 && cnt) atomicAdd(flips, cnt);
}

__global__ __launch_bounds__(kBlock) void k_decay_plain(TrapDev t, DecayParams dp, PlainPtrs s,
                                                        const int *__restrict__ n_dev)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= *n_dev) return;
    Spinor q = { s.psi[0][i], s.psi[1][i], s.psi[2][i], s.psi[3][i] };
    plain_decay(t, dp, D3{ s.d[0][i], s.d[1][i], s.d[2][i] }, q);
    s.psi[0][i] = q.ur; s.psi[1][i] = q.ui; s.psi[2][i] = q.dr; s.psi[3][i] = q.di;
}

// ---------------------------------------------------------------------------
// evaporationTag (evaporation.cu:68-106) plus the energy cut.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_evap_tag_plain(TrapDev t, EvapParams ep, PlainPtrs s,
                                                           int *__restrict__ tag,
                                                           double *__restrict__ evap_pos,
                                                           double *__restrict__ evap_vel,
                                                           double *__restrict__ evap_accum,
                                                           const int *__restrict__ n_dev)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    double e_lost = 0.0, n_lost = 0.0;
    if (i < *n_dev) {
        const D3 p = { s.d[0][i], s.d[1][i], s.d[2][i] }, v = { s.d[3][i], s.d[4][i], s.d[5][i] };
        Spinor q = { 0.0, 0.0, 0.0, 0.0 };
        if (ep.spin_loss) q = Spinor{ s.psi[0][i], s.psi[1][i], s.psi[2][i], s.psi[3][i] };
        double E;
        const bool lost = plain_lost(t, ep.mass, ep.spin_loss != 0, ep.e_cut, p, v, q, E);
        tag[i] = lost ? 1 : 0;
        if (lost) {
            const int id = s.id[i];
            evap_pos[3 * (size_t)id + 0] = p.x; evap_pos[3 * (size_t)id + 1] = p.y;
            evap_pos[3 * (size_t)id + 2] = p.z;
            evap_vel[3 * (size_t)id + 0] = v.x; evap_vel[3 * (size_t)id + 1] = v.y;
            evap_vel[3 * (size_t)id + 2] = v.z;
            e_lost = E;
            n_lost = 1.0;
        }
    }
    e_lost = wave_sum(e_lost);
    n_lost = wave_sum(n_lost);
    if ((threadIdx.x & (kWave - 1)) == 0 && n_lost > 0.0) {
        atomicAdd(&evap_accum[0], e_lost);
        atomicAdd(&evap_accum[1], n_lost);
    }
}

// ---------------------------------------------------------------------------
// FP64 observables of the current state.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_observe_plain(TrapDev t, double mass, PlainPtrs s,
                                                          const int *__restrict__ n_dev,
                                                          double *__restrict__ partials)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    const bool in = i < *n_dev;
    D3 p = { 0.0, 0.0, 0.0 }, v = p;
    bool up = true;
    if (in) {
        p = D3{ s.d[0][i], s.d[1][i], s.d[2][i] };
        v = D3{ s.d[3][i], s.d[4][i], s.d[5][i] };
        up = s.up[i] != 0;
    }
    observe_block(t, mass, in, up, p, v, partials);
}

// One block adds the block partials in a fixed order (reproducible) and
// writes the log record; it also takes and clears the collision and
// evaporation accumulators of the step.
__global__ __launch_bounds__(kBlock) void k_observe_finalize_plain(
    const int *__restrict__ n_dev, const double *__restrict__ partials, int nb,
    dsmc_observables *__restrict__ out, unsigned long long *__restrict__ coll_accum,
    double *__restrict__ evap_accum, long long step)
{
    __shared__ double tmp[(kBlock / kWave) * kObsK];
    const int n = *n_dev;
    const int used = (n + kBlock - 1) / kBlock;
    double acc[kObsK] = { 0.0, 0.0, 0.0, 0.0, 0.0 };
    for (int b = threadIdx.x; b < used && b < nb; b += kBlock) {
#pragma unroll
        for (int k = 0; k < kObsK; ++k) acc[k] += partials[(size_t)b * kObsK + k];
    }
    block_sum<kBlock, kObsK>(acc, tmp);
    if (threadIdx.x == 0) {
        out->ek = acc[0];
        out->ep = acc[1];
        out->v2[0] = acc[2]; out->v2[1] = acc[3]; out->v2[2] = acc[4];
        out->e_evap = evap_accum[0];
        out->n_alive = n;
        out->n_evap = (long long)evap_accum[1];
        out->collisions = (long long)*coll_accum;
        out->step = step;
        evap_accum[0] = 0.0; evap_accum[1] = 0.0;
        *coll_accum = 0ull;
    }
}

// ---------------------------------------------------------------------------
// Initial distribution (setUp.cu:129-252): FP64 outputs.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_init_plain(TrapDev t, InitParams ip, PlainPtrs s,
                                                       int n)
{
    const int a = blockIdx.x * kBlock + threadIdx.x;
    if (a >= n) return;
    double px, py, pz, vx, vy, vz;
    init_atom(t, ip, (uint32_t)a, px, py, pz, vx, vy, vz);
    s.d[0][a] = px; s.d[1][a] = py; s.d[2][a] = pz;
    s.d[3][a] = vx; s.d[4][a] = vy; s.d[5][a] = vz;
    const D3 acc = accel(t, px, py, pz, true);
    s.d[6][a] = acc.x; s.d[7][a] = acc.y; s.d[8][a] = acc.z;
    s.id[a] = a;
    s.up[a] = 1;
    if (ip.spin) {
        // getAlignedSpinUp/Dn (setUp.cu:236-252)
        D3 Bn;
        (void)field_dir(t, px, py, pz, Bn);
        const double rs = 1.0 / sqrt(1 + Bn.x);
        s.psi[0][a] = 0.5 * (1. + Bn.x + Bn.z) * rs;
        s.psi[1][a] = 0.5 * (-Bn.y) * rs;
        s.psi[2][a] = 0.5 * (1. + Bn.x - Bn.z) * rs;
        s.psi[3][a] = 0.5 * Bn.y * rs;
    }
}

// Accelerations for externally supplied positions (dsmc_set_state).
__global__ __launch_bounds__(kBlock) void k_accel_plain(TrapDev t, PlainPtrs s, int n)
{
    const int a = blockIdx.x * kBlock + threadIdx.x;
    if (a >= n) return;
    const D3 acc = accel(t, s.d[0][a], s.d[1][a], s.d[2][a], s.up[a] != 0);
    s.d[6][a] = acc.x; s.d[7][a] = acc.y; s.d[8][a] = acc.z;
}

// ---------------------------------------------------------------------------
// Host launchers.
// ---------------------------------------------------------------------------
static int grid_for(int n) { return div_up(n > 0 ? n : 1, kBlock); }

void launch_index_plain(const TrapDev &t, const PlainPtrs &s, uint32_t *key, const int *n_dev,
                        int n_cap, hipStream_t st, Profiler *prof)
{
    DSMC_LAUNCH(prof, "index_plain", (double)n_cap * 28.0, k_index_plain, grid_for(n_cap), kBlock,
                st, t, s.d[0], s.d[1], s.d[2], key, n_dev);
}

void launch_gather_plain(const PlainPtrs &dst, const PlainPtrs &src, const uint32_t *map,
                         const int *n_dev, int n_cap, int spin, hipStream_t st, Profiler *prof,
                         int *n_out, int *n_host)
{
    const double per = 4.0 + 2.0 * (9 * 8 + 4 + 1 + (spin ? 32 : 0));
    DSMC_LAUNCH(prof, "gather_plain", (double)n_cap * per, k_gather_plain, grid_for(n_cap), kBlock,
                st, dst, src, map, n_dev, spin, n_out, n_host);
}

void launch_cell_table_plain(const uint32_t *key, const int *n_dev, int n_cap, int2 *se,
                             int *count, int *prefix, int ncells, hipStream_t st, Profiler *prof)
{
    DSMC_LAUNCH(prof, "cell_table", (double)n_cap * 4.0 + (ncells + 1) * 16.0, k_cell_table,
                grid_for(ncells + 1), kBlock, st, key, n_dev, ncells + 1, se, count, prefix);
}

void launch_collide_plain(const TrapDev &t, const CollideParams &cp, const PlainPtrs &s,
                          double *sigvrmax, const int *prefix, int *coll_count,
                          unsigned long long *coll_total, int ncells, uint32_t step,
                          hipStream_t st, Profiler *prof)
{
    const int grid = std::min(grid_for(ncells), 8192);
    DSMC_LAUNCH(prof, "collide_plain", (double)ncells * 20.0, k_collide_plain, grid, kBlock, st, t,
                cp, s.d[3], s.d[4], s.d[5], sigvrmax, prefix, coll_count, coll_total, ncells,
                step);
}

void launch_move_plain(const TrapDev &t, double dt, double mass, const PlainPtrs &s, const int *n_dev,
                       int n_cap, double *partials, hipStream_t st, Profiler *prof)
{
    DSMC_LAUNCH(prof, "move_plain", (double)n_cap * 145.0, k_move_plain, grid_for(n_cap), kBlock,
                st, t, dt, mass, s, n_dev, partials);
}

void launch_spin_plain(const TrapDev &t, const SpinParams &sp, const PlainPtrs &s,
                       const int *n_dev, int n_cap, hipStream_t st, Profiler *prof)
{
    DSMC_LAUNCH(prof, "spin_plain", (double)n_cap * 88.0, k_spin_plain, grid_for(n_cap), kBlock,
                st, t, sp, s, n_dev);
}

void launch_normalise_plain(const PlainPtrs &s, const int *n_dev, int n_cap, hipStream_t st,
                            Profiler *prof)
{
    DSMC_LAUNCH(prof, "normalise_plain", (double)n_cap * 64.0, k_normalise_plain,
                grid_for(n_cap), kBlock, st, s, n_dev);
}

void launch_evap_tag_plain(const TrapDev &t, const EvapParams &ep, const PlainPtrs &s, int *tag,
                           double *evap_pos, double *evap_vel, double *evap_accum,
                           const int *n_dev, int n_cap, hipStream_t st, Profiler *prof)
{
    DSMC_LAUNCH(prof, "evap_tag_plain", (double)n_cap * 84.0, k_evap_tag_plain, grid_for(n_cap),
                kBlock, st, t, ep, s, tag, evap_pos, evap_vel, evap_accum, n_dev);
}

void launch_local_pops_plain(const TrapDev &t, const PlainPtrs &s, double *pops, const int *n_dev,
                             int n_cap, hipStream_t st, Profiler *prof)
{
    DSMC_LAUNCH(prof, "local_pops_plain", (double)n_cap * 76.0, k_local_pops_plain,
                grid_for(n_cap), kBlock, st, t, s, pops, n_dev);
}

void launch_flip_plain(const TrapDev &t, const FlipParams &fp, const PlainPtrs &s,
                       const double *pops, unsigned long long *flips, const int *n_dev, int n_cap,
                       hipStream_t st, Profiler *prof)
{
    DSMC_LAUNCH(prof, "flip_plain", (double)n_cap * 101.0, k_flip_plain, grid_for(n_cap), kBlock,
                st, t, fp, s, pops, flips, n_dev);
}

void launch_decay_plain(const TrapDev &t, const DecayParams &dp, const PlainPtrs &s,
                        const int *n_dev, int n_cap, hipStream_t st, Profiler *prof)
{
    DSMC_LAUNCH(prof, "decay_plain", (double)n_cap * 88.0, k_decay_plain, grid_for(n_cap), kBlock,
                st, t, dp, s, n_dev);
}

int observe_plain_blocks(int n_cap) { return grid_for(n_cap); }

void launch_observe_plain(const TrapDev &t, double mass, const PlainPtrs &s, const int *n_dev,
                          int n_cap, double *partials, hipStream_t st, Profiler *prof)
{
    DSMC_LAUNCH(prof, "observe_plain", (double)n_cap * 48.0, k_observe_plain, grid_for(n_cap),
                kBlock, st, t, mass, s, n_dev, partials);
}

void launch_observe_finalize_plain(const int *n_dev, int n_cap, const double *partials, dsmc_observables *out,
                                   unsigned long long *coll_accum, double *evap_accum, long long step,
                                   hipStream_t st, Profiler *prof)
{
    DSMC_LAUNCH(prof, "observe_finalize", (double)grid_for(n_cap) * 40.0, k_observe_finalize_plain,
                1, kBlock, st, n_dev, partials, grid_for(n_cap), out, coll_accum, evap_accum, step);
}

void launch_init_plain(const TrapDev &t, const InitParams &ip, const PlainPtrs &s, int n,
                       hipStream_t st, Profiler *prof)
{
    DSMC_LAUNCH(prof, "init_plain", (double)n * 150.0, k_init_plain, grid_for(n), kBlock, st, t,
                ip, s, n);
}

void launch_accel_plain(const TrapDev &t, const PlainPtrs &s, int n, hipStream_t st,
                        Profiler *prof)
{
    DSMC_LAUNCH(prof, "accel_plain", (double)n * 48.0, k_accel_plain, grid_for(n), kBlock, st, t,
                s, n);
}

}  // namespace dsmc
