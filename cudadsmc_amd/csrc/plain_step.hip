// plain_step.hip -- the FP64 form's whole step.
//
// dsmc_step used to run the single calls one after the other: index, a radix
// sort of every key, a gather of the state, the cell table, collide, then per
// motion step spin, move, tag, compaction (with another gather) and sums; 17
// launches a step at lpc = 1 and 11 to 13 per motion step in the reference's
// run.  At N = 1e4 that is launch latency (68 and 40 us a motion step), at 1e6
// the state crosses memory some six times (188 us).  Here a collision step of
// up to kMaxSub motion substeps is four launches (three where the finalize's
// launch holds the whole sort, up to kScanSlots atoms); every further kMaxSub
// substeps are a move and a finalize more:
//   k_ins_merge                the stable sort by (cell, slot) from the last
//                              one (primitives.hip): the same permutation as
//                              the radix sort's
//   k_collide_step             cells of two or more atoms from the sorted keys,
//                              velocities through the permutation
//   k_move_step                gathers the state through the permutation into
//                              the other buffer and runs the motion substeps
//                              up to the next collision step in registers
//                              (an atom needs no other in between): spin,
//                              Verlet, losses, sums, flips, next key
//   k_step_finalize            log records of the substeps, counters, and the
//                              next sort's first phase
// The per-atom arithmetic is that of the single calls (plain_device.hpp), so
// the state is bitwise the same.  Atoms lost in a step keep their slot, with
// the dead key, until the next sort or until somebody looks (context.hip).
// Without spin flips every atom is spin up and its acceleration a function of
// its position, so neither is read or written: 116 B per atom and step
// instead of 172.
// Measured (step, MI355X): N = 1e4 67.8 -> 15.9 us, N = 1e6 188 -> 51.9 us,
// the reference's run (N = 1e4, lpc 10, spin flips) 40.5 -> 5 us per motion
// step.
#include "cells_device.hpp"
#include "plain_device.hpp"
#include "plain_step.hpp"
#include "resort_device.hpp"

namespace dsmc {

constexpr int kCollBlock = 256;

// ---------------------------------------------------------------------------
// collide (collisions.cu:291-445): the cells of two or more atoms of a wave's
// 128 or 512 sorted slots, one per lane, trials in sequence.  Bound by its
// chain of dependent loads (keys; sigma v_r,max and permutation; velocities):
// the first trial's pair is loaded beside sigma v_r,max, before the trial
// count that needs it.
// ---------------------------------------------------------------------------
template <int ITEMS>
__global__ __launch_bounds__(kCollBlock) void k_collide_step(
    TrapDev t, CollideParams cp, const uint32_t *__restrict__ key, const uint32_t *__restrict__ perm,
    const PlainCtl *__restrict__ ctl, int n_cap, double *__restrict__ vx, double *__restrict__ vy,
    double *__restrict__ vz, double *__restrict__ sigvrmax, unsigned long long *__restrict__ cc,
    unsigned long long *__restrict__ coll_total, int *__restrict__ n_sorted, ResortBuckets rb)
{
    __shared__ WaveCells<ITEMS> cells[kCollBlock / kWave];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int chunk0 = (blockIdx.x * (kCollBlock / kWave) + w) * kWave * ITEMS;
    WaveCells<ITEMS> &L = cells[w];
    ChunkKeys<ITEMS> ck;
    chunk_load(key, n_cap, chunk0, ck);
    const int n = ctl->alive;
    const uint32_t step = (uint32_t)ctl->step;
    const unsigned long long stamp = (unsigned long long)(ctl->coll + 1u) << 32;
    if (blockIdx.x == 0 && threadIdx.x == 0) *n_sorted = n;
    resort_clear(rb, blockIdx.x * kCollBlock + threadIdx.x, gridDim.x * kCollBlock);
    uint32_t k_first, k_last;
    const int nm = wave_list_cells(key, n, chunk0, ck, L, k_first, k_last);
    unsigned long long mine = 0;
    for (int m = lane; m < nm; m += kWave) {
        const uint32_t k = L.key[m];
        const uint32_t cell = k - (uint32_t)t.key_base;
        if ((int)cell >= t.n_cells) continue;   // overflow cell: no collisions
        const int base = chunk0 + L.start[m], c = L.end[m] - base;
        int i, j;
        double u_acc;
        plain_trial(cp, t.stream, cell, step, 0, c, i, j, u_acc);
        uint32_t a = perm[base + i], b = perm[base + j];
        const double s0 = sigvrmax[k];
        D3 va = { vx[a], vy[a], vz[a] }, vb = { vx[b], vy[b], vz[b] };
        double lambda;
        const int Ncol = plain_trials(t, cp, c, s0, lambda);
        double smax = s0;
        int count = 0;
        for (int tr = 0; tr < Ncol; ++tr) {
            if (tr > 0) {
                plain_trial(cp, t.stream, cell, step, tr, c, i, j, u_acc);
                a = perm[base + i]; b = perm[base + j];
                va = D3{ vx[a], vy[a], vz[a] }; vb = D3{ vx[b], vy[b], vz[b] };
            }
            const double dx = va.x - vb.x, dy = va.y - vb.y, dz = va.z - vb.z;
            const double magVrel = sqrt(dx * dx + dy * dy + dz * dz);
            if (magVrel * cp.sigma > smax) smax = magVrel * cp.sigma;
            const double ProbCol = t.alpha * cp.lpc * cp.dt / t.cell_vol * magVrel * cp.sigma / lambda;
            if (ProbCol > u_acc) {
                plain_scatter(t, cp, cell, step, tr, magVrel, va, vb);
                vx[a] = va.x; vy[a] = va.y; vz[a] = va.z;
                vx[b] = vb.x; vy[b] = vb.y; vz[b] = vb.z;
                ++count;
            }
        }
        if (smax != s0) sigvrmax[k] = smax;
        if (count) cc[cell] = stamp | (unsigned)count;
        mine += (unsigned long long)count;
    }
    mine = wave_sum(mine);
    if (lane == 0 && mine) atomicAdd(coll_total, mine);
}

// ---------------------------------------------------------------------------
// The motion substeps.  Bound by memory at lpc = 1 without spin (gather and
// write of 52 bytes per atom, 12 bytes of keys and permutation), by FP64
// arithmetic (two sqrt and two divisions per substep, sine and cosine with
// spin) beyond.
// ---------------------------------------------------------------------------
// Wave totals of four values: lane l (l % 16 == 0) returns that of quantity
// 2 bit5(l) + bit4(l) (the exchanges of block_sum4).
__device__ __forceinline__ double wave_sum4(const double (&v)[4])
{
    const int lane = threadIdx.x & (kWave - 1);
    const bool b5 = (lane & 32) != 0, b4 = (lane & 16) != 0;
    double k0 = b5 ? v[2] : v[0], k1 = b5 ? v[3] : v[1];
    const double s0 = b5 ? v[0] : v[2], s1 = b5 ? v[1] : v[3];
    k0 += lane_xor<32>(s0);
    k1 += lane_xor<32>(s1);
    double k = b4 ? k1 : k0;
    k += lane_xor<16>(b4 ? k0 : k1);
    k += lane_xor<8>(k);
    k += lane_xor<4>(k);
    k += lane_xor<2>(k);
    k += lane_xor<1>(k);
    return k;
}

template <bool SPIN, bool STORED>
__global__ __launch_bounds__(kStepBlock) void k_move_step(
    TrapDev t, PlainStepParams sp, PlainPtrs A, PlainPtrs B, const uint32_t *__restrict__ perm,
    const uint32_t *key_in, const int *__restrict__ n_dev, const PlainCtl *__restrict__ ctl,
    uint32_t *key_out, double *__restrict__ pops, double *__restrict__ evap_pos,
    double *__restrict__ evap_vel, double *__restrict__ rec, int stride)
{
    constexpr int W = kStepBlock / kWave;
    __shared__ double red[kMaxSub][W][4];
    __shared__ double lred[kMaxSub][W][2];
    const int lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const int blk = blockIdx.x, i = blk * kStepBlock + threadIdx.x;
    const int n = *n_dev;
    const long long step0 = ctl->step;
    const bool in = i < n;
    bool alive = in;
    D3 p = { 0.0, 0.0, 0.0 }, v = p, a = p;
    Spinor q = { 0.0, 0.0, 0.0, 0.0 };
    int id = 0;
    bool up = true;
    uint32_t kold = 0;
    if (in) {
        const uint32_t j = perm ? perm[i] : (uint32_t)i;
        if (key_in) alive = key_in[i] != sp.dead_key;
        p = D3{ A.d[0][j], A.d[1][j], A.d[2][j] };
        v = D3{ A.d[3][j], A.d[4][j], A.d[5][j] };
        id = A.id[j];
        if (STORED) {
            a = D3{ A.d[6][j], A.d[7][j], A.d[8][j] };
            up = A.up[j] != 0;
        }
        if (SPIN) q = Spinor{ A.psi[0][j], A.psi[1][j], A.psi[2][j], A.psi[3][j] };
        if (sp.key_prev) kold = sp.key_prev[i];
    }
    if (!STORED) a = accel(t, p.x, p.y, p.z, true);
    double opu = 0.0, opd = 0.0;
    if (STORED && alive) {
        if (sp.phase == 0) {
            local_pops(t, p, q, opu, opd);
            pops[2 * (size_t)id] = opu;
            pops[2 * (size_t)id + 1] = opd;
        } else {
            opu = pops[2 * (size_t)id];
            opd = pops[2 * (size_t)id + 1];
        }
    }
    bool last_lost = false;
    for (int l = 0; l < sp.L; ++l) {
        double sums[4] = { 0.0, 0.0, 0.0, 0.0 }, e_lost = 0.0;
        bool lost = false;
        if (alive) {
            if (SPIN) plain_spin(t, sp.spin, p, v, a, q);
            plain_verlet(t, sp.dt, up, p, v, a);
            if (sp.spin_loss || sp.energy_cut) {
                double cut = 0.0, E;
                if (sp.energy_cut && t.kT_cut > 0.0) {
                    const double f = t.eta_steps > 0 ? fmin((double)(step0 + l) / (double)t.eta_steps, 1.0) : 1.0;
                    cut = (t.eta_start + (t.eta_end - t.eta_start) * f) * t.kT_cut;
                }
                lost = plain_lost(t, sp.mass, sp.spin_loss != 0, cut, p, v, q, E);
                if (lost) {
                    evap_pos[3 * (size_t)id + 0] = p.x; evap_pos[3 * (size_t)id + 1] = p.y;
                    evap_pos[3 * (size_t)id + 2] = p.z;
                    evap_vel[3 * (size_t)id + 0] = v.x; evap_vel[3 * (size_t)id + 1] = v.y;
                    evap_vel[3 * (size_t)id + 2] = v.z;
                    e_lost = E;
                    alive = false;
                }
            }
        }
        if (alive) {
            if (SPIN && sp.phase + l + 1 == sp.lpc) {   // end of the collision step (main.cu:501-521)
                if (STORED) {
                    FlipParams fp = sp.flip;
                    fp.step = ctl->coll + (sp.phase == 0 ? 1u : 0u);
                    (void)plain_flip(t, fp, (uint32_t)id, opu, opd, p, q, v, up);
                    plain_decay(t, sp.decay, p, q);
                }
                plain_normalise(q);
            }
            sums[0] = v.x * v.x; sums[1] = v.y * v.y; sums[2] = v.z * v.z;
            // U_up = mu (|B| - B0); a spin-down atom (after a flip) has
            // U_down = -mu (|B| + B0), so that a flip conserves E_k + U
            const double u = potential_energy(t, p.x, p.y, p.z);
            sums[3] = up ? u : -u - 2.0 * t.mu * t.B0;
        }
        const double s4 = wave_sum4(sums);
        if ((lane & 15) == 0) red[l][w][((lane >> 5) & 1) * 2 + ((lane >> 4) & 1)] = s4;
        const uint64_t lm = __ballot(lost);
        const double e = lm ? wave_sum(e_lost) : 0.0;
        if (lane == 0) { lred[l][w][0] = e; lred[l][w][1] = (double)__popcll(lm); }
        last_lost = lost;
    }
    // state, next key, masks
    const bool dead = in && !alive;
    bool moved = false;
    if (in) {
        uint32_t kout = sp.dead_key;
        if (alive)
            kout = (uint32_t)(t.key_base + (sp.fast_key ? cell_of_fast(t, p.x, p.y, p.z) : cell_of(t, p.x, p.y, p.z)));
        moved = alive && sp.key_prev && kout != kold;
        key_out[i] = kout;
        B.d[0][i] = p.x; B.d[1][i] = p.y; B.d[2][i] = p.z;
        B.d[3][i] = v.x; B.d[4][i] = v.y; B.d[5][i] = v.z;
        B.id[i] = id;
        if (STORED) {
            B.d[6][i] = a.x; B.d[7][i] = a.y; B.d[8][i] = a.z;
            B.up[i] = up ? 1 : 0;
        }
        if (SPIN) { B.psi[0][i] = q.ur; B.psi[1][i] = q.ui; B.psi[2][i] = q.dr; B.psi[3][i] = q.di; }
    }
    const uint64_t bm = __ballot(moved), bd = __ballot(dead), bl = __ballot(last_lost);
    if (lane == 0) {
        const int wd = blk * W + w;
        sp.mask_moved[wd] = bm;
        sp.mask_dead[wd] = bd;
        sp.mask_last[wd] = bl;
    }
    __syncthreads();
    // block sums: waves in order; the atoms lost are counted up to each substep
    const int tid = threadIdx.x;
    if (tid < sp.L * 4) {
        const int l = tid >> 2, k = tid & 3;
        double s = 0.0;
#pragma unroll
        for (int ww = 0; ww < W; ++ww) s += red[l][ww][k];
        rec[((size_t)l * kStepRec + k) * stride + blk] = s;
    } else if (tid >= 64 && tid < 64 + sp.L) {
        const int l = tid - 64;
        double e = 0.0, c = 0.0;
#pragma unroll
        for (int ww = 0; ww < W; ++ww) e += lred[l][ww][0];
        for (int k = 0; k <= l; ++k)
#pragma unroll
            for (int ww = 0; ww < W; ++ww) c += lred[k][ww][1];
        rec[((size_t)l * kStepRec + 4) * stride + blk] = e;
        rec[((size_t)l * kStepRec + 5) * stride + blk] = c;
    }
}
static_assert(kMaxSub * 4 <= 64, "the block sums' threads");

// Grid: one block per substep, then list.blocks blocks of the next re-sort's
// first phase.  A block adds its substep's records over the move blocks (four
// rounds of loads in flight per thread) in a fixed order.
template <bool MERGE>
__global__ __launch_bounds__(256) void k_step_finalize(
    int L, double half_mass, const int *__restrict__ n_dev, const double *__restrict__ rec, int stride,
    const PlainCtl *__restrict__ ctl, PlainCtl *__restrict__ next, int collided,
    unsigned long long *__restrict__ coll_accum, double *__restrict__ evap_accum,
    dsmc_observables *__restrict__ log, int obs_cap, ResortWork work)
{
    extern __shared__ __align__(16) uint32_t lds[];   // first phase: tiles' first keys; merge: movers' slots
    __shared__ unsigned short list_slot[kListSlots];
    __shared__ MergeLds merge_lds;
    __shared__ double red[(256 / kWave) * 8];
    if ((int)blockIdx.x >= L) {
        const int j = (int)blockIdx.x - L;
        if constexpr (MERGE) resort_scan_merge_block(work.merge, j, merge_lds, (unsigned short *)lds);
        else resort_list_block(work.list, j, lds, list_slot);
        return;
    }
    const int l = (int)blockIdx.x;
    const int n = *n_dev;
    const PlainCtl c = *ctl;
    const int nb = (n + kStepBlock - 1) / kStepBlock;
    // v_x^2, v_y^2, v_z^2, U, lost energy, lost so far; lost before this substep
    double s[8] = { 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0 };
    const double *r = rec + (size_t)l * kStepRec * stride;
    const double *before = l > 0 ? r - stride : nullptr;   // the substep before: its last row
    for (int b0 = threadIdx.x; b0 < nb; b0 += 4 * 256) {
        double x[4][7];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int b = b0 + u * 256;
#pragma unroll
            for (int k = 0; k < kStepRec; ++k) x[u][k] = b < nb ? r[(size_t)k * stride + b] : 0.0;
            x[u][6] = b < nb && before ? before[b] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int k = 0; k < 7; ++k) s[k] += x[u][k];
    }
    block_sum8<256>(s, red);
    if (threadIdx.x != 0) return;
    const long long step = c.step + l;
    dsmc_observables &o = log[step % obs_cap];
    o.ek = half_mass * (s[0] + s[1] + s[2]);
    o.ep = s[3];
    o.v2[0] = s[0]; o.v2[1] = s[1]; o.v2[2] = s[2];
    o.e_evap = s[4];
    o.n_alive = (long long)c.alive - (long long)s[5];
    o.n_evap = (long long)(s[5] - s[6]);
    o.collisions = 0;
    o.step = step;
    if (l == 0) {   // what single calls or the collide left to count
        o.collisions = (long long)*coll_accum;
        o.e_evap += evap_accum[0];
        o.n_evap += (long long)evap_accum[1];
        *coll_accum = 0ull;
        evap_accum[0] = 0.0; evap_accum[1] = 0.0;
    }
    if (l == L - 1) {
        next->step = c.step + L;
        next->coll = c.coll + (unsigned)collided;
        next->slots = n;
        next->alive = c.alive - (int)s[5];
    }
}

__global__ void k_set_ctl(PlainCtl *ctl, long long step, unsigned coll, const int *n)
{
    ctl->step = step;
    ctl->coll = coll;
    ctl->slots = *n;
    ctl->alive = *n;
}

__global__ __launch_bounds__(256) void k_prev_dead_stencil(const uint32_t *__restrict__ key,
                                                           const uint64_t *__restrict__ mask_last,
                                                           const int *__restrict__ n, uint32_t dead_key,
                                                           int *__restrict__ stencil)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < *n) stencil[i] = key[i] == dead_key && !((mask_last[i >> 6] >> (i & 63)) & 1ull);
}

__global__ __launch_bounds__(256) void k_last_tags(const uint32_t *__restrict__ map,
                                                   const uint64_t *__restrict__ mask_last,
                                                   const int *__restrict__ n, int *__restrict__ tag)
{
    const int j = blockIdx.x * 256 + threadIdx.x;
    if (j >= *n) return;
    const uint32_t i = map[j];
    tag[j] = (int)((mask_last[i >> 6] >> (i & 63)) & 1ull);
}

__global__ __launch_bounds__(256) void k_untag_counts(const unsigned long long *__restrict__ cc, unsigned coll,
                                                      int ncells, int *__restrict__ count)
{
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= ncells) return;
    const unsigned long long v = cc[c];
    count[c] = (unsigned)(v >> 32) == coll ? (int)(uint32_t)v : 0;
}

__global__ __launch_bounds__(256) void k_keys_by_slot(const uint32_t *__restrict__ key,
                                                      const uint32_t *__restrict__ perm,
                                                      const int *__restrict__ n, uint32_t *__restrict__ out)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < *n) out[perm ? perm[i] : (uint32_t)i] = key[i];
}

// ---------------------------------------------------------------------------
// Host launchers.
// ---------------------------------------------------------------------------
constexpr int kCollTwo = 1 << 19;   // largest capacity for which a lane of the collide takes two slots

void launch_collide_step(const TrapDev &t, const CollideParams &cp, const PlainPtrs &s, const uint32_t *key,
                         const uint32_t *perm, const PlainCtl *ctl, int n_cap, double *sigvrmax,
                         unsigned long long *cc, unsigned long long *coll_total, int *n_sorted,
                         const ResortBuckets &rb, hipStream_t st, Profiler *prof)
{
    auto launch = [&](auto kernel, int items) {
        DSMC_LAUNCH(prof, "collide_step", (double)n_cap * 4.0, kernel,
                    div_up(n_cap > 0 ? n_cap : 1, kCollBlock * items), kCollBlock, st, t, cp, key, perm, ctl,
                    n_cap, s.d[3], s.d[4], s.d[5], sigvrmax, cc, coll_total, n_sorted, rb);
    };
    // two slots per lane while the chip has room for the waves (one round of
    // cells each), eight beyond (step in us, eight / two: N = 1e4 23.5 / 21.2,
    // 1e5 28.6 / 25.5, 4e5 38.9 / 37.4, 1e6 55.4 / 56.7)
    if (n_cap <= kCollTwo) launch(k_collide_step<2>, 2);
    else launch(k_collide_step<8>, 8);
}

void launch_move_step(bool spin, bool stored, const TrapDev &t, const PlainStepParams &p, const PlainPtrs &src,
                      const PlainPtrs &dst, const uint32_t *perm, const uint32_t *key_in, bool after_sort,
                      const PlainCtl *ctl, uint32_t *key_out, double *pops, double *evap_pos, double *evap_vel,
                      double *rec, int stride, int n_cap, hipStream_t st, Profiler *prof)
{
    const int *n = after_sort ? &ctl->alive : &ctl->slots;
    const int grid = div_up(n_cap > 0 ? n_cap : 1, kStepBlock);
    const double bytes = (double)n_cap * (116.0 + (stored ? 50.0 : 0.0) + (spin ? 64.0 : 0.0));
#define DSMC_MOVE_STEP(S, A)                                                                            \
    DSMC_LAUNCH(prof, "move_step", bytes, (k_move_step<S, A>), grid, kStepBlock, st, t, p, src, dst, perm, \
                key_in, n, ctl, key_out, pops, evap_pos, evap_vel, rec, stride)
    if (stored) DSMC_MOVE_STEP(true, true);
    else if (spin) DSMC_MOVE_STEP(true, false);
    else DSMC_MOVE_STEP(false, false);
#undef DSMC_MOVE_STEP
}

void launch_step_finalize(const PlainStepParams &p, bool after_sort, const double *rec, int stride,
                          const PlainCtl *ctl, PlainCtl *next, unsigned long long *coll_accum,
                          double *evap_accum, dsmc_observables *log, int obs_cap, const ResortWork &work,
                          hipStream_t st, Profiler *prof)
{
    if (prof && prof->enabled) prof->begin(st, "step_finalize", (double)p.L * stride * kStepRec * 8.0);
    hipLaunchKernelGGL(work.merge.tiles > 0 ? k_step_finalize<true> : k_step_finalize<false>,
                       dim3(p.L + work.blocks()), dim3(256), resort_work_lds(work), st, p.L,
                       0.5 * p.mass, after_sort ? &ctl->alive : &ctl->slots, rec, stride, ctl, next,
                       after_sort ? 1 : 0, coll_accum, evap_accum, log, obs_cap, work);
    DSMC_HIP(hipGetLastError());
    if (prof && prof->enabled) prof->end(st);
}

void launch_set_ctl(PlainCtl *ctl, long long step, unsigned coll, const int *n, hipStream_t st)
{
    hipLaunchKernelGGL(k_set_ctl, dim3(1), dim3(1), 0, st, ctl, step, coll, n);
    DSMC_HIP(hipGetLastError());
}

void launch_prev_dead_stencil(const uint32_t *key, const uint64_t *mask_last, const PlainCtl *ctl, int n_cap,
                              uint32_t dead_key, int *stencil, hipStream_t st)
{
    hipLaunchKernelGGL(k_prev_dead_stencil, dim3(div_up(n_cap, 256)), dim3(256), 0, st, key, mask_last,
                       &ctl->slots, dead_key, stencil);
    DSMC_HIP(hipGetLastError());
}

void launch_last_tags(const uint32_t *map, const uint64_t *mask_last, const int *n, int n_cap, int *tag,
                      hipStream_t st)
{
    hipLaunchKernelGGL(k_last_tags, dim3(div_up(n_cap, 256)), dim3(256), 0, st, map, mask_last, n, tag);
    DSMC_HIP(hipGetLastError());
}

void launch_keys_by_slot(const uint32_t *key, const uint32_t *perm, const int *n, int n_cap, uint32_t *out,
                         hipStream_t st)
{
    hipLaunchKernelGGL(k_keys_by_slot, dim3(div_up(n_cap, 256)), dim3(256), 0, st, key, perm, n, out);
    DSMC_HIP(hipGetLastError());
}

void launch_untag_counts(const unsigned long long *cc, unsigned coll, int ncells, int *count, hipStream_t st)
{
    hipLaunchKernelGGL(k_untag_counts, dim3(div_up(ncells, 256)), dim3(256), 0, st, cc, coll, ncells, count);
    DSMC_HIP(hipGetLastError());
}

}  // namespace dsmc
