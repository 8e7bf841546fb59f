// context.hip -- the C ABI of include/dsmc.h: context lifetime, buffer
// ownership, the step loop of both numerical forms, HIP-graph replay, per-kernel
// profiling and the output surface.
//
// Host-side call sequence per motion step (main.cu:412-523 without the dead
// median, the MCWF spin-flip model and the HDF5 output):
//   FP64 form:  sort, collide every lpc steps, then the motion substeps up to
//               the next collision step in one kernel (plain_step.hip)
//   FP32 form:  sort, table, [collide], fused move           every step
// No call in the loop synchronises with the host.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/dsmc.h"
#include "dsmc_internal.hpp"
#include "fused.hpp"
#include "host_copy.hpp"
#include "plain.hpp"
#include "plain_step.hpp"
#include "readout.hpp"

using namespace dsmc;

// ---------------------------------------------------------------------------
// Runtime helpers
// ---------------------------------------------------------------------------
namespace dsmc {

void hip_check(hipError_t e, const char *what, const char *file, int line)
{
    if (e == hipSuccess) return;
    const int st = (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation) ? DSMC_ENOMEM
                                                                                : DSMC_EHIP;
    char buf[512];
    std::snprintf(buf, sizeof buf, "%s failed: %s (%s:%d)", what, hipGetErrorString(e), file, line);
    throw Error(st, buf);
}

hipEvent_t Profiler::take()
{
    if (!pool_.empty()) {
        hipEvent_t e = pool_.back();
        pool_.pop_back();
        return e;
    }
    hipEvent_t e;
    DSMC_HIP(hipEventCreate(&e));
    return e;
}

void Profiler::begin(hipStream_t s, const char *name, double bytes)
{
    Rec r;
    r.name = name;
    r.bytes = bytes;
    r.b = take();
    r.e = take();
    DSMC_HIP(hipEventRecord(r.b, s));
    pending_.push_back(r);
}

void Profiler::end(hipStream_t s)
{
    if (pending_.empty()) return;
    DSMC_HIP(hipEventRecord(pending_.back().e, s));
}

void Profiler::collect()
{
    for (Rec &r : pending_) {
        DSMC_HIP(hipEventSynchronize(r.e));
        float ms = 0.f;
        DSMC_HIP(hipEventElapsedTime(&ms, r.b, r.e));
        Stat &s = stats_[r.name];
        s.launches += 1;
        s.total_ms += ms;
        s.bytes = r.bytes;
        pool_.push_back(r.b);
        pool_.push_back(r.e);
    }
    pending_.clear();
}

void Profiler::reset()
{
    collect();
    stats_.clear();
}

Profiler::~Profiler()
{
    for (Rec &r : pending_) { (void)hipEventDestroy(r.b); (void)hipEventDestroy(r.e); }
    for (hipEvent_t e : pool_) (void)hipEventDestroy(e);
}

}  // namespace dsmc

// ---------------------------------------------------------------------------
// Context
// ---------------------------------------------------------------------------

static void free_kept();   // scratch kept between the primitives' calls

// Device memory, if need be without that scratch.
static void *device_alloc(size_t bytes)
{
    void *p = nullptr;
    if (hipMalloc(&p, bytes) != hipSuccess) {
        (void)hipGetLastError();
        free_kept();
        DSMC_HIP(hipMalloc(&p, bytes));
    }
    return p;
}

// A captured run of steps.
struct StepGraph {
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    void destroy()
    {
        if (exec) (void)hipGraphExecDestroy(exec);
        if (graph) (void)hipGraphDestroy(graph);
        exec = nullptr;
        graph = nullptr;
    }
};

// The captured runs of steps for one state of the double buffers: of one pair
// of steps, and of kLongPairs pairs.
struct StepGraphs {
    int srt = 0, ssel = 0, tsel = 0, cur = 0;   // the buffers current at the capture
    StepGraph one, many;
    int pairs_run = 0;   // pairs replayed (up to kLongFrom)
    bool same(const StepGraphs &o) const
    {
        return srt == o.srt && ssel == o.ssel && tsel == o.tsel && cur == o.cur;
    }
    void destroy()
    {
        one.destroy();
        many.destroy();
        pairs_run = 0;
    }
};

struct dsmc_ctx {
    dsmc_config cfg{};
    std::vector<dsmc_trap> traps;
    std::vector<TrapDev> tdev;
    std::vector<int> key_base;      // n_traps + 1; last = dead key
    std::vector<int> atom_begin;    // n_traps + 1
    int T = 0, n_cap = 0, n_keys = 0, key_bits = 0, passes = 0, ncells = 0;
    int device = 0;
    uint32_t dead_key = 0;
    bool fp32 = false;
    hipStream_t stream = nullptr;
    Profiler prof;
    std::string err;
    long long step = 0;             // motion steps taken
    long long coll_steps = 0;
    int cur = 0;                    // state buffer holding the current state
    int obs_cap = 0;
    int block = 256;                // FP32 move: threads per block
    int apt = 1;                    // FP32 move: atoms per thread
    bool have_sort = false;         // FP32: perm valid for the next move
    bool tbl_valid = false;         // FP32: trap_start and the alive count describe the
                                    // next sort's output (set by a sorted move's finalize)
    bool srt_valid = false;         // FP32: srt_k[srt_cur][i] is the key of slot i of the
                                    // current state (slots in sorted order of those keys)
    bool dead_in_state = false;     // FP32: the current state may hold atoms a move removed
                                    // (dead key in key_a, left in place until a sort)
    std::vector<void *> allocs;

    // common device buffers
    TrapDev *d_traps = nullptr;
    int *d_key_base = nullptr;
    uint32_t *key_a = nullptr, *key_b = nullptr, *val_a = nullptr, *val_b = nullptr;
    uint32_t *srt_k[2] = {nullptr, nullptr}, *srt_v[2] = {nullptr, nullptr};  // sort outputs (of a small context, the next step's in the one not current)
    int srt_cur = 0;                // FP32: srt_*[srt_cur] holds the last sort's result
    bool bucketed = false;          // the last finalize ran the re-sort's first phase, or all of it
    bool counts_clear = true;       // the buckets' counts are zero (a collide clears them)
    bool split_step = true;         // FP32: dsmc_step runs collide and move as two kernels
    const uint32_t *sorted_key = nullptr, *perm = nullptr;
    SortScratch sort;
    ResortScratch res;              // FP32: incremental re-sort
    double *sigvrmax = nullptr;     // FP64 form
    float *sigvrmax_f = nullptr;    // FP32 form: sigma v_r,max in float (half the bytes)
    uint64_t *edge_sm = nullptr;    // FP32 form, fused step: its scratch
    dsmc_observables *obs_log = nullptr;  // (obs_cap + 1) * T records
    // device step counter, double-buffered: the kernels of a step read
    // step_buf[ssel] and its finalize writes the next value to the other one
    long long *step_buf = nullptr;
    int ssel = 0;
    long long *step_save = nullptr;
    long long *step_dev() const { return step_buf + ssel; }
    unsigned long long *coll_accum = nullptr;
    int *n_dev = nullptr;           // [0], [1]: alive counts; [2]: scratch
    int *n_host = nullptr;          // pinned copy of n_dev for host reads
    dsmc_observables *obs_host = nullptr;   // pinned record (FP64 form)
    int *scan_partial = nullptr;    // partials of scans and compactions
    // FP64 form
    PlainPtrs ps[2];
    int2 *start_end = nullptr;
    int *count = nullptr, *prefix = nullptr, *coll_count = nullptr;
    int *tag = nullptr;
    uint32_t *cmap = nullptr;
    double *evap_pos_d = nullptr, *evap_vel_d = nullptr;
    double *partials = nullptr, *evap_accum = nullptr;
    double *pops = nullptr;                  // spin-flip model: populations by label
    unsigned long long *flips = nullptr;     // spin-flip model: flips of the last call
    // FP64 form, whole steps (plain_step.hip).  dsmc_step leaves some of what
    // the single calls and host reads expect to be made when they ask
    // (plain_settle, plain_need_acc, plain_need_tables).
    PlainCtl *ctl = nullptr;        // [2]: counters, ctl[csel] current
    int csel = 0;
    uint32_t *key_f = nullptr;      // the state's next keys (dead key: removed atoms)
    uint64_t *mask_d2[2] = {nullptr, nullptr};   // removed atoms; [mpar] the current state's
    uint64_t *mask_last = nullptr;
    int mpar = 0;
    double *rec64 = nullptr;        // per-block sums of a move launch
    unsigned long long *cc_tagged = nullptr;     // collision step << 32 | collisions, per cell
    bool ctl_live = false;          // ctl describes the state (else n_dev, step, coll_steps do)
    bool sorted_ok = false;         // srt_k[srt_cur][i] is the key of slot i, masks and samples too
    bool keys_ok = false;           // key_f holds the state's keys
    bool lazy_dead = false;         // removed atoms may still hold slots
    bool acc_stale = false;         // the accelerations in memory are not the state's
    bool tables_stale = false;      // cell table and counts are those of an earlier sort
    bool up_set = false;            // ps[].up hold the initial flags
    bool index_stale = false;       // key_a is not as the last step's index and sort leave it
    int perm_mask = -1;             // perm's slots count the removed atoms of mask_d2[perm_mask]
    // FP32 form
    FusedPtrs fs[2];
    uint32_t *cell_start = nullptr, *cell_end = nullptr;
    uint32_t *blk_dead = nullptr;   // removed atoms per move block (FP32)
    uint64_t *mask_moved = nullptr, *mask_dead = nullptr; // per 64 slots, for the re-sort
    // trap ranges of the slot order, double-buffered: a sorted move's
    // finalize writes the next sort's ranges to ts_buf[tsel ^ 1]
    int *ts_buf[2] = { nullptr, nullptr };
    int tsel = 0;
    int *trap_start() const { return ts_buf[tsel]; }
    double *acc = nullptr, *acc2 = nullptr;
    ObsRecords rec{};
    int *obs_first = nullptr, *obs_last = nullptr;   // on-demand observables scratch
    int max_trap_atoms = 0;
    float *evap_pos_f = nullptr, *evap_vel_f = nullptr;
    float *spin_tau = nullptr;   // (spin) the substeps' times in a step
    // captured steps (FP32: parity 0 then 1), the last used first.  Two: reads
    // of a run with losses swap the FP64 state's buffers, so runs with a read
    // after each come by two states in turn
    StepGraphs graphs[2];
    HostCopy host_copy;

    template <typename T_>
    T_ *alloc(size_t count_, bool zero = true)
    {
        const size_t bytes = std::max<size_t>(count_ * sizeof(T_), 16);
        void *p = device_alloc(bytes);
        allocs.push_back(p);
        if (zero) DSMC_HIP(hipMemsetAsync(p, 0, bytes, stream));
        return (T_ *)p;
    }

    ~dsmc_ctx()
    {
        // drain the stream before destroying a graph it may still be running
        if (stream) (void)hipStreamSynchronize(stream);
        for (StepGraphs &g : graphs) g.destroy();
        for (void *p : allocs) (void)hipFree(p);
        if (n_host) (void)hipHostFree(n_host);
        if (stream) (void)hipStreamDestroy(stream);
    }
};

static thread_local std::string g_create_error;

#define DSMC_API_BEGIN(ctx) \
    if (!(ctx)) return DSMC_EINVAL; \
    try {
#define DSMC_API_END(ctx)                                                   \
    return DSMC_OK;                                                         \
    }                                                                       \
    catch (const Error &e) { (ctx)->err = e.what(); return (dsmc_status)e.status; } \
    catch (const std::exception &e) { (ctx)->err = e.what(); return DSMC_EHIP; }

static void fail(int status, const std::string &msg) { throw Error(status, msg); }

// ---------------------------------------------------------------------------
// Parameter preparation
// ---------------------------------------------------------------------------
static TrapDev make_trapdev(const dsmc_config &c, const dsmc_trap &t, int index, int key_base,
                            int atom_begin)
{
    TrapDev d;
    std::memset(&d, 0, sizeof d);
    d.kind = t.kind;
    for (int k = 0; k < 3; ++k) {
        d.nc[k] = t.nc[k];
        d.hw[k] = t.half_width[k];
        d.gmin[k] = -1.0 * t.half_width[k];
        d.len[k] = (2.0 * t.half_width[k]) / (double)t.nc[k];
        d.inv_len[k] = 1.0 / d.len[k];
        d.f_hw[k] = (float)t.half_width[k];
        d.f_inv_len[k] = (float)d.inv_len[k];
    }
    d.f32_index = t.nc[0] <= 256 && t.nc[1] <= 256 && t.nc[2] <= 256;
    d.n_cells = t.nc[0] * t.nc[1] * t.nc[2];
    d.key_base = key_base;
    d.atom_begin = atom_begin;
    d.n_atoms0 = t.n_atoms;
    d.cell_vol = d.len[0] * d.len[1] * d.len[2];
    d.B0 = t.B0; d.dBdx = t.dBdx; d.d2Bdx2 = t.d2Bdx2; d.dBdz = t.dBdz;
    d.mu = t.mu;
    d.neg_mu_over_m = (-t.mu) / c.mass;
    // an empty trap (allowed in a batch) has no cell to collide in
    d.alpha = t.n_atoms > 0 ? t.n_real / (double)t.n_atoms : 0.0;
    d.coll_c1 = d.alpha * c.lpc * c.dt / d.cell_vol;
    d.coll_c1s = d.coll_c1 * c.sigma;
    double Tm = t.T;
    double Tax[3];
    for (int k = 0; k < 3; ++k) Tax[k] = t.T_axis[k] > 0.0 ? t.T_axis[k] : t.T;
    if (t.T_axis[0] > 0.0 || t.T_axis[1] > 0.0 || t.T_axis[2] > 0.0) Tm = (Tax[0] + Tax[1] + Tax[2]) / 3.0;
    d.sigvrmax0 = std::sqrt(16. * kKB * Tm / (kPiRef * c.mass)) * c.sigma;
    d.kT_cut = t.eta_start > 0.0 ? kKB * t.T_cut : 0.0;
    d.eta_start = t.eta_start; d.eta_end = t.eta_end; d.eta_steps = t.eta_steps;
    d.T_init = t.T;
    for (int k = 0; k < 3; ++k) d.T_axis[k] = Tax[k];
    d.periodic = t.kind == DSMC_TRAP_BOX;
    d.stream = (uint32_t)(index + t.philox_stream);
    d.f_B0 = (float)t.B0; d.f_dBdx = (float)t.dBdx; d.f_d2Bdx2 = (float)t.d2Bdx2;
    d.f_dBdz = (float)t.dBdz;
    d.f_neg_mu_over_m = (float)d.neg_mu_over_m;
    d.f_mu_dBdz = (float)(t.mu * t.dBdz);
    return d;
}

static void validate(const dsmc_config *c, const dsmc_trap *traps, int n_traps)
{
    if (!c || !traps) fail(DSMC_EINVAL, "null config or traps");
    if (c->precision != DSMC_FP64_PLAIN && c->precision != DSMC_FP32_KAHAN)
        fail(DSMC_EINVAL, "precision must be DSMC_FP64_PLAIN or DSMC_FP32_KAHAN");
    if (n_traps < 1) fail(DSMC_EINVAL, "n_traps must be >= 1");
    if (c->precision == DSMC_FP64_PLAIN && n_traps != 1)
        fail(DSMC_ENOTSUP, "the FP64 form runs one trap; use DSMC_FP32_KAHAN for batches");
    if (n_traps > fused_max_traps()) fail(DSMC_EINVAL, "too many traps");
    if (!(c->dt > 0.0) || !(c->mass > 0.0) || !(c->sigma >= 0.0))
        fail(DSMC_EINVAL, "dt and mass must be > 0, sigma >= 0");
    if (c->lpc < 1) fail(DSMC_EINVAL, "lpc must be >= 1");
    if (c->obs_capacity < 0 || (long long)c->obs_capacity * n_traps > (1LL << 28))
        fail(DSMC_EINVAL, "obs_capacity out of range");
    if (c->precision == DSMC_FP32_KAHAN && c->lpc != 1)
        fail(DSMC_ENOTSUP, "the FP32 form collides every motion step (lpc = 1)");
    if (c->spin && c->spin_substeps < 1) fail(DSMC_EINVAL, "spin_substeps must be >= 1");
    if ((c->evaporation & DSMC_EVAP_SPIN) && !c->spin)
        fail(DSMC_EINVAL, "spin-loss evaporation needs spin evolution");
    if (c->pair_mode != DSMC_PAIR_UNIFORM && c->pair_mode != DSMC_PAIR_REFERENCE)
        fail(DSMC_EINVAL, "bad pair_mode");
    if (c->sort_mode != DSMC_SORT_INCREMENTAL && c->sort_mode != DSMC_SORT_FULL)
        fail(DSMC_EINVAL, "bad sort_mode");
    if (c->mcwf && (c->precision != DSMC_FP64_PLAIN || !c->spin))
        fail(DSMC_ENOTSUP, "the spin-flip model runs in the FP64 form with spin evolution");
    const int bs = c->block_size;
    if (bs != 0 && bs != 64 && bs != 128 && bs != 256 && bs != 512 && bs != 1024)
        fail(DSMC_EINVAL, "block_size must be 0, 64, 128, 256, 512 or 1024");
    long long total = 0, keys = 0;
    for (int t = 0; t < n_traps; ++t) {
        const dsmc_trap &tr = traps[t];
        if (tr.kind < DSMC_TRAP_IP || tr.kind > DSMC_TRAP_BOX) fail(DSMC_EINVAL, "bad trap kind");
        if (tr.n_atoms < 0) fail(DSMC_EINVAL, "n_atoms < 0");
        for (int k = 0; k < 3; ++k) {
            if (tr.nc[k] < 1) fail(DSMC_EINVAL, "nc must be >= 1");
            if (!(tr.half_width[k] > 0.0)) fail(DSMC_EINVAL, "half_width must be > 0");
        }
        if (!(tr.T > 0.0)) fail(DSMC_EINVAL, "T must be > 0");
        if (tr.kind == DSMC_TRAP_QUADRUPOLE && !(tr.mu * tr.dBdz > 0.0))
            fail(DSMC_EINVAL, "quadrupole needs mu * dBdz > 0");
        if (tr.n_atoms > 0 && !(tr.n_real > 0.0)) fail(DSMC_EINVAL, "n_real must be > 0");
        if (tr.kind == DSMC_TRAP_BOX && (c->spin || (c->evaporation & DSMC_EVAP_SPIN)))
            fail(DSMC_EINVAL, "the periodic box has no field for spin evolution");
        total += tr.n_atoms;
        keys += (long long)tr.nc[0] * tr.nc[1] * tr.nc[2] + 1;
    }
    if (total < 1) fail(DSMC_EINVAL, "no atoms");
    if (total > (1LL << 30)) fail(DSMC_EINVAL, "more than 2^30 atoms");
    if (keys + 1 > (1LL << 31) - 1) fail(DSMC_EINVAL, "too many cells");
}

// ---------------------------------------------------------------------------
// Creation
// ---------------------------------------------------------------------------
static void build_context(dsmc_ctx *x, const dsmc_config *c, const dsmc_trap *traps, int n_traps)
{
    x->cfg = *c;
    x->traps.assign(traps, traps + n_traps);
    x->T = n_traps;
    x->fp32 = c->precision == DSMC_FP32_KAHAN;
    x->block = c->block_size ? c->block_size : 256;
    // DSMC_STEP_FUSED=1: dsmc_step runs the collisions inside the move kernel
    // (the fused step) instead of the collide and move kernels one after the
    // other; the results are bitwise the same.  The fused step is slower on
    // MI355X (its collision code holds the kernel to four waves per SIMD,
    // where the move alone streams at six), so it is not the default.
    if (const char *e = std::getenv("DSMC_STEP_FUSED")) x->split_step = std::atoi(e) == 0;
    DSMC_HIP(hipGetDevice(&x->device));
    DSMC_HIP(hipStreamCreateWithFlags(&x->stream, hipStreamNonBlocking));

    int kb = 0, ab = 0;
    for (int t = 0; t < n_traps; ++t) {
        x->key_base.push_back(kb);
        x->atom_begin.push_back(ab);
        x->tdev.push_back(make_trapdev(*c, traps[t], t, kb, ab));
        kb += traps[t].nc[0] * traps[t].nc[1] * traps[t].nc[2] + 1;
        ab += traps[t].n_atoms;
    }
    x->dead_key = (uint32_t)kb;
    x->key_base.push_back(kb);
    x->atom_begin.push_back(ab);
    x->n_cap = ab;
    x->n_keys = kb + 1;
    x->ncells = traps[0].nc[0] * traps[0].nc[1] * traps[0].nc[2];
    int bits = 1;
    while ((1LL << bits) < (long long)x->n_keys) ++bits;
    x->key_bits = bits;
    x->passes = bits <= kRadixBits ? 1 : div_up(bits, kRadixBits);
    const long long per_rec = (long long)sizeof(dsmc_observables) * n_traps;
    x->obs_cap = c->obs_capacity > 0
                     ? c->obs_capacity
                     : (int)std::max<long long>(16, std::min<long long>(65536, (256LL << 20) / per_rec));

    const int N = x->n_cap;
    x->d_traps = x->alloc<TrapDev>(n_traps, false);
    DSMC_HIP(hipMemcpyAsync(x->d_traps, x->tdev.data(), sizeof(TrapDev) * n_traps,
                            hipMemcpyHostToDevice, x->stream));
    x->d_key_base = x->alloc<int>(n_traps + 1, false);
    DSMC_HIP(hipMemcpyAsync(x->d_key_base, x->key_base.data(), sizeof(int) * (n_traps + 1),
                            hipMemcpyHostToDevice, x->stream));
    x->key_a = x->alloc<uint32_t>(N);
    x->key_b = x->alloc<uint32_t>(N);
    x->val_a = x->alloc<uint32_t>(N);
    x->val_b = x->alloc<uint32_t>(N);
    sort_scratch_bind(x->sort, N, x->alloc<char>(sort_scratch_bytes(N)));
    if (x->fp32) x->sigvrmax_f = x->alloc<float>(x->n_keys);
    else x->sigvrmax = x->alloc<double>(x->n_keys);
    x->obs_log = x->alloc<dsmc_observables>((size_t)(x->obs_cap + 1) * n_traps);
    x->step_buf = x->alloc<long long>(2);
    x->step_save = x->alloc<long long>(1);
    x->coll_accum = x->alloc<unsigned long long>(n_traps);
    x->n_dev = x->alloc<int>(4);
    // one pinned block: the counts, and behind them the FP64 form's record
    DSMC_HIP(hipHostMalloc((void **)&x->n_host, 64 + sizeof(dsmc_observables), hipHostMallocDefault));
    if (!x->fp32) x->obs_host = (dsmc_observables *)((char *)x->n_host + 64);
    // incremental re-sort (its counts start cleared)
    resort_scratch_bind(x->res, N, x->alloc<char>(resort_scratch_bytes(N), false));
    resort_clear_counts(x->res, x->stream, nullptr);
    // one entry per block of the smallest move block size, whole 2048-slot
    // tiles (never-written entries stay zero)
    x->blk_dead = x->alloc<uint32_t>((size_t)div_up(N, 2048) * (2048 / 64) + 64);
    x->mask_moved = x->alloc<uint64_t>(resort_mask_words(N));

    if (!x->fp32) {
        for (int b = 0; b < 2; ++b) {
            // one block for the nine arrays (each 256-byte aligned): the
            // buffer that is not current is also the staging of host reads
            const size_t pad = ((size_t)N + 31) & ~(size_t)31;
            double *block = x->alloc<double>(9 * pad);
            for (int k = 0; k < 9; ++k) x->ps[b].d[k] = block + k * pad;
            x->ps[b].id = x->alloc<int>(N);
            x->ps[b].up = x->alloc<uint8_t>(N);
            for (int k = 0; k < 4; ++k) x->ps[b].psi[k] = c->spin ? x->alloc<double>(N) : nullptr;
        }
        const int C1 = x->ncells + 1;
        x->start_end = x->alloc<int2>(C1);
        x->count = x->alloc<int>(C1);
        x->prefix = x->alloc<int>(C1);
        x->coll_count = x->alloc<int>(C1);
        x->scan_partial = x->alloc<int>(scan_partials(N));
        x->tag = x->alloc<int>(N);
        x->cmap = x->alloc<uint32_t>(N);
        x->evap_pos_d = x->alloc<double>(3 * (size_t)N);
        x->evap_vel_d = x->alloc<double>(3 * (size_t)N);
        x->partials = x->alloc<double>((size_t)observe_plain_blocks(N) * 5 + 8);
        x->evap_accum = x->alloc<double>(2);
        if (c->mcwf) {
            x->pops = x->alloc<double>(2 * (size_t)N);
            x->flips = x->alloc<unsigned long long>(1);
        }
        x->ctl = x->alloc<PlainCtl>(2);
        // few allocations: each costs a small context's creation 4 us
        const size_t row = ((size_t)N + 63) & ~(size_t)63, words = resort_mask_words(N);
        x->key_f = x->alloc<uint32_t>(5 * row);
        uint64_t *const masks = x->alloc<uint64_t>(3 * words);
        for (int b = 0; b < 2; ++b) {
            x->srt_k[b] = x->key_f + (1 + 2 * b) * row;
            x->srt_v[b] = x->key_f + (2 + 2 * b) * row;
            x->mask_d2[b] = masks + b * words;
        }
        x->mask_last = masks + 2 * words;
        x->rec64 = x->alloc<double>((size_t)std::min(c->lpc, kMaxSub) * kStepRec * step_rec_stride(N));
        x->cc_tagged = x->alloc<unsigned long long>(C1);
    } else {
        for (int b = 0; b < 2; ++b) {
            x->fs[b].r = x->alloc<f4>(rec_elems(N));
            for (int k = 0; k < 3; ++k) x->fs[b].s[k] = c->spin ? x->alloc<float>(N) : nullptr;
        }
        if (c->spin) {
            const int S = std::max(1, c->spin_substeps);
            const float dts = (float)(c->dt / S);
            std::vector<float> tau((size_t)S + 1, 0.0f);   // (the kernel reads one ahead)
            if (c->spin_interp)
                for (int k = 0; k < S; ++k) tau[k] = ((float)k + 0.5f) * dts;
            x->spin_tau = x->alloc<float>(tau.size(), false);
            DSMC_HIP(hipMemcpyAsync(x->spin_tau, tau.data(), tau.size() * sizeof(float),
                                    hipMemcpyHostToDevice, x->stream));
            DSMC_HIP(hipStreamSynchronize(x->stream));   // (tau goes)
        }
        x->mask_dead = x->alloc<uint64_t>(resort_mask_words(N));
        x->srt_k[0] = x->key_b; x->srt_v[0] = x->val_b;
        x->srt_k[1] = x->alloc<uint32_t>(N); x->srt_v[1] = x->alloc<uint32_t>(N);
        x->cell_start = x->alloc<uint32_t>(x->n_keys, false);
        x->cell_end = x->alloc<uint32_t>(x->n_keys, false);
        x->ts_buf[0] = x->alloc<int>(n_traps + 1, false);
        x->ts_buf[1] = x->alloc<int>(n_traps + 1, false);
        DSMC_HIP(hipMemcpyAsync(x->trap_start(), x->atom_begin.data(), sizeof(int) * (n_traps + 1),
                                hipMemcpyHostToDevice, x->stream));
        x->acc = x->alloc<double>((size_t)n_traps * kAccK);
        x->rec.stride = obs_record_stride(N);
        x->rec.trap = x->alloc<int>((size_t)x->rec.stride);
        x->rec.sum = x->alloc<double>((size_t)x->rec.stride * kAccK);
        x->rec.acc_over = x->acc;
        x->rec.lvl2 = x->alloc<double>((size_t)n_traps * kMaxFinalizeP * kAccK);
        x->rec.cnt = x->alloc<unsigned int>((size_t)n_traps);
        for (int t = 0; t < n_traps; ++t) x->max_trap_atoms = std::max(x->max_trap_atoms, traps[t].n_atoms);
        x->acc2 = x->alloc<double>((size_t)n_traps * kAccK);
        x->scan_partial = x->alloc<int>(scan_partials(N));
        if (!x->split_step) x->edge_sm = x->alloc<uint64_t>((size_t)edge_sm_spans(N));
        x->obs_first = x->alloc<int>((size_t)n_traps);
        x->obs_last = x->alloc<int>((size_t)n_traps);
        x->evap_pos_f = x->alloc<float>(3 * (size_t)N);
        x->evap_vel_f = x->alloc<float>(3 * (size_t)N);
    }
    DSMC_HIP(hipMemcpyAsync(x->n_dev, &x->n_cap, sizeof(int), hipMemcpyHostToDevice, x->stream));
    DSMC_HIP(hipStreamSynchronize(x->stream));
}

// ---------------------------------------------------------------------------
// Step pieces: FP64 form
// ---------------------------------------------------------------------------
static CollideParams collide_params(const dsmc_ctx *x)
{
    CollideParams cp;
    std::memset(&cp, 0, sizeof cp);
    cp.seed = x->cfg.seed;
    cp.dt = x->cfg.dt;
    cp.lpc = (double)x->cfg.lpc;
    cp.sigma = x->cfg.sigma;
    cp.pair_mode = x->cfg.pair_mode;
    return cp;
}

static void plain_index(dsmc_ctx *x)
{
    // an even number of radix passes sorts in place: the sorted keys are then
    // the array that the index overwrites
    if (x->sorted_key && x->passes % 2 == 0) x->sorted_key = x->key_a;
    x->index_stale = false;
    launch_index_plain(x->tdev[0], x->ps[x->cur], x->key_a, x->n_dev, x->n_cap, x->stream, &x->prof);
}

// Sort keys in key_a with identity values; results in (sorted_key, perm).
static void run_sort(dsmc_ctx *x, const int *n_dev)
{
    const bool odd = (x->passes % 2) == 1;
    uint32_t *ok = odd ? x->key_b : x->key_a, *ov = odd ? x->val_b : x->val_a;
    // sorting in place takes an even number of passes
    RadixPlan plan = radix_plan(x->n_cap, x->key_bits);
    if (!odd && plan.passes % 2) plan = radix_plan(x->n_cap, x->key_bits, kRadixBits);
    uint32_t *ak = odd ? x->res.alt_k : x->key_b, *av = odd ? x->res.alt_v : x->val_b;
    radix_sort(x->key_a, nullptr, ak, av, ok, ov, n_dev, plan, x->sort, x->stream, &x->prof);
    x->sorted_key = ok;
    x->perm = ov;
    x->perm_mask = -1;
}

static void plain_sort(dsmc_ctx *x)
{
    run_sort(x, x->n_dev);
    launch_gather_plain(x->ps[x->cur ^ 1], x->ps[x->cur], x->perm, x->n_dev, x->n_cap,
                        x->cfg.spin, x->stream, &x->prof);
    x->cur ^= 1;
}

static void plain_table(dsmc_ctx *x)
{
    launch_cell_table_plain(x->sorted_key, x->n_dev, x->n_cap, x->start_end, x->count, x->prefix,
                            x->ncells, x->stream, &x->prof);
}

static void plain_collide(dsmc_ctx *x)
{
    launch_collide_plain(x->tdev[0], collide_params(x), x->ps[x->cur], x->sigvrmax, x->prefix,
                         x->coll_count, x->coll_accum, x->ncells, (uint32_t)x->step, x->stream,
                         &x->prof);
    x->coll_steps++;
}

static SpinParams spin_params(const dsmc_ctx *x)
{
    SpinParams sp;
    sp.gs = x->cfg.gs;
    sp.dt = x->cfg.dt;
    sp.substeps = x->cfg.spin_substeps;
    sp.dt_spin = x->cfg.spin_substeps > 0 ? x->cfg.dt / x->cfg.spin_substeps : x->cfg.dt;
    sp.interp = x->cfg.spin_interp;
    return sp;
}

static void plain_spin(dsmc_ctx *x)
{
    const SpinParams sp = spin_params(x);
    launch_spin_plain(x->tdev[0], sp, x->ps[x->cur], x->n_dev, x->n_cap, x->stream, &x->prof);
}

// Spin-flip model pieces (FP64 form).  The flip draws use the number of
// collision steps taken so far (this one included) as counter word 1.
static void plain_local_pops(dsmc_ctx *x)
{
    launch_local_pops_plain(x->tdev[0], x->ps[x->cur], x->pops, x->n_dev, x->n_cap, x->stream,
                            &x->prof);
}

static FlipParams flip_params(const dsmc_ctx *x)
{
    FlipParams fp;
    std::memset(&fp, 0, sizeof fp);
    fp.seed = x->cfg.seed;
    fp.mass = x->cfg.mass;
    fp.gap = 2.0 * x->tdev[0].mu;
    fp.step = (uint32_t)x->coll_steps;
    return fp;
}

static void plain_flip(dsmc_ctx *x)
{
    const FlipParams fp = flip_params(x);
    launch_flip_plain(x->tdev[0], fp, x->ps[x->cur], x->pops, x->flips, x->n_dev, x->n_cap,
                      x->stream, &x->prof);
}

static DecayParams decay_params(const dsmc_ctx *x)
{
    DecayParams dp;
    dp.dt = x->cfg.lpc * x->cfg.dt;
    dp.sigma = x->cfg.sigma;
    dp.mass = x->cfg.mass;
    return dp;
}

static void plain_decay(dsmc_ctx *x)
{
    const DecayParams dp = decay_params(x);
    launch_decay_plain(x->tdev[0], dp, x->ps[x->cur], x->n_dev, x->n_cap, x->stream, &x->prof);
}

static double e_cut_now(const dsmc_ctx *x, long long step)
{
    const TrapDev &t = x->tdev[0];
    if (!(x->cfg.evaporation & DSMC_EVAP_ENERGY) || t.kT_cut <= 0.0) return 0.0;
    const double f = t.eta_steps > 0 ? std::min((double)step / (double)t.eta_steps, 1.0) : 1.0;
    return (t.eta_start + (t.eta_end - t.eta_start) * f) * t.kT_cut;
}

static void plain_evap_tag(dsmc_ctx *x)
{
    EvapParams ep;
    ep.mass = x->cfg.mass;
    ep.e_cut = e_cut_now(x, x->step);
    ep.spin_loss = (x->cfg.evaporation & DSMC_EVAP_SPIN) ? 1 : 0;
    ep.pad = 0;
    launch_evap_tag_plain(x->tdev[0], ep, x->ps[x->cur], x->tag, x->evap_pos_d, x->evap_vel_d,
                          x->evap_accum, x->n_dev, x->n_cap, x->stream, &x->prof);
}

static void plain_compact(dsmc_ctx *x)
{
    compaction_map(x->tag, x->n_dev, x->n_cap, x->cmap, x->n_dev + 2, x->scan_partial, x->stream,
                   &x->prof);
    launch_gather_plain(x->ps[x->cur ^ 1], x->ps[x->cur], x->cmap, x->n_dev + 2, x->n_cap,
                        x->cfg.spin, x->stream, &x->prof, x->n_dev, x->n_host);
    x->cur ^= 1;
}

// The record of the sums that a move or launch_observe_plain left.
static void plain_record(dsmc_ctx *x, dsmc_observables *slot, long long step)
{
    launch_observe_finalize_plain(x->n_dev, x->n_cap, x->partials, slot, x->coll_accum, x->evap_accum, step,
                                  x->stream, &x->prof);
}

// ---------------------------------------------------------------------------
// FP64 form, whole steps.
// ---------------------------------------------------------------------------
// Drops the removed atoms that still hold slots: the state is then that of the
// reference's compaction after every motion step, with the tags of the last.
static void plain_settle(dsmc_ctx *x)
{
    if (!x->lazy_dead) return;
    const PlainCtl *c = x->ctl + x->csel;
    int *stencil = (int *)x->res.alt_k;
    uint32_t *map = x->res.alt_v;
    launch_prev_dead_stencil(x->key_f, x->mask_last, c, x->n_cap, x->dead_key, stencil, x->stream);
    compaction_map(stencil, &c->slots, x->n_cap, map, x->n_dev + 2, x->scan_partial, x->stream, nullptr);
    launch_last_tags(map, x->mask_last, x->n_dev + 2, x->n_cap, x->tag, x->stream);
    launch_dead_stencil(x->key_f, &c->slots, x->n_cap, x->dead_key, stencil, x->stream);
    compaction_map(stencil, &c->slots, x->n_cap, x->cmap, x->n_dev, x->scan_partial, x->stream, nullptr);
    launch_gather_plain(x->ps[x->cur ^ 1], x->ps[x->cur], x->cmap, x->n_dev, x->n_cap, x->cfg.spin,
                        x->stream, nullptr);
    x->cur ^= 1;
    launch_set_ctl(x->ctl + x->csel, x->step, (unsigned)x->coll_steps, x->n_dev, x->stream);
    x->lazy_dead = false;
    x->sorted_ok = false;
    x->keys_ok = false;
    x->bucketed = false;
}

static void plain_need_acc(dsmc_ctx *x)
{
    if (!x->acc_stale) return;
    launch_accel_plain(x->tdev[0], x->ps[x->cur], x->n_cap, x->stream, nullptr);
    x->acc_stale = false;
}

static void plain_need_tables(dsmc_ctx *x)
{
    if (!x->tables_stale) return;
    launch_cell_table_plain(x->sorted_key, x->n_dev + 3, x->n_cap, x->start_end, x->count, x->prefix,
                            x->ncells, x->stream, nullptr);
    launch_untag_counts(x->cc_tagged, (unsigned)x->coll_steps, x->ncells, x->coll_count, x->stream);
    x->tables_stale = false;
}

// Before a single sort: key_a as the index and the sort of the last step's
// calls leave it, in place sorted (an even number of passes) or the keys of the
// slots as they were before the sort.
static void plain_need_index(dsmc_ctx *x)
{
    if (!x->index_stale) return;
    const bool in_place = x->passes % 2 == 0, gaps = x->perm_mask >= 0;
    const int *sorted = x->n_dev + 3;
    uint32_t *dst = !in_place && gaps ? x->key_f : x->key_a;
    if (!in_place && gaps) fill_u32(dst, kNoSlot, x->n_cap, x->stream, nullptr);
    launch_keys_by_slot(x->sorted_key, in_place ? nullptr : x->perm, sorted, x->n_cap, dst, x->stream);
    if (!in_place && gaps) {   // the slots were counted without the removed atoms (n_dev[1]: the capacity)
        int *stencil = (int *)x->res.alt_k;
        launch_dead_stencil(dst, x->n_dev + 1, x->n_cap, kNoSlot, stencil, x->stream);
        compaction_map(stencil, x->n_dev + 1, x->n_cap, x->cmap, x->n_dev + 2, x->scan_partial, x->stream, nullptr);
        gather_u32(x->key_a, dst, x->cmap, x->n_dev + 2, x->n_cap, x->stream, nullptr);
    }
    x->index_stale = false;
}

// Before a single call of the FP64 form: everything in memory as the calls
// leave it.  What the call changes is not in the order of the last step's sort.
static void plain_enter(dsmc_ctx *x)
{
    plain_settle(x);
    plain_need_acc(x);
    plain_need_tables(x);
    x->ctl_live = false;
    x->sorted_ok = false;
    x->keys_ok = false;
    x->bucketed = false;
}

// Small contexts re-sort in the finalize's launch; the next sort finds its
// keys and permutation in the other sort buffer.
static bool resort_early(const dsmc_ctx *x) { return x->n_cap <= kScanSlots; }

// The first phase of the re-sort that follows a move of n slots with the new
// keys key (x->bucketed: wanted), or the whole of it, for the finalize's launch.
static ResortWork resort_work(dsmc_ctx *x, const uint32_t *key, const int *n, const uint64_t *mask_dead)
{
    ResortWork w;
    if (!x->bucketed) return w;
    const bool may_remove = x->cfg.evaporation != 0;
    if (resort_early(x)) {
        w.merge = resort_merge_args(x->res, x->srt_k[x->srt_cur], n, x->dead_key, x->mask_moved, mask_dead,
                                    may_remove, x->srt_k[x->srt_cur ^ 1], x->srt_v[x->srt_cur ^ 1]);
        w.merge.key_new = key;
        return w;
    }
    if (!x->counts_clear) resort_clear_counts(x->res, x->stream, &x->prof);
    x->counts_clear = false;
    w.list = resort_list_args(x->res, key, n, x->mask_moved, mask_dead, may_remove);
    return w;
}

// Substeps of one launch: their log records are written by different blocks,
// so no two may share a place of the ring.
static int max_substeps(const dsmc_ctx *x) { return std::min(kMaxSub, x->obs_cap); }

// L motion substeps from the current one, with the sort and the collisions
// when a collision step begins (L reaches at most to its end).
static void plain_substeps(dsmc_ctx *x, int L)
{
    const int lpc = x->cfg.lpc, phase = (int)(x->step % lpc);
    const bool after = phase == 0, resort = resort_supported(x->n_cap);
    const PlainCtl *c = x->ctl + x->csel;
    const TrapDev &t = x->tdev[0];
    if (after) {
        uint32_t *ok = x->srt_k[x->srt_cur ^ 1], *ov = x->srt_v[x->srt_cur ^ 1];
        if (x->sorted_ok && x->bucketed) {
            if (!resort_early(x)) resort_merge(resort_merge_args(x->res, x->srt_k[x->srt_cur], &c->slots, x->dead_key, x->mask_moved,
                                           x->mask_d2[x->mpar], x->lazy_dead, ok, ov), x->stream, &x->prof);
        } else {
            if (!x->keys_ok)
                launch_index_plain(t, x->ps[x->cur], x->key_f, &c->slots, x->n_cap, x->stream, &x->prof);
            radix_sort(x->key_f, nullptr, x->res.alt_k, x->res.alt_v, ok, ov, &c->slots,
                       radix_plan(x->n_cap, x->key_bits), x->sort, x->stream, &x->prof);
            resort_samples(x->res, ok, x->stream, &x->prof);
        }
        x->srt_cur ^= 1;
        x->sorted_key = ok;
        x->perm = ov;
        x->perm_mask = x->lazy_dead ? x->mpar : -1;
        x->mpar ^= 1;
        launch_collide_step(t, collide_params(x), x->ps[x->cur], ok, ov, c, x->n_cap, x->sigvrmax,
                            x->cc_tagged, x->coll_accum, x->n_dev + 3, x->res.b, x->stream, &x->prof);
        x->counts_clear = true;
    }
    PlainStepParams p;
    std::memset(&p, 0, sizeof p);
    p.dt = x->cfg.dt;
    p.mass = x->cfg.mass;
    p.spin = spin_params(x);
    p.flip = flip_params(x);
    p.decay = decay_params(x);
    p.spin_loss = (x->cfg.evaporation & DSMC_EVAP_SPIN) ? 1 : 0;
    p.energy_cut = (x->cfg.evaporation & DSMC_EVAP_ENERGY) ? 1 : 0;
    p.lpc = lpc;
    p.phase = phase;
    p.L = L;
    p.fast_key = t.nc[0] < (1 << 20) && t.nc[1] < (1 << 20) && t.nc[2] < (1 << 20);
    p.dead_key = x->dead_key;
    const bool sorted = after || x->sorted_ok;
    p.key_prev = sorted ? x->srt_k[x->srt_cur] : nullptr;
    p.mask_moved = x->mask_moved; p.mask_dead = x->mask_d2[x->mpar]; p.mask_last = x->mask_last;
    launch_move_step(x->cfg.spin != 0, x->cfg.mcwf != 0, t, p, x->ps[x->cur],
                     x->ps[after ? x->cur ^ 1 : x->cur], after ? x->perm : nullptr,
                     !after && x->lazy_dead ? x->key_f : nullptr, after, c, x->key_f, x->pops,
                     x->evap_pos_d, x->evap_vel_d, x->rec64, step_rec_stride(x->n_cap), x->n_cap,
                     x->stream, &x->prof);
    x->bucketed = sorted && resort && phase + L == lpc;
    const ResortWork work = resort_work(x, x->key_f, after ? &c->alive : &c->slots, x->mask_d2[x->mpar]);
    launch_step_finalize(p, after, x->rec64, step_rec_stride(x->n_cap), c, x->ctl + (x->csel ^ 1),
                         x->coll_accum, x->evap_accum, x->obs_log, x->obs_cap, work, x->stream, &x->prof);
    x->csel ^= 1;
    if (after) {
        x->cur ^= 1;
        x->sorted_ok = true;
        x->tables_stale = true;
        x->index_stale = true;
        x->coll_steps++;
    }
    x->keys_ok = true;
    x->lazy_dead = x->cfg.evaporation != 0;
    if (!x->cfg.mcwf) x->acc_stale = true;
    x->step += L;
}

// ---------------------------------------------------------------------------
// Step pieces: FP32 form (parity p: alive count in n_dev[p], state in fs[p])
// ---------------------------------------------------------------------------
static MoveParams move_params(const dsmc_ctx *x)
{
    MoveParams mp;
    std::memset(&mp, 0, sizeof mp);
    mp.dt = x->cfg.dt;
    mp.f_dt = (float)x->cfg.dt;
    mp.mass = x->cfg.mass;
    mp.f_half_mass = (float)(0.5 * x->cfg.mass);
    mp.spin = x->cfg.spin;
    mp.substeps = std::max(1, x->cfg.spin_substeps);
    const double dts = mp.dt / mp.substeps;
    mp.f_spin_w = (float)(x->cfg.gs * kMuB * dts / kHbar);
    mp.spin_tau = x->spin_tau;
    mp.spin_loss = (x->cfg.evaporation & DSMC_EVAP_SPIN) ? 1 : 0;
    mp.energy_cut = (x->cfg.evaporation & DSMC_EVAP_ENERGY) ? 1 : 0;
    mp.n_traps = x->T;
    mp.obs_cap = x->obs_cap;
    mp.dead_key = x->dead_key;
    mp.count_moved = 0;
    mp.blk_dead = x->blk_dead;
    mp.mask_moved = x->mask_moved;
    mp.mask_dead = x->mask_dead;
    return mp;
}

static void fused_index(dsmc_ctx *x)
{
    launch_index_fused(x->d_traps, x->dead_in_state ? x->d_key_base : x->trap_start(), x->T, x->fs[x->cur],
                       x->key_a, x->n_dev + x->cur, x->n_cap, x->dead_key, x->dead_in_state, x->stream, &x->prof);
    x->tbl_valid = false;   // the new keys decide the trap ranges of the next sort
}

// Stable sort of the keys in key_a into the other sort buffer.  When the
// current state is in sorted order of the previous sort's keys (after a
// sorted move), only the atoms whose key changed are placed among the rest;
// the result is the same permutation.
static void fused_sort(dsmc_ctx *x)
{
    const int *n = x->n_dev + x->cur;
    uint32_t *ok = x->srt_k[x->srt_cur ^ 1], *ov = x->srt_v[x->srt_cur ^ 1];
    if (x->srt_valid && x->bucketed) {
        if (!resort_early(x)) resort_merge(resort_merge_args(x->res, x->srt_k[x->srt_cur], n, x->dead_key, x->mask_moved, x->mask_dead,
                                       x->dead_in_state, ok, ov), x->stream, &x->prof);
    } else {
        radix_sort(x->key_a, nullptr, x->res.alt_k, x->res.alt_v, ok, ov, n,
                   radix_plan(x->n_cap, x->key_bits), x->sort, x->stream, &x->prof);
        resort_samples(x->res, ok, x->stream, &x->prof);
    }
    x->bucketed = false;
    x->srt_cur ^= 1;
    x->sorted_key = ok;
    x->perm = ov;
    x->have_sort = true;
    x->srt_valid = false;   // the state is not yet in the new order
}

static void fused_table(dsmc_ctx *x)
{
    TableParams tp;
    tp.n_traps = x->T;
    tp.dead_key = x->dead_key;
    launch_table_fused(x->sorted_key, x->d_key_base, tp, x->n_dev + x->cur, x->n_dev + (x->cur ^ 1),
                       x->trap_start(), x->n_cap, x->stream, &x->prof);
    x->tbl_valid = true;
}

// The trap ranges and alive count of the sorted order: kept by the previous
// sorted move's finalize, else scanned from the sorted keys.
static void fused_need_table(dsmc_ctx *x)
{
    if (x->have_sort && !x->tbl_valid) fused_table(x);
}

static void fused_collide(dsmc_ctx *x)
{
    fused_need_table(x);
    launch_collide_fused(x->d_traps, x->d_key_base, x->T, collide_params(x), x->sorted_key,
                         x->perm, x->n_dev + (x->cur ^ 1), x->fs[x->cur], x->sigvrmax_f,
                         x->coll_accum, x->step_dev(), x->res.b, x->n_cap, x->stream, &x->prof);
    x->counts_clear = true;
}

// coll: the fused step (the collisions of this step run inside the move
// kernel, those of cells across its block boundaries in an edge pass before
// it); needs a pending sort.
static void fused_move(dsmc_ctx *x, bool coll = false)
{
    // atoms removed by the previous move are dropped by a sort: a second move
    // without one would move (and test) them again
    if (!x->have_sort && x->dead_in_state)
        fail(DSMC_ESTATE, "the last move removed atoms: sort before moving again");
    fused_need_table(x);
    // after a sort the alive count of the sorted order is n_dev[cur ^ 1]
    const int *n = x->have_sort ? x->n_dev + (x->cur ^ 1) : x->n_dev + x->cur;
    MoveParams mp = move_params(x);
    // a sorted move also counts, per move block, the atoms whose key changed:
    // the input of the next step's incremental re-sort
    if (x->have_sort) {
        mp.count_moved = 1;
        mp.key_prev = x->sorted_key;
    }
    StepCollide sc;
    if (coll) {
        if (!x->have_sort) fail(DSMC_ESTATE, "the fused step needs a sorted state");
        sc.cp = collide_params(x);
        sc.sigvrmax = x->sigvrmax_f;
        sc.edge_sm = x->edge_sm;
        sc.coll_accum = x->coll_accum;
        sc.dry = 0;
        launch_collide_edges(x->d_traps, x->d_key_base, x->T, sc.cp, x->sorted_key, x->perm, n,
                             x->fs[x->cur], x->sigvrmax_f, x->coll_accum, x->step_dev(),
                             64 * x->apt, x->n_cap, x->stream, &x->prof);   // one wave's span
    }
    launch_move_fused(x->block, x->apt, x->d_traps, mp, x->fs[x->cur], x->fs[x->cur ^ 1],
                      x->have_sort ? x->perm : nullptr, x->trap_start(), n, x->key_a,
                      x->evap_pos_f, x->evap_vel_f, x->rec, x->step_dev(), x->n_cap, x->stream,
                      &x->prof, coll ? &sc : nullptr);
    // a sorted move's finalize also leaves the next sort's trap ranges and
    // alive count (the removed atoms go to the end), and runs the first phase
    // of the incremental re-sort that follows
    x->bucketed = x->have_sort && x->cfg.sort_mode == DSMC_SORT_INCREMENTAL && resort_supported(x->n_cap);
    const ResortWork work = resort_work(x, x->key_a, n, x->mask_dead);
    launch_obs_finalize(x->T, x->max_trap_atoms, x->block * x->apt, x->cfg.mass, x->trap_start(),
                        x->have_sort ? x->ts_buf[x->tsel ^ 1] : nullptr, x->blk_dead,
                        x->mask_dead, x->rec, x->coll_accum, x->step_dev(),
                        x->step_buf + (x->ssel ^ 1), x->obs_log, x->obs_cap,
                        x->have_sort ? x->n_dev + x->cur : nullptr, work, x->stream, &x->prof);
    x->ssel ^= 1;
    if (x->have_sort) x->tsel ^= 1;
    if (!x->have_sort)  // keep the count with the state it describes
        DSMC_HIP(hipMemcpyAsync(x->n_dev + (x->cur ^ 1), x->n_dev + x->cur, sizeof(int),
                                hipMemcpyDeviceToDevice, x->stream));
    // a sorted move leaves the state in sorted order of the last sort's keys
    // and has counted the changed keys; after an unsorted move the next sort
    // is a full one
    x->srt_valid = x->have_sort;
    x->tbl_valid = x->have_sort;
    x->have_sort = false;
    x->dead_in_state = x->cfg.evaporation != 0;
    x->cur ^= 1;
}

static void fused_step(dsmc_ctx *x)
{
    fused_sort(x);
    if (x->split_step) {   // the collide and the move as two kernels
        fused_collide(x);
        fused_move(x);
    } else {
        fused_need_table(x);
        fused_move(x, true);
    }
    x->coll_steps++;
    x->step++;
}

static bool graph_ok(const dsmc_ctx *x) { return x->cfg.use_graph && !x->prof.enabled; }

// Destroy the captured graphs.  Their earlier launches may still be in flight
// on the stream, so the stream is drained first: an executable graph is not
// destroyed while the device may still run it.
static void drop_graphs(dsmc_ctx *x)
{
    DSMC_HIP(hipStreamSynchronize(x->stream));
    for (StepGraphs &g : x->graphs) g.destroy();
}

// The steps of one pair: two FP32 steps, or two collision steps of the FP64
// form.  Every double buffer is back where it was after them.
static int graph_len(const dsmc_ctx *x) { return x->fp32 ? 2 : 2 * x->cfg.lpc; }

static void graph_body(dsmc_ctx *x)
{
    if (x->fp32) {
        fused_step(x);
        fused_step(x);
        return;
    }
    for (int k = 0; k < 2; ++k)
        for (int done = 0; done < x->cfg.lpc;) {
            const int L = std::min(x->cfg.lpc - done, max_substeps(x));
            plain_substeps(x, L);
            done += L;
        }
}

// One graph launch leaves the device idle for some 5 us, so a long graph of
// kLongPairs pairs replays them 2.2 us a step faster than pair by pair (N = 2e4
// 22.0 -> 19.8 us a step, 1e6 53.7 -> 51.4; four pairs 20.2 and 51.9).  Its
// capture costs 145 us more, what kLongFrom pairs gain: it is captured once a
// context has replayed so many (those of the present call counted), so that no
// run loses more by it than it would have without.
constexpr int kLongPairs = 8, kLongFrom = 32;

// Captures `pairs` pairs of steps, unless there already.
static void capture_steps(dsmc_ctx *x, StepGraph &g, int pairs)
{
    if (g.exec) return;
    g.destroy();   // (what a failed instantiation left)
    DSMC_HIP(hipStreamBeginCapture(x->stream, hipStreamCaptureModeThreadLocal));
    try {
        for (int k = 0; k < pairs; ++k) graph_body(x);
    } catch (...) {
        hipGraph_t broken = nullptr;
        (void)hipStreamEndCapture(x->stream, &broken);
        if (broken) (void)hipGraphDestroy(broken);
        throw;
    }
    DSMC_HIP(hipStreamEndCapture(x->stream, &g.graph));
    DSMC_HIP(hipGraphInstantiate(&g.exec, g.graph, nullptr, nullptr, 0));
}

// `times` pairs of steps.
static void graph_steps(dsmc_ctx *x, int times)
{
    StepGraphs now;
    now.srt = x->srt_cur;
    now.ssel = x->fp32 ? x->ssel : x->csel;
    now.tsel = x->fp32 ? x->tsel : x->mpar;
    now.cur = x->cur;
    if (!x->graphs[0].same(now)) {
        std::swap(x->graphs[0], x->graphs[1]);
        if (!x->graphs[0].same(now)) {   // captured with other buffers current than these
            DSMC_HIP(hipStreamSynchronize(x->stream));
            x->graphs[0].destroy();
            x->graphs[0] = now;
        }
    }
    StepGraphs &g = x->graphs[0];
    const long long step0 = x->step, cs0 = x->coll_steps;
    g.pairs_run = (int)std::min<long long>(kLongFrom, (long long)g.pairs_run + times);
    const int longs = g.pairs_run >= kLongFrom ? times / kLongPairs : 0;
    const int singles = times - longs * kLongPairs;
    if (longs > 0) capture_steps(x, g.many, kLongPairs);
    if (singles > 0) capture_steps(x, g.one, 1);
    for (int k = 0; k < longs; ++k) DSMC_HIP(hipGraphLaunch(g.many.exec, x->stream));
    for (int k = 0; k < singles; ++k) DSMC_HIP(hipGraphLaunch(g.one.exec, x->stream));
    x->step = step0 + (long long)graph_len(x) * times;
    x->coll_steps = cs0 + 2LL * times;
    // as the captured steps leave it (a graph of an earlier run may have been
    // replayed without a step of this one before it)
    x->sorted_key = x->srt_k[x->srt_cur];
    x->perm = x->srt_v[x->srt_cur];
    if (x->fp32) {
        x->have_sort = false;
        x->srt_valid = true;
        x->tbl_valid = true;
        x->dead_in_state = x->cfg.evaporation != 0;
        x->bucketed = x->cfg.sort_mode == DSMC_SORT_INCREMENTAL && resort_supported(x->n_cap);
        return;
    }
    x->perm_mask = x->cfg.evaporation ? x->mpar ^ 1 : -1;
    x->tables_stale = true;
    x->index_stale = true;
    x->acc_stale = !x->cfg.mcwf;
    x->sorted_ok = true;
    x->keys_ok = true;
    x->lazy_dead = x->cfg.evaporation != 0;
    x->bucketed = resort_supported(x->n_cap);
}

static void do_steps(dsmc_ctx *x, int n)
{
    if (!x->fp32) {
        if (n > 0 && !x->ctl_live) {
            launch_set_ctl(x->ctl + x->csel, x->step, (unsigned)x->coll_steps, x->n_dev, x->stream);
            x->ctl_live = true;
        }
        const bool resort = resort_supported(x->n_cap);
        while (n > 0) {
            const int phase = (int)(x->step % x->cfg.lpc), len = graph_len(x);
            // a graph holds the sort that follows a step (from its buckets or
            // its keys), so the state must be as one left it, at the capture
            // and at every replay: after anything else a launched step is first
            const bool as_left = resort ? x->sorted_ok && x->bucketed : x->keys_ok;
            if (graph_ok(x) && phase == 0 && n >= len && as_left) {
                const int times = n / len;
                graph_steps(x, times);
                n -= times * len;
                continue;
            }
            const int L = std::min(std::min(x->cfg.lpc - phase, n), max_substeps(x));
            plain_substeps(x, L);
            n -= L;
        }
        return;
    }
    if (x->have_sort) fail(DSMC_ESTATE, "a sort is pending: call dsmc_move_atoms first");
    int k = 0;
    if (graph_ok(x)) {
        // the graph is captured from (and replayed at) state buffer 0 with a
        // valid previous sort
        const bool need_srt = x->cfg.sort_mode == DSMC_SORT_INCREMENTAL;
        while (k < n && (x->cur == 1 || (need_srt && !x->srt_valid))) { fused_step(x); ++k; }
        const int pairs = (n - k) / 2;
        if (pairs > 0) { graph_steps(x, pairs); k += 2 * pairs; }
    }
    for (; k < n; ++k) fused_step(x);
}

// Wait for the stream and read n_dev: n_host[k] = n_dev[k].
static void read_counts(dsmc_ctx *x)
{
    DSMC_HIP(hipMemcpyAsync(x->n_host, x->n_dev, 4 * sizeof(int), hipMemcpyDeviceToHost, x->stream));
    DSMC_HIP(hipStreamSynchronize(x->stream));
}

// FP32 form: the alive slots of the current state in slot order.  Returns
// their map (slot of each alive atom), or null when every slot is alive; n
// and n_slots receive the alive atoms and the slots (alive atoms plus the
// atoms the last move removed, which keep their slots until the next sort).
// The map is built on the device, in the re-sort's scratch, which is free
// between the calls of the C ABI.  When the trap table is valid the alive
// count is already known (the last sorted move's finalize or k_table_fused
// left it), so nothing is built if no atom was removed.
static const uint32_t *fused_live(dsmc_ctx *x, int &n, int &n_slots, bool want_map = true)
{
    read_counts(x);
    n = n_slots = x->n_host[x->cur];
    if (!x->dead_in_state || n_slots == 0) return nullptr;
    if (x->tbl_valid) {
        n = x->n_host[x->cur ^ 1];
        if (n == n_slots || !want_map) return nullptr;
    }
    int *stencil = (int *)x->res.alt_k;
    uint32_t *map = x->res.alt_v;
    launch_dead_stencil(x->key_a, x->n_dev + x->cur, n_slots, x->dead_key, stencil, x->stream);
    compaction_map(stencil, x->n_dev + x->cur, n_slots, map, x->n_dev + 2, x->scan_partial, x->stream,
                   nullptr);
    if (!x->tbl_valid) {
        read_counts(x);
        n = x->n_host[2];
        if (n == n_slots) return nullptr;
    }
    return map;
}

// Sync and read the current alive count.
static int host_alive(dsmc_ctx *x)
{
    int n = 0, n_slots = 0;
    if (x->fp32) {
        (void)fused_live(x, n, n_slots, false);
    } else {
        plain_settle(x);
        read_counts(x);
        n = x->n_host[0];
    }
    return n;
}

// Clears one 64-bit counter (a kernel, not a memset: callers may capture it).
__global__ void k_zero_u64(unsigned long long *p) { *p = 0ull; }

static void observe_now(dsmc_ctx *x, std::vector<dsmc_observables> &out)
{
    out.assign(x->T, dsmc_observables{});
    if (!x->fp32) {
        plain_settle(x);
        // the record comes back through pinned memory
        launch_observe_plain(x->tdev[0], x->cfg.mass, x->ps[x->cur], x->n_dev, x->n_cap, x->partials, x->stream,
                             &x->prof);
        plain_record(x, x->obs_host, x->step);
        DSMC_HIP(hipStreamSynchronize(x->stream));
        out[0] = *x->obs_host;
        return;
    }
    launch_observe_fused(x->d_traps, x->d_key_base, x->T, x->cfg.mass, x->fs[x->cur], x->key_a,
                         x->n_dev + x->cur, x->n_cap, x->dead_key, x->obs_first, x->obs_last,
                         x->acc2, x->stream);
    std::vector<double> a((size_t)x->T * kAccK);
    DSMC_HIP(hipStreamSynchronize(x->stream));
    DSMC_HIP(hipMemcpy(a.data(), x->acc2, sizeof(double) * a.size(), hipMemcpyDeviceToHost));
    for (int t = 0; t < x->T; ++t) {
        const double *v = a.data() + (size_t)t * kAccK;
        out[t].ek = v[kAccEk];
        out[t].ep = v[kAccEp];
        out[t].v2[0] = v[kAccV2x]; out[t].v2[1] = v[kAccV2y]; out[t].v2[2] = v[kAccV2z];
        out[t].n_alive = (long long)v[kAccN];
        out[t].step = x->step;
    }
}

// Initial per-cell state and labels (initSigvrmax, setUp.cu:287-292).  Every
// transfer goes through the context's own (non-blocking) stream, then waits.
static void reset_cells(dsmc_ctx *x)
{
    hipStream_t st = x->stream;
    if (!x->fp32) {
        plain_enter(x);   // what host reads see of the earlier run stays readable
        DSMC_HIP(hipMemsetAsync(x->cc_tagged, 0, sizeof(unsigned long long) * (x->ncells + 1), st));
        // every atom spin up, in both buffers (a move keeps the flags of the
        // one it writes unless atoms can flip)
        if (x->cfg.mcwf || !x->up_set)
            for (int b = 0; b < 2; ++b) DSMC_HIP(hipMemsetAsync(x->ps[b].up, 1, (size_t)x->n_cap, st));
        x->up_set = true;
    }
    // the double buffers as in a new context: a captured graph stays valid
    x->ssel = x->tsel = x->srt_cur = x->csel = x->mpar = 0;
    if (x->fp32)
        launch_init_sigvrmax(x->d_traps, x->d_key_base, x->T, x->n_keys, x->sigvrmax_f, st);
    else
        launch_init_sigvrmax(x->d_traps, x->d_key_base, x->T, x->n_keys, x->sigvrmax, st);
    const long long zero = 0;
    const int nn[2] = { x->n_cap, x->n_cap };
    DSMC_HIP(hipMemcpyAsync(x->step_dev(), &zero, sizeof zero, hipMemcpyHostToDevice, st));
    DSMC_HIP(hipMemsetAsync(x->coll_accum, 0, sizeof(unsigned long long) * x->T, st));
    DSMC_HIP(hipMemcpyAsync(x->n_dev, nn, sizeof nn, hipMemcpyHostToDevice, st));
    if (x->fp32)
        DSMC_HIP(hipMemcpyAsync(x->trap_start(), x->atom_begin.data(), sizeof(int) * (x->T + 1),
                                hipMemcpyHostToDevice, st));
    DSMC_HIP(hipStreamSynchronize(st));
    x->step = 0;
    x->coll_steps = 0;
    x->cur = 0;
    x->have_sort = false;
    x->srt_valid = false;
    x->dead_in_state = false;
    x->tbl_valid = true;    // all atoms alive, traps at their initial ranges
}

static InitParams init_params(const dsmc_ctx *x)
{
    InitParams ip;
    std::memset(&ip, 0, sizeof ip);
    ip.seed = x->cfg.seed;
    ip.mass = x->cfg.mass;
    ip.gs = x->cfg.gs;
    ip.spin = x->cfg.spin;
    return ip;
}

// ---------------------------------------------------------------------------
// Host reads: fields are converted to the host layout on the device, in the
// state buffer that is not current (scratch between moves: a move overwrites
// all of it), and copied from there (readout.hip).
// ---------------------------------------------------------------------------
template <typename T_>
static std::vector<T_> d2h(const T_ *d, size_t n)
{
    std::vector<T_> h(n);
    if (n) DSMC_HIP(hipMemcpy(h.data(), d, sizeof(T_) * n, hipMemcpyDeviceToHost));
    return h;
}

static void *stage(dsmc_ctx *x)
{
    return x->fp32 ? (void *)x->fs[x->cur ^ 1].r : (void *)x->ps[x->cur ^ 1].d[0];
}

static void to_host(dsmc_ctx *x, void *host, const void *dev, size_t bytes)
{
    if (bytes) x->host_copy.to_host(host, dev, bytes, x->device, x->stream);
}

static size_t field_size(dsmc_ctx *x, int field, int n)
{
    const size_t N = (size_t)n;
    switch (field) {
    case DSMC_FIELD_POS: case DSMC_FIELD_VEL: return N * 3 * sizeof(double);
    case DSMC_FIELD_ACC: return x->fp32 ? 0 : N * 3 * sizeof(double);
    case DSMC_FIELD_ATOM_ID: case DSMC_FIELD_CELL_ID: case DSMC_FIELD_PERM: return N * sizeof(int);
    case DSMC_FIELD_SPIN:
        if (!x->cfg.spin) return 0;
        return N * (x->fp32 ? 3 : 4) * sizeof(double);
    case DSMC_FIELD_EVAP_POS: case DSMC_FIELD_EVAP_VEL: return (size_t)x->n_cap * 3 * sizeof(double);
    case DSMC_FIELD_EVAP_TAG: return x->fp32 ? 0 : N * sizeof(int);
    case DSMC_FIELD_CELL_START_END:
        return x->fp32 ? (size_t)x->n_keys * 2 * sizeof(int) : (size_t)(x->ncells + 1) * 2 * sizeof(int);
    case DSMC_FIELD_CELL_COUNT: case DSMC_FIELD_CELL_PREFIX: case DSMC_FIELD_COLLISION_COUNT:
        return x->fp32 ? 0 : (size_t)(x->ncells + 1) * sizeof(int);
    case DSMC_FIELD_SIGVRMAX: return (size_t)x->n_keys * sizeof(double);
    case DSMC_FIELD_TRAP_START: return (size_t)(x->T + 1) * sizeof(int);
    case DSMC_FIELD_POS_COMP: case DSMC_FIELD_VEL_COMP: return x->fp32 ? N * 3 * sizeof(double) : 0;
    case DSMC_FIELD_OBS: return (size_t)x->obs_cap * x->T * sizeof(dsmc_observables);
    case DSMC_FIELD_SPIN_UP: return N * sizeof(int);
    case DSMC_FIELD_LOCAL_POPS: return x->pops ? (size_t)x->n_cap * 2 * sizeof(double) : 0;
    default: return 0;
    }
}

// Trap ranges of the alive atoms in slot order (traps are contiguous there),
// from their composite keys.
static void trap_ranges_of(const dsmc_ctx *x, const std::vector<uint32_t> &keys, int *out)
{
    std::vector<int> cnt(x->T, 0);
    for (uint32_t k : keys) {
        const int t = (int)(std::upper_bound(x->key_base.begin(), x->key_base.begin() + x->T, (int)k) -
                            x->key_base.begin()) - 1;
        cnt[t]++;
    }
    out[0] = 0;
    for (int t = 0; t < x->T; ++t) out[t + 1] = out[t] + cnt[t];
}

static void copy_field(dsmc_ctx *x, int field, void *host, size_t bytes)
{
    int n = 0, n_slots = 0;
    const uint32_t *live = nullptr;
    if (x->fp32) live = fused_live(x, n, n_slots);
    else n = n_slots = host_alive(x);
    const size_t need = field_size(x, field, n);
    // a field of this form has a size at one atom; at no alive atoms it is empty
    if (field_size(x, field, 1) == 0) fail(DSMC_ENOTSUP, "field not available in this form");
    if (need == 0) return;
    if (bytes < need) fail(DSMC_EINVAL, "host buffer too small");
    const size_t N = (size_t)n;
    hipStream_t st = x->stream;
    double *const sd = (double *)stage(x);
    if (!x->fp32) {
        const PlainPtrs &s = x->ps[x->cur];
        if (field == DSMC_FIELD_CELL_START_END || field == DSMC_FIELD_CELL_COUNT ||
            field == DSMC_FIELD_CELL_PREFIX || field == DSMC_FIELD_COLLISION_COUNT)
            plain_need_tables(x);
        switch (field) {
        case DSMC_FIELD_POS: case DSMC_FIELD_VEL: case DSMC_FIELD_ACC: {
            const int o = field == DSMC_FIELD_POS ? 0 : field == DSMC_FIELD_VEL ? 3 : 6;
            if (field == DSMC_FIELD_ACC) plain_need_acc(x);
            launch_pack_columns(s.d + o, 3, n, sd, st);
            to_host(x, host, sd, need);
            return;
        }
        case DSMC_FIELD_ATOM_ID: to_host(x, host, s.id, need); return;
        case DSMC_FIELD_SPIN:
            launch_pack_columns(s.psi, 4, n, sd, st);
            to_host(x, host, sd, need);
            return;
        case DSMC_FIELD_EVAP_POS: to_host(x, host, x->evap_pos_d, need); return;
        case DSMC_FIELD_EVAP_VEL: to_host(x, host, x->evap_vel_d, need); return;
        case DSMC_FIELD_EVAP_TAG: to_host(x, host, x->tag, need); return;
        case DSMC_FIELD_CELL_START_END: to_host(x, host, x->start_end, need); return;
        case DSMC_FIELD_CELL_COUNT: to_host(x, host, x->count, need); return;
        case DSMC_FIELD_CELL_PREFIX: to_host(x, host, x->prefix, need); return;
        case DSMC_FIELD_COLLISION_COUNT: to_host(x, host, x->coll_count, need); return;
        default: break;
        }
    } else {
        const FusedPtrs &s = x->fs[x->cur];
        switch (field) {
        case DSMC_FIELD_POS: case DSMC_FIELD_VEL: case DSMC_FIELD_POS_COMP: case DSMC_FIELD_VEL_COMP:
            launch_pack_records(field == DSMC_FIELD_POS   ? RecVec::Pos
                                : field == DSMC_FIELD_VEL ? RecVec::Vel
                                : field == DSMC_FIELD_POS_COMP ? RecVec::PosRem : RecVec::VelRem,
                                s, live, n, sd, st);
            to_host(x, host, sd, need);
            return;
        case DSMC_FIELD_ATOM_ID:   // the labels travel in the position remainders
            launch_pack_labels(s, live, n, (int *)sd, st);
            to_host(x, host, sd, need);
            return;
        case DSMC_FIELD_SPIN:
            launch_pack_columns(s.s, 3, live, n, sd, st);
            to_host(x, host, sd, need);
            return;
        case DSMC_FIELD_EVAP_POS: case DSMC_FIELD_EVAP_VEL:
            launch_widen(field == DSMC_FIELD_EVAP_POS ? x->evap_pos_f : x->evap_vel_f, 3LL * x->n_cap, sd, st);
            to_host(x, host, sd, need);
            return;
        case DSMC_FIELD_CELL_START_END: {
            if (!x->have_sort) fail(DSMC_ESTATE, "the cell table exists between sort and move");
            DSMC_HIP(hipMemsetAsync(x->cell_start, 0xFF, sizeof(uint32_t) * x->n_keys, x->stream));
            DSMC_HIP(hipMemsetAsync(x->cell_end, 0, sizeof(uint32_t) * x->n_keys, x->stream));
            launch_cell_range_fused(x->sorted_key, x->n_dev + (x->cur ^ 1), x->dead_key, x->cell_start,
                                    x->cell_end, x->n_cap, x->stream);
            DSMC_HIP(hipStreamSynchronize(x->stream));
            std::vector<uint32_t> a = d2h(x->cell_start, (size_t)x->n_keys);
            std::vector<uint32_t> b = d2h(x->cell_end, (size_t)x->n_keys);
            int *hi_ = (int *)host;
            for (int k = 0; k < x->n_keys; ++k) { hi_[2 * k] = (int)a[k]; hi_[2 * k + 1] = (int)b[k] - 1; }
            return;
        }
        case DSMC_FIELD_TRAP_START: {
            std::vector<uint32_t> lk(N);
            const uint32_t *src = x->key_a;
            if (live) {
                gather_u32((uint32_t *)sd, x->key_a, live, nullptr, n, st, nullptr);
                src = (const uint32_t *)sd;
            }
            to_host(x, lk.data(), src, sizeof(uint32_t) * N);
            trap_ranges_of(x, lk, (int *)host);
            return;
        }
        case DSMC_FIELD_CELL_ID:
            if (!x->have_sort) {   // keys of the alive slots (unsorted order)
                const uint32_t *src = x->key_a;
                if (live) {
                    gather_u32((uint32_t *)sd, x->key_a, live, nullptr, n, st, nullptr);
                    src = (const uint32_t *)sd;
                }
                to_host(x, host, src, need);
                return;
            }
            break;
        default: break;
        }
    }
    switch (field) {
    case DSMC_FIELD_CELL_ID: {
        // FP64 form: the keys of the last index or sort; FP32 form after a
        // sort: the sorted keys (the alive atoms; removed atoms sort last)
        const uint32_t *src = (x->fp32 && !x->have_sort) ? x->key_a : x->sorted_key;
        if (!src) src = x->key_a;
        to_host(x, host, src, need);
        return;
    }
    case DSMC_FIELD_PERM:
        if (!x->perm) fail(DSMC_ESTATE, "no sort has run yet");
        to_host(x, host, x->perm, need);
        if (!x->fp32 && x->perm_mask >= 0) {
            // slots as they were counted without the removed atoms among them
            const std::vector<uint64_t> m = d2h(x->mask_d2[x->perm_mask], resort_mask_words(x->n_cap));
            std::vector<uint32_t> before(m.size() + 1, 0u);
            for (size_t w = 0; w < m.size(); ++w) before[w + 1] = before[w] + (uint32_t)__builtin_popcountll(m[w]);
            uint32_t *h = (uint32_t *)host;
            for (size_t i = 0; i < N; ++i) {
                const uint32_t v = h[i], w = v >> 6;
                h[i] = v - before[w] - (uint32_t)__builtin_popcountll(m[w] & ((1ull << (v & 63)) - 1ull));
            }
        }
        return;
    case DSMC_FIELD_SIGVRMAX:
        if (x->fp32) {
            // widened in pieces that fit the staging (48 bytes per atom)
            const long long piece = std::max<long long>(1, 6LL * x->n_cap);
            for (long long k = 0; k < x->n_keys; k += piece) {
                const long long m = std::min<long long>(piece, x->n_keys - k);
                launch_widen(x->sigvrmax_f + k, m, sd, st);
                to_host(x, (double *)host + k, sd, sizeof(double) * (size_t)m);
            }
        } else {
            to_host(x, host, x->sigvrmax, need);
        }
        return;
    case DSMC_FIELD_TRAP_START: {
        int *h = (int *)host;
        h[0] = 0;
        h[1] = n;
        return;
    }
    case DSMC_FIELD_OBS: to_host(x, host, x->obs_log, need); return;
    case DSMC_FIELD_SPIN_UP: {
        int *h = (int *)host;
        if (x->fp32) {   // the FP32 form removes atoms instead of flipping them
            for (size_t i = 0; i < N; ++i) h[i] = 1;
            return;
        }
        // widened on the host: a quarter of the bytes to copy (1e4 atoms 59 -> 40 us, 1e6 267 -> 160)
        std::vector<uint8_t> up(N);
        to_host(x, up.data(), x->ps[x->cur].up, N);
        for (size_t i = 0; i < N; ++i) h[i] = up[i] ? 1 : 0;
        return;
    }
    case DSMC_FIELD_LOCAL_POPS: to_host(x, host, x->pops, need); return;
    default: break;
    }
    fail(DSMC_EINVAL, "unknown field");
}

#define PRIM_BEGIN try {
#define PRIM_END                                                              \
    return DSMC_OK;                                                           \
    }                                                                         \
    catch (const Error &e) { g_create_error = e.what(); return (dsmc_status)e.status; } \
    catch (const std::exception &e) { g_create_error = e.what(); return DSMC_EHIP; }

// Device scratch of one primitive call.  A call allocated its scratch and
// freed it (which waits for the device): some 70 us a sort, of 95 at n = 1000
// and 195 at n = 1e6.  A few idle blocks are kept for the next call instead:
// at most kKeptBlocks, of at most kKeptBytes together, per process; one that
// kKeptUnused calls did not use is freed, and all are when an allocation of
// this library fails.  A block belongs to one call at a time and the calls wait for their
// stream before they return, so threads and streams never share one (a call
// that fails does not keep its block).
constexpr int kKeptBlocks = 8;
constexpr size_t kKeptBytes = (size_t)512 << 20;
constexpr int kKeptUnused = 64;

struct KeptBlock {
    void *p;
    int *host;      // 64 bytes of pinned host memory, for a result
    size_t bytes;
    int device;
    int unused;
};
static std::mutex g_kept_mu;
static std::vector<KeptBlock> *const g_kept = new std::vector<KeptBlock>();   // outlives static destructors

static void free_kept()
{
    std::lock_guard<std::mutex> lock(g_kept_mu);
    for (const KeptBlock &b : *g_kept) { (void)hipFree(b.p); (void)hipHostFree(b.host); }
    g_kept->clear();
}

struct Workspace {
    KeptBlock b{ nullptr, nullptr, 0, 0, 0 };
    explicit Workspace(size_t bytes)
    {
        bytes = (std::max<size_t>(bytes, 16) + 65535) & ~(size_t)65535;
        DSMC_HIP(hipGetDevice(&b.device));
        {
            std::lock_guard<std::mutex> lock(g_kept_mu);
            int best = -1;
            for (size_t i = 0; i < g_kept->size(); ++i) {
                KeptBlock &k = (*g_kept)[i];
                ++k.unused;
                if (k.device == b.device && k.bytes >= bytes && (best < 0 || k.bytes < (*g_kept)[best].bytes))
                    best = (int)i;
            }
            if (best >= 0) {
                b = (*g_kept)[best];
                g_kept->erase(g_kept->begin() + best);
                return;
            }
        }
        b.bytes = bytes;
        b.p = device_alloc(bytes);
        if (hipHostMalloc((void **)&b.host, 64, hipHostMallocDefault) != hipSuccess) {
            (void)hipFree(b.p);
            fail(DSMC_ENOMEM, "no pinned host memory for a primitive's result");
        }
    }
    ~Workspace()
    {
        if (!b.p) return;
        if (std::uncaught_exceptions() > 0) {   // the stream may still use it: hipFree waits
            (void)hipFree(b.p);
            (void)hipHostFree(b.host);
            return;
        }
        b.unused = 0;
        std::vector<KeptBlock> gone;
        {
            std::lock_guard<std::mutex> lock(g_kept_mu);
            g_kept->push_back(b);
            size_t total = 0;
            for (const KeptBlock &k : *g_kept) total += k.bytes;
            // the longest unused first
            for (size_t i = 0; i < g_kept->size();) {
                size_t old = 0;
                for (size_t j = 1; j < g_kept->size(); ++j)
                    if ((*g_kept)[j].unused > (*g_kept)[old].unused) old = j;
                const KeptBlock k = (*g_kept)[old];
                if (total <= kKeptBytes && g_kept->size() <= (size_t)kKeptBlocks && k.unused < kKeptUnused) break;
                total -= k.bytes;
                gone.push_back(k);
                g_kept->erase(g_kept->begin() + old);
            }
        }
        for (const KeptBlock &k : gone) { (void)hipFree(k.p); (void)hipHostFree(k.host); }
    }
    Workspace(const Workspace &) = delete;
    Workspace &operator=(const Workspace &) = delete;
    template <typename T_> T_ *as() const { return (T_ *)b.p; }
};

// ---------------------------------------------------------------------------
// Scratch of the allocation-free sort (dsmc_sort_by_key_noalloc): a
// file-scope device array, one copy per device, resident until the process
// ends.  Layout: the radix digit totals and histograms for kNoAllocMaxPairs
// pairs, then the alternate key and value buffers of the passes.  Host code never uses the array's
// name as an address: the address on each device comes from
// hipGetSymbolAddress with that device current (noalloc_scratch()).
// ---------------------------------------------------------------------------
constexpr int kNoAllocMaxPairs = 1 << 20;
constexpr size_t kNoAllocSortBytes =
    ((size_t)kRadix * (kNoAllocMaxPairs / kSortTile) * 4 + (size_t)kRadix * 4 + 256 + 255) & ~(size_t)255;
constexpr size_t kNoAllocBytes = kNoAllocSortBytes + 2 * (size_t)kNoAllocMaxPairs * 4;
static_assert(kNoAllocMaxPairs % kSortTile == 0, "whole sort tiles");

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

constexpr int kNoAllocMaxDevices = 64;
static std::mutex g_noalloc_mu;
static void *g_noalloc_ptr[kNoAllocMaxDevices] = {};

// Device address of `scratch` on the current device, looked up once per
// device (first call there).
static char *noalloc_scratch()
{
    int dev = 0;
    DSMC_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= kNoAllocMaxDevices) fail(DSMC_EINVAL, "device index out of range");
    std::lock_guard<std::mutex> lock(g_noalloc_mu);
    if (!g_noalloc_ptr[dev]) {
        void *p = nullptr;
        DSMC_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) fail(DSMC_EHIP, "hipGetSymbolAddress returned no address for the sort scratch");
        g_noalloc_ptr[dev] = p;
    }
    return (char *)g_noalloc_ptr[dev];
}

__global__ __launch_bounds__(256) void k_copy_pairs(uint32_t *__restrict__ dk, uint32_t *__restrict__ dv,
                                                    const uint32_t *__restrict__ sk,
                                                    const uint32_t *__restrict__ sv, int n)
{
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        dk[i] = sk[i];
        dv[i] = sv[i];
    }
}

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
extern "C" {

int dsmc_abi_version(void) { return DSMC_ABI_VERSION; }

const char *dsmc_last_error(const dsmc_ctx *ctx)
{
    if (!ctx) return g_create_error.c_str();
    return ctx->err.c_str();
}

dsmc_status dsmc_create(const dsmc_config *cfg, const dsmc_trap *traps, int n_traps, dsmc_ctx **out)
{
    if (!out) return DSMC_EINVAL;
    *out = nullptr;
    dsmc_ctx *x = nullptr;
    try {
        validate(cfg, traps, n_traps);
        x = new dsmc_ctx();
        build_context(x, cfg, traps, n_traps);
        reset_cells(x);
        *out = x;
        g_create_error.clear();
        return DSMC_OK;
    } catch (const Error &e) {
        g_create_error = e.what();
        delete x;
        return (dsmc_status)e.status;
    } catch (const std::exception &e) {
        g_create_error = e.what();
        delete x;
        return DSMC_ENOMEM;
    }
}

dsmc_status dsmc_destroy(dsmc_ctx *ctx)
{
    delete ctx;
    return DSMC_OK;
}

dsmc_status dsmc_init_distribution(dsmc_ctx *ctx)
{
    DSMC_API_BEGIN(ctx)
    reset_cells(ctx);
    const InitParams ip = init_params(ctx);
    if (!ctx->fp32) {
        launch_init_plain(ctx->tdev[0], ip, ctx->ps[0], ctx->n_cap, ctx->stream, &ctx->prof);
        plain_index(ctx);
    } else {
        launch_init_fused(ctx->d_traps, ctx->trap_start(), ctx->T, ip, ctx->fs[0], ctx->n_cap,
                          ctx->stream, &ctx->prof);
        fused_index(ctx);
    }
    DSMC_HIP(hipStreamSynchronize(ctx->stream));
    DSMC_API_END(ctx)
}

dsmc_status dsmc_set_state(dsmc_ctx *ctx, const double *pos, const double *vel, int n)
{
    DSMC_API_BEGIN(ctx)
    if (!pos || !vel || n != ctx->n_cap) fail(DSMC_EINVAL, "set_state needs n_capacity atoms");
    reset_cells(ctx);
    // the rows go to the other state buffer (reset_cells made 0 current) and
    // are laid out from there
    const size_t N = (size_t)n;
    double *const sp = (double *)stage(ctx), *const sv = sp + 3 * N;
    hipStream_t st = ctx->stream;
    DSMC_HIP(hipMemcpyAsync(sp, pos, 3 * N * sizeof(double), hipMemcpyHostToDevice, st));
    DSMC_HIP(hipMemcpyAsync(sv, vel, 3 * N * sizeof(double), hipMemcpyHostToDevice, st));
    if (!ctx->fp32) {
        const PlainPtrs &s = ctx->ps[0];
        launch_unpack_columns(sp, 3, n, s.d, st);
        launch_unpack_columns(sv, 3, n, s.d + 3, st);
        launch_iota(s.id, n, st);
        launch_accel_plain(ctx->tdev[0], s, n, st, &ctx->prof);
        plain_index(ctx);
    } else {
        // slot i holds atom i: its label in the position remainders
        launch_unpack_records(sp, sv, n, ctx->fs[0], st);
        fused_index(ctx);
    }
    DSMC_HIP(hipStreamSynchronize(ctx->stream));
    DSMC_API_END(ctx)
}

dsmc_status dsmc_set_spin(dsmc_ctx *ctx, const double *spin, int n, int components)
{
    DSMC_API_BEGIN(ctx)
    if (!ctx->cfg.spin) fail(DSMC_ENOTSUP, "spin evolution is off in this context");
    int n_alive = 0, n_slots = 0;
    const uint32_t *live = nullptr;
    if (ctx->fp32) live = fused_live(ctx, n_alive, n_slots);
    else n_alive = host_alive(ctx);
    if (!spin || n != n_alive) fail(DSMC_EINVAL, "set_spin needs one row per alive atom");
    double *const sd = (double *)stage(ctx);
    if (!ctx->fp32 && components != 4) fail(DSMC_EINVAL, "the FP64 form stores spinors (4 components)");
    if (ctx->fp32 && components != 3) fail(DSMC_EINVAL, "the FP32 form stores Bloch vectors (3 components)");
    if (n > 0) {
        DSMC_HIP(hipMemcpyAsync(sd, spin, sizeof(double) * (size_t)components * (size_t)n, hipMemcpyHostToDevice,
                                ctx->stream));
        // FP32 form: rows go to the alive slots; slots of removed atoms keep their values
        if (!ctx->fp32) launch_unpack_columns(sd, 4, n, ctx->ps[ctx->cur].psi, ctx->stream);
        else launch_unpack_columns(sd, 3, live, n, ctx->fs[ctx->cur].s, ctx->stream);
        DSMC_HIP(hipStreamSynchronize(ctx->stream));
    }
    DSMC_API_END(ctx)
}

dsmc_status dsmc_index_atoms(dsmc_ctx *ctx)
{
    DSMC_API_BEGIN(ctx)
    if (ctx->fp32) {
        if (ctx->have_sort) fail(DSMC_ESTATE, "a sort is pending: call dsmc_move_atoms first");
        fused_index(ctx);
    } else {
        plain_enter(ctx);
        plain_index(ctx);
    }
    DSMC_API_END(ctx)
}

dsmc_status dsmc_sort_arrays(dsmc_ctx *ctx)
{
    DSMC_API_BEGIN(ctx)
    if (ctx->fp32) {
        if (ctx->have_sort) fail(DSMC_ESTATE, "a sort is pending: call dsmc_move_atoms first");
        fused_sort(ctx);
    } else {
        plain_enter(ctx);
        plain_need_index(ctx);
        plain_sort(ctx);
    }
    DSMC_API_END(ctx)
}

dsmc_status dsmc_build_cell_table(dsmc_ctx *ctx)
{
    DSMC_API_BEGIN(ctx)
    if (!ctx->sorted_key) fail(DSMC_ESTATE, "no sort has run yet");
    if (ctx->fp32) {
        if (!ctx->have_sort) fail(DSMC_ESTATE, "build the table right after dsmc_sort_arrays");
        fused_table(ctx);
    } else {
        plain_enter(ctx);
        plain_table(ctx);
    }
    DSMC_API_END(ctx)
}

dsmc_status dsmc_collide(dsmc_ctx *ctx)
{
    DSMC_API_BEGIN(ctx)
    if (ctx->fp32) {
        if (!ctx->have_sort) fail(DSMC_ESTATE, "collide needs a sorted state and its table");
        fused_collide(ctx);
        ctx->coll_steps++;
    } else {
        plain_enter(ctx);
        plain_collide(ctx);
    }
    DSMC_API_END(ctx)
}

dsmc_status dsmc_evolve_spin(dsmc_ctx *ctx)
{
    DSMC_API_BEGIN(ctx)
    if (!ctx->cfg.spin) fail(DSMC_ENOTSUP, "spin evolution is off in this context");
    if (ctx->fp32) fail(DSMC_ENOTSUP, "the FP32 form evolves spins inside dsmc_move_atoms");
    plain_enter(ctx);
    plain_spin(ctx);
    launch_normalise_plain(ctx->ps[ctx->cur], ctx->n_dev, ctx->n_cap, ctx->stream, &ctx->prof);
    DSMC_API_END(ctx)
}

dsmc_status dsmc_move_atoms(dsmc_ctx *ctx)
{
    DSMC_API_BEGIN(ctx)
    if (ctx->fp32) {
        fused_move(ctx);
    } else {
        plain_enter(ctx);
        launch_move_plain(ctx->tdev[0], ctx->cfg.dt, ctx->cfg.mass, ctx->ps[ctx->cur], ctx->n_dev, ctx->n_cap,
                          ctx->partials, ctx->stream, &ctx->prof);
        plain_record(ctx, ctx->obs_log + (ctx->step % ctx->obs_cap), ctx->step);
    }
    ctx->step++;
    DSMC_API_END(ctx)
}

dsmc_status dsmc_calculate_temp(dsmc_ctx *ctx, double *T)
{
    DSMC_API_BEGIN(ctx)
    if (!T) fail(DSMC_EINVAL, "null output");
    std::vector<dsmc_observables> o;
    observe_now(ctx, o);
    const double v2 = o[0].v2[0] + o[0].v2[1] + o[0].v2[2];
    *T = o[0].n_alive > 0 ? ctx->cfg.mass / 3. / kKB * (v2 / (double)o[0].n_alive) : 0.0;
    DSMC_API_END(ctx)
}

dsmc_status dsmc_local_populations(dsmc_ctx *ctx)
{
    DSMC_API_BEGIN(ctx)
    if (!ctx->pops) fail(DSMC_ENOTSUP, "the spin-flip model is off in this context (cfg.mcwf)");
    plain_enter(ctx);
    plain_local_pops(ctx);
    DSMC_API_END(ctx)
}

dsmc_status dsmc_flip_atoms(dsmc_ctx *ctx, long long *n_flipped)
{
    DSMC_API_BEGIN(ctx)
    if (!ctx->pops) fail(DSMC_ENOTSUP, "the spin-flip model is off in this context (cfg.mcwf)");
    plain_enter(ctx);
    hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(1), 0, ctx->stream, ctx->flips);
    DSMC_HIP(hipGetLastError());
    plain_flip(ctx);
    if (n_flipped) {
        unsigned long long f = 0;
        DSMC_HIP(hipMemcpyAsync(&f, ctx->flips, sizeof f, hipMemcpyDeviceToHost, ctx->stream));
        DSMC_HIP(hipStreamSynchronize(ctx->stream));
        *n_flipped = (long long)f;
    }
    DSMC_API_END(ctx)
}

dsmc_status dsmc_exponential_decay(dsmc_ctx *ctx)
{
    DSMC_API_BEGIN(ctx)
    if (!ctx->pops) fail(DSMC_ENOTSUP, "the spin-flip model is off in this context (cfg.mcwf)");
    plain_enter(ctx);
    plain_decay(ctx);
    DSMC_API_END(ctx)
}

dsmc_status dsmc_evaporation_tag(dsmc_ctx *ctx)
{
    DSMC_API_BEGIN(ctx)
    if (ctx->fp32) fail(DSMC_ENOTSUP, "the FP32 form tags inside dsmc_move_atoms");
    plain_enter(ctx);
    plain_evap_tag(ctx);
    DSMC_API_END(ctx)
}

dsmc_status dsmc_compact(dsmc_ctx *ctx, int *n_alive)
{
    DSMC_API_BEGIN(ctx)
    if (ctx->fp32) fail(DSMC_ENOTSUP, "the FP32 form compacts inside the sort");
    plain_enter(ctx);
    plain_compact(ctx);
    if (n_alive) {   // the gather left the count in n_host
        DSMC_HIP(hipStreamSynchronize(ctx->stream));
        *n_alive = ctx->n_host[0];
    }
    DSMC_API_END(ctx)
}

dsmc_status dsmc_step(dsmc_ctx *ctx, int n_steps)
{
    DSMC_API_BEGIN(ctx)
    if (n_steps < 0) fail(DSMC_EINVAL, "n_steps < 0");
    do_steps(ctx, n_steps);
    DSMC_API_END(ctx)
}

dsmc_status dsmc_sync(dsmc_ctx *ctx)
{
    DSMC_API_BEGIN(ctx)
    DSMC_HIP(hipStreamSynchronize(ctx->stream));
    DSMC_API_END(ctx)
}

dsmc_status dsmc_get_info(dsmc_ctx *ctx, dsmc_info *info)
{
    DSMC_API_BEGIN(ctx)
    if (!info) fail(DSMC_EINVAL, "null output");
    info->precision = ctx->cfg.precision;
    info->n_traps = ctx->T;
    info->n_capacity = ctx->n_cap;
    info->n_alive = host_alive(ctx);
    info->n_keys = ctx->n_keys;
    info->key_bits = ctx->key_bits;
    info->radix_passes = ctx->passes;
    info->block_size = ctx->block;
    info->step = ctx->step;
    info->collision_steps = ctx->coll_steps;
    info->obs_capacity = ctx->obs_cap;
    DSMC_API_END(ctx)
}

dsmc_status dsmc_observe(dsmc_ctx *ctx, dsmc_observables *per_trap, int n_traps)
{
    DSMC_API_BEGIN(ctx)
    if (!per_trap || n_traps < ctx->T) fail(DSMC_EINVAL, "need one record per trap");
    std::vector<dsmc_observables> o;
    observe_now(ctx, o);
    std::memcpy(per_trap, o.data(), sizeof(dsmc_observables) * ctx->T);
    DSMC_API_END(ctx)
}

dsmc_status dsmc_copy_out(dsmc_ctx *ctx, int field, void *host, size_t bytes)
{
    DSMC_API_BEGIN(ctx)
    if (!host) fail(DSMC_EINVAL, "null output");
    copy_field(ctx, field, host, bytes);
    DSMC_API_END(ctx)
}

dsmc_status dsmc_field_bytes(dsmc_ctx *ctx, int field, size_t *bytes)
{
    DSMC_API_BEGIN(ctx)
    if (!bytes) fail(DSMC_EINVAL, "null output");
    *bytes = field_size(ctx, field, host_alive(ctx));
    DSMC_API_END(ctx)
}

dsmc_status dsmc_time_steps(dsmc_ctx *ctx, int n_steps, double *ms)
{
    DSMC_API_BEGIN(ctx)
    if (!ms || n_steps < 0) fail(DSMC_EINVAL, "bad arguments");
    hipEvent_t b, e;
    DSMC_HIP(hipEventCreate(&b));
    DSMC_HIP(hipEventCreate(&e));
    try {
        DSMC_HIP(hipStreamSynchronize(ctx->stream));
        DSMC_HIP(hipEventRecord(b, ctx->stream));
        do_steps(ctx, n_steps);
        DSMC_HIP(hipEventRecord(e, ctx->stream));
        DSMC_HIP(hipEventSynchronize(e));
        float f = 0.f;
        DSMC_HIP(hipEventElapsedTime(&f, b, e));
        *ms = f;
    } catch (...) {
        (void)hipEventDestroy(b);
        (void)hipEventDestroy(e);
        throw;
    }
    DSMC_HIP(hipEventDestroy(b));
    DSMC_HIP(hipEventDestroy(e));
    DSMC_API_END(ctx)
}

// ---- several contexts stepped together ------------------------------------
// Independent groups of traps in separate contexts (each with its own stream
// and graph) are stepped in turns of `chunk` steps, so that every stream has
// work queued and the GPU runs one group's latency-bound kernels (re-sort,
// collide, finalize) beside another's bandwidth-bound move.
static void check_group(dsmc_ctx *const *ctxs, int n_ctx, int n_steps, int chunk)
{
    if (n_steps < 0 || chunk < 1) fail(DSMC_EINVAL, "n_steps < 0 or chunk < 1");
    for (int i = 0; i < n_ctx; ++i) {
        if (!ctxs[i]) fail(DSMC_EINVAL, "null context in the group");
        if (ctxs[i]->device != ctxs[0]->device) fail(DSMC_EINVAL, "the group's contexts are on different devices");
        for (int j = 0; j < i; ++j)
            if (ctxs[j] == ctxs[i]) fail(DSMC_EINVAL, "a context appears twice in the group");
    }
}

static void group_steps(dsmc_ctx *const *ctxs, int n_ctx, int n_steps, int chunk)
{
    for (int done = 0; done < n_steps; done += chunk) {
        const int k = std::min(chunk, n_steps - done);
        for (int i = 0; i < n_ctx; ++i) do_steps(ctxs[i], k);
    }
}

dsmc_status dsmc_step_group(dsmc_ctx *const *ctxs, int n_ctx, int n_steps, int chunk)
{
    if (!ctxs || n_ctx < 1) return DSMC_EINVAL;
    DSMC_API_BEGIN(ctxs[0])
    check_group(ctxs, n_ctx, n_steps, chunk);
    group_steps(ctxs, n_ctx, n_steps, chunk);
    DSMC_API_END(ctxs[0])
}

dsmc_status dsmc_time_steps_group(dsmc_ctx *const *ctxs, int n_ctx, int n_steps, int chunk, double *ms)
{
    if (!ctxs || n_ctx < 1) return DSMC_EINVAL;
    DSMC_API_BEGIN(ctxs[0])
    if (!ms) fail(DSMC_EINVAL, "null output");
    check_group(ctxs, n_ctx, n_steps, chunk);
    std::vector<hipEvent_t> ev((size_t)n_ctx + 1, nullptr);
    auto destroy = [&]() {
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
    };
    try {
        for (auto &e : ev) DSMC_HIP(hipEventCreate(&e));
        for (int i = 0; i < n_ctx; ++i) DSMC_HIP(hipStreamSynchronize(ctxs[i]->stream));
        // one start for all: every other stream waits for the first's event
        DSMC_HIP(hipEventRecord(ev[0], ctxs[0]->stream));
        for (int i = 1; i < n_ctx; ++i) DSMC_HIP(hipStreamWaitEvent(ctxs[i]->stream, ev[0], 0));
        group_steps(ctxs, n_ctx, n_steps, chunk);
        for (int i = 0; i < n_ctx; ++i) DSMC_HIP(hipEventRecord(ev[i + 1], ctxs[i]->stream));
        float worst = 0.f;
        for (int i = 0; i < n_ctx; ++i) {
            DSMC_HIP(hipEventSynchronize(ev[i + 1]));
            float f = 0.f;
            DSMC_HIP(hipEventElapsedTime(&f, ev[0], ev[i + 1]));
            worst = std::max(worst, f);
        }
        *ms = worst;
    } catch (...) {
        destroy();
        throw;
    }
    destroy();
    DSMC_API_END(ctxs[0])
}

dsmc_status dsmc_profile_enable(dsmc_ctx *ctx, int enable)
{
    DSMC_API_BEGIN(ctx)
    ctx->prof.collect();
    if (enable) ctx->prof.reset();
    ctx->prof.enabled = enable != 0;
    DSMC_API_END(ctx)
}

dsmc_status dsmc_profile_read(dsmc_ctx *ctx, dsmc_kernel_stat *stats, int max_stats, int *n_stats)
{
    DSMC_API_BEGIN(ctx)
    DSMC_HIP(hipStreamSynchronize(ctx->stream));
    ctx->prof.collect();
    int k = 0;
    for (const auto &kv : ctx->prof.stats()) {
        if (stats && k < max_stats) {
            dsmc_kernel_stat &s = stats[k];
            std::memset(&s, 0, sizeof s);
            std::snprintf(s.name, sizeof s.name, "%s", kv.first.c_str());
            s.launches = kv.second.launches;
            s.total_ms = kv.second.total_ms;
            s.bytes_per_launch = kv.second.bytes;
        }
        ++k;
    }
    if (n_stats) *n_stats = k;
    DSMC_API_END(ctx)
}

dsmc_status dsmc_autotune(dsmc_ctx *ctx, int *block_size_out)
{
    DSMC_API_BEGIN(ctx)
    if (!ctx->fp32) {
        if (block_size_out) *block_size_out = 256;
        return DSMC_OK;
    }
    if (ctx->have_sort) fail(DSMC_ESTATE, "a sort is pending: call dsmc_move_atoms first");
    // Time the fused move on the current state without committing it: the move
    // writes the other state buffer and a scratch key buffer, evaporation is
    // off, and the device step counter is restored afterwards.  When the state
    // is in the order of a sort (as in the step loop), the trial moves also
    // compare with that sort's keys and leave the re-sort's masks, counts and
    // samples, as the step's move does; the next sort is then a full one.
    DSMC_HIP(hipStreamSynchronize(ctx->stream));
    DSMC_HIP(hipMemcpyAsync(ctx->step_save, ctx->step_dev(), sizeof(long long),
                            hipMemcpyDeviceToDevice, ctx->stream));
    MoveParams mp = move_params(ctx);
    mp.spin_loss = 0;
    mp.energy_cut = 0;
    if (ctx->srt_valid) {
        mp.count_moved = 1;
        mp.key_prev = ctx->sorted_key;
    }
    // (threads per block, atoms per thread): shapes of at least 512 atoms per
    // block.  Smaller blocks multiply the per-block work that trial moves do
    // not weigh (each move block's trap table and sums, the finalize's
    // records, the re-sort's counts): on MI355X a 128 x 2 move made the
    // batched step 26 % slower, and a 64 x 2 move that won the trials made
    // the spin step 2 % slower.
    const int cands[4][2] = { { 512, 1 }, { 1024, 1 }, { 256, 2 }, { 512, 2 } };
    double best = 1e30, pref = 1e30;
    int best_bs = ctx->block, best_apt = ctx->apt;
    // 256 threads x 2 atoms measured best in the step on MI355X (batched,
    // single-trap and spin workloads); the trial moves cannot reproduce the
    // step's cache state, so another candidate must beat it by more than 5 %
    // to be taken
    const int pref_bs = 256, pref_apt = 2;
    hipEvent_t b, e;
    DSMC_HIP(hipEventCreate(&b));
    DSMC_HIP(hipEventCreate(&e));
    const bool was = ctx->prof.enabled;
    ctx->prof.enabled = false;
    // on sorted state the trials time the fused step kernel (its collisions
    // computed but not stored), as the step loop runs it
    StepCollide sc;
    sc.cp = collide_params(ctx);
    sc.sigvrmax = ctx->sigvrmax_f;
    sc.edge_sm = ctx->edge_sm;
    sc.coll_accum = ctx->coll_accum;
    sc.dry = 1;
    const StepCollide *coll = (ctx->srt_valid && !ctx->split_step) ? &sc : nullptr;
    for (const auto &cand : cands) {
        const int bs = cand[0], apt = cand[1];
        float f = 1e30f;
        for (int rep = 0; rep < 3; ++rep) {  // first repetition warms up
            float g = 0.f;
            DSMC_HIP(hipEventRecord(b, ctx->stream));
            for (int k = 0; k < 5; ++k)
                launch_move_fused(bs, apt, ctx->d_traps, mp, ctx->fs[ctx->cur], ctx->fs[ctx->cur ^ 1],
                                  nullptr, ctx->trap_start(), ctx->n_dev + ctx->cur, ctx->res.alt_k,
                                  ctx->evap_pos_f, ctx->evap_vel_f, ctx->rec, ctx->step_dev(),
                                  ctx->n_cap, ctx->stream, nullptr, coll);
            DSMC_HIP(hipEventRecord(e, ctx->stream));
            DSMC_HIP(hipEventSynchronize(e));
            DSMC_HIP(hipEventElapsedTime(&g, b, e));
            if (rep > 0) f = std::min(f, g);
        }
        if (f < best) { best = f; best_bs = bs; best_apt = apt; }
        if (bs == pref_bs && apt == pref_apt) pref = f;
    }
    if (pref <= 1.05 * best) { best_bs = pref_bs; best_apt = pref_apt; }
    ctx->prof.enabled = was;
    (void)hipEventDestroy(b);
    (void)hipEventDestroy(e);
    DSMC_HIP(hipMemcpyAsync(ctx->step_dev(), ctx->step_save, sizeof(long long),
                            hipMemcpyDeviceToDevice, ctx->stream));
    DSMC_HIP(hipMemsetAsync(ctx->acc, 0, sizeof(double) * kAccK * ctx->T, ctx->stream));
    DSMC_HIP(hipStreamSynchronize(ctx->stream));
    if (mp.count_moved) ctx->srt_valid = false;
    if (ctx->block != best_bs || ctx->apt != best_apt) {
        drop_graphs(ctx);
        // the per-block counts of the last move are for the old block size
        ctx->srt_valid = false;
    }
    ctx->block = best_bs;
    ctx->apt = best_apt;
    if (block_size_out) *block_size_out = best_bs;
    DSMC_API_END(ctx)
}

// ---- device primitives on caller memory -----------------------------------

dsmc_status dsmc_sort_by_key(unsigned int *d_keys, unsigned int *d_values, int n, int key_bits,
                             void *stream)
{
    PRIM_BEGIN
    if (n < 0 || key_bits < 1 || key_bits > 32 || (n > 0 && (!d_keys || !d_values)))
        fail(DSMC_EINVAL, "bad sort arguments");
    if (n == 0) return DSMC_OK;
    hipStream_t st = (hipStream_t)stream;
    const RadixPlan plan = radix_plan(n, key_bits);
    const size_t row = ((size_t)n + 63) & ~(size_t)63;
    Workspace ws(2 * row * sizeof(uint32_t) + sort_scratch_bytes(n));
    uint32_t *tk = ws.as<uint32_t>(), *tv = tk + row;
    SortScratch s;
    sort_scratch_bind(s, n, tv + row);
    if (plan.passes % 2 == 0) {
        radix_sort(d_keys, d_values, tk, tv, d_keys, d_values, nullptr, plan, s, st, nullptr);
    } else {
        radix_sort(d_keys, d_values, d_keys, d_values, tk, tv, nullptr, plan, s, st, nullptr);
        hipLaunchKernelGGL(k_copy_pairs, dim3(std::min(div_up(n, 256), 2048)), dim3(256), 0, st, d_keys,
                           d_values, tk, tv, n);
        DSMC_HIP(hipGetLastError());
    }
    DSMC_HIP(hipStreamSynchronize(st));
    PRIM_END
}

dsmc_status dsmc_sort_by_key_noalloc(unsigned int *d_keys, unsigned int *d_values, int n,
                                     int key_bits, void *stream)
{
    PRIM_BEGIN
    if (n < 0 || key_bits < 1 || key_bits > 32 || (n > 0 && (!d_keys || !d_values)))
        fail(DSMC_EINVAL, "bad sort arguments");
    if (n > kNoAllocMaxPairs)
        fail(DSMC_EINVAL, "dsmc_sort_by_key_noalloc sorts at most 1048576 pairs (use dsmc_sort_by_key)");
    char *base = noalloc_scratch();
    if (n == 0) return DSMC_OK;
    hipStream_t st = (hipStream_t)stream;
    SortScratch s;
    sort_scratch_bind(s, n, base, kRadix);
    uint32_t *tk = (uint32_t *)(base + kNoAllocSortBytes);
    uint32_t *tv = tk + kNoAllocMaxPairs;
    const RadixPlan plan = radix_plan(n, key_bits, kRadixBits);   // its fixed scratch holds 256 digits
    if (plan.passes % 2 == 0) {
        radix_sort(d_keys, d_values, tk, tv, d_keys, d_values, nullptr, plan, s, st, nullptr);
    } else {
        radix_sort(d_keys, d_values, d_keys, d_values, tk, tv, nullptr, plan, s, st, nullptr);
        hipLaunchKernelGGL(k_copy_pairs, dim3(std::min(div_up(n, 256), 2048)), dim3(256), 0, st,
                           d_keys, d_values, tk, tv, n);
        DSMC_HIP(hipGetLastError());
    }
    PRIM_END
}

dsmc_status dsmc_exclusive_scan(const int *d_in, int *d_out, int n, void *stream)
{
    PRIM_BEGIN
    if (n < 0 || (n > 0 && (!d_in || !d_out))) fail(DSMC_EINVAL, "bad scan arguments");
    if (n == 0) return DSMC_OK;
    hipStream_t st = (hipStream_t)stream;
    Workspace part(sizeof(int) * (scan_partials(n)));
    exclusive_scan(d_in, d_out, n, part.as<int>(), st, nullptr);
    DSMC_HIP(hipStreamSynchronize(st));
    PRIM_END
}

dsmc_status dsmc_remove_if(int *d_values, const int *d_stencil, int n, int *n_out, void *stream)
{
    PRIM_BEGIN
    if (n < 0 || (n > 0 && (!d_values || !d_stencil))) fail(DSMC_EINVAL, "bad remove_if arguments");
    if (n == 0) { if (n_out) *n_out = 0; return DSMC_OK; }
    hipStream_t st = (hipStream_t)stream;
    Workspace ws(sizeof(int) * ((size_t)n + scan_partials(n)));
    int *tmp = ws.as<int>();
    remove_if(d_values, d_stencil, n, tmp, tmp + n, ws.b.host, st);
    DSMC_HIP(hipStreamSynchronize(st));
    const int kept = *ws.b.host;
    if (n_out) *n_out = kept;
    PRIM_END
}

dsmc_status dsmc_philox(unsigned int *d_out, int n, const unsigned int ctr[4],
                        const unsigned int key[2], void *stream)
{
    PRIM_BEGIN
    if (n < 0 || !ctr || !key || (n > 0 && !d_out)) fail(DSMC_EINVAL, "bad philox arguments");
    philox_fill(d_out, n, ctr, key, (hipStream_t)stream);
    DSMC_HIP(hipStreamSynchronize((hipStream_t)stream));
    PRIM_END
}

dsmc_status dsmc_stream_copy(void *d_dst, const void *d_src, size_t bytes, int repeats,
                             double *ms)
{
    PRIM_BEGIN
    if (!d_dst || !d_src || bytes % 16 || repeats < 1) fail(DSMC_EINVAL, "bad stream_copy arguments");
    hipEvent_t b, e;
    DSMC_HIP(hipEventCreate(&b));
    DSMC_HIP(hipEventCreate(&e));
    stream_copy(d_dst, d_src, bytes, nullptr);  // warm-up
    DSMC_HIP(hipEventRecord(b, nullptr));
    for (int r = 0; r < repeats; ++r) stream_copy(d_dst, d_src, bytes, nullptr);
    DSMC_HIP(hipEventRecord(e, nullptr));
    DSMC_HIP(hipEventSynchronize(e));
    float f = 0.f;
    DSMC_HIP(hipEventElapsedTime(&f, b, e));
    (void)hipEventDestroy(b);
    (void)hipEventDestroy(e);
    if (ms) *ms = f / repeats;
    PRIM_END
}

dsmc_status dsmc_gather_copy(void *d_dst, const void *d_src, const unsigned int *d_map, int n_slots,
                             int repeats, double *ms)
{
    PRIM_BEGIN
    if (!d_dst || !d_src || !d_map || n_slots < 1 || repeats < 1)
        fail(DSMC_EINVAL, "bad gather_copy arguments");
    hipEvent_t b, e;
    DSMC_HIP(hipEventCreate(&b));
    DSMC_HIP(hipEventCreate(&e));
    gather_copy(d_dst, d_src, d_map, n_slots, nullptr);  // warm-up
    DSMC_HIP(hipEventRecord(b, nullptr));
    for (int r = 0; r < repeats; ++r) gather_copy(d_dst, d_src, d_map, n_slots, nullptr);
    DSMC_HIP(hipEventRecord(e, nullptr));
    DSMC_HIP(hipEventSynchronize(e));
    float f = 0.f;
    DSMC_HIP(hipEventElapsedTime(&f, b, e));
    (void)hipEventDestroy(b);
    (void)hipEventDestroy(e);
    if (ms) *ms = f / repeats;
    PRIM_END
}

dsmc_status dsmc_device_alloc(void **d_ptr, size_t bytes)
{
    PRIM_BEGIN
    if (!d_ptr) fail(DSMC_EINVAL, "null output");
    *d_ptr = device_alloc(std::max<size_t>(bytes, 16));
    PRIM_END
}

dsmc_status dsmc_device_free(void *d_ptr)
{
    PRIM_BEGIN
    if (d_ptr) DSMC_HIP(hipFree(d_ptr));
    PRIM_END
}

dsmc_status dsmc_memcpy_htod(void *d_dst, const void *h_src, size_t bytes)
{
    PRIM_BEGIN
    DSMC_HIP(hipMemcpy(d_dst, h_src, bytes, hipMemcpyHostToDevice));
    PRIM_END
}

dsmc_status dsmc_memcpy_dtoh(void *h_dst, const void *d_src, size_t bytes)
{
    PRIM_BEGIN
    DSMC_HIP(hipMemcpy(h_dst, d_src, bytes, hipMemcpyDeviceToHost));
    PRIM_END
}

}  // extern "C"
