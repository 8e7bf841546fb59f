// plain_step.hpp -- the FP64 form's whole step (dsmc_step): launchers of the
// kernels that replace the one-kernel-per-call sequence inside it.
#pragma once

#include "plain.hpp"

namespace dsmc {

constexpr int kStepBlock = 256;   // slots per move block
constexpr int kMaxSub = 16;       // motion substeps of one move launch
constexpr int kStepRec = 6;       // sums per block and substep: v_x^2, v_y^2, v_z^2, U, lost energy,
                                  // atoms lost so far in the launch

// Device-side counters of the step loop, double-buffered: a step's kernels
// read one and its finalize writes the other.
struct PlainCtl {
    long long step;      // motion steps taken
    unsigned  coll;      // collision steps taken
    int       slots;     // slots of the state (alive atoms and those removed since the last sort)
    int       alive;     // alive atoms; after a sort they are the first slots
    int       pad;
};

struct PlainStepParams {
    double dt, mass;
    SpinParams  spin;
    FlipParams  flip;
    DecayParams decay;
    int spin_loss, energy_cut;
    int pad;          // the fields behind it at their places: without it the compiler's move is
                      // 3 % slower (the reference's run, 500 steps: 2.26 ms instead of 2.19)
    int lpc;          // motion substeps per collision step
    int phase;        // substeps of the collision step already taken
    int L;            // substeps of this launch (<= kMaxSub)
    int fast_key;     // every nc below 2^20: cell_of_fast
    uint32_t dead_key;
    // incremental re-sort (key_prev null: the slots are in no sorted order)
    const uint32_t *key_prev;
    uint64_t *mask_moved, *mask_dead, *mask_last;   // mask_last: removed in the launch's last substep
};

// Collisions of the sorted slots (key, perm) on the state in its previous
// order.  cc[cell] = collision step << 32 | accepted collisions, written for
// cells with any; *n_sorted receives the slots.
void launch_collide_step(const TrapDev &t, const CollideParams &cp, const PlainPtrs &s, const uint32_t *key,
                         const uint32_t *perm, const PlainCtl *ctl, int n_cap, double *sigvrmax,
                         unsigned long long *cc, unsigned long long *coll_total, int *n_sorted,
                         const ResortBuckets &rb, hipStream_t st, Profiler *prof);
// Motion substeps of src (slot i taken from perm[i]; perm null: in place) into
// dst.  after_sort: the launch covers ctl->alive slots, all alive; else
// ctl->slots slots, of which key_in (when not null) marks the removed ones.
// spin: evolve spinors; stored: keep the accelerations and spin states in
// memory (the spin-flip model), else both are those of spin up at the position.
void launch_move_step(bool spin, bool stored, const TrapDev &t, const PlainStepParams &p, const PlainPtrs &src,
                      const PlainPtrs &dst, const uint32_t *perm, const uint32_t *key_in, bool after_sort,
                      const PlainCtl *ctl, uint32_t *key_out, double *pops, double *evap_pos, double *evap_vel,
                      double *rec, int stride, int n_cap, hipStream_t st, Profiler *prof);
inline int step_rec_stride(int n_cap) { return div_up(n_cap > 0 ? n_cap : 1, kStepBlock); }
// Log records of the launch's L substeps, the next counters, and (list.blocks
// > 0) the next re-sort's first phase.
void launch_step_finalize(const PlainStepParams &p, bool after_sort, const double *rec, int stride,
                          const PlainCtl *ctl, PlainCtl *next, unsigned long long *coll_accum,
                          double *evap_accum, dsmc_observables *log, int obs_cap, const ResortWork &work,
                          hipStream_t st, Profiler *prof);
void launch_set_ctl(PlainCtl *ctl, long long step, unsigned coll, const int *n, hipStream_t st);
// out[perm[i]] (perm null: out[i]) = key[i], i < *n.
constexpr uint32_t kNoSlot = 0xFFFFFFFFu;   // no key: no such slot
void launch_keys_by_slot(const uint32_t *key, const uint32_t *perm, const int *n, int n_cap, uint32_t *out,
                         hipStream_t st);
// stencil = 1 for slots whose atom was removed before the launch's last substep.
void launch_prev_dead_stencil(const uint32_t *key, const uint64_t *mask_last, const PlainCtl *ctl, int n_cap,
                              uint32_t dead_key, int *stencil, hipStream_t st);
// tag[j] = 1 if the atom of slot map[j] was removed in the last substep, j < *n.
void launch_last_tags(const uint32_t *map, const uint64_t *mask_last, const int *n, int n_cap, int *tag,
                      hipStream_t st);
// Collision counts of the collision step `coll` from the tagged counts.
void launch_untag_counts(const unsigned long long *cc, unsigned coll, int ncells, int *count, hipStream_t st);

}  // namespace dsmc
