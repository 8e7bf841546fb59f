// readout.hpp -- conversion of the state between its device layout and the
// host layout of the C ABI (double precision, AoS rows), on the device: host
// reads and writes are then one conversion kernel and one copy.
#pragma once

#include "fused.hpp"
#include "plain.hpp"

namespace dsmc {

// Which vector of the FP32 state records: the position or velocity (value +
// remainder) or the remainder alone.
enum class RecVec { Pos, Vel, PosRem, VelRem };

// out row i = the vector of slot map[i] (slot i when map is null), i < n.
void launch_pack_records(RecVec what, const FusedPtrs &s, const uint32_t *map, int n, double *out,
                         hipStream_t st);
// out[i] = the label of slot map[i].
void launch_pack_labels(const FusedPtrs &s, const uint32_t *map, int n, int *out, hipStream_t st);
// FP32 state of atom i (slot i, label i) from rows i of pos and vel (n x 3).
void launch_unpack_records(const double *pos, const double *vel, int n, const FusedPtrs &s,
                           hipStream_t st);
// out (n x ncols) from ncols columns: out row i = element map[i] of each.
void launch_pack_columns(const double *const *cols, int ncols, int n, double *out, hipStream_t st);
void launch_pack_columns(const float *const *cols, int ncols, const uint32_t *map, int n, double *out,
                         hipStream_t st);
// The reverse: element i (map[i]) of each column = row i of in.
void launch_unpack_columns(const double *in, int ncols, int n, double *const *cols, hipStream_t st);
void launch_unpack_columns(const double *in, int ncols, const uint32_t *map, int n, float *const *cols,
                           hipStream_t st);
// out[i] = in[i], widened.
void launch_widen(const float *in, long long n, double *out, hipStream_t st);
void launch_iota(int *out, int n, hipStream_t st);
// stencil[i] = 1 for slots with the dead key, 0 for the alive ones.
void launch_dead_stencil(const uint32_t *key, const int *n_dev, int n_cap, uint32_t dead_key,
                         int *stencil, hipStream_t st);
// Initial sigma v_r,max of every composite key (initSigvrmax, setUp.cu:287-292;
// the dead key after the traps gets zero).
void launch_init_sigvrmax(const TrapDev *traps, const int *key_base, int n_traps, int n_keys, double *out,
                          hipStream_t st);
void launch_init_sigvrmax(const TrapDev *traps, const int *key_base, int n_traps, int n_keys, float *out,
                          hipStream_t st);

}  // namespace dsmc
