// What the workgroups of a direct encode leave in the scratch for the run after
// theirs and for a reader behind them on the stream.
//
// Workgroups start in no guaranteed order and act on the words as they found
// them when they started, while others of the same run may have changed them
// since: one that starts after the last chunk's has given up finds the count
// moved on and the abort mark set.  Whatever a run says about ITSELF therefore
// goes by its nonce, which every workgroup has from the host, and never by the
// count.
#pragma once

#include <stdint.h>

#include "nz_format.h"

#define NZ_LOOKBACK_ABORT 0xAB0F7EDDu

// Whatever the memory held before its first use is as good a start as any.
struct NzLbWords {
  uint32_t runs;      // direct encodes that have used this scratch, advanced by the workgroup of the last chunk: the
                      // announcements' mark is made of it and the nonce, so those of an earlier run of the
                      // very same call (a replayed graph) do not pass for this run's
  uint32_t abort;     // NZ_LOOKBACK_ABORT after a run in which a workgroup gave up: the next run then leaves the placing
                      // to nz_compact_kernel as well (and says so through the same flags) and takes the mark away
  uint64_t left_out;  // nonce of the last run that left a record out of the container, whatever the reason
};

template <typename T>
NZ_HD static inline void nz_lb_put(T* at, T v) {
#ifdef __HIP_DEVICE_COMPILE__
  __hip_atomic_store(at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#else
  *at = v;
#endif
}
// a workgroup of run `nonce` leaves a record out of the container
NZ_HD static inline void nz_lb_left_out(NzLbWords* w, uint64_t nonce) { nz_lb_put(&w->left_out, nonce); }
// ... all of its records, because it found the abort mark when it started (with the count at `runs`)
NZ_HD static inline void nz_lb_unplaced(NzLbWords* w, uint64_t nonce, uint32_t runs, bool last_chunk) {
  nz_lb_left_out(w, nonce);
  if (last_chunk) {
    nz_lb_put(&w->runs, runs + 1u);
    nz_lb_put(&w->abort, 0u);
  }
}
// ... all of its records, because it has given up waiting
NZ_HD static inline void nz_lb_gave_up(NzLbWords* w, uint64_t nonce, uint32_t runs, bool last_chunk) {
  nz_lb_put(&w->abort, NZ_LOOKBACK_ABORT);
  nz_lb_left_out(w, nonce);
  if (last_chunk) nz_lb_put(&w->runs, runs + 1u);
}
// the last chunk's workgroup has found its place: every other has announced, so all of them have read the count
NZ_HD static inline void nz_lb_placed(NzLbWords* w, uint32_t runs, bool last_chunk) {
  if (last_chunk) nz_lb_put(&w->runs, runs + 1u);
}
// behind the run `nonce`: is its container not whole?
NZ_HD static inline bool nz_lb_not_whole(const NzLbWords* w, uint64_t nonce) { return w->left_out == nonce; }
