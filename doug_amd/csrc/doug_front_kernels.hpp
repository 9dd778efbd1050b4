// Launch wrappers of the frontal subdomain factors (doug_fronts.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

#include "doug_fronts.hpp"

namespace doug {

// One subdomain on the device: where its panels and vectors start, and its
// pattern's arrays (FrontPattern).
struct FrontSub {
  int64_t base;  // first panel element
  int64_t vec;   // offset into the concatenated subdomain vectors
  int64_t sch;   // first element of its update matrices (set-up)
  const Front* fronts;
  const uint16_t* rpos;
  const uint32_t* src;
  const uint16_t* colfront;
  const int32_t* hptr;
  const uint16_t* hlist;
  const FrontUnit *units_f, *units_b;
  const int32_t *list_f, *list_b;
  const FrontUnit *bunits_f, *bunits_b;  // subtrees of several workgroups
  const int32_t *blist_f, *blist_b, *gpos, *gtop, *uoff;
  const uint16_t* uidx;
  int64_t ub;  // first of its entries between the workgroups' updates
  int32_t n, top0, work, nheights;
};

// The lower entries of each subdomain's matrix (converted to T) into its
// zeroed panels; A must hold no (i, j) pair twice.
template <typename T>
void launch_front_scatter(T* tiles, const FrontSub* subs, int nsub, const int32_t* inds, const int32_t* occ_ptr,
                          const int32_t* occ_pos, const int32_t* a_ptr, const int32_t* a_col, const double* a_val,
                          hipStream_t st);
// Factorises every front of height h (at most maxcount per subdomain; `wide`:
// some have more than 32 columns), all lower heights being done.  `flag` receives the first failing subdomain + 1
// on a non-positive pivot.
template <typename T>
void launch_front_factor(T* tiles, T* schur, const FrontSub* subs, int nsub, int h, int maxcount, bool wide, int* flag,
                         hipStream_t st);
// Solve of every subdomain by `groups` workgroups of nw wavefronts each
// (`updates` holds what several hand over): gathers r(inds), writes the solution to sol (FP64,
// concatenated layout).  maxwork: the largest pattern's work vector; call
// prepare_front_solve<T>() once before on a device.  skip (device, optional): the
// launch does nothing when *skip != 0.
template <typename T>
hipError_t prepare_front_solve();
template <typename T>
void launch_front_solve(const T* tiles, const FrontSub* subs, int nsub, int nw, int groups, int maxwork, const int32_t* inds,
                        const double* r, double* updates, double* sol, hipStream_t st, const double* skip = nullptr);

}  // namespace doug
