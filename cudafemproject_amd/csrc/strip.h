// strip.h -- patch kernels whose threads take strips of elements (StripPlan)
// instead of single ones: the matvec and the PCG step of plans that run in
// launches (strip.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"

namespace femgpu {

// Threads of a strip workgroup: at most a quarter more than the patch's nodes.
constexpr int STRIP_THREADS_MAX = 640;

// Strips are planned for plans of 512 threads and for those of 256 with more than
// RES_PATCHES_MAX patches (the others run resident with an element per thread,
// resident.h), where every patch has at most 5/4 as many strips as threads.
inline bool has_strips(const DevMesh &dm) { return dm.strip_rec != nullptr; }

// Whether the kernels of arithmetic T take strips.  In FP64 not with a wave more
// than the patch's nodes need: it costs the fourth workgroup of a compute unit
// (47^3 hexes: 31.5 us per iteration against 25.2 element by element; FP32 17.8
// against 18.2).
template <typename T>
inline bool use_strips(const DevMesh &dm) {
  return has_strips(dm) && (sizeof(T) == 4 || dm.strip_threads <= dm.patch_threads);
}

// y = K x as launch_matvec_patch (owned nodes final, interface nodes to slots).
template <typename T>
void launch_strip_matvec(const DevMesh &dm, const T *x, T *y, T *partial, hipStream_t s);

// The same on FP64 vectors in user order (launch_matvec_user).
template <typename T>
void launch_strip_matvec_user(const DevMesh &dm, const double *x, double *y, T *partial,
                              hipStream_t s);

// The patch kernel of a PCG iteration (launch_pcg_iter).
template <typename T>
struct StripPcg {
  const T *r, *invD;
  T *x, *p, *q, *partial;
  OpShift<T> sh;
  CgScalars *sc;
  double *part;
  const double *prz, *prr;
  int parity;
};
template <typename T>
void launch_strip_pcg(const DevMesh &dm, const StripPcg<T> &a, hipStream_t s);

hipError_t prepare_strip_kernels();

}  // namespace femgpu
