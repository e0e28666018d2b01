// resident.h -- PCG solves and explicit time steps that stay on the chip: one
// launch runs many iterations (steps), one workgroup per patch, the patch's
// mesh data and node state in registers and LDS throughout (resident.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"
#include "resident_gate.h"

namespace femgpu {

// The workgroups' exchange buffer for np patches, in 8-byte words: the tag of
// the last exchange, the abort flag, the bound of a wait (0: a second), the tags
// of the last trade of entries (FP32, FP64; every launch advances its tags), and
// the tagged partials in EX_COPIES copies on pages of their own.  The interface entries are tagged
// words too (res_entry_words).  Both are zeroed when they are allocated or the
// plan changes, and after an aborted launch.
constexpr int EX_COPIES = 8;
constexpr size_t RES_HEAD = 512;
constexpr int RES_SUMS = 5;  // sums of a PCG iteration, in two places in turn
__host__ __device__ inline size_t res_copy_words(int np) {
  return (size_t(4 * RES_SUMS) * size_t(np) + 511) & ~size_t(511);
}
inline size_t res_words(int np) { return RES_HEAD + EX_COPIES * res_copy_words(np); }
// Words of an entry: dim values of tb bytes, 48 bits to a word.
__host__ __device__ constexpr int res_entry_size(int dim, int tb) { return (dim * tb * 8 + 47) / 48; }
template <typename T>
inline size_t res_entry_words(int64_t n_entries, int dim) {
  return size_t(n_entries) * res_entry_size(dim, int(sizeof(T))) + 1;
}

// The largest plan the exchange tables are built for (compute units).
constexpr int RES_PATCHES_MAX = 256;

// One resident PCG launch.  r, x, p: node vectors in internal order; the
// solve starts from r_in (x = p = 0) when fresh, else from r_in, x, p and
// the scalars of an earlier launch.
template <typename T>
struct ResPcg {
  const T *r_in;
  T *x, *p, *r_out;
  const T *invD;
  unsigned long long *entries;  // two sets of interface entries
  size_t entry_words;           // of a set (res_entry_words)
  unsigned long long *words;    // res_words(np)
  CgScalars *sc;              // the scalars at the end (host-visible memory)
  int fresh, kind;
  double eps;             // fresh: tolerance (threshold formed from the initial residual)
  double gamma0, rr0, thresh, g_prev;  // not fresh
  int late;               // tests: the last patch's workgroup gives up at its end
  double pause;           // stop with done = 5 once r'r < pause (fresh: times
                          // the initial r'r; 0: never)
  int it0, max_iter, cap; // updates done before, in all, and at most in this launch
};

// done codes of a resident launch besides CgScalars': 6 the launch did not
// complete (its workgroups were not on the chip together), 7 cap reached; within
// the kernels 8 the sums underflowed (3 or 4 to the host).  Every workgroup that
// gives up sets gave_up itself: it may be after the one that writes the scalars
// has ended, in the last exchange.
constexpr int RES_ABORTED = 6, RES_CAP = 7, RES_FAINT = 8;

// Whether the plan's PCG runs resident: patches of up to 512 nodes and 1536
// elements, every workgroup on a compute unit of its own.  Several workgroups
// per unit would fit, and lose to the launch-per-kernel form (a 40^3-hex cube
// in 500 patches, with two trips per iteration: FP64 32.3 against 18.1 us, mixed
// 20.4 against 15.3), whose launches cost less the more work there is between
// them; in 256 patches of twice the size the resident form is ahead, 14.5 and
// 9.9 us.
template <typename T>
bool res_pcg_fit(const DevMesh &dm, int device, ResFit *fit);

// (short_grid: tests; a workgroup that others wait for is left out)
template <typename T>
void launch_res_pcg(const DevMesh &dm, const ResPcg<T> &a, hipStream_t s, bool short_grid);

// Receivers of a resident run (rec_of null: none): per node its first receiver
// or -1, the receivers of one node linked by rec_next.
template <typename T>
struct ResRecv {
  const int32_t *rec_of, *rec_next;
  int n_rec, rec_every, rec_samples, rec_quantity;
  T *traces;
};

// Explicit GN22 steps step0 .. step0 + n_steps - 1 (1-based) in one launch;
// from d = v = a = 0 when fresh, else from d, v, a, which hold the state at
// the end.
template <typename T>
struct ResDyn : ResRecv<T> {
  T *d, *v, *a;
  const T *f_file, *f_unit, *invM;
  const double *coef_file, *coef_unit;   // per step
  T dt, c1, c2, c3, alpha, scale;        // DynCoeffs
  unsigned long long *entries;           // two sets of entry_words
  size_t entry_words;
  unsigned long long *abort;             // zero; nonzero after a launch that did not complete;
                                         // then the bound of a wait (0: a second)
  unsigned tag0;                         // tags tag0 .. tag0 + n_steps - 1, following the last launch's
  int fresh, step0, n_steps;
};

template <typename T>
bool res_dyn_fit(const DevMesh &dm, int device, ResFit *fit);

template <typename T>
void launch_res_dyn(const DevMesh &dm, const ResDyn<T> &a, hipStream_t s, bool short_grid);

// Implicit GN22 steps in one launch, likewise; a launch ends early when its PCG
// iterations reach it_budget, within a step's solve (sc->done RES_CAP: d, v, a, r, p
// and the scalars are the solve's, the next launch continues it, mid) or between
// two.  At the end sc->done is 1, RES_CAP or the done code of the step that failed,
// sc->par_final the steps completed and sc->it[0] the launch's PCG iterations.
template <typename T>
struct ResImpl : ResRecv<T> {
  T *d, *v, *a, *r, *p;
  const T *f_file, *f_unit, *mlump, *invA;
  const double *coef_file, *coef_unit;
  T dt, c1, c2, c3, c4, alpha, beta;
  T cK, cM;               // operator cK K + cM diag(mlump) (cM 0: no mass)
  double eps;             // nested PCG: gamma < eps gamma0
  int max_iter, it_budget;
  unsigned long long *words, *entries;
  size_t entry_words;     // as ResPcg
  CgScalars *sc;
  int late;               // as ResPcg
  int fresh, step0, n_steps;
  int mid, it0;           // mid: the launch before ended in step0's solve after it0 iterations
  double gamma0, rr0, thresh, g_prev;  // and these are its scalars
};

template <typename T>
bool res_impl_fit(const DevMesh &dm, int device, ResFit *fit);

template <typename T>
void launch_res_impl(const DevMesh &dm, const ResImpl<T> &a, hipStream_t s, bool short_grid);

hipError_t prepare_resident_kernels();

// Workgroups of a kernel that a compute unit holds, and the device's units
// (asked of the runtime once per kernel and LDS size).
int blocks_per_cu(const void *fn, int threads, int lds);
int compute_units(int device);

}  // namespace femgpu
