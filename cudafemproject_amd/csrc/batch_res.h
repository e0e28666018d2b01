// batch_res.h -- resident form of the lockstep schedule for 2D batches: every
// instance's PCG for NR right-hand sides runs in its own workgroups, one per
// patch, that stay on the chip until the instance is done (batch_res.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "batch_ls.h"

namespace femgpu {

constexpr int BR_THREADS = 512;              // a DOF and an element per thread
constexpr int BR_NODES = BR_THREADS / 2;
constexpr int BR_ELEMS = BR_THREADS;

// Most neighbours of a node within its patch: regular triangulations have six,
// and with 8 the rows of four systems fit the registers of two workgroups per
// compute unit; a mesh with more (counted on the host when it is loaded) runs
// with 12, which spill (60 plates of 80 x 40, four load cases, FP64, all with 8
// or all with 12: 21.9 against 24.7 ms).
constexpr int BR_DEGREE = 8, BR_DEGREE_MAX = 12;

// Words of a patch in its instance's exchange (three places of 2 nr values).
constexpr size_t br_patch_words(int nr) { return size_t(3) * 4 * nr; }
// Words of an interface entry: nr times two doubles, 48 bits to a word.
constexpr int br_entry_words(int nr) { return nr * 3; }

struct BRArgs {
  const PatchInfo *patches;            // of the lockstep plans (pad: instance)
  const uint32_t *erec;
  const int4 *sh_info;
  const uint16_t *node_end;
  const uint8_t *fixmask;
  const double *coords, *diagK;
  const BLInst *inst;
  const ExchangePatch *xpatch;
  const uint32_t *out_entry;
  const uint16_t *out_src, *in_pos, *src_end, *own_pos;
  const int32_t *order;                // patch of each ticket: instances in turn
  int np, ent, pn, n_in_max, n_src_max;
  const double *f, *invD;              // [node][rhs][2], [node][2]
  double *x;                           // solution, likewise
  unsigned long long *entries, *words; // zero before the launch
  unsigned long long *abort;           // zero; nonzero after a launch that did not complete; then
                                       // the bound of a wait (0: a second), the ticket counter,
                                       // the time of the last sign of progress (zero both)
  BLState *st;                         // per (instance, rhs), written at the end
  int max_iter;
  double tol2;
};

// LDS of a workgroup, and how many workgroups the device holds (0: the kernel
// does not run there); block: the part of a compute unit that one takes.
int br_lds_bytes(int nr, int pn, int ent, int n_in, int n_src);
int br_capacity(int nr, int degree, int lds, int device, double *block);

// groups: at least as many as the patches of any instance, and at most
// br_groups_max, what the registers let the device hold (those that start late
// find no ticket left, so more would do no harm).
int br_groups_max(int device);
void launch_batch_resident(int nr, int degree, const BRArgs &a, int groups, hipStream_t s);

// Right-hand sides to internal node order padded to nr, and solutions back.
void launch_br_rhs_in(int64_t n, int n_rhs, int nr, const int32_t *perm, const double *user,
                      double *f, hipStream_t s);
void launch_br_rhs_out(int64_t n, int n_rhs, int nr, const int32_t *perm, const double *x,
                       double *user, hipStream_t s);

hipError_t prepare_br_kernels();

}  // namespace femgpu
