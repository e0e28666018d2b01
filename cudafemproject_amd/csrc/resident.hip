// resident.hip -- the PCG iteration (femfunc.cpp:59-111) and the explicit and
// implicit time steps (femfunc.cpp:247-343) as one launch per solve or run.
//
// A launch costs about 4 us on gfx950 even when it does nothing, and the
// launch-per-kernel forms of kernels.hip pay it once a step and twice an
// iteration, and re-read their mesh data and vectors every time.  Here one
// workgroup per patch stays on its compute unit throughout: element records
// and geometry, node state and coordinates are loaded once and kept in
// registers and LDS; between workgroups only the interface nodes' partial
// sums and the dot products' partials travel, through memory, at agent scope.
//
// What bounds it, in kcycles of 2.4 GHz: an iteration's (a step's) trip through
// memory (from the first store to the last load 3.5 at 10 workgroups, 4 to 7 at
// 100 to 230) and the element phase of one patch on one compute unit (FP64
// tets: 4 for 768 elements; for 1536 12 one by one, 8 in strips; bound by LDS
// traffic and FP64 issue).
// Measured, launch per kernel -> resident:
//   us per PCG iteration: 12x7 plate FP64 10.2 -> 1.7 (one workgroup, no
//   trip), 64x32 plate FP64 10.2 -> 3.7, 24^3 hexes FP64 14.0 -> 6.9 and mixed
//   14.0 -> 6.6, 40^3 hexes (1536 elements per patch) FP64 18.1 -> 14.5 and
//   mixed 15.3 -> 9.9; with a trip for p'K p and one for r'z, as the
//   launch-per-kernel recurrence has it, 5.3 for the 64x32 plate, 9.0 and 8.2,
//   16.7 and 12.5;
//   us per explicit step: 63x31 plate FP32 with receivers 9.1 -> 2.0, 160x80
//   plate FP64 5.7 -> 2.3, 16x16x256 column FP64 15.5 -> 8.2 and FP32
//   10.7 -> 5.9;
//   20 implicit steps of an 11x11x80 column (870 iterations) 13.4 -> 5.7 ms.
//
// Every workgroup forms every scalar itself from all partials in the same
// order, and every patch holding an interface node carries its own copy of
// the node's state, updated with the same operations: no workgroup waits for
// another's decision, and all copies have the same bits.
//
// Exchange: a workgroup's partials and its interface sums are published as
// 8-byte words that carry the number of the exchange beside their payload
// (partials: 32 bits under a 32-bit tag, interface sums: 48 under 16), so that a
// value and its arrival are one load and nothing has to be ordered.  A
// workgroup that has everyone's words of one exchange knows that everyone has
// read those of the one before, so two places (and, for the interface sums, two
// sets of entries) take turns.  Stores and loads of shared data are relaxed
// agent-scope atomics (written through, not served from a stale cache); an
// agent-scope fence would write the XCD's L2 back, some 40 us.
//
// Waiting needs all workgroups on the chip: the host launches this form only
// where they fit (res_pcg_fit), and a wait is bounded (WAIT_TICKS): past it
// the launch ends, every workgroup that gave up says so to the host, and the
// call goes on in the launch-per-kernel form.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <tuple>

#include "element.h"
#include "kernels.h"
#include "patch_common.h"
#include "resident.h"
#include "resident_dev.h"
#include "strip.h"

namespace femgpu {

namespace {

using namespace elem;
using namespace patch;
using namespace resident;

// LDS of a resident workgroup: node coordinates and vector, `comps` components
// of the node-sorted element entries, the interface nodes' contributions
// slot by slot, the tables of what the patch sends (entry and place of its
// own contribution) and where a received entry goes.
struct ResLds {
  int off_x, off_res, off_in, off_oe, off_os, off_ip, off_red, total;
};
__host__ __device__ inline ResLds res_lds(int dim, int tb, int pn, int ent, int comps, int n_in,
                                          int n_src) {
  ResLds L;
  L.off_x = al32(pn * dim * tb);
  L.off_res = L.off_x + al32(pn * dim * tb);
  L.off_in = L.off_res + al32(comps * ent * tb);
  L.off_oe = L.off_in + al32(n_src * dim * tb);
  L.off_os = L.off_oe + al32(n_in * 4);
  L.off_ip = L.off_os + al32(n_in * 2);
  L.off_red = L.off_ip + al32(n_in * 2);
  L.total = L.off_red + (16 * RES_SUMS + 8) * 8;
  return L;
}

// Resident kernels' view of the mesh.
template <typename T>
struct ResMesh {
  const PatchInfo *patches;
  const uint32_t *erec_s;
  int emax;
  const uint4 *strip_rec;  // strips (NE = 3)
  const uint32_t *strip_rec2;
  int strip_stride;
  const int32_t *pgid, *pslot;
  const uint16_t *pend;
  int pstride;             // of pgid, pslot, pend
  const uint8_t *fixmask;
  const T *coords, *escale, *diagK;
  T lam, mu;
  int np, p8, ent, pn;
  const ExchangePatch *xpatch;
  const uint32_t *out_entry;
  const uint16_t *out_src, *in_pos, *src_end, *own_pos;
  int n_in_max, n_src_max;
};

// One patch in one workgroup of PT threads for a whole launch.  NE = 1: one
// element and one DOF per thread (thread t: node t / DIM, component t % DIM),
// the element entries of every component in LDS at once, one barrier instead
// of 2 DIM - 1 per product.  Else (patches of up to 512 nodes) a node with its
// DIM DOFs in each of the first threads and the components' entries in turn
// through one list, with NE = 3 a strip of up to three elements per thread
// (StripPlan), with NE = 2 two elements one by one.
template <typename T, int DIM, int PT, int NE>
struct ResPatch {
  static constexpr bool DOF = NE == 1, STRIPS = NE == 3;
  static constexpr int ND = DOF ? 1 : DIM;     // DOFs per thread
  static constexpr int COMPS = DOF ? DIM : 1;  // components in the entry list
  static constexpr int NPE = DIM + 1, NDE = DIM * NPE;
  static constexpr int NS = DIM + STRIP_ELEMS;  // nodes of a full strip
  // the elements' geometry in registers for the whole launch, where they hold
  // it (FP64 with two elements per thread: formed again in every product)
  static constexpr bool GEOM = NE != 2 || sizeof(T) == 4;
  static constexpr int NGEO = GEOM ? DIM * DIM + 1 : 1;

  T *s_c, *s_x, *s_res, *s_in;
  uint32_t *s_oe;
  uint16_t *s_os, *s_ip;
  double *s_red;
  int ent, n_elem, n_in, in_start;
  T lam, mu;
  uint3 rec[STRIPS ? 1 : NE];  // elements
  uint4 srec;                  // the strip
  uint32_t srec2;
  T esc[NE];
  bool has, own, first;  // first: this patch accounts for the node
  unsigned fm;           // fixed DOFs of this thread
  int go;                // global DOF of this thread's first
  int gid;               // its node
  int b0, b1, l0, l1, lo;
  T dK[ND];              // diagonal of a constrained row
  T geo[NE][NGEO];

  __device__ __forceinline__ int local(int i) const {
    return DOF ? int(threadIdx.x) : int(threadIdx.x) * DIM + i;
  }
  __device__ __forceinline__ int comp(int i) const { return DOF ? int(threadIdx.x) % DIM : i; }
  __device__ __forceinline__ bool fixed(int i) const { return ((fm >> i) & 1u) != 0u; }

  // Loads the patch (one barrier; the exchange tables are ready after the
  // next).
  __device__ __forceinline__ void load(const ResMesh<T> &a, int pid, unsigned char *lds) {
    const ResLds L = res_lds(DIM, int(sizeof(T)), a.pn, a.ent, COMPS, a.n_in_max, a.n_src_max);
    s_c = reinterpret_cast<T *>(lds);
    s_x = reinterpret_cast<T *>(lds + L.off_x);
    s_res = reinterpret_cast<T *>(lds + L.off_res);
    s_in = reinterpret_cast<T *>(lds + L.off_in);
    s_oe = reinterpret_cast<uint32_t *>(lds + L.off_oe);
    s_os = reinterpret_cast<uint16_t *>(lds + L.off_os);
    s_ip = reinterpret_cast<uint16_t *>(lds + L.off_ip);
    s_red = reinterpret_cast<double *>(lds + L.off_red);
    const int t = threadIdx.x;
    const PatchInfo P = a.patches[pid];
    const ExchangePatch E = a.xpatch[pid];
    ent = a.ent;
    n_elem = P.n_elem;
    n_in = E.n_in;
    in_start = E.in_start;
    lam = a.lam;
    mu = a.mu;
    if constexpr (STRIPS) {
      const size_t i = size_t(pid) * a.strip_stride + t;
      srec = a.strip_rec[i];
      srec2 = a.strip_rec2[i];
#pragma unroll
      for (int e = 0; e < NE; ++e)
        esc[e] = a.escale ? a.escale[(size_t(pid) * NE + e) * a.strip_stride + t] : T(1);
    } else {
      const uint3 *prec = reinterpret_cast<const uint3 *>(a.erec_s) + size_t(pid) * unsigned(a.emax);
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        const int i = t + e * PT;
        rec[e] = prec[unsigned(min(i, a.emax - 1))];
        esc[e] = a.escale && i < n_elem ? a.escale[P.elem_start + i] : T(1);
      }
    }
    clear_entries<T, PT>(s_res, COMPS * ent);
    const int k = DOF ? t / DIM : t;
    has = k < P.n_own + P.n_sh;
    first = own = k < P.n_own;
    fm = 0;
    go = gid = b0 = b1 = l0 = l1 = lo = 0;
#pragma unroll
    for (int i = 0; i < ND; ++i) dK[i] = T(0);
    if (has) {
      const size_t pbase = size_t(pid) * a.pstride;
      gid = a.pgid[pbase + k];
      go = gid * DIM + (DOF ? t % DIM : 0);
      b1 = int(a.pend[pbase + k]);
      b0 = k ? int(a.pend[pbase + k - 1]) : 0;
      fm = a.fixmask[gid] & ((1u << DIM) - 1u);
      if constexpr (DOF) fm = (fm >> (t % DIM)) & 1u;
      if (!own) {
        const int j = P.sh_start + k - P.n_own;
        first = a.pslot[pbase + k] < 0;
        l1 = int(a.src_end[j]);
        l0 = k > P.n_own ? int(a.src_end[j - 1]) : 0;
        lo = int(a.own_pos[j]);
      }
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        s_c[local(i)] = a.coords[go + i];
        if (fixed(i) && first) dK[i] = a.diagK[go + i];
      }
    }
    __syncthreads();
    if constexpr (GEOM) {
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        int l[4] = {0, 0, 0, 0}, q[4];
        if constexpr (STRIPS) {
          // (node 0 past a strip's end: its elements are not formed)
#pragma unroll
          for (int n = 0; n < NPE; ++n) l[n] = int(strip_node(srec, e + n));
        } else {
          decode_rec(rec[e], l, q);
        }
        T X[NDE];
#pragma unroll
        for (int n = 0; n < NPE; ++n)
#pragma unroll
          for (int c = 0; c < DIM; ++c) X[n * DIM + c] = s_c[l[n] * DIM + c];
        elem_geometry<T, DIM>(X, esc[e], geo[e]);
      }
    }
    for (int i = t; i < n_in; i += PT) {
      s_oe[i] = a.out_entry[E.out_start + i];
      s_os[i] = a.out_src[E.out_start + i];
      s_ip[i] = a.in_pos[E.out_start + i];
    }
  }

  __device__ __forceinline__ void force(int e, T *F, int *q) const {
    int l[4];
    decode_rec(rec[e], l, q);
    T U[NDE];
#pragma unroll
    for (int n = 0; n < NPE; ++n)
#pragma unroll
      for (int c = 0; c < DIM; ++c) U[n * DIM + c] = s_x[l[n] * DIM + c];
    if constexpr (GEOM) {
      (void)elem_force_geo<T, DIM>(geo[e], U, lam, mu, F);
    } else {
      T X[NDE];
#pragma unroll
      for (int n = 0; n < NPE; ++n)
#pragma unroll
        for (int c = 0; c < DIM; ++c) X[n * DIM + c] = s_c[l[n] * DIM + c];
      (void)elem_force_free<T, DIM>(X, U, lam, mu, esc[e], F);
    }
  }

  // y = this patch's part of K x at this thread's DOFs (x: their values; the
  // other threads' through LDS).  A constrained row is its assembled diagonal,
  // in the patch that accounts for the node.
  __device__ __forceinline__ void product(const T (&x)[ND], T (&y)[ND]) {
    const int t = threadIdx.x;
    if (has)
#pragma unroll
      for (int i = 0; i < ND; ++i) s_x[local(i)] = fixed(i) ? T(0) : x[i];
    __syncthreads();
    if constexpr (DOF) {
      if (t < n_elem) {
        int q[4];
        T F[NDE];
        force(0, F, q);
#pragma unroll
        for (int c = 0; c < DIM; ++c)
#pragma unroll
          for (int n = 0; n < NPE; ++n) s_res[c * ent + q[n]] = F[n * DIM + c];
      }
      __syncthreads();
      y[0] = run_sum<T>(s_res + (t % DIM) * ent, b0, b1);
    } else if constexpr (STRIPS) {
      const int count = int(srec.x >> 30);
      T F[NS * DIM];
      if (count) {
        T U[NS * DIM];
        auto load = [&](int n) {
          const unsigned l = strip_node(srec, n) * unsigned(DIM);
#pragma unroll
          for (int c = 0; c < DIM; ++c) U[n * DIM + c] = s_x[l + c];
        };
#pragma unroll
        for (int n = 0; n < DIM; ++n) load(n);
#pragma unroll
        for (int k = 0; k < STRIP_ELEMS; ++k) {
#pragma unroll
          for (int c = 0; c < DIM; ++c) F[(k + DIM) * DIM + c] = T(0);
          if (k < count) {
            load(k + DIM);
            T f[NDE];
            (void)elem_force_geo<T, DIM>(geo[k], U + k * DIM, lam, mu, f);
#pragma unroll
            for (int i = 0; i < NDE; ++i)
              F[k * DIM + i] = k == 0 || i >= DIM * DIM ? f[i] : F[k * DIM + i] + f[i];
          }
        }
      }
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        if (c) __syncthreads();
        if (count)
#pragma unroll
          for (int n = 0; n < NS; ++n)
            if (n <= DIM || n < count + DIM) s_res[strip_entry(srec, srec2, n)] = F[n * DIM + c];
        __syncthreads();
        y[c] = run_sum<T>(s_res, b0, b1);
      }
    } else {
      // (corner 0's force is minus the others', formed again at the scatter:
      // fewer live registers)
      T F[NE][NDE - DIM];
#pragma unroll
      for (int e = 0; e < NE; ++e) {
        if (t + e * PT >= n_elem) continue;
        int q[4];
        T Fe[NDE];
        force(e, Fe, q);
#pragma unroll
        for (int j = 0; j < NDE - DIM; ++j) F[e][j] = Fe[DIM + j];
      }
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        if (c) __syncthreads();
#pragma unroll
        for (int e = 0; e < NE; ++e)
          if (t + e * PT < n_elem) {
            int l[4], q[4];
            decode_rec(rec[e], l, q);
            T f0 = F[e][c];
            s_res[q[1]] = F[e][c];
#pragma unroll
            for (int n = 2; n < NPE; ++n) {
              f0 += F[e][(n - 1) * DIM + c];
              s_res[q[n]] = F[e][(n - 1) * DIM + c];
            }
            s_res[q[0]] = -f0;
          }
        __syncthreads();
        y[c] = run_sum<T>(s_res, b0, b1);
      }
    }
    if (fm)
#pragma unroll
      for (int i = 0; i < ND; ++i)
        if (fixed(i)) y[i] = dK[i] * x[i];
  }

  // An interface node's contribution of this patch to its place (before a
  // barrier that precedes trade).
  __device__ __forceinline__ void put(const T (&y)[ND]) {
    if (has && !own)
#pragma unroll
      for (int i = 0; i < ND; ++i) s_in[lo * DIM + comp(i)] = y[i];
  }

  // Sends this patch's contributions and receives the others', an entry per
  // thread.  False when the wait ran out; the contributions are complete after
  // the next barrier.
  __device__ __forceinline__ bool trade(u64 *entries, unsigned tag, u64 *abort) {
    for (int i = threadIdx.x; i < n_in; i += PT)
      send_entry<T, DIM>(entries, s_oe[i], tag, &s_in[int(s_os[i]) * DIM]);
    for (int i = threadIdx.x; i < n_in; i += PT)
      if (!recv_entry<T, DIM>(entries, unsigned(in_start + i), tag, Patience{abort}, &s_in[int(s_ip[i]) * DIM]))
        return false;
    return true;
  }

  // The interface node's sums from all its patches, in slot order.
  __device__ __forceinline__ void collect(T (&y)[ND]) const {
    if (has && !own)
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        T q = T(0);
        for (int l = l0; l < l1; ++l) q += s_in[l * DIM + comp(i)];
        y[i] = q;
      }
  }
};

// The PCG of one workgroup: r, p, x of this thread's DOFs, the scalars the same in
// every workgroup.  One trip through memory per iteration: K z (z = invD r) is
// formed and traded instead of K p, s = K p follows from the recurrence
// s = K z + beta s (Chronopoulos and Gear, J. Comput. Appl. Math. 25 (1989)), and
//   p'Kp = z'Kz + 2 beta z's + beta^2 p's  (p, s of the last iteration)
// from sums that travel beside r'z and r'r.  Neither beta nor the step length
// uses an orthogonality that rounding loses, and every RENEW iterations (or
// where the sums cancel) s = K p and p's are formed anew, so r keeps to f - K x
// as it does with a product K p in every iteration: iterations and errors are
// those of that recurrence (64 x 32 plate, FP64 to 1e-10: 620 both, error
// 6.9e-12 both).
// (Mixed solves of the batch workload's plates and of cubes: 98.7, 93.9 and
// 91.1 ms in all with 8, 16 and 32; iterations within 3 %.)
constexpr int RENEW = 32;

// Below this r'z every iteration forms s = K p and p's, as the two-trip form
// does: its own rounding, at the end of the number range no longer relative to the
// values, would stay in a recurrence.  FP32: z or r of some 2^-100 (a solve of a 9^3
// cube run on at tolerance 0 left that floor again and was at 1e24 ||f|| after
// 12000 iterations; so it stays at the floor, as there).  FP64: the sums
// themselves end at 2^-1074.
template <typename T>
constexpr double FAINT = sizeof(T) == 8 ? 0x1p-1000 : 0x1p-160;

template <typename T, int DIM, int PT, int NE>
struct ResSolver {
  using Patch = ResPatch<T, DIM, PT, NE>;
  static constexpr int ND = Patch::ND;
  Patch &P;
  Exchange ex;
  u64 *entries;
  size_t entry_words;
  unsigned tag, entry_tag;
  int pid;
  bool alone;            // one workgroup: no exchange
  int *s_flag;           // LDS: a wait ran out
  double *s_red, *s_bc;  // LDS: the waves' sums; the totals
  double g, q2, g_prev;  // r'z, r'r; the r'z that p was formed with
  double gamma0, rr0, thresh, pause;
  int n_upd;

  __device__ __forceinline__ ResSolver(Patch &patch, const ResMesh<T> &m, u64 *words, u64 *ent,
                                       size_t ent_words, int b, int id, int *flag)
      : P(patch), entries(ent), entry_words(ent_words), pid(id), alone(m.np == 1), s_flag(flag),
        s_red(patch.s_red), s_bc(patch.s_red + 16 * RES_SUMS), g(0.0), q2(0.0), g_prev(1.0),
        n_upd(0) {
    ex = Exchange{words + RES_HEAD, res_copy_words(m.np), words + 1, m.np, b % EX_COPIES};
    // (workgroup 0 advances the tags at its end, after an exchange that every
    // workgroup took part in with the tags it reads here)
    tag = unsigned(ld_agent(words));
    entry_tag = unsigned(ld_agent(words + 3 + (sizeof(T) == 8 ? 1 : 0)));
  }

  __device__ __forceinline__ void store_tags(u64 *words) const {
    st_agent(words, u64(tag));
    st_agent(words + 3 + (sizeof(T) == 8 ? 1 : 0), u64(entry_tag));
  }

  // A trade; the sets of entries take turns, as in the explicit steps: a
  // neighbour may still be reading the last trade's.
  __device__ __forceinline__ void trade() {
    ++entry_tag;
    if (!P.trade(entries + (entry_tag & 1u) * entry_words, entry_tag, ex.abort)) *s_flag = 1;
  }

  // y = K x, complete.  False: a wait ran out.
  __device__ __forceinline__ bool apply(const T (&x)[ND], T (&y)[ND]) {
    P.product(x, y);
    if (alone) return true;
    P.put(y);
    __syncthreads();
    trade();
    __syncthreads();
    P.collect(y);
    return *s_flag == 0;
  }

  // v summed over all workgroups; with_trade: the trade of what was put beside
  // it.  False: a wait ran out.
  __device__ __forceinline__ bool sums(double (&v)[RES_SUMS], bool with_trade = false) {
    ++tag;
    const double sum = sum_by_wave<PT>(v, s_red);
    Exchange e = ex;
    e.words += (tag & 1u) * size_t(2 * RES_SUMS) * ex.np;
    if (!alone) {
      publish(e, pid, tag, sum);
      if (with_trade) trade();
    }
    return gather(e, tag, sum, v, s_bc, s_flag, alone);
  }

  // s = (cK K + diag(cMm)) p.
  __device__ __forceinline__ bool refresh(const T (&p)[ND], T (&s)[ND], T cK, const T (&cMm)[ND]) {
    const bool ok = apply(p, s);
#pragma unroll
    for (int i = 0; i < ND; ++i) s[i] = cK * s[i] + cMm[i] * p[i];
    return ok;
  }

  // Iterates from r, p, x until a stop; returns the done code.  fresh: p = 0,
  // and the threshold and the pause are formed from the first sums (eps, and
  // pause relative to r'r); else p, g_prev, thresh and pause are an earlier
  // run's.  cMm: the mass shift of this thread's DOFs.
  __device__ __forceinline__ int run(T (&r)[ND], T (&p)[ND], T (&x)[ND], const T (&invd)[ND], T cK,
                                     const T (&cMm)[ND], bool fresh, int kind, double eps,
                                     int max_iter, int last) {
    T s[ND];
    if (fresh) {
#pragma unroll
      for (int i = 0; i < ND; ++i) s[i] = T(0);
    } else if (!refresh(p, s, cK, cMm)) {
      return RES_ABORTED;
    }
    for (;;) {
      T z[ND], w[ND];
#pragma unroll
      for (int i = 0; i < ND; ++i) z[i] = mul_rn(invd[i], r[i]);
      P.product(z, w);
      double v[RES_SUMS] = {0.0, 0.0, 0.0, 0.0, 0.0};
      if (P.has)
#pragma unroll
        for (int i = 0; i < ND; ++i) {
          w[i] = cK * w[i];
          if (P.own) w[i] += cMm[i] * z[i];
          const double zi = double(z[i]);
          v[2] += zi * double(w[i]);
          if (P.first) {
            v[0] += double(r[i]) * zi;
            v[1] += double(r[i]) * double(r[i]);
            v[3] += zi * double(s[i]);
            v[4] += double(p[i]) * double(s[i]);
            // the mass shift belongs to the patch that accounts for the node
            if (!P.own) v[2] += double(cMm[i]) * zi * zi;
          }
        }
      P.put(w);
      if (!sums(v, true)) return RES_ABORTED;
      g = v[0];
      q2 = v[1];
      if (fresh) {
        fresh = false;
        gamma0 = g;
        rr0 = q2;
        thresh = kind == 0 ? eps * g : eps * eps * q2;
        pause *= q2;
      }
      if (n_upd >= 1) {
        if (kind == 0 ? g < thresh : q2 <= thresh) return 1;
      } else if (q2 == 0.0) {
        return 1;
      }
      if (!isfinite(g)) return 2;
      if (n_upd >= max_iter) return 4;
      // (looked at every eighth iteration: r'r is not monotone, and a
      // replacement at a single dip can cost directions -- a 160 x 80-class
      // plate under body force took 3225 iterations with a look at every one,
      // 1953 so, 1950 in the launch-per-kernel form)
      if ((n_upd & 7) == 0 && q2 < pause) return 5;
      if (n_upd >= last) return RES_CAP;
      const double beta_d = g / g_prev, own = v[2] + beta_d * beta_d * v[4];
      double pq = v[2] + beta_d * (2.0 * v[3] + beta_d * v[4]);
      const T beta = T(beta_d);
      // (beyond the range of T: the state of the last completed iteration)
      if (!isfinite(beta)) return 2;
      P.collect(w);
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        if (P.has && !P.own) w[i] += cMm[i] * z[i];
        p[i] = fma(beta, p[i], z[i]);
        s[i] = fma(beta, s[i], w[i]);
      }
      const bool faint = fabs(g) < FAINT<T>;
      if (faint || n_upd % RENEW == RENEW - 1 || !(pq > 0x1p-10 * own)) {
        // (or where the sums cancel)
        if (!refresh(p, s, cK, cMm)) return RES_ABORTED;
        double u[RES_SUMS] = {0.0, 0.0, 0.0, 0.0, 0.0};
        if (P.first)
#pragma unroll
          for (int i = 0; i < ND; ++i) u[0] += double(p[i]) * double(s[i]);
        if (!sums(u)) return RES_ABORTED;
        pq = u[0];
      }
      const double alpha_d = g / pq;
      // (no x or r has changed: the state of the last completed iteration)
      if (!(pq > 0.0) || !isfinite(pq) || !isfinite(alpha_d))
        return faint ? RES_FAINT : isfinite(pq) ? 3 : 2;
      g_prev = g;
      const T alpha = T(alpha_d);
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        x[i] = x[i] + alpha * p[i];
        r[i] = r[i] - alpha * s[i];
      }
      ++n_upd;
    }
  }
};

template <typename T>
struct PcgArgs {
  ResMesh<T> m;
  ResPcg<T> s;
};

template <typename T, int DIM, int PT, int NE>
__global__ __launch_bounds__(PT) void k_pcg_resident(PcgArgs<T> a) {
  using Patch = ResPatch<T, DIM, PT, NE>;
  constexpr int ND = Patch::ND;
  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ int s_flag;
  const int b = blockIdx.x;
  const int pid = (b & 7) * a.m.p8 + (b >> 3);
  if (pid >= a.m.np) return;
  if (threadIdx.x == 0) s_flag = 0;
  Patch P;
  P.load(a.m, pid, lds);
  T r[ND], p[ND], x[ND], d[ND], cMm[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    r[i] = p[i] = x[i] = d[i] = cMm[i] = T(0);
    if (P.has) {
      r[i] = a.s.r_in[P.go + i];
      d[i] = a.s.invD[P.go + i];
      if (!a.s.fresh) {
        p[i] = a.s.p[P.go + i];
        x[i] = a.s.x[P.go + i];
      }
    }
  }
  ResSolver<T, DIM, PT, NE> S(P, a.m, a.s.words, a.s.entries, a.s.entry_words, b, pid, &s_flag);
  S.n_upd = a.s.it0;
  S.gamma0 = a.s.gamma0;
  S.rr0 = a.s.rr0;
  S.thresh = a.s.thresh;
  S.pause = a.s.pause;
  if (!a.s.fresh) S.g_prev = a.s.g_prev;
  int done = S.run(r, p, x, d, T(1), cMm, a.s.fresh != 0, a.s.kind, a.s.eps, a.s.max_iter,
                   a.s.it0 + a.s.cap);
  if (done == RES_FAINT) {
    // (without a tolerance a solve goes on to its cap, and changes nothing more)
    if (!(a.s.eps > 0.0)) S.n_upd = a.s.max_iter;
    done = a.s.eps > 0.0 ? 3 : 4;
  }
  if (a.s.late && pid == a.m.np - 1) done = RES_ABORTED;
  if (done == RES_ABORTED) {
    if (threadIdx.x == 0) a.s.sc->gave_up = 1;
    return;
  }
  if (P.first)
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      a.s.x[P.go + i] = x[i];
      a.s.p[P.go + i] = p[i];
      a.s.r_out[P.go + i] = r[i];
    }
  if (pid == 0 && threadIdx.x == 0) {
    CgScalars *sc = a.s.sc;
    sc->gamma0 = S.gamma0;
    sc->rr0 = S.rr0;
    sc->thresh = S.thresh;
    sc->g[0] = sc->g[1] = S.g_prev;
    sc->g_final = S.g;
    sc->rr_final = S.q2;
    sc->iter_final = S.n_upd;
    sc->pause = S.pause;
    S.store_tags(a.s.words);
    sc->done = done;
  }
}

// Implicit GN22 steps: the predictor (k_dyn_predict), K (d~ + beta v~) and its
// trade, the residual (k_dyn_correct), the nested PCG for the acceleration,
// the corrector (k_dyn_implicit_post).
template <typename T>
struct ImplArgs {
  ResMesh<T> m;
  ResImpl<T> s;
};

// One receiver sample of this thread's DOFs, if its node has receivers.
template <typename T, int DIM, typename Patch, typename R>
__device__ __forceinline__ void record(const Patch &P, const R &s, int rec, int step, const T *d,
                                       const T *v, const T *a) {
  if (rec < 0 || step % s.rec_every != 0) return;
  const int smp = step / s.rec_every - 1;
  if (smp >= s.rec_samples) return;
  const T *src = s.rec_quantity == 0 ? d : s.rec_quantity == 1 ? v : a;
  for (int k = rec; k >= 0; k = s.rec_next[k])
#pragma unroll
    for (int i = 0; i < Patch::ND; ++i)
      s.traces[(int64_t(smp) * s.n_rec + k) * DIM + P.comp(i)] = src[i];
}

// MID: the launch begins within a step's solve.  Not a run-time flag: with both
// entries to run() in one kernel, a column of 11 x 11 x 80 hexes took 6.29 ms
// for 20 steps, in a kernel of its own 6.14.
template <typename T, int DIM, int PT, int NE, bool MID>
__global__ __launch_bounds__(PT) void k_impl_resident(ImplArgs<T> arg) {
  using Patch = ResPatch<T, DIM, PT, NE>;
  constexpr int ND = Patch::ND;
  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ int s_flag;
  const int b = blockIdx.x;
  const int pid = (b & 7) * arg.m.p8 + (b >> 3);
  if (pid >= arg.m.np) return;
  if (threadIdx.x == 0) s_flag = 0;
  Patch P;
  P.load(arg.m, pid, lds);
  const ResImpl<T> &s = arg.s;
  T d[ND], v[ND], a[ND], invd[ND], cMm[ND], ml[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    d[i] = v[i] = a[i] = invd[i] = cMm[i] = ml[i] = T(0);
    if (P.has) {
      invd[i] = s.invA[P.go + i];
      ml[i] = s.mlump[P.go + i];
      if (s.cM != T(0)) cMm[i] = s.cM * ml[i];
      if (!s.fresh) {
        d[i] = s.d[P.go + i];
        v[i] = s.v[P.go + i];
        a[i] = s.a[P.go + i];
      }
    }
  }
  const int rec = s.rec_of && P.has && P.first ? s.rec_of[P.gid] : -1;
  ResSolver<T, DIM, PT, NE> S(P, arg.m, s.words, s.entries, s.entry_words, b, pid, &s_flag);
  int done = 1, n = 0, total = 0;
  bool mid = MID;
  T x[ND], r[ND], p[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    x[i] = r[i] = p[i] = T(0);
    if (P.has && mid) {
      x[i] = a[i];
      r[i] = s.r[P.go + i];
      p[i] = s.p[P.go + i];
    }
  }
  if (mid) {
    S.n_upd = s.it0;
    S.gamma0 = s.gamma0;
    S.rr0 = s.rr0;
    S.thresh = s.thresh;
    S.g_prev = s.g_prev;
  }
  S.pause = 0.0;
  for (; n < s.n_steps && total < s.it_budget; ++n) {
    if (!mid) {
      const int step = s.step0 + n;
      const T cf = T(s.coef_file[step]), cu = T(s.coef_unit[step]);
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        d[i] = d[i] + s.dt * v[i];
        d[i] = d[i] + s.c1 * a[i];
        v[i] = v[i] + s.c2 * a[i];
        x[i] = s.beta != T(0) ? d[i] + s.beta * v[i] : d[i];
      }
      done = RES_ABORTED;
      if (!S.apply(x, r)) break;
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        const T kd = r[i];
        p[i] = x[i] = r[i] = T(0);
        if (P.has) {
          const T f = cf * s.f_file[P.go + i] + cu * s.f_unit[P.go + i] - kd;
          r[i] = s.alpha != T(0) ? f - s.alpha * ml[i] * v[i] : f;
        }
      }
      S.n_upd = 0;
      S.g_prev = 1.0;
    }
    const int it0 = S.n_upd;
    done = S.run(r, p, x, invd, s.cK, cMm, !mid, 0, s.eps, s.max_iter, it0 + s.it_budget - total);
    total += S.n_upd - it0;
    mid = false;
    if (done == RES_FAINT) done = 3;
    if (done != 1) break;
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      a[i] = x[i];
      v[i] = v[i] + s.c3 * a[i];
      d[i] = d[i] + s.c4 * a[i];
    }
    record<T, DIM>(P, s, rec, s.step0 + n, d, v, a);
  }
  if (s.late && pid == arg.m.np - 1) done = RES_ABORTED;
  if (done == RES_ABORTED) {
    if (threadIdx.x == 0) s.sc->gave_up = 1;
    return;
  }
  if (P.first && (done == 1 || done == RES_CAP))
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      s.d[P.go + i] = d[i];
      s.v[P.go + i] = v[i];
      s.a[P.go + i] = done == RES_CAP ? x[i] : a[i];
      if (done == RES_CAP) {
        s.r[P.go + i] = r[i];
        s.p[P.go + i] = p[i];
      }
    }
  if (pid == 0 && threadIdx.x == 0) {
    CgScalars *sc = s.sc;
    sc->gamma0 = S.gamma0;
    sc->rr0 = S.rr0;
    sc->thresh = S.thresh;
    sc->g[1] = S.g_prev;
    sc->iter_final = S.n_upd;
    sc->it[0] = total;
    sc->par_final = n;
    S.store_tags(s.words);
    sc->done = done;
  }
}

// Explicit GN22 steps (gn22_correct's operations, the predictor of
// k_dyn_predict): a step is one product and one trade with the patches that
// share nodes; no workgroup waits for one it has no node in common with.  The
// entries alternate between two sets (by the tag's parity): a neighbour may
// still be reading the previous step's when this patch, with that neighbour's
// in hand, writes the next.
template <typename T>
struct DynArgs {
  ResMesh<T> m;
  ResDyn<T> s;
};

template <typename T, int DIM, int PT, int NE>
__global__ __launch_bounds__(PT) void k_dyn_resident(DynArgs<T> a) {
  using Patch = ResPatch<T, DIM, PT, NE>;
  constexpr int ND = Patch::ND;
  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ int s_flag;
  const int b = blockIdx.x;
  const int pid = (b & 7) * a.m.p8 + (b >> 3);
  if (pid >= a.m.np) return;
  const bool alone = a.m.np == 1;
  if (threadIdx.x == 0) s_flag = 0;
  Patch P;
  P.load(a.m, pid, lds);
  const ResDyn<T> &s = a.s;
  T d[ND], v[ND], ac[ND], ff[ND], fu[ND], im[ND];
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    d[i] = v[i] = ac[i] = ff[i] = fu[i] = im[i] = T(0);
    if (P.has) {
      ff[i] = s.f_file[P.go + i];
      fu[i] = s.f_unit[P.go + i];
      im[i] = s.invM[P.go + i];
      if (!s.fresh) {
        d[i] = s.d[P.go + i];
        v[i] = s.v[P.go + i];
        ac[i] = s.a[P.go + i];
      }
    }
  }
  const int rec = s.rec_of && P.has && P.first ? s.rec_of[P.gid] : -1;
  bool alive = true;
  for (int n = 0; n < s.n_steps; ++n) {
    const int step = s.step0 + n;
    const T cf = T(s.coef_file[step]), cu = T(s.coef_unit[step]);
    T x[ND], kd[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) x[i] = (d[i] + s.dt * v[i]) + s.c1 * ac[i];
    P.product(x, kd);
    if (!alone) {
      P.put(kd);
      __syncthreads();
      const unsigned tag = s.tag0 + unsigned(n);
      if (!P.trade(s.entries + ((tag & 1u) ? s.entry_words : 0), tag, s.abort)) s_flag = 1;
    }
    __syncthreads();
    alive = s_flag == 0;
    if (!alive) break;
    if (!alone) P.collect(kd);
    if (P.has)
#pragma unroll
      for (int i = 0; i < ND; ++i) {
        gn22_correct<T>(cf, cu, ff[i], fu[i], kd[i], im[i], s.c2, s.c3, s.alpha, s.scale, ac[i], v[i]);
        d[i] = x[i];
      }
    record<T, DIM>(P, s, rec, step, d, v, ac);
  }
  if (P.first && alive)
#pragma unroll
    for (int i = 0; i < ND; ++i) {
      s.d[P.go + i] = d[i];
      s.v[P.go + i] = v[i];
      s.a[P.go + i] = ac[i];
    }
}

// The kernels' forms: 768 threads with one element and one DOF each (patches
// of up to 256 nodes and 768 elements; 512 threads hold the 2D patches, which
// mostly run into the node limit first); patches of up to 512 nodes: 512 threads
// with a strip and a node each, whose registers hold the strips' geometry, else
// 768 with two elements each (us per explicit step of the 16x16x256 column FP64
// 10.2 -> 8.4 and FP32 6.3 -> 5.8, per implicit iteration 15.2 -> 12.0; with 640
// threads for more strips a 40^3 cube slows from 14.5 to 15.4 us per iteration).
struct Form {
  int threads, ne;
};
constexpr int RES_NODES[] = {0, 256, 512}, RES_THREADS = 768, RES_STRIPS = 512;
constexpr int RES_LDS_MAX = 160 * 1024 - 256;

Form res_form(const DevMesh &dm) {
  if (dm.pn <= RES_NODES[1] && dm.emax <= RES_THREADS)
    return {dm.dim == 2 && dm.emax <= 512 ? 512 : RES_THREADS, 1};
  if (dm.pn > RES_NODES[2]) return {0, 0};
  if (has_strips(dm) && dm.strip_threads <= RES_STRIPS) return {RES_STRIPS, 3};
  return dm.emax <= 2 * RES_THREADS ? Form{RES_THREADS, 2} : Form{0, 0};
}

template <typename T>
ResMesh<T> res_mesh(const DevMesh &dm) {
  ResMesh<T> a{};
  a.patches = dm.patches;
  a.erec_s = dm.erec_s;
  a.emax = dm.emax;
  a.pgid = dm.pgid;
  a.pslot = dm.pslot;
  const bool strips = res_form(dm).ne == 3;
  a.pend = strips ? dm.strip_pend : dm.pend;
  a.strip_rec = dm.strip_rec;
  a.strip_rec2 = dm.strip_rec2;
  a.strip_stride = dm.strip_stride;
  a.pstride = dm.patch_threads;
  a.fixmask = dm.fixmask;
  if constexpr (sizeof(T) == 8) {
    a.coords = reinterpret_cast<const T *>(dm.coords64);
    a.escale = strips ? dm.strip_escale64 : dm.escale64;
    a.diagK = reinterpret_cast<const T *>(dm.diag64);
  } else {
    a.coords = reinterpret_cast<const T *>(dm.coords32);
    a.escale = strips ? dm.strip_escale32 : dm.escale32;
    a.diagK = reinterpret_cast<const T *>(dm.diag32);
  }
  a.lam = T(dm.lam);
  a.mu = T(dm.mu);
  a.np = dm.np;
  a.p8 = (dm.np + 7) / 8;
  a.ent = strips ? dm.strip_ent : dm.ent;
  a.pn = dm.pn;
  a.xpatch = dm.xpatch;
  a.out_entry = dm.x_out_entry;
  a.out_src = dm.x_out_src;
  a.in_pos = dm.x_in_pos;
  a.src_end = dm.x_src_end;
  a.own_pos = dm.x_own_pos;
  a.n_in_max = dm.x_in_max;
  a.n_src_max = dm.x_src_max;
  return a;
}

int res_lds_bytes(const DevMesh &dm, int tb) {
  const bool strips = res_form(dm).ne == 3;
  return res_lds(dm.dim, tb, dm.pn, strips ? dm.strip_ent : dm.ent,
                 res_form(dm).ne == 1 ? dm.dim : 1, dm.x_in_max, dm.x_src_max)
      .total;
}

template <typename T>
using PcgKernel = void (*)(PcgArgs<T>);
template <typename T>
using DynKernel = void (*)(DynArgs<T>);
template <typename T>
using ImplKernel = void (*)(ImplArgs<T>);

#define FEMGPU_RES_KERNEL(OF, KIND, NAME, ...)                                              \
  template <typename T>                                                                     \
  KIND<T> OF(int dim, Form f) {                                                             \
    if (f.ne == 3)                                                                          \
      return dim == 3 ? KIND<T>(NAME<T, 3, 512, 3 __VA_ARGS__>)                             \
                      : KIND<T>(NAME<T, 2, 512, 3 __VA_ARGS__>);                            \
    if (f.ne == 2)                                                                          \
      return dim == 3 ? KIND<T>(NAME<T, 3, 768, 2 __VA_ARGS__>)                             \
                      : KIND<T>(NAME<T, 2, 768, 2 __VA_ARGS__>);                            \
    if (dim == 3) return NAME<T, 3, 768, 1 __VA_ARGS__>;                                    \
    return f.threads == 512 ? KIND<T>(NAME<T, 2, 512, 1 __VA_ARGS__>)                       \
                            : KIND<T>(NAME<T, 2, 768, 1 __VA_ARGS__>);                      \
  }
FEMGPU_RES_KERNEL(k_pcg_resident_of, PcgKernel, k_pcg_resident)
FEMGPU_RES_KERNEL(k_dyn_resident_of, DynKernel, k_dyn_resident)
FEMGPU_RES_KERNEL(k_impl_resident_of, ImplKernel, k_impl_resident, , false)
FEMGPU_RES_KERNEL(k_impl_mid_resident_of, ImplKernel, k_impl_resident, , true)
#undef FEMGPU_RES_KERNEL

// Workgroups of a launch (short_grid: up to the last patch's, and without it).
int grid_of(int np, int p8, bool short_grid) {
  int n = 8 * p8;
  if (short_grid && np > 1)
    while (((n - 1) & 7) * p8 + ((n - 1) >> 3) >= np) --n;
  return short_grid && np > 1 ? n - 1 : n;
}

// Whether a kernel of this form fits the plan, a workgroup per compute unit.
bool fits(const DevMesh &dm, int device, const void *fn, int lds, ResFit *fit) {
  const int cu = compute_units(device);
  if (cu < 1 || lds > RES_LDS_MAX) return false;
  const int per = blocks_per_cu(fn, res_form(dm).threads, lds);
  const int grid = 8 * ((dm.np + 7) / 8);
  if (per < 1 || grid > cu) return false;
  fit->block = 1.0 / per;
  fit->share = double(grid) / (double(per) * cu);
  fit->groups = grid;
  return true;
}

}  // namespace

int blocks_per_cu(const void *fn, int threads, int lds) {
  static std::mutex mu;
  static std::map<std::tuple<const void *, int, int>, int> seen;
  std::lock_guard<std::mutex> lock(mu);
  auto key = std::make_tuple(fn, threads, lds);
  auto it = seen.find(key);
  if (it != seen.end()) return it->second;
  int n = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, fn, threads, size_t(lds)) != hipSuccess) {
    (void)hipGetLastError();
    n = 0;
  }
  seen[key] = n;
  return n;
}

int compute_units(int device) {
  static std::mutex mu;
  static std::map<int, int> seen;
  std::lock_guard<std::mutex> lock(mu);
  auto it = seen.find(device);
  if (it != seen.end()) return it->second;
  int n = 0;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) {
    (void)hipGetLastError();
    n = 0;
  }
  seen[device] = n;
  return n;
}

template <typename T>
bool res_pcg_fit(const DevMesh &dm, int device, ResFit *fit) {
  const Form f = res_form(dm);
  return dm.xpatch && f.ne && fits(dm, device, reinterpret_cast<const void *>(k_pcg_resident_of<T>(dm.dim, f)),
                                   res_lds_bytes(dm, int(sizeof(T))), fit);
}

template <typename T>
void launch_res_pcg(const DevMesh &dm, const ResPcg<T> &s, hipStream_t st, bool short_grid) {
  const PcgArgs<T> a{res_mesh<T>(dm), s};
  const Form f = res_form(dm);
  hipLaunchKernelGGL(k_pcg_resident_of<T>(dm.dim, f), dim3(grid_of(a.m.np, a.m.p8, short_grid)),
                     dim3(f.threads),
                     res_lds_bytes(dm, int(sizeof(T))), st, a);
}

template <typename T>
bool res_dyn_fit(const DevMesh &dm, int device, ResFit *fit) {
  const Form f = res_form(dm);
  return dm.xpatch && f.ne && fits(dm, device, reinterpret_cast<const void *>(k_dyn_resident_of<T>(dm.dim, f)),
                                   res_lds_bytes(dm, int(sizeof(T))), fit);
}

template <typename T>
void launch_res_dyn(const DevMesh &dm, const ResDyn<T> &s, hipStream_t st, bool short_grid) {
  const DynArgs<T> a{res_mesh<T>(dm), s};
  const Form f = res_form(dm);
  hipLaunchKernelGGL(k_dyn_resident_of<T>(dm.dim, f), dim3(grid_of(a.m.np, a.m.p8, short_grid)),
                     dim3(f.threads),
                     res_lds_bytes(dm, int(sizeof(T))), st, a);
}

template <typename T>
bool res_impl_fit(const DevMesh &dm, int device, ResFit *fit) {
  const Form f = res_form(dm);
  const int lds = res_lds_bytes(dm, int(sizeof(T)));
  ResFit mid;
  if (!dm.xpatch || !f.ne ||
      !fits(dm, device, reinterpret_cast<const void *>(k_impl_resident_of<T>(dm.dim, f)), lds, fit) ||
      !fits(dm, device, reinterpret_cast<const void *>(k_impl_mid_resident_of<T>(dm.dim, f)), lds, &mid))
    return false;
  // (either may be launched under one turn)
  fit->share = std::max(fit->share, mid.share);
  fit->block = std::max(fit->block, mid.block);
  return true;
}

template <typename T>
void launch_res_impl(const DevMesh &dm, const ResImpl<T> &s, hipStream_t st, bool short_grid) {
  const ImplArgs<T> a{res_mesh<T>(dm), s};
  const Form f = res_form(dm);
  hipLaunchKernelGGL(s.mid ? k_impl_mid_resident_of<T>(dm.dim, f) : k_impl_resident_of<T>(dm.dim, f),
                     dim3(grid_of(a.m.np, a.m.p8, short_grid)), dim3(f.threads),
                     res_lds_bytes(dm, int(sizeof(T))), st, a);
}

template <typename T>
static hipError_t prepare_t() {
  hipError_t e = hipSuccess, r;
  for (int dim : {2, 3})
    for (Form f : {Form{512, 1}, Form{768, 1}, Form{512, 3}, Form{768, 2}})
      for (const void *fn : {reinterpret_cast<const void *>(k_pcg_resident_of<T>(dim, f)),
                             reinterpret_cast<const void *>(k_dyn_resident_of<T>(dim, f)),
                             reinterpret_cast<const void *>(k_impl_resident_of<T>(dim, f)),
                             reinterpret_cast<const void *>(k_impl_mid_resident_of<T>(dim, f))})
        if ((r = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, RES_LDS_MAX)) !=
            hipSuccess)
          e = r;
  return e;
}

hipError_t prepare_resident_kernels() {
  const hipError_t e = prepare_t<double>(), r = prepare_t<float>();
  return e != hipSuccess ? e : r;
}

#define FEMGPU_RES_INST(T)                                                    \
  template bool res_pcg_fit<T>(const DevMesh &, int, ResFit *);               \
  template void launch_res_pcg<T>(const DevMesh &, const ResPcg<T> &, hipStream_t, bool); \
  template bool res_dyn_fit<T>(const DevMesh &, int, ResFit *);               \
  template void launch_res_dyn<T>(const DevMesh &, const ResDyn<T> &, hipStream_t, bool); \
  template bool res_impl_fit<T>(const DevMesh &, int, ResFit *);              \
  template void launch_res_impl<T>(const DevMesh &, const ResImpl<T> &, hipStream_t, bool);
FEMGPU_RES_INST(double)
FEMGPU_RES_INST(float)

}  // namespace femgpu
