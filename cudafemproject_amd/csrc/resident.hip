// resident.hip -- the PCG iteration (femfunc.cpp:59-111) as one launch per
// solve.
//
// A launch costs about 4 us on gfx950 even when it does nothing, and the
// two-launch iteration of kernels.hip pays it twice and re-reads its mesh
// data and vectors every time.  Here one workgroup per patch stays on its
// compute unit for the whole solve: element records, coordinates, r, p, x
// and M^-1 are loaded once and kept in registers and LDS; between
// workgroups only the interface nodes' partial sums and the dot products'
// partials travel, through memory, at agent scope.  What bounds an iteration
// now is those two trips, some 3.5 kcycles each from the first store to the
// last load (10 workgroups; 4 to 7 at 100), then the element phase of one
// workgroup on one compute unit (2 to 5 kcycles in FP64).  Measured, us per
// iteration, launch per kernel -> resident: 12x7 plate FP64 10.2 -> 1.9 (one
// workgroup, no trips), 64x32 plate FP64 10.2 -> 5.6, 24^3-hex cube FP64
// 14.0 -> 10.0 and mixed 14.0 -> 8.9, 32^3 hexes FP64 14.4 -> 12.0.
//
// Every workgroup forms every scalar itself from all partials in the same
// order, and every patch holding an interface node carries its own copy of
// the node's state, updated with the same operations: no workgroup waits for
// another's decision, and all copies have the same bits.
//
// Exchange: a workgroup's partials and its interface sums are published as
// 8-byte words, 32 bits of payload under a 32-bit tag (the number of the
// exchange), so that a value and its arrival are one load and nothing has to
// be ordered: an iteration is two trips through memory.  Every workgroup has
// read an exchange's words before it publishes in the next one, so each word
// has one place.  Stores and loads of shared data are relaxed agent-scope
// atomics (written through, not served from a stale cache); an agent-scope
// fence would write the XCD's L2 back, some 40 us.
//
// Waiting needs all workgroups on the chip: the host launches this form only
// where they fit (res_pcg_fits), and a wait is bounded (WAIT_TICKS): past it
// the launch ends with an abort flag and the host runs the launch-per-kernel
// form instead.
#include <hip/hip_runtime.h>

#include <map>
#include <mutex>
#include <tuple>

#include "element.h"
#include "kernels.h"
#include "patch_common.h"
#include "resident.h"

namespace femgpu {

namespace {

using namespace elem;
using namespace patch;

using u64 = unsigned long long;

constexpr u64 WAIT_TICKS = 100000000ull;  // one second of the 100 MHz clock

__device__ __forceinline__ void st_agent(u64 *p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 ld_agent(const u64 *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A value as tagged words (one for FP32, two for FP64), and back.
template <typename T>
constexpr int NW = sizeof(T) / 4;

__device__ __forceinline__ void tag_words(float v, unsigned tag, u64 (&w)[1]) {
  w[0] = (u64(tag) << 32) | __float_as_uint(v);
}
__device__ __forceinline__ void tag_words(double v, unsigned tag, u64 (&w)[2]) {
  const u64 b = static_cast<u64>(__double_as_longlong(v));
  w[0] = (u64(tag) << 32) | (b & 0xffffffffull);
  w[1] = (u64(tag) << 32) | (b >> 32);
}
__device__ __forceinline__ float untag(const u64 (&w)[1]) { return __uint_as_float(unsigned(w[0])); }
__device__ __forceinline__ double untag(const u64 (&w)[2]) {
  return __longlong_as_double(static_cast<long long>((w[1] << 32) | (w[0] & 0xffffffffull)));
}

// A bounded wait: true once the caller should give up (another workgroup
// did, or WAIT_TICKS have passed since the 256th look).
struct Patience {
  u64 *abort;
  u64 start = 0;
  __device__ __forceinline__ bool over(int spin) {
    if ((spin & 255) != 255) return false;
    const u64 now = wall_clock64();
    if (start == 0) start = now;
    if (ld_agent(abort) == 0 && now - start <= WAIT_TICKS) return false;
    st_agent(abort, 1);
    return true;
  }
};

// Interface sums travel as entries (femgpu_internal.h): DIM values of W words,
// word w of 64 consecutive entries together.
template <typename T, int DIM>
__device__ __forceinline__ size_t entry_word(unsigned e, int w) {
  return (size_t(e >> 6) * (DIM * NW<T>) + w) * 64 + (e & 63u);
}

// Component c of an entry.
template <typename T, int DIM>
__device__ __forceinline__ void send_entry(u64 *entries, unsigned e, int c, unsigned tag, T v) {
  u64 w[NW<T>];
  tag_words(v, tag, w);
#pragma unroll
  for (int h = 0; h < NW<T>; ++h) st_agent(&entries[entry_word<T, DIM>(e, c * NW<T> + h)], w[h]);
}

// Component c of the entries e0 + i (i = i0, i0 + 256, ... below n) into
// v[pos[i] * DIM + c], four of them in flight.  False when the wait ran out.
template <typename T, int DIM>
__device__ __forceinline__ bool recv_entries(const u64 *entries, unsigned e0, int i0, int n, int c,
                                             unsigned tag, u64 *abort, T *v, const uint16_t *pos) {
  constexpr int W = NW<T>, NB = 4;
  for (int ib = i0; ib < n; ib += 256 * NB) {
    u64 h[NB][W];
    Patience wait{abort};
    for (int spin = 0;; ++spin) {
      bool all = true;
#pragma unroll
      for (int m = 0; m < NB; ++m)
        if (ib + 256 * m < n)
#pragma unroll
          for (int k = 0; k < W; ++k)
            h[m][k] = ld_agent(&entries[entry_word<T, DIM>(e0 + ib + 256 * m, c * W + k)]);
#pragma unroll
      for (int m = 0; m < NB; ++m)
        if (ib + 256 * m < n)
#pragma unroll
          for (int k = 0; k < W; ++k) all = all && unsigned(h[m][k] >> 32) == tag;
      if (all) break;
      if (wait.over(spin)) return false;
    }
#pragma unroll
    for (int m = 0; m < NB; ++m)
      if (ib + 256 * m < n) v[int(pos[ib + 256 * m]) * DIM + c] = untag(h[m]);
  }
  return true;
}

// The exchange words lie in EX_COPIES copies, each read by every
// EX_COPIES-th workgroup (a copy per XCD): all workgroups polling one copy
// of a few kilobytes queue up at the memory channels that hold it.
struct Exchange {
  u64 *words;      // copy 0 of this exchange: [2 * NV][np]
  size_t stride;   // words from copy to copy
  u64 *abort;      // nonzero: a workgroup gave up waiting
  int np, copy;    // copy: the one this workgroup reads
};

// Sums of NV values over the workgroup's threads, valid in wave 0 (the same
// bits in every lane; fixed order).  s_red: NV * PT / 64 doubles that no
// thread still reads or writes for another sum.
template <int PT, int NV>
__device__ __forceinline__ void sum_to_wave0(double (&v)[NV], double *s_red) {
  constexpr int W = PT / 64;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
  if (l == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) s_red[k * W + w] = v[k];
  __syncthreads();
  if (w == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      // (at most 16 waves: one row, its sum in every lane of the row)
      double q = s_red[k * W + min(l & 15, W - 1)];
      if ((l & 15) >= W) q = 0.0;
      q += dpp_f64<0xB1>(q);
      q += dpp_f64<0x4E>(q);
      q += dpp_f64<0x141>(q);
      q += dpp_f64<0x140>(q);
      v[k] = q;
    }
}

// Wave 0 publishes the workgroup's NV values under `tag`.
template <int NV>
__device__ __forceinline__ void publish(const Exchange &x, int pid, unsigned tag,
                                        const double (&v)[NV]) {
  const int t = threadIdx.x;
  if (t < 2 * NV * EX_COPIES) {
    const int k = t % (2 * NV), copy = t / (2 * NV);
    double d = v[0];
#pragma unroll
    for (int i = 1; i < NV; ++i) d = (k >> 1) == i ? v[i] : d;
    u64 w[2];
    tag_words(d, tag, w);
    st_agent(&x.words[copy * x.stride + size_t(k) * x.np + pid], (k & 1) ? w[1] : w[0]);
  }
}

// Wave 0 gathers every workgroup's NV values of `tag` (NB loads of each lane
// in flight) and sums them in a fixed order; the sums reach every thread
// through s_bc (NV doubles) behind a barrier, which also ends the wait for
// the entries.  alone: v is the sum already.  False when a workgroup gave up
// (or *s_flag was set).
template <int NV>
__device__ __forceinline__ bool gather(const Exchange &x, unsigned tag, double (&v)[NV],
                                       double *s_bc, int *s_flag, bool alone) {
  constexpr int NB = 4;
  if (threadIdx.x < 64 && !alone) {
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = 0.0;
    const u64 *words = x.words + x.copy * x.stride;
    bool ok = true;
    for (int i0 = threadIdx.x; ok && i0 < x.np; i0 += 64 * NB) {
      u64 h[NB][NV][2];
      Patience wait{x.abort};
      for (int spin = 0;; ++spin) {
        bool all = true;
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int k = 0; k < 2 * NV; ++k)
            if (i0 + 64 * i < x.np)
              h[i][k >> 1][k & 1] = ld_agent(&words[size_t(k) * x.np + i0 + 64 * i]);
#pragma unroll
        for (int i = 0; i < NB; ++i)
#pragma unroll
          for (int k = 0; k < 2 * NV; ++k)
            if (i0 + 64 * i < x.np) all = all && unsigned(h[i][k >> 1][k & 1] >> 32) == tag;
        if (all) break;
        if (wait.over(spin)) {
          ok = false;
          break;
        }
      }
#pragma unroll
      for (int i = 0; i < NB; ++i)
        if (i0 + 64 * i < x.np)
#pragma unroll
          for (int k = 0; k < NV; ++k) v[k] += untag(h[i][k]);
    }
    if (!ok) *s_flag = 1;
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] = wave_sum(v[k]);
  }
  if (threadIdx.x == 0)
#pragma unroll
    for (int k = 0; k < NV; ++k) s_bc[k] = v[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = s_bc[k];
  return *s_flag == 0;
}

// LDS of a resident workgroup: node coordinates and vector, the node-sorted
// element entries of every component, the interface nodes' contributions
// slot by slot, the tables of what the patch sends (entry and place of its
// own contribution) and where a received entry goes.
struct ResLds {
  int off_x, off_res, off_in, off_oe, off_os, off_ip, off_red, total;
};
__host__ __device__ inline ResLds res_lds(int dim, int tb, int pn, int ent, int n_in, int n_src) {
  ResLds L;
  L.off_x = al32(pn * dim * tb);
  L.off_res = L.off_x + al32(pn * dim * tb);
  L.off_in = L.off_res + al32(dim * ent * tb);
  L.off_oe = L.off_in + al32(n_src * dim * tb);
  L.off_os = L.off_oe + al32(n_in * 4);
  L.off_ip = L.off_os + al32(n_in * 2);
  L.off_red = L.off_ip + al32(n_in * 2);
  L.total = L.off_red + (3 * 16 + 4) * 8;
  return L;
}

template <typename T>
struct ResArgs {
  const PatchInfo *patches;
  const uint32_t *erec_s;
  int emax;
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
  ResPcg<T> s;
};

// Sum of the entry run [b0, b1) (multiples of 4) in a fixed order.
template <typename T>
__device__ __forceinline__ T run_sum(const T *s_res, int b0, int b1) {
  using V4 = typename Vec4<T>::type;
  const V4 *rp = reinterpret_cast<const V4 *>(s_res) + (b0 >> 2);
  T s0 = T(0), s1 = T(0), s2 = T(0), s3 = T(0);
  const int n4 = (b1 - b0) >> 2;
  for (int m = n4 >> 1; m > 0; --m, rp += 2) {
    const V4 u = rp[0], v = rp[1];
    s0 += Vec4<T>::get(u, 0) + Vec4<T>::get(v, 0);
    s1 += Vec4<T>::get(u, 1) + Vec4<T>::get(v, 1);
    s2 += Vec4<T>::get(u, 2) + Vec4<T>::get(v, 2);
    s3 += Vec4<T>::get(u, 3) + Vec4<T>::get(v, 3);
  }
  if (n4 & 1) {
    const V4 u = rp[0];
    s0 += Vec4<T>::get(u, 0);
    s1 += Vec4<T>::get(u, 1);
    s2 += Vec4<T>::get(u, 2);
    s3 += Vec4<T>::get(u, 3);
  }
  return (s0 + s1) + (s2 + s3);
}

// This thread's DOF (node t / DIM of the patch, component t % DIM) of K x by
// one thread per element and per DOF: patch_common.h's assemble with every
// component's entries in LDS at once, one barrier instead of 2 DIM - 1.
template <typename T, int DIM>
__device__ __forceinline__ T assemble_dof(const T *s_c, const T *s_x, T *s_res, int ent, uint3 rec,
                                          T esc, int n_elem, T lam, T mu, int b0, int b1) {
  constexpr int NPE = DIM + 1, NDE = DIM * NPE;
  if (int(threadIdx.x) < n_elem) {
    int l[4], q[4];
    decode_rec(rec, l, q);
    T X[NDE], U[NDE], F[NDE];
#pragma unroll
    for (int n = 0; n < NPE; ++n)
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        X[n * DIM + c] = s_c[l[n] * DIM + c];
        U[n * DIM + c] = s_x[l[n] * DIM + c];
      }
    (void)elem_force_free<T, DIM>(X, U, lam, mu, esc, F);
#pragma unroll
    for (int c = 0; c < DIM; ++c)
#pragma unroll
      for (int n = 0; n < NPE; ++n) s_res[c * ent + q[n]] = F[n * DIM + c];
  }
  __syncthreads();
  return run_sum<T>(s_res + (int(threadIdx.x) % DIM) * ent, b0, b1);
}

template <typename T, int DIM, int PT>
__global__ __launch_bounds__(PT) void k_pcg_resident(ResArgs<T> a) {
  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ int s_flag;
  const int b = blockIdx.x;
  const int pid = (b & 7) * a.p8 + (b >> 3);
  if (pid >= a.np) return;
  const bool alone = a.np == 1;  // no exchange
  const ResLds L = res_lds(DIM, int(sizeof(T)), a.pn, a.ent, a.n_in_max, a.n_src_max);
  T *s_c = reinterpret_cast<T *>(lds);
  T *s_x = reinterpret_cast<T *>(lds + L.off_x);
  T *s_res = reinterpret_cast<T *>(lds + L.off_res);
  T *s_in = reinterpret_cast<T *>(lds + L.off_in);
  uint32_t *s_oe = reinterpret_cast<uint32_t *>(lds + L.off_oe);
  uint16_t *s_os = reinterpret_cast<uint16_t *>(lds + L.off_os);
  uint16_t *s_ip = reinterpret_cast<uint16_t *>(lds + L.off_ip);
  double *s_red = reinterpret_cast<double *>(lds + L.off_red);  // p'q; r'z and r'r
  double *s_bc = s_red + 48;
  const int t = threadIdx.x;
  if (t == 0) s_flag = 0;

  // the patch, this thread's element and DOF (node k, component c)
  const PatchInfo P = a.patches[pid];
  const ExchangePatch E = a.xpatch[pid];
  const size_t pbase = size_t(pid) * a.pstride;
  const int k = t / DIM, c = t - k * DIM;
  const bool has = k < P.n_own + P.n_sh;
  const bool own = k < P.n_own;
  const uint3 rec = reinterpret_cast<const uint3 *>(
      a.erec_s)[size_t(pid) * unsigned(a.emax) + unsigned(min(t, a.emax - 1))];
  const T esc = a.escale && t < P.n_elem ? a.escale[P.elem_start + t] : T(1);
  clear_entries<T, PT>(s_res, DIM * a.ent);
  int go = 0, b0 = 0, b1 = 0, l0 = 0, l1 = 0, lo = 0;
  bool first = own, fixed = false;  // first: this patch accounts for the node
  T r = T(0), p = T(0), x = T(0), d = T(0);
  if (has) {
    const int gid = a.pgid[pbase + k];
    go = gid * DIM + c;
    b1 = int(a.pend[pbase + k]);
    b0 = k ? int(a.pend[pbase + k - 1]) : 0;
    fixed = ((a.fixmask[gid] >> c) & 1) != 0;
    if (!own) {
      const int j = P.sh_start + k - P.n_own;
      first = a.pslot[pbase + k] < 0;
      l1 = int(a.src_end[j]);
      l0 = k > P.n_own ? int(a.src_end[j - 1]) : 0;
      lo = int(a.own_pos[j]);
    }
    s_c[t] = a.coords[go];
    r = a.s.r_in[go];
    d = a.s.invD[go];
    if (!a.s.fresh) {
      p = a.s.p[go];
      x = a.s.x[go];
    }
  }
  // the operator's diagonal of a constrained row, its mass shift
  const T dK = fixed && first ? a.diagK[go] : T(0);
  const T cK = a.s.sh.cK, cMm = has && a.s.sh.m ? a.s.sh.cM * a.s.sh.m[go] : T(0);
  for (int i = t; i < E.n_in; i += PT) {
    s_oe[i] = a.out_entry[E.out_start + i];
    s_os[i] = a.out_src[E.out_start + i];
    s_ip[i] = a.in_pos[E.out_start + i];
  }
  const int xc = t >> 8, xi = t & 255;  // entries xi, xi + 256, ... of component xc
  // (workgroup 0 advances the epoch at its end, after an exchange that every
  // workgroup took part in with the tag it reads here)
  u64 *const epoch = a.s.words;
  const size_t stride = res_copy_words(a.np);
  const Exchange xpq{a.s.words + RES_HEAD, stride, epoch + 1, a.np, b % EX_COPIES};
  const Exchange xrz{xpq.words + size_t(2) * a.np, stride, epoch + 1, a.np, b % EX_COPIES};
  unsigned tag = unsigned(ld_agent(epoch));

  // r'z and r'r over all patches
  double g = 0.0, q2 = 0.0;
  auto dots = [&]() -> bool {
    double v[2] = {0.0, 0.0};
    if (first) {
      v[0] = double(r) * double(mul_rn(d, r));
      v[1] = double(r) * double(r);
    }
    sum_to_wave0<PT, 2>(v, s_red + 16);
    ++tag;
    if (!alone && t < 64) publish<2>(xrz, pid, tag, v);
    const bool ok = gather<2>(xrz, tag, v, s_bc, &s_flag, alone);
    g = v[0];
    q2 = v[1];
    return ok;
  };

  bool alive = dots();
  double g_prev = a.s.fresh ? 1.0 : a.s.g_prev;
  const double gamma0 = a.s.fresh ? g : a.s.gamma0, rr0 = a.s.fresh ? q2 : a.s.rr0;
  const double pause = a.s.fresh ? a.s.pause * q2 : a.s.pause;
  const double thresh = !a.s.fresh ? a.s.thresh : a.s.kind == 0 ? a.s.eps * g : a.s.eps * a.s.eps * q2;
  int n_upd = a.s.it0;
  int done = RES_ABORTED;
  while (alive) {
    int stop = 0;
    if (n_upd >= 1) {
      if (a.s.kind == 0 ? g < thresh : q2 <= thresh) stop = 1;
    } else if (q2 == 0.0) {
      stop = 1;
    }
    if (!stop && !isfinite(g)) stop = 2;
    if (!stop && n_upd >= a.s.max_iter) stop = 4;
    // (looked at every eighth iteration: r'r is not monotone, and a replacement
    // at a single dip can cost directions -- a 160 x 80-class plate under body
    // force took 3225 iterations with a look at every one, 1953 so, 1950 in the
    // launch-per-kernel form)
    if (!stop && (n_upd & 7) == 0 && q2 < pause) stop = 5;
    if (!stop && n_upd - a.s.it0 >= a.s.cap) stop = RES_CAP;
    if (stop) {
      done = stop;
      break;
    }
    const T beta = T(g / g_prev);
    g_prev = g;
    if (has) {
      p = pcg_dir(d, r, beta, p);
      s_x[t] = fixed ? T(0) : p;
    }
    __syncthreads();
    T q = assemble_dof<T, DIM>(s_c, s_x, s_res, a.ent, rec, esc, P.n_elem, a.lam, a.mu, b0, b1);
    // the row of a constrained DOF: the assembled diagonal only; the mass
    // shift belongs to the patch that accounts for the node
    if (fixed) q = dK * p;
    q = cK * q;
    double vpq[1] = {0.0};
    if (has) {
      if (own) q += cMm * p;
      vpq[0] = double(p) * double(q);
      if (!own) {
        s_in[lo * DIM + c] = q;
        if (first) vpq[0] += double(cMm) * double(p) * double(p);
      }
    }
    ++tag;
    sum_to_wave0<PT, 1>(vpq, s_red);
    if (!alone) {
      if (t < 64) publish<1>(xpq, pid, tag, vpq);
      if (xc < DIM) {
        for (int i = xi; i < E.n_in; i += 256)
          send_entry<T, DIM>(a.s.entries, s_oe[i], xc, tag, s_in[int(s_os[i]) * DIM + xc]);
        if (!recv_entries<T, DIM>(a.s.entries, unsigned(E.in_start), xi, E.n_in, xc, tag, epoch + 1,
                                  s_in, s_ip))
          s_flag = 1;
      }
    }
    alive = gather<1>(xpq, tag, vpq, s_bc + 2, &s_flag, alone);
    if (!alive) break;
    const double pq = vpq[0], alpha_d = g / pq;
    if (!(pq > 0.0) || !isfinite(alpha_d)) {
      // no x or r has changed: the state of the last completed iteration
      done = isfinite(pq) ? 3 : 2;
      break;
    }
    const T alpha = T(alpha_d);
    if (has) {
      if (!own) {
        // the DOF's contributions from all its patches, in slot order
        q = T(0);
        for (int l = l0; l < l1; ++l) q += s_in[l * DIM + c];
        q += cMm * p;
      }
      x = x + alpha * p;
      r = r - alpha * q;
    }
    alive = dots();
    ++n_upd;
  }
  if (first) {
    a.s.x[go] = x;
    a.s.p[go] = p;
    a.s.r_out[go] = r;
  }
  if (pid == 0 && t == 0) {
    CgScalars *sc = a.s.sc;
    sc->gamma0 = gamma0;
    sc->rr0 = rr0;
    sc->thresh = thresh;
    sc->g[0] = sc->g[1] = g_prev;
    sc->g_final = g;
    sc->rr_final = q2;
    sc->iter_final = n_upd;
    sc->pause = pause;
    st_agent(epoch, u64(tag));
    if (ld_agent(epoch + 1) != 0) done = RES_ABORTED;
    sc->done = done;
  }
}

template <typename T>
ResArgs<T> res_args(const DevMesh &dm, const ResPcg<T> &s) {
  ResArgs<T> a{};
  a.patches = dm.patches;
  a.erec_s = dm.erec_s;
  a.emax = dm.emax;
  a.pgid = dm.pgid;
  a.pslot = dm.pslot;
  a.pend = dm.pend;
  a.pstride = dm.patch_threads;
  a.fixmask = dm.fixmask;
  if constexpr (sizeof(T) == 8) {
    a.coords = reinterpret_cast<const T *>(dm.coords64);
    a.escale = reinterpret_cast<const T *>(dm.escale64);
    a.diagK = reinterpret_cast<const T *>(dm.diag64);
  } else {
    a.coords = reinterpret_cast<const T *>(dm.coords32);
    a.escale = reinterpret_cast<const T *>(dm.escale32);
    a.diagK = reinterpret_cast<const T *>(dm.diag32);
  }
  a.lam = T(dm.lam);
  a.mu = T(dm.mu);
  a.np = dm.np;
  a.p8 = (dm.np + 7) / 8;
  a.ent = dm.ent;
  a.pn = dm.pn;
  a.xpatch = dm.xpatch;
  a.out_entry = dm.x_out_entry;
  a.out_src = dm.x_out_src;
  a.in_pos = dm.x_in_pos;
  a.src_end = dm.x_src_end;
  a.own_pos = dm.x_own_pos;
  a.n_in_max = dm.x_in_max;
  a.n_src_max = dm.x_src_max;
  a.s = s;
  return a;
}

// One thread per element and per DOF: patches of up to 256 nodes and 768
// elements.
constexpr int RES_NODES = 256, RES_ELEMS = 768;

template <typename T>
using PcgKernel = void (*)(ResArgs<T>);

// 2D patches mostly run into the node limit first: 512 threads hold them.
int res_threads(const DevMesh &dm) { return dm.dim == 2 && dm.emax <= 512 ? 512 : 768; }

template <typename T>
PcgKernel<T> pcg_kernel(const DevMesh &dm) {
  if (dm.dim == 3) return k_pcg_resident<T, 3, 768>;
  return res_threads(dm) == 512 ? PcgKernel<T>(k_pcg_resident<T, 2, 512>)
                                : PcgKernel<T>(k_pcg_resident<T, 2, 768>);
}

// Workgroups of a kernel that a compute unit holds, and the device's units
// (asked of the runtime once per kernel and LDS size).
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

int res_lds_bytes(const DevMesh &dm, int tb) {
  return res_lds(dm.dim, tb, dm.pn, dm.ent, dm.x_in_max, dm.x_src_max).total;
}

constexpr int RES_LDS_MAX = 160 * 1024 - 256;

}  // namespace

template <typename T>
bool res_pcg_fit(const DevMesh &dm, int device, ResFit *fit) {
  const int lds = res_lds_bytes(dm, int(sizeof(T))), cu = compute_units(device);
  if (!dm.xpatch || cu < 1 || dm.pn > RES_NODES || dm.emax > RES_ELEMS || lds > RES_LDS_MAX)
    return false;
  const int per = blocks_per_cu(reinterpret_cast<const void *>(pcg_kernel<T>(dm)), res_threads(dm), lds);
  const int grid = 8 * ((dm.np + 7) / 8);
  if (per < 1 || grid > cu) return false;
  fit->block = 1.0 / per;
  fit->share = double(grid) / (double(per) * cu);
  return true;
}

template <typename T>
void launch_res_pcg(const DevMesh &dm, const ResPcg<T> &s, hipStream_t st) {
  const ResArgs<T> a = res_args<T>(dm, s);
  hipLaunchKernelGGL(pcg_kernel<T>(dm), dim3(8 * a.p8), dim3(res_threads(dm)),
                     res_lds_bytes(dm, int(sizeof(T))), st, a);
}

hipError_t prepare_resident_kernels() {
  hipError_t e = hipSuccess, r;
  for (const void *f : {reinterpret_cast<const void *>(&k_pcg_resident<double, 3, 768>),
                        reinterpret_cast<const void *>(&k_pcg_resident<double, 2, 768>),
                        reinterpret_cast<const void *>(&k_pcg_resident<double, 2, 512>),
                        reinterpret_cast<const void *>(&k_pcg_resident<float, 3, 768>),
                        reinterpret_cast<const void *>(&k_pcg_resident<float, 2, 768>),
                        reinterpret_cast<const void *>(&k_pcg_resident<float, 2, 512>)})
    if ((r = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, RES_LDS_MAX)) != hipSuccess)
      e = r;
  return e;
}

#define FEMGPU_RES_INST(T)                                              \
  template bool res_pcg_fit<T>(const DevMesh &, int, ResFit *);         \
  template void launch_res_pcg<T>(const DevMesh &, const ResPcg<T> &, hipStream_t);
FEMGPU_RES_INST(double)
FEMGPU_RES_INST(float)

}  // namespace femgpu
