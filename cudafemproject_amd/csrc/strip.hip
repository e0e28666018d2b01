// strip.hip -- y = K x and the patch half of a PCG iteration (k_ebe_patch MODE 0
// and 1, kernels.hip), a strip of up to three elements per thread.
//
// What bounds the element-wise kernel is LDS traffic: per tetrahedron in FP64
// 192 bytes of corner data read, 96 written into the entry list and read back
// for the node sums, all at scattered addresses.  Three tetrahedra in a strip
// (StripPlan) have 6 nodes instead of 12 corners: corner data is read once per
// strip node, the forces of a node's elements within the strip are added in
// registers, and the entry list has half as many entries.  Measured on the 64^3-hex
// cube, element by element -> strips (the PCG step with its loads reordered):
// FP64 matvec patch kernel 22.1 -> 18.1 us, PCG step 28.6 -> 23.6 us; FP32 PCG
// step 16.2 -> 14.5 us.  Of a workgroup's 18 kcycles (2.4 GHz) some 9 are now
// the node and partial loads, 3 to 5 the strips, 3 the node sums.
//
// The user-order product reads x and writes y through the patch's node ids, in
// two launches instead of four: 36.8 -> 23.5 us.
#include <hip/hip_runtime.h>

#include <cmath>

#include "element.h"
#include "patch_common.h"
#include "strip.h"

namespace femgpu {

namespace {

using namespace elem;
using namespace patch;

enum { MATVEC = 0, PCG = 1, USER = 2 };

template <typename T>
struct StripArgs {
  const PatchInfo *patches;
  const uint4 *rec;
  const uint32_t *rec2;
  const uint16_t *pend;
  const int32_t *pgid, *pslot, *puser;
  int stride, nstride;       // of rec, rec2; of pend, pgid, pslot, puser
  const uint8_t *fixmask;
  const T *coords, *diagK;
  const T *escale;           // per strip element k at (pid * 3 + k) * stride, or null
  T lam, mu;
  int np, p8, ent, pn;
  const T *x;                // MATVEC: x
  T *y;
  const double *xu;          // USER: x and y in user order
  double *yu;
  StripPcg<T> s;             // PCG
  T *partial;
};

// Sum over the workgroup in every thread; sh: blockDim / 64 doubles that no
// thread still reads or writes.
__device__ __forceinline__ double block_sum_n(double v, double *sh) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = 0.0;
  for (unsigned i = 0; i < blockDim.x >> 6; ++i) r += sh[i];
  return r;
}

// Waves per SIMD asked of the register allocator: FP64 fits 128 registers, four
// workgroups of 256 threads per CU (96 spill: 34.9 -> 43.9 us per iteration of
// the 64^3 cube), FP32 64.
template <typename T, int DIM, int MODE>
__global__ __launch_bounds__(STRIP_THREADS_MAX)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 ? 4 : 8))) void k_strip(StripArgs<T> a) {
  constexpr unsigned FMASK = (1u << DIM) - 1u;
  constexpr int NS = DIM + STRIP_ELEMS;  // nodes of a full strip
  extern __shared__ __align__(16) unsigned char lds[];
  const int b = blockIdx.x;
  // (XCD-aware, as k_ebe_patch: neighbouring patches share an XCD's L2)
  const int pid = (b & 7) * a.p8 + (b >> 3);
  if (pid >= a.np) return;
  const LdsLayout L = lds_layout(DIM, int(sizeof(T)), a.pn, a.ent);
  T *s_c = reinterpret_cast<T *>(lds + L.off_c);
  T *s_x = reinterpret_cast<T *>(lds + L.off_x);      // constrained components zeroed
  T *s_res = reinterpret_cast<T *>(lds + L.off_res);  // one component of the entries
  double *s_red = reinterpret_cast<double *>(lds + L.off_red);
  const int t = threadIdx.x;

  // Loads first, in the order of their use: the scalars and partial sums that
  // beta comes from are on their way together with the node data, which does
  // not wait for them (formed first, beta took 6 of a workgroup's 22 kcycles).
  const size_t nbase = size_t(pid) * a.nstride;
  int gid = 0, b1 = 0, b0 = 0, slot = 0, uo = 0;
  if (t < a.pn) {
    gid = a.pgid[nbase + t];
    slot = a.pslot[nbase + t];
    if constexpr (MODE == USER) uo = a.puser[nbase + t] * DIM;
    b1 = int(a.pend[nbase + t]);
    b0 = t ? int(a.pend[nbase + t - 1]) : 0;
  }
  const PatchInfo P = a.patches[pid];
  constexpr int NL = NODE_PARTS / 64;
  double gv[NL], qv[NL], thresh = 0.0, g_prev = 1.0, x_pend = 0.0;
  int done = 0, kind = 0, n_upd = 0, max_iter = 0;
  if constexpr (MODE == PCG) {
    const CgScalars *sc = a.s.sc;
    done = sc->done;
    kind = sc->kind;
    n_upd = sc->it[a.s.parity ^ 1] + 1;
    max_iter = sc->max_iter;
    thresh = sc->thresh;
    g_prev = sc->g[a.s.parity ^ 1];
    x_pend = sc->x_pend;
    if (t < 64)
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        gv[j] = a.s.prz[t + 64 * j];
        qv[j] = a.s.prr[t + 64 * j];
      }
  }
  const uint4 rec = a.rec[size_t(pid) * a.stride + t];
  const uint32_t rec2 = a.rec2[size_t(pid) * a.stride + t];
  const bool has_node = t < P.n_own + P.n_sh, own = t < P.n_own;
  const bool first = own || slot < 0;
  const int go = gid * DIM;
  T xin[DIM], co[DIM], rv[DIM], dv[DIM];
  unsigned fm = 0;
  if (has_node) {
    fm = a.fixmask[gid] & FMASK;
#pragma unroll
    for (int c = 0; c < DIM; ++c) co[c] = a.coords[go + c];
    if constexpr (MODE == PCG) {
#pragma unroll
      for (int c = 0; c < DIM; ++c) xin[c] = a.s.p[go + c];
#pragma unroll
      for (int c = 0; c < DIM; ++c) rv[c] = a.s.r[go + c];
#pragma unroll
      for (int c = 0; c < DIM; ++c) dv[c] = a.s.invD[go + c];
    } else {
#pragma unroll
      for (int c = 0; c < DIM; ++c) xin[c] = MODE == USER ? T(a.xu[uo + c]) : a.x[go + c];
    }
  }
  {
    using V4 = typename Vec4<T>::type;
    V4 *r4 = reinterpret_cast<V4 *>(s_res);
    for (int i = t; i < (a.ent >> 2); i += int(blockDim.x)) r4[i] = Vec4<T>::zero();
  }
  T beta = T(0);
  if constexpr (MODE == PCG) {
    // the stop test and beta (k_ebe_patch MODE 1): wave 0 sums the partials
    if (t < 64) {
      double g = 0.0, q = 0.0;
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        g += gv[j];
        q += qv[j];
      }
      g = wave_sum(g);
      q = wave_sum(q);
      if (t == 0) {
        s_red[0] = g;
        s_red[1] = q;
      }
    }
    lds_barrier();
    const double g = s_red[0], q = s_red[1];
    if (done) return;
    int stop = 0;
    if (n_upd >= 1) {
      if (kind == 0 ? (g < thresh) : (q <= thresh)) stop = 1;
    } else if (q == 0.0) {
      stop = 1;
    }
    if (!stop && !isfinite(g)) stop = 2;
    if (!stop && n_upd >= max_iter) stop = 4;
    const double bt = g / g_prev;
    if (pid == 0 && t == 0) {
      CgScalars *sc = a.s.sc;
      sc->g_final = g;
      sc->rr_final = q;
      sc->iter_final = n_upd;
      if (stop) {
        sc->done = stop;
        sc->par_final = a.s.parity;
      } else {
        sc->g[a.s.parity] = g;
        sc->b[a.s.parity] = bt;
        sc->it[a.s.parity] = n_upd;
      }
    }
    if (stop) return;
    beta = T(bt);
  }
  if (has_node) {
#pragma unroll
    for (int c = 0; c < DIM; ++c) s_c[t * DIM + c] = co[c];
    if constexpr (MODE == PCG) {
      // (FP64: the previous update's x += alpha p, as in k_ebe_patch)
      if (sizeof(T) == 8 && first) {
        const T xstep = T(x_pend);
#pragma unroll
        for (int c = 0; c < DIM; ++c) a.s.x[go + c] += xstep * xin[c];
      }
#pragma unroll
      for (int c = 0; c < DIM; ++c) xin[c] = pcg_dir(dv[c], rv[c], beta, xin[c]);
      if (own) {
#pragma unroll
        for (int c = 0; c < DIM; ++c) a.s.p[go + c] = xin[c];
      }
    }
#pragma unroll
    for (int c = 0; c < DIM; ++c) s_x[t * DIM + c] = ((fm >> c) & 1u) ? T(0) : xin[c];
  }
  lds_barrier();

  // The strip's elements: element k has its nodes k .. k + DIM.
  const int count = int(rec.x >> 30);
  T F[NS * DIM];
  if (count) {
    T X[NS * DIM], U[NS * DIM];
    auto load = [&](int n) {
      const unsigned l = strip_node(rec, n) * unsigned(DIM);
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        X[n * DIM + c] = s_c[l + c];
        U[n * DIM + c] = s_x[l + c];
      }
    };
#pragma unroll
    for (int n = 0; n < DIM; ++n) load(n);
    const T *esc = a.escale ? a.escale + size_t(pid) * 3 * unsigned(a.stride) + t : nullptr;
#pragma unroll
    for (int k = 0; k < STRIP_ELEMS; ++k) {
#pragma unroll
      for (int c = 0; c < DIM; ++c) F[(k + DIM) * DIM + c] = T(0);
      if (k < count) {
        load(k + DIM);
        T f[(DIM + 1) * DIM];
        (void)elem_force_free<T, DIM>(X + k * DIM, U + k * DIM, a.lam, a.mu,
                                      esc ? esc[k * a.stride] : T(1), f);
#pragma unroll
        for (int i = 0; i < (DIM + 1) * DIM; ++i)
          F[k * DIM + i] = k == 0 || i >= DIM * DIM ? f[i] : F[k * DIM + i] + f[i];
      }
    }
  }
  T acc[DIM];
#pragma unroll
  for (int c = 0; c < DIM; ++c) {
    if (c) lds_barrier();
    if (count) {
#pragma unroll
      for (int n = 0; n < NS; ++n)
        if (n <= DIM || n < count + DIM) s_res[strip_entry(rec, rec2, n)] = F[n * DIM + c];
    }
    lds_barrier();
    using V4 = typename Vec4<T>::type;
    const V4 *rp = reinterpret_cast<const V4 *>(s_res) + (b0 >> 2);
    T s0 = T(0), s1 = T(0), s2 = T(0), s3 = T(0);
    for (int m = (b1 - b0) >> 2; m > 0; --m, ++rp) {
      const V4 u = rp[0];
      s0 += Vec4<T>::get(u, 0);
      s1 += Vec4<T>::get(u, 1);
      s2 += Vec4<T>::get(u, 2);
      s3 += Vec4<T>::get(u, 3);
    }
    acc[c] = (s0 + s1) + (s2 + s3);
  }

  // Rows of constrained components: the assembled diagonal, by the node's first
  // patch (k_ebe_patch).
  double en = 0.0;
  if (has_node) {
    const unsigned so = unsigned(slot & 0x7fffffff) * unsigned(DIM);
#pragma unroll
    for (int c = 0; c < DIM; ++c) xin[c] = MODE == PCG ? s_x[t * DIM + c] : T(0);
    if (fm)
#pragma unroll
      for (int c = 0; c < DIM; ++c)
        if ((fm >> c) & 1u) {
          if constexpr (MODE == MATVEC)
            xin[c] = a.x[go + c];
          else if constexpr (MODE == USER)
            xin[c] = T(a.xu[uo + c]);
          else
            xin[c] = own ? a.s.p[go + c] : pcg_dir(a.s.invD[go + c], a.s.r[go + c], beta, a.s.p[go + c]);
          acc[c] = first ? a.diagK[go + c] * xin[c] : T(0);
        }
    if constexpr (MODE == PCG) {
      const T *m = a.s.sh.m;
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        T v = a.s.sh.cK * acc[c];
        if (m && own) v += a.s.sh.cM * m[go + c] * xin[c];
        en += double(xin[c]) * double(v);
        // (an interface node's mass term: once)
        if (m && !own && first) en += double(a.s.sh.cM) * double(m[go + c]) * double(xin[c]) * double(xin[c]);
        acc[c] = v;
      }
    }
    if (own) {
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        if constexpr (MODE == USER)
          a.yu[uo + c] = double(acc[c]);
        else
          a.y[go + c] = acc[c];
      }
    } else {
#pragma unroll
      for (int c = 0; c < DIM; ++c) a.partial[so + c] = acc[c];
    }
  }
  if constexpr (MODE == PCG) {
    const double tot = block_sum_n(en, s_red + 16);
    if (t == 0) a.s.part[pid] = tot;
  }
}

template <typename T>
StripArgs<T> strip_args(const DevMesh &dm) {
  StripArgs<T> a{};
  a.patches = dm.patches;
  a.rec = dm.strip_rec;
  a.rec2 = dm.strip_rec2;
  a.pend = dm.strip_pend;
  a.pgid = dm.pgid;
  a.pslot = dm.pslot;
  a.puser = dm.puser;
  a.stride = dm.strip_stride;
  a.nstride = dm.patch_threads;
  a.fixmask = dm.fixmask;
  if constexpr (sizeof(T) == 8) {
    a.coords = dm.coords64;
    a.diagK = dm.diag64;
    a.escale = dm.strip_escale64;
  } else {
    a.coords = dm.coords32;
    a.diagK = dm.diag32;
    a.escale = dm.strip_escale32;
  }
  a.lam = T(dm.lam);
  a.mu = T(dm.mu);
  a.np = dm.np;
  a.p8 = (dm.np + 7) / 8;
  a.ent = dm.strip_ent;
  a.pn = dm.pn;
  return a;
}

template <typename T, int MODE>
void launch(const DevMesh &dm, const StripArgs<T> &a, hipStream_t s) {
  const LdsLayout L = lds_layout(dm.dim, int(sizeof(T)), a.pn, a.ent);
  if (dm.dim == 3)
    hipLaunchKernelGGL((k_strip<T, 3, MODE>), dim3(8 * a.p8), dim3(dm.strip_threads), L.total, s, a);
  else
    hipLaunchKernelGGL((k_strip<T, 2, MODE>), dim3(8 * a.p8), dim3(dm.strip_threads), L.total, s, a);
}

}  // namespace

template <typename T>
void launch_strip_matvec(const DevMesh &dm, const T *x, T *y, T *partial, hipStream_t s) {
  StripArgs<T> a = strip_args<T>(dm);
  a.x = x;
  a.y = y;
  a.partial = partial;
  launch<T, MATVEC>(dm, a, s);
}

template <typename T>
void launch_strip_matvec_user(const DevMesh &dm, const double *x, double *y, T *partial,
                              hipStream_t s) {
  StripArgs<T> a = strip_args<T>(dm);
  a.xu = x;
  a.yu = y;
  a.partial = partial;
  launch<T, USER>(dm, a, s);
}

template <typename T>
void launch_strip_pcg(const DevMesh &dm, const StripPcg<T> &p, hipStream_t s) {
  StripArgs<T> a = strip_args<T>(dm);
  a.s = p;
  a.y = p.q;
  a.partial = p.partial;
  launch<T, PCG>(dm, a, s);
}

hipError_t prepare_strip_kernels() {
  hipError_t e = hipSuccess, r;
#define FEMGPU_STRIP_ATTR(T, D, M)                                                          \
  if ((r = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_strip<T, D, M>),           \
                               hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024)) !=  \
      hipSuccess)                                                                           \
    e = r;
#define FEMGPU_STRIP_ATTRS(T, D) FEMGPU_STRIP_ATTR(T, D, 0) FEMGPU_STRIP_ATTR(T, D, 1) FEMGPU_STRIP_ATTR(T, D, 2)
  FEMGPU_STRIP_ATTRS(double, 3)
  FEMGPU_STRIP_ATTRS(double, 2)
  FEMGPU_STRIP_ATTRS(float, 3)
  FEMGPU_STRIP_ATTRS(float, 2)
#undef FEMGPU_STRIP_ATTRS
#undef FEMGPU_STRIP_ATTR
  return e;
}

#define FEMGPU_STRIP_INST(T)                                                                       \
  template void launch_strip_matvec<T>(const DevMesh &, const T *, T *, T *, hipStream_t);         \
  template void launch_strip_matvec_user<T>(const DevMesh &, const double *, double *, T *,        \
                                            hipStream_t);                                          \
  template void launch_strip_pcg<T>(const DevMesh &, const StripPcg<T> &, hipStream_t);
FEMGPU_STRIP_INST(double)
FEMGPU_STRIP_INST(float)

}  // namespace femgpu
