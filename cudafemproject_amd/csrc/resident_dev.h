// resident_dev.h -- device pieces of the kernels whose workgroups stay on the
// chip and exchange through memory while they run (resident.hip,
// batch_res.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <climits>

#include "element.h"
#include "patch_common.h"
#include "resident.h"

namespace femgpu {
namespace resident {

using namespace elem;
using namespace patch;

using u64 = unsigned long long;

constexpr int WAIT_TICKS = 100000000;  // one second of the 100 MHz clock

__device__ __forceinline__ void st_agent(u64 *p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 ld_agent(const u64 *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// A double as two tagged words, and back.
__device__ __forceinline__ void tag_words(double v, unsigned tag, u64 (&w)[2]) {
  const u64 b = static_cast<u64>(__double_as_longlong(v));
  w[0] = (u64(tag) << 32) | (b & 0xffffffffull);
  w[1] = (u64(tag) << 32) | (b >> 32);
}
__device__ __forceinline__ double untag(const u64 (&w)[2]) {
  return __longlong_as_double(static_cast<long long>((w[1] << 32) | (w[0] & 0xffffffffull)));
}

// A bounded wait: true once the caller should give up (another workgroup
// did, or WAIT_TICKS -- or what the host put beside the abort word -- have
// passed since the 256th look).  (Times in 32 bits, 42 s round: the wait loops
// stand where registers are short.)
struct Patience {
  u64 *abort;
  unsigned start = 0;
  __device__ __forceinline__ bool over(int spin) {
    if ((spin & 255) != 255) return false;
    const unsigned now = unsigned(wall_clock64());
    if (start == 0) start = now | 1u;
    return expired(abort, int(now - start));
  }
  static __device__ __forceinline__ bool expired(u64 *abort, int waited) {
    const int limit = int(ld_agent(abort + 1));
    if (ld_agent(abort) == 0 && waited <= (limit ? limit : WAIT_TICKS)) return false;
    st_agent(abort, 1);
    return true;
  }
};

// The same in a launch whose workgroups take tickets: the bound runs from the
// last sign of progress of any workgroup (its time, in abort[3]).  The peers waited
// for may still be busy with earlier instances, which may take long, but ends.
struct QueuePatience {
  u64 *abort;
  unsigned start = 0;
  __device__ __forceinline__ bool over(int spin) {
    if ((spin & 255) != 255) return false;
    const unsigned now = unsigned(wall_clock64());
    if (start == 0) start = now | 1u;
    const unsigned sign = unsigned(ld_agent(abort + 3));
    return Patience::expired(abort, min(int(now - start), sign ? int(now - sign) : INT_MAX));
  }
};

// Interface sums travel as entries (femgpu_internal.h): the bits of DIM values
// in words of 48 under a 16-bit tag (a third fewer words than 32 under 32;
// the traffic of some hundred kilobytes a step per workgroup is what bounds a
// trade).  The tag counts the trades through a set of entries, and every trade
// writes them all: a stale word carries the tag before the one awaited.  Word
// w of 64 consecutive entries lie together.
template <typename T, int DIM>
constexpr int EW = res_entry_size(DIM, int(sizeof(T)));

template <typename T, int DIM>
__device__ __forceinline__ size_t entry_word(unsigned e, int w) {
  return (size_t(e >> 6) * EW<T, DIM> + w) * 64 + (e & 63u);
}

template <typename T>
__device__ __forceinline__ void to_bits(T v, unsigned *u) {
  if constexpr (sizeof(T) == 8) {
    const u64 b = static_cast<u64>(__double_as_longlong(v));
    u[0] = unsigned(b);
    u[1] = unsigned(b >> 32);
  } else {
    u[0] = __float_as_uint(v);
  }
}
template <typename T>
__device__ __forceinline__ T from_bits(const unsigned *u) {
  if constexpr (sizeof(T) == 8)
    return __longlong_as_double(static_cast<long long>((u64(u[1]) << 32) | u[0]));
  else
    return __uint_as_float(u[0]);
}

template <typename T, int DIM>
__device__ __forceinline__ void send_entry(u64 *entries, unsigned e, unsigned tag, const T *v) {
  constexpr int W = EW<T, DIM>, U = sizeof(T) / 4;
  unsigned u[DIM * U + 2];
#pragma unroll
  for (int c = 0; c < DIM; ++c) to_bits<T>(v[c], &u[c * U]);
  u[DIM * U] = u[DIM * U + 1] = 0u;
  // 16-bit unit j of the payload: half j & 1 of u[j >> 1]
  auto unit = [&](int j) { return j >= 2 * DIM * U ? 0u : (j & 1) ? u[j >> 1] >> 16 : u[j >> 1] & 0xffffu; };
#pragma unroll
  for (int w = 0; w < W; ++w)
    st_agent(&entries[entry_word<T, DIM>(e, w)],
             (u64((tag << 16) | unit(3 * w + 2)) << 32) | (unit(3 * w + 1) << 16) | unit(3 * w));
}

// Entry e into v; false when the wait ran out.
template <typename T, int DIM, typename Wait>
__device__ __forceinline__ bool recv_entry(const u64 *entries, unsigned e, unsigned tag, Wait wait,
                                           T *v) {
  constexpr int W = EW<T, DIM>, U = sizeof(T) / 4;
  u64 h[W];
  for (int spin = 0;; ++spin) {
    bool all = true;
#pragma unroll
    for (int w = 0; w < W; ++w) h[w] = ld_agent(&entries[entry_word<T, DIM>(e, w)]);
#pragma unroll
    for (int w = 0; w < W; ++w) all = all && unsigned(h[w] >> 48) == (tag & 0xffffu);
    if (all) break;
    if (wait.over(spin)) return false;
  }
  auto unit = [&](int j) { return unsigned(h[j / 3] >> (16 * (j % 3))) & 0xffffu; };
#pragma unroll
  for (int c = 0; c < DIM; ++c) {
    unsigned u[U];
#pragma unroll
    for (int i = 0; i < U; ++i) u[i] = unit(2 * (c * U + i)) | (unit(2 * (c * U + i) + 1) << 16);
    v[c] = from_bits<T>(u);
  }
  return true;
}

// The exchange words lie in EX_COPIES copies, each read by every
// EX_COPIES-th workgroup (a copy per XCD): all workgroups polling one copy
// of a few kilobytes queue up at the memory channels that hold it.
struct Exchange {
  u64 *words;      // copy 0 of this exchange: [2 * RES_SUMS][np]
  size_t stride;   // words from copy to copy
  u64 *abort;      // nonzero: a workgroup gave up waiting
  int np, copy;    // copy: the one this workgroup reads
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

// v, its value unknown to the compiler: what is computed from it is computed
// where it is used, not kept in registers through a loop that has none to spare.
template <typename V>
__device__ __forceinline__ V fresh(V v) {
  asm volatile("" : "+v"(v));
  return v;
}

// A DOF's row of its patch's part of K, kept in registers: K of an element
// annihilates translations, so row i is sum_j K_ij (u_j - u_i) over the other
// nodes j of the node's elements -- differences, as in the element-wise product
// and as accurate.  Constrained components count as zero: a neighbour's goes
// into the node's own coefficients.  Up to D neighbours, in order of first
// touch.
template <typename T, int DIM, int D>
struct PatchRow {
  static constexpr int NPE = DIM + 1;
  static constexpr unsigned NONE = 0xffffu;
  static_assert(D % 2 == 0 && D >= 6, "two offsets to a word");
  unsigned off[D / 2];  // neighbour d's byte offset in a node vector: half d & 1 of off[d >> 1]
  T k[D][DIM], self[DIM];
  unsigned zero;        // the node's own components to take as zero
  int n;                // neighbours (the most of a lane of the wave)

  // Component c of node `node`, whose entries (patch_common.h) are [b0, b1):
  // s_ent: element * 4 + corner + 1 per entry (0: padding), s_el: an element's
  // local nodes, 10 bits each, s_fix: the nodes' constrained components.  diag:
  // the row's diagonal where it is constrained.  False: more than D neighbours.
  __device__ __forceinline__ bool build(int node, int c, int b0, int b1, const uint16_t *s_ent,
                                        const uint32_t *s_el, const uint8_t *s_fix, const T *s_c,
                                        T diag, T lam, T mu) {
    unsigned id[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      id[d] = NONE;
#pragma unroll
      for (int j = 0; j < DIM; ++j) k[d][j] = T(0);
    }
#pragma unroll
    for (int j = 0; j < DIM; ++j) self[j] = T(0);
    zero = s_fix[node];
    const bool fixed = (zero >> c) & 1u;
    if (fixed) {
      zero = 0u;
#pragma unroll
      for (int j = 0; j < DIM; ++j) self[j] = j == c ? diag : T(0);
    }
    bool ok = true;
    for (int b = fixed ? b1 : b0; b < b1; ++b) {
      if (!s_ent[b]) continue;
      const int a = (int(s_ent[b]) - 1) & 3;
      const uint32_t w = s_el[(int(s_ent[b]) - 1) >> 2];
      T X[NPE * DIM], g[DIM * DIM + 1];
#pragma unroll
      for (int m = 0; m < NPE; ++m)
#pragma unroll
        for (int j = 0; j < DIM; ++j) X[m * DIM + j] = s_c[((w >> (10 * m)) & 1023u) * DIM + j];
      elem_geometry<T, DIM>(X, T(1), g);
#pragma unroll
      for (int m = 0; m < NPE; ++m) {
        if (m == a) continue;
        const unsigned nb = (w >> (10 * m)) & 1023u, fm = s_fix[nb];
        T kk[DIM];
#pragma unroll
        for (int j = 0; j < DIM; ++j) {
          T U[NPE * DIM], F[NPE * DIM];
#pragma unroll
          for (int i = 0; i < NPE * DIM; ++i) U[i] = i == m * DIM + j ? T(1) : T(0);
          (void)elem_force_geo<T, DIM>(g, U, lam, mu, F);
          kk[j] = F[0];
#pragma unroll
          for (int i = 1; i < NPE * DIM; ++i) kk[j] = i == a * DIM + c ? F[i] : kk[j];
          if ((fm >> j) & 1u) {
            self[j] -= kk[j];
            kk[j] = T(0);
          }
        }
        const unsigned to = nb * unsigned(DIM * sizeof(T));
        bool found = false;
#pragma unroll
        for (int d = 0; d < D; ++d) {
          const bool hit = !found && (id[d] == to || id[d] == NONE);
          id[d] = hit ? to : id[d];
#pragma unroll
          for (int j = 0; j < DIM; ++j) k[d][j] = hit ? k[d][j] + kk[j] : k[d][j];
          found = found || hit;
        }
        ok = ok && found;
      }
    }
    n = 0;
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (__ballot(id[d] != NONE)) n = d + 1;
      if (id[d] == NONE) id[d] = unsigned(node) * unsigned(DIM * sizeof(T));
    }
#pragma unroll
    for (int d = 0; d < D; ++d) off[d >> 1] = d & 1 ? off[d >> 1] | (id[d] << 16) : id[d];
    return ok;
  }

  // The row times a node vector in LDS.
  __device__ __forceinline__ T times(const T *s_x, int node) const {
    T u[DIM], y = T(0);
#pragma unroll
    for (int j = 0; j < DIM; ++j) u[j] = (zero >> j) & 1u ? T(0) : s_x[node * DIM + j];
#pragma unroll
    for (int j = 0; j < DIM; ++j) y += self[j] * u[j];
    auto add2 = [&](int d) {
      const unsigned o2 = fresh(off[d >> 1]);
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const T *x = reinterpret_cast<const T *>(reinterpret_cast<const char *>(s_x) +
                                                 (e ? o2 >> 16 : o2 & 0xffffu));
#pragma unroll
        for (int j = 0; j < DIM; ++j) y += k[d + e][j] * (x[j] - u[j]);
      }
    };
    // (a regular triangulation's six at once, the others in pairs)
#pragma unroll
    for (int d = 0; d < 6; d += 2) add2(d);
#pragma unroll
    for (int d = 6; d < D; d += 2)
      if (d < n) add2(d);
    return y;
  }
};

// Value of the lane 8, 16 or 32 away (xor); t: the thread (a caller without
// registers to spare passes it formed anew, fresh(threadIdx.x)).
template <int O>
__device__ __forceinline__ unsigned lane_xor(unsigned v, unsigned t) {
  static_assert(O == 8 || O == 16 || O == 32, "");
  if constexpr (O == 8) {
    return unsigned(__builtin_amdgcn_update_dpp(0, int(v), 0x128, 0xf, 0xf, false));
  } else if constexpr (O == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return t & 16u ? r[0] : r[1];
  } else {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return t & 32u ? r[0] : r[1];
  }
}
template <int O>
__device__ __forceinline__ double lane_xor(double v, unsigned t) {
  return __hiloint2double(int(lane_xor<O>(unsigned(__double2hiint(v)), t)),
                          int(lane_xor<O>(unsigned(__double2loint(v)), t)));
}
// a + (a's partner) in the lower half (of 32: rows 0, 2), b + (b's partner) in the
// upper (rows 1, 3).
template <int O>
__device__ __forceinline__ double fold(double a, double b) {
  static_assert(O == 16 || O == 32, "");
  unsigned al = unsigned(__double2loint(a)), ah = unsigned(__double2hiint(a));
  unsigned bl = unsigned(__double2loint(b)), bh = unsigned(__double2hiint(b));
  if constexpr (O == 32) {
    const auto l = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
    const auto h = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
    return __hiloint2double(int(h[0]), int(l[0])) + __hiloint2double(int(h[1]), int(l[1]));
  } else {
    const auto l = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
    const auto h = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
    return __hiloint2double(int(h[0]), int(l[0])) + __hiloint2double(int(h[1]), int(l[1]));
  }
}
// Sum over the lane's eight.
__device__ __forceinline__ double sum8(double v) {
  v += dpp_f64<0xB1>(v);
  v += dpp_f64<0x4E>(v);
  return v + dpp_f64<0x141>(v);
}

// Sums of NV values over a wave; lane l gets value l / (64 / NV)'s.  Each step
// halves the values with the lanes that hold them: 8 values in 10 additions
// instead of 48.
template <int NV>
__device__ __forceinline__ double wave_sums(const double (&v)[NV], unsigned t) {
  if constexpr (NV == 8) {
    const double s0 = fold<16>(fold<32>(v[0], v[4]), fold<32>(v[2], v[6]));
    const double s1 = fold<16>(fold<32>(v[1], v[5]), fold<32>(v[3], v[7]));
    const bool hi = t & 8u;
    return sum8((hi ? s1 : s0) + lane_xor<8>(hi ? s0 : s1, t));
  } else {
    double s;
    if constexpr (NV == 4) {
      s = fold<16>(fold<32>(v[0], v[2]), fold<32>(v[1], v[3]));
    } else {
      s = fold<32>(v[0], v[NV - 1]);
      s += lane_xor<16>(s, t);
    }
    return sum8(s + lane_xor<8>(s, t));
  }
}

// Sums of RES_SUMS values over the workgroup's threads: wave v < RES_SUMS gets value
// v's in every lane of its first row (fixed order).  s_red: RES_SUMS * 16 doubles
// that no thread still reads or writes.
template <int PT>
__device__ __forceinline__ double sum_by_wave(const double (&v)[RES_SUMS], double *s_red) {
  constexpr int W = PT / 64;
  static_assert(RES_SUMS <= 8 && W >= RES_SUMS && W <= 16, "");
  double v8[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) v8[k] = k < RES_SUMS ? v[k < RES_SUMS ? k : 0] : 0.0;
  const double s = wave_sums<8>(v8, threadIdx.x);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if ((l & 7) == 0 && l < 8 * RES_SUMS) s_red[(l >> 3) * 16 + w] = s;
  __syncthreads();
  double q = w < RES_SUMS && l < W ? s_red[w * 16 + l] : 0.0;
  q += dpp_f64<0xB1>(q);
  q += dpp_f64<0x4E>(q);
  q += dpp_f64<0x141>(q);
  return q + dpp_f64<0x140>(q);
}

// Wave v publishes the workgroup's value v under `tag`, a copy to two lanes.
__device__ __forceinline__ void publish(const Exchange &x, int pid, unsigned tag, double v) {
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (w < RES_SUMS && l < 2 * EX_COPIES) {
    u64 h[2];
    tag_words(v, tag, h);
    st_agent(&x.words[(l >> 1) * x.stride + size_t(2 * w + (l & 1)) * x.np + pid], h[l & 1]);
  }
}

// Wave v gathers every workgroup's value v of `tag` (NB loads of each lane in
// flight) and sums them in a fixed order; the sums reach every thread through
// s_bc (RES_SUMS doubles) behind a barrier, which also ends the wait for the
// entries.  alone: v is the sum already.  False when a workgroup gave up (or
// *s_flag was set).
__device__ __forceinline__ bool gather(const Exchange &x, unsigned tag, double v,
                                       double (&sums)[RES_SUMS], double *s_bc, int *s_flag,
                                       bool alone) {
  constexpr int NB = 4;
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  if (w < RES_SUMS) {
    if (!alone) {
      v = 0.0;
      const u64 *words = x.words + x.copy * x.stride + size_t(2 * w) * x.np;
      bool ok = true;
      for (int i0 = l; ok && i0 < x.np; i0 += 64 * NB) {
        u64 h[NB][2];
        Patience wait{x.abort};
        for (int spin = 0;; ++spin) {
          bool all = true;
#pragma unroll
          for (int i = 0; i < NB; ++i)
#pragma unroll
            for (int k = 0; k < 2; ++k)
              if (i0 + 64 * i < x.np) h[i][k] = ld_agent(&words[size_t(k) * x.np + i0 + 64 * i]);
#pragma unroll
          for (int i = 0; i < NB; ++i)
            if (i0 + 64 * i < x.np)
              all = all && unsigned(h[i][0] >> 32) == tag && unsigned(h[i][1] >> 32) == tag;
          if (all) break;
          if (wait.over(spin)) {
            ok = false;
            break;
          }
        }
#pragma unroll
        for (int i = 0; i < NB; ++i)
          if (i0 + 64 * i < x.np) v += untag(h[i]);
      }
      if (!ok) *s_flag = 1;
      v = wave_sum(v);
    }
    if (l == 0) s_bc[w] = v;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < RES_SUMS; ++k) sums[k] = s_bc[k];
  return *s_flag == 0;
}

}  // namespace resident
}  // namespace femgpu
