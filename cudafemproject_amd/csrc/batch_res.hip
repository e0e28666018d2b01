// batch_res.hip -- the lockstep schedule's PCG with every instance in
// workgroups of its own that stay on the chip (batch_res.h); exchange between
// an instance's workgroups, waiting and determinism as in resident.hip.
//
// The launch-per-iteration form (batch_ls.hip) advances all systems together:
// every iteration streams the patches' mesh data and the systems' vectors
// through memory, waits for the slowest instance, and a system that pauses for
// its residual replacement idles to the end of the replay.  Here matrix rows
// and residuals stay in registers, directions and solutions in LDS, an
// instance waits only for its own workgroups, replaces a residual at once and
// makes room for the next when it is done.  Measured, device time of FP64
// solves to 1e-10, launch per iteration -> resident: 60 equal plates of 80 x 40
// with four load cases 44.7 -> 21.2 ms (830 iterations), with one 16.2 -> 10.0;
// one plate of 160 x 80, four load cases, 33.9 -> 16.3; one of 300 x 220 to 1e-8
// 110 -> 71; 200 plates of [16, 160] x [16, 80] to 1e-9 230 -> 127 ms (mixed in
// launches 192).
//
// The patch's part of K is applied by rows (PatchRow) instead of element by
// element: a product is the patch's 7 neighbour reads per DOF and system with
// no barrier between, where the entry lists of an element-wise product take 13
// LDS accesses and two barriers per system (four systems 2.6 kcycles of 2.4 GHz
// each against 1.06).  What bounds an iteration of four systems, 18 kcycles in
// one workgroup: the products 4.2, two trips through memory 3.6 + 2.2 and 4.6,
// interface sums 1.9, block sums 2; two workgroups per compute unit overlap.
//
// Workgroups take tickets, a patch each, and the tickets run instance by instance;
// one that is done takes the next.  Whoever waits for a ticket that nobody has
// taken waits for earlier instances only, and those end: the earliest one that
// has not ended has all its patches in hand, as long as as many workgroups as
// its patches are on the chip.  A launch has no more workgroups than the chip
// holds.  (With a workgroup per ticket the later ones start when places become
// free, and the hardware does not always start the next one that some compute
// unit has room for: three plates of some 320 patches each stood still in one
// run of three, some 100 places empty, until the waits ran out.)  Waits are
// bounded all the same, from the launch's last sign of progress.
//
// All arithmetic is FP64.  A system ends on its FP64 residual f - K x, formed
// when the recurrence's meets the tolerance.
//
// Reference: the PCG of gpuPCG_EbE_vec (femfunc.cpp:25-128) with the
// relative-residual rule.
#include <hip/hip_runtime.h>

#include "batch_res.h"
#include "element.h"
#include "femgpu.h"
#include "patch_common.h"
#include "resident.h"
#include "resident_dev.h"

namespace femgpu {

namespace {

using namespace elem;
using namespace patch;
using namespace resident;

constexpr int PT = BR_THREADS;
constexpr int DIM = 2;

// Directions and solutions of the NR systems (while the rows are formed: the
// entries' elements, the elements' nodes, the constrained components; the node
// coordinates), the interface contributions of all systems, the exchange
// tables, the sums.
struct BRLds {
  int off_el, off_fix, off_x, off_in, off_oe, off_os, off_ip, off_red, total;
};
__host__ __device__ inline BRLds br_lds(int nr, int pn, int ent, int n_in, int n_src) {
  BRLds L;
  L.off_el = al32(ent * 2);
  L.off_fix = L.off_el + BR_ELEMS * 4;
  const int v = nr * BR_NODES * DIM * 8, rows = L.off_fix + al32(pn);
  L.off_x = v > rows ? v : rows;
  L.off_in = L.off_x + v;
  L.off_oe = L.off_in + al32(n_src * DIM * nr * 8);
  L.off_os = L.off_oe + al32(n_in * 4);
  L.off_ip = L.off_os + al32(n_in * 2);
  L.off_red = L.off_ip + al32(n_in * 2);
  L.total = L.off_red + (3 * nr * (PT / 64) + nr) * 8;
  return L;
}

// Sums over the workgroup, in wave 0: lane l's value is (l / 8) % NV.  s_red:
// NV * PT / 64 doubles that no thread still reads or writes for another sum.
template <int NV>
__device__ __forceinline__ double block_sums(const double (&v)[NV], double *s_red) {
  static_assert(PT == 512, "eight waves: a value's in eight lanes");
  const double s = wave_sums<NV>(v, fresh(threadIdx.x));
  const int tx = fresh(threadIdx.x), w = tx >> 6, l = tx & 63;
  if (l % (64 / NV) == 0) s_red[(l / (64 / NV)) * 8 + w] = s;
  __syncthreads();
  return w == 0 ? sum8(s_red[((l >> 3) % NV) * 8 + (l & 7)]) : 0.0;
}
// Exchange of these sums between an instance's np workgroups, words
// [workgroup][value][2]: wave 0 publishes workgroup i's and gathers everyone's
// (64 / NV workgroups at a time, NB loads of each lane in flight) in a fixed
// order.  False when a workgroup gave up.
template <int NV>
__device__ __forceinline__ void publish_lanes(u64 *words, int i, unsigned tag, double v) {
  const int l = fresh(threadIdx.x);
  u64 w[2];
  tag_words(v, tag, w);
  if (l < 8 * NV && (l & 7) < 2) st_agent(&words[(size_t(i) * NV + (l >> 3)) * 2 + (l & 1)], l & 1 ? w[1] : w[0]);
}
template <int NV>
__device__ __forceinline__ bool gather_lanes(const u64 *words, int np, unsigned tag, u64 *abort,
                                             double &sum) {
  constexpr int G = 64 / NV, NB = 4;
  const int l = fresh(threadIdx.x), v = (l >> 3) % NV;
  sum = 0.0;
  bool ok = true;
  for (int i0 = (l & 7) + 8 * ((l >> 3) / NV); ok && i0 < np; i0 += G * NB) {
    u64 h[NB][2];
    QueuePatience wait{abort};
    for (int spin = 0;; ++spin) {
      bool all = true;
#pragma unroll
      for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int k = 0; k < 2; ++k)
          if (i0 + G * b < np) h[b][k] = ld_agent(&words[(size_t(i0 + G * b) * NV + v) * 2 + k]);
#pragma unroll
      for (int b = 0; b < NB; ++b)
        if (i0 + G * b < np)
          all = all && unsigned(h[b][0] >> 32) == tag && unsigned(h[b][1] >> 32) == tag;
      if (all) break;
      if (wait.over(spin)) {
        ok = false;
        break;
      }
    }
#pragma unroll
    for (int b = 0; b < NB; ++b)
      if (i0 + G * b < np) sum += untag(h[b]);
  }
  sum = sum8(sum);
  if constexpr (NV == 1) sum += lane_xor<8>(sum, l);
  if constexpr (NV <= 2) sum += lane_xor<16>(sum, l);
  if constexpr (NV <= 4) sum += lane_xor<32>(sum, l);
  return __all(ok);
}

// A system, advanced by the lanes of wave 0 that hold its sums, all alike (and
// in every workgroup): in registers what every iteration needs, the rest in
// LDS (every lane writes the same).
struct BRRest {
  double ff, rr_last, rr;  // ||f||^2; r'r at the last replacement and at the last look
  int status, nrep, stag;
};
struct BRSystem {
  double thr, g;  // tol^2 ||f||^2; r'z that p was formed with
  int state;      // 0 iterating, 1 residual wanted, 2 residual wanted to end, 3 ended
  int it;

  __device__ __forceinline__ void end(BRRest &R, int s, int st) {
    R.status = s;
    state = st;
  }
  // r = f formed: whether to iterate.
  __device__ __forceinline__ void start(BRRest &R, double gv, double rrv, double tol2) {
    R.ff = R.rr = R.rr_last = rrv;
    thr = tol2 * rrv;
    g = gv;
    it = R.nrep = R.stag = state = 0;
    if (!isfinite(gv) || !isfinite(rrv)) end(R, FEMGPU_E_NONFINITE, 3);
    else if (rrv <= thr) end(R, FEMGPU_OK, 3);
  }
  // After an update: r'z and r'r of the recurrence.
  __device__ __forceinline__ void look(BRRest &R, double gv, double rrv, int max_iter) {
    if (!isfinite(gv) || !isfinite(rrv)) {
      end(R, FEMGPU_E_NONFINITE, 2);
    } else if (rrv <= thr) {
      R.rr = rrv;
      state = 1;
    } else if (it >= max_iter) {
      end(R, FEMGPU_E_MAXIT, 2);
    }
  }
  // After a replacement; true: restart the directions (the FP64 residual did
  // not halve since the last one, or the recurrence's had drifted from it).
  // Two in a row without a decrease end the system: its tolerance is below the
  // attainable accuracy.
  __device__ __forceinline__ bool replaced(BRRest &R, double gv, double rrv, int max_iter) {
    const double last = R.rr_last;
    const int nrep = R.nrep, stag = nrep >= 1 && rrv >= last ? R.stag + 1 : 0;
    const bool restart = rrv > 0.25 * last || rrv > 4.0 * R.rr;
    R.stag = stag;
    R.rr = R.rr_last = rrv;
    R.nrep = nrep + 1;
    state = 0;
    if (!isfinite(gv) || !isfinite(rrv)) end(R, FEMGPU_E_NONFINITE, 3);
    else if (rrv <= thr) end(R, FEMGPU_OK, 3);
    else if (stag >= 2) end(R, FEMGPU_E_STAGNATION, 3);
    else if (it >= max_iter) end(R, FEMGPU_E_MAXIT, 3);
    return restart;
  }
};

// One patch from the first residual to the end of its instance's systems.
// s_flag: 0; false: a wait ran out.
template <int NR, int DEGREE>
__device__ __forceinline__ bool solve_patch(const BRArgs &a, int pid, unsigned char *lds, int &s_flag) {
  constexpr int W = PT / 64;
  constexpr int NPE = DIM + 1, NX = DIM * NR;
  __shared__ BRRest s_rest[NR];
  __shared__ int s_iter, s_want;  // systems that iterate, whose residual is wanted
  const int t = fresh(threadIdx.x);  // (nothing of a patch is kept for the next)
  const BRLds L = br_lds(NR, a.pn, a.ent, a.n_in_max, a.n_src_max);
  double *s_p = reinterpret_cast<double *>(lds);
  uint16_t *s_ent = reinterpret_cast<uint16_t *>(lds);
  uint32_t *s_el = reinterpret_cast<uint32_t *>(lds + L.off_el);
  uint8_t *s_fix = reinterpret_cast<uint8_t *>(lds + L.off_fix);
  double *s_x = reinterpret_cast<double *>(lds + L.off_x);
  double *s_c = s_x;
  double *s_in = reinterpret_cast<double *>(lds + L.off_in);
  uint32_t *s_oe = reinterpret_cast<uint32_t *>(lds + L.off_oe);
  uint16_t *s_os = reinterpret_cast<uint16_t *>(lds + L.off_os);
  uint16_t *s_ip = reinterpret_cast<uint16_t *>(lds + L.off_ip);
  double *s_red = reinterpret_cast<double *>(lds + L.off_red);
  double *s_co = s_red + 3 * NR * W;  // beta or alpha per system

  const PatchInfo P = a.patches[pid];
  const ExchangePatch E = a.xpatch[pid];
  const BLInst I = a.inst[P.pad];
  const int np = I.p1 - I.p0, lp = pid - I.p0;
  const bool alone = np == 1;
  // p'q, r'z and r'r, the same of a replaced residual (three places: one is
  // written again only after two exchanges that every workgroup took part in)
  u64 *xpq = a.words + br_patch_words(NR) * size_t(I.p0);
  u64 *xrz = xpq + size_t(4) * NR * np, *xrep = xrz + size_t(4) * NR * np;
  unsigned tag = 0, entry_tag = 0;

  const int k = t / DIM, c = t % DIM;
  const bool has = k < P.n_own + P.n_sh, own = k < P.n_own;
  for (int i = t; i < a.ent; i += PT) s_ent[i] = 0;
  bool first = own;
  int gid = 0;
  unsigned places = 0;  // an interface node's: first, and end in the upper half
  int lo = 0;           // the patch's own
  double invd = 0.0;
  PatchRow<double, DIM, DEGREE> row;
  {
    double diag = 0.0;
    int b0 = 0, b1 = 0;
    if (has) {
      b1 = int(a.node_end[P.pnode_start + k]);
      b0 = k ? int(a.node_end[P.pnode_start + k - 1]) : 0;
      gid = P.own_start + k;
      if (!own) {
        const int j = P.sh_start + k - P.n_own;
        const int4 sh = a.sh_info[j];
        gid = sh.x;
        first = sh.y == sh.z;
        places = (k > P.n_own ? unsigned(a.src_end[j - 1]) : 0u) | unsigned(a.src_end[j]) << 16;
        lo = int(a.own_pos[j]);
      }
      const unsigned fm = a.fixmask[gid];
      if (c == 0) s_fix[k] = uint8_t(fm & ((1u << DIM) - 1u));
      s_c[t] = a.coords[size_t(gid) * DIM + c];
      invd = a.invD[size_t(gid) * DIM + c];
      // (a constrained row counts in the patch that accounts for the node)
      if (((fm >> c) & 1u) && first) diag = a.diagK[size_t(gid) * DIM + c];
    }
    for (int i = t; i < E.n_in; i += PT) {
      s_oe[i] = a.out_entry[E.out_start + i];
      s_os[i] = a.out_src[E.out_start + i];
      s_ip[i] = a.in_pos[E.out_start + i];
    }
    __syncthreads();
    if (t < P.n_elem) {
      int l[4], q[4];
      decode_rec(reinterpret_cast<const uint3 *>(a.erec)[P.elem_start + t], l, q);
      s_el[t] = unsigned(l[0]) | unsigned(l[1]) << 10 | unsigned(l[2]) << 20;
#pragma unroll
      for (int n = 0; n < NPE; ++n) s_ent[q[n]] = uint16_t(t * 4 + n + 1);
    }
    __syncthreads();
    if (!row.build(has ? k : 0, c, b0, b1, s_ent, s_el, s_fix, s_c, diag, I.lam, I.mu)) {
      st_agent(a.abort, 1);  // (the host counted wrongly)
      s_flag = 1;
    }
    __syncthreads();
    if (s_flag) return false;
  }
  const int node = has ? k : 0;
  constexpr int sv = BR_NODES * DIM;  // a system's stride in s_p, s_x
  double r[NR];
#pragma unroll
  for (int v = 0; v < NR; ++v) {
    r[v] = has ? a.f[(size_t(gid) * NR + v) * DIM + c] : 0.0;
    if (has) s_p[v * sv + t] = s_x[v * sv + t] = 0.0;
  }

  // y = this patch's part of K u at this thread's DOF for the systems of mask
  // (u complete in LDS); interface contributions to their places.  Ends with a
  // barrier.
  auto product = [&](unsigned mask, const double *s_u, double (&y)[NR]) {
#pragma unroll
    for (int v = 0; v < NR; ++v) {
      y[v] = 0.0;
      if (!((mask >> v) & 1u)) continue;
      y[v] = row.times(s_u + v * sv, node);
      if (has && !own) s_in[lo * NX + v * DIM + c] = y[v];
    }
    __syncthreads();
  };
  // Sends the contributions, receives the others' (complete after a barrier),
  // a system's by PT / NR threads.
  auto trade = [&](unsigned mask) {
    constexpr int TV = PT / NR;
    const int t = fresh(threadIdx.x), v = t / TV;
    ++entry_tag;
    if (!((mask >> v) & 1u)) return;
    auto at = [&](unsigned e) { return ((e >> 6) * unsigned(NR) + unsigned(v)) * 64u + (e & 63u); };
    for (int i = t % TV; i < E.n_in; i += TV)
      send_entry<double, DIM>(a.entries, at(s_oe[i]), entry_tag, &s_in[int(s_os[i]) * NX + v * DIM]);
    for (int i = t % TV; i < E.n_in; i += TV)
      if (!recv_entry<double, DIM>(a.entries, at(unsigned(E.in_start + i)), entry_tag,
                                   QueuePatience{a.abort}, &s_in[int(s_ip[i]) * NX + v * DIM]))
        s_flag = 1;
  };
  auto collect = [&](double (&y)[NR]) {
    if (has && !own) {
#pragma unroll
      for (int v = 0; v < NR; ++v) y[v] = 0.0;
      for (int j = int(places & 0xffffu); j < int(places >> 16); ++j)
#pragma unroll
        for (int v = 0; v < NR; ++v) y[v] += s_in[j * NX + v * DIM + c];
    }
  };
  // Wave 0: the lane's system's r'z and r'r over the instance.
  auto dots = [&](u64 *ex, double &g, double &rr) {
    double v[2 * NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      v[i] = first ? r[i] * mul_rn(invd, r[i]) : 0.0;
      v[NR + i] = first ? r[i] * r[i] : 0.0;
    }
    double s = block_sums<2 * NR>(v, s_red + NR * W);
    ++tag;
    if (t < 64) {
      if (!alone) {
        publish_lanes<2 * NR>(ex, lp, tag, s);
        if (!gather_lanes<2 * NR>(ex, np, tag, a.abort, s)) s_flag = 1;
      }
      const double o = lane_xor<8 * NR>(s, fresh(threadIdx.x));
      const bool second = t & (8 * NR);
      g = second ? o : s;
      rr = second ? s : o;
    }
  };
  // Wave 0: a coefficient per system and the systems' states to everyone
  // (behind a barrier).
  BRSystem S;
  BRRest &R = s_rest[(t >> 3) % NR];
  auto tell = [&](double coef) {
    const u64 run = __ballot(S.state == 0), want = __ballot(S.state == 1 || S.state == 2);
    if ((t & 7) == 0 && t < 8 * NR) s_co[t >> 3] = coef;
    if (t == 0) {
      int m = 0, w = 0;
#pragma unroll
      for (int v = 0; v < NR; ++v) {
        m |= int((run >> (8 * v)) & 1u) << v;
        w |= int((want >> (8 * v)) & 1u) << v;
      }
      s_iter = m;
      s_want = w;
    }
  };

  {
    double g, rr;
    dots(xrz, g, rr);
    if (t < 64) {
      S.start(R, g, rr, a.tol2);
      tell(0.0);
    }
    __syncthreads();
  }
  bool ok = s_flag == 0;
  while (ok) {
    unsigned iter = __builtin_amdgcn_readfirstlane(s_iter);
    const unsigned want = __builtin_amdgcn_readfirstlane(s_want);
    if (!(iter | want)) break;
    if (want) {
      // r = f - K x of the systems that stopped; their next step
      double y[NR], beta = t < 64 ? s_co[(t >> 3) % NR] : 0.0;
      product(want, s_x, y);
      if (!alone) trade(want);
      __syncthreads();
      collect(y);
#pragma unroll
      for (int v = 0; v < NR; ++v)
        if (((want >> v) & 1u) && has) r[v] = a.f[(size_t(gid) * NR + v) * DIM + c] - y[v];
      double g, rr;
      dots(xrep, g, rr);
      if (t < 64) {
        if (S.state == 1) {
          beta = S.replaced(R, g, rr, a.max_iter) ? 0.0 : g / S.g;
          S.g = g;
        } else if (S.state == 2) {
          R.rr = rr;
          S.state = 3;
        }
        tell(beta);
      }
      __syncthreads();
      ok = s_flag == 0;
      iter = __builtin_amdgcn_readfirstlane(s_iter);
      if (!ok || !iter) break;
    }
    double y[NR], pq[NR];
    if (has)
#pragma unroll
      for (int v = 0; v < NR; ++v)
        if ((iter >> v) & 1u) s_p[v * sv + t] = pcg_dir(invd, r[v], s_co[v], s_p[v * sv + t]);
    __syncthreads();
    product(iter, s_p, y);
#pragma unroll
    for (int v = 0; v < NR; ++v) pq[v] = has ? s_p[v * sv + t] * y[v] : 0.0;
    double d = block_sums<NR>(pq, s_red);
    ++tag;
    if (!alone) {
      if (t < 64) publish_lanes<NR>(xpq, lp, tag, d);
      trade(iter);
    }
    if (t < 64) {
      if (!alone && !gather_lanes<NR>(xpq, np, tag, a.abort, d)) s_flag = 1;
      // every 32 iterations a sign of progress to those who wait (here: at the
      // loop's begin it moved the spills about, and four systems took 6 %
      // longer)
      if ((tag & 62u) == 0 && t == 0) st_agent(a.abort + 3, wall_clock64());
      double alpha = 0.0;
      if (S.state == 0) {
        alpha = S.g / d;
        if (!(d > 0.0) || !isfinite(alpha)) {
          // (no x or r changes: the state of the last completed iteration)
          S.end(R, isfinite(d) ? FEMGPU_E_BREAKDOWN : FEMGPU_E_NONFINITE, 2);
          alpha = 0.0;
        } else {
          ++S.it;
        }
      }
      tell(alpha);
    }
    __syncthreads();
    ok = s_flag == 0;
    if (!ok) break;
    iter = __builtin_amdgcn_readfirstlane(s_iter);
    collect(y);
    if (has)
#pragma unroll
      for (int v = 0; v < NR; ++v)
        if ((iter >> v) & 1u) {
          s_x[v * sv + t] = s_x[v * sv + t] + s_co[v] * s_p[v * sv + t];
          r[v] = r[v] - s_co[v] * y[v];
        }
    double g, rr;
    dots(xrz, g, rr);
    if (t < 64) {
      double beta = 0.0;
      if (S.state == 0) {
        S.look(R, g, rr, a.max_iter);
        if (S.state == 0) {
          beta = g / S.g;
          S.g = g;
        }
      }
      tell(beta);
    }
    __syncthreads();
    ok = s_flag == 0;
  }
  if (first)
#pragma unroll
    for (int v = 0; v < NR; ++v) a.x[(size_t(gid) * NR + v) * DIM + c] = s_x[v * sv + t];
  if (lp == 0 && (t & 7) == 0 && t < 8 * NR) {
    BLState &o = a.st[size_t(P.pad) * NR + (t >> 3)];
    o.state = 3;
    o.status = R.status;
    o.iters = S.it;
    o.nrep = R.nrep;
    o.ff = R.ff;
    o.rr = R.rr;
  }
  return ok;
}

template <int NR, int DEGREE>
__global__ __launch_bounds__(PT, 4) void k_batch_resident(BRArgs a) {
  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ int s_flag, s_ticket;
  if (threadIdx.x == 0) s_flag = 0;
  for (;;) {
    __syncthreads();  // (the last patch's values are read)
    if (threadIdx.x == 0) s_ticket = int(atomicAdd(reinterpret_cast<unsigned *>(a.abort + 2), 1u));
    __syncthreads();
    const int ticket = __builtin_amdgcn_readfirstlane(s_ticket);
    if (ticket >= a.np || !solve_patch<NR, DEGREE>(a, a.order[ticket], lds, s_flag)) return;
  }
}

// One value per thread: node, rhs, component.
__global__ void k_br_rhs_in(int64_t n, int n_rhs, int nr, const int32_t *perm, const double *user,
                            double *f) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const int m = nr * DIM;
  if (i >= n * m) return;
  const int64_t g = i / m;
  const int j = int(i % m);
  f[i] = j < n_rhs * DIM ? user[int64_t(perm[g]) * n_rhs * DIM + j] : 0.0;
}
__global__ void k_br_rhs_out(int64_t n, int n_rhs, int nr, const int32_t *perm, const double *x,
                             double *user) {
  const int64_t i = int64_t(blockIdx.x) * 256 + threadIdx.x;
  const int m = n_rhs * DIM;
  if (i >= n * m) return;
  const int64_t g = i / m;
  user[int64_t(perm[g]) * m + i % m] = x[g * nr * DIM + i % m];
}

using Kernel = void (*)(BRArgs);
Kernel kernel_of(int nr, int degree) {
  if (degree == BR_DEGREE)
    return nr == 1   ? k_batch_resident<1, BR_DEGREE>
           : nr == 2 ? k_batch_resident<2, BR_DEGREE>
                     : k_batch_resident<4, BR_DEGREE>;
  return nr == 1   ? k_batch_resident<1, BR_DEGREE_MAX>
         : nr == 2 ? k_batch_resident<2, BR_DEGREE_MAX>
                   : k_batch_resident<4, BR_DEGREE_MAX>;
}

int blocks(int64_t n) { return int((n + 255) / 256); }

constexpr int BR_LDS_MAX = 160 * 1024 - 1024;  // (and the static part)

}  // namespace

int br_lds_bytes(int nr, int pn, int ent, int n_in, int n_src) {
  return br_lds(nr, pn, ent, n_in, n_src).total;
}

int br_capacity(int nr, int degree, int lds, int device, double *block) {
  const int cu = compute_units(device);
  if (cu < 1 || lds > BR_LDS_MAX) return 0;
  const int per = blocks_per_cu(reinterpret_cast<const void *>(kernel_of(nr, degree)), PT, lds);
  *block = per > 0 ? 1.0 / per : 1.0;
  return per * cu;
}

int br_groups_max(int device) { return 2 * compute_units(device); }

void launch_batch_resident(int nr, int degree, const BRArgs &a, int groups, hipStream_t s) {
  const int lds = br_lds_bytes(nr, a.pn, a.ent, a.n_in_max, a.n_src_max);
  hipLaunchKernelGGL(kernel_of(nr, degree), dim3(groups), dim3(PT), lds, s, a);
}

void launch_br_rhs_in(int64_t n, int n_rhs, int nr, const int32_t *perm, const double *user,
                      double *f, hipStream_t s) {
  hipLaunchKernelGGL(k_br_rhs_in, dim3(blocks(n * nr * DIM)), dim3(256), 0, s, n, n_rhs, nr, perm,
                     user, f);
}
void launch_br_rhs_out(int64_t n, int n_rhs, int nr, const int32_t *perm, const double *x,
                       double *user, hipStream_t s) {
  hipLaunchKernelGGL(k_br_rhs_out, dim3(blocks(n * n_rhs * DIM)), dim3(256), 0, s, n, n_rhs, nr,
                     perm, x, user);
}

hipError_t prepare_br_kernels() {
  hipError_t e = hipSuccess, r;
  for (int nr : {1, 2, 4})
    for (int degree : {BR_DEGREE, BR_DEGREE_MAX})
      if ((r = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel_of(nr, degree)),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, BR_LDS_MAX)) !=
          hipSuccess)
        e = r;
  return e;
}

}  // namespace femgpu
