// mesh_plan.cpp -- host-side preparation of the device mesh layout.
//
// Replaces the reference's per-iteration sort-based assembly set-up
// (genMask + sort + reduce_by_key, fem_utils/src/cpu_fem_utils.cpp:182-219 and
// fem_utils/src/cu/cuda_fem_utils.cpp:178-216): instead of sorting all
// element-local entries by DOF every PCG iteration, the element -> patch and
// node -> owner maps are built once here, and the kernels assemble in LDS and
// through fixed-order interface sums.  See femgpu_internal.h for the layout.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <new>
#include <numeric>
#include <thread>

#include "femgpu_internal.h"

namespace femgpu {

namespace {

uint64_t spread3(uint64_t v) {  // 21 bits -> every third bit
  v &= 0x1fffffULL;
  v = (v | v << 32) & 0x1f00000000ffffULL;
  v = (v | v << 16) & 0x1f0000ff0000ffULL;
  v = (v | v << 8) & 0x100f00f00f00f00fULL;
  v = (v | v << 4) & 0x10c30c30c30c30c3ULL;
  v = (v | v << 2) & 0x1249249249249249ULL;
  return v;
}

uint64_t spread2(uint64_t v) {  // 31 bits -> every second bit
  v &= 0x7fffffffULL;
  v = (v | v << 16) & 0x0000ffff0000ffffULL;
  v = (v | v << 8) & 0x00ff00ff00ff00ffULL;
  v = (v | v << 4) & 0x0f0f0f0f0f0f0f0fULL;
  v = (v | v << 2) & 0x3333333333333333ULL;
  v = (v | v << 1) & 0x5555555555555555ULL;
  return v;
}

// Entry positions within the padded node runs of one patch.  The patch
// kernels write the entries with one instruction per (element slot e,
// corner a): thread t writes the entry of its element t + e * pn_max.  Any
// position of a node's run may hold any of the node's entries (the padding
// positions are the unused ones, which stay zero), so the positions are
// chosen to spread the lanes of each write instruction over the LDS banks
// (4-byte words: 64 banks per wave, 32 per half wave): a greedy pass in
// the kernel's write order, then two sweeps of pairwise swaps inside each run
// that lower sum_W (2 * sum_b n64(W,b)^2 + sum_h,b n32(W,h,b)^2), n = lanes of
// write instruction W on a bank.  The order of the entries inside a run is
// the summation order of the node's sum; it is fixed by the plan.
struct BankScratch {
  std::vector<int32_t> occ, rstart, wid;
  std::vector<uint8_t> half;
  std::vector<int16_t> c64, c32;
};

// Items of up to `corners` entries (elements, strips), item i's local nodes at
// lid[4 or more * i] (NO_NODE: none), one item per thread and round of pn_max.
// node_end: ends of the nodes' runs.
constexpr uint16_t NO_NODE = 0xffff;

bool spread_entry_banks(const uint16_t *lid, uint16_t *epos, int stride, int corners, int32_t items,
                        int pn_max, const uint16_t *node_end, int32_t nloc, int32_t run,
                        BankScratch &B) {
  const int32_t nwave = (pn_max + 63) / 64;
  const int32_t slots_e = (items + pn_max - 1) / pn_max;
  const int32_t n_w = slots_e * corners * nwave;
  B.occ.assign(size_t(run), -1);
  B.rstart.resize(nloc);
  for (int32_t k = 0; k < nloc; ++k) B.rstart[k] = k ? int32_t(node_end[k - 1]) : 0;
  B.wid.assign(size_t(items) * stride, 0);
  B.half.assign(size_t(items) * stride, 0);
  B.c64.assign(size_t(n_w) * 64, 0);
  B.c32.assign(size_t(n_w) * 64, 0);
  for (int32_t e = 0; e < slots_e; ++e)
    for (int a = 0; a < corners; ++a)
      for (int32_t t = 0; t < pn_max; ++t) {
        const int32_t i = e * pn_max + t;
        if (i >= items) break;
        const int32_t j = i * stride + a, l = lid[j];
        if (l == NO_NODE) continue;
        const int32_t W = (e * corners + a) * nwave + t / 64, h = (t & 63) >> 5;
        int16_t *u64 = &B.c64[size_t(W) * 64], *u32 = &B.c32[size_t(W) * 64 + h * 32];
        const int32_t r1 = int32_t(node_end[l]);
        int32_t best = -1, best_cost = INT32_MAX;
        for (int32_t p = B.rstart[l]; p < r1; ++p) {
          if (B.occ[p] >= 0) continue;
          const int32_t cost = 2 * u64[p & 63] + u32[p & 31];
          if (cost < best_cost) {
            best_cost = cost;
            best = p;
            if (cost == 0) break;
          }
        }
        if (best < 0) return false;  // (the run is full)
        B.occ[best] = j;
        B.wid[j] = W;
        B.half[j] = uint8_t(h);
        ++u64[best & 63];
        ++u32[best & 31];
      }
  // cost change of moving entry j from position p to q (applied)
  auto move = [&](int32_t j, int32_t p, int32_t q) {
    int16_t *u64 = &B.c64[size_t(B.wid[j]) * 64], *u32 = &B.c32[size_t(B.wid[j]) * 64 + B.half[j] * 32];
    int32_t d = 0;
    if ((p ^ q) & 63) {
      d += 4 * (u64[q & 63] - u64[p & 63] + 1);
      --u64[p & 63];
      ++u64[q & 63];
    }
    if ((p ^ q) & 31) {
      d += 2 * (u32[q & 31] - u32[p & 31] + 1);
      --u32[p & 31];
      ++u32[q & 31];
    }
    return d;
  };
  for (int sweep = 0; sweep < 2; ++sweep) {
    int32_t improved = 0;
    for (int32_t k = 0; k < nloc; ++k) {
      const int32_t r0 = B.rstart[k], r1 = int32_t(node_end[k]);
      for (int32_t p = r0; p < r1; ++p)
        for (int32_t q = p + 1; q < r1; ++q) {
          const int32_t x = B.occ[p], y = B.occ[q];
          if (x < 0 && y < 0) continue;
          int32_t d = 0;
          if (x >= 0) d += move(x, p, q);
          if (y >= 0) d += move(y, q, p);
          if (d < 0) {
            B.occ[p] = y;
            B.occ[q] = x;
            ++improved;
          } else {
            if (y >= 0) move(y, p, q);
            if (x >= 0) move(x, q, p);
          }
        }
    }
    if (!improved) break;
  }
  for (int32_t p = 0; p < run; ++p)
    if (B.occ[p] >= 0) epos[B.occ[p]] = uint16_t(p);
  return true;
}

// fn(i) for i in [0, n) by up to 8 threads (fewer when the system gives fewer),
// in no order.  Calls that throw make it throw std::bad_alloc, once all have
// ended.
template <typename F>
void for_each_patch(int32_t n, F fn) {
  std::atomic<int32_t> next{0};
  std::atomic<bool> failed{false};
  auto work = [&] {
    try {
      auto f = fn();
      for (int32_t i = next++; i < n && !failed; i = next++) f(i);
    } catch (...) {
      failed = true;
    }
  };
  // (below some 64 patches a thread costs more than it takes over)
  const int n_threads = std::min({8, int(std::thread::hardware_concurrency()), int(n / 32)});
  std::vector<std::thread> threads;
  try {
    for (int i = 1; i < n_threads; ++i) threads.emplace_back(work);
  } catch (...) {
  }
  work();
  for (std::thread &t : threads) t.join();
  if (failed) throw std::bad_alloc();
}

}  // namespace

std::string build_plan(int dim, int64_t nn, const double *nodes, int64_t ne,
                       const int32_t *elems, int emax, int pn_max, bool pad_runs,
                       MeshPlan &plan) {
  if (dim != 2 && dim != 3) return "dim must be 2 or 3";
  if (nn <= 0 || ne <= 0) return "empty mesh";
  if (nn >= (int64_t(1) << 31) / 3 || ne >= (int64_t(1) << 31) / 12)
    return "mesh too large for int32 DOF indexing";
  if (emax < 16 || emax > EMAX_LIMIT) return "elements per patch out of range";
  if (pn_max < 16 || pn_max > PN_LIMIT) return "nodes per patch out of range";
  const int npe = dim + 1;
  plan = MeshPlan();
  plan.dim = dim;
  plan.npe = npe;
  plan.nde = dim * npe;
  plan.nn = nn;
  plan.ne = ne;
  plan.emax = emax;
  plan.padded = pad_runs;

  for (int64_t e = 0; e < ne; ++e) {
    for (int a = 0; a < npe; ++a) {
      int32_t v = elems[e * npe + a];
      if (v < 0 || v >= nn) return "element node index out of range";
      for (int b = 0; b < a; ++b)
        if (elems[e * npe + b] == v) return "element with a repeated node";
    }
  }

  // 1. Morton order of element centroids.
  double lo[3] = {0, 0, 0}, hi[3] = {0, 0, 0};
  for (int c = 0; c < dim; ++c) lo[c] = hi[c] = nodes[c];
  for (int64_t i = 0; i < nn; ++i)
    for (int c = 0; c < dim; ++c) {
      double v = nodes[i * dim + c];
      if (!std::isfinite(v)) return "non-finite node coordinate";
      lo[c] = std::min(lo[c], v);
      hi[c] = std::max(hi[c], v);
    }
  const int bits = dim == 3 ? 21 : 31;
  const double qmax = double((uint64_t(1) << bits) - 1);
  std::vector<std::pair<uint64_t, int32_t>> key(ne);
  for (int64_t e = 0; e < ne; ++e) {
    uint64_t q[3] = {0, 0, 0};
    for (int c = 0; c < dim; ++c) {
      double s = 0;
      for (int a = 0; a < npe; ++a) s += nodes[int64_t(elems[e * npe + a]) * dim + c];
      s /= npe;
      double span = hi[c] - lo[c];
      double t = span > 0 ? (s - lo[c]) / span : 0.0;
      q[c] = uint64_t(std::min(qmax, std::max(0.0, t * qmax)));
    }
    uint64_t k = dim == 3 ? (spread3(q[0]) | spread3(q[1]) << 1 | spread3(q[2]) << 2)
                          : (spread2(q[0]) | spread2(q[1]) << 1);
    key[e] = {k, int32_t(e)};
  }
  std::sort(key.begin(), key.end());
  plan.elem_perm.resize(ne);
  for (int64_t i = 0; i < ne; ++i) plan.elem_perm[i] = key[i].second;
  key.clear();
  key.shrink_to_fit();

  // 2. Greedy patches over the sorted elements.
  std::vector<int32_t> stamp(nn, -1);
  std::vector<int32_t> pstart;  // element start per patch
  {
    int32_t pid = 0, cur_nodes = 0, cur_elems = 0;
    pstart.push_back(0);
    for (int64_t i = 0; i < ne; ++i) {
      const int32_t *en = &elems[int64_t(plan.elem_perm[i]) * npe];
      int add = 0;
      for (int a = 0; a < npe; ++a) add += stamp[en[a]] != pid;
      if (cur_elems > 0 && (cur_elems + 1 > emax || cur_nodes + add > pn_max)) {
        ++pid;
        pstart.push_back(int32_t(i));
        cur_nodes = 0;
        cur_elems = 0;
        add = npe;
      }
      for (int a = 0; a < npe; ++a)
        if (stamp[en[a]] != pid) {
          stamp[en[a]] = pid;
          ++cur_nodes;
        }
      ++cur_elems;
    }
    pstart.push_back(int32_t(ne));
  }
  const int32_t np = int32_t(pstart.size()) - 1;

  // 3. Touch counts: how many patches reference each node.
  std::vector<int32_t> touches(nn, 0);
  std::fill(stamp.begin(), stamp.end(), -1);
  for (int32_t p = 0; p < np; ++p)
    for (int32_t i = pstart[p]; i < pstart[p + 1]; ++i) {
      const int32_t *en = &elems[int64_t(plan.elem_perm[i]) * npe];
      for (int a = 0; a < npe; ++a)
        if (stamp[en[a]] != p) {
          stamp[en[a]] = p;
          ++touches[en[a]];
        }
    }

  // 4. Internal node numbering: owned runs per patch, then interface, then isolated.
  std::vector<int32_t> inv(nn, -1);
  int32_t next = 0;
  for (int32_t p = 0; p < np; ++p)
    for (int32_t i = pstart[p]; i < pstart[p + 1]; ++i) {
      const int32_t *en = &elems[int64_t(plan.elem_perm[i]) * npe];
      for (int a = 0; a < npe; ++a)
        if (touches[en[a]] == 1 && inv[en[a]] < 0) inv[en[a]] = next++;
    }
  plan.n_owned = next;
  for (int32_t p = 0; p < np; ++p)
    for (int32_t i = pstart[p]; i < pstart[p + 1]; ++i) {
      const int32_t *en = &elems[int64_t(plan.elem_perm[i]) * npe];
      for (int a = 0; a < npe; ++a)
        if (touches[en[a]] > 1 && inv[en[a]] < 0) inv[en[a]] = next++;
    }
  plan.n_iface = next - plan.n_owned;
  for (int64_t v = 0; v < nn; ++v)
    if (inv[v] < 0) inv[v] = next++;
  plan.n_isolated = nn - plan.n_owned - plan.n_iface;
  plan.node_inv = inv;
  plan.node_perm.assign(nn, 0);
  for (int64_t v = 0; v < nn; ++v) plan.node_perm[inv[v]] = int32_t(v);

  // 5. Interface slots (contiguous per node, patch order).
  plan.slot_start.assign(plan.n_iface + 1, 0);
  for (int64_t j = 0; j < plan.n_iface; ++j)
    plan.slot_start[j + 1] = plan.slot_start[j] + touches[plan.node_perm[plan.n_owned + j]];
  plan.n_slots = plan.slot_start[plan.n_iface];
  std::vector<int32_t> slot_next(plan.slot_start.begin(), plan.slot_start.end() - 1);

  // 6. Per-patch local numbering, packed ids and node-sorted entry positions.
  plan.patches.resize(np);
  plan.elem_lid.assign(size_t(ne) * 4, 0);
  plan.epos.assign(size_t(ne) * 4, 0);
  plan.elems_int.assign(size_t(ne) * npe, 0);
  std::vector<int32_t> local(nn, -1);
  std::vector<int32_t> loc_nodes;
  std::vector<int32_t> cnt;
  for (int32_t p = 0; p < np; ++p) {
    PatchInfo &P = plan.patches[p];
    P.elem_start = pstart[p];
    P.n_elem = pstart[p + 1] - pstart[p];
    P.sh_start = int32_t(plan.sh_gid.size());
    P.pnode_start = int32_t(plan.node_end.size());
    P.pad = 0;
    // owned nodes: internal ids of this patch are one contiguous run
    int32_t omin = INT32_MAX, omax = -1, n_own = 0;
    loc_nodes.clear();
    for (int32_t i = pstart[p]; i < pstart[p + 1]; ++i) {
      const int32_t *en = &elems[int64_t(plan.elem_perm[i]) * npe];
      for (int a = 0; a < npe; ++a) {
        int32_t v = en[a];
        if (local[v] != -1) continue;
        local[v] = -2;  // seen
        loc_nodes.push_back(v);
        if (touches[v] == 1) {
          omin = std::min(omin, inv[v]);
          omax = std::max(omax, inv[v]);
          ++n_own;
        }
      }
    }
    if (n_own > 0 && omax - omin + 1 != n_own) return "internal error: owned run not contiguous";
    P.own_start = n_own > 0 ? omin : 0;
    P.n_own = n_own;
    int32_t n_sh = 0;
    for (int32_t v : loc_nodes) {
      if (touches[v] == 1) {
        local[v] = inv[v] - P.own_start;
      } else {
        local[v] = n_own + n_sh++;
        plan.sh_gid.push_back(inv[v]);
        int64_t j = inv[v] - plan.n_owned;
        plan.sh_slot.push_back(slot_next[j]++);
      }
    }
    P.n_sh = n_sh;
    const int32_t nloc = n_own + n_sh;
    if (nloc > pn_max) return "internal error: patch node overflow";
    plan.pn_used = std::max(plan.pn_used, int(nloc));
    plan.emax_used = std::max(plan.emax_used, int(P.n_elem));
    // packed ids + counts for the incidence lists
    cnt.assign(nloc, 0);
    for (int32_t i = pstart[p]; i < pstart[p + 1]; ++i) {
      const int32_t *en = &elems[int64_t(plan.elem_perm[i]) * npe];
      for (int a = 0; a < npe; ++a) {
        int32_t l = local[en[a]];
        plan.elem_lid[size_t(i) * 4 + a] = uint16_t(l);
        ++cnt[l];
        plan.elems_int[size_t(i) * npe + a] = inv[en[a]];
      }
    }
    // end offsets, then each (element, corner) entry's position in the
    // node-sorted order (within a node: by element, then corner)
    std::vector<int32_t> pos(nloc);
    int32_t run = 0;
    for (int32_t k = 0; k < nloc; ++k) {
      pos[k] = run;
      run += cnt[k];
      if (pad_runs) run = (run + 3) & ~3;
      plan.node_end.push_back(uint16_t(run));
    }
    if (run >= 16384) return "internal error: entry list above 14-bit positions";
    plan.ent_used = std::max(plan.ent_used, int(run));
    if (!pad_runs) {
      for (int32_t i = 0; i < P.n_elem; ++i)
        for (int a = 0; a < npe; ++a) {
          int32_t l = plan.elem_lid[size_t(P.elem_start + i) * 4 + a];
          plan.epos[size_t(P.elem_start + i) * 4 + a] = uint16_t(pos[l]++);
        }
    }
    for (int32_t v : loc_nodes) local[v] = -1;
  }
  if (!pad_runs) return "";
  // Patch by patch and most of the planning time: a context with the 64^3-hex
  // cube set up in 870 ms with this on one thread, in 228 ms on eight; the
  // 393,216-element column, which is planned twice, in 212 and 59 ms.
  std::atomic<bool> full{false};
  for_each_patch(np, [&] {
    return [&, bank = BankScratch()](int32_t p) mutable {
      const PatchInfo &P = plan.patches[p];
      const int32_t nloc = P.n_own + P.n_sh;
      const uint16_t *end = &plan.node_end[P.pnode_start];
      if (!spread_entry_banks(&plan.elem_lid[size_t(P.elem_start) * 4], &plan.epos[size_t(P.elem_start) * 4],
                              4, npe, P.n_elem, pn_max, end, nloc, end[nloc - 1], bank))
        full = true;
    };
  });
  return full ? "internal error: node run full" : "";
}

void pack_records(const MeshPlan &plan, std::vector<uint32_t> &rec) {
  rec.assign(size_t(plan.ne) * 3, 0u);
  for (int64_t e = 0; e < plan.ne; ++e) {
    uint32_t l[4] = {0, 0, 0, 0}, q[4] = {0, 0, 0, 0};
    for (int a = 0; a < plan.npe; ++a) {
      l[a] = plan.elem_lid[size_t(e) * 4 + a];
      q[a] = plan.epos[size_t(e) * 4 + a];
    }
    rec[size_t(e) * 3 + 0] = l[0] | l[1] << 10 | l[2] << 20 | (l[3] & 3u) << 30;
    rec[size_t(e) * 3 + 1] = l[3] >> 2 | q[0] << 8 | (q[1] & 1023u) << 22;
    rec[size_t(e) * 3 + 2] = q[1] >> 10 | q[2] << 4 | q[3] << 18;
  }
}

bool stride_records(const MeshPlan &plan, std::vector<uint32_t> &rec,
                    std::vector<uint32_t> &rec_s) {
  const size_t emax = size_t(plan.emax_used);
  bool regular = true;
  for (size_t p = 0; p < plan.patches.size(); ++p)
    regular = regular && size_t(plan.patches[p].elem_start) == p * emax;
  rec_s.clear();
  if (regular) {
    rec.resize(rec.size() + emax * 3, 0u);
    return true;
  }
  rec_s.assign(plan.patches.size() * emax * 3, 0u);
  for (size_t p = 0; p < plan.patches.size(); ++p)
    std::copy(rec.begin() + size_t(plan.patches[p].elem_start) * 3,
              rec.begin() + (size_t(plan.patches[p].elem_start) + plan.patches[p].n_elem) * 3,
              rec_s.begin() + p * emax * 3);
  return false;
}

void pack_patch_nodes(const MeshPlan &plan, int stride, std::vector<int32_t> &pgid,
                      std::vector<int32_t> &pslot, std::vector<uint16_t> &pend) {
  const size_t np = plan.patches.size();
  pgid.assign(np * size_t(stride), 0);
  pslot.assign(np * size_t(stride), 0);
  pend.assign(np * size_t(stride), 0);
  for (size_t p = 0; p < np; ++p) {
    const PatchInfo &Q = plan.patches[p];
    for (int k = 0; k < Q.n_own + Q.n_sh; ++k) {
      const size_t i = p * size_t(stride) + size_t(k);
      if (k < Q.n_own) {
        pgid[i] = Q.own_start + k;
      } else {
        const int32_t gid = plan.sh_gid[size_t(Q.sh_start + k - Q.n_own)];
        const int32_t slot = plan.sh_slot[size_t(Q.sh_start + k - Q.n_own)];
        const bool first = slot == plan.slot_start[size_t(gid - plan.n_owned)];
        pgid[i] = gid;
        pslot[i] = int32_t(uint32_t(slot) | (first ? 0x80000000u : 0u));
      }
      pend[i] = plan.node_end[size_t(Q.pnode_start + k)];
    }
  }
}

namespace {

// The strips of one patch: elements joined across shared faces (2D: edges).
struct StripScratch {
  std::vector<std::pair<uint32_t, int32_t>> face;  // hash table: key + 1, element * 4 + face
  std::vector<int32_t> adj;                        // 4 per element: neighbour * 4 + its face, or -1
  std::vector<uint8_t> used;
  std::vector<int32_t> deg, queue[5];              // free neighbours; elements by their number
  std::vector<int32_t> strip;                      // 3 elements per strip, -1: none
  std::vector<uint16_t> lid, epos, end;            // 6 per strip; per node
  std::vector<int32_t> cnt;
  BankScratch bank;
};

void strip_neighbours(const uint16_t *lid, int32_t n, int dim, StripScratch &S) {
  size_t size = 64;
  while (size < size_t(n) * 8) size *= 2;
  S.face.assign(size, {0u, 0});
  S.adj.assign(size_t(n) * 4, -1);
  for (int32_t e = 0; e < n; ++e)
    for (int f = 0; f <= dim; ++f) {  // the face opposite corner f
      uint32_t v[3] = {0, 0, 0};
      for (int a = 0, m = 0; a <= dim; ++a)
        if (a != f) v[m++] = lid[size_t(e) * 4 + a];
      if (v[0] > v[1]) std::swap(v[0], v[1]);
      if (dim == 3) {
        if (v[1] > v[2]) std::swap(v[1], v[2]);
        if (v[0] > v[1]) std::swap(v[0], v[1]);
      }
      const uint32_t key = (v[0] | v[1] << 10 | v[2] << 20) + 1;
      size_t h = (key * 2654435761u >> 8) & (size - 1);
      while (S.face[h].first && S.face[h].first != key) h = (h + 1) & (size - 1);
      if (!S.face[h].first) {
        S.face[h] = {key, e * 4 + f};
      } else if (S.face[h].second >= 0) {  // (of more than two elements at a face, the first two)
        S.adj[size_t(e) * 4 + f] = S.face[h].second;
        S.adj[size_t(S.face[h].second)] = e * 4 + f;
        S.face[h].second = -1;
      }
    }
}

// Greedy strips, each begun at an element with the fewest free neighbours (it is
// the first to be left alone) and continued to those with the fewest, among
// equals the nearest in the order; or (!by_degree) in the order and to the
// nearest.  The number of strips; S.strip: their elements, S.lid: their nodes.
int32_t find_strips(const uint16_t *lid, int32_t n, int dim, bool by_degree, StripScratch &S) {
  int32_t n_strips = 0;
  S.strip.clear();
  S.lid.clear();
  auto out = [&](const int32_t *el, const uint16_t *nd) {
    S.strip.insert(S.strip.end(), el, el + 3);
    S.lid.insert(S.lid.end(), nd, nd + 6);
    ++n_strips;
  };
  S.used.assign(size_t(n), 0);
  S.deg.assign(size_t(n), 0);
  for (auto &q : S.queue) q.clear();
  for (int32_t e = 0; e < n; ++e) {
    for (int f = 0; f <= dim; ++f) S.deg[e] += S.adj[size_t(e) * 4 + f] >= 0;
    S.queue[by_degree ? S.deg[e] : 0].push_back(e);
  }
  size_t at[5] = {0, 0, 0, 0, 0};
  // an element with the fewest free neighbours (entries may be out of date)
  auto pick = [&]() -> int32_t {
    for (int d = 0; d <= dim + 1; ++d)
      while (at[d] < S.queue[d].size()) {
        const int32_t e = S.queue[d][at[d]++];
        if (!S.used[e] && (!by_degree || S.deg[e] == d)) return e;
      }
    return -1;
  };
  auto use = [&](int32_t e) {
    S.used[e] = 1;
    for (int f = 0; f <= dim; ++f) {
      const int32_t a = S.adj[size_t(e) * 4 + f];
      if (a < 0 || S.used[a >> 2]) continue;
      const int32_t m = a >> 2;
      if (!by_degree) continue;
      S.queue[--S.deg[m]].push_back(m);
      at[S.deg[m]] = std::min(at[S.deg[m]], S.queue[S.deg[m]].size() - 1);
    }
  };
  // the face of e to the next element of its strip, or -1
  auto next = [&](int32_t e) {
    int best = -1, cost = INT32_MAX;
    for (int f = 0; f <= dim; ++f) {
      const int32_t a = S.adj[size_t(e) * 4 + f];
      if (a < 0 || S.used[a >> 2]) continue;
      const int c = (by_degree ? S.deg[a >> 2] * 65536 : 0) + std::abs((a >> 2) - e);
      if (c < cost) {
        cost = c;
        best = f;
      }
    }
    return best;
  };
  auto node = [&](int32_t e, int a) { return lid[size_t(e) * 4 + a]; };
  for (int32_t e; (e = pick()) >= 0;) {
    int32_t el[3] = {e, -1, -1};
    uint16_t nd[6] = {NO_NODE, NO_NODE, NO_NODE, NO_NODE, NO_NODE, NO_NODE};
    use(e);
    const int f0 = next(e);
    if (f0 < 0) {
      for (int a = 0; a <= dim; ++a) nd[a] = node(e, a);
      out(el, nd);
      continue;
    }
    const int32_t mid = S.adj[size_t(e) * 4 + f0] >> 2, f1 = S.adj[size_t(e) * 4 + f0] & 3;
    el[1] = mid;
    use(mid);
    const int f2 = next(mid);
    // nodes: the first element's own, those of both or all, the last one's own
    int m = 0;
    nd[m++] = node(e, f0);
    if (f2 >= 0) nd[m++] = node(mid, f2);
    for (int a = 0; a <= dim; ++a)
      if (a != f1 && a != f2) nd[m++] = node(mid, a);
    nd[m++] = node(mid, f1);
    if (f2 >= 0) {
      const int32_t C = S.adj[size_t(mid) * 4 + f2];
      el[2] = C >> 2;
      use(C >> 2);
      nd[m++] = node(C >> 2, C & 3);
    }
    out(el, nd);
  }
  return n_strips;
}

}  // namespace

bool build_strips(const MeshPlan &plan, int node_stride, int stride, StripPlan &x) {
  const size_t np = plan.patches.size();
  x = StripPlan();
  x.rec.assign(np * size_t(stride) * 4, 0u);
  x.rec2.assign(np * size_t(stride), 0u);
  x.pend.assign(np * size_t(node_stride), 0);
  x.elems.assign(np * size_t(stride) * STRIP_ELEMS, -1);
  std::vector<int32_t> n_strips(np), n_ent(np);
  std::atomic<bool> failed{false};
  for_each_patch(int32_t(np), [&] {
    return [&, S = StripScratch()](int32_t p) mutable {
      const PatchInfo &P = plan.patches[p];
      const int32_t nloc = P.n_own + P.n_sh;
      const size_t base = size_t(p) * stride;
      const uint16_t *lid = &plan.elem_lid[size_t(P.elem_start) * 4];
      strip_neighbours(lid, P.n_elem, plan.dim, S);
      // (in the order a regular grid divides without remainder; elsewhere by
      // degree leaves a tenth fewer strips)
      int32_t n = find_strips(lid, P.n_elem, plan.dim, false, S);
      if (n > (P.n_elem + 2) / 3) n = find_strips(lid, P.n_elem, plan.dim, true, S);
      n_strips[p] = n;
      if (n > stride) {
        failed = true;
        return;
      }
      for (int32_t s = 0; s < n; ++s) {
        uint32_t count = 0;
        for (int k = 0; k < STRIP_ELEMS; ++k)
          if (S.strip[size_t(s) * 3 + k] >= 0) {
            x.elems[(base + s) * 3 + k] = P.elem_start + S.strip[size_t(s) * 3 + k];
            ++count;
          }
        x.rec[(base + s) * 4] = count << 30;
      }
      S.cnt.assign(nloc, 0);
      for (uint16_t l : S.lid)
        if (l != NO_NODE) ++S.cnt[l];
      S.end.resize(nloc);
      int32_t run = 0;
      for (int32_t k = 0; k < nloc; ++k) {
        run = (run + S.cnt[k] + 3) & ~3;
        S.end[k] = x.pend[size_t(p) * node_stride + k] = uint16_t(run);
      }
      n_ent[p] = run;
      S.epos.assign(S.lid.size(), 0);
      if (!spread_entry_banks(S.lid.data(), S.epos.data(), 6, plan.dim + STRIP_ELEMS, n, stride,
                              S.end.data(), nloc, run, S.bank)) {
        failed = true;
        return;
      }
      for (int32_t s = 0; s < n; ++s) {
        uint32_t l[6], q[6];
        for (int a = 0; a < 6; ++a) {
          const uint16_t v = S.lid[size_t(s) * 6 + a];
          l[a] = v == NO_NODE ? 0u : v;
          q[a] = S.epos[size_t(s) * 6 + a];
        }
        uint32_t *r = &x.rec[(base + s) * 4];
        r[0] |= l[0] | l[1] << 10 | l[2] << 20;
        r[1] = l[3] | l[4] << 10 | l[5] << 20;
        r[2] = q[0] | q[1] << 14;
        r[3] = q[2] | q[3] << 14;
        x.rec2[base + s] = q[4] | q[5] << 14;
      }
    };
  });
  for (size_t p = 0; p < np; ++p) {
    x.strips_used = std::max(x.strips_used, int(n_strips[p]));
    x.ent_used = std::max(x.ent_used, int(n_ent[p]));
  }
  return !failed;
}

bool build_exchange(const MeshPlan &plan, ExchangePlan &x) {
  const size_t np = plan.patches.size();
  x = ExchangePlan();
  x.patches.assign(np, ExchangePatch{});
  x.src_end.assign(plan.sh_gid.size(), 0);
  x.own_pos.assign(plan.sh_gid.size(), 0);
  // the patch of every slot and the place that its node's first slot has there
  std::vector<int32_t> slot_patch(size_t(plan.n_slots)), slot_place(size_t(plan.n_slots));
  for (size_t p = 0; p < np; ++p) {
    const PatchInfo &Q = plan.patches[p];
    int32_t n = 0;
    for (int32_t i = Q.sh_start; i < Q.sh_start + Q.n_sh; ++i) {
      const size_t v = size_t(plan.sh_gid[size_t(i)] - plan.n_owned);
      const int32_t s = plan.sh_slot[size_t(i)], s0 = plan.slot_start[v];
      slot_patch[size_t(s)] = int32_t(p);
      slot_place[size_t(s)] = n;
      if (n + (plan.slot_start[v + 1] - s0) > 0xffff) return false;
      x.own_pos[size_t(i)] = uint16_t(n + (s - s0));
      n += plan.slot_start[v + 1] - s0;
      x.src_end[size_t(i)] = uint16_t(n);
    }
    x.n_src_max = std::max(x.n_src_max, int(n));
  }
  // senders in order: a receiver's entries come sender by sender
  struct Out {
    int32_t to, entry;  // receiver and its entry (receiver-local)
    uint16_t src, pos;  // places at the sender and at the receiver
  };
  std::vector<std::vector<Out>> out(np);
  for (size_t p = 0; p < np; ++p) {
    const PatchInfo &Q = plan.patches[p];
    for (int32_t i = Q.sh_start; i < Q.sh_start + Q.n_sh; ++i) {
      const size_t v = size_t(plan.sh_gid[size_t(i)] - plan.n_owned);
      const int32_t mine = plan.sh_slot[size_t(i)], s0 = plan.slot_start[v];
      for (int32_t s = s0; s < plan.slot_start[v + 1]; ++s)
        if (s != mine) {
          const size_t q = size_t(slot_patch[size_t(s)]);
          out[p].push_back({int32_t(q), x.patches[q].n_in++, x.own_pos[size_t(i)],
                            uint16_t(slot_place[size_t(s)] + (mine - s0))});
        }
    }
  }
  int64_t n_out = 0;
  for (size_t p = 0; p < np; ++p) {
    ExchangePatch &E = x.patches[p];
    E.in_start = int32_t(x.n_entries);
    E.out_start = int32_t(n_out);
    x.n_entries += (int64_t(E.n_in) + 63) & ~int64_t(63);
    n_out += E.n_in;  // (each node's patches send to each other: as many as received)
    if (x.n_entries > INT32_MAX / 64) return false;
    x.n_in_max = std::max(x.n_in_max, int(E.n_in));
  }
  x.out_entry.resize(size_t(n_out));
  x.out_src.resize(size_t(n_out));
  x.in_pos.resize(size_t(n_out));
  for (size_t p = 0; p < np; ++p) {
    std::stable_sort(out[p].begin(), out[p].end(),
                     [](const Out &a, const Out &b) { return a.to < b.to; });
    size_t k = size_t(x.patches[p].out_start);
    for (const Out &o : out[p]) {
      const ExchangePatch &R = x.patches[size_t(o.to)];
      x.out_entry[k] = uint32_t(R.in_start + o.entry);
      x.out_src[k] = o.src;
      x.in_pos[size_t(R.out_start + o.entry)] = o.pos;
      ++k;
    }
  }
  return true;
}

}  // namespace femgpu
