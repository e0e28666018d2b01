// The exchange tables of a plan (build_exchange) as the resident kernels use
// them: every patch sends its contribution of every interface node to each
// other patch of the node, through entries written once and read once, and
// every patch ends with all contributions of its nodes in slot order.
// Usage: exchange_check <dim> <n> <elems_per_patch>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "femgpu_internal.h"
using namespace femgpu;
#define CHK(c) do { if (!(c)) { printf("FAIL %s line %d\n", #c, __LINE__); exit(1); } } while (0)

int main(int argc, char **argv) {
  const int dim = atoi(argv[1]), n = atoi(argv[2]), emax = atoi(argv[3]);
  (void)argc;
  std::vector<double> nodes;
  std::vector<int32_t> elems;
  const int N = n + 1;
  if (dim == 3) {
    for (int k = 0; k < N; ++k)
      for (int j = 0; j < N; ++j)
        for (int i = 0; i < N; ++i) nodes.insert(nodes.end(), {double(i), double(j), double(k)});
    const int perms[6][3] = {{0, 1, 2}, {0, 2, 1}, {1, 0, 2}, {1, 2, 0}, {2, 0, 1}, {2, 1, 0}};
    const int st[3] = {1, N, N * N};
    for (int k = 0; k < n; ++k)
      for (int j = 0; j < n; ++j)
        for (int i = 0; i < n; ++i)
          for (auto &p : perms) {
            const int v0 = i + N * (j + N * k), v1 = v0 + st[p[0]], v2 = v1 + st[p[1]];
            elems.insert(elems.end(), {v0, v1, v2, v2 + st[p[2]]});
          }
  } else {
    for (int j = 0; j < N; ++j)
      for (int i = 0; i < N; ++i) nodes.insert(nodes.end(), {double(i), double(j)});
    for (int j = 0; j < n; ++j)
      for (int i = 0; i < n; ++i) {
        const int a = i + N * j;
        elems.insert(elems.end(), {a, a + 1, a + N + 1, a, a + N + 1, a + N});
      }
  }
  const int64_t nn = int64_t(nodes.size()) / dim, ne = int64_t(elems.size()) / (dim + 1);
  MeshPlan P;
  CHK(build_plan(dim, nn, nodes.data(), ne, elems.data(), emax, 256, true, P).empty());
  ExchangePlan X;
  CHK(build_exchange(P, X));
  const size_t np = P.patches.size();
  CHK(X.patches.size() == np);
  // contributions: the slot number itself; entries start unwritten
  std::vector<int64_t> entry(size_t(X.n_entries) + 1, -1);
  std::vector<std::vector<int64_t>> place(np);
  for (size_t p = 0; p < np; ++p) {
    const PatchInfo &Q = P.patches[p];
    const int n_src = Q.n_sh ? X.src_end[size_t(Q.sh_start + Q.n_sh - 1)] : 0;
    CHK(n_src <= X.n_src_max && X.patches[p].n_in <= X.n_in_max);
    CHK(X.patches[p].n_in + Q.n_sh == n_src && X.patches[p].in_start % 64 == 0);
    place[p].assign(size_t(n_src) + 1, -1);
    for (int i = 0; i < Q.n_sh; ++i) place[p][X.own_pos[size_t(Q.sh_start + i)]] = P.sh_slot[size_t(Q.sh_start + i)];
  }
  for (size_t p = 0; p < np; ++p)
    for (int i = 0; i < X.patches[p].n_in; ++i) {
      const uint32_t e = X.out_entry[size_t(X.patches[p].out_start + i)];
      const uint16_t s = X.out_src[size_t(X.patches[p].out_start + i)];
      CHK(int64_t(e) < X.n_entries && s < place[p].size() && place[p][s] >= 0 && entry[e] < 0);
      entry[e] = place[p][s];
    }
  for (size_t p = 0; p < np; ++p)
    for (int i = 0; i < X.patches[p].n_in; ++i) {
      const size_t e = size_t(X.patches[p].in_start + i), at = X.in_pos[size_t(X.patches[p].out_start + i)];
      CHK(int64_t(e) < X.n_entries && entry[e] >= 0 && at < place[p].size() && place[p][at] < 0);
      place[p][at] = entry[e];
    }
  for (size_t p = 0; p < np; ++p) {
    const PatchInfo &Q = P.patches[p];
    size_t l = 0;
    for (int i = 0; i < Q.n_sh; ++i) {
      const size_t v = size_t(P.sh_gid[size_t(Q.sh_start + i)] - P.n_owned);
      for (int s = P.slot_start[v]; s < P.slot_start[v + 1]; ++s, ++l) CHK(place[p][l] == s);
      CHK(l == X.src_end[size_t(Q.sh_start + i)]);
    }
  }
  printf("ok: %zu patches, %ld entries, at most %d in and %d places\n", np, long(X.n_entries), X.n_in_max, X.n_src_max);
  return 0;
}
