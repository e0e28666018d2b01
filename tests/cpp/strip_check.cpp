// The strips of a plan (build_strips) as the strip kernels use them: every element
// lies in one strip of its patch, element k of a strip has its nodes
// k .. k + dim, and every strip node has an entry of its own in its node's run.
// Usage: strip_check <dim> <n> <elems_per_patch> [shuffle]
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <set>
#include <vector>

#include "femgpu_internal.h"
using namespace femgpu;
#define CHK(c) do { if (!(c)) { printf("FAIL %s line %d\n", #c, __LINE__); exit(1); } } while (0)

int main(int argc, char **argv) {
  const int dim = atoi(argv[1]), n = atoi(argv[2]), emax = atoi(argv[3]);
  std::vector<double> nodes;
  std::vector<int32_t> elems;
  const int N = n + 1;
  const bool jitter = argc > 4;  // nodes and elements in no order
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
  if (jitter) {
    unsigned long long z = 12345;
    auto rnd = [&] { return double((z = z * 6364136223846793005ull + 1442695040888963407ull) >> 33) / 2147483648.0; };
    for (double &v : nodes) v += 0.5 * rnd() - 0.25;
    for (int64_t e = 0; e < ne; ++e)
      for (int a = dim; a > 0; --a)
        std::swap(elems[size_t(e * (dim + 1) + a)], elems[size_t(e * (dim + 1)) + size_t(rnd() * (a + 1))]);
  }
  const int threads = 256, stride = 320;
  MeshPlan P;
  CHK(build_plan(dim, nn, nodes.data(), ne, elems.data(), emax, threads, true, P).empty());
  StripPlan S;
  CHK(build_strips(P, threads, stride, S));
  const size_t np = P.patches.size();
  std::vector<int> seen(size_t(ne), 0);
  int most = 0;
  size_t total = 0;
  for (size_t p = 0; p < np; ++p) {
    const PatchInfo &Q = P.patches[p];
    std::set<int> taken;
    int n_strips = 0;
    for (int s = 0; s < stride; ++s) {
      const uint32_t *r = &S.rec[(p * stride + size_t(s)) * 4], r2 = S.rec2[p * stride + size_t(s)];
      const int count = int(r[0] >> 30);
      if (!count) {
        CHK(!r[0] && !r[1] && !r[2] && !r[3] && !r2);
        continue;
      }
      CHK(s == n_strips);
      ++n_strips;
      const int l[6] = {int(r[0] & 1023), int(r[0] >> 10 & 1023), int(r[0] >> 20 & 1023),
                        int(r[1] & 1023), int(r[1] >> 10 & 1023), int(r[1] >> 20 & 1023)};
      const int q[6] = {int(r[2] & 16383), int(r[2] >> 14), int(r[3] & 16383),
                        int(r[3] >> 14), int(r2 & 16383), int(r2 >> 14)};
      for (int k = 0; k < 3; ++k) {
        const int e = S.elems[(p * stride + size_t(s)) * 3 + size_t(k)];
        CHK((e >= 0) == (k < count));
        if (e < 0) continue;
        CHK(e >= Q.elem_start && e < Q.elem_start + Q.n_elem);
        ++seen[size_t(e)];
        std::set<int> a, b;
        for (int c = 0; c <= dim; ++c) {
          a.insert(P.elem_lid[size_t(e) * 4 + size_t(c)]);
          b.insert(l[k + c]);
        }
        CHK(a == b && int(a.size()) == dim + 1);
      }
      for (int m = 0; m < count + dim; ++m) {
        CHK(l[m] < Q.n_own + Q.n_sh);
        const int b0 = l[m] ? S.pend[p * threads + size_t(l[m]) - 1] : 0, b1 = S.pend[p * threads + size_t(l[m])];
        CHK(q[m] >= b0 && q[m] < b1 && b1 <= S.ent_used && b0 % 4 == 0 && b1 % 4 == 0);
        CHK(taken.insert(q[m]).second);
      }
    }
    CHK(n_strips >= (Q.n_elem + 2) / 3);
    most = std::max(most, n_strips);
    total += size_t(n_strips);
  }
  CHK(most == S.strips_used);
  for (int v : seen) CHK(v == 1);
  printf("ok: %zu patches, %.2f elements per strip\n", np, double(ne) / double(total));
  return 0;
}
