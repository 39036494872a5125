// GPU test driver: plans of the force phase and the adjoint when the device
// has room for the coarse cut of the lists but not for the finer one that
// short lists take.  The program defines hipMalloc itself (the library's
// calls bind to it): it passes requests on, and refuses those above a limit
// that the program sets, as a full device does.  Prints a line per step.
#include <dlfcn.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "hacc_sr.h"

static size_t g_limit = 0;  // 0: none
static int g_refused = 0;

extern "C" int hipMalloc(void **p, size_t bytes) {
  using Fn = int (*)(void **, size_t);
  static Fn real = (Fn)dlsym(RTLD_NEXT, "hipMalloc");
  if (g_limit && bytes > g_limit) {
    ++g_refused;
    *p = nullptr;
    return 2;  // hipErrorOutOfMemory
  }
  return real(p, bytes);
}

static int fails = 0;
static void expect(bool ok, const char *what) {
  printf("%s: %s%s\n", what, ok ? "ok" : "FAILED ", ok ? "" : hsr_last_error());
  fflush(stdout);
  if (!ok) ++fails;
}

static double rel(const std::vector<float> &a, const std::vector<float> &b) {
  double d = 0, s = 0;
  for (size_t i = 0; i < a.size(); ++i) {
    d += ((double)a[i] - b[i]) * ((double)a[i] - b[i]);
    s += (double)b[i] * b[i];
  }
  return std::sqrt(d / s);
}

int main() {
  const int64_t n = 20000;
  const float box = 10.f;
  std::vector<float> a[8];
  for (auto &v : a) v.assign(n, 0.f);
  unsigned long long r = 7;
  for (int k = 0; k < 3; ++k)
    for (int64_t i = 0; i < n; ++i) {
      r = r * 6364136223846793005ull + 1442695040888963407ull;
      a[k][i] = box * (float)((r >> 40) * (1.0 / 16777216.0));
    }
  a[6].assign(n, 1.f);  // masses
  std::vector<int64_t> id(n, 0);
  std::vector<uint16_t> mask(n, 0);
  hsr_params p = {};
  p.tdpts = 1;
  p.law = HSR_LAW_STEP16;
  p.nd = 64;
  p.ds = 2;
  p.tmin = 128;
  p.fsrrmax = 3.12f;
  p.rsm = 0.1f;
  p.oa = 0.1f;
  p.tan_oa = tanf(0.1f);
  p.ppc = 0.9f;
  hsr_ctx *c = nullptr;
  if (hsr_create(&c, &p)) {
    printf("%s\n", hsr_last_error());
    return 2;
  }
  const float lo[3] = {0, 0, 0}, hi[3] = {box, box, box}, flo[3] = {-1, -1, -1},
              fhi[3] = {box + 1, box + 1, box + 1};
  hsr_tuning t;
  auto chunk = [&](int entries) {
    hsr_get_tuning(c, &t);
    t.chunk = entries;
    return hsr_set_tuning(c, &t) == HSR_OK;
  };
  std::vector<float> F[3], G[3], f[3], g[3], l[3];
  for (int k = 0; k < 3; ++k) {
    for (auto *v : {&F[k], &G[k], &f[k], &g[k]}) v->assign(n, 0.f);
    l[k].resize(n);
    for (int64_t i = 0; i < n; ++i) l[k][i] = (float)((i * 37 + k * 11) % 101) * 0.01f - 0.5f;
  }
  auto forces = [&](std::vector<float> *o) {
    return hsr_forces(c, o[0].data(), o[1].data(), o[2].data(), HSR_HOST_PTRS) == HSR_OK;
  };
  auto adjoint = [&](std::vector<float> *o) {
    return hsr_adjoint(c, l[0].data(), l[1].data(), l[2].data(), o[0].data(), o[1].data(), o[2].data(),
                       HSR_HOST_PTRS) == HSR_OK;
  };
  // the coarse cut: every buffer but the finer plan's is there afterwards
  expect(chunk(8192), "coarse cut set");
  expect(hsr_build(c, n, a[0].data(), a[1].data(), a[2].data(), a[3].data(), a[4].data(), a[5].data(),
                   a[6].data(), a[7].data(), id.data(), mask.data(), lo, hi, HSR_HOST_PTRS) == HSR_OK &&
             hsr_lists(c, flo, fhi) == HSR_OK,
         "build and lists");
  expect(forces(F) && adjoint(G), "forces and adjoint with the coarse cut");
  // 1e-5 and 1e-4: the tolerances of the force and of the adjoint
  g_limit = 1 << 20;
  expect(chunk(0), "plan of the force phase without room for the finer cut");
  expect(g_refused > 0, "an allocation was refused");
  expect(forces(f) && rel(f[0], F[0]) < 1e-5 && rel(f[2], F[2]) < 1e-5, "its forces");
  g_limit = 0;
  expect(chunk(8192) && chunk(0) && forces(f) && rel(f[1], F[1]) < 1e-5, "forces with the finer cut");
  g_refused = 0;
  g_limit = 1 << 20;
  expect(adjoint(g), "adjoint without room for the finer cut");
  expect(g_refused > 0, "an allocation was refused");
  expect(rel(g[0], G[0]) < 1e-4 && rel(g[1], G[1]) < 1e-4 && rel(g[2], G[2]) < 1e-4, "its gradient");
  hsr_destroy(c);
  // no room at all: an error, and the context goes on when there is room
  int64_t kept = 0;
  expect(hsr_release_buffers(0, &kept) == HSR_OK && kept > 0, "kept buffers released");
  c = nullptr;
  expect(hsr_create(&c, &p) == HSR_OK, "another context");
  auto build = [&] {
    return hsr_build(c, n, a[0].data(), a[1].data(), a[2].data(), a[3].data(), a[4].data(), a[5].data(),
                     a[6].data(), a[7].data(), id.data(), mask.data(), lo, hi, HSR_HOST_PTRS) == HSR_OK &&
           hsr_lists(c, flo, fhi) == HSR_OK;
  };
  g_limit = 1;
  expect(!build(), "no room for the build");
  g_limit = 0;
  // (the arrays are in tree order now: the same tree, its particles as they lie)
  expect(build() && forces(f) && rel(f[0], F[0]) < 1e-5, "build, lists and forces afterwards");
  hsr_destroy(c);
  printf("%d failed\n", fails);
  return fails ? 1 : 0;
}
