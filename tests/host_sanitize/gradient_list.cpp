// Host-sanitizer driver of the gradient list and the plans made from it (test
// infrastructure; see the Makefile beside this file).  With HOST_ONLY it needs
// no GPU: the list's definition, entry by entry, its refusals, and the host
// stage of gradient plans over the whole list, parts of it and an empty one.
// Without, it runs the entry points end to end and holds the reduced list's
// gradient to the one of every (i, j, k >= l).  Any sanitizer finding aborts;
// a failed check exits with 1.  Prints "gradient_list ok" at the end.
#include <hip/hip_runtime.h>
#include <sanitizer/lsan_interface.h>
#include <unistd.h>

#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <tuple>
#include <algorithm>
#include <vector>

#include "../../libcint_amd/csrc/host_internal.h"
#include "mcint.h"
#include "synth_basis.h"

namespace {

using synth::SynthBasis;

void expect(long long got, long long want, const char* what) {
  if (got == want) return;
  std::fprintf(stderr, "FAIL %s: got %lld, expected %lld (%s)\n", what, got, want, mcint_last_error());
  std::exit(1);
}

struct List {
  std::vector<int> shls, refs;
  size_t n = 0;
};

// The list, checked against its definition.
List gradient_list(const mcint_basis* b, const SynthBasis& B) {
  List L;
  expect(mcint_gradient_list(b, nullptr, nullptr, 0, &L.n), MCINT_OK, "count");
  L.shls.resize(4 * L.n);
  L.refs.resize(L.n);
  size_t n = 0;
  expect(mcint_gradient_list(b, L.shls.data(), L.refs.data(), L.n, &n), MCINT_OK, "list");
  expect((long long)n, (long long)L.n, "entries");
  auto atom = [&](int s) { return B.bas[8 * s]; };
  // one reference atom per unordered quartet, one of its own
  std::map<std::vector<int>, int> ref;
  std::map<std::tuple<int, int, int, int>, int> seen;
  for (size_t q = 0; q < n; ++q) {
    const int* s = &L.shls[4 * q];
    expect(s[2] >= s[3], 1, "k >= l");
    expect(atom(s[0]) != L.refs[q], 1, "no derivative on the reference atom");
    std::vector<int> bra = {std::min(s[0], s[1]), std::max(s[0], s[1])}, ket = {s[3], s[2]};
    std::vector<int> key = std::min(bra, ket), hi = std::max(bra, ket);
    key.insert(key.end(), hi.begin(), hi.end());
    const auto it = ref.emplace(key, L.refs[q]).first;
    expect(it->second, L.refs[q], "the same reference atom in every order");
    expect(seen.emplace(std::make_tuple(s[0], s[1], s[2], s[3]), 0).second, 1, "listed once");
  }
  // every ordered quartet is listed unless it differentiates its reference atom
  long long want = 0;
  for (int i = 0; i < B.nbas; ++i)
    for (int j = 0; j < B.nbas; ++j)
      for (int k = 0; k < B.nbas; ++k)
        for (int l = 0; l <= k; ++l) {
          std::vector<int> bra = {std::min(i, j), std::max(i, j)}, ket = {l, k};
          std::vector<int> key = std::min(bra, ket), hi = std::max(bra, ket);
          key.insert(key.end(), hi.begin(), hi.end());
          const auto it = ref.find(key);
          if (it == ref.end()) {  // never listed: all four shells on one atom
            expect(atom(i) == atom(j) && atom(j) == atom(k) && atom(k) == atom(l), 1, "unlisted quartet");
            continue;
          }
          expect(it->second == atom(i) || it->second == atom(j) || it->second == atom(k) || it->second == atom(l), 1,
                 "the reference is one of the quartet's atoms");
          want += it->second != atom(i);
        }
  expect((long long)n, want, "every other derivative is listed");
  if (L.n) {
    expect(mcint_gradient_list(b, L.shls.data(), L.refs.data(), L.n - 1, &n), MCINT_ERR_ARG, "a list too short");
    expect(mcint_gradient_list(b, nullptr, L.refs.data(), L.n, &n), MCINT_ERR_ARG, "no shells");
    expect(mcint_gradient_list(b, L.shls.data(), nullptr, L.n, &n), MCINT_ERR_ARG, "no references");
  }
  expect(mcint_gradient_list(b, nullptr, nullptr, 0, nullptr), MCINT_ERR_ARG, "no count");
  expect(mcint_gradient_list(nullptr, nullptr, nullptr, 0, &n), MCINT_ERR_ARG, "no basis");
  return L;
}

#ifdef HOST_ONLY
void run(const SynthBasis& B) {
  mcint_basis* b = nullptr;
  expect(mcint::basis_create_host_only(&b, B.atm.data(), B.natm, B.bas.data(), B.nbas, B.env.data()), MCINT_OK,
         "basis");
  const List L = gradient_list(b, B);
  std::vector<uint8_t> flags(L.n + 1);
  for (size_t q = 0; q < L.n; ++q) flags[q] = q % 3 == 0;
  for (size_t first : {(size_t)0, L.n / 3, L.n}) {
    long long tasks = 0;
    for (size_t q = first; q < L.n; ++q) {
      long long t = 1;
      for (int c = 0; c < 4; ++c) t *= B.bas[8 * L.shls[4 * q + c] + 3];
      tasks += t;
    }
    for (const uint8_t* f : {(const uint8_t*)nullptr, (const uint8_t*)flags.data()}) {
      int64_t st[6];
      expect(mcint::gradient_plan_host_only(b, L.shls.data() + 4 * first, L.refs.data() + first, L.n - first, f, st),
             MCINT_OK, "gradient plan");
      expect(st[0], tasks, "tasks of a gradient plan");
    }
  }
  if (L.n) {
    int64_t st[6];
    for (int bad : {-2, B.natm}) {
      std::vector<int> refs = L.refs;
      refs.back() = bad;
      expect(mcint::gradient_plan_host_only(b, L.shls.data(), refs.data(), L.n, nullptr, st), MCINT_ERR_ARG,
             "a reference that is no atom");
    }
    expect(mcint::gradient_plan_host_only(b, L.shls.data(), nullptr, L.n, nullptr, st), MCINT_ERR_ARG, "no references");
  }
  mcint_basis_destroy(b);
  std::printf("  %d atoms, %d shells: %zu entries\n", B.natm, B.nbas, L.n);
}
#else
void hipcheck(hipError_t e, const char* what) { expect(e, hipSuccess, what); }

void run(const SynthBasis& B) {
  mcint_basis* b = nullptr;
  expect(mcint_basis_create(&b, B.atm.data(), B.natm, B.bas.data(), B.nbas, B.env.data()), MCINT_OK, "basis");
  const List L = gradient_list(b, B);
  const int nao = synth::nao_sph(B), ng = 3 * B.natm;
  std::vector<double> dm((size_t)nao * nao);
  for (int i = 0; i < nao; ++i)
    for (int j = 0; j < nao; ++j) dm[(size_t)i * nao + j] = std::cos(0.7 * (i + 1) * (j + 1)) / (1.0 + std::abs(i - j));
  double *dm_d = nullptr, *g_d = nullptr, *out_d = nullptr;
  hipcheck(hipMalloc(&dm_d, sizeof(double) * dm.size()), "density");
  hipcheck(hipMalloc(&g_d, sizeof(double) * ng), "gradient");
  hipcheck(hipMalloc(&out_d, 1 << 20), "blocks");
  hipcheck(hipMemcpy(dm_d, dm.data(), sizeof(double) * dm.size(), hipMemcpyHostToDevice), "density");
  auto gradient = [&](mcint_plan* p) {
    std::vector<double> g(ng, 0.0);
    hipcheck(hipMemcpy(g_d, g.data(), sizeof(double) * ng, hipMemcpyHostToDevice), "zero");
    expect(mcint_plan_execute_grad(p, dm_d, nao, g_d, nullptr), MCINT_OK, "execute_grad");
    hipcheck(hipMemcpy(g.data(), g_d, sizeof(double) * ng, hipMemcpyDeviceToHost), "gradient");
    return g;
  };
  std::vector<int> all;
  for (int i = 0; i < B.nbas; ++i)
    for (int j = 0; j < B.nbas; ++j)
      for (int k = 0; k < B.nbas; ++k)
        for (int l = 0; l <= k; ++l) all.insert(all.end(), {i, j, k, l});
  mcint_plan* p = nullptr;
  int64_t osz = 0;
  expect(mcint_plan_create(&p, b, MCINT_INT2E_IP1_SPH, all.data(), all.size() / 4, nullptr, &osz), MCINT_OK, "full");
  const std::vector<double> want = gradient(p);
  mcint_plan_destroy(p);
  expect(mcint_plan_create_gradient(&p, b, L.shls.data(), L.refs.data(), L.n, nullptr), MCINT_OK, "gradient plan");
  const std::vector<double> got = gradient(p);
  double big = 1.0;
  for (double v : want) big = std::max(big, std::fabs(v));
  // one atom's list is empty: nothing is added (the full list's sum there is
  // the rounding of terms that cancel)
  for (int i = 0; i < ng; ++i)
    expect(L.n ? std::fabs(got[i] - want[i]) <= 1e-10 * big : got[i] == 0.0, 1, "reduced and full gradient");
  // such a plan stores no blocks, by no route (the buffer is real)
  if (L.n) {
    expect(mcint_plan_execute(p, out_d, nullptr, nullptr), MCINT_ERR_ARG, "stored blocks");
    expect(mcint_plan_execute_direct(p, out_d, nullptr, nullptr), MCINT_ERR_ARG, "stored blocks, direct");
    expect(mcint_plan_execute_bucket(p, 0, out_d, nullptr, nullptr), MCINT_ERR_ARG, "stored blocks, one bucket");
    expect(mcint_plan_execute_noalloc(p, out_d, nullptr, nullptr), MCINT_ERR_ARG, "stored blocks, no-alloc");
  }
  mcint_plan_destroy(p);
  expect(mcint_plan_create_gradient(&p, b, nullptr, nullptr, 0, nullptr), MCINT_OK, "empty list");
  for (double v : gradient(p)) expect(v == 0.0, 1, "the empty list's gradient");
  mcint_plan_destroy(p);
  hipcheck(hipDeviceSynchronize(), "wait");
  hipcheck(hipFree(dm_d), "free");
  hipcheck(hipFree(g_d), "free");
  hipcheck(hipFree(out_d), "free");
  mcint_basis_destroy(b);
  std::printf("  %d atoms, %d shells: %zu entries, |g| up to %.3g\n", B.natm, B.nbas, L.n, big);
}
#endif

}  // namespace

int main() {
  for (int natm : {1, 2, 3}) run(synth::make_basis(natm, 0.0, 5 + natm));
  run(synth::make_basis(2, 0.3, 11));
  std::fflush(stdout);
  __lsan_do_leak_check();
  std::printf("gradient_list ok\n");
  std::fflush(stdout);
  std::fflush(stderr);
  _exit(0);  // without the ROCm runtime's exit-time teardown (plan_sanitize.cpp)
}
