// CPU check, under AddressSanitizer / UBSan, of the batch buffers that grow
// with the number of frequencies: solve and backward of one batch at several
// sizes, and with allocations that fail (the library's own ed_batch.hip on the
// device emulation, as batch_check.cpp).
//
// Arguments: a script of steps run on one batch of two small models,
//   sN  solve with N frequencies       b   backward
//   fN  the N-th allocation from here (0 = the next) fails; with kK before it,
//       and the K - 1 after it
//   z   solve with 3 frequencies, the last of them zero (refused)
// Output: "solve rc" / "grad rc v..." per step.
#include <fstream>
#include <string>

#include <hip/hip_runtime.h>

static long g_fail_in = -1, g_fail_count = 1;
template <class T>
static hipError_t counted_malloc(T** p, size_t n) {
  if (g_fail_in == 0) {
    if (--g_fail_count == 0) g_fail_in = -1;
    return hipErrorOutOfMemory;
  }
  if (g_fail_in > 0) --g_fail_in;
  return hipMalloc(p, n);
}
#define hipMalloc counted_malloc
#include "cmpy_amd/csrc/ed_batch.cpp"

namespace ed {
int set_error(int code, const char*, ...) { return code; }
void clear_error() {}
}  // namespace ed

int main(int argc, char** argv) {
  const int M = 2, mb = 2;
  const int32_t nb[M] = {1, 2}, nu[M] = {1, 1}, nd[M] = {1, 1};
  const double u[M] = {2.0, 3.0}, ei[M] = {-1.0, -1.5}, eb[M * mb] = {0.3, 0.0, -0.4, 0.7},
               v[M * mb] = {0.5, 0.0, 0.6, 0.9};
  ed_batch_desc d{};
  d.num_models = M;
  d.num_bath = nb;
  d.n_up = nu;
  d.n_dn = nd;
  d.u = u;
  d.eps_imp = ei;
  d.eps_bath = eb;
  d.v = v;
  d.max_bath = mb;
  d.max_iter = 40;
  d.cf_steps = 16;
  d.check_every = 8;
  d.keep_basis = 1;
  d.tol = 1e-10;
  d.seed = 0x5EED;
  d.cf_tol = 1e-13;
  ed_batch* b = nullptr;
  if (ed_batch_create(&b, &d, nullptr) != ED_OK || ed_batch_config(b, -1, 2, 0, nullptr) != ED_OK) return 1;
  int nw = 0;
  for (int i = 1; i < argc; ++i) {
    const char op = argv[i][0];
    const long n = std::atol(argv[i] + 1);
    if (op == 'f') g_fail_in = n;
    if (op == 'k') g_fail_count = n;
    if (op == 's' || op == 'z') {
      const int k = op == 'z' ? 3 : (int)n;
      std::vector<double> wn(k), g(2 * M * k);
      for (int q = 0; q < k; ++q) wn[q] = (2 * q + 1) * M_PI / 10.0;
      if (op == 'z') wn[k - 1] = 0.0;
      const int rc = ed_batch_solve(b, wn.data(), k, nullptr, g.data(), nullptr, nullptr, nullptr, nullptr);
      if (rc == ED_OK) nw = k;
      std::printf("solve %d\n", rc);
    }
    if (op == 'b') {  // gradients of the exact size that the last solve asks for
      std::vector<double> dre(M * nw, 1.0), dim(M * nw, 0.5), ge(M * mb, 0.0), gv(M * mb, 0.0);
      const int rc = ed_batch_backward(b, dre.data(), dim.data(), ge.data(), gv.data(), nullptr, nullptr, nullptr);
      std::printf("grad %d", rc);
      for (int m = 0; m < M; ++m)
        for (int k = 0; k < nb[m]; ++k) std::printf(" %.17g %.17g", ge[m * mb + k], gv[m * mb + k]);
      std::printf("\n");
    }
  }
  std::fflush(stdout);
  ed_batch_destroy(b);
  emu::release_fibers();
  return 0;
}
