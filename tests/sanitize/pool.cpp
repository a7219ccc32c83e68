// The pool of device memory that a system keeps (DevPool), without a GPU: hipMalloc,
// hipFree and hipDeviceSynchronize are replaced here by malloc, free and a counter.
// A block that was returned may still be in use on any stream the system was on since
// it was taken, so the first scope after a change of stream has to wait for the device,
// also when the system is back on the stream of the last scope (A, B, A); while the
// stream stays the same, no scope waits.  Exit status 0 means clean.
#include <cstdio>
#include <cstdlib>

#include "../../nalu_amd/csrc/internal.hpp"

static int g_waits = 0, g_fail = 0;
extern "C" hipError_t hipMalloc(void** p, size_t n) {
  *p = std::malloc(n);
  return *p ? hipSuccess : hipErrorOutOfMemory;
}
extern "C" hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
extern "C" hipError_t hipDeviceSynchronize(void) {
  ++g_waits;
  return hipSuccess;
}

// waits of one scope that takes a block and returns it
static int scope_waits(nalu_linsys* ls) {
  const int before = g_waits;
  nalu::PoolScope scope(ls->pool);
  nalu::DevBuf<int> b(1000);
  return g_waits - before;
}
static void expect(const char* what, int got, int want) {
  if (got == want) return;
  std::fprintf(stderr, "pool: %s: %d waits, expected %d\n", what, got, want);
  g_fail = 1;
}

int main() {
  int a, b;  // stand for two streams
  nalu_solver_config cfg{};
  cfg.method = NALU_METHOD_CG;
  cfg.precond = NALU_PREC_SGS;
  cfg.max_iterations = 1;
  cfg.kspace = 1;
  nalu_linsys* ls = nullptr;
  if (nalu_linsys_create(1, &cfg, &ls) != NALU_OK) return 1;
  nalu_linsys_set_stream(ls, &a);
  expect("first scope", scope_waits(ls), 0);
  expect("same stream", scope_waits(ls), 0);
  nalu_linsys_set_stream(ls, &a);
  expect("same stream set again", scope_waits(ls), 0);
  nalu_linsys_set_stream(ls, &b);
  nalu_linsys_set_stream(ls, &a);
  expect("A, B, A", scope_waits(ls), 1);
  expect("after it", scope_waits(ls), 0);
  nalu_linsys_set_stream(ls, &b);
  expect("A, B", scope_waits(ls), 1);
  nalu_linsys_set_stream(ls, nullptr);  // destroy synchronizes the stream it is on
  nalu_linsys_destroy(ls);
  if (!g_fail) std::printf("pool: ok\n");
  return g_fail;
}
