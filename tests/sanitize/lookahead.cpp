// The look-ahead of (F)GMRES (lookahead.hpp) over residual histories, as gmres_t applies
// it: a column that converges, or is orthogonalized a second time, discards the product
// enqueued with it.  A steady fall discards none and looks ahead at every column but the
// last; one that reaches the target a column early discards one; systems past the size,
// V-cycles of FP32 solves and the network never look ahead.  Exit status 0 means clean.
#include <cmath>
#include <cstdio>
#include <vector>

#include "../../nalu_amd/csrc/lookahead.hpp"

struct Count {
  int columns, ahead, lost;
};

// res[k]: residual after column k (1 before the first); twice[k]: column k is orthogonalized a second time
static Count run(nalu::LookAhead look, const std::vector<double>& res, double target, const std::vector<int>& twice = {}) {
  Count c{0, 0, 0};
  double r = 1.0;
  for (size_t k = 0; k < res.size(); ++k) {
    ++c.columns;
    const bool ahead = look(r, target);
    c.ahead += ahead;
    look.cancelled = k < twice.size() && twice[k];
    if (ahead && (look.cancelled || res[k] <= target)) ++c.lost;
    look.fall = res[k] / r;
    r = res[k];
    if (r <= target) break;
  }
  return c;
}

static int g_fail = 0;
static void expect(const char* what, const Count& c, int ahead, int lost) {
  if (c.ahead == ahead && c.lost == lost) return;
  std::fprintf(stderr, "lookahead: %s: %d ahead, %d lost of %d columns, expected %d and %d\n", what, c.ahead, c.lost,
               c.columns, ahead, lost);
  g_fail = 1;
}

int main() {
  const int64_t small = 1 << 20;
  for (double f : {0.15, 0.5, 0.9}) {
    std::vector<double> res;
    for (int k = 1; k <= 400; ++k) res.push_back(std::pow(f, k));
    const double target = 1.0001e-8;  // no column lands on it
    const int n = (int)std::ceil(std::log(target) / std::log(f));
    expect("steady fall", run({small, NALU_PREC_SGS, false}, res, target), n - 1, 0);
    expect("steady fall, FP32", run({small, NALU_PREC_JACOBI, true}, res, target), n - 1, 0);
    expect("steady fall, V-cycle", run({small, NALU_PREC_MUELU, false}, res, target), n - 1, 0);
    expect("too large", run({small + 1, NALU_PREC_SGS, false}, res, target), 0, 0);
    expect("V-cycle, FP32", run({small, NALU_PREC_MUELU, true}, res, target), 0, 0);
    expect("network", run({small, NALU_PREC_LEARNED, true}, res, target), 0, 0);
  }
  expect("one column", run({small, NALU_PREC_SGS, false}, {1e-9}, 1e-8), 1, 1);
  expect("sudden end", run({small, NALU_PREC_SGS, false}, {0.5, 0.25, 1e-9}, 1e-8), 3, 1);
  expect("second pass", run({small, NALU_PREC_SGS, true}, {0.5, 0.25, 0.125, 0.0625, 0.03}, 1e-8, {0, 1, 1, 0, 0}), 3, 1);
  if (!g_fail) std::printf("lookahead: ok\n");
  return g_fail;
}
