// When (F)GMRES enqueues the next column's preconditioner and product before the host
// has read the current column's norm (host code only).
#pragma once

#include <cstdint>

#include "../../include/nalu_hip.h"

namespace nalu {

// The host decides from each column's norm whether to go on, and the device idles for
// that read (about 7 us) unless the next column is enqueued already.  That product is
// lost where the column turns out to be the last one, or is orthogonalized a second
// time, and then costs more than many reads.  So a column looks ahead only where
//  * a product is short: at most 2^20 unknowns.  Heat conduction, FP64, with and without
//    looking ahead: 10^3 1.75 and 1.90 ms, 32^3 4.61 and 4.96, 64^3 12.6 and 13.0; three
//    momentum solves 96^3 9.42 and 9.52 ms, 128^3 14.60 and 14.60.  Enqueuing every
//    column at 128^3 took 15.4 ms;
//  * the preconditioner is not a V-cycle of an FP32 solve, where nearly every column is
//    orthogonalized twice (64^3: 2.95 ms without, 3.48 ms with), nor the network, which
//    may end a cycle at any column;
//  * the residual, falling as it fell in the last column, stays above the target;
//  * the last column was not orthogonalized a second time.
struct LookAhead {
  bool allowed;
  double fall = 1.0;       // residual over that of the column before it
  bool cancelled = false;  // the last column took a second orthogonalization

  LookAhead(int64_t unknowns, int precond, bool fp32)
      : allowed(unknowns <= ((int64_t)1 << 20) && precond != NALU_PREC_LEARNED &&
                !(fp32 && precond == NALU_PREC_MUELU)) {}
  // for the column after one that starts from residual res
  bool operator()(double res, double target) const { return allowed && !cancelled && res * fall > target; }
};

}  // namespace nalu
