// Score-writer instances for score rows that do not all start on 64-byte
// boundaries (odd key counts).
#include "fas_fwd.hpp"

namespace fas {

hipError_t launch_fwd_scores_unaligned(const FwdParams& p, int dtype, int d, hipStream_t s) {
  if (p.pack > 1) return launch_fwd_mode<kFwdScores, 8, false, true, false, false>(p, dtype, d, s);
  if (p.dropout) return launch_fwd_mode<kFwdScores, 8, true, false, false, false>(p, dtype, d, s);
  if (p.bm == 64) return launch_fwd_mode<kFwdScores, 4, false, false, true, false>(p, dtype, d, s);
  if (p.bm == 128)
    return launch_fwd_mode<kFwdScores, 8, false, false, true, false>(p, dtype, d, s);
  if (p.bm != 256) return hipErrorInvalidValue;
  return launch_fwd_mode<kFwdScores, 8, false, false, false, false>(p, dtype, d, s);
}

}  // namespace fas
