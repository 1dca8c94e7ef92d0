// Forward-pass instances with 128-row blocks whose key tiles are split
// between wave pairs: plain output (+ base-2 LSE) and per-row sums, one head
// or several packed heads per workgroup.
#include "fas_fwd.hpp"

namespace fas {

hipError_t launch_fwd_key_split(const FwdParams& p, int mode, int dtype, int d, hipStream_t s) {
  if (mode == kFwdPlain)
    return p.pack > 1 ? launch_fwd_mode<kFwdPlain, 8, false, true, true>(p, dtype, d, s)
                      : launch_fwd_mode<kFwdPlain, 8, false, false, true>(p, dtype, d, s);
  if (mode == kFwdRowSum)
    return p.pack > 1 ? launch_fwd_mode<kFwdRowSum, 8, false, true, true>(p, dtype, d, s)
                      : launch_fwd_mode<kFwdRowSum, 8, false, false, true>(p, dtype, d, s);
  return hipErrorInvalidValue;
}

}  // namespace fas
