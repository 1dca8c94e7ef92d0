// Forward-pass instances with dropout and 128-row blocks whose key tiles are
// split between wave pairs.
#include "fas_fwd.hpp"

namespace fas {

hipError_t launch_fwd_dropout_key_split(const FwdParams& p, int mode, int dtype, int d,
                                        hipStream_t s) {
  switch (mode) {
    case kFwdPlain: return launch_fwd_mode<kFwdPlain, 8, true, false, true>(p, dtype, d, s);
    case kFwdPlainKeepBits:
      return launch_fwd_mode<kFwdPlainKeepBits, 8, true, false, true>(p, dtype, d, s);
    case kFwdRowSum: return launch_fwd_mode<kFwdRowSum, 8, true, false, true>(p, dtype, d, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace fas
