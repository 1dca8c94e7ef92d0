// Dispatch of the forward pass to its per-mode translation units.
#include "fas_launch.hpp"

namespace fas {

hipError_t launch_fwd_plain(const FwdParams& p, int dtype, int d, hipStream_t s);
hipError_t launch_fwd_rowsum(const FwdParams& p, int dtype, int d, hipStream_t s);
hipError_t launch_fwd_scores(const FwdParams& p, int dtype, int d, hipStream_t s);
hipError_t launch_fwd_scores_unaligned(const FwdParams& p, int dtype, int d, hipStream_t s);
hipError_t launch_fwd_region(const FwdParams& p, int dtype, int d, hipStream_t s);
hipError_t launch_fwd_key_split(const FwdParams& p, int mode, int dtype, int d, hipStream_t s);
hipError_t launch_fwd_few(const FwdParams& p, int dtype, int d, hipStream_t s);
hipError_t launch_fwd_dropout(const FwdParams& p, int mode, int dtype, int d, hipStream_t s);
hipError_t launch_fwd_packed(const FwdParams& p, int mode, int dtype, int d, hipStream_t s);
hipError_t launch_fwd_scores_packed(const FwdParams& p, int dtype, int d, hipStream_t s);

// GQA-packed launches (p.pack > 1) take their own instances; the host never
// packs a launch with dropout.
hipError_t launch_fwd(const FwdParams& p, int mode, int dtype, int d, hipStream_t s) {
  // Row blocks below 256: the unpacked score writer without dropout (128 and
  // 64 rows) and, without a key split over workgroups, the plain and row-sum
  // modes (128 rows).
  if (p.bm != kFwdRows) {
    if (mode == kFwdScores
            ? p.dropout || p.pack != 1 || (p.bm != kFwdRows / 2 && p.bm != kFwdRows / 4)
            : mode == kFwdRegion || mode == kFwdFewRows || p.bm != kFwdRows / 2 || p.nsplit != 1)
      return hipErrorInvalidValue;
    if (mode != kFwdScores && !p.dropout) return launch_fwd_key_split(p, mode, dtype, d, s);
  }
  if (mode == kFwdFewRows) return launch_fwd_few(p, dtype, d, s);
  if (mode == kFwdScores && !p.scores_aligned) {
    if (p.pack > 1 && p.dropout) return hipErrorInvalidValue;
    return launch_fwd_scores_unaligned(p, dtype, d, s);
  }
  if (p.pack > 1) {
    if (p.dropout && mode != kFwdRegion) return hipErrorInvalidValue;
    return mode == kFwdScores ? launch_fwd_scores_packed(p, dtype, d, s)
                              : launch_fwd_packed(p, mode, dtype, d, s);
  }
  if (p.dropout && mode != kFwdRegion) return launch_fwd_dropout(p, mode, dtype, d, s);
  switch (mode) {
    case kFwdPlain: return launch_fwd_plain(p, dtype, d, s);
    case kFwdRowSum: return launch_fwd_rowsum(p, dtype, d, s);
    case kFwdScores: return launch_fwd_scores(p, dtype, d, s);
    case kFwdRegion: return launch_fwd_region(p, dtype, d, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace fas
