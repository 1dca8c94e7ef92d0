// Stand-ins for the kernel launchers: each appends one line with the launch's
// plan to a log that the test reads, and launches nothing.
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdio>
#include <string>

#include "fas_launch.hpp"

static std::string g_log, g_taken;

static hipError_t log_line(const char* fmt, ...) {
  char line[256];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(line, sizeof line, fmt, ap);
  va_end(ap);
  g_log += line;
  g_log += '\n';
  return hipSuccess;
}

extern "C" const char* plan_log_take() {
  g_taken = g_log;
  g_log.clear();
  return g_taken.c_str();
}

// A device and its scratch array for the entry point that allocates nothing.
extern "C" hipError_t hipGetDevice(int* device) {
  *device = 0;
  return hipSuccess;
}
extern "C" hipError_t hipGetSymbolAddress(void** ptr, const void*) {
  *ptr = reinterpret_cast<void*>(0x2000000);
  return hipSuccess;
}

namespace fas {

hipError_t launch_fwd(const FwdParams& p, int mode, int, int, hipStream_t) {
  return log_line("fwd mode=%d bm=%d nrb=%d pack=%d nsplit=%d tps=%d kept=%d aligned=%d", mode, p.bm,
                  p.nrb, p.pack, p.nsplit, p.tps, p.few != nullptr, p.scores_aligned);
}
hipError_t launch_few_cols(const FwdParams& p, int, int, hipStream_t) {
  return log_line("few_cols nsplit=%d", p.nsplit);
}
hipError_t launch_colsm(const ColsmParams& p, int, int, bool buffered, hipStream_t) {
  return log_line("colsm fold=%d nsplit=%d buffered=%d dropout=%d", p.fold, p.nsplit, buffered,
                  p.dropout);
}
hipError_t launch_rawsum(const RawParams& p, int, bool suffix, hipStream_t) {
  return log_line("rawsum nblk=%d suffix=%d", p.nblk, suffix);
}
hipError_t launch_bwd(const BwdParams& p, int, int, hipStream_t) {
  return log_line("bwd pieces=%d ds=%d", p.pieces, p.ds != nullptr);
}
hipError_t launch_scores(const ScoresParams& p, int, int, hipStream_t) {
  return log_line("scores ngrp=%d nkb=%d nrs=%d pshift=%d mask=%d aligned=%d", p.ngrp, p.nkb, p.nrs,
                  p.pshift, p.mask, p.aligned);
}
hipError_t launch_fill_zero(float*, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t,
                            hipStream_t) {
  return log_line("fill_zero");
}

}  // namespace fas
