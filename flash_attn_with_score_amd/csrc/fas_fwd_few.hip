// Forward-pass instances for at most 32 query rows per KV head that keep the
// scores of every key, and their second pass.
#include "fas_fwd.hpp"
#include "fas_launch.hpp"

namespace fas {

hipError_t launch_fwd_few(const FwdParams& p, int dtype, int d, hipStream_t s) {
  if (p.pack != p.G || (int64_t)p.G * p.M > kFwdFewMax || p.dropout) return hipErrorInvalidValue;
  return p.pack > 1 ? launch_fwd_mode<kFwdFewRows, 8, false, true>(p, dtype, d, s)
                    : launch_fwd_mode<kFwdFewRows, 8>(p, dtype, d, s);
}

template <class E, int D>
static hipError_t few_cols_t(const FwdParams& p, hipStream_t s) {
  const int64_t nblk = (p.M + 2048 / D - 1) / (2048 / D);
  const int64_t ncombine = p.nsplit > 1 ? nblk * p.B * p.H : 0;
  const int64_t grid = ncombine + (int64_t)p.B * (p.H / p.G) * ((p.N + 1023) / 1024);
  if (grid > INT32_MAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL((few_cols_kernel<E, D>), dim3((unsigned)grid), dim3(256), 0, s, p,
                     (int)ncombine);
  return hipGetLastError();
}

hipError_t launch_few_cols(const FwdParams& p, int dtype, int d, hipStream_t s) {
  switch (d) {
    case 16: return dtype == 0 ? few_cols_t<F16, 16>(p, s) : few_cols_t<BF16, 16>(p, s);
    case 32: return dtype == 0 ? few_cols_t<F16, 32>(p, s) : few_cols_t<BF16, 32>(p, s);
    case 64: return dtype == 0 ? few_cols_t<F16, 64>(p, s) : few_cols_t<BF16, 64>(p, s);
    case 128: return dtype == 0 ? few_cols_t<F16, 128>(p, s) : few_cols_t<BF16, 128>(p, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace fas
