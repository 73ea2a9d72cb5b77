// FP64 instantiations of the hop kernels (RB = 1): many right-hand sides go to
// the t-marching one (wc_hop_march.h).
#include "wc_hop.h"
#include "wc_hop_march.h"
#include "wc_hop_split.h"

namespace wck {
template <> bool hop_march_applies<double>(const HopLaunch &a) { return march_applies<double>(a); }
template <> bool hop_split_applies<double>(const HopLaunch &a) { return split_applies<double>(a); }
template <> bool hop<double>(const HopLaunch &a, hipStream_t s) {
  if (split_applies<double>(a)) return hop_split<double>(a, s);
  return march_applies<double>(a) ? hop_march<double>(a, s) : hop_launch<double>(a, s);
}
}  // namespace wck
