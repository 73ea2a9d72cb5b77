// FP64 instantiations of the hop kernels (RB = 1): many right-hand sides go to
// the t-marching one (wc_hop_march.h).
#include "wc_hop.h"
#include "wc_hop_march.h"

namespace wck {
template <> bool hop_march_applies<double>(const HopLaunch &a) { return march_applies<double>(a); }
template <> bool hop<double>(const HopLaunch &a, hipStream_t s) {
  return march_applies<double>(a) ? hop_march<double>(a, s) : hop_launch<double>(a, s);
}
}  // namespace wck
