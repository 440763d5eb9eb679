// gsg_solo64.hip -- the resident small-solve kernel, FP64 (gsg_solo.hpp)
#include "gsg_solo.hpp"

namespace gsg {

template <int D>
static hipError_t solo64_d(int K, const SoloArgs& a, int nsolve, int threads, int lds_bytes, hipStream_t s) {
#define GSG_SOLO(KK)                                                                                   \
  case KK:                                                                                             \
    if constexpr (solo_shape_ok(D, KK)) return solo::launch_one<D, KK, double, false>(a, nsolve, threads, lds_bytes, s); \
    return hipErrorInvalidValue;
  switch (K) {
    GSG_SOLO(1) GSG_SOLO(2) GSG_SOLO(3) GSG_SOLO(4) GSG_SOLO(5)
    default: return hipErrorInvalidValue;
  }
#undef GSG_SOLO
}

hipError_t launch_solo(int D, int K, bool fp32, bool segr, const SoloArgs& a, int nsolve, int threads, int lds_bytes,
                       hipStream_t s) {
  if (nsolve <= 0 || a.nsteps <= 0) return hipSuccess;
  if (threads <= 0 || threads > SOLO_MAXT || threads % 64 || lds_bytes > SOLO_LDS) return hipErrorInvalidValue;
  if (fp32) return launch_solo32(D, K, segr, a, nsolve, threads, lds_bytes, s);
  switch (D) {
    case 1: return solo64_d<1>(K, a, nsolve, threads, lds_bytes, s);
    case 2: return solo64_d<2>(K, a, nsolve, threads, lds_bytes, s);
    case 3: return solo64_d<3>(K, a, nsolve, threads, lds_bytes, s);
    case 4: return solo64_d<4>(K, a, nsolve, threads, lds_bytes, s);
    case 5: return solo64_d<5>(K, a, nsolve, threads, lds_bytes, s);
    case 6: return solo64_d<6>(K, a, nsolve, threads, lds_bytes, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace gsg
