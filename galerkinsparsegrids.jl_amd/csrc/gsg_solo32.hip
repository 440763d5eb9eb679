// gsg_solo32.hip -- the resident small-solve kernel, FP32 operator (gsg_solo.hpp)
#include "gsg_solo.hpp"

namespace gsg {

template <int D, int K>
static hipError_t solo32_dk(bool segr, const SoloArgs& a, int nsolve, int threads, int lds_bytes, hipStream_t s) {
  if constexpr (solo_shape_ok(D, K)) {
    if constexpr (seg_ok(D, K) && seg_cpw(D, K) > 1) {
      if (segr) return solo::launch_one<D, K, float, true>(a, nsolve, threads, lds_bytes, s);
    }
    if (segr) return hipErrorInvalidValue;
    return solo::launch_one<D, K, float, false>(a, nsolve, threads, lds_bytes, s);
  }
  return hipErrorInvalidValue;
}

template <int D>
static hipError_t solo32_d(int K, bool segr, const SoloArgs& a, int nsolve, int threads, int lds_bytes,
                           hipStream_t s) {
  switch (K) {
    case 1: return solo32_dk<D, 1>(segr, a, nsolve, threads, lds_bytes, s);
    case 2: return solo32_dk<D, 2>(segr, a, nsolve, threads, lds_bytes, s);
    case 3: return solo32_dk<D, 3>(segr, a, nsolve, threads, lds_bytes, s);
    case 4: return solo32_dk<D, 4>(segr, a, nsolve, threads, lds_bytes, s);
    case 5: return solo32_dk<D, 5>(segr, a, nsolve, threads, lds_bytes, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_solo32(int D, int K, bool segr, const SoloArgs& a, int nsolve, int threads, int lds_bytes,
                         hipStream_t s) {
  switch (D) {
    case 1: return solo32_d<1>(K, segr, a, nsolve, threads, lds_bytes, s);
    case 2: return solo32_d<2>(K, segr, a, nsolve, threads, lds_bytes, s);
    case 3: return solo32_d<3>(K, segr, a, nsolve, threads, lds_bytes, s);
    case 4: return solo32_d<4>(K, segr, a, nsolve, threads, lds_bytes, s);
    case 5: return solo32_d<5>(K, segr, a, nsolve, threads, lds_bytes, s);
    case 6: return solo32_d<6>(K, segr, a, nsolve, threads, lds_bytes, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace gsg
