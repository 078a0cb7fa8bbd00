// The FP32 Coulomb kernels.
#include "flosic_coulomb_fp.h"

namespace flosic {

template void launch_frag_h<float>(const FpSegs &, const double *, int, int, float *, hipStream_t);
template void launch_coulomb_mfma<float>(const FpSegs &, const double4 *, const float *, const double *, const double *,
                                      const double *, int64_t, const double *, int, double *, int64_t, hipStream_t, int);
template void launch_coulomb_batch_all<float>(const CoulJob<float> *, const int64_t *, int, int64_t, const double *,
                                           hipStream_t);

}  // namespace flosic
