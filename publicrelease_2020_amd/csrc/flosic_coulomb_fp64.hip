// The FP64 Coulomb kernels.
#include "flosic_coulomb_fp.h"

namespace flosic {

int64_t fp_steps(const FpSegs &seg) { return seg_step0(seg, 5); }

template void launch_frag_h<double>(const FpSegs &, const double *, int, int, double *, hipStream_t);
template void launch_coulomb_mfma<double>(const FpSegs &, const double4 *, const double *, const double *, const double *,
                                      const double *, int64_t, const double *, int, double *, int64_t, hipStream_t, int);
template void launch_coulomb_batch_all<double>(const CoulJob<double> *, const int64_t *, int, int64_t, const double *,
                                           hipStream_t);

}  // namespace flosic
