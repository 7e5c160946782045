/* gemm_f32_split_iq.hip - the fp32 product on split activations (IQ3_S, IQ2_XXS): instances of gemm_f32_split.h */
#include "gemm_f32_split.h"

namespace qlin {
hipError_t f32_split_iq3s(const F32SplitCall &c) { return split_format<TIQ3S, T_IQ3_S>(c); }
hipError_t f32_split_iq2xxs(const F32SplitCall &c) { return split_format<TIQ2XXS, T_IQ2_XXS>(c); }
}  // namespace qlin
