/* gemm_f32_split_b32.hip - the fp32 product on split activations (Q4_0, IQ4_NL, IQ4_XS): instances of gemm_f32_split.h */
#include "gemm_f32_split.h"

namespace qlin {
hipError_t f32_split_q4_0(const F32SplitCall &c) { return split_format<TQ4_0, T_Q4_0>(c); }
hipError_t f32_split_iq4nl(const F32SplitCall &c) { return split_format<TIQ4NL, T_IQ4_NL>(c); }
hipError_t f32_split_iq4xs(const F32SplitCall &c) { return split_format<TIQ4XS, T_IQ4_XS>(c); }
}  // namespace qlin
