/* gemm_f32_split_k6.hip - the fp32 product on split activations (Q6_K, Q3_K, Q8_0): instances of gemm_f32_split.h */
#include "gemm_f32_split.h"

namespace qlin {
hipError_t f32_split_q6k(const F32SplitCall &c) { return split_format<TQ6K, T_Q6_K>(c); }
hipError_t f32_split_q3k(const F32SplitCall &c) { return split_format<TQ3K, T_Q3_K>(c); }
hipError_t f32_split_q8_0(const F32SplitCall &c) { return split_format<TQ8_0, T_Q8_0>(c); }
}  // namespace qlin
