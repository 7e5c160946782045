/* gemm_f32_split_k4.hip - the fp32 product on split activations (Q4_K, Q5_K, Q2_K): instances of gemm_f32_split.h */
#include "gemm_f32_split.h"

namespace qlin {
hipError_t f32_split_q4k(const F32SplitCall &c) { return split_format<TQ4K, T_Q4_K>(c); }
hipError_t f32_split_q5k(const F32SplitCall &c) { return split_format<TQ5K, T_Q5_K>(c); }
hipError_t f32_split_q2k(const F32SplitCall &c) { return split_format<TQ2K, T_Q2_K>(c); }
}  // namespace qlin
