/* gemm_fewtok_k4.hip - the few-token product (Q4_K, Q5_K, Q2_K): instances of gemm_fewtok.h */
#include "gemm_fewtok.h"

namespace qlin {
hipError_t fewtok_q4k(const FewtokCall &c) { return fewtok_format<TQ4K>(c); }
hipError_t fewtok_q5k(const FewtokCall &c) { return fewtok_format<TQ5K>(c); }
hipError_t fewtok_q2k(const FewtokCall &c) { return fewtok_format<TQ2K>(c); }
}  // namespace qlin
