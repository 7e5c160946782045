/* gemm_fewtok_k6.hip - the few-token product (Q6_K, Q3_K): instances of gemm_fewtok.h */
#include "gemm_fewtok.h"

namespace qlin {
hipError_t fewtok_q6k(const FewtokCall &c) { return fewtok_format<TQ6K>(c); }
hipError_t fewtok_q3k(const FewtokCall &c) { return fewtok_format<TQ3K>(c); }
}  // namespace qlin
