/* gemm_fewtok_b32.hip - the few-token product (Q8_0, Q4_0, IQ4_NL): instances of gemm_fewtok.h */
#include "gemm_fewtok.h"

namespace qlin {
hipError_t fewtok_q8_0(const FewtokCall &c) { return fewtok_format<TQ8_0>(c); }
hipError_t fewtok_q4_0(const FewtokCall &c) { return fewtok_format<TQ4_0>(c); }
hipError_t fewtok_iq4nl(const FewtokCall &c) { return fewtok_format<TIQ4NL>(c); }
}  // namespace qlin
