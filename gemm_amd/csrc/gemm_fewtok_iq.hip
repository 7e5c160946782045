/* gemm_fewtok_iq.hip - the few-token product (IQ4_XS, IQ3_S, IQ2_XXS): instances of gemm_fewtok.h */
#include "gemm_fewtok.h"

namespace qlin {
hipError_t fewtok_iq4xs(const FewtokCall &c) { return fewtok_format<TIQ4XS>(c); }
hipError_t fewtok_iq3s(const FewtokCall &c) { return fewtok_format<TIQ3S>(c); }
hipError_t fewtok_iq2xxs(const FewtokCall &c) { return fewtok_format<TIQ2XXS>(c); }
}  // namespace qlin
