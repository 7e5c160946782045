/* gemm_kq_wave4_iq.hip - the tiles of 128 rows (IQ4_NL, IQ4_XS): instances of gemm_kq_wave4.h */
#include "gemm_kq_wave4.h"

namespace qlin {
hipError_t wave4_iq4nl(const Wave4Call &c) { return wave4_format<FIQ4NL>(c); }
hipError_t wave4_iq4xs(const Wave4Call &c) { return wave4_format<FIQ4XS>(c); }
}  // namespace qlin
