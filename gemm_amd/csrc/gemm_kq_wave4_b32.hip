/* gemm_kq_wave4_b32.hip - the tiles of 128 rows (Q8_0, Q4_0): instances of gemm_kq_wave4.h */
#include "gemm_kq_wave4.h"

namespace qlin {
hipError_t wave4_q8_0(const Wave4Call &c) { return wave4_format<FQ8_0>(c); }
hipError_t wave4_q4_0(const Wave4Call &c) { return wave4_format<FQ4_0>(c); }
}  // namespace qlin
