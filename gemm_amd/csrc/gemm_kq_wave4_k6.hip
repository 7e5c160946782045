/* gemm_kq_wave4_k6.hip - the tiles of 128 rows (Q6_K, Q3_K): instances of gemm_kq_wave4.h */
#include "gemm_kq_wave4.h"

namespace qlin {
hipError_t wave4_q6k(const Wave4Call &c) { return wave4_format<FQ6K>(c); }
hipError_t wave4_q3k(const Wave4Call &c) { return wave4_format<FQ3K>(c); }
}  // namespace qlin
