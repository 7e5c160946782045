/* gemm_kq_wave4_k4.hip - the tiles of 128 rows (Q4_K, Q5_K, Q2_K): instances of gemm_kq_wave4.h */
#include "gemm_kq_wave4.h"

namespace qlin {
hipError_t wave4_q4k(const Wave4Call &c) { return wave4_format<FQ4K>(c); }
hipError_t wave4_q5k(const Wave4Call &c) { return wave4_format<FQ5K>(c); }
hipError_t wave4_q2k(const Wave4Call &c) { return wave4_format<FQ2K>(c); }
}  // namespace qlin
