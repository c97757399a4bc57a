// Instantiations of gemvk.h.
#include "gemvk.h"

namespace hq {

int launch_krows_q4k(hipStream_t s, KRowsArgs& a, bool f32, uint32_t cus) { return launch_krows_t<HQ_Q4_K>(s, a, f32, cus); }
int launch_krows_q5k(hipStream_t s, KRowsArgs& a, bool f32, uint32_t cus) { return launch_krows_t<HQ_Q5_K>(s, a, f32, cus); }

}  // namespace hq
