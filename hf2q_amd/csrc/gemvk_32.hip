// Instantiations of gemvk.h.
#include "gemvk.h"

namespace hq {

int launch_krows_q80(hipStream_t s, KRowsArgs& a, bool f32, uint32_t cus) { return launch_krows_t<HQ_Q8_0>(s, a, f32, cus); }
int launch_krows_q40(hipStream_t s, KRowsArgs& a, bool f32, uint32_t cus) { return launch_krows_t<HQ_Q4_0>(s, a, f32, cus); }

}  // namespace hq
