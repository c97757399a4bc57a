// Instantiations of gemvk.h.
#include "gemvk.h"

namespace hq {

int launch_krows_q6k(hipStream_t s, KRowsArgs& a, bool f32, uint32_t cus) { return launch_krows_t<HQ_Q6_K>(s, a, f32, cus); }

}  // namespace hq
