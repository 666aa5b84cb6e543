// k_gemm_q4k.hip -- the Q4_K instances of the prefill GEMM (gemm_kq.h).
#include "gemm_kq.h"

namespace aq {

hipError_t launch_kq_q4k(const KqParams &p, int form, bool dump, hipStream_t s) {
    return kq::launch<TYPE_Q4_K>(p, form, dump, s);
}

}  // namespace aq
