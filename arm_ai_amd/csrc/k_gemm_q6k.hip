// k_gemm_q6k.hip -- the Q6_K instances of the prefill GEMM (gemm_kq.h).
#include "gemm_kq.h"

namespace aq {

hipError_t launch_kq_q6k(const KqParams &p, int form, bool dump, hipStream_t s) {
    return kq::launch<TYPE_Q6_K>(p, form, dump, s);
}

}  // namespace aq
