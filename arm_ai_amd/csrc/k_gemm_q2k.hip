// k_gemm_q2k.hip -- the Q2_K instances of the prefill GEMM (gemm_kq.h).
#include "gemm_kq.h"

namespace aq {

hipError_t launch_kq_q2k(const KqParams &p, int form, bool dump, hipStream_t s) {
    return kq::launch<TYPE_Q2_K>(p, form, dump, s);
}

}  // namespace aq
