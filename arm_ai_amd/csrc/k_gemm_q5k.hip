// k_gemm_q5k.hip -- the Q5_K instances of the prefill GEMM (gemm_kq.h).
#include "gemm_kq.h"

namespace aq {

hipError_t launch_kq_q5k(const KqParams &p, int form, bool dump, hipStream_t s) {
    return kq::launch<TYPE_Q5_K>(p, form, dump, s);
}

}  // namespace aq
