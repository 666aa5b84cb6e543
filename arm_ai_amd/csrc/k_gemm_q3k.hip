// k_gemm_q3k.hip -- the Q3_K instances of the prefill GEMM (gemm_kq.h).
#include "gemm_kq.h"

namespace aq {

hipError_t launch_kq_q3k(const KqParams &p, int form, bool dump, hipStream_t s) {
    return kq::launch<TYPE_Q3_K>(p, form, dump, s);
}

}  // namespace aq
