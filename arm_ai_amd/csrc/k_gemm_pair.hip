// k_gemm_pair.hip -- two K-quant weights on one activation in one launch of
// the prefill GEMM (gemm_kq.h): llama's wq|wk and wv.
#include "gemm_kq.h"

namespace aq {

hipError_t launch_kq_pair(const KqParams &p1, const KqParams &p2, int type2, hipStream_t s) {
    const int b1 = p1.per_xcd * kq::NXCD, b2 = p2.per_xcd * kq::NXCD;
    if (type2 == TYPE_Q6_K) kq::pair_kernel<TYPE_Q6_K><<<(unsigned)(b1 + b2), 256, 0, s>>>(p1, p2, b1);
    else if (type2 == TYPE_Q5_K) kq::pair_kernel<TYPE_Q5_K><<<(unsigned)(b1 + b2), 256, 0, s>>>(p1, p2, b1);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace aq
