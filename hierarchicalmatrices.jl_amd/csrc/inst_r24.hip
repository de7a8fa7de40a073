// inst_r24.hip -- kernels for ranks in bucket 24 (r <= 24).
#include "nested1.h"

hipError_t hmx_matvec_r24(const DevPlan &p, const MvArgs &a, bool tr, int mode, int kb,
                          hipStream_t s, const hipEvent_t *ev) {
    return hmxk::matvec_r<double, 24>(p, a, tr, mode, kb, s, ev);
}

hipError_t hmx_grad_r24(const DevPlan &p, const MvArgs &a, bool tr, double *y2, int64_t incy2,
                        const double *sv, int64_t incs, hipStream_t s) {
    return hmxk::grad_r<double, 24>(p, a, tr, y2, incy2, sv, incs, s);
}

hipError_t hmx_gen_basis_r24(const DevPlan &p, hipStream_t s) { return hmxk::gen_basis_r<double, 24>(p, s); }

hipError_t hmx_matvec_m_r24(const DevPlan &p, const MvArgs &a, int mode, int prec, int nq,
                            hipStream_t s) {
    return hmxk::matvec_m_r<32>(p, a, mode, prec, nq, s);
}

hipError_t hmx_matvec_n1_r24(const DevPlan &p, const MvArgs &a, bool tr, int src, int nq,
                           hipStream_t s, const hipEvent_t *ev) {
    return hmxk::matvec_n1<double, 24>(p, a, tr, src, nq, s, ev);
}
