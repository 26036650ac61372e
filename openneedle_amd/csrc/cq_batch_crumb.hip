// The batch GEMV of cq_batch.h for 2-bit device codes (CQ2, ternary).
#include "cq_batch.h"

namespace nd {

void launch_cq_gemv_batch_crumb(const CqGeom &g, const CqJob &job0, const CqJob *jobs, int njobs, int blocks, int batch,
                                bool x_raw, hipStream_t s) {
    launch_kind<kCrumb>(g, job0, jobs, njobs, blocks, batch, x_raw, s);
}

}  // namespace nd
