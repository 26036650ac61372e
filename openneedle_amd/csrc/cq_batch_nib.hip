// The batch GEMV of cq_batch.h for 4-bit device codes (CQ4, CQ3), and its entry point.
#include "cq_batch.h"

namespace nd {

void launch_cq_gemv_batch_crumb(const CqGeom &g, const CqJob &job0, const CqJob *jobs, int njobs, int blocks, int batch,
                                bool x_raw, hipStream_t s);

void launch_cq_gemv_batch(const CqGeom &g, const CqJob &job0, const CqJob *jobs, int njobs, int blocks, int batch,
                          bool x_raw, hipStream_t s) {
    if (g.kind == kNib) launch_kind<kNib>(g, job0, jobs, njobs, blocks, batch, x_raw, s);
    else launch_cq_gemv_batch_crumb(g, job0, jobs, njobs, blocks, batch, x_raw, s);
}

}  // namespace nd
