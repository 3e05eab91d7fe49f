// pcg_batch_lean.hip -- the persistent kernels in their lean form (LEAN in
// pcg_persist.hpp): a file of its own, so that the two forms build in
// parallel.
#include "pcg_persist.hpp"

namespace pcg {

void launch_jobs_lean(const DevBatch *jobs, JobSlot *slots, int njobs, int prec, int block,
                      int nsteps, size_t lds_bytes, hipStream_t s) {
  launch_jobs_b<true>(jobs, slots, njobs, prec, block, nsteps, lds_bytes, s);
}

void launch_batch_lean(const DevBatch &b, int prec, int block, int nsteps, size_t lds_bytes,
                       hipStream_t s) {
  launch_batch_b<true>(b, prec, block, nsteps, lds_bytes, s);
}

} // namespace pcg
