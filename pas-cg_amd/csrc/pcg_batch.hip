// pcg_batch.hip -- the persistent kernels in their general form (every term of
// the force field), and the launchers that choose between it and the lean
// form.
#include "pcg_persist.hpp"

namespace pcg {

void launch_persistent_jobs(const DevBatch *jobs, JobSlot *slots, int njobs, bool lean, int prec,
                            int block, int nsteps, size_t lds_bytes, hipStream_t s) {
  if (lean) launch_jobs_lean(jobs, slots, njobs, prec, block, nsteps, lds_bytes, s);
  else launch_jobs_b<false>(jobs, slots, njobs, prec, block, nsteps, lds_bytes, s);
}

void launch_persistent(const DevBatch &b, bool lean, int prec, int block, int nsteps,
                       size_t lds_bytes, hipStream_t s) {
  if (lean) launch_batch_lean(b, prec, block, nsteps, lds_bytes, s);
  else launch_batch_b<false>(b, prec, block, nsteps, lds_bytes, s);
}

} // namespace pcg
