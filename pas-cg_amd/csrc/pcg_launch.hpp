// pcg_launch.hpp -- launchers of the grid-wide stage kernels (pcg_kernels.hip)
// and of the persistent batched kernel (pcg_batch.hip).
#pragma once
#include "pcg_kernels.hpp"

namespace pcg {
void launch_begin(const DevBatch &b, hipStream_t s);
// forces, energies and wall reactions to zero before an evaluation outside a step
void launch_eval_begin(const DevBatch &b, hipStream_t s);
// the FP64 force accumulators into FP32 force arrays
void launch_store_forces(const DevBatch &b, hipStream_t s);
// and back
void launch_load_forces(const DevBatch &b, hipStream_t s);
// completes near lists of the persistent kernel for the stage kernels
void launch_near_fields(const DevBatch &b, hipStream_t s);
void launch_mark_invalid(const DevBatch &b, hipStream_t s);
// device data into mapped pinned host memory: bytes of src as words, and three
// columns of n values (FP32 or FP64) as FP64 triples; then seq into flag. acc
// (with f32): the columns are forces still in these accumulators, n of each
// component, and are stored on the way.
struct Fetch {
  const void *src = nullptr;
  void *dst = nullptr;
  size_t bytes = 0;
  const void *cols[3] = {nullptr, nullptr, nullptr};
  bool f32 = false;
  const double *acc = nullptr;
  int n = 0;
  double *out = nullptr;
  int *flag = nullptr;  // null: no flag
  int seq = 0;
};
void launch_fetch(const Fetch &f, hipStream_t s);
// the host's noise of one step into the device's
void launch_noise_in(const DevBatch &b, const double *src, hipStream_t s);
void launch_prepare_nh(const DevBatch &b, hipStream_t s);
// The list rebuild of every system that needs one. step: the first kernels of
// a full step, which also take the verify decision, clear the forces and
// energies and (qa_on) compute n and h; else the systems marked invalid, and
// the rebuild is closed here.
void launch_fix_nl(const DevBatch &b, int max_n, int cell_words, hipStream_t s, bool step,
                   int qa_on);
// and its launches in a step
int fix_nl_launches(int max_n, int cell_words);
// every term, of a step or (step false) of an evaluation outside one
void launch_step_terms(const DevBatch &b, int prec, int max_n, bool step, hipStream_t s);
// a single term outside a step
void launch_terms(const DevBatch &b, int prec, int max_items, int term, int from, int to,
                  hipStream_t s);
void launch_qa_finish(const DevBatch &b, int max_n, hipStream_t s);
// tick: the step's k_tick (advance, close a rebuild) by the wave that
// completes each system, log: after the wall forces' log of the box protocol
// noise: RAN2 draws in host memory, or null for those on the device
void launch_lang(const DevBatch &b, int prec, int noise_mode, const double *noise, hipStream_t s,
                 bool tick = false, bool log = false);
void launch_tick(const DevBatch &b, int advance, hipStream_t s);
// walls and the box protocol of a plain context (b.wall set): LJ candidate
// processing; box set-up, and the phase logic before a step. P and sd are the
// writable device parameters and system descriptor.
void launch_ljw_process(const DevBatch &b, hipStream_t s);
void launch_box_setup(const DevBatch &b, DevParams *P, SysDesc *sd, hipStream_t s);
void launch_box_phase(const DevBatch &b, DevParams *P, SysDesc *sd, hipStream_t s);
// persistent form: every system of the batch advances nsteps in one launch;
// lean: the lean kernels (pcg_batch_lean.hip), for batches lean_batch allows
void launch_persistent(const DevBatch &b, bool lean, int prec, int block, int nsteps,
                       size_t lds_bytes, hipStream_t s);
void launch_persistent_jobs(const DevBatch *jobs, JobSlot *slots, int njobs, bool lean, int prec,
                            int block, int nsteps, size_t lds_bytes, hipStream_t s);
void launch_batch_lean(const DevBatch &b, int prec, int block, int nsteps, size_t lds_bytes,
                       hipStream_t s);
void launch_jobs_lean(const DevBatch *jobs, JobSlot *slots, int njobs, int prec, int block,
                      int nsteps, size_t lds_bytes, hipStream_t s);
// report sums of every system (pcg_report.hip)
void launch_report(const DevBatch &b, int pid_on, ReportSums *out, hipStream_t s);
// the same into the library's own device array (no allocation), for batches
// of at most REPORT_STATIC_MAX systems, with `device` current: 0, or -1 for
// too many systems, -2 for a device index beyond the library's table, -3 for
// a HIP failure
constexpr int REPORT_STATIC_MAX = 4096;
int report_static_sums(const DevBatch &b, int device, int pid_on, hipStream_t s,
                       ReportSums **sums);
} // namespace pcg
