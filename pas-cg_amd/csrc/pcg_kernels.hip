// pcg_kernels.hip -- grid-wide kernels of the per-step loop and their
// launchers. Each stage of thread::advance_by_step
// (cg/src/cg/simul/thread_main.cpp:373-536) is one launch over all systems of
// a batch; stages that the reference runs conditionally (NL rebuild and list
// updates) exit on the device when not needed, so that a step never waits on
// the host and can be captured in a hipGraph.
#include <algorithm>

#include "pcg_launch.hpp"
#include "pcg_stages.hpp"

namespace pcg {

// ------------------------------------------------------------ begin step ----
// NL verify decision (nl::verify, cg/src/cg/nl/verify.cpp:3-34) from the
// displacement maximum the previous Langevin step left behind. Read only: in a
// step, every thread of the first kernel takes it, and a later kernel
// (k_step_terms) resets the scalars it reads.
__device__ __forceinline__ bool rebuild_due(const DevBatch &b, int s) {
#pragma clang fp contract(off)
  const SysState &st = b.st[s];
  if (!b.P->nl_required) return st.nl_invalid != 0;
  if (st.verify_first) return true;
  SysDescC &d = b.sys[s];
  const double maxd = __longlong_as_double((long long)st.max_disp_bits);
  const double box = fabs(d.cell[0] - st.orig_cell[0]) + fabs(d.cell[1] - st.orig_cell[1]) +
                     fabs(d.cell[2] - st.orig_cell[2]);
  return __dadd_rn(__dmul_rn(2.0, maxd), box) > st.orig_pad;
}
// a system's energies and the walls' reaction forces at zero
// (dynamics::reset, dynamics.cpp:11-19)
__device__ __forceinline__ void clear_system(const DevBatch &b, int s) {
  for (int k = 0; k < NT; ++k) b.st[s].V[k] = 0.0;
  if (b.wall)
    for (int w = 0; w < 6; ++w)
      for (int c = 0; c < 3; ++c) b.wall->wall_F[w][c] = 0.0;
}
// the verify outside a step
__device__ __forceinline__ void begin_system(const DevBatch &b, int s) {
  SysState &st = b.st[s];
  if (!st.active) return;
  clear_system(b, s);
  st.nl_invalid = rebuild_due(b, s) ? 1 : 0;
  if (b.P->nl_required) st.verify_first = 0;
  st.max_disp_bits = 0ull;
}

__global__ void k_begin(DevBatch b) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= b.nsys) return;
  begin_system(b, s);
}

// Residue i before an evaluation: its force at zero; the system's first one
// clears the rest.
__device__ __forceinline__ void clear_residue(const DevBatch &b, int i, int s) {
  if (b.local[i] == 0) clear_system(b, s);
  for (int c = 0; c < 3; ++c) b.acc[c][i] = 0.0;
}
// an evaluation outside a step
__global__ void k_eval_begin(DevBatch b) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= b.ntot) return;
  const int s = b.sysid[i];
  if (!b.st[s].active) return;
  clear_residue(b, i, s);
}
// Residue i at the start of a step: cleared, its n and h (qa_on); the
// system's first residue writes down whether the step rebuilds its lists
// (due), for the kernels after this one.
__device__ __forceinline__ void begin_residue(const DevBatch &b, int i, int s, bool due, int qa_on) {
  if (!b.st[s].active) return;
  clear_residue(b, i, s);
  if (b.local[i] == 0) b.st[s].nl_invalid = due ? 1 : 0;
  if (qa_on) {
    GeoG g{b.y[0][0], b.y[0][1], b.y[0][2]};
    prepare_nh_item(b, g, i);
  }
}
// the forces of an evaluation, accumulated in FP64, into the FP32 arrays
// (STORE), or back for an integration outside a step
template <bool STORE> __global__ void k_move_forces(DevBatch b) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= b.ntot) return;
  for (int c = 0; c < 3; ++c) {
    float *f = (float *)b.F[c];
    if (STORE) f[i] = (float)b.acc[c][i];
    else b.acc[c][i] = f[i];
  }
}

// The near list's fields that only the stage kernels read, from those the
// persistent kernel keeps: before a plain context's calls term by term on the
// lists of persistent steps. (Written by the persistent rebuild itself they
// cost steps that have no such call after them: 3% of a 56-residue chain's,
// 5% of the batch of 30 to 600 residues.)
__global__ void k_near_fields(DevBatch b) {
  const int s = blockIdx.y;
  SysDescC &sd = b.sys[s];
  for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < b.st[s].qh_n; k += gridDim.x * blockDim.x) {
    const int h = sd.qf0 + k;
    const uint32_t ij = b.qh_ij[h];
    const float thr2 = b.qh_thr2[h];
    const int i1 = sd.res0 + (int)(ij & 0xFFFF), i2 = sd.res0 + (int)(ij >> 16);
    float of_types;
    b.qh_i[0][h] = i1;
    b.qh_i[1][h] = i2;
    b.qh_vac[h] = thr2 < 0.0f;  // as an accepted candidate leaves it
    qa_near_filters(b, i1, i2, b.qh_req[h], of_types);
  }
}

// The next rebuild of every system is due.
__global__ void k_mark_invalid(DevBatch b) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= b.nsys) return;
  b.st[s].nl_invalid = 1;
  b.st[s].verify_first = 0;
}

// Device data into mapped pinned host memory: words as they are, and three
// columns as interleaved FP64 triples. One workgroup then writes seq to the
// host's flag, so that the host sees the result arrive by reading the flag
// instead of waiting for the stream (9 us a call for a system's positions;
// 14 us with a wait for the stream, 47 us as three staged column copies).
// Without a flag, any number of workgroups.
template <typename T>
__global__ __launch_bounds__(1024) void k_fetch(const uint32_t *words, uint32_t *words_out, int nw,
                                                const T *x, const T *y, const T *z,
                                                const double *acc, double *out, int n, int *flag,
                                                int seq) {
  const int i0 = blockIdx.x * blockDim.x + threadIdx.x, stride = gridDim.x * blockDim.x;
  for (int i = i0; i < nw; i += stride) words_out[i] = words[i];
  for (int i = i0; i < 3 * n; i += stride) {
    const int k = i / 3, c = i - 3 * k;
    const T *col = c == 0 ? x : c == 1 ? y : z;
    if (acc) ((T *)col)[k] = (T)acc[(size_t)c * n + k];
    out[i] = (double)col[k];
  }
  // A barrier waits for no store, and thread 0's release for its own wave's
  // only. So every wave waits until its stores are in the L2, which is the
  // workgroup's waves' own and which thread 0 then writes back to the system:
  // also without a flag, as the flagged fetch behind on the stream may run on
  // another XCD. (A system release by every wave does it too, but 16
  // write-backs of the L2 took 5 us more a call.)
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  __syncthreads();
  if (threadIdx.x == 0) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "");
    if (flag) __hip_atomic_store(flag, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}
// the host's noise for one step (ntot x, then y, then z) into the device's
__global__ void k_noise_in(DevBatch b, const double *src) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= b.ntot) return;
  for (int c = 0; c < 3; ++c) b.noise[c][i] = src[(size_t)c * b.ntot + i];
}

// ------------------------------------------------------------ NL rebuild ----
// nl::legacy_update (cg/src/cg/nl/legacy_update.cpp:11-55): all pairs i < j
// of a system, same-chain |seq difference| < 3 skipped, kept if the wrapped
// distance is below max(nl.cutoff, dh.cutoff) + pad. One wavefront per row;
// rows come out in (i1, i2) order, which is the reference's sorted order.
__device__ __forceinline__ bool nl_pred(const DevBatch &b, SysDescC &s, const GeoG &g,
                                        int i, int j, double req, double &dist) {
  if (b.chain[i] == b.chain[j]) {
    int d = b.seq[i] - b.seq[j];
    if (d < 0) d = -d;
    if (d < 3) return false;
  }
  v3<double> dd = xwrapd(xsub(g.r(j), g.r(i)), s);
  dist = xnorm3(dd);
  return dist < req;
}

// Completion count of a per-item stage kernel: every lane with `mine` (an
// item of system `sys`) counts itself toward the system's residue count
// (and extra more items) in the SysState field `done`; a wave whose counted lanes share one system
// adds them with one atomic. Returns, in the lane whose add completed a
// system, that system (-1 elsewhere); with fence, what every lane wrote before
// the call is visible to it then.
__device__ __forceinline__ int count_done(const DevBatch &b, int SysState::*done, bool mine,
                                          int sys, bool fence = true, int extra = 0) {
  // a wave with nothing to count skips the fence: an agent-scope release
  // writes back the L2, and on a step without a rebuild every wave of the
  // cell count has nothing to count
  if (!__any(mine)) return -1;
  if (fence) __threadfence();
  else __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");  // what was read, was read
  const int lane = threadIdx.x & 63;
  const unsigned long long m = __ballot(mine);
  const int sys0 = __shfl(sys, 0, 64);
  const bool uni = __all(!mine || sys == sys0) && ((m & 1ull) != 0ull);
  int who = -1, add = 0;
  if (uni) {
    if (lane == 0) who = sys0, add = __popcll(m);
  } else if (mine) {
    who = sys, add = 1;
  }
  if (who < 0) return -1;
  const int old = atomicAdd(&(b.st[who].*done), add);
  if (old + add != b.sys[who].n + extra) return -1;
  if (fence) __threadfence();
  return who;
}

// Inclusive scan of x over the wave's 64 lanes: four DPP row shifts give
// each 16-lane row its own prefix (a lane shifted in from outside the row
// reads 0), three readlanes carry the rows' totals across. Every lane of the
// wave must be active; `total` is the wave's sum.
__device__ __forceinline__ int wave_incl(int x, int &total) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xf, 0xf, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xf, 0xf, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xf, 0xf, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xf, 0xf, false);  // row_shr:8
  const int r0 = __builtin_amdgcn_readlane(x, 15), r1 = __builtin_amdgcn_readlane(x, 31);
  const int r2 = __builtin_amdgcn_readlane(x, 47), r3 = __builtin_amdgcn_readlane(x, 63);
  const int row = (threadIdx.x & 63) >> 4;
  x += (row > 0 ? r0 : 0) + (row > 1 ? r1 : 0) + (row > 2 ? r2 : 0);
  total = r0 + r1 + r2 + r3;
  return x;
}

// One wave's exclusive scans of M arrays v[m][0..n) in place, the first one
// also into also[0..n) when given; their totals in every lane. The wave walks
// the arrays in stripes of 64 consecutive entries, loading SB stripes of each
// at once (coalesced, all in flight together) and carrying the running sums
// from stripe to stripe. Every lane of the wave must be active.
template <int M, int SB>
__device__ __forceinline__ void wave_scan(int *const (&v)[M], int n, int *also, int (&total)[M]) {
  const int lane = threadIdx.x & 63;
  for (int m = 0; m < M; ++m) total[m] = 0;
  for (int base = 0; base < n; base += 64 * SB) {
    int x[M][SB];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int j = 0; j < SB; ++j) {
        const int k = base + j * 64 + lane;
        x[m][j] = k < n ? v[m][k] : 0;
      }
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int j = 0; j < SB; ++j) {
        int tot;
        const int inc = wave_incl(x[m][j], tot);
        const int k = base + j * 64 + lane;
        if (k < n) {
          v[m][k] = total[m] + inc - x[m][j];
          if (m == 0 && also) also[k] = total[m] + inc - x[m][j];
        }
        total[m] += tot;
      }
  }
}

// ------------------------------------------------------------- cell grid ----
// A large periodic system can take its NL rows from a cell grid instead of
// every later residue: the periodic cell cut into cg[a] >= 3 cells a side,
// each at least the NL radius wide (with a relative 1e-6 to spare), so every
// pair within the radius sits in neighbouring cells (the 27 of the stencil,
// periodic). A row's candidates from those cells go into a bitmask over the
// system's residues, which the row then walks in increasing column order:
// the same pairs, tested by the same predicate, in the same order as the
// scan over all columns. When the cell has shrunk below that (the box
// protocol), the rebuild scans every column.
__device__ __forceinline__ bool use_cells(const DevBatch &b, SysDescC &sd) {
  if (sd.cg[0] <= 0) return false;
  const double req = (b.P->nl_eff_cutoff + b.P->p.nl_pad) * (1.0 + 1e-6);
  for (int a = 0; a < 3; ++a)
    if (!(sd.cell[a] >= req * (double)sd.cg[a])) return false;
  return true;
}
__device__ __forceinline__ int cell_coord(SysDescC &sd, int a, double x) {
  // the position wrapped into [0, cell), then its cell along the axis
  const double u = x - sd.cell[a] * floor(x * sd.cell_inv[a]);
  const int k = (int)(u * sd.cell_inv[a] * (double)sd.cg[a]);
  return k < 0 ? 0 : (k >= sd.cg[a] ? sd.cg[a] - 1 : k);
}

// A step's first kernel when a system is on a cell grid (begin): the residues'
// begin work. Each residue's cell; cell_end counts the residues of each cell; the wave
// whose residue completes a system turns its counts into the cells' first
// slots (cell_start) and fill pointers (cell_end)
__global__ void k_cell_count(DevBatch b, int begin, int qa_on) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  bool mine = false;
  int sys = -1;
  if (i < b.ntot) {
    sys = b.sysid[i];
    const SysState &st = b.st[sys];
    SysDescC &sd = b.sys[sys];
    const bool due = begin ? rebuild_due(b, sys) : st.nl_invalid != 0;
    if (begin) begin_residue(b, i, sys, due, qa_on);
    if (st.active && due && use_cells(b, sd)) {
      mine = true;
      const int c = (cell_coord(sd, 2, b.y[0][2][i]) * sd.cg[1] + cell_coord(sd, 1, b.y[0][1][i])) *
                        sd.cg[0] + cell_coord(sd, 0, b.y[0][0][i]);
      b.cell_of[i] = c;
      atomicAdd(&b.cell_end[sd.cell0 + c], 1);
    }
  }
  const int done = count_done(b, &SysState::done_cells, mine, sys);
  unsigned long long dm = __ballot(done >= 0);
  while (dm) {
    const int src = __ffsll((long long)dm) - 1;
    dm &= dm - 1ull;
    const int ds = __shfl(done, src, 64);
    SysDescC &sd = b.sys[ds];
    int *const v[1] = {b.cell_end + sd.cell0};
    int total[1];
    wave_scan<1, 16>(v, sd.cg[0] * sd.cg[1] * sd.cg[2], b.cell_start + sd.cell0, total);
    if ((threadIdx.x & 63) == 0) b.st[ds].done_cells = 0;
  }
}

// the cell counts back to zero for the next rebuild, once the rows are written
__device__ __forceinline__ void clear_cells(const DevBatch &b, SysDescC &sd, int t, int nt) {
  const int nc = sd.cg[0] > 0 ? sd.cg[0] * sd.cg[1] * sd.cg[2] : 0;
  for (int c = t; c < nc; c += nt) b.cell_end[sd.cell0 + c] = 0;
}

// the residues into their cells' slots (any order within a cell: a row's
// candidates go through a bitmask); cell_end ends at each cell's end
__global__ void k_cell_fill(DevBatch b) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= b.ntot) return;
  const int s = b.sysid[i];
  const SysState &st = b.st[s];
  if (!st.active || !st.nl_invalid) return;
  SysDescC &sd = b.sys[s];
  if (!use_cells(b, sd)) return;
  const int slot = atomicAdd(&b.cell_end[sd.cell0 + b.cell_of[i]], 1);
  b.cell_items[sd.res0 + slot] = i - sd.res0;
}

// Per-row counts of a rebuild: the NL pairs in row_cnt, the lists the pairs go
// to (RC_*) in the system's candidate scratch, which only a step's QA stage
// uses; [class][residue within the system]. After the scan, the rows' first
// slots.
enum { RC_NC, RC_QA, RC_NEAR, RC_PID, RC_DH, RC_PAULI, RC_N };
__device__ __forceinline__ int *row_counts(const DevBatch &b, SysDescC &sd, int cls) {
  return b.cand_perm + sd.nl0 + cls * sd.n;
}

__device__ __forceinline__ int *nl_counts(const DevBatch &b, SysDescC &sd) {
  return b.row_cnt + sd.res0;
}

// the length of the NL (cls -1) or of one of the lists
__device__ __forceinline__ void set_length(SysState &st, SysDescC &sd, int cls, int tot) {
  const int qf = min(tot, sd.qfcap), nl = min(tot, sd.nlcap);
  switch (cls) {
  case -1:
    st.nl_n = nl;
    if (tot > sd.nlcap) st.overflow = 1;
    break;
  case RC_NC: st.nc_n = tot; break;
  case RC_QA:
    st.qf_n = qf;
    st.qf_store = qf;
    if (tot > sd.qfcap) st.overflow = 1;
    break;
  case RC_NEAR: st.qh_n = qf; break;
  case RC_PID: st.pid_n = nl; break;
  case RC_DH: st.dh_n = nl; break;
  case RC_PAULI: st.pauli_n = nl; break;
  }
}

// One row of the sorted NL by one wave, with the ordered list updates of
// thread::fix_nl_async (thread_main.cpp:409-423): native contacts take first
// (nat_cont/update_contacts.cpp:7-37), then QA free pairs
// (qa/update_free_pairs.cpp:4-25), PID bundles and DH pairs see the rest
// without taking (pid/update_bundles.cpp:4-34, dh/update_pairs.cpp:4-25),
// Pauli takes last (pauli/update_pairs.cpp:4-20). Each pair's destination
// depends only on the pair, so the first pass counts each list's pairs per row
// (WRITE false), a scan gives every row its slots, and the second pass writes
// the NL pair and its list entries there. (Classifying in the rows instead of
// over the finished NL saves two launches, 5.7 us of a step with or without a
// rebuild, and the NL's reading back.)
template <bool WRITE> struct RowOut {
  const DevBatch &b;
  SysDescC &sd;
  int row, il, out, at[RC_N];
  int c0, nc;     // the row's native contacts [c0, c0 + nc) of all
  int partner;    // their second residues, one a lane (of the first 64)
  __device__ __forceinline__ RowOut(const DevBatch &b_, SysDescC &sd_, int row_)
      : b(b_), sd(sd_), row(row_), il(row_ - sd_.res0) {
    const int lane = threadIdx.x & 63;
    out = WRITE ? b.row_cnt[row] : 0;
    for (int c = 0; c < RC_N; ++c) at[c] = WRITE ? row_counts(b, sd, c)[il] : 0;
    // contacts are sorted by (i1, i2): the first of this row by bisection
    int lo = sd.nc0, hi = sd.nc0 + (b.P->p.nat_cont_on ? sd.nnc : 0);
    const int end = hi;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (b.nc_i[0][mid] < row) lo = mid + 1;
      else hi = mid;
    }
    c0 = __builtin_amdgcn_readfirstlane(lo);
    const bool mine = c0 + lane < end && b.nc_i[0][c0 + lane] == row;
    partner = mine ? b.nc_i[1][c0 + lane] : -1;
    nc = __popcll(__ballot(mine));
  }
  // the contact of residue j in this row, or -1
  __device__ __forceinline__ int contact(int j) const {
    int found = -1;
    for (int m = nc - 1; m >= 0; --m)
      if (__builtin_amdgcn_readlane(partner, m) == j) found = c0 + m;
    if (nc == 64 && found < 0) found = find_contact(b, sd, row, j);  // more than 64 contacts
    return found;
  }
  // 64 pairs (row, j), of which the lanes with `in` are NL pairs at distance d
  __device__ __forceinline__ void pairs(int j, bool in, double d) {
    const unsigned long long m = __ballot(in);
    if (!m) return;
    const int nat = contact(j);
    const int cls = in ? classify(b, sd, row, j, d, nat >= 0) : 0;
    const unsigned long long mm[RC_N] = {
        __ballot(cls & CL_NC), __ballot(cls & CL_QA), __ballot(cls & CL_NEAR),
        __ballot(cls & CL_PID), __ballot(cls & CL_DH), __ballot(cls & CL_PAULI)};
    if (WRITE && in) {
      const unsigned long long below = (1ull << (threadIdx.x & 63)) - 1ull;
      auto slot = [&](int c) { return at[c] + __popcll(mm[c] & below); };
      const int pos = out + __popcll(m & below);
      if (pos < sd.nlcap) {
        b.nl_i[0][sd.nl0 + pos] = row;
        b.nl_i[1][sd.nl0 + pos] = j;
        b.nl_d[sd.nl0 + pos] = d;
      }
      if (cls & CL_NC) set_current_contact(b, sd.nc0 + slot(RC_NC), nat, sd.res0);
      if (cls & CL_QA) {
        const int p = slot(RC_QA), q = sd.qf0 + p;
        if (p < sd.qfcap) {
          b.qf_i[0][q] = row;
          b.qf_i[1][q] = j;
          b.qf_d[q] = d;
          b.qf_vac[q] = 0;
          if (cls & CL_NEAR) {
            // near list entry: the free pair in slot p (its order is the
            // free pairs' order)
            const int h = sd.qf0 + slot(RC_NEAR);
            b.qh_slot[h] = p;
            b.qh_i[0][h] = row;
            b.qh_i[1][h] = j;
            b.qh_vac[h] = 0;
            qa_near_filters(b, row, j, b.qh_req[h], b.qh_thr2[h]);
            b.qh_ij[h] = (uint32_t)il | ((uint32_t)(j - sd.res0) << 16);
          }
        }
      }
      if (cls & CL_PID) {
        const int p = slot(RC_PID), q = sd.nl0 + p;
        if (p < sd.nlcap) {
          b.pid_i[0][q] = row;
          b.pid_i[1][q] = j;
          b.pid_d[q] = d;
          b.pid_t[q] = (int16_t)(b.atype[row] * 21 + b.atype[j]);
        }
      }
      if (cls & CL_DH) {
        const int p = slot(RC_DH), q = sd.nl0 + p;
        if (p < sd.nlcap) {
          b.dh_i[0][q] = row;
          b.dh_i[1][q] = j;
          b.dh_q[q] = b.P->p.charge[b.atype[row]] * b.P->p.charge[b.atype[j]];
        }
      }
      if (cls & CL_PAULI) {
        const int p = slot(RC_PAULI), q = sd.nl0 + p;
        if (p < sd.nlcap) {
          b.pauli_i[0][q] = row;
          b.pauli_i[1][q] = j;
        }
      }
    }
    out += __popcll(m);
    for (int c = 0; c < RC_N; ++c) at[c] += __popcll(mm[c]);
  }
};

// cell_words: 64-bit mask words of the largest system on the grid (the
// dynamic LDS holds one row mask a wave), 0 without a grid. begin (the count
// pass, without a grid): the step's first kernel, whose first threads do the
// residues' begin work.
template <bool WRITE>
__global__ void k_nl_rows(DevBatch b, int cell_words, int fuse_scan, int begin, int qa_on) {
  extern __shared__ unsigned long long row_mask[];
  if (!WRITE && begin) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < b.ntot) begin_residue(b, i, b.sysid[i], rebuild_due(b, b.sysid[i]), qa_on);
  }
  const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (row >= b.ntot) return;
  const int s = b.sysid[row];
  SysState &st = b.st[s];
  if (!st.active || !(!WRITE && begin ? rebuild_due(b, s) : st.nl_invalid != 0)) return;
  SysDescC &sd = b.sys[s];
  GeoG g{b.y[0][0], b.y[0][1], b.y[0][2]};
  // the snapshot of the rebuild's positions, pad and cell
  // (legacy_update.cpp:80-89); in the second pass, as a step's verify, taken
  // by the threads of the first, reads the old one
  if (WRITE && lane == 0) {
    for (int c = 0; c < 3; ++c) b.orig_r[c][row] = b.y[0][c][row];
    if (row == sd.res0) {
      st.orig_pad = b.P->p.nl_pad;
      for (int c = 0; c < 3; ++c) st.orig_cell[c] = sd.cell[c];
    }
  }
  const double req = b.P->nl_eff_cutoff + b.P->p.nl_pad;
  const int end = sd.res0 + sd.n;
  RowOut<WRITE> o(b, sd, row);
  if (cell_words > 0 && use_cells(b, sd)) {
    unsigned long long *m = row_mask + (size_t)(threadIdx.x >> 6) * cell_words;
    const int il = o.il, W = (sd.n + 63) >> 6, w0 = (il + 1) >> 6;
    for (int w = w0 + lane; w < W; w += 64) m[w] = 0ull;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int c = b.cell_of[row], gx = sd.cg[0], gy = sd.cg[1], gz = sd.cg[2];
    const int cx = c % gx, cy = (c / gx) % gy, cz = c / (gx * gy);
    for (int dz = -1; dz <= 1; ++dz)
      for (int dy = -1; dy <= 1; ++dy)
        for (int dx = -1; dx <= 1; ++dx) {
          const int nx = (cx + dx + gx) % gx, ny = (cy + dy + gy) % gy, nz = (cz + dz + gz) % gz;
          const int ncell = sd.cell0 + (nz * gy + ny) * gx + nx;
          const int t1 = b.cell_end[ncell];
          for (int t = b.cell_start[ncell] + lane; t < t1; t += 64) {
            const int j = b.cell_items[sd.res0 + t];
            if (j > il) atomicOr(&m[j >> 6], 1ull << (j & 63));
          }
        }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int wb = w0; wb < W; wb += 64) {
      const int w = wb + lane;
      const unsigned long long bits = w < W ? m[w] : 0ull;
      unsigned long long nz = __ballot(bits != 0ull);
      while (nz) {
        const int k = __ffsll((long long)nz) - 1;
        nz &= nz - 1ull;
        const unsigned lo = __shfl((unsigned)bits, k, 64), hi = __shfl((unsigned)(bits >> 32), k, 64);
        const unsigned long long bw = (unsigned long long)lo | ((unsigned long long)hi << 32);
        const int j = sd.res0 + (wb + k) * 64 + lane;
        double dist = 0.0;
        const bool in = ((bw >> lane) & 1ull) && nl_pred(b, sd, g, row, j, req, dist);
        o.pairs(j, in, dist);
      }
    }
  } else {
    for (int j0 = row + 1; j0 < end; j0 += 64) {
      const int j = j0 + lane;
      double dist = 0.0;
      const bool in = j < end && nl_pred(b, sd, g, row, j, req, dist);
      o.pairs(j, in, dist);
    }
  }
  if (!WRITE) {
    // the row counts; with fuse_scan the wave of the system's last row to
    // finish scans them into the rows' first slots, else k_nl_scan does
    if (lane == 0) {
      b.row_cnt[row] = o.out;
      for (int c = 0; c < RC_N; ++c) row_counts(b, sd, c)[o.il] = o.at[c];
    }
    if (!fuse_scan) return;
    int fin = 0;
    if (lane == 0) {
      __threadfence();
      fin = atomicAdd(&st.done_rows, 1) == sd.n - 1;
    }
    if (__shfl(fin, 0, 64)) {
      __threadfence();
      int *const v[RC_N + 1] = {nl_counts(b, sd),         row_counts(b, sd, 0),
                                row_counts(b, sd, 1), row_counts(b, sd, 2),
                                row_counts(b, sd, 3), row_counts(b, sd, 4),
                                row_counts(b, sd, 5)};
      int total[RC_N + 1];
      wave_scan<RC_N + 1, 4>(v, sd.n, nullptr, total);
      if (lane == 0) {
        for (int c = -1; c < RC_N; ++c) set_length(st, sd, c, total[c + 1]);
        st.done_rows = 0;
      }
    }
  }
}

// The row scan as a launch of its own, one wave a system and list: for systems
// of ROWS_FUSE_MAX residues or more. Every row's count comes to its system's
// counter through an agent-scope fence, and on this device such a fence
// writes back and invalidates the L2: in the trace of a 6400-residue box a
// rebuild's count pass took 131 us with the fused scan and about 20 us
// without it.
__global__ void k_nl_scan(DevBatch b) {
  const int s = blockIdx.x;
  if (s >= b.nsys) return;
  SysState &st = b.st[s];
  if (!st.active || !st.nl_invalid) return;
  SysDescC &sd = b.sys[s];
  const int cls = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6) - 1);
  int *const v[1] = {cls < 0 ? nl_counts(b, sd) : row_counts(b, sd, cls)};
  int total[1];
  wave_scan<1, 16>(v, sd.n, nullptr, total);
  if ((threadIdx.x & 63) == 0) set_length(st, sd, cls, total[0]);
}

// A rebuild outside a step is complete: record it and clear nl_invalid and the
// cell counts; one block a system.
__global__ void k_nl_done(DevBatch b) {
  const int s = blockIdx.x;
  SysState &st = b.st[s];
  const bool inv = st.active && st.nl_invalid;
  __syncthreads();
  if (!inv) return;
  clear_cells(b, b.sys[s], threadIdx.x, blockDim.x);
  if (threadIdx.x == 0) {
    st.nl_invalid = 0;
    st.rebuilds += 1;
  }
}

// ------------------------------------------------------------------ terms ----
// Forces accumulate in FP64 in every precision: FP64 atomics cost the L2 what
// FP32 ones do.

// A single term, as the host's per-term calls ask for it: blockIdx.y is the
// system, blockIdx.x strides over the term's list.
template <typename R> __global__ void k_terms(DevBatch b, int term, int from, int to) {
  int s = blockIdx.y;
  SysState &st = b.st[s];
  if (!st.active || !term_on(*b.P, term)) return;
  SysDescC &sd = b.sys[s];
  int n = term_size(sd, st, term);
  int lo = from > 0 ? from : 0, hi = (to >= 0 && to < n) ? to : n;
  GeoG g{b.y[0][0], b.y[0][1], b.y[0][2]};
  AccG acc{b.acc[0], b.acc[1], b.acc[2]};
  double v = 0.0;
  for (int k = lo + blockIdx.x * blockDim.x + threadIdx.x; k < hi; k += gridDim.x * blockDim.x)
    v += eval_item<R>(b, sd, st, g, acc, term, k, st.t);
  v = block_sum(v);
  if (threadIdx.x == 0 && v != 0.0) atomicAdd(&st.V[term], v);
}

// The sum of v over the wave in lane 63: row shifts within 16 lanes, then the
// rows' totals broadcast along (a DPP move is one vector instruction; a
// cross-lane shuffle an LDS round trip).
template <int CTRL, int ROWS> __device__ __forceinline__ double dpp_add(double v) {
  const long long x = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)x, CTRL, ROWS, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(x >> 32), CTRL, ROWS, 0xf, true);
  return v + __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}
__device__ __forceinline__ double wave_total(double v) {
  v = dpp_add<0x111, 0xf>(v);
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);  // row_bcast:15 into rows 1 and 3
  v = dpp_add<0x143, 0xc>(v);  // row_bcast:31 into rows 2 and 3
  return v;
}
__device__ __forceinline__ void add_energy(SysState &st, int term, double v) {
  v = wave_total(v);
  if ((threadIdx.x & 63) == 63 && v != 0.0) atomicAdd(&st.V[term], v);
}

// 64 base residues' chain-local bonded items (bond_regular): every lane
// evaluates the items that start at its residue, in FP64 as eval_item does,
// from one read of its four residues; a residue's force is its own share plus
// those lanes 1..3 below computed for it, so a residue takes 3 atomics a group
// where its items would take 9 or 12 each. Shares past the wave's last lane go
// out directly. The items fall into three groups for different waves, as one
// wave's chain of all seven would be the step's longest.
enum { BG_DIH, BG_CHIR, BG_SHORT, BG_N };
template <int GROUP>
__device__ __forceinline__ void bonded_chunk(const DevBatch &b, SysDescC &sd, SysState &st,
                                             const GeoG &g, AccG &acc, int chunk) {
  ParamsC &p = b.P->p;
  const int lane = threadIdx.x & 63, k = chunk * 64 + lane, last = sd.res0 + sd.n - 1;
  const bool mine = k < sd.n;
  const int r = min(sd.res0 + k, last);
  GeoR q;
  q.base = r;
  for (int j = 0; j < 4; ++j) q.p[j] = g.r(min(r + j, last));
  AccSlots<double> a;
  a.base = r;
  for (int s = 0; s < 4; ++s) a.c[s][0] = a.c[s][1] = a.c[s][2] = 0.0;
  const int variant = p.nat_dih_variant;
  auto part = [&](int term, int L, auto item) {
    const int t = mine ? b.bond_item[L][r] : -1;
    if (!__any(t >= 0)) return;
    double v = 0.0;
    if (t >= 0) v = item(t);
    add_energy(st, term, v);
  };
  if (GROUP == BG_SHORT) {
    part(PCG_TETHER, BOND_TETHER,
         [&](int t) { return tether_core<double>(p, q, a, r, r + 1, b.teth_nat[t]); });
    part(PCG_LREP, BOND_LREP, [&](int) { return lrep_core<double>(p, q, a, r, r + 2); });
    part(PCG_NAT_ANG, BOND_NAT_ANG,
         [&](int t) { return nat_ang_core<double>(p, q, a, r, r + 1, r + 2, b.nang_th[t]); });
    part(PCG_HEUR_ANG, BOND_HEUR_ANG,
         [&](int t) { return heur_ang_core<double>(p, q, a, r, r + 1, r + 2, b.hang_t[t]); });
  } else if (GROUP == BG_DIH) {
    part(variant ? PCG_SND : PCG_CND, BOND_NAT_DIH, [&](int t) {
      const double phi0 = b.ndih_ph[t];
      double s0 = 0.0, c0 = 1.0;
      if (variant == 0) sincos(phi0, &s0, &c0);
      return nat_dih_core<double>(p, q, a, r, r + 1, r + 2, r + 3, phi0, c0, s0, variant);
    });
    part(PCG_HEUR_DIH, BOND_HEUR_DIH, [&](int t) {
      return heur_dih_core<double>(p, q, a, r, r + 1, r + 2, r + 3, b.hdih_t[t]);
    });
  } else {
    part(PCG_CHIR, BOND_CHIR, [&](int t) {
      return chir_core<double>(p, q, a, r, r + 1, r + 2, r + 3, b.chir_f0[t], b.chir_f1[t]);
    });
  }
  double f[3];
  for (int c = 0; c < 3; ++c) {
    const double s1 = __shfl_up(a.c[1][c], 1, 64), s2 = __shfl_up(a.c[2][c], 2, 64),
                 s3 = __shfl_up(a.c[3][c], 3, 64);
    f[c] = a.c[0][c];
    if (lane >= 1) f[c] += s1;
    if (lane >= 2) f[c] += s2;
    if (lane >= 3) f[c] += s3;
  }
  if (!mine) return;
  acc.add(r, v3<double>{f[0], f[1], f[2]});
  for (int s = 1; s < 4; ++s)
    if (lane + s >= 64 && (a.c[s][0] != 0.0 || a.c[s][1] != 0.0 || a.c[s][2] != 0.0))
      acc.add(r + s, v3<double>{a.c[s][0], a.c[s][1], a.c[s][2]});
}

template <int T> struct Term {
  static constexpr int value = T;
};
// Every enabled term of a step in one launch: blockIdx.y is the system, whose
// waves stride over the 64-item chunks of all its terms, the long chains of
// bonded items first. Each wave finds its chunk from the list sizes on the
// device, so the grid follows the work. A wave's chunk is a serial chain of
// some thousand instructions on almost empty SIMDs, which bounds the kernel: a
// grid of blocks for every term at its largest size was 11 000 blocks, nearly
// all empty, and took 18.4 us for a box of 64 chains of 100, 18 for 2000
// residues in one chain and 12.9 for 480 between walls; this one takes 14.0,
// 15.5 and 10.3 (29 and more with one chunk of all the bonded items). Also
// resets what the step's verify read.
template <typename R> __global__ __launch_bounds__(BLK) void k_step_terms(DevBatch b, int step) {
  const int s = blockIdx.y;
  SysState &st = b.st[s];
  if (!st.active) return;
  SysDescC &sd = b.sys[s];
  const int nwaves = gridDim.x * (BLK / 64);
  const int w0 = __builtin_amdgcn_readfirstlane(blockIdx.x * (BLK / 64) + (threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  if (step && st.nl_invalid) clear_cells(b, sd, w0 * 64 + lane, nwaves * 64);
  if (step && blockIdx.x == 0 && threadIdx.x == 0) {
    st.max_disp_bits = 0ull;
    if (b.P->nl_required) st.verify_first = 0;
  }
  GeoG g{b.y[0][0], b.y[0][1], b.y[0][2]};
  AccG acc{b.acc[0], b.acc[1], b.acc[2]};
  const double t = st.t;
  for (int w = w0;; w += nwaves) {
    int c = w;  // the wave's chunk, counted down through the terms
    // (uniform) chunk c of term T, or past its end
    auto term = [&](auto tag) -> bool {
      constexpr int T = decltype(tag)::value;
      if (!term_on(*b.P, T)) return false;
      const int n = __builtin_amdgcn_readfirstlane(term_size(sd, st, T)), chunks = (n + 63) >> 6;
      if (c >= chunks) {
        c -= chunks;
        return false;
      }
      const int k = c * 64 + lane;
      double v = 0.0;
      if (k < n) v = eval_item<R>(b, sd, st, g, acc, T, k, t);
      add_energy(st, T, v);
      return true;
    };
    if (sd.bond_regular) {
      const int chunks = (sd.n + 63) >> 6;
      // chunk c of a group with items
      auto group = [&](auto tag, bool any) -> bool {
        if (!any) return false;
        if (c >= chunks) {
          c -= chunks;
          return false;
        }
        bonded_chunk<decltype(tag)::value>(b, sd, st, g, acc, c);
        return true;
      };
      if (group(Term<BG_DIH>(), sd.nndih > 0 || sd.nhdih > 0) ||
          group(Term<BG_CHIR>(), sd.nchir > 0) ||
          group(Term<BG_SHORT>(), sd.nteth > 0 || sd.nlrep > 0 || sd.nnang > 0 || sd.nhang > 0))
        continue;
    } else if (term(Term<PCG_CHIR>()) || term(Term<PCG_TETHER>()) || term(Term<PCG_LREP>()) ||
               term(Term<PCG_NAT_ANG>()) || term(Term<PCG_HEUR_ANG>()) ||
               term(Term<PCG_HEUR_DIH>()) || term(Term<PCG_CND>()) || term(Term<PCG_SND>())) {
      continue;
    }
    if (term(Term<PCG_QA_CONT>()) || term(Term<PCG_NAT_CONT>()) || term(Term<PCG_PID>()) ||
        term(Term<PCG_QA_CAND>()) || term(Term<PCG_PAULI>()) || term(Term<PCG_CONST_DH>()) ||
        term(Term<PCG_REL_DH>()) || term(Term<PCG_VEL_AFM>()) || term(Term<PCG_FORCE_AFM>()) ||
        term(Term<PCG_SOLID_WALL>()) || term(Term<PCG_HW_FREE>()) || term(Term<PCG_HW_CONN>()) ||
        term(Term<PCG_LJW_FREE>()) || term(Term<PCG_LJW_CONN>()))
      continue;
    break;
  }
}

// ------------------------------------------------------------------- QA ----
__global__ void k_prepare_nh(DevBatch b) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= b.ntot) return;
  if (!b.st[b.sysid[i]].active) return;
  GeoG g{b.y[0][0], b.y[0][1], b.y[0][2]};
  prepare_nh_item(b, g, i);
}

// Sums and differences of four int8 side by side, each on its own.
__device__ __forceinline__ uint32_t add4(uint32_t x, uint32_t y) {
  return ((x & 0x7f7f7f7fu) + (y & 0x7f7f7f7fu)) ^ ((x ^ y) & 0x80808080u);
}
__device__ __forceinline__ uint32_t sub4(uint32_t x, uint32_t y) {
  return ((x | 0x80808080u) - (y & 0x7f7f7f7fu)) ^ ((x ^ ~y) & 0x80808080u);
}
// LDS of the QA finish beside the budgets: the candidates as they come and in
// the order they are taken, and the removed contacts as they come
struct QfLds {
  long long key[QF_CAND_LDS];   // by distance; then the accepted ones' ranks
  uint64_t sd[QF_CAND_LDS];     // by rank: budget changes of the two residues,
  int i1[QF_CAND_LDS], i2[QF_CAND_LDS], sc[QF_CAND_LDS];  // the residues, the slot
  int idx[QF_CAND_LDS];
  int rem[QF_REM_LDS];          // 2 * contact + near
  int wave[16];
  int near, accepted, live, overflow;
};

// budget word w takes the four changes in d (they commute: any order)
__device__ __forceinline__ void give_back(uint32_t *w, uint32_t d) {
  uint32_t old = *w;
  for (;;) {
    const uint32_t seen = atomicCAS(w, old, add4(old, d));
    if (seen == old) return;
    old = seen;
  }
}
// qa_finish_block (pcg_stages.hpp) by a whole workgroup of 1024, the budgets
// in LDS (sy: one word of four a residue). Removed contacts and candidates are
// ranked in parallel, one thread decides which candidates are taken, in order,
// on LDS alone, and the lists are written and compressed in parallel. (With
// that thread writing the lists too, a contact cost some 1 us of waits on HBM:
// 11 us a step for a box of 64 chains of 100 and 2400 us for its first, where
// it is 6.7 and 575 so; what is left is the chain of loads and barriers.)
// Removed contacts beyond QF_REM_LDS are ranked where they are, in HBM.
__device__ __forceinline__ void qa_finish_wide(const DevBatch &b, SysDescC &sd, SysState &st,
                                               uint32_t *sy, QfLds &q, int cand_n, int rem_n) {
  const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wv = tid >> 6;
  const int r0 = sd.res0, qc_n0 = st.qc_n, store0 = st.qf_store, qh0 = st.qh_n;
  const int num0 = st.num_qa;
  if (tid == 0) q.near = 0, q.overflow = 0;
  for (int c = tid; c < cand_n; c += nt) {
    q.key[c] = total_key(b.cand_dist[sd.nl0 + c]);
    q.idx[c] = b.cand_idx[sd.nl0 + c];
  }
  const bool rem_lds = rem_n <= QF_REM_LDS;
  for (int a = tid; a < rem_n; a += nt) {
    const int v = b.rem[sd.qc0 + a], w = 2 * v + (b.qc_d[sd.qc0 + v] > b.P->qa_max_req ? 0 : 1);
    if (rem_lds) q.rem[a] = w;
    else b.rem[sd.qc0 + a] = w;
  }
  for (int k = tid; k < sd.n; k += nt) sy[k] = *(const uint32_t *)(b.sync + 4 * (r0 + k));
  __syncthreads();
  // candidates by (distance, free-pair index); ties, from evaluations repeated
  // outside a step, as they came
  for (int c = tid; c < cand_n; c += nt) {
    const int sc = sd.nl0 + c, ic = q.idx[c];
    const long long kc = q.key[c];
    int rank = 0;
    for (int o = 0; o < cand_n; ++o) {
      const long long kd = q.key[o];
      rank += (kd < kc || (kd == kc && (q.idx[o] < ic || (q.idx[o] == ic && o < c)))) ? 1 : 0;
    }
    q.sc[rank] = sc;
    q.i1[rank] = b.cand_i[0][sc];
    q.i2[rank] = b.cand_i[1][sc];
    q.sd[rank] = *(const uint64_t *)(b.cand_sd + 8 * (size_t)sc);
  }
  // removed contacts in increasing index order, back among the free pairs
  const int *rem_hbm = b.rem + sd.qc0;
  for (int a = tid; a < rem_n; a += nt) {
    const int own = rem_lds ? q.rem[a] : rem_hbm[a];
    const int v = own >> 1, near = own & 1, qc = sd.qc0 + v;
    int rank = 0, nearer = 0;
    auto behind = [&](int o, int w) {
      const bool before = (w >> 1) < v || ((w >> 1) == v && o < a);
      rank += before ? 1 : 0;
      nearer += before ? (w & 1) : 0;
    };
    if (rem_lds) {
      for (int o = 0; o < rem_n; ++o) behind(o, q.rem[o]);
    } else {
#pragma clang loop unroll_count(8)
      for (int o = 0; o < rem_n; ++o) behind(o, rem_hbm[o]);
    }
    const int i1 = b.qc_i[0][qc], i2 = b.qc_i[1][qc];
    const uint64_t back = *(const uint64_t *)(b.qc_sd + 8 * (size_t)qc);
    give_back(sy + (i1 - r0), (uint32_t)back);
    give_back(sy + (i2 - r0), (uint32_t)(back >> 32));
    b.qc_vac[qc] = 1;
    const int slot = store0 + rank;
    if (slot >= sd.qfcap) {
      q.overflow = 1;
      continue;
    }
    const int f = sd.qf0 + slot;
    b.qf_i[0][f] = i1;
    b.qf_i[1][f] = i2;
    b.qf_d[f] = b.qc_d[qc];
    b.qf_vac[f] = 0;
    if (near) {
      // appended at the end, so the near list stays in slot order
      const int h = sd.qf0 + qh0 + nearer;
      b.qh_slot[h] = slot;
      b.qh_i[0][h] = i1;
      b.qh_i[1][h] = i2;
      b.qh_vac[h] = 0;
      qa_near_filters(b, i1, i2, b.qh_req[h], b.qh_thr2[h]);
      b.qh_ij[h] = (uint32_t)(i1 - r0) | ((uint32_t)(i2 - r0) << 16);
      atomicAdd(&q.near, 1);
    }
  }
  __syncthreads();
  int *taken = (int *)q.key;
  if (tid == 0) {
    int n = 0;
    for (int a = 0; a < cand_n; ++a) {
      const int i1 = q.i1[a] - r0, i2 = q.i2[a] - r0;
      const uint64_t v = q.sd[a];
      const uint32_t n1 = sub4(sy[i1], (uint32_t)v), n2 = sub4(sy[i2], (uint32_t)(v >> 32));
      if ((n1 | n2) & 0x80808080u) continue;
      if (qc_n0 + n >= sd.qccap) {
        q.overflow = 1;
        continue;
      }
      taken[n++] = a;
      sy[i1] = n1;
      sy[i2] = n2;
    }
    q.accepted = n;
  }
  __syncthreads();
  for (int k = tid; k < sd.n; k += nt) *(uint32_t *)(b.sync + 4 * (r0 + k)) = sy[k];
  const int acc_n = q.accepted;
  for (int k = tid; k < acc_n; k += nt) {
    const int a = taken[k], sc = q.sc[a], qc = sd.qc0 + qc_n0 + k;
    b.qc_i[0][qc] = q.i1[a];
    b.qc_i[1][qc] = q.i2[a];
    b.qc_d[qc] = b.cand_od[sc];
    b.qc_t[qc] = b.cand_t[sc];
    b.qc_sat[qc] = 0.0;
    *(uint64_t *)(b.qc_sd + 8 * (size_t)qc) = q.sd[a];
    b.qc_vac[qc] = 0;
    const int h = sd.qf0 + b.cand_h[sc];
    b.qf_vac[sd.qf0 + b.cand_idx[sc]] = 1;
    b.qh_vac[h] = 1;
    b.qh_thr2[h] = -1.0f;
  }
  // compress: the contacts still there move to the front, in order, a block
  // of them at a time (a contact never moves up, so no block's reads meet
  // another's writes)
  const int num = num0 - rem_n + acc_n;
  int qc_n = qc_n0 + acc_n;
  if (2 * num < qc_n) {
    int slot = 0;
    for (int base = 0; base < qc_n; base += nt) {
      __syncthreads();
      const int cur = base + tid, qc = sd.qc0 + cur;
      const bool live = cur < qc_n && !b.qc_vac[qc];
      const unsigned long long m = __ballot(live);
      if (lane == 0) q.wave[wv] = __popcll(m);
      int i1 = 0, i2 = 0;
      double d = 0.0, sat = 0.0;
      int16_t t = 0;
      uint64_t v = 0;
      if (live) {
        i1 = b.qc_i[0][qc], i2 = b.qc_i[1][qc];
        d = b.qc_d[qc], sat = b.qc_sat[qc];
        t = b.qc_t[qc];
        v = *(const uint64_t *)(b.qc_sd + 8 * (size_t)qc);
      }
      __syncthreads();
      int at = slot + __popcll(m & ((1ull << lane) - 1ull));
      for (int w = 0; w < nt >> 6; ++w) {
        at += w < wv ? q.wave[w] : 0;
        slot += q.wave[w];
      }
      if (live && at != cur) {
        const int qs = sd.qc0 + at;
        b.qc_i[0][qs] = i1;
        b.qc_i[1][qs] = i2;
        b.qc_d[qs] = d;
        b.qc_t[qs] = t;
        b.qc_sat[qs] = sat;
        *(uint64_t *)(b.qc_sd + 8 * (size_t)qs) = v;
        // the vacancy flag of the destination slot stays as it was
      }
    }
    qc_n = slot;
  }
  if (tid == 0) {
    const int back = min(rem_n, sd.qfcap - store0);
    st.qf_n += back;
    st.qf_store = store0 + back;
    st.qh_n = qh0 + q.near;
    st.num_qa = num;
    st.qc_n = qc_n;
    if (q.overflow) st.overflow = 1;
    st.cand_n = 0;
    st.rem_n = 0;
  }
}

// The QA finish of a step, one workgroup a system: qa_finish_wide where the
// budgets fit its LDS (sync_lds) and the candidates their staging, which only
// the first steps of a large system outgrow.
__global__ __launch_bounds__(1024) void k_qa_finish(DevBatch b, int sync_lds) {
  extern __shared__ __align__(16) unsigned char qf_lds[];
  int s = blockIdx.x;
  SysState &st = b.st[s];
  if (!st.active || !b.P->p.qa_on) return;
  SysDescC &sd = b.sys[s];
  // nothing removed and no candidate
  if (st.cand_n == 0 && st.rem_n == 0) return;
  const int rem_n = min(st.rem_n, sd.qccap), cand_n = min(st.cand_n, sd.nlcap);
  if (!sync_lds) {
    qa_finish_block(b, sd, st, b.sync, 0);
    return;
  }
  const int n = sd.n, r0 = sd.res0;
  QfLds &q = *(QfLds *)qf_lds;
  uint32_t *syl = (uint32_t *)(qf_lds + sizeof(QfLds));
  if (cand_n <= QF_CAND_LDS) {
    qa_finish_wide(b, sd, st, syl, q, cand_n, rem_n);
    return;
  }
  for (int k = threadIdx.x; k < n; k += blockDim.x) syl[k] = *(const uint32_t *)(b.sync + 4 * (r0 + k));
  __syncthreads();
  qa_finish_block(b, sd, st, (int8_t *)syl, r0);
  for (int k = threadIdx.x; k < n; k += blockDim.x) *(uint32_t *)(b.sync + 4 * (r0 + k)) = syl[k];
}

// wall::log_forces (cg/src/cg/wall/log_forces.cpp:4-17) after the forces of
// a step: every plane on a box side, then once more the -axis plane of each
// LJ axis (the reference's wall list holds it twice, state.cpp:680-681);
// work += F . shift; the z force averaged. One thread a side, as the planes
// keep apart, and one for the z force (threads 0..6; by one thread in turn the
// log took 5.6 us of the 44 a 480-residue box step ran).
__device__ __forceinline__ void box_log(const DevBatch &b) {
#pragma clang fp contract(off)
  WallDev &W = *b.wall;
  const SysState &st = b.st[0];
  if (!st.active || !W.log_on) return;
  ParamsC &p = b.P->p;
  const double t = st.t;
  auto one = [&](int w) {
    mavg_add(W.avg_F[w], t, W.wall_F[w], 3);
    W.work[w] += W.wall_F[w][0] * W.shift[w][0] + W.wall_F[w][1] * W.shift[w][1] +
                 W.wall_F[w][2] * W.shift[w][2];
  };
  const int side = threadIdx.x;
  if (side < 6) {
    const int w = W.side_wall[side];
    if (w >= 0) one(w);
    if (w >= 0 && (side & 1) == 0 && p.wall_kind[w] == 2) one(w);
  }
  if (side != 6) return;
  const int wn = W.side_wall[4], wp = W.side_wall[5];
  const double zf = (W.wall_F[wn][0] * p.wall_normal[wn][0] + W.wall_F[wn][1] * p.wall_normal[wn][1] +
                     W.wall_F[wn][2] * p.wall_normal[wn][2]) +
                    (W.wall_F[wp][0] * p.wall_normal[wp][0] + W.wall_F[wp][1] * p.wall_normal[wp][1] +
                     W.wall_F[wp][2] * p.wall_normal[wp][2]);
  mavg_add(W.avg_z, t, &zf, 1);
}

// time and energy bookkeeping at the end of a step (step.cpp:157-162)
// v: the sum of its energies
__device__ __forceinline__ void tick_system(const DevBatch &b, int s, int advance, bool nl_done,
                                            double v) {
  SysState &st = b.st[s];
  // (all reads first: one wait instead of one for each)
  const int invalid = st.nl_invalid, rebuilds = st.rebuilds, overflow = st.overflow;
  const double t = st.true_t + b.P->dt;
  const auto step = st.step;
  const int lang = b.P->p.lang_on;
  // a full step's rebuild, if it made one, is complete (k_nl_done)
  if (nl_done && invalid) {
    st.nl_invalid = 0;
    st.rebuilds = rebuilds + 1;
  }
  st.Vtot = v;
  if (b.ovf && overflow) *b.ovf = 1;
  if (advance && lang) {
    st.true_t = t;
    st.t = t;
    st.step = step + 1;
  }
}
__device__ __forceinline__ double sum_energies(const SysState &st) {
  double v = 0.0;
  for (int k = 0; k < NT; ++k) v += st.V[k];
  return v;
}

// the tick outside a step, where k_nl_done closes rebuilds
__global__ void k_tick(DevBatch b, int advance) {
  int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= b.nsys) return;
  if (!b.st[s].active) return;
  tick_system(b, s, advance, false, sum_energies(b.st[s]));
}


// The displacement maximum goes to the system's state with one atomic per
// wave when the wave's residues belong to one system (a system of the plain
// context has thousands of residues: one atomic per residue on one address
// serialised the whole kernel), else one per residue. The forces come from the
// FP64 accumulators and go to the force arrays in their precision.
//
// The step's tick is run by the wave that completes its system. It waits for
// no other wave's results, only for every wave to have read the time and step
// it advances, which a wave has when it counts itself: so the count needs no
// fence (an agent-scope one writes back the L2; 8.8 us with it, 7.9 without,
// for 6400 residues). What the tick adds up is
// read before the count, as it is final by then. log (one system): one more
// block than the residues need keeps the wall forces' log, which reads the
// time too, and counts itself as one more item.
//
// noise (RAN2): the step's draws where the host put them (ntot x, then y, then
// z), or null for the device's copy. Read from host memory here, they cost a
// step 1.1 us; a kernel that copied them took 4.8.
template <typename RF>
__global__ void k_lang(DevBatch b, int noise_mode, const double *noise, int tick, int log) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  int s = -1, sys = -1;
  bool mine = false;   // a residue of an active system
  double disp = -1.0;  // below every displacement: lanes without a residue
  if (i < b.ntot) {
    // (the longest wait first)
    double nz[3];
    if (noise_mode == PCG_NOISE_RAN2)
      for (int c = 0; c < 3; ++c) nz[c] = noise ? noise[(size_t)c * b.ntot + i] : b.noise[c][i];
    s = sys = b.sysid[i];
    SysState &st = b.st[s];
    mine = st.active != 0;
    if (st.active && b.P->p.lang_on) {
      SysDescC &sd = b.sys[s];
      if (noise_mode != PCG_NOISE_RAN2) philox_normals(sd.philox_key, st.step, b.local[i], nz);
      const double F[3] = {b.acc[0][i], b.acc[1][i], b.acc[2][i]};
      double r[3];
      gear_update(b, sd, st, i, F[0], F[1], F[2], nz, r);
      if (sizeof(RF) == 4)
        for (int c = 0; c < 3; ++c) ((RF *)b.F[c])[i] = (RF)F[c];
      disp = disp_from_orig(b, sd, i, r);
    } else {
      s = -1;
      // without Langevin steps the forces are a step's result all the same
      if (sizeof(RF) == 4 && mine)
        for (int c = 0; c < 3; ++c) ((RF *)b.F[c])[i] = (RF)b.acc[c][i];
    }
  } else if (log && blockIdx.x == gridDim.x - 1 && threadIdx.x < 7) {
    mine = threadIdx.x == 0 && b.st[0].active != 0;
    sys = 0;
    box_log(b);
  }
  // the energies of the wave's first system, one a lane, for the tick
  const int sys0 = __shfl(sys, 0, 64), lane = threadIdx.x & 63;
  const double vk = tick && sys0 >= 0 && lane < NT ? b.st[sys0].V[lane] : 0.0;
  const int s0 = __shfl(s, 0, 64);
  if (__all(s == s0)) {
    double m = disp;
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0 && s0 >= 0)
      atomicMax(&b.st[s0].max_disp_bits, (unsigned long long)__double_as_longlong(m));
  } else if (s >= 0) {
    atomicMax(&b.st[s].max_disp_bits, (unsigned long long)__double_as_longlong(disp));
  }
  if (tick) {
    const int done = count_done(b, &SysState::done_lang, mine, sys, false, log);
    double v = 0.0;
    if (__any(done >= 0))
      for (int k = 0; k < NT; ++k) v += __shfl(vk, k, 64);
    if (done >= 0) {
      tick_system(b, done, 1, true, done == sys0 ? v : sum_energies(b.st[done]));
      b.st[done].done_lang = 0;
    }
  }
}


// ------------------------------------------------------------------ walls ----
// wall::lj::process_candidates (cg/src/cg/wall/lj/process_candidates.cpp:5-31)
// in one workgroup: the released slots leave (their residue unconnected, the
// plane's count down) and the live slots close up in order; then the
// candidates, sorted by distance (ties by residue, then plane: the order
// sift_free emits them in), connect one by one while their plane is below its
// limit and their residue is not connected, with the bead at the residue's
// projection on the plane. As in the reference a new connection does not
// mark its residue connected. The candidates are consumed.
constexpr int LJW_SORT_MAX = 4096;
__global__ void __launch_bounds__(1024) k_ljw_process(DevBatch b) {
#pragma clang fp contract(off)
  WallDev &W = *b.wall;
  SysState &st = b.st[0];
  ParamsC &p = b.P->p;
  const int tid = threadIdx.x, B = blockDim.x;
  __shared__ double key[LJW_SORT_MAX];
  __shared__ int val[LJW_SORT_MAX];
  __shared__ int scan[1024];
  __shared__ int base;
  const int n_lj = st.n_lj;
  // releases
  for (int k = tid; k < n_lj; k += B)
    if (W.lj_gone[k]) {
      W.is_conn[W.lj_res[k]] = 0;
      atomicSub(&W.num_conns[W.lj_wall[k]], 1);
    }
  if (tid == 0) base = 0;
  __syncthreads();
  // ordered compaction, one chunk of B slots at a time (reads before writes)
  for (int c0 = 0; c0 < n_lj; c0 += B) {
    const int k = c0 + tid;
    const bool keep = k < n_lj && !W.lj_gone[k];
    int res = 0, wl = 0;
    double o0 = 0, o1 = 0, o2 = 0, sat = 0;
    if (keep) {
      res = W.lj_res[k], wl = W.lj_wall[k], sat = W.lj_sat[k];
      o0 = W.lj_off[0][k], o1 = W.lj_off[1][k], o2 = W.lj_off[2][k];
    }
    scan[tid] = keep ? 1 : 0;
    __syncthreads();
    for (int off = 1; off < B; off <<= 1) {
      int v = tid >= off ? scan[tid - off] : 0;
      __syncthreads();
      scan[tid] += v;
      __syncthreads();
    }
    const int pos = base + scan[tid] - (keep ? 1 : 0);
    const int total = scan[B - 1];
    __syncthreads();
    if (keep) {
      W.lj_res[pos] = res, W.lj_wall[pos] = wl, W.lj_sat[pos] = sat;
      W.lj_off[0][pos] = o0, W.lj_off[1][pos] = o1, W.lj_off[2][pos] = o2;
      W.lj_gone[pos] = 0;
    }
    __syncthreads();
    if (tid == 0) base += total;
    __syncthreads();
  }
  int live = base;
  for (int k = live + tid; k < n_lj; k += B) W.lj_gone[k] = 0;
  // candidates by (distance, residue, plane)
  int nc = W.n_cand < W.cand_cap ? W.n_cand : W.cand_cap;
  if (nc > LJW_SORT_MAX) {
    if (tid == 0) W.overflow = 1;
    nc = LJW_SORT_MAX;
  }
  int m = 1;
  while (m < nc) m <<= 1;
  for (int k = tid; k < m; k += B) {
    key[k] = k < nc ? W.cand_d[k] : __builtin_inf();
    val[k] = k < nc ? k : -1;
  }
  __syncthreads();
  auto before = [&](int a, int c) {  // entry a sorts before entry c
    if (key[a] != key[c]) return key[a] < key[c];
    const int va = val[a], vc = val[c];
    if (va < 0 || vc < 0) return vc < 0 && va >= 0;
    const int ra = W.cand_res[va], rc = W.cand_res[vc];
    if (ra != rc) return ra < rc;
    return W.cand_wall[va] < W.cand_wall[vc];
  };
  for (int size = 2; size <= m; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int i = tid; i < m; i += B) {
        const int j = i ^ stride;
        if (j > i) {
          const bool up = (i & size) == 0;
          if (before(j, i) == up) {
            const double tk = key[i];
            key[i] = key[j], key[j] = tk;
            const int tv = val[i];
            val[i] = val[j], val[j] = tv;
          }
        }
      }
      __syncthreads();
    }
  if (tid == 0) {
    for (int a = 0; a < nc; ++a) {
      const int c = val[a], res = W.cand_res[c], w = W.cand_wall[c];
      if (W.is_conn[res] || W.num_conns[w] >= p.wall_limit[w]) continue;
      if (live >= W.lj_cap) {
        W.overflow = 1;
        break;
      }
      const double nx = p.wall_normal[w][0], ny = p.wall_normal[w][1], nz = p.wall_normal[w][2];
      const double ox = p.wall_origin[w][0], oy = p.wall_origin[w][1], oz = p.wall_origin[w][2];
      const double rx = b.y[0][0][res], ry = b.y[0][1][res], rz = b.y[0][2][res];
      const double sd = nx * (rx - ox) + ny * (ry - oy) + nz * (rz - oz);
      W.lj_res[live] = res, W.lj_wall[live] = w, W.lj_sat[live] = 0.0, W.lj_gone[live] = 0;
      W.lj_off[0][live] = (rx - sd * nx) - ox;
      W.lj_off[1][live] = (ry - sd * ny) - oy;
      W.lj_off[2][live] = (rz - sd * nz) - oz;
      ++live;
      ++W.num_conns[w];
    }
    W.n_cand = 0;
    W.n_gone = 0;
    st.n_lj = live;
  }
}

// ------------------------------------------------------------- box protocol ----
// state::reinit_wall_values (cg/src/cg/simul/state.cpp:708-729): each plane
// on a box side goes to the centre plus the projection on its normal of the
// vector to its face; shift = new origin - old; periodic axes take the box
// extent as their PBC cell
__device__ void box_reinit(WallDev &W, DevParams *P, SysDesc *sd) {
#pragma clang fp contract(off)
  double center[3], ext[3];
  for (int c = 0; c < 3; ++c) {
    center[c] = (W.box_max[c] + W.box_min[c]) / 2.0;
    ext[c] = W.box_max[c] - W.box_min[c];
  }
  for (int side = 0; side < 6; ++side) {
    const int w = W.side_wall[side];
    if (w < 0) continue;
    double d[3], *o = P->p.wall_origin[w];
    const double *n = P->p.wall_normal[w];
    for (int c = 0; c < 3; ++c) d[c] = (side % 2 == 1 ? W.box_max[c] : W.box_min[c]) - center[c];
    const double proj = d[0] * n[0] + d[1] * n[1] + d[2] * n[2];
    for (int c = 0; c < 3; ++c) {
      const double next = center[c] + n[c] * proj;
      W.shift[w][c] = next - o[c];
      o[c] = next;
    }
  }
  for (int c = 0; c < 3; ++c) {
    const double cell = W.bx.pbc[c] ? ext[c] : 0.0;
    sd->cell[c] = cell;
    sd->cell_inv[c] = cell != 0.0 ? 1.0 / cell : 0.0;
  }
}

// state::adjust_wall_pos (state.cpp:702-706) along z, or with the same
// change on every axis
__device__ __forceinline__ void box_adjust(WallDev &W, DevParams *P, SysDesc *sd, const double *size_change) {
#pragma clang fp contract(off)
  for (int c = 0; c < 3; ++c) {
    W.box_min[c] += -size_change[c] + 0.0;
    W.box_max[c] += size_change[c] + 0.0;
  }
  box_reinit(W, P, sd);
}

// state::setup_walls' box part: averages reset, planes to the faces
__global__ void k_box_setup(DevBatch b, DevParams *P, SysDesc *sd) {
  if (threadIdx.x != 0) return;
  WallDev &W = *b.wall;
  for (int w = 0; w < 6; ++w) {
    W.avg_F[w] = MAvg{};
    W.avg_F[w].window = W.bx.avg_forces_over;
    W.work[w] = 0.0;
  }
  W.avg_z = MAvg{};
  W.avg_z.window = W.bx.avg_forces_over;
  box_reinit(W, P, sd);
}

// The phase logic of thread_main.cpp:144-330 before a step: the phase
// changes of this time (which take no step in the reference) and the wall
// move of the phase that then advances.
__global__ void k_box_phase(DevBatch b, DevParams *P, SysDesc *sd) {
#pragma clang fp contract(off)
  if (threadIdx.x != 0) return;
  WallDev &W = *b.wall;
  const SysState &st = b.st[0];
  if (!st.active || W.phase == PCG_PHASE_NONE) return;
  const pcg_box &bx = W.bx;
  const double t = st.t, dt = P->p.dt, num_res = (double)sd->n;
  const double pi = 3.14159265358979323846, pi_2 = 1.57079632679489661923;
  for (int guard = 0; guard < 16; ++guard) {
    switch (W.phase) {
    case PCG_PHASE_SQUEEZING: {  // squeezing_step, thread_main.cpp:144-181
      if (!bx.squeezing) {
        W.since = t;
        W.phase = PCG_PHASE_FIND_FORCE_MIN;
        continue;
      }
      const double ex = W.box_max[0] - W.box_min[0], ey = W.box_max[1] - W.box_min[1],
                   ez = W.box_max[2] - W.box_min[2];
      const double cur_vol = ex * ey * ez, target_vol = num_res / bx.target_density;
      if (cur_vol <= target_vol) {
        W.until = fmin(t + bx.rest_period, bx.total_time);
        W.phase = PCG_PHASE_REST_AFTER_SQUEEZING;
        continue;
      }
      double vel;
      if (cur_vol > 2.0 * target_vol) {
        const double accel_time = bx.accel_dist / bx.vel_above_2V;
        vel = fmin((t - W.since) / accel_time, 1.0) * bx.vel_above_2V;
      } else {
        const double accel_time = bx.accel_dist / bx.target_vel;
        vel = fmin((t - W.since) / accel_time, 1.0) * bx.target_vel;
      }
      const double sh = 0.5 * vel * dt, ch[3] = {-sh, -sh, -sh};
      box_adjust(W, P, sd, ch);
      return;
    }
    case PCG_PHASE_REST_AFTER_SQUEEZING:  // :183-191
      if (t < W.until) return;
      W.phase = PCG_PHASE_FIND_FORCE_MIN;
      continue;
    case PCG_PHASE_FIND_FORCE_MIN: {  // :193-222
      if (!bx.force_min) {
        W.phase = PCG_PHASE_FREEFORM;
        continue;
      }
      if (W.avg_z.has && fabs(W.avg_z.avg[0]) < 5e-2 + 5e-5 * num_res) {
        W.until = t + bx.rest_period;
        W.phase = PCG_PHASE_REST_AFTER_FORCE_MIN;
        continue;
      }
      const double accel_time = bx.accel_dist / bx.target_vel;
      const double time_vel_frac = fmin((t - W.since) / accel_time, 1.0);
      double fvf = (W.avg_z.has ? W.avg_z.avg[0] : 0.0) / bx.force_for_max_vel;
      fvf = copysign(fmin(fabs(fvf), 1.0), fvf);
      const double vel = bx.target_vel * time_vel_frac * fvf;
      const double sh = 0.5 * vel * dt, ch[3] = {0.0, 0.0, sh};
      box_adjust(W, P, sd, ch);
      return;
    }
    case PCG_PHASE_REST_AFTER_FORCE_MIN:  // :224-243
      if (t < W.until) return;
      if (!bx.amp_relative) {
        W.amplitude = bx.amp_abs;
      } else {
        W.shear = bx.osc_shear != 0;
        const double base_val = W.shear ? W.box_max[0] - W.box_min[0] : W.box_max[2] - W.box_min[2];
        W.amplitude = bx.amp_rel * base_val;
      }
      W.since = t;
      W.phase = PCG_PHASE_MAX_AMPLITUDE;
      continue;
    case PCG_PHASE_MAX_AMPLITUDE: {  // :245-276
      if (!bx.oscillations) {
        W.phase = PCG_PHASE_FREEFORM;
        continue;
      }
      const double accel_time = bx.accel_dist / bx.target_vel;
      const double vel = fmin((t - W.since) / accel_time, 1.0) * bx.target_vel;
      const double sh = vel * dt;
      if (W.displacement > 0.5 * W.amplitude) {
        W.until = t + bx.rest_period;
        W.phase = PCG_PHASE_REST_AFTER_MAX_AMP;
        continue;
      }
      W.displacement += sh;
      if (W.shear) {
        for (int side = 4; side < 6; ++side)
          if (W.side_wall[side] >= 0) P->p.wall_normal[W.side_wall[side]][0] += sh;
      } else {
        const double ch[3] = {0.0, 0.0, -sh};
        box_adjust(W, P, sd, ch);
      }
      return;
    }
    case PCG_PHASE_REST_AFTER_MAX_AMP:  // :278-293
      if (t < W.until) return;
      W.since = t;
      W.omega = bx.angular_freq;
      W.until = t + (pi * 2 * bx.num_of_cycles + pi_2) / W.omega;
      W.phase = PCG_PHASE_OSCILLATIONS;
      continue;
    case PCG_PHASE_OSCILLATIONS: {  // :295-320
      if (t >= W.until) {
        W.until = t + bx.rest_period;
        W.phase = PCG_PHASE_REST_AFTER_OSCILLATIONS;
        continue;
      }
      const double vel = 0.5 * W.amplitude * W.omega * sin(W.omega * (t - W.since));
      const double sh = vel * dt;
      if (W.shear) {
        for (int side = 4; side < 6; ++side)
          if (W.side_wall[side] >= 0) P->p.wall_normal[W.side_wall[side]][0] += sh;
      } else {
        const double ch[3] = {0.0, 0.0, sh};
        box_adjust(W, P, sd, ch);
      }
      return;
    }
    case PCG_PHASE_REST_AFTER_OSCILLATIONS:  // :322-330
      if (t < W.until) return;
      W.phase = PCG_PHASE_FREEFORM;
      continue;
    default:
      return;
    }
  }
}

// ------------------------------------------------------------- launchers ----
static inline dim3 grid1(int n, int blk = BLK) { return dim3((unsigned)((n + blk - 1) / blk)); }

void launch_begin(const DevBatch &b, hipStream_t s) {
  hipLaunchKernelGGL(k_begin, grid1(b.nsys, 64), dim3(64), 0, s, b);
}
void launch_eval_begin(const DevBatch &b, hipStream_t s) {
  hipLaunchKernelGGL(k_eval_begin, grid1(b.ntot), dim3(BLK), 0, s, b);
}
void launch_store_forces(const DevBatch &b, hipStream_t s) {
  hipLaunchKernelGGL(k_move_forces<true>, grid1(b.ntot), dim3(BLK), 0, s, b);
}
void launch_load_forces(const DevBatch &b, hipStream_t s) {
  hipLaunchKernelGGL(k_move_forces<false>, grid1(b.ntot), dim3(BLK), 0, s, b);
}
void launch_near_fields(const DevBatch &b, hipStream_t s) {
  hipLaunchKernelGGL(k_near_fields, dim3(16, (unsigned)b.nsys), dim3(BLK), 0, s, b);
}
void launch_mark_invalid(const DevBatch &b, hipStream_t s) {
  hipLaunchKernelGGL(k_mark_invalid, grid1(b.nsys, 64), dim3(64), 0, s, b);
}
void launch_fetch(const Fetch &f, hipStream_t s) {
  const int most = std::max((int)(f.bytes / 4), 3 * f.n);
  const dim3 block((unsigned)std::min(1024, std::max(64, (most + 63) / 64 * 64)));
  const dim3 grid(f.flag ? 1u : (unsigned)std::min(64, std::max(1, (most + 1023) / 1024)));
  if (f.f32)
    hipLaunchKernelGGL(k_fetch<float>, grid, block, 0, s, (const uint32_t *)f.src,
                       (uint32_t *)f.dst, (int)(f.bytes / 4), (const float *)f.cols[0],
                       (const float *)f.cols[1], (const float *)f.cols[2], f.acc, f.out, f.n, f.flag,
                       f.seq);
  else
    hipLaunchKernelGGL(k_fetch<double>, grid, block, 0, s, (const uint32_t *)f.src,
                       (uint32_t *)f.dst, (int)(f.bytes / 4), (const double *)f.cols[0],
                       (const double *)f.cols[1], (const double *)f.cols[2], (const double *)nullptr, f.out, f.n,
                       f.flag, f.seq);
}
void launch_noise_in(const DevBatch &b, const double *src, hipStream_t s) {
  hipLaunchKernelGGL(k_noise_in, grid1(b.ntot), dim3(BLK), 0, s, b, src);
}
void launch_prepare_nh(const DevBatch &b, hipStream_t s) {
  hipLaunchKernelGGL(k_prepare_nh, grid1(b.ntot), dim3(BLK), 0, s, b);
}
void launch_fix_nl(const DevBatch &b, int max_n, int cell_words, hipStream_t s, bool step,
                   int qa_on) {
  int rows_per_block = BLK / 64;
  dim3 rg((unsigned)((b.ntot + rows_per_block - 1) / rows_per_block));
  const size_t mask_lds = (size_t)rows_per_block * cell_words * sizeof(unsigned long long);
  const int begin = step ? 1 : 0, cells = cell_words > 0;
  // the cell counts and, for smaller systems, the row counts are scanned by
  // the wave that completes them
  if (cells) {
    hipLaunchKernelGGL(k_cell_count, grid1(b.ntot), dim3(BLK), 0, s, b, begin, qa_on);
    hipLaunchKernelGGL(k_cell_fill, grid1(b.ntot), dim3(BLK), 0, s, b);
  }
  const int fuse = max_n < ROWS_FUSE_MAX;
  hipLaunchKernelGGL(k_nl_rows<false>, rg, dim3(BLK), mask_lds, s, b, cell_words, fuse,
                     cells ? 0 : begin, qa_on);
  if (!fuse) hipLaunchKernelGGL(k_nl_scan, dim3((unsigned)b.nsys), dim3(64 * (RC_N + 1)), 0, s, b);
  hipLaunchKernelGGL(k_nl_rows<true>, rg, dim3(BLK), mask_lds, s, b, cell_words, fuse, 0, 0);
  if (!step) hipLaunchKernelGGL(k_nl_done, dim3((unsigned)b.nsys), dim3(BLK), 0, s, b);
}
int fix_nl_launches(int max_n, int cell_words) {
  return (cell_words > 0 ? 2 : 0) + (max_n < ROWS_FUSE_MAX ? 2 : 3);
}
void launch_terms(const DevBatch &b, int prec, int max_items, int term, int from, int to,
                  hipStream_t s) {
  int gx = (max_items + BLK - 1) / BLK;
  if (gx < 1) gx = 1;
  if (gx > 512) gx = 512;
  dim3 g((unsigned)gx, (unsigned)b.nsys);
  if (prec == PCG_FP64)
    hipLaunchKernelGGL(k_terms<double>, g, dim3(BLK), 0, s, b, term, from, to);
  else
    hipLaunchKernelGGL(k_terms<float>, g, dim3(BLK), 0, s, b, term, from, to);
}
void launch_step_terms(const DevBatch &b, int prec, int max_n, bool step, hipStream_t s) {
  // a wave for some four residues: the chunks of the usual force field (bonded
  // n / 64, native contacts and QA near pairs n / 4 and more); longer lists
  // stride. At most eight waves a SIMD of the chip.
  const int gx = std::max(16, std::min((max_n / 4 + 3) / 4, 2048));
  dim3 g((unsigned)gx, (unsigned)b.nsys);
  if (prec == PCG_FP64)
    hipLaunchKernelGGL(k_step_terms<double>, g, dim3(BLK), 0, s, b, step ? 1 : 0);
  else
    hipLaunchKernelGGL(k_step_terms<float>, g, dim3(BLK), 0, s, b, step ? 1 : 0);
}
size_t qa_finish_lds(int max_n) {
  return sizeof(QfLds) + 4 * (((size_t)max_n + 1) & ~(size_t)1);
}
void launch_qa_finish(const DevBatch &b, int max_n, hipStream_t s) {
  // the budgets in LDS while they and the candidates fit QF_LDS_MAX
  const size_t lds = qa_finish_lds(max_n);
  const int sync_lds = lds <= QF_LDS_MAX ? max_n : 0;
  hipLaunchKernelGGL(k_qa_finish, dim3(b.nsys), dim3(1024), sync_lds ? lds : 0, s, b, sync_lds);
}
void launch_lang(const DevBatch &b, int prec, int noise_mode, const double *noise,
                 hipStream_t s, bool tick, bool log) {
  const int t = tick ? 1 : 0, l = log ? 1 : 0;
  dim3 g = grid1(b.ntot);
  g.x += l;
  if (prec == PCG_FP64)
    hipLaunchKernelGGL(k_lang<double>, g, dim3(BLK), 0, s, b, noise_mode, noise, t, l);
  else
    hipLaunchKernelGGL(k_lang<float>, g, dim3(BLK), 0, s, b, noise_mode, noise, t, l);
}
void launch_tick(const DevBatch &b, int advance, hipStream_t s) {
  hipLaunchKernelGGL(k_tick, grid1(b.nsys, 64), dim3(64), 0, s, b, advance);
}
void launch_ljw_process(const DevBatch &b, hipStream_t s) {
  hipLaunchKernelGGL(k_ljw_process, dim3(1), dim3(1024), 0, s, b);
}
void launch_box_setup(const DevBatch &b, DevParams *P, SysDesc *sd, hipStream_t s) {
  hipLaunchKernelGGL(k_box_setup, dim3(1), dim3(64), 0, s, b, P, sd);
}
void launch_box_phase(const DevBatch &b, DevParams *P, SysDesc *sd, hipStream_t s) {
  hipLaunchKernelGGL(k_box_phase, dim3(1), dim3(64), 0, s, b, P, sd);
}
} // namespace pcg
