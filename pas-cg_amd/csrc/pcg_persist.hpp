// pcg_persist.hpp -- the persistent form's device code: one workgroup owns one
// system and runs many whole steps of thread::advance_by_step
// (cg/src/cg/simul/thread_main.cpp:373-536) inside a single launch.
//
// Positions (FP64) and forces (R) of the system stay in LDS across steps;
// force terms accumulate with LDS atomics; the NL rebuild, the ordered list
// partition and the QA finish run inside the workgroup; the Gear-5 state is
// in LDS too, or streamed from/to HBM where it does not fit. Systems are
// independent, so workgroups never synchronise with each other.
//
// pcg_batch.hip instantiates the general kernels, pcg_batch_lean.hip the lean
// ones.
#pragma once
#include "pcg_launch.hpp"
#include "pcg_stages.hpp"

namespace pcg {

// The batch descriptor in constant memory (the kernel's arguments, or the
// served form's job array). A phase of the step takes its own copy of the
// fields it uses through unpack(): the address passes through an empty asm
// statement, so the compiler cannot hoist those scalar loads out of the step
// loop. Hoisted, the descriptor's pointers and the parameters they lead to
// (some 400 scalar registers) were spilled into VGPR lanes and read back at
// every use.
typedef const PCG_CONST_AS DevBatch DevBatchC;
__device__ __forceinline__ DevBatch unpack(DevBatchC *bp) {
  asm volatile("" : "+s"(bp));
  DevBatch b;
  __builtin_memcpy_inline(&b, (const DevBatch *)bp, sizeof(DevBatch));
  return b;
}

// Whose turn it is: each force term's items start at the wave after the one
// that took the term before's last item, so that short terms spread over the
// workgroup's waves instead of all falling on the first.
struct TermTurn {
  int wave, nw;  // uniform
  // the thread's first item of a term of n items
  __device__ __forceinline__ int first(int n) {
    int w = (int)(threadIdx.x >> 6) - wave;
    if (w < 0) w += nw;
    skip(n);
    return w * 64 + (int)(threadIdx.x & 63);
  }
  __device__ __forceinline__ void skip(int n) {
    const int used = wave + ((n + 63) >> 6);
    wave = used < nw ? used : used % nw;
  }
};

// Geometry and per-residue QA data of the workgroup's system, from LDS.
struct GeoL {
  const double *x, *y, *z;
  int res0;
  const uint8_t *at;       // residue type | has chain predecessor << 6 | successor << 7
  const uint32_t *sync;    // the four sync budgets of each residue, one byte each
  const int8_t *ptype_t;   // polarity class per residue type
  const double *req_t;     // r_high[type] * (1 + formation_tol) per QA type
  __device__ __forceinline__ v3<double> r(int i) const {
    int k = i - res0;
    return v3<double>{x[k], y[k], z[k]};
  }
  __device__ __forceinline__ int atype(const DevBatch &, int i) const { return at[i - res0] & 63; }
  __device__ __forceinline__ int ptype(const DevBatch &, int a) const { return ptype_t[a]; }
  __device__ __forceinline__ uint32_t sync4(const DevBatch &, int i) const { return sync[i - res0]; }
  __device__ __forceinline__ double type_req(const DevBatch &, int t) const { return req_t[t]; }
  // n and h of residue i as wg_prepare_nh left them for this step
  __device__ __forceinline__ void nh(const DevBatch &b, int i, double out[6]) const {
    for (int c = 0; c < 6; ++c) out[c] = b.nh[c][i];
  }
};

// qa::prepare_nh (cg/src/cg/qa/prepare_nh.cpp:10-19) over the workgroup's
// system, from the LDS positions, into the batch's n and h arrays (the chain
// neighbours of residue i are i - 1 and i + 1; zero at chain ends, where
// prepare_nh writes nothing). Run once per step after the positions move,
// so that a QA pair reads its residues' vectors instead of recomputing them.
__device__ __forceinline__ void wg_prepare_nh(DevBatchC *bp, const GeoL &g, int n, int r0,
                                              TermTurn &turn) {
  const DevBatch b = unpack(bp);
  for (int k = turn.first(n); k < n; k += blockDim.x) {
    const int i = r0 + k;
    double o[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if ((g.at[k] & 0xC0) == 0xC0) nh_from(g.r(i), g.r(i - 1), g.r(i + 1), o);
    for (int c = 0; c < 6; ++c) b.nh[c][i] = o[c];
  }
}

template <typename RF> struct AccL {
  RF *fx, *fy, *fz;
  int res0;
  template <typename T> __device__ __forceinline__ void add(int i, v3<T> f) {
    int k = i - res0;
    atomicAdd(fx + k, (RF)f.x);
    atomicAdd(fy + k, (RF)f.y);
    atomicAdd(fz + k, (RF)f.z);
  }
};

// Maximum over the workgroup, in every thread: each wave's maximum goes to
// part[wave], then, past the barrier, every thread reads them all. part is
// next written one step later, past the barrier that ends that step's force
// terms, so one barrier suffices.
__device__ __forceinline__ double block_max(double v, double *part) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_down(v, o, 64));
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) part[w] = v;
  __syncthreads();
  double m = 0.0;
  for (int k = 0; k < (int)(blockDim.x >> 6); ++k) m = fmax(m, part[k]);
  return m;
}

// Tallies of the list rebuild: NL pairs, then the pairs of each list the
// ordered partition fills (native contacts, QA free pairs, the QA free pairs
// that can become candidates, PID, DH, Pauli).
enum { KC_NEAR = 1, KC_PID = 2, KC_DH = 4, KC_PAULI = 8 };  // a kept pair's lists
enum { RB_NL = 0, RB_NC, RB_QA, RB_NEAR, RB_PID, RB_DH, RB_PAULI, RB_N };

// Cost of the rows before row k in the rebuild's first pass, in 64-column
// chunks: row k visits the chunks from its next residue's to the last, and
// costs about a chunk and a half of its own.
__device__ __forceinline__ int rb_cost(int k, int n) {
  const int W = (n + 63) >> 6, q = k >> 6, r = k & 63;
  return 2 * (k * W - (32 * q * (q - 1) + q * (r + 1))) + 3 * k;  // in half chunks
}
// First row of wave w's block when nw waves split the rows into contiguous
// blocks of about equal cost. Monotone in w, 0 for w = 0 and n for w = nw.
__device__ __forceinline__ int rb_row_start(int w, int nw, int n) {
  if (w <= 0) return 0;
  if (w >= nw) return n;
  const int want = (int)((float)rb_cost(n, n) * ((float)w / (float)nw));
  int lo = 0, hi = n;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (rb_cost(mid, n) < want) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ float lane_f32(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

__device__ __forceinline__ unsigned long long lane_u64(unsigned long long v, int lane) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)v, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(v >> 32), lane);
  return (unsigned long long)lo | ((unsigned long long)hi << 32);
}

// nl::legacy_update (cg/src/cg/nl/legacy_update.cpp:11-55) fused with the
// ordered list updates of thread_main.cpp:409-423 and the QA near list,
// inside the workgroup and without writing the NL itself. The rows of the
// sorted NL (pairs i < j) are split into contiguous blocks of about equal
// cost, one per wave, and handled in three stages:
//
// scan      each row against every later column, 64 at a time: the pairs
//           within the NL radius and within the native-contact radius are
//           counted, the pairs that may join a list kept in order;
// classify  the kept pairs, 64 at a time, as the partition would classify the
//           NL pair (native contacts and QA free pairs take; PID bundle, DH
//           pair, Pauli pair), by their exact FP64 distance;
// write     once a scan over the waves has given each wave its offsets: every
//           kept pair at its wave's offset plus its rank among the block's
//           earlier pairs of that list, so the lists come out exactly in the
//           order of partitioning the sorted NL.
//
// The native contacts come from their own sorted list, which is the NL's
// order, a contiguous run of contacts a wave.
//
// The scan tests all n (n - 1) / 2 pairs. It is bound by the instructions each
// wave runs through one after another (measured: 5 cycles a dependent vector
// instruction, 7 a scalar one, 10 where a scalar one waits for a compare),
// not by the vector unit: classifying each 64 columns on the spot took 2500
// cycles for them, mostly scalar logic and branches. Now 64 columns cost one
// 16-byte LDS read of FP32 positions (relative to residue 0, staged over the
// force accumulators, which are zero during a rebuild), the squared distance,
// two counts and one test for every reason to keep a pair; the row's data come
// from registers by readlane. A rebuild of a 600-residue protein on 1024
// threads takes 95 us instead of 280, of a 56-residue one 15 us instead of 41.
//
// Every decision is the FP64 one of the reference's expressions. The scan's
// FP32 comparison counts a pair when its squared distance is clear of the
// threshold by a relative margin of 2e-5 + 1e-6 M / d (M the largest
// coordinate staged, d the threshold): staging rounds a coordinate by at most
// 2^-24 M and the difference, squares and sums round by at most a few 2^-24,
// together less than 4.2e-7 M / d + 4e-7. Pairs inside a margin are kept and
// counted by the classification. In a periodic cell, and in a system with a
// coordinate beyond 1e4 NL radii or none at all (a diverged one: up to there
// the margin is a hundredth, an infinite one would keep every column), the
// differences are formed (and wrapped) in FP64 and rounded afterwards (M = 0).
//
// QA free pairs beyond the QA maximum required distance are counted (qf_n,
// which sizes the contact loop as the reference's free-pair count does) but
// not stored: with total_disp reset after every verify
// (cg/src/cg/nl/verify.cpp:31-32) loop_over_candidates skips them until the
// next rebuild (qa/loop_over_candidates.cpp:20), and the stored pairs keep
// their relative order, so the (distance, free-pair index) order of the QA
// finish is unchanged.
//
// rb: the LDS region of the QA stacks, free during a rebuild: the residues'
// sequence words, the row starts of the static native contacts and the
// contacts' second residues. force: the force accumulators (24 n bytes from a
// multiple of 8, zero again after); pos4: the multiple of 16 from there.
// (inlined: as a call it would make the kernel save every live register)
__device__ __forceinline__ void wg_fix_nl(DevBatchC *bp, int s, SysState &st, const GeoL &g,
                                          void *rb, double *force, float4 *pos4,
                                          uint32_t chg) {
#pragma clang fp contract(off)
  typedef unsigned long long u64;
  const DevBatch b = unpack(bp);
  SysDescC &sd = b.sys[s];
  DevParamsC &P = *b.P;
  ParamsC &p = P.p;
  const int n = sd.n, r0 = sd.res0;
  // the wave's index, known to the compiler as uniform: the row loops below
  // are then scalar loops and the running counts scalar registers
  const int nw = blockDim.x >> 6, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int nnc = p.nat_cont_on ? sd.nnc : 0;
  // each residue's sequence index, chain and type in one word (seq | chain
  // << 12 | type << 24: a persistent system has fewer than 4096 residues)
  uint32_t *csq = (uint32_t *)rb;
  int *rs = (int *)(csq + n);  // rs[0..n]
  uint16_t *pj = (uint16_t *)(rs + n + 1);               // [nnc]
  __shared__ int wcnt[16][RB_N];
  __shared__ float wspan[16];
  __shared__ int wirr[16];
  __shared__ u64 charge_mask[64];  // the charged residues of each 64
  const bool cell = has_cell(sd);
  const float far_from = 1e4f * (float)(P.nl_eff_cutoff + p.nl_pad);
  const double ox = g.x[0], oy = g.y[0], oz = g.z[0];
  float span = 0.0f;
  bool irr = false, far = false;
  for (int k0 = threadIdx.x - lane; k0 < n; k0 += blockDim.x) {
    const int k = k0 + lane;
    const u64 cm = __ballot(k < n && ((chg >> (g.at[min(k, n - 1)] & 31)) & 1u));
    if (lane == 0) charge_mask[k0 >> 6] = cm;
    if (k >= n) continue;
    const int ch = b.chain[r0 + k], sq = b.seq[r0 + k];
    csq[k] = (uint32_t)sq | ((uint32_t)ch << 12) | ((uint32_t)(g.at[k] & 63) << 24);
    // the usual numbering: chains one after another, consecutive sequence
    // indices within one; then a pair's sequence distance is j - k, and the
    // exclusions concern only the four columns after the row's residue: bit
    // d - 1 of mate tells whether residue k + d is of the same chain
    uint32_t mate = 0u;
    for (int d = 1; d <= 4; ++d)
      if (k + d < n && b.chain[r0 + k + d] == ch) mate |= 1u << (d - 1);
    if (k + 1 < n) {
      const int c1 = b.chain[r0 + k + 1];
      irr |= c1 < ch || (c1 == ch && b.seq[r0 + k + 1] != sq + 1);
    }
    const float fx = (float)(g.x[k] - ox), fy = (float)(g.y[k] - oy), fz = (float)(g.z[k] - oz);
    span = fmaxf(span, fmaxf(fabsf(fx), fmaxf(fabsf(fy), fabsf(fz))));
    far |= !(fabsf(fx) <= far_from) | !(fabsf(fy) <= far_from) | !(fabsf(fz) <= far_from);
    pos4[k] = make_float4(fx, fy, fz, __builtin_bit_cast(float, (uint32_t)(g.at[k] & 31) | (mate << 8)));
  }
  for (int o = 32; o > 0; o >>= 1) span = fmaxf(span, __shfl_down(span, o, 64));
  const int wave_irr = (__any(irr) ? 1 : 0) | (__any(far) ? 2 : 0);
  if (lane == 0) {
    wspan[w] = span;
    wirr[w] = wave_irr;
  }
  // contacts sd.nc0 + [rs[k], rs[k + 1]) of the list sorted by (i1, i2) are
  // those of residue r0 + k with later residues; pj holds their second
  // residues within the system
  if (nnc == 0) {
    for (int k = threadIdx.x; k <= n; k += blockDim.x) rs[k] = 0;
  } else {
    for (int c = threadIdx.x; c < nnc; c += blockDim.x) {
      const int a = b.nc_i[0][sd.nc0 + c] - r0;
      const int prev = c > 0 ? b.nc_i[0][sd.nc0 + c - 1] - r0 : -1;
      pj[c] = (uint16_t)(b.nc_i[1][sd.nc0 + c] - r0);
      for (int r = prev + 1; r <= a; ++r) rs[r] = c;
      if (c == nnc - 1)
        for (int r = a + 1; r <= n; ++r) rs[r] = nnc;
    }
  }
  const double pad = p.nl_pad;
  const double t_nl = __dadd_rn(P.nl_eff_cutoff, pad);
  const double t_nc = __dadd_rn(p.nl_cutoff, pad);
  const double t_dh = __dadd_rn(p.dh_cutoff, pad);
  const double t_rep = __dadd_rn(p.rep_cutoff, pad);
  const double t_near = P.qa_max_req;
  const double rt_dh = __ddiv_rn(1.0, t_dh);
  const bool qa_on = p.qa_on, pid_on = p.pid_on, dh_on = p.dh_on, pauli_on = P.pauli_on;
  const bool qa4 = p.qa_include4, pid4 = p.pid_include4;
  __syncthreads();
  int all_irr = 0;
  span = 0.0f;
  for (int v = 0; v < nw; ++v) {
    span = fmaxf(span, wspan[v]);
    all_irr |= wirr[v];
  }
  const bool regular = !(all_irr & 1), by64 = cell | ((all_irr & 2) != 0);
  if (by64) span = 0.0f;
  // squared thresholds in FP32, their margins (half) in the FP32 comparisons,
  // and the bounds clear of them; in scalar registers
  auto half = [&](double t) {
    const float tf = (float)t;
    return tf * tf * (2e-5f + 1e-6f * span * rcpR(tf));
  };
  auto sq32 = [&](double t) { return (float)(t * t); };
  auto uni = [&](float x) { return lane_f32(x, 0); };
  const float nl_c = uni(sq32(t_nl)), nc_c = uni(sq32(t_nc));
  // the NL and native-contact radii share the wider of their margins
  const float h_nl = uni(fmaxf(half(t_nl), half(t_nc)));
  const float nl_lo = nl_c - h_nl, nl_hi = nl_c + h_nl, nc_lo = nc_c - h_nl, nc_hi = nc_c + h_nl;
  const float band = h_nl * 1.001f;  // (with the comparison's own rounding)
  const float dh_lo = uni(sq32(t_dh) - half(t_dh)), dh_hi = uni(sq32(t_dh) + half(t_dh));
  const float near_lo = uni(sq32(t_near) - half(t_near)), near_hi = uni(sq32(t_near) + half(t_near));
  const float rep_lo = uni(sq32(t_rep) - half(t_rep)), rep_hi = uni(sq32(t_rep) + half(t_rep));
  // every pair this close is kept for the classification
  float keep_to = -1.0f;
  if (qa_on) keep_to = fmaxf(keep_to, near_hi);
  if (pauli_on) keep_to = fmaxf(keep_to, rep_hi);
  if (pid_on && !qa_on) keep_to = fmaxf(keep_to, nc_hi);
  const float keep_c = keep_to * 1.00001f - band;
  // pairs four apart are told apart by the lists' own options
  const bool keep4 = (qa_on && !qa4) || (pid_on && !pid4);
  const int kbeg = rb_row_start(w, nw, n), kend = rb_row_start(w + 1, nw, n);
  // the kept pairs, k | j << 12 | classes << 24, go to nl_i[0]: when every
  // pair fits the NL capacity a wave's region starts at the index of its
  // block's first pair, which no other wave's pairs reach; else each wave has
  // an equal share and takes its rows in batches whose pairs fit it, scanned
  // and classified in both passes
  const bool compact = (long long)n * (n - 1) / 2 <= (long long)sd.nlcap;
  const int share = compact ? 0 : sd.nlcap / nw;
  uint32_t *kp = (uint32_t *)b.nl_i[0] + sd.nl0 +
                 (compact ? (int)((long long)kbeg * (n - 1) - (long long)kbeg * (kbeg - 1) / 2)
                          : w * share);
  const int batch = compact ? max(kend - kbeg, 1) : max(share / n, 1);
  const int W = (n + 63) >> 6;
  const u64 last_cols = (n & 63) ? ~0ull >> (64 - (n & 63)) : ~0ull;
  const u64 charged = lane < W ? charge_mask[lane] : 0ull;  // of chunk l, in lane l
  // the wave's native contacts: whole 64s of the list
  const int nc64 = (nnc + 63) >> 6, cper = ((nc64 + nw - 1) / nw) << 6;
  const int cbeg = min(w * cper, nnc), cend = min(cbeg + cper, nnc);
  auto word_same = [&](uint32_t wa, uint32_t wb) {
    return ((wa >> 12) & 0xFFFu) == ((wb >> 12) & 0xFFFu);
  };
  auto word_gap = [&](uint32_t wa, uint32_t wb) {
    return abs((int)(wa & 0xFFFu) - (int)(wb & 0xFFFu));
  };
  auto pair_dist = [&](int k, int j) {
    v3<double> dd = xsub(v3<double>{g.x[j], g.y[j], g.z[j]}, v3<double>{g.x[k], g.y[k], g.z[k]});
    if (cell) dd = xwrapd(dd, sd);
    return xnorm3(dd);
  };
  // a pair's squared distance as the scan sees it
  auto scan_d2 = [&](float4 q, float xi, float yi, float zi, int k, int j) {
    float dx = q.x - xi, dy = q.y - yi, dz = q.z - zi;
    if (by64) {
      const v3<double> dd = xwrapd(xsub(v3<double>{g.x[j], g.y[j], g.z[j]},
                                        v3<double>{g.x[k], g.y[k], g.z[k]}), sd);
      dx = (float)dd.x, dy = (float)dd.y, dz = (float)dd.z;
    }
    return __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
  };
  auto rank_in = [&](u64 m, int base = 0) {  // base plus the earlier lanes of the mask
    return (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                          __builtin_amdgcn_mbcnt_lo((uint32_t)m, base));
  };
  const bool plain = regular && !by64 && !keep4;
  int kept = 0;
  u64 native_in = 0ull;
  for (int pass = 0; pass < 2; ++pass) {
    int off[RB_N];
    for (int c = 0; c < RB_N; ++c) off[c] = pass ? __builtin_amdgcn_readfirstlane(wcnt[w][c]) : 0;
    for (int ka = kbeg; ka < kend; ka += batch) {
      const int kb = min(ka + batch, kend);
      if (!pass || !compact) {
        // ---- scan: the rows' pairs counted against the NL radius and the
        // native-contact radius, the close ones and those in a margin kept
        int lane_in = 0, lane_inner = 0;
        kept = 0;
        for (int kg = ka; kg < kb; kg += 64) {
          const float4 rp = pos4[min(kg + lane, n - 1)];  // 64 rows' data, one a lane
          const int kn = min(kb - kg, 64);
          if (plain) {
            // the next chunk's columns (or the next row's first) are loaded a
            // chunk ahead
            float4 nq = pos4[min((((kg + 1) >> 6) << 6) + lane, n - 1)];
            for (int r = 0; r < kn; ++r) {
              const int k = kg + r;
              const float xi = lane_f32(rp.x, r), yi = lane_f32(rp.y, r), zi = lane_f32(rp.z, r);
              const uint32_t wk = (uint32_t)__builtin_amdgcn_readlane(__builtin_bit_cast(int, rp.w), r);
              const bool row_dh = dh_on && ((chg >> (wk & 31)) & 1u);
              // the columns past the row's residue, without the two after it
              // that are of its chain, in the row's first two chunks
              const int sh = (k + 1) & 63;
              const u64 ex = (wk >> 8) & 3u;
              u64 cols = (~0ull << sh) & ~(ex << sh), cols1 = sh ? ~(ex >> (64 - sh)) : ~0ull;
              for (int jc = (k + 1) >> 6; jc < W; ++jc) {
                const int j = jc * 64 + lane;
                const float4 q = nq;
                nq = pos4[min(jc + 1 < W ? j + 64 : (((k + 2) >> 6) << 6) + lane, n - 1)];
                if (jc == W - 1) cols &= last_cols;
                const float dx = q.x - xi, dy = q.y - yi, dz = q.z - zi;
                float d2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                // (no comparison takes a NaN, whatever the thresholds)
                d2 = __builtin_amdgcn_inverse_ballot_w64(cols) ? d2 : __builtin_nanf("");
                lane_in += d2 < nl_lo ? 1 : 0;
                lane_inner += d2 < nc_lo ? 1 : 0;
                // one test for all reasons to keep a pair: inside keep_to, or
                // within band of the NL or the native-contact radius
                const float why = fminf(fminf(fabsf(d2 - nl_c), fabsf(d2 - nc_c)), d2 - keep_c);
                u64 keep = __ballot(why <= band);
                if (row_dh) {
                  u64 dm = lane_u64(charged, jc) & __ballot(d2 <= dh_hi);
                  if (qa_on) dm &= ~__ballot(d2 < nc_lo);
                  keep |= dm;
                }
                if (__builtin_amdgcn_inverse_ballot_w64(keep))
                  *(uint32_t *)((char *)kp + 4u * (uint32_t)rank_in(keep, kept)) =
                      (uint32_t)k | ((uint32_t)j << 12);
                kept += __popcll(keep);
                cols = cols1;
                cols1 = ~0ull;
              }
            }
          } else {
            for (int r = 0; r < kn; ++r) {
              const int k = kg + r;
              const float xi = lane_f32(rp.x, r), yi = lane_f32(rp.y, r), zi = lane_f32(rp.z, r);
              const uint32_t wi = csq[k];
              const bool row_dh = dh_on && ((chg >> ((wi >> 24) & 31)) & 1u);
              for (int jc = (k + 1) >> 6; jc < W; ++jc) {
                const int j = jc * 64 + lane, jj = min(j, n - 1);
                const float d2 = scan_d2(pos4[jj], xi, yi, zi, k, jj);
                const uint32_t wj = csq[jj];
                const bool same = word_same(wi, wj);
                const u64 cols = __ballot(j > k & j < n & !(same & (word_gap(wi, wj) < 3)));
                const bool col = __builtin_amdgcn_inverse_ballot_w64(cols);
                lane_in += (col & (d2 < nl_lo)) ? 1 : 0;
                lane_inner += (col & (d2 < nc_lo)) ? 1 : 0;
                const float why = fminf(fminf(fabsf(d2 - nl_c), fabsf(d2 - nc_c)), d2 - keep_c);
                u64 keep = __ballot(why <= band);
                if (keep4) keep |= __ballot(same & (word_gap(wi, wj) == 4));
                if (row_dh) {
                  u64 dm = lane_u64(charged, jc) & __ballot(d2 <= dh_hi);
                  if (qa_on) dm &= ~__ballot(d2 < nc_lo);
                  keep |= dm;
                }
                keep &= cols;
                if (__builtin_amdgcn_inverse_ballot_w64(keep))
                  kp[rank_in(keep, kept)] = (uint32_t)k | ((uint32_t)j << 12);
                kept += __popcll(keep);
              }
            }
          }
        }
        for (int o = 32; o > 0; o >>= 1) {
          lane_in += __shfl_xor(lane_in, o, 64);
          lane_inner += __shfl_xor(lane_inner, o, 64);
        }
        int n_in = __builtin_amdgcn_readfirstlane(lane_in);
        int n_inner = __builtin_amdgcn_readfirstlane(lane_inner);
        // the stores above before the loads of other lanes' pairs below
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
        // ---- classify
        int n_four = 0;
        int cnt[RB_N] = {0};
        uint32_t next = lane < kept ? kp[lane] : 0u;
        for (int t0 = 0; t0 < kept; t0 += 64) {
          const int t = t0 + lane;
          const bool valid = t < kept;
          const uint32_t word = next;
          next = t + 64 < kept ? kp[t + 64] : 0u;
          const int k = (int)(word & 0xFFFu), j = (int)((word >> 12) & 0xFFFu);
          const float4 pk = pos4[k], pl = pos4[j];
          // a native partner? the row's contacts, eight at a time
          bool native = false;
#pragma clang loop unroll(disable)
          for (int c = rs[k], ce = rs[k + 1]; c < ce; c += 8) {
            uint16_t e[8];
            __builtin_memcpy(e, pj + c, 16);
            for (int m = 0; m < 8; ++m) native |= (c + m < ce) & (e[m] == j);
          }
          const float d2 = scan_d2(pl, pk.x, pk.y, pk.z, k, j);
          bool in = d2 < nl_lo, inner = d2 < nc_lo, b_near = d2 < near_lo, b_dh = d2 < dh_lo,
               b_rep = d2 < rep_lo;
          const bool edge = valid & ((in != (d2 <= nl_hi)) | (inner != (d2 <= nc_hi)) |
                                     (b_near != (d2 <= near_hi)) | (b_dh != (d2 <= dh_hi)) |
                                     (b_rep != (d2 <= rep_hi)));
          if (__ballot(edge)) {  // the exact FP64 decisions of the pairs in a margin
            const double dist = pair_dist(k, j);
            // (what the scan did not count)
            n_in += __popcll(__ballot(edge & !in & (dist < t_nl)));
            n_inner += __popcll(__ballot(edge & !inner & (dist < t_nl) & (dist < t_nc)));
            if (edge) {
              in = dist < t_nl;
              inner = in & (dist < t_nc);
              b_near = !(dist > t_near);
              b_dh = __ddiv_rn(1.0, dist) > rt_dh;
              b_rep = dist < t_rep;
            }
          }
          in &= valid;
          inner &= valid;
          const bool is_nc = inner & native;
          bool is4 = false;
          if (keep4) {
            const uint32_t wi = csq[k], wj = csq[j];
            is4 = word_same(wi, wj) & (word_gap(wi, wj) == 4);
            n_four += __popcll(__ballot(inner & !is_nc & is4));
          }
          const bool is_qa = qa_on & inner & !is_nc & (qa4 | !is4);
          const bool near = is_qa & b_near;
          const bool rest = in & !is_nc & !is_qa;
          const bool is_pid = pid_on & rest & inner & (pid4 | !is4);
          const uint32_t ti = __builtin_bit_cast(uint32_t, pk.w), tj = __builtin_bit_cast(uint32_t, pl.w);
          const bool is_dh = dh_on & rest & b_dh & (bool)((chg >> (ti & 31)) & (chg >> (tj & 31)) & 1u);
          const bool is_pauli = pauli_on & rest & b_rep;
          cnt[RB_NEAR] += __popcll(__ballot(near));
          cnt[RB_PID] += __popcll(__ballot(is_pid));
          cnt[RB_DH] += __popcll(__ballot(is_dh));
          cnt[RB_PAULI] += __popcll(__ballot(is_pauli));
          const uint32_t cls = (near ? KC_NEAR : 0) | (is_pid ? KC_PID : 0) | (is_dh ? KC_DH : 0) |
                               (is_pauli ? KC_PAULI : 0);
          if (valid) kp[t] = word | (cls << 24);
        }
        if (!pass) {
          off[RB_NL] += n_in;
          // the native contacts among them are taken off once they are counted
          if (qa_on) off[RB_QA] += n_inner - (qa4 ? 0 : n_four);
          off[RB_NEAR] += cnt[RB_NEAR];
          off[RB_PID] += cnt[RB_PID];
          off[RB_DH] += cnt[RB_DH];
          off[RB_PAULI] += cnt[RB_PAULI];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");
      }
      if (pass) {
        // ---- write: each kept pair into its lists at the wave's running
        // offset plus its rank among the 64's earlier pairs of the list
        uint32_t next = lane < kept ? kp[lane] : 0u;
        for (int t0 = 0; t0 < kept; t0 += 64) {
          const uint32_t word = next;
          next = t0 + 64 + lane < kept ? kp[t0 + 64 + lane] : 0u;
          const int k = (int)(word & 0xFFFu), j = (int)((word >> 12) & 0xFFFu);
          const uint32_t cls = word >> 24;  // 0 past the end
          const bool near = cls & KC_NEAR, is_pid = cls & KC_PID, is_dh = cls & KC_DH,
                     is_pauli = cls & KC_PAULI;
          const int i = r0 + k, jg = r0 + j, ai = g.at[k] & 63, aj = g.at[j] & 63;
          const u64 m_near = __ballot(near), m_pid = __ballot(is_pid), m_dh = __ballot(is_dh),
                    m_pauli = __ballot(is_pauli);
          double d64 = 0.0;
          if (near | is_pid) d64 = pair_dist(k, j);
          if (near) {
            const int fslot = off[RB_NEAR] + rank_in(m_near);
            if (fslot < sd.qfcap) {
              const int q = sd.qf0 + fslot;
              b.qf_i[0][q] = i;
              b.qf_i[1][q] = jg;
              b.qf_d[q] = d64;
              b.qf_vac[q] = 0;
              // near list entry fslot: the free pair in slot fslot (the
              // fields only the stage kernels read are left out)
              const double req = fmax(fmax(fmax(g.req_t[1], g.req_t[2]), g.req_t[3]),
                                      g.req_t[4 + ai + 21 * aj]);
              const double thr = fmin(P.qa_max_req, fmax(p.rep_cutoff, req)) * (1.0 + 1e-5);
              b.qh_slot[q] = fslot;
              b.qh_thr2[q] = (float)(thr * thr);
              b.qh_ij[q] = (uint32_t)k | ((uint32_t)j << 16);
            }
          }
          if (is_pid) {
            const int pos = off[RB_PID] + rank_in(m_pid);
            if (pos < sd.nlcap) {
              const int q = sd.nl0 + pos;
              b.pid_i[0][q] = i;
              b.pid_i[1][q] = jg;
              b.pid_d[q] = d64;
              b.pid_t[q] = (int16_t)(ai * 21 + aj);
            }
          }
          if (is_dh) {
            const int pos = off[RB_DH] + rank_in(m_dh);
            if (pos < sd.nlcap) {
              const int q = sd.nl0 + pos;
              b.dh_i[0][q] = i;
              b.dh_i[1][q] = jg;
              b.dh_q[q] = p.charge[ai] * p.charge[aj];
            }
          }
          if (is_pauli) {
            const int pos = off[RB_PAULI] + rank_in(m_pauli);
            if (pos < sd.nlcap) {
              const int q = sd.nl0 + pos;
              b.pauli_i[0][q] = i;
              b.pauli_i[1][q] = jg;
            }
          }
          off[RB_NEAR] += __popcll(m_near);
          off[RB_PID] += __popcll(m_pid);
          off[RB_DH] += __popcll(m_dh);
          off[RB_PAULI] += __popcll(m_pauli);
        }
      }
    }
    // ---- the native contacts, each from its own entry of the sorted list: a
    // wave takes a contiguous run of them, the first pass leaving the mask of
    // the t-th 64 that are in range in lane t (a wave has fewer than 4096)
    for (int c0 = cbeg; c0 < cend; c0 += 64) {
      const int c = min(c0 + lane, cend - 1), turn = (c0 - cbeg) >> 6;
      u64 m;
      if (!pass || turn >= 64) {
        const int i = b.nc_i[0][sd.nc0 + c], jg = b.nc_i[1][sd.nc0 + c];
        // (a pair listed twice counts once)
        const bool twice = c > 0 && b.nc_i[0][sd.nc0 + c - 1] == i && b.nc_i[1][sd.nc0 + c - 1] == jg;
        const uint32_t wi = csq[i - r0], wj = csq[jg - r0];
        const double dist = pair_dist(i - r0, jg - r0);
        m = __ballot((c0 + lane < cend) & !twice & (dist < t_nl) & (dist < t_nc) &
                     !(word_same(wi, wj) & (word_gap(wi, wj) < 3)));
        if (lane == turn) native_in = m;
      } else {
        m = lane_u64(native_in, turn);
      }
      if (pass && __builtin_amdgcn_inverse_ballot_w64(m))
        set_current_contact(b, sd.nc0 + off[RB_NC] + rank_in(m), sd.nc0 + c, r0);
      off[RB_NC] += __popcll(m);
    }
    if (!pass) {
      if (qa_on) off[RB_QA] -= off[RB_NC];
      if (lane == 0)
        for (int c = 0; c < RB_N; ++c) wcnt[w][c] = off[c];
      __syncthreads();
      // the waves' offsets: an exclusive scan over the waves, in wave order
      if (threadIdx.x < RB_N) {
        const int c = threadIdx.x;
        int run = 0;
        for (int v = 0; v < nw; ++v) {
          const int x = wcnt[v][c];
          wcnt[v][c] = run;
          run += x;
        }
        switch (c) {
        case RB_NL: st.nl_n = run; break;
        case RB_NC: st.nc_n = run; break;
        case RB_QA: st.qf_n = run; break;
        case RB_NEAR:
          st.qf_store = run < sd.qfcap ? run : sd.qfcap;
          st.qh_n = st.qf_store;
          if (run > sd.qfcap) st.overflow = 1;
          break;
        case RB_PID:
          st.pid_n = run < sd.nlcap ? run : sd.nlcap;
          if (run > sd.nlcap) st.overflow = 1;
          break;
        case RB_DH:
          st.dh_n = run < sd.nlcap ? run : sd.nlcap;
          if (run > sd.nlcap) st.overflow = 1;
          break;
        case RB_PAULI:
          st.pauli_n = run < sd.nlcap ? run : sd.nlcap;
          if (run > sd.nlcap) st.overflow = 1;
          break;
        }
      }
      __syncthreads();
    }
  }
  __syncthreads();
  // snapshot (legacy_update.cpp:80-89); the force accumulators back to zero
  for (int k = threadIdx.x; k < n; k += blockDim.x) {
    b.orig_r[0][r0 + k] = g.x[k];
    b.orig_r[1][r0 + k] = g.y[k];
    b.orig_r[2][r0 + k] = g.z[k];
    for (int c = 0; c < 3; ++c) force[c * n + k] = 0.0;
  }
  if (threadIdx.x == 0) {
    st.orig_pad = pad;
    for (int c = 0; c < 3; ++c) st.orig_cell[c] = sd.cell[c];
    st.nl_invalid = 0;
    st.verify_first = 0;
    st.rebuilds += 1;
  }
  __syncthreads();
}

// Per-residue bonded parameters of a chain-local system in LDS: the item
// starting at residue k of each list exists if its flag bit is set.
enum { BF_TETHER = 1, BF_LREP = 2, BF_NAT_ANG = 4, BF_HEUR_ANG = 8, BF_NAT_DIH = 16,
       BF_HEUR_DIH = 32, BF_CHIR = 64 };
struct BondLds {
  // [6][n]: tether length, native angle, native dihedral (phi0 of the simple
  // variant, cos phi0 of the complex one), sin phi0, chiral f0, f1
  double *d;
  uint8_t *u;  // [3][n]: flags, heuristic angle type, heuristic dihedral type
  int n;
  __device__ double &teth(int k) const { return d[k]; }
  __device__ double &ang(int k) const { return d[n + k]; }
  __device__ double &dih(int k) const { return d[2 * n + k]; }
  __device__ double &dihs(int k) const { return d[3 * n + k]; }
  __device__ double &c0(int k) const { return d[4 * n + k]; }
  __device__ double &c1(int k) const { return d[5 * n + k]; }
  __device__ uint8_t &flag(int k) const { return u[k]; }
  __device__ uint8_t &at(int k) const { return u[n + k]; }
  __device__ uint8_t &dt(int k) const { return u[2 * n + k]; }
};

// Once per launch: the static bonded items of every base residue, from HBM
// into LDS (the per-step loop then reads no list of these terms from HBM).
__device__ __forceinline__ void stage_bonded(const DevBatch &b, SysDescC &sd, const BondLds &bl) {
  for (int k = threadIdx.x; k < sd.n; k += blockDim.x) {
    int r = sd.res0 + k, it;
    uint8_t f = 0;
    if ((it = b.bond_item[BOND_TETHER][r]) >= 0) f |= BF_TETHER, bl.teth(k) = b.teth_nat[it];
    if ((it = b.bond_item[BOND_LREP][r]) >= 0) f |= BF_LREP;
    if ((it = b.bond_item[BOND_NAT_ANG][r]) >= 0) f |= BF_NAT_ANG, bl.ang(k) = b.nang_th[it];
    if ((it = b.bond_item[BOND_HEUR_ANG][r]) >= 0) f |= BF_HEUR_ANG, bl.at(k) = b.hang_t[it];
    if ((it = b.bond_item[BOND_NAT_DIH][r]) >= 0) {
      f |= BF_NAT_DIH;
      const double phi0 = b.ndih_ph[it];
      if (b.P->p.nat_dih_variant == 0) {
        double s0, c0;
        sincos(phi0, &s0, &c0);
        bl.dih(k) = c0;
        bl.dihs(k) = s0;
      } else {
        bl.dih(k) = phi0;
      }
    }
    if ((it = b.bond_item[BOND_HEUR_DIH][r]) >= 0) f |= BF_HEUR_DIH, bl.dt(k) = b.hdih_t[it];
    if ((it = b.bond_item[BOND_CHIR][r]) >= 0) {
      f |= BF_CHIR;
      bl.c0(k) = b.chir_f0[it];
      bl.c1(k) = b.chir_f1[it];
    }
    bl.flag(k) = f;
  }
}

template <typename RF> __device__ __forceinline__ RF shfl_up_rf(RF v, int d) {
  return __shfl_up(v, (unsigned)d, 64);
}

// The static bonded terms of a system whose items are all chain-local. Each
// thread takes one base residue per pass (consecutive residues on consecutive
// lanes) and evaluates the items that start there; a residue's force is its
// own share plus the shares lanes 1..3 below it computed for it, gathered
// with cross-lane shifts, and one LDS add per component. Shares that would
// cross into the next wave go to LDS directly.
template <typename RF, bool STAGED, bool LEAN>
__device__ __forceinline__ void bonded_by_base(DevBatchC *bp, int sys, SysState &st,
                                               const GeoL &g, const BondLds &bl, double *fx,
                                               double *fy, double *fz, double *vacc, bool want_v) {
  const DevBatch b = unpack(bp);
  ParamsC &p = b.P->p;
  const int n = b.sys[sys].n, r0 = b.sys[sys].res0, lane = threadIdx.x & 63;
  // energies only on the step that reports them, added per item (no
  // accumulators live across the items: registers are the scarce resource)
  auto ev = [&](int term, double V) {
    if (want_v && V != 0.0) atomicAdd(&vacc[term], V);
  };
  const int dih_variant = p.nat_dih_variant, dih_term = dih_variant ? PCG_SND : PCG_CND;
  // waves past the system's last residue have nothing to do
  for (int base = (int)threadIdx.x - lane; base < n; base += blockDim.x) {
    const int k = base + lane;
    AccSlots<RF> a;
    a.base = r0 + k;
    for (int s = 0; s < 4; ++s) a.c[s][0] = a.c[s][1] = a.c[s][2] = (RF)0;
    if (STAGED && k < n) {
      const int r = r0 + k;
      const uint8_t f = bl.flag(k);
      GeoR q;
      q.base = r;
      for (int j = 0; j < 4; ++j) q.p[j] = g.r(r0 + min(k + j, n - 1));
      if (f & BF_TETHER) ev(PCG_TETHER, tether_core<double>(p, q, a, r, r + 1, bl.teth(k)));
      // local repulsion and chirality have no ill-conditioned step: in R
      if (f & BF_LREP) ev(PCG_LREP, lrep_core<RF>(p, q, a, r, r + 2));
      // the mixed form's FP32 angles on every step but the one that reports
      // energies (want_v, uniform), which takes FP64
      if (sizeof(RF) == 4 && !want_v) {
        if (f & BF_NAT_ANG) ev(PCG_NAT_ANG, nat_ang_mixed(p, q, a, r, r + 1, r + 2, bl.ang(k)));
        if (f & BF_HEUR_ANG) ev(PCG_HEUR_ANG, heur_ang_mixed(p, q, a, r, r + 1, r + 2, bl.at(k)));
      } else {
        if (f & BF_NAT_ANG) ev(PCG_NAT_ANG, nat_ang_core<double>(p, q, a, r, r + 1, r + 2, bl.ang(k)));
        if (f & BF_HEUR_ANG) ev(PCG_HEUR_ANG, heur_ang_core<double>(p, q, a, r, r + 1, r + 2, bl.at(k)));
      }
      if (f & BF_NAT_DIH)
        ev(dih_term, nat_dih_core<double>(p, q, a, r, r + 1, r + 2, r + 3, bl.dih(k), bl.dih(k),
                                          bl.dihs(k), LEAN ? 0 : dih_variant));
      if (f & BF_HEUR_DIH)
        ev(PCG_HEUR_DIH, heur_dih_core<double>(p, q, a, r, r + 1, r + 2, r + 3, bl.dt(k)));
      if (f & BF_CHIR)
        ev(PCG_CHIR, chir_core<RF>(p, q, a, r, r + 1, r + 2, r + 3, bl.c0(k), bl.c1(k)));
    } else if (!STAGED && k < n) {
      int r = r0 + k, it;
      if ((it = b.bond_item[BOND_TETHER][r]) >= 0) ev(PCG_TETHER, tether_item<double>(b, g, a, it));
      if ((it = b.bond_item[BOND_LREP][r]) >= 0) ev(PCG_LREP, lrep_item<double>(b, g, a, it));
      if ((it = b.bond_item[BOND_NAT_ANG][r]) >= 0) ev(PCG_NAT_ANG, nat_ang_item<double>(b, g, a, it));
      if ((it = b.bond_item[BOND_HEUR_ANG][r]) >= 0) ev(PCG_HEUR_ANG, heur_ang_item<double>(b, g, a, it));
      if ((it = b.bond_item[BOND_NAT_DIH][r]) >= 0)
        ev(dih_term, nat_dih_item<double>(b, g, a, it, dih_variant));
      if ((it = b.bond_item[BOND_HEUR_DIH][r]) >= 0) ev(PCG_HEUR_DIH, heur_dih_item<double>(b, g, a, it));
      if ((it = b.bond_item[BOND_CHIR][r]) >= 0) ev(PCG_CHIR, chir_item<double>(b, g, a, it));
    }
    RF t[3];
    for (int c = 0; c < 3; ++c) {
      RF s1 = shfl_up_rf(a.c[1][c], 1), s2 = shfl_up_rf(a.c[2][c], 2), s3 = shfl_up_rf(a.c[3][c], 3);
      t[c] = a.c[0][c];
      if (lane >= 1) t[c] += s1;
      if (lane >= 2) t[c] += s2;
      if (lane >= 3) t[c] += s3;
    }
    if (k < n) {
      atomicAdd(fx + k, (double)t[0]);
      atomicAdd(fy + k, (double)t[1]);
      atomicAdd(fz + k, (double)t[2]);
      // shares for residues handled by the next wave (they exist: an item
      // only reaches residues of its own system)
      for (int s = 1; s < 4; ++s)
        if (lane + s >= 64 && (a.c[s][0] != (RF)0 || a.c[s][1] != (RF)0 || a.c[s][2] != (RF)0)) {
          atomicAdd(fx + k + s, (double)a.c[s][0]);
          atomicAdd(fy + k + s, (double)a.c[s][1]);
          atomicAdd(fz + k + s, (double)a.c[s][2]);
        }
    }
  }
}

// Native contacts, NK items per thread per pass, with every item's list
// fields loaded before any is evaluated (their chains of list load -> LDS
// positions -> decisions overlap). The step takes NK = 1: on the ragged
// 256-protein workload NK = 1, 2, 3, 4 and 6 measured 34.9, 35.1, 35.6,
// 36.6 and 37.7 us a step (the larger NK keep more registers live across
// the loop, in a kernel already limited to 128 VGPRs).
template <int NK, typename R, bool LEAN>
__device__ __forceinline__ void nat_cont_loop(DevBatchC *bp, int s, SysState &st,
                                              const GeoL &g, AccL<double> &acc, TermTurn &turn, double t,
                                              double *vacc, bool want_v) {
  const int n = __builtin_amdgcn_readfirstlane(st.nc_n), B = blockDim.x;
  if (n <= 0) return;
  const DevBatch b = unpack(bp);
  SysDescC &sd = b.sys[s];
  int k = turn.first(n);
  double v = 0.0;
  ParamsC &p = b.P->p;
  if constexpr (sizeof(R) == 4) {
    if (LEAN || p.nc_ss_kind == 0) {
      // the FP32 form of nat_cont_core's plain-LJ case, in stages over the NK
      // items so that the items' loads and arithmetic overlap: the geometry
      // and the FP32-first decisions of every item, straight-line; the exact
      // FP64 decisions of the few inside the margins; the forces of every
      // item, straight-line; then the adds and the state transitions
      const float cut2 = (float)(p.nl_cutoff * p.nl_cutoff), lo = 1.0f - 2e-5f, hi = 1.0f + 2e-5f;
      const float depth = (float)p.nat_cont_depth;
      const int r0 = sd.res0;
      for (; k < n; k += NK * B) {
        // three loads an item: the packed residues, type and state; the
        // native length; the FP32 squared transition distance
        uint32_t ijt[NK];
        double nat[NK];
        float th2[NK];
        for (int j = 0; j < NK; ++j) {
          const int kk = sd.nc0 + min(k + j * B, n - 1);
          ijt[j] = b.ncur_ijt[kk];
          nat[j] = b.ncur_nat[kk];
          th2[j] = b.ncur_th2[kk];
        }
        for (int j = 0; j < NK; ++j) {
          keep(ijt[j]);
          keep(nat[j]);
          keep(th2[j]);
        }
        v3<double> d[NK];
        v3<float> r12[NK];
        float rn[NK];
        int now[NK];
        bool act[NK], exact[NK];
        for (int j = 0; j < NK; ++j) {
          const int i1 = r0 + (int)(ijt[j] & 0xFFFu), i2 = r0 + (int)((ijt[j] >> 12) & 0xFFFu);
          d[j] = xwrapd(xsub(g.r(i2), g.r(i1)), sd);
          r12[j] = cast3<float>(d[j]);
          const float d2 = nsq(r12[j]);
          act[j] = k + j * B < n && !(d2 > cut2 * hi);
          exact[j] = !(d2 < cut2 * lo && (d2 < th2[j] * lo || d2 > th2[j] * hi));
          now[j] = d2 < th2[j] * lo ? 1 : 0;
          rn[j] = sq(d2);
        }
        for (int j = 0; j < NK; ++j)
          if (act[j] && exact[j]) {
            const double rnx = xnorm3(d[j]);
            act[j] = rnx < p.nl_cutoff;
            rn[j] = (float)rnx;
            now[j] = rnx <= __dmul_rn(__dmul_rn(nat[j], C216_INV), p.counting_factor) ? 1 : 0;
          }
        float Vj[NK];
        v3<float> f[NK];
        for (int j = 0; j < NK; ++j) {
          float dV;
          ljR<float>(depth, (float)nat[j], rcpR(rn[j]), Vj[j], dV);
          dV = clampR(dV, -1e3f, 1e3f);
          f[j] = (dV * rcpR(rn[j])) * r12[j];
        }
        for (int j = 0; j < NK; ++j)
          if (act[j]) {
            acc.add(r0 + (int)(ijt[j] & 0xFFFu), f[j]);
            acc.add(r0 + (int)((ijt[j] >> 12) & 0xFFFu), -f[j]);
            if (want_v) v += (double)Vj[j];
            if ((uint32_t)now[j] != (ijt[j] >> 31)) {
              // a transition (rare): the contact's index into the list of all
              const DevBatch bb = unpack(bp);
              const int kk = sd.nc0 + k + j * B, c = bb.ncur[kk];
              bb.nc_active[c] = (uint8_t)now[j];
              bb.ncur_t[kk] = (uint8_t)(((ijt[j] >> 24) & 0x7Fu) | ((uint32_t)now[j] << 7));
              bb.ncur_ijt[kk] = (ijt[j] & 0x7FFFFFFFu) | ((uint32_t)now[j] << 31);
              if (bb.nc_change_t[c] < 0) {
                bb.nc_change_t[c] = t;
                atomicAdd(&st.num_changed, 1);
              }
            }
          }
      }
      if (want_v && v != 0.0) atomicAdd(&vacc[PCG_NAT_CONT], v);
      return;
    }
  }
  for (; k < n; k += NK * B) {
    NcFetch q[NK];
    for (int j = 0; j < NK; ++j)
      if (k + j * B < n) q[j] = nat_cont_fetch(b, sd.nc0 + k + j * B);
    for (int j = 0; j < NK; ++j)
      if (k + j * B < n) keep_fetch(q[j]);
    for (int j = 0; j < NK; ++j)
      if (k + j * B < n) v += nat_cont_core<R>(b, sd, st, g, acc, q[j], t, true);
  }
  if (want_v && v != 0.0) atomicAdd(&vacc[PCG_NAT_CONT], v);
}

// QA near pairs without workgroup barriers. Thread t of the workgroup takes
// near pairs t, t + B, ...; every pair takes the cheap FP32 first test, and
// the ones that pass (about one near pair in seven) are stacked in the
// wave's own 128-entry LDS segment. Whenever 64 are stacked, the wave takes
// the newest 64 through the exact path, one a lane, so that path runs on
// full waves; the last few go after the loop. The next pair is fetched
// before the stack is drained, so its load overlaps the exact path. No wave
// waits for another: the force terms before and after this one flow on. The
// exact path reads nothing from HBM but n and h (a pair's formation
// distance bound comes from the LDS tables, its free-pair slot is loaded
// only if it becomes a candidate), and the order in which candidates are
// found does not matter: qa::finish ranks them by (distance, free-pair
// index).
template <typename R>
__device__ __forceinline__ void qa_cand_waves(DevBatchC *bp, int s, SysState &st,
                                              const GeoL &g, AccL<double> &acc,
                                              uint2 *queue, double *vacc, bool want_v) {
  constexpr int WCAP = 128;  // stacked pairs per wave: fewer than 64 + 64
  static_assert(16 * WCAP * sizeof(uint2) <= LdsLayout::QA_QUEUE * sizeof(int),
                "the QA queue holds every wave's stack");
  const int n = __builtin_amdgcn_readfirstlane(st.qh_n), B = blockDim.x;
  if (n <= 0) return;
  const DevBatch b = unpack(bp);
  SysDescC &sd = b.sys[s];
  const int tid = threadIdx.x, lane = tid & 63, r0 = sd.res0;
  const unsigned long long below = (1ull << lane) - 1ull;
  uint2 *wq = queue + (tid >> 6) * WCAP;
  auto fetch = [&](int hk) { return hk < n ? qa_cand_fetch_lite(b, sd, hk) : QhLite{0u, -1.0f}; };
  // the exact path's q: every field but the free-pair slot
  auto full = [&](int hk, int i1, int i2) {
    const int a1 = g.atype(b, i1), a2 = g.atype(b, i2);
    double req = fmax(fmax(fmax(g.req_t[1], g.req_t[2]), g.req_t[3]), g.req_t[4 + a1 + 21 * a2]);
    return QhFetch{hk, i1, i2, 0.f, 0, req, -1};
  };
  const int iters = (n + B - 1) / B;  // the same for every thread
  int pend = 0;                       // stacked pairs of this wave (uniform)
  double v = 0.0;
  QhLite cur = fetch(tid);
  for (int t = 0; t <= iters; ++t) {
    if (t < iters) {
      bool act = false;
      if (cur.thr2 >= 0.0f) {  // a vacant pair has thr2 < 0
        const v3<double> d = xwrapd(xsub(g.r(r0 + (int)(cur.ij >> 16)), g.r(r0 + (int)(cur.ij & 0xFFFFu))), sd);
        const float dx = (float)d.x, dy = (float)d.y, dz = (float)d.z;
        act = !(dx * dx + dy * dy + dz * dz > cur.thr2);
      }
      const unsigned long long m = __ballot(act);
      if (act) wq[pend + __popcll(m & below)] = make_uint2((unsigned)(tid + t * B), cur.ij);
      pend += __popcll(m);
      cur = fetch(tid + (t + 1) * B);
    }
    if (pend >= 64 || (t == iters && pend > 0)) {
      const int take = pend < 64 ? pend : 64;
      pend -= take;
      // the lanes' stack writes before the reads of other lanes' entries
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      if (lane < take) {
        const uint2 w = wq[pend + lane];
        v += qa_cand_exact<R>(b, sd, st, g, acc,
                              full((int)w.x, r0 + (int)(w.y & 0xFFFFu), r0 + (int)(w.y >> 16)));
      }
      // and those reads before the slots take new pairs
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
  if (want_v && v != 0.0) atomicAdd(&vacc[PCG_QA_CAND], v);
}

// The items of one term, one a thread and pass, starting at the wave the
// terms before it left off at.
template <int T, typename R>
__device__ __forceinline__ void term_loop(DevBatchC *bp, int s, uint32_t on, SysState &st,
                                          const GeoL &g, AccL<double> &acc, TermTurn &turn, double t,
                                          double *vacc, bool want_v) {
  if (!(on & (1u << T))) return;
  const DevBatch b = unpack(bp);
  SysDescC &sd = b.sys[s];
  const int n = __builtin_amdgcn_readfirstlane(term_size(sd, st, T)), B = blockDim.x;
  if (n <= 0) return;
  int k = turn.first(n);
  double v = 0.0;
  for (; k < n; k += B) v += eval_item<R>(b, sd, st, g, acc, T, k, t, want_v);
  if (want_v && v != 0.0) atomicAdd(&vacc[T], v);
}

// nl::verify's test (cg/src/cg/nl/verify.cpp:3-34) for the displacement
// maximum maxd since the last rebuild.
__device__ __forceinline__ bool nl_moved(DevBatchC *bp, int s, const SysState &st, double maxd) {
#pragma clang fp contract(off)
  const DevBatch b = unpack(bp);
  SysDescC &sd = b.sys[s];
  const double box = fabs(sd.cell[0] - st.orig_cell[0]) + fabs(sd.cell[1] - st.orig_cell[1]) +
                     fabs(sd.cell[2] - st.orig_cell[2]);
  return __dadd_rn(__dmul_rn(2.0, maxd), box) > st.orig_pad;
}

// LEAN: the common force field, without what the host has ruled out for every
// system of the launch (lean_batch in pcg_host.hip): bonded items outside LDS
// or not chain-local, the simple native dihedral, disulfide contacts, PID
// pairs, the relative Debye-Hueckel term and walls. A step is a chain of
// short dependent phases, bound by latency and instruction issue, and the
// general form's unused code is half of the kernel: 23 600 instructions
// against 12 400, 204 spilled VGPRs against 65 on 1024 threads. With LEAN,
// unpack() and the step's decisions taken by every thread, a step of one
// 56-residue Go chain takes 5.5 us instead of 9.4, of a 301-residue protein
// in the full force field 17.3 us instead of 22.0.
template <typename R, typename RF, bool LEAN>
__device__ __forceinline__ void persistent_body(DevBatchC *bp, int s, int nsteps,
                                                JobSlot *slot = nullptr) {
#pragma clang fp contract(off)
  __shared__ SysState st;
  __shared__ double minv_t[21], sqminv_t[21], req_t[445];
  __shared__ int8_t ptype_t[21];
  __shared__ double vacc[NT];
  __shared__ double wave_max[16];
  extern __shared__ __align__(16) unsigned char lds[];
  int n, r0, nftip;
  int64_t target;
  bool staged, regular, gear_l, energy_off, nl_required, lang_on;
  uint32_t on = 0u;   // the enabled terms
  uint32_t chg = 0u;  // the residue types with a charge (q1 q2 != 0 iff both are set)
  {
    const DevBatch b = unpack(bp);
    SysDescC &sd = b.sys[s];
    if (!b.st[s].active) return;
    DevParamsC &P = *b.P;
    n = sd.n;
    r0 = sd.res0;
    nftip = sd.nftip;
    target = slot ? slot->target : sd.steps_target;
    regular = LEAN || sd.bond_regular;
    staged = LEAN || (sd.bond_regular && b.bond_lds);
    gear_l = b.gear_lds != 0;
    energy_off = b.energy_off != 0;
    nl_required = P.nl_required != 0;
    lang_on = P.p.lang_on != 0;
    for (int t = 0; t < NT; ++t) on |= (term_on(P, t) ? 1u : 0u) << t;
    for (int t = 0; t < 21; ++t) chg |= (P.p.charge[t] != 0.0 ? 1u : 0u) << t;
  }
  const bool qa_on = on & (1u << PCG_QA_CAND);
  // forces accumulate in FP64 in LDS: on gfx950 an LDS FP64 atomic add
  // (ds_add_f64) runs at integer-atomic speed, an FP32 one far slower
  const LdsLayout lay((size_t)n, sizeof(double), staged, gear_l);
  double *rx = (double *)lds, *ry = rx + n, *rz = ry + n;
  double *fx = (double *)(lds + lay.f), *fy = fx + n, *fz = fy + n;
  BondLds bl{(double *)(lds + lay.bd), (uint8_t *)(lds + lay.bu), n};
  uint8_t *atl = (uint8_t *)(lds + lay.at);      // residue types and chain flags
  uint32_t *syl = (uint32_t *)(lds + lay.sy);     // QA sync budgets
  uint2 *qa_queue = (uint2 *)(lds + lay.q);
  double *ys = (double *)(lds + lay.g);  // [15][n]: y1..y5 x, y, z (gear_l)
  GeoL g{rx, ry, rz, r0, atl, syl, ptype_t, req_t};
  AccL<double> acc{fx, fy, fz, r0};
  {
    const DevBatch b = unpack(bp);
    DevParamsC &P = *b.P;
    // the system's scalars live in LDS for the launch (only this workgroup
    // touches them) and go back to HBM at its end
    if (threadIdx.x == 0) st = b.st[s];
    // 1 / mass and its square root per residue type, for the Langevin step;
    // the QA polarity classes and per-type formation distances
    if (threadIdx.x < 21) {
      minv_t[threadIdx.x] = 1.0 / P.p.mass[threadIdx.x];
      sqminv_t[threadIdx.x] = sqrt(minv_t[threadIdx.x]);
      ptype_t[threadIdx.x] = (int8_t)P.p.ptype[threadIdx.x];
    }
    for (int t = threadIdx.x; t < 445; t += blockDim.x)
      req_t[t] = __dmul_rn(P.p.qa_lj_r_high[t], __dadd_rn(1.0, P.p.qa_formation_tol));
    if (threadIdx.x < NT) vacc[threadIdx.x] = 0.0;
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
      rx[k] = b.y[0][0][r0 + k];
      ry[k] = b.y[0][1][r0 + k];
      rz[k] = b.y[0][2][r0 + k];
      // chain neighbours are always the adjacent residues (i - 1, i + 1)
      atl[k] = (uint8_t)(b.atype[r0 + k] | (b.prev[r0 + k] >= 0 ? 0x40 : 0) |
                         (b.next[r0 + k] >= 0 ? 0x80 : 0));
      syl[k] = *(const uint32_t *)(b.sync + 4 * (r0 + k));
      // forces start at zero; afterwards each step's Langevin pass clears them
      fx[k] = 0;
      fy[k] = 0;
      fz[k] = 0;
    }
    if (staged) stage_bonded(b, b.sys[s], bl);
    if (gear_l)
      for (int k = threadIdx.x; k < n; k += blockDim.x)
        for (int j = 0; j < 15; ++j) ys[j * n + k] = b.y[1 + j / 3][j % 3][r0 + k];
  }
  __syncthreads();

  // Each thread keeps the step counter, the time and the displacement
  // maximum and takes the step's decisions from them itself. With one thread
  // doing that for the workgroup, the others waited 3900 cycles a step for
  // it, a sixth of a 56-residue system's step.
  int64_t step = st.step;
  double t = st.t, true_t = st.true_t, dt;
  {
    const DevBatch b = unpack(bp);
    dt = b.P->dt;
  }
  bool ran = false, with_v = false;
  double maxd = __longlong_as_double((long long)st.max_disp_bits);
  bool first = st.verify_first != 0, invalid = st.nl_invalid != 0;
  for (int it = 0; it < nsteps; ++it) {
    // a finished system keeps the forces of its last evaluation
    if (step >= target) break;
    // the last step this launch makes for the system: energies (unless
    // off) and the write-back of its forces
    const bool last = (it == nsteps - 1) || (step + 1 >= target);
    const bool wv = !energy_off && last;
    // nl::verify (cg/src/cg/nl/verify.cpp:3-34)
    if (nl_required) invalid = first || nl_moved(bp, s, st, maxd);
    first = first && !nl_required;
    if (invalid) {
      wg_fix_nl(bp, s, st, g, (void *)(lds + lay.q), fx,
                (float4 *)(lds + ((lay.f + 15) & ~(size_t)15)), chg);
      invalid = false;
    }
    TermTurn turn{0, (int)(blockDim.x >> 6)};
    // every term's items, a thread moving on to the next term without
    // waiting; one loop per term so each keeps only its own constants in
    // registers
    if (staged) {
      bonded_by_base<RF, true, LEAN>(bp, s, st, g, bl, fx, fy, fz, vacc, wv);
      turn.skip(n);
    } else if (regular) {
      bonded_by_base<RF, false, LEAN>(bp, s, st, g, bl, fx, fy, fz, vacc, wv);
      turn.skip(n);
    } else {
      term_loop<PCG_CHIR, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
      term_loop<PCG_TETHER, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
      term_loop<PCG_LREP, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
      term_loop<PCG_NAT_ANG, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
      term_loop<PCG_HEUR_ANG, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
      term_loop<PCG_HEUR_DIH, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
      term_loop<PCG_CND, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
      term_loop<PCG_SND, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
    }
    // n and h of this step's positions, which the barrier before the QA pairs
    // makes visible
    if (qa_on) wg_prepare_nh(bp, g, n, r0, turn);
    if (on & (1u << PCG_NAT_CONT)) nat_cont_loop<1, R, LEAN>(bp, s, st, g, acc, turn, t, vacc, wv);
    term_loop<PCG_PAULI, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
    term_loop<PCG_CONST_DH, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
    if (!LEAN) {
      term_loop<PCG_REL_DH, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
      term_loop<PCG_PID, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
      term_loop<PCG_SOLID_WALL, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
    }
    term_loop<PCG_VEL_AFM, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
    term_loop<PCG_FORCE_AFM, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
    if (qa_on) {
      __syncthreads();  // n and h
      qa_cand_waves<R>(bp, s, st, g, acc, qa_queue, vacc, wv);
      term_loop<PCG_QA_CONT, R>(bp, s, on, st, g, acc, turn, t, vacc, wv);
    }
    __syncthreads();
    if (qa_on && (st.cand_n != 0 || st.rem_n != 0)) {
      const DevBatch b = unpack(bp);
      qa_finish_block(b, b.sys[s], st, (int8_t *)syl, r0);
    }
    // lang::step (cg/src/cg/langevin/step.cpp:23-77); each residue's force,
    // once used, goes to HBM on the launch's last step and restarts at 0
    double md = 0.0;
    {
      const DevBatch b = unpack(bp);
      SysDescC &sd = b.sys[s];
      auto flush_force = [&](int k) {
        if (last) {
          ((RF *)b.F[0])[r0 + k] = (RF)fx[k];
          ((RF *)b.F[1])[r0 + k] = (RF)fy[k];
          ((RF *)b.F[2])[r0 + k] = (RF)fz[k];
        }
        fx[k] = 0;
        fy[k] = 0;
        fz[k] = 0;
      };
      if (lang_on) {
        for (int k = threadIdx.x; k < n; k += blockDim.x) {
          int i = r0 + k;
          // the rebuild snapshot is loaded first: its latency hides behind
          // the noise and the corrector
          const double o[3] = {b.orig_r[0][i], b.orig_r[1][i], b.orig_r[2][i]};
          double nz[3];
          philox_normals(sd.philox_key, step, k, nz);
          double r[3], vel[3];
          const int aa = atl[k] & 63;  // the type, without the chain flags
          const double Fx = fx[k], Fy = fy[k], Fz = fz[k];
          flush_force(k);
          if (gear_l) {
            gear_core(b, sd, t == 0.0, minv_t[aa], sqminv_t[aa], Fx, Fy, Fz, nz, r, vel,
                      [&](int kk, int c) -> double & {
                        return kk == 0 ? (c == 0 ? rx[k] : c == 1 ? ry[k] : rz[k])
                                       : ys[((kk - 1) * 3 + c) * n + k];
                      });
            // a force tip averages its residue's velocity in the next
            // evaluation, which reads it from HBM
            if (nftip > 0)
              for (int c = 0; c < 3; ++c) b.vel[c][i] = vel[c];
          } else {
            gear_core(b, sd, t == 0.0, minv_t[aa], sqminv_t[aa], Fx, Fy, Fz, nz, r, vel,
                      [&](int kk, int c) -> double & { return b.y[kk][c][i]; });
            for (int c = 0; c < 3; ++c) b.vel[c][i] = vel[c];
          }
          rx[k] = r[0];
          ry[k] = r[1];
          rz[k] = r[2];
          md = fmax(md, disp2_from(sd, o, r));  // squared; the root is taken once below
        }
      } else {
        for (int k = threadIdx.x; k < n; k += blockDim.x) flush_force(k);
      }
    }
    // every position has moved past this barrier
    maxd = __dsqrt_rn(block_max(md, wave_max));
    if (lang_on) {
      ++step;
      true_t += dt;
      t = true_t;
    }
    ran = true;
    with_v = wv;
  }
  // scalars and the forces of the last evaluation back to HBM
  __syncthreads();
  const DevBatch b = unpack(bp);
  if (threadIdx.x == 0) {
    st.step = step;
    st.t = t;
    st.true_t = true_t;
    if (ran) {
      st.max_disp_bits = (unsigned long long)__double_as_longlong(maxd);
      if (nl_required && step < target) st.nl_invalid = nl_moved(bp, s, st, maxd);
    }
    if (with_v) {
      double v = 0.0;
      for (int k = 0; k < NT; ++k) {
        st.V[k] = vacc[k];
        v += vacc[k];
      }
      st.Vtot = v;
    }
    b.st[s] = st;
    if (b.ovf && st.overflow) *b.ovf = 1;
    if (slot) {
      slot->step = st.step;
      slot->Vtot = st.Vtot;
      slot->overflow = st.overflow;
    }
  }
  if (gear_l)
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
      b.y[0][0][r0 + k] = rx[k];
      b.y[0][1][r0 + k] = ry[k];
      b.y[0][2][r0 + k] = rz[k];
      for (int j = 0; j < 15; ++j) b.y[1 + j / 3][j % 3][r0 + k] = ys[j * n + k];
      for (int c = 0; c < 3; ++c) b.vel[c][r0 + k] = ys[c * n + k] * b.P->dt_inv;
    }
  if (qa_on)
    for (int k = threadIdx.x; k < n; k += blockDim.x) *(uint32_t *)(b.sync + 4 * (r0 + k)) = syl[k];
}

// Persistent kernels over every system of a batch, and over the resident jobs
// of the served form (one-system batches).
//
// The launch bound sets the register budget: 1024 threads leave 128 VGPRs
// per lane, 768 leave 168, 512 leave 256.
template <typename R, typename RF, int MAXT, bool LEAN>
__global__ __launch_bounds__(MAXT) void k_persistent(DevBatch b, int nsteps) {
  // the descriptor is the first kernel argument
  persistent_body<R, RF, LEAN>((DevBatchC *)__builtin_amdgcn_kernarg_segment_ptr(), blockIdx.x,
                               nsteps);
}

template <typename R, typename RF, int MAXT, bool LEAN>
__global__ __launch_bounds__(MAXT) void k_persistent_jobs(const DevBatch *jobs, JobSlot *slots,
                                                          int nsteps) {
  persistent_body<R, RF, LEAN>((DevBatchC *)(jobs + blockIdx.x), 0, nsteps, slots + blockIdx.x);
}

template <bool LEAN, int MAXT>
void launch_jobs_t(const DevBatch *jobs, JobSlot *slots, int njobs, int prec, int block, int nsteps,
                   size_t lds_bytes, hipStream_t s) {
  if (prec == PCG_FP64)
    hipLaunchKernelGGL((k_persistent_jobs<double, double, MAXT, LEAN>), dim3(njobs), dim3(block),
                       lds_bytes, s, jobs, slots, nsteps);
  else
    hipLaunchKernelGGL((k_persistent_jobs<float, float, MAXT, LEAN>), dim3(njobs), dim3(block),
                       lds_bytes, s, jobs, slots, nsteps);
}

template <bool LEAN, int MAXT>
void launch_batch_t(const DevBatch &b, int prec, int block, int nsteps, size_t lds_bytes,
                    hipStream_t s) {
  if (prec == PCG_FP64)
    hipLaunchKernelGGL((k_persistent<double, double, MAXT, LEAN>), dim3(b.nsys), dim3(block),
                       lds_bytes, s, b, nsteps);
  else
    hipLaunchKernelGGL((k_persistent<float, float, MAXT, LEAN>), dim3(b.nsys), dim3(block),
                       lds_bytes, s, b, nsteps);
}

template <bool LEAN>
void launch_jobs_b(const DevBatch *jobs, JobSlot *slots, int njobs, int prec, int block, int nsteps,
                   size_t lds_bytes, hipStream_t s) {
  if (block > 768) launch_jobs_t<LEAN, 1024>(jobs, slots, njobs, prec, block, nsteps, lds_bytes, s);
  else if (block > 512) launch_jobs_t<LEAN, 768>(jobs, slots, njobs, prec, block, nsteps, lds_bytes, s);
  else launch_jobs_t<LEAN, 512>(jobs, slots, njobs, prec, block, nsteps, lds_bytes, s);
}

template <bool LEAN>
void launch_batch_b(const DevBatch &b, int prec, int block, int nsteps, size_t lds_bytes,
                    hipStream_t s) {
  if (block > 768) launch_batch_t<LEAN, 1024>(b, prec, block, nsteps, lds_bytes, s);
  else if (block > 512) launch_batch_t<LEAN, 768>(b, prec, block, nsteps, lds_bytes, s);
  else launch_batch_t<LEAN, 512>(b, prec, block, nsteps, lds_bytes, s);
}

} // namespace pcg
