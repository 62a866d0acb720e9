// Readout reductions: norm / branch probability, collapse, Pauli
// expectation, marginals and shot sampling.  All accumulation is FP64
// (also for complex64 states, as crates/aleph-cuda/src/sv/readout_f32.cu:1-8
// requires).  Norms, branch probabilities and the sampler's block sums are
// Neumaier-compensated per thread and combined with error-free two-sums across
// lanes and workgroups.  Marginals, the sampler's prefix over the blocks and
// Pauli sums add plainly (a relative rounding of 1e-16 per addition, at most a
// few hundred in sequence): they decide nothing about the state's validity
// near the edge of its budget, where the compensated norm is taken.
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace aleph {
namespace {

constexpr uint32_t kThreads = 256;

struct KSum {
  double s, c;
};

__device__ __forceinline__ void kadd(KSum& k, double x) {
  const double t = k.s + x;
  if (fabs(k.s) >= fabs(x)) k.c += (k.s - t) + x;
  else k.c += (x - t) + k.s;
  k.s = t;
}

__device__ __forceinline__ KSum kmerge(KSum a, KSum b) {
  KSum r = a;
  kadd(r, b.s);
  r.c += b.c;
  return r;
}

__device__ __forceinline__ KSum wave_reduce(KSum v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    KSum o;
    o.s = __shfl_down(v.s, off, 64);
    o.c = __shfl_down(v.c, off, 64);
    v = kmerge(v, o);
  }
  return v;
}

// Block-wide reduction of up to 3 compensated sums; result valid in thread 0.
template <int N>
__device__ void block_reduce(KSum (&v)[N]) {
  __shared__ KSum sh[N][kThreads / 64];
  const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < N; i++) v[i] = wave_reduce(v[i]);
  if (lane == 0)
#pragma unroll
    for (int i = 0; i < N; i++) sh[i][wid] = v[i];
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int i = 0; i < N; i++) {
      KSum acc = sh[i][0];
      for (uint32_t w = 1; w < blockDim.x / 64; w++) acc = kmerge(acc, sh[i][w]);
      v[i] = acc;
    }
  }
}

// Compensated column sums of `rows` rows of three partials into total[0..3)
// (LDS), one wavefront per column.
__device__ __forceinline__ void sum_rows(const double* partials, uint32_t rows, double* total) {
  const uint32_t lane = threadIdx.x & 63u, col = threadIdx.x >> 6;
  if (col < 3) {
    KSum v = {0, 0};
#pragma unroll 4
    for (uint32_t b = lane; b < rows; b += 64) kadd(v, partials[3 * (uint64_t)b + col]);
    v = wave_reduce(v);
    if (lane == 0) total[col] = v.s + v.c;
  }
  __syncthreads();
}

// A workgroup's three sums (valid in thread 0) into its row.  A second launch
// adds the rows: with the last workgroup of the same launch doing it, the
// device-wide fence of every workgroup cost more (19 qubits: 18 us against
// 6.6 + 5.7).
__device__ __forceinline__ void store_row(const KSum (&v)[3], double* partials) {
  if (threadIdx.x == 0)
    for (int w = 0; w < 3; w++) partials[3 * (uint64_t)blockIdx.x + w] = v[w].s + v[w].c;
}

// Sweeps take kUnroll amplitudes per thread per iteration, all loads issued
// before any arithmetic, so each wave keeps several 16-byte loads in flight.
constexpr int kUnroll = 4;
constexpr int kMarginalUnroll = 8;
// Workgroups of a reduction: four per CU, a tile of kUnroll * kThreads
// consecutive amplitudes at a time, so that a row of partials sums many reads
// (the second launch then takes 7 us at 27 qubits where 4096 rows took 16).
// Twice as many for FP32, whose loads are half as long: the norm at 27 qubits
// takes 309 us with 1024, 217 with 2048 and 223 with 4096 (FP64 374, 384, 382).
constexpr uint32_t kReduceGrid = 1024;

// MODE 0: [sum over bit q clear, sum over bit q set, non-finite count] of p = |a|^2.
// MODE 1: [sum of p^2, sum of p, non-finite count] (collision probability).
template <typename T, int MODE>
__global__ void __launch_bounds__(kThreads) k_reduce_branch(const C2<T>* __restrict__ s, uint64_t len, uint64_t qmask,
                                                            double* __restrict__ partials) {
  KSum v[3] = {{0, 0}, {0, 0}, {0, 0}};
  const uint64_t tile = kUnroll * kThreads;
  for (uint64_t i0 = (uint64_t)blockIdx.x * tile + threadIdx.x; i0 < len; i0 += gridDim.x * tile) {
    C2<T> a[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
      const uint64_t i = i0 + u * kThreads;
      if (i < len) a[u] = s[i];
      else a[u].x = a[u].y = 0;
    }
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
      const uint64_t i = i0 + u * kThreads;
      const double p = (double)a[u].x * (double)a[u].x + (double)a[u].y * (double)a[u].y;
      if (!isfinite(p)) {
        v[2].s += 1.0;
        continue;
      }
      if (MODE == 0) {
        if (i & qmask) kadd(v[1], p);
        else kadd(v[0], p);
      } else {
        kadd(v[0], p * p);
        kadd(v[1], p);
      }
    }
  }
  block_reduce<3>(v);
  store_row(v, partials);
}

// Sums `count` rows of three partials into out[0..3) (device or pinned memory).
__global__ void __launch_bounds__(kThreads) k_reduce_final(const double* __restrict__ partials, uint32_t count,
                                                           double* out) {
  __shared__ double total[3];
  sum_rows(partials, count, total);
  if (threadIdx.x < 3) out[threadIdx.x] = total[threadIdx.x];
}

// Zero the amplitudes with bit q != outcome and scale the others, a pair
// {q clear, q set} at a time: the zeroed half is only written.
template <typename T>
__device__ __forceinline__ void collapse_pairs(C2<T>* s, uint64_t pairs, uint32_t q, bool outcome, double scale,
                                               uint64_t first, uint64_t stride) {
  for (uint64_t p = first; p < pairs; p += stride) {
    const uint64_t i0 = insert_zero(p, q), i1 = i0 | (1ull << q);
    const uint64_t keep = outcome ? i1 : i0, drop = outcome ? i0 : i1;
    C2<T> a = s[keep], zero;
    a.x = (T)((double)a.x * scale);
    a.y = (T)((double)a.y * scale);
    zero.x = zero.y = 0;
    s[keep] = a;
    s[drop] = zero;
  }
}

// A measurement without a round trip to the host: every workgroup adds the
// rows of the preceding reduction (at most 2 * kReduceGrid, a few microseconds)
// and comes to the same decision the host reads from host[0..3); an invalid
// state or a degenerate branch is left alone.  The reduction's second launch,
// the copy back, a synchronisation and the reads of the zeroed half go (19
// qubits, two rounds of 9 parity measurements with their 56 gates: 1.24 ->
// 0.99 ms).
template <typename T>
__global__ void __launch_bounds__(kThreads) k_measure(C2<T>* __restrict__ s, uint64_t pairs, uint32_t q,
                                                      const double* __restrict__ partials, uint32_t rows, double u,
                                                      double tol, double* host) {
  __shared__ double total[3];
  sum_rows(partials, rows, total);
  if (blockIdx.x == 0 && threadIdx.x < 3) host[threadIdx.x] = total[threadIdx.x];
  const MeasureChoice c = measure_choice(total[0], total[1], total[2], u, tol);
  if (!c.apply) return;
  collapse_pairs(s, pairs, q, c.outcome, c.scale, (uint64_t)blockIdx.x * blockDim.x + threadIdx.x,
                 (uint64_t)gridDim.x * blockDim.x);
}

// The same for large states in three launches: one workgroup adds the rows and
// decides, and a collapse with a grid of an amplitude a thread reads the
// decision.  FP64 27 qubits 1039 -> 923 us, 28 qubits 2101 -> 1817 (FP32 622
// -> 508, 1245 -> 946); 24 qubits 113 either way, below the launch counts.
struct MeasureDecision {
  double scale;
  uint32_t apply, outcome;
};

__global__ void __launch_bounds__(kThreads) k_measure_decide(const double* __restrict__ partials, uint32_t rows,
                                                             double u, double tol, MeasureDecision* decision,
                                                             double* host) {
  __shared__ double total[3];
  sum_rows(partials, rows, total);
  if (threadIdx.x < 3) host[threadIdx.x] = total[threadIdx.x];
  if (threadIdx.x == 0) {
    const MeasureChoice c = measure_choice(total[0], total[1], total[2], u, tol);
    *decision = MeasureDecision{c.scale, c.apply ? 1u : 0u, c.outcome ? 1u : 0u};
  }
}

template <typename T>
__global__ void __launch_bounds__(kThreads) k_collapse(C2<T>* __restrict__ s, uint64_t len, uint64_t qmask,
                                                       const MeasureDecision* __restrict__ decision) {
  const MeasureDecision d = *decision;
  if (!d.apply) return;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < len; i += (uint64_t)gridDim.x * blockDim.x) {
    C2<T> a;
    a.x = a.y = 0;
    if (((i & qmask) != 0) == (d.outcome != 0)) {
      a = s[i];
      a.x = (T)((double)a.x * d.scale);
      a.y = (T)((double)a.y * d.scale);
    }
    s[i] = a;
  }
}

// The same for a state of one workgroup's size, in one launch.
template <typename T>
__global__ void __launch_bounds__(kThreads) k_measure_small(C2<T>* __restrict__ s, uint64_t len, uint32_t q, double u,
                                                            double tol, double* host) {
  __shared__ double total[3];
  KSum v[3] = {{0, 0}, {0, 0}, {0, 0}};
  for (uint64_t i = threadIdx.x; i < len; i += blockDim.x) {
    const C2<T> a = s[i];
    const double p = (double)a.x * (double)a.x + (double)a.y * (double)a.y;
    if (!isfinite(p)) v[2].s += 1.0;
    else if ((i >> q) & 1ull) kadd(v[1], p);
    else kadd(v[0], p);
  }
  block_reduce<3>(v);
  if (threadIdx.x == 0)
    for (int w = 0; w < 3; w++) host[w] = total[w] = v[w].s + v[w].c;
  __syncthreads();
  const MeasureChoice c = measure_choice(total[0], total[1], total[2], u, tol);
  if (c.apply) collapse_pairs(s, len / 2, q, c.outcome, c.scale, threadIdx.x, blockDim.x);
}

// All Pauli terms that share one X mask `x` in one read of the state.
// With z = conj(psi[i ^ x]) psi[i] and s_t(i) = (-1)^{|i & zy_t|}, term t
// needs R_t = sum_i s_t(i) Re z(i) and I_t = sum_i s_t(i) Im z(i).  For
// x != 0 the sum runs over pairs {i, j = i ^ x} (i with x's top bit clear),
// each amplitude read once: z(j) = conj z(i) and s_t(j) = c_t s_t(i) with
// c_t = (-1)^{|x & zy_t|}, so the pair adds 2 s_t(i) Re z(i) to R_t when
// c_t = 1 (I_t gets 0) and 2 s_t(i) Im z(i) to I_t when c_t = -1 (R_t
// gets 0).  Hence one accumulator per term: acc_t = sum s_t(i) w_t(i) with
// w_t = Re z or Im z; the factor 2 and the placement are applied on the host.
// For x = 0, w = |psi_i|^2 over every i.
constexpr int kGroupTerms = (int)kExpectGroup;
struct GroupTerms {
  uint64_t zy[kGroupTerms];
  uint32_t use_im;   // bit t: term t accumulates Im z
  uint32_t count;
};

template <typename T>
__global__ void __launch_bounds__(kThreads) k_expect_group(const C2<T>* __restrict__ s, uint64_t pairs, uint64_t x,
                                                           uint32_t hbit, GroupTerms g,
                                                           double* __restrict__ partials) {
  double acc[kGroupTerms];
#pragma unroll
  for (int t = 0; t < kGroupTerms; t++) acc[t] = 0.0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t lo_mask = (1ull << hbit) - 1ull;
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < pairs; k += stride) {
    // k enumerates indices with bit hbit clear (every index when x == 0).
    const uint64_t i = x ? (((k & ~lo_mask) << 1) | (k & lo_mask)) : k;
    const C2<T> a = s[i];
    double re, im;
    if (x) {
      const C2<T> b = s[i ^ x];
      re = (double)b.x * (double)a.x + (double)b.y * (double)a.y;
      im = (double)b.x * (double)a.y - (double)b.y * (double)a.x;
    } else {
      re = (double)a.x * (double)a.x + (double)a.y * (double)a.y;
      im = 0.0;
    }
#pragma unroll
    for (int t = 0; t < kGroupTerms; t++) {
      if (t < (int)g.count) {
        const double w = ((g.use_im >> t) & 1u) ? im : re;
        acc[t] += (__popcll(i & g.zy[t]) & 1) ? -w : w;
      }
    }
  }
  // Block reduction per term: wave shuffles, then the block's waves in LDS.
  __shared__ double sh[kGroupTerms][kThreads / 64];
  const uint32_t lane = threadIdx.x & 63u, wid = threadIdx.x >> 6;
#pragma unroll
  for (int t = 0; t < kGroupTerms; t++) {
    double v = acc[t];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
    if (lane == 0) sh[t][wid] = v;
  }
  __syncthreads();
  if (threadIdx.x < (uint32_t)g.count) {
    double v = 0.0;
    for (uint32_t w = 0; w < blockDim.x / 64; w++) v += sh[threadIdx.x][w];
    partials[(uint64_t)blockIdx.x * kGroupTerms + threadIdx.x] = v;
  }
}

// Sums `count` rows of `width` partials column-wise into out[0..width)
// (compensated), one workgroup.
__global__ void __launch_bounds__(kThreads) k_reduce_columns(const double* __restrict__ partials, uint32_t count,
                                                             uint32_t width, double* __restrict__ out) {
  __shared__ double sh[kThreads];
  for (uint32_t w = 0; w < width; w++) {
    KSum v = {0, 0};
    for (uint32_t b = threadIdx.x; b < count; b += blockDim.x) kadd(v, partials[(uint64_t)width * b + w]);
    v = wave_reduce(v);
    if ((threadIdx.x & 63u) == 0) sh[threadIdx.x >> 6] = v.s + v.c;
    __syncthreads();
    if (threadIdx.x == 0) {
      KSum acc = {0, 0};
      for (uint32_t i = 0; i < blockDim.x / 64; i++) kadd(acc, sh[i]);
      out[w] = acc.s + acc.c;
    }
    __syncthreads();
  }
}

// Marginal histogram.  The index bits are split so that a thread's loop runs
// over bits outside the marginal only: its bin is fixed, the sum stays in a
// register, and one atomic per thread (into the workgroup's LDS bins, then
// one per workgroup and bin) replaces one per amplitude.  Thread bits are the
// low 8 (coalesced); loop bits the lowest bits above them that the marginal
// does not ask for, as many as leave kMarginalGroups workgroups; the rest
// number the workgroups.  The norm of the validity check is the sum of the
// same reads.  27 qubits FP64, 9 of them random: 678 us and a separate check
// of 428 us -> 352 us (6.1 TB/s, what a plain read reaches; 424 us with four
// loads in flight instead of eight).
constexpr uint32_t kMarginalGroups = 2048;
// Marginal qubits above the thread bits: with more, workgroups would outnumber
// the rows of the reduction, and bins the atomics saved (k_marginal_wide).
constexpr uint32_t kMarginalHigh = 12;
static_assert((1u << kMarginalHigh) <= kReduceBlocks, "one row per workgroup");

struct MarginalBits {
  uint64_t loop_mask;          // index bits of a thread's loop
  uint32_t n_group;            // workgroup bits
  uint32_t group_pos[40];      // their index bits
  uint32_t n_low;              // marginal bits among the thread bits
  uint32_t low_pos[8], low_bin[8];    // their index bits and bin bits
  uint32_t n_high;             // marginal bits among the workgroup bits
  uint32_t high_pos[32], high_bin[32];
};

template <typename T>
__global__ void __launch_bounds__(kThreads) k_marginal(const C2<T>* __restrict__ s, uint64_t len, MarginalBits d,
                                                       double* __restrict__ bins, double* __restrict__ partials) {
  __shared__ double h[kThreads];
  const uint32_t tid = threadIdx.x;
  h[tid] = 0.0;
  uint64_t base = tid;
  for (uint32_t j = 0; j < d.n_group; j++) base |= (uint64_t)((blockIdx.x >> j) & 1u) << d.group_pos[j];
  double acc[kMarginalUnroll];
#pragma unroll
  for (int u = 0; u < kMarginalUnroll; u++) acc[u] = 0.0;
  if (tid < len) {
    uint64_t x = 0;
    bool more = true;
    while (more) {
      C2<T> a[kMarginalUnroll];
#pragma unroll
      for (int u = 0; u < kMarginalUnroll; u++) {
        if (more) a[u] = s[base | x];
        else a[u].x = a[u].y = 0;
        x = ((x | ~d.loop_mask) + 1) & d.loop_mask;      // next setting of the loop bits
        more = more && x != 0;
      }
#pragma unroll
      for (int u = 0; u < kMarginalUnroll; u++)
        acc[u] += (double)a[u].x * (double)a[u].x + (double)a[u].y * (double)a[u].y;
    }
  }
  double mine = 0.0;
#pragma unroll
  for (int u = 0; u < kMarginalUnroll; u++) mine += acc[u];
  uint32_t low = 0;
  for (uint32_t j = 0; j < d.n_low; j++) low |= ((tid >> d.low_pos[j]) & 1u) << j;
  __syncthreads();
  atomicAdd(&h[low], mine);
  KSum v[3] = {{mine, 0}, {0, 0}, {0, 0}};
  block_reduce<3>(v);
  __syncthreads();
  if (tid < (1u << d.n_low)) {
    uint32_t bin = 0;
    for (uint32_t j = 0; j < d.n_low; j++) bin |= ((tid >> j) & 1u) << d.low_bin[j];
    for (uint32_t j = 0; j < d.n_high; j++) bin |= (uint32_t)((base >> d.high_pos[j]) & 1ull) << d.high_bin[j];
    atomicAdd(&bins[bin], h[tid]);
  }
  store_row(v, partials);
}

struct Qubits64 { uint32_t q[64]; };

// Wide marginals: one global atomic per amplitude.
template <typename T>
__global__ void __launch_bounds__(kThreads) k_marginal_wide(const C2<T>* __restrict__ s, uint64_t len, uint32_t k,
                                                            Qubits64 qs, double* __restrict__ out) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < len; i += (uint64_t)gridDim.x * blockDim.x) {
    const C2<T> a = s[i];
    const double p = (double)a.x * (double)a.x + (double)a.y * (double)a.y;
    uint32_t bin = 0;
    for (uint32_t j = 0; j < k; j++) bin |= (uint32_t)((i >> qs.q[j]) & 1ull) << j;
    atomicAdd(&out[bin], p);
  }
}

__global__ void k_zero(double* __restrict__ p, uint64_t count) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = 0.0;
}

// ---- sampler ----
constexpr uint32_t kSampleBlock = 1u << kSampleBlockBits;

template <typename T>
__global__ void __launch_bounds__(kThreads) k_block_sums(const C2<T>* __restrict__ s, uint64_t len,
                                                         double* __restrict__ sums, double* __restrict__ prefix) {
  const uint64_t base = (uint64_t)blockIdx.x * kSampleBlock;
  const uint32_t per = kSampleBlock / kThreads;
  KSum v[1] = {{0, 0}};
  const uint64_t lim = len < base + kSampleBlock ? len : base + kSampleBlock;
  for (uint32_t j = 0; j < per; j++) {
    const uint64_t i = base + (uint64_t)j * kThreads + threadIdx.x;
    if (i < lim) {
      const C2<T> a = s[i];
      kadd(v[0], (double)a.x * (double)a.x + (double)a.y * (double)a.y);
    }
  }
  block_reduce<1>(v);
  if (threadIdx.x == 0) {
    const double t = v[0].s + v[0].c;
    sums[blockIdx.x] = t;
    prefix[blockIdx.x] = t;
  }
}

// Exclusive prefix of `count` sums in place, one workgroup of 1024 threads;
// the grand total lands in total[0] and, if host is not null, in host[0].
// 32768 sums: 72 us with the 1024 partials added by one thread, 30 us with
// the lane scan.
__global__ void __launch_bounds__(1024) k_scan(double* __restrict__ v, uint64_t count, double* __restrict__ total,
                                               double* host) {
  __shared__ double wave_total[16];
  const uint32_t t = threadIdx.x, nt = blockDim.x, lane = t & 63u, wave = t >> 6;
  const uint64_t per = (count + nt - 1) / nt;
  const uint64_t b = t * per, e = b + per < count ? b + per : count;
  double acc = 0.0;
#pragma unroll 8
  for (uint64_t i = b; i < e; i++) acc += v[i];
  double incl = acc;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const double o = __shfl_up(incl, off, 64);
    if ((int)lane >= off) incl += o;
  }
  if (lane == 63) wave_total[wave] = incl;
  __syncthreads();
  double run = 0.0, all = 0.0;
  for (uint32_t w = 0; w < nt / 64; w++) {
    if (w < wave) run += wave_total[w];
    all += wave_total[w];
  }
  const double before = __shfl_up(incl, 1, 64);
  if (lane) run += before;
  if (t == 0) {
    total[0] = all;
    if (host) host[0] = all;
  }
#pragma unroll 8
  for (uint64_t i = b; i < e; i++) {
    const double x = v[i];
    v[i] = run;
    run += x;
  }
}

// One wavefront per shot: a 64-way search over the block prefixes, then the
// chosen block in sub-blocks of 256 amplitudes (4 consecutive ones per lane,
// 16 loads of a lane in flight) until the one that holds the target, then a
// lane scan inside it.  Zero-probability amplitudes are never returned
// (strict `target < cumulative`, as crates/aleph-sv/src/sampling.rs:61-83
// does).  4096 shots at 27 qubits: 158 us with a binary search and 64
// amplitudes a lane -> 50 us.
template <typename T>
__global__ void __launch_bounds__(kThreads) k_sample(const C2<T>* __restrict__ s, uint64_t len,
                                                     const double* __restrict__ prefix, const double* __restrict__ sums,
                                                     uint64_t nblocks, const double* __restrict__ total,
                                                     const double* __restrict__ uni, uint32_t shots,
                                                     uint64_t* __restrict__ out) {
  constexpr uint32_t kSub = kSampleBlock / 256;
  const uint32_t lane = threadIdx.x & 63u;
  const uint64_t waves = ((uint64_t)gridDim.x * blockDim.x) >> 6;
  for (uint64_t shot = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6; shot < shots; shot += waves) {
    const double target = uni[shot] * total[0];
    // last block whose prefix <= target among blocks with positive mass
    uint64_t lo = 0, hi = nblocks;  // invariant: answer in [lo, hi)
    while (hi - lo > 1) {
      const uint64_t step = (hi - lo + 63) / 64, at = lo + lane * step;
      const uint64_t below = __ballot(at < hi && prefix[at] <= target);
      const uint64_t count = below ? __popcll(below) : 1;
      lo += (count - 1) * step;
      hi = lo + step < hi ? lo + step : hi;
    }
    uint64_t blk = lo;
    while (blk > 0 && sums[blk] <= 0.0) blk--;          // never land in an empty block
    while (blk + 1 < nblocks && sums[blk] <= 0.0) blk++;
    double local = target - prefix[blk];
    const uint64_t base = blk * kSampleBlock;
    // Sub-blocks in order until local falls inside one; `keep` is this lane's
    // mass in it, or in the last one with any mass when rounding leaves none.
    double keep = 0.0, keep_local = 1e308;
    uint32_t sub = 0;
    bool inside = false;
    for (uint32_t j0 = 0; j0 < kSub && !inside; j0 += 4) {
      double mine[4];
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) {
        mine[j] = 0.0;
#pragma unroll
        for (uint32_t r = 0; r < 4; r++) {
          const uint64_t i = base + (j0 + j) * 256 + lane * 4 + r;
          if (i < len) {
            const C2<T> a = s[i];
            mine[j] += (double)a.x * (double)a.x + (double)a.y * (double)a.y;
          }
        }
      }
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) {
        double sum = mine[j];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
        if (!inside && sum > 0.0) {
          keep = mine[j];
          sub = j0 + j;
          if (local < sum) {
            keep_local = local;
            inside = true;
          } else {
            local -= sum;
          }
        }
      }
    }
    // inclusive scan over lanes
    double incl = keep;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const double o = __shfl_up(incl, off, 64);
      if ((int)lane >= off) incl += o;
    }
    const double excl = incl - keep;
    const bool hit = inside && keep > 0.0 && keep_local < incl && keep_local >= excl;
    const uint64_t hits = __ballot(hit);
    const uint64_t pos_lanes = __ballot(keep > 0.0);
    int who;
    if (hits) who = __ffsll((long long)hits) - 1;
    else who = pos_lanes ? 63 - __clzll((long long)pos_lanes) : 0;   // rounding overflow: last positive lane
    if ((int)lane == who) {
      const double rem = hits ? keep_local - excl : 1e308;
      double cum = 0.0;
      const uint64_t first = base + sub * 256 + lane * 4;
      uint64_t pick = first, last_pos = first;
      bool found = false;
#pragma unroll
      for (uint32_t j = 0; j < 4; j++) {
        const uint64_t i = first + j;
        if (i >= len) break;
        const C2<T> a = s[i];
        const double p = (double)a.x * (double)a.x + (double)a.y * (double)a.y;
        if (p > 0.0) {
          last_pos = i;
          cum += p;
          if (!found && rem < cum) {
            pick = i;
            found = true;
          }
        }
      }
      out[shot] = found ? pick : last_pos;
    }
  }
}

// Capped so that a dispatch stays under 2^32 work-items; kernels that can
// exceed the cap loop grid-stride (k_sample's grid is shots * 64 threads).
// psi *= 1 / sqrt(norm[0] + norm[1]), the FP64 norm a preceding reduce left
// on the device; a non-finite or zero norm leaves the state alone.
template <typename T>
__global__ void __launch_bounds__(kThreads) k_scale_by_norm(C2<T>* __restrict__ s, uint64_t len,
                                                             const double* __restrict__ norm) {
  const double t = norm[0] + norm[1];
  if (norm[2] != 0.0 || !(t > 0.0) || !isfinite(t)) return;
  const double f = 1.0 / sqrt(t);
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i0 = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i0 < len; i0 += kUnroll * stride) {
    C2<T> a[kUnroll];
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
      const uint64_t i = i0 + u * stride;
      if (i < len) a[u] = s[i];
    }
#pragma unroll
    for (int u = 0; u < kUnroll; u++) {
      const uint64_t i = i0 + u * stride;
      if (i < len) {
        a[u].x = (T)((double)a[u].x * f);
        a[u].y = (T)((double)a[u].y * f);
        s[i] = a[u];
      }
    }
  }
}

// Per block: Re and Im of sum conj(a_i) b_i, sum |a_i - b_i|^2 (compensated,
// FP64) and max |a_i - b_i|^2; a and b may differ in precision.
template <typename TA, typename TB>
__global__ void __launch_bounds__(kThreads) k_compare(const C2<TA>* __restrict__ a, const C2<TB>* __restrict__ b,
                                                       uint64_t len, double* __restrict__ partials) {
  KSum v[3] = {{0, 0}, {0, 0}, {0, 0}};
  double mx = 0.0;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < len; i += (uint64_t)gridDim.x * blockDim.x) {
    const double ar = a[i].x, ai = a[i].y, br = b[i].x, bi = b[i].y;
    kadd(v[0], ar * br + ai * bi);
    kadd(v[1], ar * bi - ai * br);
    const double dr = ar - br, di = ai - bi, d2 = dr * dr + di * di;
    kadd(v[2], d2);
    mx = fmax(mx, d2);
  }
  block_reduce<3>(v);
  __shared__ double shm[kThreads / 64];
  for (int off = 32; off > 0; off >>= 1) mx = fmax(mx, __shfl_down(mx, off, 64));
  if ((threadIdx.x & 63u) == 0) shm[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (uint32_t w = 1; w < blockDim.x / 64; w++) mx = fmax(mx, shm[w]);
    partials[4 * blockIdx.x + 0] = v[0].s + v[0].c;
    partials[4 * blockIdx.x + 1] = v[1].s + v[1].c;
    partials[4 * blockIdx.x + 2] = v[2].s + v[2].c;
    partials[4 * blockIdx.x + 3] = mx;
  }
}

inline uint32_t grid_for(uint64_t items) {
  uint64_t g = (items + kThreads - 1) / kThreads;
  if (g > (1ull << 20)) g = 1ull << 20;
  return (uint32_t)(g == 0 ? 1 : g);
}

}  // namespace

namespace {
template <typename T>
uint32_t reduce_blocks(uint64_t len) {
  // Four tiles a workgroup before the next one: fewer rows for the second
  // launch to add (19 qubits: a measurement's two kernels
  // 17.7 -> 14.5 us, with the rows added by a wavefront per column).
  const uint64_t tiles = (uint64_t)kUnroll * kThreads * 4;
  return (uint32_t)std::min<uint64_t>((len + tiles - 1) / tiles, sizeof(T) == 8 ? kReduceGrid : 2 * kReduceGrid);
}
}  // namespace

void launch_reduce_rows(hipStream_t st, const double* partials, uint32_t rows, double* out) {
  hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(kThreads), 0, st, partials, rows, out);
  ALEPH_HIP_CHECK(hipGetLastError());
}

template <typename T>
void launch_reduce_branch(hipStream_t st, const void* state, uint32_t n, int32_t qubit, double* partials,
                          double* out) {
  const uint64_t len = 1ull << n;
  const uint64_t qmask = qubit >= 0 ? (1ull << qubit) : 0ull;
  hipLaunchKernelGGL((k_reduce_branch<T, 0>), dim3(reduce_blocks<T>(len)), dim3(kThreads), 0, st, (const C2<T>*)state,
                     len, qmask, partials);
  launch_reduce_rows(st, partials, reduce_blocks<T>(len), out);
}

template <typename T>
void launch_sum_p2(hipStream_t st, const void* state, uint32_t n, double* partials, double* out) {
  const uint64_t len = 1ull << n;
  hipLaunchKernelGGL((k_reduce_branch<T, 1>), dim3(reduce_blocks<T>(len)), dim3(kThreads), 0, st, (const C2<T>*)state,
                     len, 0ull, partials);
  launch_reduce_rows(st, partials, reduce_blocks<T>(len), out);
}

template <typename T>
void launch_expect_group(hipStream_t st, const void* state, uint32_t n, uint64_t xmask, const uint64_t* zy,
                         const uint8_t* use_im, uint32_t count, double* partials, double* out) {
  if (count == 0 || count > (uint32_t)kGroupTerms) throw Failure{ALEPH_HIP_ERR_INVALID_ARGUMENT, "group size"};
  GroupTerms g{};
  for (uint32_t t = 0; t < count; t++) {
    g.zy[t] = zy[t];
    if (use_im[t]) g.use_im |= 1u << t;
  }
  g.count = count;
  uint32_t hbit = 0;
  if (xmask) hbit = 63 - __builtin_clzll(xmask);
  const uint64_t pairs = xmask ? (1ull << (n - 1)) : (1ull << n);
  uint32_t blocks = grid_for(pairs);
  if (blocks > kReduceBlocks) blocks = kReduceBlocks;
  hipLaunchKernelGGL(k_expect_group<T>, dim3(blocks), dim3(kThreads), 0, st, (const C2<T>*)state, pairs, xmask, hbit,
                     g, partials);
  hipLaunchKernelGGL(k_reduce_columns, dim3(1), dim3(kThreads), 0, st, partials, blocks, (uint32_t)kGroupTerms, out);
  ALEPH_HIP_CHECK(hipGetLastError());
}

// One workgroup up to 11 qubits (8 amplitudes a thread).
constexpr uint32_t kMeasureSmallQubits = 11;
// From here the collapse's own traffic outweighs a third launch.
constexpr uint32_t kMeasureLargeQubits = 25;

template <typename T>
void launch_measure(hipStream_t st, void* state, uint32_t n, uint32_t qubit, double u, double tol, double* partials,
                    double* host) {
  const uint64_t len = 1ull << n;
  if (n <= kMeasureSmallQubits) {
    hipLaunchKernelGGL(k_measure_small<T>, dim3(1), dim3(kThreads), 0, st, (C2<T>*)state, len, qubit, u, tol, host);
  } else {
    const uint32_t rows = reduce_blocks<T>(len);
    hipLaunchKernelGGL((k_reduce_branch<T, 0>), dim3(rows), dim3(kThreads), 0, st, (const C2<T>*)state, len,
                       1ull << qubit, partials);
    if (n >= kMeasureLargeQubits) {
      MeasureDecision* d = reinterpret_cast<MeasureDecision*>(partials + 3 * (size_t)kReduceBlocks);
      hipLaunchKernelGGL(k_measure_decide, dim3(1), dim3(kThreads), 0, st, (const double*)partials, rows, u, tol, d,
                         host);
      hipLaunchKernelGGL(k_collapse<T>, dim3(grid_for(len)), dim3(kThreads), 0, st, (C2<T>*)state, len, 1ull << qubit,
                         (const MeasureDecision*)d);
    } else {
      hipLaunchKernelGGL(k_measure<T>, dim3(std::min<uint32_t>(grid_for(len / 2), 2 * kReduceGrid)), dim3(kThreads), 0,
                         st, (C2<T>*)state, len / 2, qubit, (const double*)partials, rows, u, tol, host);
    }
  }
  ALEPH_HIP_CHECK(hipGetLastError());
}

template <typename T>
bool launch_marginal(hipStream_t st, const void* state, uint32_t n, uint32_t k, const uint32_t* qubits, double* bins,
                     double* partials, double* host) {
  const uint64_t len = 1ull << n;
  hipLaunchKernelGGL(k_zero, dim3(grid_for(1ull << k)), dim3(kThreads), 0, st, bins, 1ull << k);
  MarginalBits d{};
  uint64_t asked = 0;
  for (uint32_t j = 0; j < k; j++) asked |= 1ull << qubits[j];
  const uint32_t tb = std::min<uint32_t>(8u, n);
  if ((uint32_t)__builtin_popcountll(asked >> tb) > kMarginalHigh) {
    Qubits64 qs{};
    for (uint32_t j = 0; j < k && j < 64; j++) qs.q[j] = qubits[j];
    hipLaunchKernelGGL(k_marginal_wide<T>, dim3(std::min<uint32_t>(grid_for(len), kReduceBlocks)), dim3(kThreads), 0,
                       st, (const C2<T>*)state, len, k, qs, bins);
    ALEPH_HIP_CHECK(hipGetLastError());
    return false;
  }
  // kMarginalGroups workgroups where there are as many bits; every workgroup
  // is a row of the reduction's partials.
  uint32_t left = n - tb;
  for (uint32_t q = tb; q < n && (1ull << left) > kMarginalGroups; q++)
    if (!((asked >> q) & 1ull)) {
      d.loop_mask |= 1ull << q;
      left--;
    }
  for (uint32_t q = tb; q < n; q++)
    if (!((d.loop_mask >> q) & 1ull)) d.group_pos[d.n_group++] = q;
  for (uint32_t j = 0; j < k; j++) {
    if (qubits[j] < tb) {
      d.low_pos[d.n_low] = qubits[j];
      d.low_bin[d.n_low++] = j;
    } else {
      d.high_pos[d.n_high] = qubits[j];
      d.high_bin[d.n_high++] = j;
    }
  }
  hipLaunchKernelGGL(k_marginal<T>, dim3(1u << d.n_group), dim3(kThreads), 0, st, (const C2<T>*)state, len, d, bins,
                     partials);
  launch_reduce_rows(st, partials, 1u << d.n_group, host);
  return true;
}

template <typename T>
void launch_sample(hipStream_t st, const void* state, uint32_t n, double* block_sums, double* scan_tmp,
                   const double* uniforms, uint32_t shots, uint64_t* out, double* host_total) {
  const uint64_t len = 1ull << n;
  const uint64_t nb = n > kSampleBlockBits ? (1ull << (n - kSampleBlockBits)) : 1ull;
  double* sums = block_sums;       // nb
  double* prefix = block_sums + nb;  // nb
  double* total = scan_tmp;
  hipLaunchKernelGGL(k_block_sums<T>, dim3((uint32_t)nb), dim3(kThreads), 0, st, (const C2<T>*)state, len, sums,
                     prefix);
  hipLaunchKernelGGL(k_scan, dim3(1), dim3(1024), 0, st, prefix, nb, total, host_total);
  if (shots) {
    const uint64_t threads = (uint64_t)shots * 64;
    hipLaunchKernelGGL(k_sample<T>, dim3(grid_for(threads)), dim3(kThreads), 0, st, (const C2<T>*)state, len, prefix,
                       sums, nb, total, uniforms, shots, out);
  }
  ALEPH_HIP_CHECK(hipGetLastError());
}

template <typename T>
void launch_normalize(hipStream_t st, void* state, uint32_t n, double* partials, double* res) {
  launch_reduce_branch<T>(st, state, n, -1, partials, res);
  const uint64_t len = 1ull << n;
  hipLaunchKernelGGL(k_scale_by_norm<T>, dim3(grid_for((len + kUnroll - 1) / kUnroll)), dim3(kThreads), 0, st,
                     (C2<T>*)state, len,
                     (const double*)res);
  ALEPH_HIP_CHECK(hipGetLastError());
}

template <typename TA, typename TB>
uint32_t launch_compare(hipStream_t st, const void* a, const void* b, uint32_t n, double* partials) {
  const uint64_t len = 1ull << n;
  uint32_t blocks = grid_for(len);
  if (blocks > kReduceBlocks) blocks = kReduceBlocks;
  hipLaunchKernelGGL((k_compare<TA, TB>), dim3(blocks), dim3(kThreads), 0, st, (const C2<TA>*)a, (const C2<TB>*)b,
                     len, partials);
  ALEPH_HIP_CHECK(hipGetLastError());
  return blocks;
}

template uint32_t launch_compare<double, double>(hipStream_t, const void*, const void*, uint32_t, double*);
template uint32_t launch_compare<double, float>(hipStream_t, const void*, const void*, uint32_t, double*);
template uint32_t launch_compare<float, double>(hipStream_t, const void*, const void*, uint32_t, double*);
template uint32_t launch_compare<float, float>(hipStream_t, const void*, const void*, uint32_t, double*);

#define ALEPH_INST(T)                                                                                           \
  template void launch_reduce_branch<T>(hipStream_t, const void*, uint32_t, int32_t, double*, double*);         \
  template void launch_sum_p2<T>(hipStream_t, const void*, uint32_t, double*, double*);                         \
  template void launch_normalize<T>(hipStream_t, void*, uint32_t, double*, double*);                            \
  template void launch_expect_group<T>(hipStream_t, const void*, uint32_t, uint64_t, const uint64_t*,           \
                                       const uint8_t*, uint32_t, double*, double*);                             \
  template void launch_measure<T>(hipStream_t, void*, uint32_t, uint32_t, double, double, double*, double*);    \
  template bool launch_marginal<T>(hipStream_t, const void*, uint32_t, uint32_t, const uint32_t*, double*,      \
                                   double*, double*);                                                           \
  template void launch_sample<T>(hipStream_t, const void*, uint32_t, double*, double*, const double*, uint32_t, \
                                 uint64_t*, double*);
ALEPH_INST(double)
ALEPH_INST(float)
#undef ALEPH_INST

}  // namespace aleph
