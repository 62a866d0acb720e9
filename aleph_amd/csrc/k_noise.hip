// Noise trajectories: one workgroup runs one whole trajectory at a time,
// gate by gate and channel by channel, then draws its terminal outcome.
// Staged programs keep the state in registers (k_staged, up to 14 qubits);
// for the others states of up to 13 qubits live in LDS (one read of the
// program from L2, no HBM traffic per gate) and wider ones in the
// workgroup's own slice of a device buffer (k_trajectories).  The RNG is
// counter-based, so every thread of the workgroup computes the same draw
// without communication.
#include "common.hpp"
#include "inplace.hpp"
#include "noise.hpp"

namespace aleph {
namespace {

constexpr uint64_t kGolden = 0x9E3779B97F4A7C15ull;

// splitmix64 finaliser (Steele, Lea & Flood, OOPSLA 2014).
__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// Per-shot key: crates/aleph-sv/src/noise/apply.rs:169-180.
__device__ __forceinline__ uint64_t shot_key(uint64_t seed, uint64_t shot) {
  return mix64(seed * kGolden + shot + kGolden);
}

// Draw c (0-based) of the splitmix64 stream seeded with `key`, as a
// 53-bit uniform in [0, 1).
__device__ __forceinline__ double uniform(uint64_t key, uint32_t c) {
  return (double)(mix64(key + (uint64_t)(c + 1) * kGolden) >> 11) * (1.0 / 9007199254740992.0);
}

__device__ __forceinline__ uint64_t insert_zero(uint64_t x, uint32_t b) {
  return ((x >> b) << (b + 1)) | (x & ((1ull << b) - 1ull));
}

// z * i^e for e in 0..3 (exact: component swaps and negations).
__device__ __forceinline__ double2 mul_ipow(double2 z, uint32_t e) {
  switch (e & 3u) {
    case 0: return z;
    case 1: return make_double2(-z.y, z.x);
    case 2: return make_double2(-z.x, -z.y);
    default: return make_double2(z.y, -z.x);
  }
}

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// Sum over the workgroup; every thread returns the same value (the wave
// partials are added in one fixed order by every thread).
__device__ double block_sum(double v, double* red) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double t = 0.0;
  const uint32_t nw = (blockDim.x + 63u) >> 6;
#pragma nounroll
  for (uint32_t w = 0; w < nw; w++) t += red[w];
  __syncthreads();
  return t;
}

template <int K>
__device__ void apply_dense(double2* s, uint32_t n, const TrajOp& op, const double* m) {
  constexpr uint32_t D = 1u << K;
  uint32_t sorted[K];
#pragma unroll
  for (int i = 0; i < K; i++) sorted[i] = op.q[i];
#pragma unroll
  for (int i = 0; i < K; i++)
#pragma unroll
    for (int j = 0; j + 1 < K - i; j++)
      if (sorted[j] > sorted[j + 1]) {
        const uint32_t t = sorted[j];
        sorted[j] = sorted[j + 1];
        sorted[j + 1] = t;
      }
  const uint64_t groups = 1ull << (n - K);
  for (uint64_t g = threadIdx.x; g < groups; g += blockDim.x) {
    uint64_t base = g;
#pragma unroll
    for (int i = 0; i < K; i++) base = insert_zero(base, sorted[i]);
    if ((base & op.cmask) != op.cmask) continue;
    double2 a[D];
    uint64_t idx[D];
#pragma unroll
    for (uint32_t j = 0; j < D; j++) {
      uint64_t x = base;
#pragma unroll
      for (int t = 0; t < K; t++)
        if ((j >> (K - 1 - t)) & 1u) x |= 1ull << op.q[t];
      idx[j] = x;
      a[j] = s[x];
    }
#pragma unroll
    for (uint32_t r = 0; r < D; r++) {
      double re = 0.0, im = 0.0;
#pragma unroll
      for (uint32_t c = 0; c < D; c++) {
        const double mr = m[2 * (r * D + c)], mi = m[2 * (r * D + c) + 1];
        re += mr * a[c].x - mi * a[c].y;
        im += mr * a[c].y + mi * a[c].x;
      }
      s[idx[r]] = make_double2(re, im);
    }
  }
}

__device__ void apply_diag(double2* s, uint32_t n, const TrajOp& op, const double* d) {
  const uint64_t N = 1ull << n;
  for (uint64_t x = threadIdx.x; x < N; x += blockDim.x) {
    if ((x & op.cmask) != op.cmask) continue;
    uint32_t j = 0;
    for (uint32_t t = 0; t < op.k; t++) j = (j << 1) | (uint32_t)((x >> op.q[t]) & 1ull);
    s[x] = cmul(s[x], make_double2(d[2 * j], d[2 * j + 1]));
  }
}

// DiagonalPhase (crates/aleph-ir/src/diagonal_phase.rs:60-72): term t adds
// angles[t] when popcount(cond & x) is odd for each of its conditions.
__device__ void apply_phase(double2* s, uint32_t n, const TrajOp& op, const double* angles, const uint64_t* conds,
                            const uint32_t* offsets) {
  const uint64_t N = 1ull << n;
  for (uint64_t x = threadIdx.x; x < N; x += blockDim.x) {
    double phi = 0.0;
    for (uint32_t t = 0; t < op.count; t++) {
      bool fire = true;
      for (uint32_t c = offsets[t]; c < offsets[t + 1]; c++)
        if ((__popcll(conds[c] & x) & 1) == 0) fire = false;
      if (fire) phi += angles[t];
    }
    double sn, cs;
    sincos(phi, &sn, &cs);
    s[x] = cmul(s[x], make_double2(cs, sn));
  }
}

// Pauli string i^ny X^xm Z^zm (Y = i X Z on its qubit):
// psi'[x ^ xm] = i^ny (-1)^popcount(zm & x) psi[x].
__device__ void apply_pauli(double2* s, uint32_t n, uint64_t xm, uint64_t zm) {
  const uint32_t ny = (uint32_t)__popcll(xm & zm);
  const uint64_t N = 1ull << n;
  if (xm == 0) {
    for (uint64_t x = threadIdx.x; x < N; x += blockDim.x)
      s[x] = mul_ipow(s[x], ny + 2u * ((uint32_t)__popcll(zm & x) & 1u));
    return;
  }
  const uint32_t lb = (uint32_t)__ffsll((long long)xm) - 1u;
  for (uint64_t t = threadIdx.x; t < N / 2; t += blockDim.x) {
    const uint64_t x = insert_zero(t, lb), y = x ^ xm;
    const double2 a = s[x], b = s[y];
    s[y] = mul_ipow(a, ny + 2u * ((uint32_t)__popcll(zm & x) & 1u));
    s[x] = mul_ipow(b, ny + 2u * ((uint32_t)__popcll(zm & y) & 1u));
  }
}

// One-qubit quantum jump (crates/aleph-sv/src/noise/apply.rs:68-133).
// Branch probabilities are summed only until the drawn branch is known.
__device__ void apply_kraus(double2* s, uint32_t n, const TrajOp& op, const double* kraus, double u, double* red) {
  const uint32_t q = op.q[0];
  const uint64_t qb = 1ull << q, half = (1ull << n) / 2;
  double acc = 0.0, pc = 0.0;
  uint32_t chosen = op.count;
  for (uint32_t b = 0; b < op.count; b++) {
    const double* k = kraus + 8 * b;
    double part = 0.0;
    for (uint64_t t = threadIdx.x; t < half; t += blockDim.x) {
      const uint64_t i0 = insert_zero(t, q), i1 = i0 | qb;
      const double2 a0 = s[i0], a1 = s[i1];
      const double o0r = k[0] * a0.x - k[1] * a0.y + k[2] * a1.x - k[3] * a1.y;
      const double o0i = k[0] * a0.y + k[1] * a0.x + k[2] * a1.y + k[3] * a1.x;
      const double o1r = k[4] * a0.x - k[5] * a0.y + k[6] * a1.x - k[7] * a1.y;
      const double o1i = k[4] * a0.y + k[5] * a0.x + k[6] * a1.y + k[7] * a1.x;
      part += o0r * o0r + o0i * o0i + o1r * o1r + o1i * o1i;
    }
    const double pb = block_sum(part, red);
    acc += pb;
    pc = pb;
    if (u < acc) {
      chosen = b;
      break;
    }
  }
  if (chosen == op.count) chosen = op.count - 1;   // the last branch absorbs rounding (pc is its probability)
  if (pc < 1e-300) return;                          // degenerate branch: keep the pre-channel state
  const double inv = 1.0 / sqrt(pc);
  const double* k = kraus + 8 * chosen;
  for (uint64_t t = threadIdx.x; t < half; t += blockDim.x) {
    const uint64_t i0 = insert_zero(t, q), i1 = i0 | qb;
    const double2 a0 = s[i0], a1 = s[i1];
    const double o0r = k[0] * a0.x - k[1] * a0.y + k[2] * a1.x - k[3] * a1.y;
    const double o0i = k[0] * a0.y + k[1] * a0.x + k[2] * a1.y + k[3] * a1.x;
    const double o1r = k[4] * a0.x - k[5] * a0.y + k[6] * a1.x - k[7] * a1.y;
    const double o1i = k[4] * a0.y + k[5] * a0.x + k[6] * a1.y + k[7] * a1.x;
    s[i0] = make_double2(o0r * inv, o0i * inv);
    s[i1] = make_double2(o1r * inv, o1i * inv);
  }
}

template <bool kLds>
__global__ void __launch_bounds__(kLds ? kNoiseThreadsLds : kNoiseThreadsWide) k_trajectories(TrajProgram p, double2* slices, uint64_t* out) {
  extern __shared__ double2 lds_state[];
  __shared__ double red[16];
  __shared__ double scan[16];
  __shared__ unsigned long long found, last_pos;
  const uint32_t n = p.n;
  const uint64_t N = 1ull << n;
  double2* s = kLds ? lds_state : slices + (size_t)blockIdx.x * N;
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, nw = (blockDim.x + 63u) >> 6;
  for (uint64_t shot = blockIdx.x; shot < p.shots; shot += gridDim.x) {
    const uint64_t key = shot_key(p.seed, p.shot0 + shot);
    uint32_t draw = 0;
    for (uint64_t i = threadIdx.x; i < N; i += blockDim.x) s[i] = make_double2(i == 0 ? 1.0 : 0.0, 0.0);
    if (threadIdx.x == 0) {
      found = ~0ull;
      last_pos = 0;
    }
    __syncthreads();
    for (uint32_t o = 0; o < p.n_ops; o++) {
      const TrajOp& op = p.ops[o];
      switch (op.kind) {
        case TrajOp::DENSE:
          if (op.k == 1) apply_dense<1>(s, n, op, p.reals + op.off);
          else if (op.k == 2) apply_dense<2>(s, n, op, p.reals + op.off);
          else apply_dense<3>(s, n, op, p.reals + op.off);
          break;
        case TrajOp::DIAG:
          apply_diag(s, n, op, p.reals + op.off);
          break;
        case TrajOp::PHASE:
          apply_phase(s, n, op, p.reals + op.off, p.masks + op.off2, p.index + op.off3);
          break;
        case TrajOp::PAULI: {
          // crates/aleph-sv/src/noise/apply.rs:46-66: one draw, cumulative
          // weights, the last term absorbs rounding.
          const double u = uniform(key, draw++);
          const double* w = p.reals + op.off;
          uint32_t chosen = op.count - 1;
          double acc = 0.0;
          for (uint32_t b = 0; b < op.count; b++) {
            acc += w[b];
            if (u < acc) {
              chosen = b;
              break;
            }
          }
          const uint64_t xm = p.masks[op.off2 + 2 * chosen], zm = p.masks[op.off2 + 2 * chosen + 1];
          if (xm | zm) apply_pauli(s, n, xm, zm);
          break;
        }
        default:
          apply_kraus(s, n, op, p.reals + op.off, uniform(key, draw++), red);
          break;
      }
      __syncthreads();
    }
    // Terminal draw (crates/aleph-sv/src/sampling.rs:61-91): the first index
    // whose running sum of |psi|^2 exceeds u * total, zero-mass bins
    // skipped, the last positive bin when rounding leaves nothing.  Each
    // thread owns a contiguous segment; a wave scan gives its offset.
    const uint64_t seg = N >= blockDim.x ? N / blockDim.x : 1ull;
    const uint64_t lo = (uint64_t)threadIdx.x * seg, hi = lo < N ? lo + seg : lo;
    double part = 0.0;
    uint64_t mine_last = 0;
    bool any = false;
    for (uint64_t i = lo; i < hi; i++) {
      const double2 a = s[i];
      const double pr = a.x * a.x + a.y * a.y;
      if (pr > 0.0) {
        part += pr;
        mine_last = i;
        any = true;
      }
    }
    double incl = part;
    for (int d = 1; d < 64; d <<= 1) {
      const double y = __shfl_up(incl, d);
      if ((int)lane >= d) incl += y;
    }
    double excl = __shfl_up(incl, 1);
    if (lane == 0) excl = 0.0;
    if (lane == 63) scan[wave] = incl;
    if (any) atomicMax(&last_pos, (unsigned long long)mine_last);
    __syncthreads();
    double woff = 0.0, total = 0.0;
    for (uint32_t w = 0; w < nw; w++) {
      if (w < wave) woff += scan[w];
      total += scan[w];
    }
    const double target = uniform(key, draw++) * total;
    double cum = woff + excl;
    if (cum <= target) {
      for (uint64_t i = lo; i < hi; i++) {
        const double2 a = s[i];
        const double pr = a.x * a.x + a.y * a.y;
        if (pr > 0.0) {
          cum += pr;
          if (target < cum) {
            atomicMin(&found, (unsigned long long)i);
            break;
          }
        }
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      uint64_t idx = found != ~0ull ? (uint64_t)found : (uint64_t)last_pos;
      // Readout error (apply.rs:135-158): one draw per qubit that has one,
      // in ascending qubit order, flipping the bit with P(1-t | t).
      for (uint32_t q = 0; q < n; q++) {
        if (!((p.readout_mask >> q) & 1ull)) continue;
        const uint32_t bit = (uint32_t)((idx >> q) & 1ull);
        if (uniform(key, draw++) < p.readout[2 * q + bit]) idx ^= 1ull << q;
      }
      out[shot] = idx;
    }
    __syncthreads();
  }
}


// ---- register-resident trajectories (TStage, noise.hpp) ----
//
// Measured on MI355X against k_trajectories (state in LDS, one op at a time with
// barriers, a norm reduction per Kraus channel): the 12-qubit depth-10 noisy
// brickwall, 20 000 shots, 46.9 -> 9.3 ms a call (5.8 ms of it this kernel, the
// rest on the host); 14 qubits, 2 048 shots, 63.3 -> 7.6 ms.  Bound by issue: four
// waves per SIMD, vector instructions for the amplitudes and scalar ones for the
// records.

// Register-slot patterns of register bit g: bit r of kSlots[g] is bit g of r.
__device__ __constant__ constexpr uint32_t kSlots[4] = {0xAAAAu, 0xCCCCu, 0xF0F0u, 0xFF00u};

__device__ __forceinline__ double flip_hi(double x, uint32_t s) {
  return __builtin_bit_cast(double, __builtin_bit_cast(uint64_t, x) ^ ((uint64_t)s << 32));
}

// Conditions of the record loop go through opaque() so that exclusive ifs are
// not rebuilt into a switch.
using fused::opaque;
using fused::pair_update;

// Plain components: arrays of the HIP vector type stay in scratch memory.
using Amp = C2<double>;

struct Mat2 {
  double v[8];
};

// F^dagger M F of a one-qubit matrix: rows and columns swapped under an X
// frame, off-diagonal entries negated under a Z frame.
__device__ __forceinline__ Mat2 in_frame(const Mat2& in, bool x, bool z) {
  const double (&m)[8] = in.v;
  Mat2 o;
  const uint32_t s = z ? 0x80000000u : 0u;
#pragma unroll
  for (int e = 0; e < 2; e++) {
    o.v[e] = x ? m[6 + e] : m[e];
    o.v[6 + e] = x ? m[e] : m[6 + e];
    o.v[2 + e] = flip_hi(x ? m[4 + e] : m[2 + e], s);
    o.v[4 + e] = flip_hi(x ? m[2 + e] : m[4 + e], s);
  }
  return o;
}

__device__ __forceinline__ double uniform_value(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)u), hi = __builtin_amdgcn_readfirstlane((uint32_t)(u >> 32));
  return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}

__device__ __forceinline__ Mat2 load_mat(Prog<double>* m) {
  Mat2 o;
#pragma unroll
  for (int e = 0; e < 8; e++) o.v[e] = m[e];
  return o;
}

// A TOp in scalar registers, as two 16-dword loads.
typedef uint32_t u32x16 __attribute__((ext_vector_type(16)));
struct Record {
  u32x16 w, v;
  __device__ __forceinline__ double f64(uint32_t lo, uint32_t hi) const {
    return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
  }
  __device__ __forceinline__ double lam() const { return f64(w[12], w[13]); }
  __device__ __forceinline__ double m(int e) const { return f64(v[2 * e], v[2 * e + 1]); }
};
__device__ __forceinline__ Record record(const TOp* ops, uint32_t o) {
  Prog<u32x16>* p = (Prog<u32x16>*)(uintptr_t)(ops + o);
  Record r;
  r.w = p[0];
  r.v = p[1];
  return r;
}
constexpr uint32_t kLook = 0x80000000u;   // the Kraus channel has to look at the state

template <int G, int B, bool kCtl>
__device__ __forceinline__ void one_qubit(Amp (&a)[1 << G], const Mat2& m, uint32_t tctl, const uint32_t (&rl)[G],
                                          uint32_t fx, uint32_t cm) {
#pragma unroll
  for (int r = 0; r < (1 << G); r++) {
    if (r & (1 << B)) continue;
    bool on = true;
    if constexpr (kCtl) {
      uint32_t ro = 0;
#pragma unroll
      for (int g = 0; g < G; g++)
        if (r & (1 << g)) ro |= rl[g];
      on = (((tctl | ro) ^ fx) & cm) == cm;
    }
    if (on) pair_update(a[r], a[r | (1 << B)], m.v);
  }
}

// sel: bit B for an uncontrolled operator on register bit B, bit 4 + B for a
// controlled one, none to do nothing.
template <int G, bool kRare, int B = 0>
__device__ __forceinline__ void dispatch_one(Amp (&a)[1 << G], uint32_t sel, const Mat2& m, uint32_t tctl,
                                             const uint32_t (&rl)[G], uint32_t fx, uint32_t cm) {
  if constexpr (B < G) {
    if (sel & (1u << B)) one_qubit<G, B, false>(a, m, tctl, rl, fx, cm);
    if (kRare && (sel & (16u << B))) one_qubit<G, B, true>(a, m, tctl, rl, fx, cm);
    dispatch_one<G, kRare, B + 1>(a, sel, m, tctl, rl, fx, cm);
  }
}

// Sum over this thread of |row 0|^2 + |row 1|^2 of K applied to the pairs of
// register bit B.
template <int G, int B = 0>
__device__ __forceinline__ double branch_sum(const Amp (&a)[1 << G], uint32_t bit, const Mat2& k) {
  if constexpr (B < G) {
    if (bit != (uint32_t)B) return branch_sum<G, B + 1>(a, bit, k);
    double part = 0.0;
#pragma unroll
    for (int r = 0; r < (1 << G); r++) {
      if (r & (1 << B)) continue;
      const Amp x = a[r], y = a[r | (1 << B)];
      const double pr = k.v[0] * x.x - k.v[1] * x.y + k.v[2] * y.x - k.v[3] * y.y;
      const double pi = k.v[0] * x.y + k.v[1] * x.x + k.v[2] * y.y + k.v[3] * y.x;
      const double qr = k.v[4] * x.x - k.v[5] * x.y + k.v[6] * y.x - k.v[7] * y.y;
      const double qi = k.v[4] * x.y + k.v[5] * x.x + k.v[6] * y.y + k.v[7] * y.x;
      part += pr * pr + pi * pi + qr * qr + qi * qi;
    }
    return part;
  } else {
    return 0.0;
  }
}

// Uncontrolled 4x4 on register bits A > B (A the matrix MSB), rows and
// columns permuted by xm and signed by zm (both over the matrix index).
template <int G, int A, int B, int Q = 0>
__device__ __forceinline__ void two_qubit(Amp (&a)[1 << G], Prog<double>* m, uint32_t xm, uint32_t zm) {
  if constexpr (Q < (1 << (G - 2))) {
    constexpr int lo = (Q & ((1 << B) - 1)) | ((Q >> B) << (B + 1));
    constexpr int r = (lo & ((1 << A) - 1)) | ((lo >> A) << (A + 1));
    const Amp v0 = a[r], v1 = a[r | (1 << B)], v2 = a[r | (1 << A)], v3 = a[r | (1 << A) | (1 << B)];
    Amp o[4];
#pragma unroll
    for (uint32_t row = 0; row < 4; row++) {
      asm volatile("" ::: "memory");   // matrix rows are read just before use, not all held in registers
      double re = 0.0, im = 0.0;
#pragma unroll
      for (uint32_t col = 0; col < 4; col++) {
        const uint32_t e = 2 * (4 * (row ^ xm) + (col ^ xm));
        const uint32_t s = (uint32_t)__popc(zm & (row ^ col)) << 31;
        const double mr = flip_hi(m[e], s), mi = flip_hi(m[e + 1], s);
        const Amp v = col == 0 ? v0 : col == 1 ? v1 : col == 2 ? v2 : v3;
        re += mr * v.x - mi * v.y;
        im += mr * v.y + mi * v.x;
      }
      o[row] = Amp{re, im};
    }
    a[r] = o[0];
    a[r | (1 << B)] = o[1];
    a[r | (1 << A)] = o[2];
    a[r | (1 << A) | (1 << B)] = o[3];
    two_qubit<G, A, B, Q + 1>(a, m, xm, zm);
  }
}

template <int G, int A = 1, int B = 0>
__device__ __forceinline__ void dispatch_two(Amp (&a)[1 << G], uint32_t sel, Prog<double>* m, uint32_t xm,
                                             uint32_t zm) {
  if constexpr (A < G) {
    if constexpr (B < A) {
      if (sel & (1u << (A * (A - 1) / 2 + B))) two_qubit<G, A, B>(a, m, xm, zm);
      dispatch_two<G, A, B + 1>(a, sel, m, xm, zm);
    } else {
      dispatch_two<G, A + 1, 0>(a, sel, m, xm, zm);
    }
  }
}

// Negate the slots whose bit is set in sgn.
template <int G>
__device__ __forceinline__ void flip_slots(Amp (&a)[1 << G], uint32_t sgn) {
#pragma unroll
  for (int r = 0; r < (1 << G); r++) {
    const uint32_t s = (sgn << (31 - r)) & 0x80000000u;
    a[r].x = flip_hi(a[r].x, s);
    a[r].y = flip_hi(a[r].y, s);
  }
}

// Diagonal over k targets (4 bits each in `targets`, MSB first) with
// controls cm; `phys` is the thread's physical index with the register bits
// as the frame leaves them.
template <int G>
__device__ __forceinline__ void diagonal(Amp (&a)[1 << G], const double* d, uint32_t targets, uint32_t k, uint32_t phys,
                                         const uint32_t (&rl)[G], uint32_t cm) {
  uint32_t tsel = 0, rsel[G];
#pragma unroll
  for (int g = 0; g < G; g++) rsel[g] = 0;
#pragma nounroll
  for (uint32_t t = 0; t < k; t++) {
    const uint32_t b = 1u << (k - 1 - t), qb = 1u << ((targets >> (4 * t)) & 15u);
    if (phys & qb) tsel |= b;
#pragma unroll
    for (int g = 0; g < G; g++)
      if (rl[g] == qb) rsel[g] = b;
  }
#pragma unroll
  for (int r = 0; r < (1 << G); r++) {
    uint32_t sel = tsel, ro = 0;
#pragma unroll
    for (int g = 0; g < G; g++)
      if (r & (1 << g)) {
        sel ^= rsel[g];
        ro |= rl[g];
      }
    const bool on = ((phys ^ ro) & cm) == cm;
    const Amp v = cmul(a[r], Amp{d[2 * sel], d[2 * sel + 1]});
    a[r].x = on ? v.x : a[r].x;
    a[r].y = on ? v.y : a[r].y;
  }
}

// kRare: the program has two-qubit matrices, diagonals other than signs, or
// controlled gates; without them the kernel needs far fewer registers.
template <int G, bool kRare, int TH, int W>
__global__ void __launch_bounds__(TH, W) k_staged(TrajProgram p, StagedProgram sp, uint64_t* __restrict__ out) {
  constexpr int N = 1 << G;
  extern __shared__ double2 lds_state[];
  __shared__ double red[16];
  __shared__ double scan[16];
  __shared__ uint32_t xscan[16];
  __shared__ unsigned long long found, last_pos;
  const uint32_t n = p.n, tid = threadIdx.x, T = 1u << (n - G);
  const bool active = tid < T;
  const uint32_t lane = tid & 63u, wave = tid >> 6, nw = (blockDim.x + 63u) >> 6;
  // Per record: the frame before it (low word) and the frame before its
  // Kraus channel with the look flag on top (high word); then the exchange
  // buffer, which holds the channels' frames and flags before stage 0.
  uint64_t* const words = reinterpret_cast<uint64_t*>(lds_state);       // n_ops + 1
  double* const buf = reinterpret_cast<double*>(words + sp.n_ops + 1);  // 2^n + 2^n / 16 doubles
  uint32_t* const frames = reinterpret_cast<uint32_t*>(buf);            // n_chan + 1
  uint8_t* const look = reinterpret_cast<uint8_t*>(frames + sp.n_chan + 1);   // n_chan
  for (uint64_t shot = blockIdx.x; shot < p.shots; shot += gridDim.x) {
    const uint64_t key = shot_key(p.seed, p.shot0 + shot);
    // Every channel's draw, one lane each: the Pauli drawn (x in the low and
    // z in the high half-word) or whether a Kraus channel must look at the
    // state; then the frame before every channel as a prefix XOR.
    if (tid == 0) {
      frames[0] = 0;
      found = ~0ull;
      last_pos = 0;
    }
    uint32_t carry = 0;
    for (uint32_t c0 = 0; c0 < sp.n_chan; c0 += blockDim.x) {
      const uint32_t c = c0 + tid;
      uint32_t mask = 0;
      if (c < sp.n_chan) {
        const TChan& ch = sp.chans[c];
        const double u = uniform(key, c);
        uint8_t need = 0;
        if (ch.pauli) {
          const double* w = p.reals + ch.off;
          uint32_t chosen = ch.count - 1;
          double acc = 0.0;
#pragma nounroll
          for (uint32_t b = 0; b < ch.count; b++) {
            acc += w[b];
            if (u < acc) {
              chosen = b;
              break;
            }
          }
          mask = (uint32_t)p.masks[ch.off2 + 2 * chosen] | ((uint32_t)p.masks[ch.off2 + 2 * chosen + 1] << 16);
        } else {
          need = u < ch.thr ? 0 : 1;
        }
        look[c] = need;
      }
      uint32_t incl = mask;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const uint32_t y = __shfl_up(incl, d);
        if ((int)lane >= d) incl ^= y;
      }
      if (lane == 63) xscan[wave] = incl;
      __syncthreads();
      uint32_t before = carry;
#pragma nounroll
      for (uint32_t w = 0; w < nw; w++) {
        if (w < wave) before ^= xscan[w];
        carry ^= xscan[w];
      }
      if (c < sp.n_chan) frames[c + 1] = before ^ incl;
      __syncthreads();
    }
    __syncthreads();
    for (uint32_t o = tid; o <= sp.n_ops; o += blockDim.x) {
      const TOp& op = sp.ops[o];
      const uint32_t f1 = frames[op.f1] | (op.chan != ~0u && look[op.chan] ? kLook : 0u);
      words[o] = (uint64_t)frames[op.f0] | ((uint64_t)f1 << 32);
    }
    __syncthreads();
    Amp a[N];
    bool repeat_full = false;    // the record that runs again has to look at the state
    double floor_norm = 1.0;     // lower bound of the squared norm since the last normalisation
    uint32_t rl[G];
    uint32_t tidx = 0, tslot = 0;
    Record cur = record(sp.ops, 0);
    uint64_t word = words[0];
    for (uint32_t si = 0; si < sp.n_stages; si++) {
      Prog<TStage>& st = prog(sp.stages)[si];
      uint32_t idx = 0, slot = 0;
#pragma nounroll
      for (uint32_t j = 0; j < st.n_tb; j++)
        if ((tid >> j) & 1u) {
          idx |= st.tl[j];
          slot ^= st.ts[j];
        }
      if (si == 0) {
#pragma unroll
        for (int r = 0; r < N; r++) a[r] = Amp{0.0, 0.0};
        if (tid == 0) a[0].x = 1.0;
      } else {
        // Real parts, then imaginary parts, through 2^n doubles.
        Prog<TStage>& pv = prog(sp.stages)[si - 1];
        if (active) {
#pragma unroll
          for (int r = 0; r < N; r++) buf[tslot ^ pv.ls[r]] = a[r].x;
        }
        __syncthreads();
        if (active) {
#pragma unroll
          for (int r = 0; r < N; r++) a[r].x = buf[slot ^ st.ls[r]];
        }
        __syncthreads();
        // Opaque to the compiler: the addresses are formed again instead of
        // staying in registers from the real parts.
        asm volatile("" : "+v"(tslot), "+v"(slot));
        if (active) {
#pragma unroll
          for (int r = 0; r < N; r++) buf[tslot ^ pv.ls[r]] = a[r].y;
        }
        __syncthreads();
        if (active) {
#pragma unroll
          for (int r = 0; r < N; r++) a[r].y = buf[slot ^ st.ls[r]];
        }
        __syncthreads();
      }
      tidx = idx;
      tslot = slot;
      uint32_t rall = 0;
#pragma unroll
      for (int g = 0; g < G; g++) {
        rl[g] = st.rl[g];
        rall |= rl[g];
      }
      uint32_t sgn = 0;        // bit r: amplitude r is to be negated
      bool pending = false;
      // The loop body is a row of plain ifs, each changing the amplitudes in
      // place: with else chains, continues or an inner loop the compiler
      // moves all of them to new registers at every join.
      bool gate_applied = false;
      uint32_t o = st.op_begin;
      while (o < st.op_end) {
        const uint32_t kind = cur.w[0], cm = cur.w[4], qb = cur.w[2], chan = cur.w[8];
        const uint32_t f0 = __builtin_amdgcn_readfirstlane((uint32_t)word);
        const uint32_t f1k = __builtin_amdgcn_readfirstlane((uint32_t)(word >> 32));
        const uint32_t f1 = f1k & ~kLook, fx = f0 & 0x3FFFu, fz = (f0 >> 16) & 0x3FFFu;
        if (kind == TOp::SIGN) {
          // Signs are only noted per slot (one bit each) and applied before
          // the next operator that mixes amplitudes.
          const uint32_t tm = cm & ~rall;
          uint32_t pat = 0xFFFFu;
#pragma unroll
          for (int g = 0; g < G; g++)
            if (cm & rl[g]) pat &= (fx & rl[g]) ? ~kSlots[g] : kSlots[g];
          sgn ^= (((tidx ^ fx) & tm) == tm) ? pat : 0u;
          pending = true;
        }
        const uint32_t flush = opaque(pending && kind != TOp::SIGN && kind != TOp::DIAG ? 1u : 0u);
        if (flush) flip_slots<G>(a, sgn);
        sgn = flush ? 0u : sgn;
        pending = pending && !flush;
        if (kRare && opaque(kind) == TOp::DIAG) diagonal<G>(a, p.reals + cur.w[5], cur.w[2], cur.w[3], tidx ^ fx, rl, cm);
        if (kRare) {
          const uint32_t xm = ((fx & qb) ? 2u : 0u) | ((fx & cur.w[3]) ? 1u : 0u);
          const uint32_t zm = ((fz & qb) ? 2u : 0u) | ((fz & cur.w[3]) ? 1u : 0u);
          dispatch_two<G>(a, opaque(kind == TOp::TWO ? 1u << cur.w[1] : 0u), prog(p.reals) + cur.w[5], xm, zm);
        }
        // A one-qubit operator: a gate (controls only without a channel), a
        // Kraus channel, or a gate with the channel's K_0 folded in.  When
        // the fold does not hold (a Pauli drawn in between changed the
        // frame, or the channel has to look at the state) the record runs
        // twice: the bare gate, then the chosen Kraus operator.
        bool advance = true;
        uint32_t bit = kind == TOp::ONE || kind == TOp::KRAUS ? cur.w[1] : ~0u;
        bool x = (fx & qb) != 0, z = (fz & qb) != 0, look_now = false, kraus_now = false;
        Mat2 m;
#pragma unroll
        for (int e = 0; e < 8; e++) m.v[e] = cur.m(e);
        if (chan != ~0u) {
          bool full = (f1k & kLook) != 0;
          if (!full && !gate_applied) {
            floor_norm = uniform_value(floor_norm * cur.lam());
            full = floor_norm < 1e-60;
          }
          const bool split = full || gate_applied || (kind == TOp::ONE && ((f0 ^ f1) & (qb | (qb << 16))) != 0);
          if (split && kind == TOp::ONE && !gate_applied) {
            m = load_mat(prog(p.reals) + cur.w[5]);
            advance = false;
            repeat_full = full;
          } else if (split) {
            kraus_now = true;
            look_now = kind == TOp::ONE ? repeat_full : full;
          }
        }
        if (kraus_now) {
          x = (f1 & qb) != 0;
          z = ((f1 >> 16) & qb) != 0;
          uint32_t chosen = 0;
          double scale = 1.0;
          if (look_now) {
            // Branch probabilities relative to the norm, summed until the
            // drawn branch is known (as apply_kraus).
            double part = 0.0;
#pragma unroll
            for (int r = 0; r < N; r++) part += a[r].x * a[r].x + a[r].y * a[r].y;
            const double norm = uniform_value(block_sum(part, red));
            const double u = uniform_value(uniform(key, chan) * norm);
            double acc = 0.0, pc = 0.0;
            bool found_branch = false;
            uint32_t b = 0;
            while (b < cur.w[7] && !found_branch) {
              pc = uniform_value(block_sum(branch_sum<G>(a, bit, in_frame(load_mat(prog(p.reals) + cur.w[6] + 8 * b), x, z)), red));
              acc += pc;
              found_branch = u < acc;
              b++;
            }
            chosen = b - 1;      // the last branch absorbs rounding
            if (pc < 1e-300 * norm) bit = ~0u;     // degenerate branch: keep the pre-channel state
            else scale = 1.0 / sqrt(pc);
            floor_norm = 1.0;
          }
          m = load_mat(prog(p.reals) + cur.w[6] + 8 * chosen);
#pragma unroll
          for (int e = 0; e < 8; e++) m.v[e] = uniform_value(m.v[e] * scale);
        }
        const uint32_t sel = bit == ~0u ? 0u : (kRare && cm != 0 ? 16u : 1u) << bit;
        dispatch_one<G, kRare>(a, opaque(sel), in_frame(m, x, z), tidx, rl, fx, cm);
        gate_applied = !advance;
        if (advance) {
          o++;
          cur = record(sp.ops, o);
          word = words[o];
        }
      }
      if (pending) flip_slots<G>(a, sgn);
    }
    // Terminal draw as in k_trajectories, over the physical index: the
    // probabilities go to LDS (one slot of padding per 16), each thread owns
    // a contiguous segment.
    const uint32_t fx = carry & 0x3FFFu;
    if (active) {
#pragma unroll
      for (int r = 0; r < N; r++) {
        uint32_t i = tidx ^ fx;
#pragma unroll
        for (int g = 0; g < G; g++)
          if (r & (1 << g)) i ^= rl[g];
        buf[i + (i >> 4)] = a[r].x * a[r].x + a[r].y * a[r].y;
      }
    }
    __syncthreads();
    double part = 0.0;
    uint32_t mine_last = 0;
    bool any = false;
    if (active) {
#pragma unroll
      for (int r = 0; r < N; r++) {
        const uint32_t i = tid * N + r;
        const double pr = buf[i + (i >> 4)];
        if (pr > 0.0) {
          part += pr;
          mine_last = i;
          any = true;
        }
      }
    }
    double incl = part;
    for (int d = 1; d < 64; d <<= 1) {
      const double y = __shfl_up(incl, d);
      if ((int)lane >= d) incl += y;
    }
    double excl = __shfl_up(incl, 1);
    if (lane == 0) excl = 0.0;
    if (lane == 63) scan[wave] = incl;
    if (any) atomicMax(&last_pos, (unsigned long long)mine_last);
    __syncthreads();
    double woff = 0.0, total = 0.0;
#pragma nounroll
    for (uint32_t w = 0; w < nw; w++) {
      if (w < wave) woff += scan[w];
      total += scan[w];
    }
    uint32_t draw = sp.n_chan;
    const double target = uniform(key, draw++) * total;
    double cum = woff + excl;
    if (active && cum <= target) {
      for (uint32_t r = 0; r < (uint32_t)N; r++) {
        const uint32_t i = tid * N + r;
        const double pr = buf[i + (i >> 4)];
        if (pr > 0.0) {
          cum += pr;
          if (target < cum) {
            atomicMin(&found, (unsigned long long)i);
            break;
          }
        }
      }
    }
    __syncthreads();
    if (tid == 0) {
      uint64_t idx = found != ~0ull ? (uint64_t)found : (uint64_t)last_pos;
#pragma nounroll
      for (uint32_t q = 0; q < n; q++) {
        if (!((p.readout_mask >> q) & 1ull)) continue;
        const uint32_t b = (uint32_t)((idx >> q) & 1ull);
        if (uniform(key, draw++) < p.readout[2 * q + b]) idx ^= 1ull << q;
      }
      out[shot] = idx;
    }
    __syncthreads();
  }
}

template <int G, bool kRare, int TH, int W>
void staged_launch(hipStream_t s, const TrajProgram& p, const StagedProgram& sp, uint64_t* out) {
  const uint32_t threads = std::max<uint32_t>(64u, 1u << (p.n - G));
  const size_t len = (size_t)1 << p.n;
  const size_t lds = (sp.n_ops + 1) * sizeof(uint64_t) +
                     std::max((len + len / 16) * sizeof(double), ((size_t)sp.n_chan + 1) * sizeof(uint32_t) + sp.n_chan);
  // 14 qubits and kStagedMaxOps records: 136 + 16 KiB of the CU's 160.
  allow_full_lds((const void*)k_staged<G, kRare, TH, W>, 158 * 1024);
  const uint32_t groups = std::max<uint32_t>(1u, std::min<uint32_t>(p.shots, 16384u));
  hipLaunchKernelGGL((k_staged<G, kRare, TH, W>), dim3(groups), dim3(threads), lds, s, p, sp, out);
  ALEPH_HIP_CHECK(hipGetLastError());
}

}  // namespace

void trajectory_geometry(uint32_t n, uint32_t shots, size_t budget, uint32_t* workgroups, size_t* bytes) {
  if (n <= kNoiseLdsMaxQubits) {
    *workgroups = std::max<uint32_t>(1u, std::min<uint32_t>(shots, 16384u));
    *bytes = 0;
    return;
  }
  const size_t slice = (size_t{1} << n) * sizeof(double2);
  const size_t fit = std::max<size_t>(1, budget / slice);
  *workgroups = (uint32_t)std::max<size_t>(1, std::min<size_t>({(size_t)shots, fit, 1024}));
  *bytes = (size_t)*workgroups * slice;
}

void launch_staged(hipStream_t s, const TrajProgram& p, const StagedProgram& sp, uint64_t* out) {
  if (p.shots == 0) return;
  // Amplitudes per thread follow staged_reg_bits; workgroups of up to 256 threads
  // (12 qubits) fit four to a CU, larger ones fill it alone.
  if (p.n <= 8) staged_launch<2, true, 64, 4>(s, p, sp, out);
  else if (p.n == 9) staged_launch<3, true, 64, 4>(s, p, sp, out);
  else if (p.n <= 12) sp.rare ? staged_launch<4, true, 256, 4>(s, p, sp, out) : staged_launch<4, false, 256, 4>(s, p, sp, out);
  else sp.rare ? staged_launch<4, true, 1024, 4>(s, p, sp, out) : staged_launch<4, false, 1024, 4>(s, p, sp, out);
}

void launch_trajectories(hipStream_t s, const TrajProgram& p, uint32_t workgroups, void* slices, uint64_t* out) {
  if (p.shots == 0) return;
  if (p.n <= kNoiseLdsMaxQubits) {
    const uint32_t threads = std::min<uint32_t>(kNoiseThreadsLds, std::max<uint32_t>(64u, (1u << p.n) / 2u));
    const size_t lds = ((size_t)1 << p.n) * sizeof(double2);
    // The largest state (13 qubits, 128 KiB) plus the kernel's static LDS fits the CU's 160 KiB.
    allow_full_lds((const void*)k_trajectories<true>, (int)((size_t{1} << kNoiseLdsMaxQubits) * sizeof(double2)));
    hipLaunchKernelGGL(k_trajectories<true>, dim3(workgroups), dim3(threads), lds, s, p, (double2*)nullptr, out);
  } else {
    hipLaunchKernelGGL(k_trajectories<false>, dim3(workgroups), dim3(kNoiseThreadsWide), 0, s, p, (double2*)slices,
                       out);
  }
  ALEPH_HIP_CHECK(hipGetLastError());
}

}  // namespace aleph
