// Pauli-string sums: sum_t c_t <psi|P_t|psi> and the state's norm in as few
// reads of the state as the strings' X masks allow.
//
// With z(i) = conj(psi[i ^ x]) psi[i] and s_t(i) = (-1)^{|i & zy_t|}, a string
// with X mask x contributes c_t Re(i^ny sum_i s_t(i) z(i)).  A workgroup takes
// chunks of 2^m amplitudes spanned by m chunk qubits (the others fixed by the
// chunk number), so every pair {i, i ^ x} with x inside the chunk qubits meets
// in one chunk: one sweep serves every string whose X mask fits, and the
// diagonal strings and the norm of the validity check ride on the first.
// Strings whose X mask does not fit any chunk keep k_expect_group.
//
// Per thread 16 amplitudes sit in registers.  All strings of a group (one X
// mask, Re or Im) share the 16 products w_r; a string's sign splits into a
// register part and a thread part, so the products go through one 16-point
// Walsh-Hadamard transform and each string costs one parity and one addition
// per thread, not per amplitude.  Groups whose strings touch no register
// qubit with Z (a transverse field) need the plain sum only.  Full chunks are
// read in up to three layouts (register bits 8..11 from memory, 4..7 and 0..3
// from the LDS copy): a plain-sum group whose X mask is one qubit runs in the
// layout that has it in a register bit, without LDS; the others take their
// partners from LDS (up to 16 reads of an amplitude per thread and group).
//
// The 26-qubit FP64 Ising chain (25 ZZ + 26 X) is 3 sweeps of 1.07 GB at 301 us
// each (3.6 TB/s of the 6.1 a plain read reaches; the scalar loads of the
// records and the per-group arithmetic, two waves per SIMD, hold it there:
// loading the next chunk ahead left it at 308 us).  The whole call, with the
// validity check, took 28 group reads and 7.6 ms before and takes 0.89 ms.
// Partners of one-qubit masks from LDS instead of the second and third layout:
// 483 us a sweep.
#include <algorithm>
#include <cmath>
#include <vector>

#include "common.hpp"
#include "kernels.hpp"
#include "pauli.hpp"

namespace aleph {
namespace {

constexpr uint32_t kRegs = 4;
constexpr uint32_t kSlots = 1u << kRegs;
constexpr uint32_t kChunkBits = 12;      // 64 KiB FP64, 32 KiB FP32: two and more workgroups per CU
constexpr uint32_t kMaxSweeps = 4096;    // bounds the search for a sweep that a string fits
constexpr uint32_t kRunBits = 4;         // chunks keep the 4 lowest qubits: runs of 16 amplitudes

struct alignas(16) PauliTermDev {
  uint64_t z_out;      // Z part outside the chunk qubits
  double c;
  uint32_t z_thread;   // Z part on thread bits (chunk-local)
  uint32_t pad[3];
};

struct alignas(16) PauliGroupDev {
  uint32_t x_thread;   // X mask on thread bits (chunk-local)
  uint32_t x_reg;      // X mask on register bits
  uint32_t half;       // lowest register bit of x_reg: slots with it set are the partners of the others
  uint32_t use_im;
  uint32_t flat;       // no string has Z on a register bit (the `half` bit aside)
  uint32_t in_reg;     // flat, and the X mask is one of the layout's register bits
  uint32_t bound[kSlots + 1];   // strings sorted by their register Z part
  uint32_t pad;
};
static_assert(sizeof(PauliGroupDev) % 16 == 0, "PauliGroupDev layout");

constexpr uint32_t kLayouts = kChunkBits / kRegs;

struct SweepArgs {
  uint32_t m;
  uint32_t group_end[kLayouts];   // groups of layout k end here (cumulative)
  uint32_t pos[kChunkBits];   // ascending chunk qubits
  uint32_t first;             // the call's first sweep: carries the norm and starts the rows of partial sums
};

__device__ __forceinline__ double signed_one(uint32_t parity) {
  return __builtin_bit_cast(double, ((uint64_t)(0x3FF00000u ^ (parity << 31))) << 32);
}

// Sum of the group's coefficients of strings [b, e), each with the sign of
// its thread and chunk part.
__device__ __forceinline__ double signed_coeffs(Prog<PauliTermDev>* terms, uint32_t b, uint32_t e, uint64_t base,
                                                uint32_t tl) {
  double acc = 0.0;
  for (uint32_t t = b; t < e; t++) {
    const uint32_t out = (uint32_t)__popcll(base & terms[t].z_out);
    acc += terms[t].c * signed_one(((uint32_t)__popc(tl & terms[t].z_thread) + out) & 1u);
  }
  return acc;
}

// LDS slot of chunk-local index li (linear over XOR): 16 consecutive lanes
// hit distinct 16-byte banks in all three layouts.
__device__ __forceinline__ uint32_t slot(uint32_t li) { return li ^ ((li >> 4) & 15u) ^ ((li >> 8) & 15u); }

// Sum over the slots with bit XR clear of Re or Im of conj(a[r ^ XR]) a[r],
// XR one register bit.  A row of ifs on a value the compiler knows nothing
// about: a chain of alternatives made it compute all of them side by side and
// spill.
template <typename T, uint32_t XR = 1>
__device__ __forceinline__ double pair_sum(const C2<T> (&a)[kSlots], uint32_t xr, uint32_t im) {
  double sum = 0.0;
  if constexpr (XR < kSlots) {
    if (__builtin_amdgcn_readfirstlane(xr) & XR) {
#pragma unroll
      for (uint32_t r = 0; r < kSlots; r++) {
        if (r & XR) continue;
        __builtin_amdgcn_sched_barrier(0);
        const double ar = a[r].x, ai = a[r].y, br = a[r | XR].x, bi = a[r | XR].y;
        sum += im ? br * ai - bi * ar : br * ar + bi * ai;
      }
    }
    sum += pair_sum<T, 2 * XR>(a, xr, im);
  }
  return sum;
}

template <typename T>
__global__ void __launch_bounds__(256, 2) k_pauli_sweep(const C2<T>* __restrict__ s, uint64_t n_chunks, SweepArgs d,
                                                        const PauliGroupDev* __restrict__ groups,
                                                        const PauliTermDev* __restrict__ terms,
                                                        double* __restrict__ partials) {
  extern __shared__ __align__(16) unsigned char smem[];
  C2<T>* const lds = reinterpret_cast<C2<T>*>(smem);
  __shared__ double red[3][4];
  const uint32_t tb = d.m - kRegs, T0 = 1u << tb, tid = threadIdx.x;
  const bool active = tid < T0;
  uint64_t toff = 0, rg[kRegs];
  for (uint32_t j = 0; j < tb; j++)
    if ((tid >> j) & 1u) toff |= 1ull << d.pos[j];
#pragma unroll
  for (uint32_t g = 0; g < kRegs; g++) rg[g] = 1ull << d.pos[tb + g];
  double acc = 0.0, norm = 0.0, bad = 0.0;
  for (uint64_t chunk = blockIdx.x; chunk < n_chunks; chunk += gridDim.x) {
    uint64_t base = chunk;
    for (uint32_t j = 0; j < d.m; j++) base = insert_zero(base, d.pos[j]);
    C2<T> a[kSlots];
    const C2<T>* const p = s + (base | toff);
#pragma unroll
    for (uint32_t r = 0; r < kSlots; r++) {
      uint64_t o = 0;
#pragma unroll
      for (uint32_t g = 0; g < kRegs; g++)
        if (r & (1u << g)) o |= rg[g];
      if (active) a[r] = p[o];
      else a[r].x = a[r].y = 0;
    }
    if (d.first) {
      double part = 0.0;
#pragma unroll
      for (uint32_t r = 0; r < kSlots; r++) part += (double)a[r].x * (double)a[r].x + (double)a[r].y * (double)a[r].y;
      norm += part;
      if (!isfinite(part)) {   // tell non-finite amplitudes from an overflow of the sum
#pragma unroll
        for (uint32_t r = 0; r < kSlots; r++)
          if (!isfinite((double)a[r].x * (double)a[r].x + (double)a[r].y * (double)a[r].y)) bad += 1.0;
      }
    }
    __syncthreads();           // the partners of the previous chunk have been read
    if (active) {
#pragma unroll
      for (uint32_t r = 0; r < kSlots; r++) lds[slot(tid) ^ slot(r << tb)] = a[r];
    }
    __syncthreads();
    uint32_t gi = 0, tl = tid;       // tl: chunk-local index of the thread in the current layout
#pragma nounroll
    for (uint32_t layout = 0; layout < kLayouts; layout++) {
      const uint32_t end = d.group_end[layout];
      if (gi == end) continue;
      if (layout) {                    // full chunks only: the register bits move down
        const uint32_t rb = tb - kRegs * layout;
        tl = (tid & ((1u << rb) - 1u)) | ((tid >> rb) << (rb + kRegs));
        const uint32_t ts = slot(tl);
#pragma unroll
        for (uint32_t r = 0; r < kSlots; r++) a[r] = lds[ts ^ slot(r << rb)];
      }
      for (; gi < end; gi++) {
        Prog<PauliGroupDev>& g = prog(groups)[gi];
        // Keeps the products of every kind of group from being hoisted out of
        // this loop (they are invariant, and together take 200 registers).
#pragma unroll
        for (uint32_t r = 0; r < kSlots; r++) asm volatile("" : "+v"(a[r].x), "+v"(a[r].y));
        if (g.in_reg) {
          acc += pair_sum<T>(a, g.x_reg, g.use_im) * signed_coeffs(prog(terms), g.bound[0], g.bound[1], base, tl);
          continue;
        }
        const uint32_t xt = g.x_thread, xr = g.x_reg, half = g.half, im = g.use_im;
        const bool diagonal = (xt | xr) == 0;
        double w[kSlots];
        const uint32_t q = active ? slot(tid ^ xt) : 0u;
#pragma unroll
        for (uint32_t r = 0; r < kSlots; r++) {
          w[r] = 0.0;
          if (r & half) continue;
          const double ar = a[r].x, ai = a[r].y;
          double br = ar, bi = ai;
          if (!diagonal) {
            const C2<T> b = lds[q ^ slot((r ^ xr) << tb)];
            br = b.x;
            bi = b.y;
          }
          w[r] = im ? br * ai - bi * ar : br * ar + bi * ai;
        }
        if (g.flat) {
          double sum = 0.0;
#pragma unroll
          for (uint32_t r = 0; r < kSlots; r++) sum += w[r];
          acc += sum * signed_coeffs(prog(terms), g.bound[0], g.bound[1], base, tid);
        } else {
#pragma unroll
          for (uint32_t h = 1; h < kSlots; h <<= 1) {
#pragma unroll
            for (uint32_t r = 0; r < kSlots; r++) {
              if (r & h) continue;
              const double u = w[r], v = w[r | h];
              w[r] = u + v;
              w[r | h] = u - v;
            }
          }
#pragma unroll
          for (uint32_t k = 0; k < kSlots; k++)
            if (g.bound[k] < g.bound[k + 1])
              acc += w[k] * signed_coeffs(prog(terms), g.bound[k], g.bound[k + 1], base, tid);
        }
      }
    }
  }
  if (!active) acc = 0.0;
  double v[3] = {acc, norm, bad};
#pragma unroll
  for (int k = 0; k < 3; k++) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v[k] += __shfl_down(v[k], off, 64);
    if ((tid & 63u) == 0) red[k][tid >> 6] = v[k];
  }
  __syncthreads();
  if (tid < 3) {
    double t = 0.0;
    for (uint32_t w = 0; w < (blockDim.x + 63u) / 64u; w++) t += red[tid][w];
    double* const row = partials + 3 * (uint64_t)blockIdx.x;
    row[tid] = d.first ? t : row[tid] + t;
  }
}

}  // namespace

PauliPlan plan_pauli_sum(const std::vector<PauliTerm>& terms, uint32_t n) {
  PauliPlan plan;
  std::vector<uint32_t> order(terms.size());
  for (uint32_t t = 0; t < order.size(); t++) order[t] = t;
  std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return terms[a].x < terms[b].x; });
  if (n < kRegs) {
    plan.rest = std::move(order);
    return plan;
  }
  const uint32_t m = std::min(n, kChunkBits), L = std::min(kRunBits, m);
  const uint64_t low = (1ull << L) - 1ull;
  plan.sweeps.push_back(PauliSweep{low, {}});
  size_t k = 0;
  uint64_t last = 0;
  for (uint32_t t : order) {
    const uint64_t x = terms[t].x;
    if ((uint32_t)__builtin_popcountll(low | x) > m) {
      plan.rest.push_back(t);
      continue;
    }
    if (x != last) k = 0;      // strings with one X mask follow each other and share a sweep
    last = x;
    while (k < plan.sweeps.size() && (uint32_t)__builtin_popcountll(plan.sweeps[k].qubits | x) > m) k++;
    if (k == kMaxSweeps) {
      plan.rest.push_back(t);
      continue;
    }
    if (k == plan.sweeps.size()) plan.sweeps.push_back(PauliSweep{low, {}});
    plan.sweeps[k].qubits |= x;
    plan.sweeps[k].terms.push_back(t);
  }
  for (PauliSweep& s : plan.sweeps)
    for (uint32_t q = 0; q < n && (uint32_t)__builtin_popcountll(s.qubits) < m; q++) s.qubits |= 1ull << q;
  return plan;
}

// Device records of one sweep; coefficients are scaled by 2^-shift.
static void sweep_records(const PauliSweep& sw, const std::vector<PauliTerm>& terms, uint32_t n, int shift,
                          SweepArgs& d, std::vector<PauliGroupDev>& groups, std::vector<PauliTermDev>& out) {
  d = SweepArgs{};
  for (uint32_t q = 0; q < n; q++)
    if ((sw.qubits >> q) & 1ull) d.pos[d.m++] = q;
  const uint32_t tb = d.m - kRegs;
  auto local = [&](uint64_t mask) {
    uint32_t l = 0;
    for (uint32_t j = 0; j < d.m; j++)
      if ((mask >> d.pos[j]) & 1ull) l |= 1u << j;
    return l;
  };
  // Layout of an X mask: of one bit, the one that has it in a register bit; else layout 0.
  const uint32_t layouts = d.m == kChunkBits ? kLayouts : 1u;
  struct Item {
    uint64_t x;
    uint32_t layout, im, zr, id;
  };
  std::vector<Item> items;
  for (uint32_t t : sw.terms) {
    const uint32_t xl = local(terms[t].x);
    uint32_t lay = 0;
    for (uint32_t k = 0; k < layouts; k++)
      if (__builtin_popcount(xl) == 1 && (xl & ((kSlots - 1u) << (tb - kRegs * k)))) lay = k;
    const uint32_t xr = (xl >> (tb - kRegs * lay)) & (kSlots - 1u);
    // Slots with the half bit set are never evaluated: Z there has no effect.
    const uint32_t zr = (local(terms[t].zy) >> (tb - kRegs * lay)) & (kSlots - 1u) & ~(xr & (0u - xr));
    if (lay && zr) lay = 0;          // the other layouts run plain sums only
    items.push_back(Item{terms[t].x, lay, (uint32_t)(terms[t].ny & 1), 0u, t});
  }
  for (Item& it : items) {
    const uint32_t rb = tb - kRegs * it.layout, xr = (local(it.x) >> rb) & (kSlots - 1u);
    it.zr = (local(terms[it.id].zy) >> rb) & (kSlots - 1u) & ~(xr & (0u - xr));
  }
  std::stable_sort(items.begin(), items.end(), [](const Item& a, const Item& b) {
    if (a.layout != b.layout) return a.layout < b.layout;
    if (a.x != b.x) return a.x < b.x;
    if (a.im != b.im) return a.im < b.im;
    return a.zr < b.zr;
  });
  const uint32_t g0 = (uint32_t)groups.size();
  auto same = [](const Item& a, const Item& b) { return a.layout == b.layout && a.x == b.x && a.im == b.im; };
  for (size_t i = 0; i < items.size();) {
    size_t j = i;
    PauliGroupDev g{};
    const uint32_t rb = tb - kRegs * items[i].layout, regs = (kSlots - 1u) << rb;
    const uint32_t xl = local(items[i].x), t0 = (uint32_t)out.size();
    g.x_thread = xl & ~regs;
    g.x_reg = (xl & regs) >> rb;
    g.half = g.x_reg & (0u - g.x_reg);
    g.use_im = items[i].im;
    g.flat = 1;
    for (; j < items.size() && same(items[i], items[j]); j++) {
      const PauliTerm& t = terms[items[j].id];
      PauliTermDev td{};
      td.z_out = t.zy & ~sw.qubits;
      td.z_thread = local(t.zy) & ~regs;
      // Re(i^ny (re + i im)): +re, -im, -re, +im; each pair counted once when
      // a register bit picks its half.
      td.c = std::ldexp(((t.ny & 3) == 1 || (t.ny & 3) == 2) ? -t.coeff : t.coeff, -shift);
      if (g.half) td.c *= 2.0;
      if (items[j].zr) g.flat = 0;
      out.push_back(td);
    }
    g.in_reg = g.flat && !g.x_thread && __builtin_popcount(g.x_reg) == 1;
    uint32_t at = (uint32_t)i;
    for (uint32_t k = 0; k <= kSlots; k++) {
      while (at < j && items[at].zr < k) at++;
      g.bound[k] = t0 + (at - (uint32_t)i);
    }
    groups.push_back(g);
    for (uint32_t k = items[i].layout; k < kLayouts; k++) d.group_end[k] = (uint32_t)groups.size() - g0;
    i = j;
  }
}

template <typename T>
void run_pauli_sweeps(hipStream_t st, const void* state, uint32_t n, const PauliPlan& plan,
                      const std::vector<PauliTerm>& terms, void* dev, size_t dev_bytes, double* partials,
                      double* result) {
  const uint64_t len = 1ull << n;
  std::vector<SweepArgs> args(plan.sweeps.size());
  std::vector<PauliGroupDev> groups;
  std::vector<PauliTermDev> recs;
  std::vector<uint32_t> first(plan.sweeps.size());
  // The kernel adds coefficients, twice those of pairs, before it multiplies:
  // very large ones are scaled down (exactly) so that only a sum that is
  // itself out of range overflows.
  double largest = 0.0;
  for (const PauliTerm& t : terms) largest = std::max(largest, std::fabs(t.coeff));
  const int shift = largest > std::ldexp(1.0, 960) ? 128 : 0;
  for (size_t k = 0; k < plan.sweeps.size(); k++) {
    first[k] = (uint32_t)groups.size();
    sweep_records(plan.sweeps[k], terms, n, shift, args[k], groups, recs);
    args[k].first = k == 0;
  }
  const size_t gb = groups.size() * sizeof(PauliGroupDev), tb = recs.size() * sizeof(PauliTermDev);
  std::vector<unsigned char> host(gb + tb);
  if (gb) std::memcpy(host.data(), groups.data(), gb);
  if (tb) std::memcpy(host.data() + gb, recs.data(), tb);
  struct Own {
    void* p = nullptr;
    ~Own() {
      if (p) (void)hipFree(p);
    }
  } own;
  if (host.size() > dev_bytes) {
    ALEPH_HIP_CHECK(hipMalloc(&own.p, host.size()));
    dev = own.p;
  }
  if (!host.empty()) ALEPH_HIP_CHECK(hipMemcpyAsync(dev, host.data(), host.size(), hipMemcpyHostToDevice, st));
  const PauliGroupDev* dg = reinterpret_cast<const PauliGroupDev*>(dev);
  const PauliTermDev* dt = reinterpret_cast<const PauliTermDev*>((const unsigned char*)dev + gb);
  allow_full_lds(reinterpret_cast<const void*>(&k_pauli_sweep<T>), 96 * 1024);
  // Every sweep has the same number of chunks and adds its sums to the same
  // rows of partials, so each gets a full grid however many there are: 1000
  // random strings on two to eight of 24 qubits are 120 sweeps and take 143 ms
  // with the rows divided between them (34 workgroups each), 13.8 ms now (89 ms as group
  // reads); 200 strings on four of 26 qubits 29.2 -> 10.8 ms (group reads 48.3).
  uint32_t rows = 0;
  for (size_t k = 0; k < plan.sweeps.size(); k++) {
    const uint64_t chunks = len >> args[k].m;
    const uint32_t threads = std::max<uint32_t>(64u, 1u << (args[k].m - kRegs));
    rows = (uint32_t)std::min<uint64_t>(chunks, kPauliRows);
    hipLaunchKernelGGL(k_pauli_sweep<T>, dim3(rows), dim3(threads), sizeof(C2<T>) << args[k].m, st,
                       (const C2<T>*)state, chunks, args[k], dg + first[k], dt, partials);
  }
  ALEPH_HIP_CHECK(hipGetLastError());
  launch_reduce_rows(st, partials, rows, result);
  ALEPH_HIP_CHECK(hipStreamSynchronize(st));   // before `host` and an own buffer go
  result[0] = std::ldexp(result[0], shift);
}

template void run_pauli_sweeps<double>(hipStream_t, const void*, uint32_t, const PauliPlan&,
                                       const std::vector<PauliTerm>&, void*, size_t, double*, double*);
template void run_pauli_sweeps<float>(hipStream_t, const void*, uint32_t, const PauliPlan&,
                                      const std::vector<PauliTerm>&, void*, size_t, double*, double*);

}  // namespace aleph
