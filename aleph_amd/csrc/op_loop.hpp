// The fused pass as an op loop: the kernel body of plans without generated
// kernels (k_fused.hip) and of the batched executors (k_batch.hip).
//
// One chunk of 2^m amplitudes (the index bits outside the pass's chunk
// qubits fixed by the chunk number) is read from HBM once, every op of the
// pass is applied to registers (2^G amplitudes per thread), the chunk is
// re-distributed through LDS between stages and written back once.
//
// Bound by vector issue and by how much latency its waves hide, so it is
// written for few vector registers (92 to 128 in FP64 with 4x4 or phase ops,
// 144 with both; 60 to 117 in FP32; none spilled), and a workgroup with its
// SIMDs to itself by the scalar loads of the ops:
//  - the loop body is a row of plain ifs on selector words the compiler knows
//    nothing about, behind one if per kind of op, and the operators change the
//    amplitudes in place (one asm block per pair or quartet): with a chain of
//    alternatives in C++ it moved all amplitudes to new registers at every
//    join and took 250 registers;
//  - descriptors and matrices come through the constant address space, so
//    they are scalar loads and the matrices SGPR operands; every op's cache
//    lines are read ahead, and no more lines than it uses (the misses of the
//    scalar cache are served one after the other: all five lines of every op
//    made small passes a quarter slower);
//  - nothing is kept across ops but the amplitudes and the thread's index: the
//    slots' indices alone took 32 registers;
//  - FP64 stages exchange real and imaginary parts in turn through 2^m
//    doubles (32 KiB at m = 12), half of what whole amplitudes need;
//  - a phase op forms one class factor at a time.
// MI355X, a pass list run 20 times, against the C++ chains: FP64 QFT of 24
// qubits 23.7 -> 13.1 ms, CX-ladder ansatz of 22 qubits 7.2 -> 5.2 ms and of
// 10 qubits (one workgroup) 0.75 ms both; FP32 24-qubit QFT 18.8 -> 10.0 ms,
// brickwall of 10 qubits 0.63 -> 0.60 ms.
#pragma once

#include "common.hpp"
#include "fused_chunk.hpp"
#include "inplace.hpp"

namespace aleph {
namespace fused {

// Waves per SIMD the op loop is compiled for.
template <typename T, int G>
struct OpLoopWaves {
  static constexpr int kWaves = G > 4 ? 2 : sizeof(T) == 8 ? 3 : 4;
};

template <typename T, int G, int B, bool CTL>
__device__ __forceinline__ void loop_1q(C2<T> (&a)[1 << G], const T (&m)[8], uint64_t tgo, const uint64_t (&rg)[G],
                                        uint64_t cm) {
#pragma unroll
  for (int r = 0; r < (1 << G); r++) {
    if (r & (1 << B)) continue;
    if (CTL && ((tgo | roff<G>(rg, r)) & cm) != cm) continue;
    pair_update(a[r], a[r | (1 << B)], m);
  }
}

// Rows 0 and 1 (m: 16 entries) of quartet Q and up into p.
template <typename T, int G, int A, int B, int Q = 0>
__device__ __forceinline__ void upper_rows(C2<T> (&a)[1 << G], C2<T> (&p)[1 << (G - 1)], const T* m) {
  if constexpr (Q < (1 << (G - 2))) {
    constexpr int r = ins0(ins0(Q, B), A);
    two_rows<true>(a[r], a[r | (1 << B)], p[2 * Q], p[2 * Q + 1], m);
    two_rows<false>(a[r | (1 << A)], a[r | (1 << A) | (1 << B)], p[2 * Q], p[2 * Q + 1], m + 4);
    upper_rows<T, G, A, B, Q + 1>(a, p, m);
  }
}

// Rows 2 and 3 of quartet Q and up, and the quartet's results into place.
template <typename T, int G, int A, int B, bool CTL, int Q = 0>
__device__ __forceinline__ void lower_rows(C2<T> (&a)[1 << G], const C2<T> (&p)[1 << (G - 1)], const T* m,
                                           uint64_t tgo, const uint64_t (&rg)[G], uint64_t cm) {
  if constexpr (Q < (1 << (G - 2))) {
    constexpr int r = ins0(ins0(Q, B), A), r1 = r | (1 << B), r2 = r | (1 << A), r3 = r1 | r2;
    C2<T> p2, p3;
    two_rows<true>(a[r], a[r1], p2, p3, m);
    two_rows<false>(a[r2], a[r3], p2, p3, m + 4);
    if (!CTL || ((tgo | roff<G>(rg, r)) & cm) == cm) {
      put(a[r], p[2 * Q]);
      put(a[r1], p[2 * Q + 1]);
      put(a[r2], p2);
      put(a[r3], p3);
    }
    lower_rows<T, G, A, B, CTL, Q + 1>(a, p, m, tgo, rg, cm);
  }
}

// A = matrix MSB register bit, B = LSB, A > B.  The matrix is used a half at
// a time (32 SGPRs in FP64): rows 0 and 1 of every quartet, whose results
// wait in temporaries, then rows 2 and 3.
template <typename T, int G, int A, int B, bool CTL>
__device__ __forceinline__ void loop_2q(C2<T> (&a)[1 << G], const T* upper, Prog<T>* mm, uint64_t tgo,
                                        const uint64_t (&rg)[G], uint64_t cm) {
  C2<T> p[1 << (G - 1)];
  upper_rows<T, G, A, B>(a, p, upper);
  asm volatile("" : "+s"(mm));      // the second half takes the scalar registers of the first
  T lower[16];
#pragma unroll
  for (int e = 0; e < 16; e++) lower[e] = mm[16 + e];
  lower_rows<T, G, A, B, CTL>(a, p, lower, tgo, rg, cm);
}

// Selector words: 1q op on register bit B: bit B, controlled bit 8 + B;
// 2q op on bits A > B: bit A (A - 1) / 2 + B, controlled 16 above.
template <typename T, int G, bool CTL, int B = 0>
__device__ __forceinline__ void select_1q(C2<T> (&a)[1 << G], uint32_t sel, const T (&m)[8], uint64_t tgo,
                                          const uint64_t (&rg)[G], uint64_t cm) {
  if constexpr (B < G) {
    if (sel & (1u << B)) loop_1q<T, G, B, CTL>(a, m, tgo, rg, cm);
    select_1q<T, G, CTL, B + 1>(a, sel, m, tgo, rg, cm);
  }
}

template <typename T, int G, bool CTL, int A = 1, int B = 0>
__device__ __forceinline__ void select_2q(C2<T> (&a)[1 << G], uint32_t sel, const T* upper, Prog<T>* mm, uint64_t tgo,
                                          const uint64_t (&rg)[G], uint64_t cm) {
  if constexpr (A < G) {
    if constexpr (B < A) {
      if (sel & (1u << (A * (A - 1) / 2 + B))) loop_2q<T, G, A, B, CTL>(a, upper, mm, tgo, rg, cm);
      select_2q<T, G, CTL, A, B + 1>(a, sel, upper, mm, tgo, rg, cm);
    } else {
      select_2q<T, G, CTL, A + 1, 0>(a, sel, upper, mm, tgo, rg, cm);
    }
  }
}

// Multiply class K's factor into the slots it selects: class 0 every slot,
// linear classes the slots with that register bit, pair classes those with both.
template <typename T, int G, int K = 0>
__device__ __forceinline__ void select_class(C2<T> (&a)[1 << G], uint32_t sel, T fr, T fi) {
  if constexpr (K < PhaseSlots<G>::kCount) {
    if (sel & (1u << K)) {
#pragma unroll
      for (int r = 0; r < (1 << G); r++) {
        bool in = K == 0;
#pragma unroll
        for (int g = 0; g < G; g++) {
          if (K == PhaseSlots<G>::linear(g) && ((r >> g) & 1)) in = true;
#pragma unroll
          for (int h = g + 1; h < G; h++)
            if (K == PhaseSlots<G>::pair(g, h) && ((r >> g) & 1) && ((r >> h) & 1)) in = true;
        }
        if (in) rotate(a[r], fr, fi);
      }
    }
    select_class<T, G, K + 1>(a, sel, fr, fi);
  }
}

// Angle of class [b, e) of a phase op for this thread, summed in FP64.
__device__ __forceinline__ double class_angle(Prog<PhaseTerm>* terms, uint32_t b, uint32_t e, uint64_t tgo) {
  double phi = 0.0;
#pragma unroll 4
  for (uint32_t t = b; t < e; t++) {
    const uint64_t mo = terms[t].mask_out;
    phi += ((tgo & mo) == mo) ? terms[t].angle : 0.0;
  }
  return phi;
}

// psi *= e^{i phi} on FP64 amplitudes: one factor per non-empty class (FP64
// angle sum, one sincos as for a state of type T), then the terms on three and
// more register bits with their own unit factors.
template <typename T, int G>
__device__ __forceinline__ void rotate_classes(C2<double> (&a)[1 << G], Prog<DevOp>* op, Prog<PhaseTerm>* terms,
                                               uint64_t tgo) {
  const Prog<uint32_t>* bounds = (const Prog<uint32_t>*)op->m;
  const uint32_t t0 = op->term_off;
#pragma nounroll
  for (uint32_t left = op->a; left; left &= left - 1) {
    const uint32_t k = (uint32_t)__builtin_ctz(left);
    double s, c;
    phase_sincos<T>(class_angle(terms, t0 + bounds[k], t0 + bounds[k + 1], tgo), &s, &c);
    select_class<double, G>(a, opaque(1u << k), c, s);
  }
  const uint32_t g0 = t0 + op->n_terms, g1 = g0 + op->b;
#pragma nounroll
  for (uint32_t t = g0; t < g1; t++) {
    const uint64_t mo = terms[t].mask_out;
    const uint32_t rm = opaque(terms[t].rmask);
    const bool on = (tgo & mo) == mo;
    const double c = on ? terms[t].c : 1.0, s = on ? terms[t].s : 0.0;
#pragma unroll
    for (int r = 0; r < (1 << G); r++)
      if (((uint32_t)r & rm) == rm) rotate(a[r], c, s);
  }
}

// FP32 amplitudes are rotated in FP64 and rounded once, at the end of the op:
// a rotation in FP32 per factor rounds an amplitude up to eleven times an op,
// and once more per term on three and more register bits (1.29e-7 RMS an op
// with all classes filled, against 1.17e-7 for one rotation by the product).
// An FP64 multiply-add takes no longer than an unpacked FP32 one.
template <typename T, int G>
__device__ __forceinline__ void loop_phase(C2<T> (&a)[1 << G], Prog<DevOp>* op, Prog<PhaseTerm>* terms, uint64_t tgo) {
  if constexpr (sizeof(T) == 8) {
    rotate_classes<T, G>(a, op, terms, tgo);
  } else {
    C2<double> d[1 << G];
#pragma unroll
    for (int r = 0; r < (1 << G); r++) d[r] = C2<double>{a[r].x, a[r].y};
    rotate_classes<T, G>(d, op, terms, tgo);
#pragma unroll
    for (int r = 0; r < (1 << G); r++) a[r] = C2<float>{(float)d[r].x, (float)d[r].y};
  }
}

// A phase op in CutPhase form: the integer K of each amplitude from parities
// and popcounts, its factor from the op's table in LDS, whose entries the
// threads form here (one sincos a thread and op, where a class factor each
// takes up to 11).  Three MaxCut layers run 20 times, against the same with
// unequal weights (one sincos per class and a pass over the terms per thread):
// 20 qubits FP64 3.03 -> 2.36 ms, 24 qubits FP32 14.3 -> 12.7 ms.
template <typename T>
__device__ __forceinline__ void loop_cut(C2<T> (&a)[16], Prog<CutPhase>* c, uint64_t tgo, C2<T>* table) {
  const uint32_t x = (uint32_t)tgo, size = c->size;
  __syncthreads();                         // the previous op's table has been read
  for (uint32_t i = threadIdx.x; i < size; i += blockDim.x) {
    double sn, cs;
    phase_sincos<T>(fma(c->theta, (double)(c->k_min + (int32_t)i), c->phi0), &sn, &cs);
    table[i].x = (T)cs;
    table[i].y = (T)sn;
  }
  int32_t pairs = 0;
  const uint32_t n = c->n;
#pragma unroll 4
  for (uint32_t u = 0; u < n; u++) pairs += (int32_t)(__popc(x & c->below[u]) & (0u - ((x >> u) & 1u)));
  const int32_t pk = c->pair;
  int32_t k0 = pk * pairs - c->k_min + (int32_t)(__popc(x & c->linear[0]) + 2 * __popc(x & c->linear[1]) +
                                                4 * __popc(x & c->linear[2]));
  int32_t lin[4];
#pragma unroll
  for (int g = 0; g < 4; g++) lin[g] = c->reg_linear[g] + pk * (int32_t)__popc(x & c->reg_adj[g]);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 16; r++) {
    int32_t k = k0 + c->slot[r];
#pragma unroll
    for (int g = 0; g < 4; g++)
      if (r & (1 << g)) k += lin[g];
    const C2<T> f = table[k];
    rotate(a[r], f.x, f.y);
  }
}

template <typename T, int G>
__device__ __forceinline__ void loop_diag(C2<T> (&a)[1 << G], Prog<DevOp>* op, uint64_t tgo, const uint64_t (&rg)[G]) {
  const uint64_t ma = op->ma, mb = op->mb, cm = op->cmask;
  Prog<T>* d = (Prog<T>*)op->m;
#pragma unroll
  for (int r = 0; r < (1 << G); r++) {
    const uint64_t idx = tgo | roff<G>(rg, r);
    const bool hi = (idx & ma) != 0, lo = (idx & mb) != 0, on = (idx & cm) == cm;
    const T dr = hi ? (lo ? d[6] : d[4]) : (lo ? d[2] : d[0]);
    const T di = hi ? (lo ? d[7] : d[5]) : (lo ? d[3] : d[1]);
    rotate(a[r], on ? dr : (T)1, on ? di : (T)0);
  }
}

// Process chunk `chunk` of pass `pd` on `state`.  With GUARD, threads with
// tid >= 2^(m - G) hold no amplitudes but take part in every barrier, so a
// workgroup sized for the largest chunk can run smaller passes; without it
// the workgroup has exactly 2^(m - G) threads, or is one wavefront whose spare
// lanes repeat the others' work.  `lds` holds 2^m scalars of 8 bytes: the
// real, then the imaginary parts of FP64 amplitudes, whole FP32 ones.
template <typename T, int G, int FEAT, bool NT, bool GUARD>
__device__ __forceinline__ void fused_chunk(C2<T>* __restrict__ state, const PassDev* __restrict__ pass,
                                            const StageDev* __restrict__ stage_list, const DevOp* __restrict__ op_list,
                                            const PhaseTerm* __restrict__ term_list, uint64_t chunk,
                                            unsigned char* __restrict__ lds) {
  constexpr int SW = sizeof(T) == 8 ? 3 : 4;
  constexpr int N = 1 << G;
  using V = typename std::conditional<sizeof(T) == 8, v2f64, v2f32>::type;
  Prog<PassDev>* const pd = prog(pass);
  Prog<DevOp>* const ops = prog(op_list);
  Prog<PhaseTerm>* const terms = prog(term_list);
  const uint32_t m = pd->m, ns = pd->n_stages, tid = threadIdx.x;
  Prog<StageDev>* const stages = prog(stage_list) + pd->stage_begin;
  const uint32_t last_op = stages[ns - 1].op_end;
  uint32_t lines = pd->first_lines;
  uint64_t base = chunk;
  for (uint32_t i = 0; i < m; i++) base = insert_zero(base, pd->local_pos[i]);
  const bool active = !GUARD || tid < (1u << (m - G));
  C2<T> a[N];
#pragma unroll
  for (int r = 0; r < N; r++) a[r].x = a[r].y = 0;
  uint64_t tgo = 0;
  uint32_t slot = 0;       // byte offset of the thread's part in LDS
  for (uint32_t s = 0; s < ns; s++) {
    Prog<StageDev>* const sd = stages + s;
    const uint32_t ntb = sd->n_thread_bits, from = slot;
    uint32_t tlo = 0;
    tgo = base;
    for (uint32_t j = 0; j < ntb; j++) {
      if ((tid >> j) & 1u) {
        tgo |= sd->tg[j];
        tlo |= sd->tl[j];
      }
    }
    slot = swz<SW>(tlo) * 8u;
    uint64_t rg[G];
#pragma unroll
    for (int g = 0; g < G; g++) rg[g] = sd->rg[g];
    if (s == 0) {
      if (active) {
        const C2<T>* const tp = state + tgo;
#pragma unroll
        for (int r = 0; r < N; r++) {
          const V v = gload<NT>(reinterpret_cast<const V*>(tp + sd->go[r]));
          a[r].x = v.x;
          a[r].y = v.y;
        }
      }
    } else {
      // Thread and register bits are disjoint and the swizzle is linear over
      // XOR: an element's byte offset is the thread's XOR the slot's (lb).
      Prog<StageDev>* const pv = sd - 1;
      if (s > 1) __syncthreads();      // the previous exchange has been read
      if constexpr (sizeof(T) == 8) {
        uint32_t w = from, g = slot;
        if (active) {
#pragma unroll
          for (int r = 0; r < N; r++) *reinterpret_cast<T*>(lds + (w ^ pv->lb[r])) = a[r].x;
        }
        __syncthreads();
        if (active) {
#pragma unroll
          for (int r = 0; r < N; r++) a[r].x = *reinterpret_cast<const T*>(lds + (g ^ sd->lb[r]));
        }
        __syncthreads();
        // Opaque: the addresses are formed again instead of kept.
        asm volatile("" : "+v"(w), "+v"(g));
        if (active) {
#pragma unroll
          for (int r = 0; r < N; r++) *reinterpret_cast<T*>(lds + (w ^ pv->lb[r])) = a[r].y;
        }
        __syncthreads();
        if (active) {
#pragma unroll
          for (int r = 0; r < N; r++) a[r].y = *reinterpret_cast<const T*>(lds + (g ^ sd->lb[r]));
        }
      } else {
        if (active) {
#pragma unroll
          for (int r = 0; r < N; r++) *reinterpret_cast<V*>(lds + (from ^ pv->lb[r])) = V{a[r].x, a[r].y};
        }
        __syncthreads();
        if (active) {
#pragma unroll
          for (int r = 0; r < N; r++) {
            const V v = *reinterpret_cast<const V*>(lds + (slot ^ sd->lb[r]));
            a[r].x = v.x;
            a[r].y = v.y;
          }
        }
      }
    }
    const uint32_t end = sd->op_end;
    for (uint32_t o = sd->op_begin; o < end; o++) {
      // Opaque: the slots' indices (tgo with the register bits) are formed
      // where a controlled or diagonal op needs them; hoisted out of the loop
      // they took 32 vector or scalar registers and spilled others.
      asm volatile("" : "+v"(tgo));
#pragma unroll
      for (int g = 0; g < G; g++) asm volatile("" : "+s"(rg[g]));
      Prog<DevOp>* const op = ops + o;
      const uint32_t type = op->type, ra = op->a, rb = op->b;
      const uint64_t cm = op->cmask;
      // The first line of the matrix slots (FP64) or the first half of an FP32
      // 4x4 is read with the header, one memory latency for both; an op
      // without a matrix reads its header in that place.
      constexpr int H = (FEAT & kFeat2Q) != 0 && sizeof(T) == 4 ? 16 : 8;
      Prog<T>* const mm = (Prog<T>*)op->m;
      Prog<T>* const m0 = lines > 1 ? mm : (Prog<T>*)op;
      T head[H], one[8];
#pragma unroll
      for (int e = 0; e < H; e++) head[e] = m0[e];
      // Then one word of each line of the next op (the pass's last op reads
      // its own again): a workgroup with a SIMD to itself otherwise waits on
      // memory for every op's header and matrix.  The asm keeps these loads
      // behind the wait for the header and the matrix.
      lines = op->next_lines;
      Prog<uint32_t>* ahead = (Prog<uint32_t>*)(ops + (o + 1 < last_op ? o + 1 : o));
      asm volatile("" : "+s"(ahead) : "s"(head[0]), "s"(head[H - 1]), "s"(type), "s"(lines));
      constexpr uint32_t kLines = sizeof(DevOp) / 64;
      uint32_t touched[kLines];
#pragma unroll
      for (uint32_t e = 0; e < kLines; e++) touched[e] = ahead[16 * (e < lines ? e : 0u)];
#pragma unroll
      for (int e = 0; e < 8; e++) one[e] = head[e];
      const uint32_t s1 = opaque(type == OP_1Q ? (cm ? 256u : 1u) << ra : 0u);
      if (s1) {
        select_1q<T, G, false>(a, s1, one, tgo, rg, cm);
        if (s1 >> 8) select_1q<T, G, true>(a, s1 >> 8, one, tgo, rg, cm);
      }
      if constexpr ((FEAT & kFeat2Q) != 0) {
        const uint32_t s2 = opaque(type == OP_2Q ? (cm ? 65536u : 1u) << (ra * (ra - 1) / 2 + rb) : 0u);
        if (s2) {
          T upper[16];
#pragma unroll
          for (int e = 0; e < 16; e++) upper[e] = e < H ? head[e] : mm[e];
          select_2q<T, G, false>(a, s2, upper, mm, tgo, rg, cm);
          if (s2 >> 16) select_2q<T, G, true>(a, s2 >> 16, upper, mm, tgo, rg, cm);
        }
      }
      if (opaque(type != OP_1Q && type != OP_2Q ? 1u : 0u)) {
        if (opaque(type) == OP_SIGN) {
          // Sign-bit XOR with (thread condition) & (uniform slot condition).
          const uint32_t tm = ((tgo & cm) == cm) ? ~0u : 0u;
#pragma unroll
          for (int r = 0; r < N; r++) {
            const uint32_t sr = (((uint32_t)r & ra) == ra) ? 0x80000000u : 0u;
            a[r].x = flip_sign(a[r].x, sr, tm);
            a[r].y = flip_sign(a[r].y, sr, tm);
          }
        }
        if (opaque(type) == OP_DIAG) loop_diag<T, G>(a, op, tgo, rg);
        if constexpr ((FEAT & kFeatPhase) != 0) {
          const uint32_t cut = type == OP_PHASE ? op->cut : 0u;
          if (G == 4 && opaque(cut)) {
            __shared__ C2<T> table[kCutTable];
            loop_cut<T>(reinterpret_cast<C2<T>(&)[16]>(a), prog(reinterpret_cast<const CutPhase*>(term_list + cut - 1)),
                        tgo, table);
          }
          if (opaque(type == OP_PHASE && !(G == 4 && cut) ? 1u : 0u)) loop_phase<T, G>(a, op, terms, tgo);
        }
      }
#pragma unroll
      for (uint32_t e = 0; e < kLines; e++) asm volatile("" : : "s"(touched[e]));
    }
  }
  if (active) {
    Prog<StageDev>* const sd = stages + (ns - 1);
    C2<T>* const tp = state + tgo;
#pragma unroll
    for (int r = 0; r < N; r++) {
      V v;
      v.x = a[r].x;
      v.y = a[r].y;
      gstore<NT>(reinterpret_cast<V*>(tp + sd->go[r]), v);
    }
  }
}

}  // namespace fused
}  // namespace aleph
