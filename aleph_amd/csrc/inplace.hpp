// Operators that change amplitudes in their own registers, for kernels whose
// amplitudes live across a loop over operators (op_loop.hpp, k_noise.hip).
//
// One asm block per pair or quartet: with the 2x2 in C++ the compiler puts
// every result into a new register and copies all amplitudes back where the
// branches around the operator join (in k_noise.hip 250 moves a record beside
// 128 multiply-adds).
#pragma once

#include "common.hpp"
#include "device_types.hpp"

namespace aleph {
namespace fused {

// A uniform value the compiler knows nothing about.
__device__ __forceinline__ uint32_t opaque(uint32_t v) { return __builtin_amdgcn_readfirstlane(v); }

// In-place operators.  s_nop: a matrix entry may have been written to its
// SGPR by a vector instruction (a reloaded spill), which needs two wait
// states before a vector read; every block with matrix operands starts with it.
#define ALEPH_ROWS_TAIL(FMA)                                                                                         \
  FMA " %[pr], -%[b], %[xi], %[pr]\n" FMA " %[pi], %[b], %[xr], %[pi]\n" FMA " %[qr], -%[f], %[xi], %[qr]\n" FMA      \
      " %[qi], %[f], %[xr], %[qi]\n" FMA " %[pr], %[c], %[yr], %[pr]\n" FMA " %[pi], %[c], %[yi], %[pi]\n" FMA        \
      " %[qr], %[g], %[yr], %[qr]\n" FMA " %[qi], %[g], %[yi], %[qi]\n" FMA " %[pr], -%[d], %[yi], %[pr]\n" FMA       \
      " %[pi], %[d], %[yr], %[pi]\n" FMA " %[qr], -%[h], %[yi], %[qr]\n" FMA " %[qi], %[h], %[yr], %[qi]\n"
#define ALEPH_ROWS_IN(v0, v1, m)                                                                                     \
  [xr] "v"((v0).x), [xi] "v"((v0).y), [yr] "v"((v1).x), [yi] "v"((v1).y), [a] "s"((m)[0]), [b] "s"((m)[1]),          \
      [c] "s"((m)[2]), [d] "s"((m)[3]), [e] "s"((m)[8]), [f] "s"((m)[9]), [g] "s"((m)[10]), [h] "s"((m)[11])
#define ALEPH_PAIR_UPDATE(T, MUL, FMA, MOV)                                                                          \
  __device__ __forceinline__ void pair_update(C2<T>& x, C2<T>& y, const T (&m)[8]) {                                 \
    T t0, t1, t2, t3;                                                                                                \
    asm volatile("s_nop 1\n" MUL " %[t0], %[a], %[xr]\n" MUL " %[t1], %[a], %[xi]\n" MUL " %[t2], %[e], %[xr]\n" MUL \
                 " %[t3], %[e], %[xi]\n" FMA " %[t0], -%[b], %[xi], %[t0]\n" FMA                                     \
                 " %[t1], %[b], %[xr], %[t1]\n" FMA " %[t2], -%[f], %[xi], %[t2]\n" FMA                              \
                 " %[t3], %[f], %[xr], %[t3]\n" FMA " %[t0], %[c], %[yr], %[t0]\n" FMA                               \
                 " %[t1], %[c], %[yi], %[t1]\n" FMA " %[t2], %[g], %[yr], %[t2]\n" FMA                               \
                 " %[t3], %[g], %[yi], %[t3]\n" FMA " %[xr], -%[d], %[yi], %[t0]\n" FMA                              \
                 " %[xi], %[d], %[yr], %[t1]\n" FMA " %[t3], %[h], %[yr], %[t3]\n" FMA                               \
                 " %[yr], -%[h], %[yi], %[t2]\n" MOV " %[yi], %[t3]\n"                                               \
                 : [xr] "+v"(x.x), [xi] "+v"(x.y), [yr] "+v"(y.x), [yi] "+v"(y.y), [t0] "=&v"(t0), [t1] "=&v"(t1),   \
                   [t2] "=&v"(t2), [t3] "=&v"(t3)                                                                    \
                 : [a] "s"(m[0]), [b] "s"(m[1]), [c] "s"(m[2]), [d] "s"(m[3]), [e] "s"(m[4]), [f] "s"(m[5]),         \
                   [g] "s"(m[6]), [h] "s"(m[7]));                                                                    \
  }                                                                                                                  \
  /* Two matrix rows (m: 16 entries) times a half of (v0, v1, v2, v3): into (p, q), or added to them. */             \
  template <bool FIRST>                                                                                              \
  __device__ __forceinline__ void two_rows(const C2<T>& v0, const C2<T>& v1, C2<T>& p, C2<T>& q, const T* m) {       \
    if constexpr (FIRST) {                                                                                           \
      asm volatile("s_nop 1\n" MUL " %[pr], %[a], %[xr]\n" MUL " %[pi], %[a], %[xi]\n"                               \
                   MUL " %[qr], %[e], %[xr]\n" MUL " %[qi], %[e], %[xi]\n" ALEPH_ROWS_TAIL(FMA)                      \
                   : [pr] "=&v"(p.x), [pi] "=&v"(p.y), [qr] "=&v"(q.x), [qi] "=&v"(q.y)                              \
                   : ALEPH_ROWS_IN(v0, v1, m));                                                                      \
    } else {                                                                                                         \
      asm volatile("s_nop 1\n" FMA " %[pr], %[a], %[xr], %[pr]\n" FMA " %[pi], %[a], %[xi], %[pi]\n"                 \
                   FMA " %[qr], %[e], %[xr], %[qr]\n" FMA " %[qi], %[e], %[xi], %[qi]\n" ALEPH_ROWS_TAIL(FMA)        \
                   : [pr] "+v"(p.x), [pi] "+v"(p.y), [qr] "+v"(q.x), [qi] "+v"(q.y)                                  \
                   : ALEPH_ROWS_IN(v0, v1, m));                                                                      \
    }                                                                                                                \
  }                                                                                                                  \
  /* a = v, in a's own registers. */                                                                                 \
  __device__ __forceinline__ void put(C2<T>& a, const C2<T>& v) {                                                    \
    asm volatile(MOV " %0, %2\n" MOV " %1, %3\n" : "+v"(a.x), "+v"(a.y) : "v"(v.x), "v"(v.y));                       \
  }                                                                                                                  \
  /* a *= (fr, fi), per-lane factor. */                                                                              \
  __device__ __forceinline__ void rotate(C2<T>& a, T fr, T fi) {                                                     \
    T t0, t1;                                                                                                        \
    asm volatile(MUL " %[t0], %[fi], %[ai]\n" MUL " %[t1], %[fi], %[ar]\n" FMA " %[ar], %[fr], %[ar], -%[t0]\n" FMA  \
                 " %[ai], %[fr], %[ai], %[t1]\n"                                                                     \
                 : [ar] "+v"(a.x), [ai] "+v"(a.y), [t0] "=&v"(t0), [t1] "=&v"(t1)                                    \
                 : [fr] "v"(fr), [fi] "v"(fi));                                                                      \
  }
ALEPH_PAIR_UPDATE(double, "v_mul_f64", "v_fma_f64", "v_mov_b64")
ALEPH_PAIR_UPDATE(float, "v_mul_f32", "v_fma_f32", "v_mov_b32")
#undef ALEPH_PAIR_UPDATE
#undef ALEPH_ROWS_TAIL
#undef ALEPH_ROWS_IN

}  // namespace fused
}  // namespace aleph
