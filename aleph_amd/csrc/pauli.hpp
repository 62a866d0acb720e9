// Pauli-string sums in few reads of the state (k_pauli.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstring>
#include <vector>

namespace aleph {

// coeff * P: X on the bits of x (Y included), sign mask zy (Z and Y), ny Ys.
struct PauliTerm {
  uint64_t x = 0, zy = 0;
  int ny = 0;
  double coeff = 0.0;
};

// One read of the state: its chunk qubits and the terms it evaluates.
struct PauliSweep {
  uint64_t qubits = 0;
  std::vector<uint32_t> terms;
};

// sweeps[0] always exists when n >= 4 and carries the norm; `rest` lists the
// terms that no sweep can hold (all of them when n < 4), ordered by X mask so
// that those with the same one share a read.
struct PauliPlan {
  std::vector<PauliSweep> sweeps;
  std::vector<uint32_t> rest;
};

PauliPlan plan_pauli_sum(const std::vector<PauliTerm>& terms, uint32_t n);

// Workgroups of a sweep at most, each with a row of three partial sums.
constexpr uint32_t kPauliRows = 1024;

// Runs the sweeps and waits: result = {sum of the sweeps' terms, sum |psi|^2,
// amplitudes with a non-finite |psi|^2} (host-visible).  `dev` is scratch for
// the records (an allocation is made when it is too small), `partials` holds
// 3 * kPauliRows doubles.
template <typename T>
void run_pauli_sweeps(hipStream_t st, const void* state, uint32_t n, const PauliPlan& plan,
                      const std::vector<PauliTerm>& terms, void* dev, size_t dev_bytes, double* partials,
                      double* result);

}  // namespace aleph
