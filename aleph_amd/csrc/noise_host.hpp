// Host lowering of a program and its noise channels into trajectory records.
#pragma once

#include <cstdint>
#include <vector>

#include "../../include/aleph_hip.h"
#include "engine.hpp"
#include "noise.hpp"

namespace aleph {

struct TrajHost {
  std::vector<TrajOp> ops;
  std::vector<double> reals;
  std::vector<uint64_t> masks;
  std::vector<uint32_t> index;
  std::vector<double> readout;   // n x 2 flip probabilities
  uint64_t readout_mask = 0;
};

// Validates channels and readout errors (throws Failure, kind
// "invalid-channel" or "unsupported") and lowers gates, diagonal phases and
// channels in program order.  Channels must be sorted by `after`.
TrajHost build_trajectories(const std::vector<ProgInstr>& prog, uint32_t n, const aleph_hip_channel* channels,
                            uint32_t n_channels, const double* readout, uint64_t readout_mask);

// The staged form of a lowered program, for register-resident trajectories.
struct StagedHost {
  std::vector<TStage> stages;
  std::vector<TOp> ops;
  std::vector<TChan> chans;
};

// Cuts `h` into stages (appending fused matrices to h.reals); false when a
// record has no staged form (DiagonalPhase, a dense gate on three qubits
// that is not a controlled one-qubit gate, a controlled two-qubit gate), or
// the qubit or channel count is out of the staged range.
bool build_staged(TrajHost& h, uint32_t n, StagedHost& out);

}  // namespace aleph
