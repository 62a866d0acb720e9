// Monte-Carlo noise trajectories on the device (quantum-jump unravelling).
//
// Semantics follow crates/aleph-sv/src/noise: after every gate the channels
// attached to it fire in order (execution.rs:102-135); a Pauli channel picks
// one Pauli string from its fixed weights with one uniform draw and applies
// it (apply.rs:46-66); a one-qubit Kraus channel computes p_i = |K_i psi|^2,
// draws one uniform, applies K_i / sqrt(p_i) and leaves the state alone
// when p_i < 1e-300 (apply.rs:68-133); the terminal outcome is one
// cumulative-inversion draw (sampling.rs:61-91), then one draw per qubit
// with a readout error flips that bit with probability m[t][1-t]
// (apply.rs:135-158).  Every trajectory draws from its own counter-based
// stream keyed by the reference's splitmix64 shot seed (apply.rs:160-180),
// so shot s's outcome depends only on (seed, s), never on how shots are
// spread over workgroups or calls.
//
// Device layout: one workgroup owns one trajectory at a time.  Programs of
// one- and two-qubit gates and diagonals on 2..14 qubits keep the state in
// registers (TStage below); other programs of up to 13 qubits (FP64, 128 KiB)
// keep it in LDS, and wider states live in a per-workgroup slice of a device
// buffer.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace aleph {

// One trajectory-program record.
struct TrajOp {
  enum Kind : uint32_t { DENSE = 0, DIAG = 1, PHASE = 2, PAULI = 3, KRAUS = 4 };
  uint32_t kind = DENSE;
  uint32_t k = 0;          // DENSE / DIAG: target count (DENSE <= 3, DIAG <= 6)
  uint32_t q[6] = {0};     // targets, q[0] = most significant bit of the matrix index
  uint32_t count = 0;      // PHASE: terms; PAULI / KRAUS: branches
  uint32_t off = 0;        // doubles into `reals`: DENSE matrix (2*4^k), DIAG entries (2*2^k),
                           // PHASE angles, PAULI weights, KRAUS matrices (8 per branch)
  uint32_t off2 = 0;       // PHASE: u64 conds into `masks`; PAULI: (x, z) mask pairs into `masks`
  uint32_t off3 = 0;       // PHASE: u32 CSR offsets (count + 1) into `index`
  uint64_t cmask = 0;      // DENSE / DIAG: control qubits
};
static_assert(sizeof(TrajOp) == 56, "TrajOp layout");

constexpr uint32_t kNoiseLdsMaxQubits = 13;     // 2^13 complex128 = 128 KiB of LDS
constexpr uint32_t kNoiseMaxQubits = 24;        // per-workgroup device slices beyond 13 qubits
constexpr uint32_t kNoiseMaxKraus = 64;         // branches of one Kraus channel
constexpr uint32_t kNoiseThreadsLds = 256;
constexpr uint32_t kNoiseThreadsWide = 1024;

// ---- register-resident trajectories ----
// A staged program is the record list of a trajectory in program order, cut
// into stages: in a stage every thread holds the 2^G amplitudes spanned by G
// register qubits, dense operators act on register qubits, and the state is
// re-distributed through LDS only where a stage ends.
//
// Pauli channels cost nothing in the record loop.  The physical state is kept
// as psi = X^x Z^z phi (up to a global phase) with the stored phi; a drawn
// Pauli only changes the frame (x, z), and an operator O acts on phi as
// F^dagger O F: rows and columns of its matrix permuted by x and signed by z,
// diagonals and controls evaluated at the stored index XOR x.  Every channel
// draws exactly once, so all draws of a shot are made first, one lane per
// channel, and a prefix XOR gives the frame before every record.
//
// A Kraus channel whose first operator K_0 has K_0^dagger K_0 >= lam takes
// branch 0 without looking at the state when the draw is below lam (p_0 >=
// lam whatever the state is); the state is then left unnormalised, and the
// branch probabilities of a channel that does need them are taken relative
// to the norm.  K_0 is multiplied into the gate before it on the host.
constexpr uint32_t kStagedMinQubits = 2;
constexpr uint32_t kStagedMaxQubits = 14;     // 2^14 amplitudes in 1024 threads, 128 KiB exchange buffer
constexpr uint32_t kStagedMaxChannels = 4096; // 5 bytes of LDS each, shared with the exchange buffer
constexpr uint32_t kStagedMaxOps = 2048;      // 8 bytes of LDS each

// Two 64-byte halves, each read with one scalar load; the next record is
// read while the current one runs.
struct alignas(64) TOp {
  enum Kind : uint32_t { ONE = 0, TWO = 1, SIGN = 2, DIAG = 3, KRAUS = 4 };
  uint32_t kind = ONE;
  uint32_t bit = 0;        // register bit of the target (ONE, KRAUS); A (A - 1) / 2 + B, A > B the matrix MSB (TWO)
  uint32_t qmask = 0;      // physical target (ONE, KRAUS); A's qubit (TWO); DIAG: 4-bit target list, MSB first
  uint32_t qmask2 = 0;     // TWO: B's qubit; DIAG: target count
  uint32_t cmask = 0;      // controls (ONE, DIAG) or the sign mask (SIGN)
  uint32_t off = 0;        // reals: ONE with a Kraus channel: the bare gate; TWO: 4x4; DIAG: entries
  uint32_t koff = 0;       // reals: Kraus matrices
  uint32_t count = 0;      // Kraus branches
  uint32_t chan = ~0u;     // Kraus channel of the record, ~0: none
  uint32_t f0 = 0;         // frame entry before the record
  uint32_t f1 = 0;         // frame entry before its Kraus channel
  uint32_t pad = 0;
  double lam = 1.0;        // lower bound of the K_0 branch's probability
  double pad2 = 0.0;
  double m[8] = {0};       // ONE: gate (times K_0); KRAUS: K_0
};
static_assert(sizeof(TOp) == 128, "TOp layout");

struct TChan {
  uint32_t pauli = 0;      // 1: Pauli channel (weights, masks), 0: Kraus
  uint32_t count = 0;
  uint32_t off = 0;        // reals: Pauli weights
  uint32_t off2 = 0;       // masks: (x, z) pairs
  double thr = 0.0;        // Kraus: draws below it take branch 0 without the state
};

struct TStage {
  uint32_t op_begin = 0, op_end = 0;
  uint32_t n_tb = 0;
  uint32_t pad = 0;
  uint32_t tl[12] = {0};   // qubit mask of thread-id bit j
  uint32_t ts[12] = {0};   // its swizzled LDS index
  uint32_t rl[4] = {0};    // qubit mask of register bit g
  uint32_t ls[16] = {0};   // swizzled LDS index of register slot r
};

// LDS index swizzle of the stage exchange (linear over XOR): bits 5.. folded
// into the low 5, so 32 lanes on bits distinct modulo 5 hit distinct banks.
__host__ __device__ inline uint32_t traj_swz(uint32_t x) { return x ^ ((x >> 5) & 31u) ^ ((x >> 10) & 31u); }

struct StagedProgram {
  const TStage* stages = nullptr;
  const TOp* ops = nullptr;
  const TChan* chans = nullptr;
  uint32_t n_stages = 0;
  uint32_t n_ops = 0;      // records; one more follows them for the read-ahead
  uint32_t n_chan = 0;
  bool rare = false;       // has two-qubit matrices, diagonals other than signs, or controlled gates
};

// Register qubits of an n-qubit staged trajectory: 16 amplitudes per thread
// where that still fills a wavefront, fewer below.
inline uint32_t staged_reg_bits(uint32_t n) { return n >= 10 ? 4u : n == 9 ? 3u : 2u; }

struct TrajProgram {
  const TrajOp* ops = nullptr;
  uint32_t n_ops = 0;
  uint32_t n = 0;
  const double* reals = nullptr;
  const uint64_t* masks = nullptr;
  const uint32_t* index = nullptr;
  const double* readout = nullptr;   // n x 2: P(flip | true 0), P(flip | true 1)
  uint64_t readout_mask = 0;         // qubits with a readout error
  uint64_t seed = 0;
  uint64_t shot0 = 0;                // absolute index of the first shot of this launch
  uint32_t shots = 0;
};

// Runs `p.shots` trajectories; outcome of shot i -> out[i].  `slices` is
// null for n <= kNoiseLdsMaxQubits, else `workgroups` * 2^n complex128.
void launch_trajectories(hipStream_t s, const TrajProgram& p, uint32_t workgroups, void* slices, uint64_t* out);

// The same for a program that lowered to stages; state in registers.
void launch_staged(hipStream_t s, const TrajProgram& p, const StagedProgram& sp, uint64_t* out);

// Workgroups and device bytes the launch for an n-qubit program uses
// (bytes = 0 when the state fits in LDS).  `budget` bounds the slices.
void trajectory_geometry(uint32_t n, uint32_t shots, size_t budget, uint32_t* workgroups, size_t* bytes);

}  // namespace aleph
