// Host side of the noise trajectories: validation of channels and readout
// errors (crates/aleph-sv/src/noise/execution.rs:207-300) and lowering of a
// decoded program plus its channels into trajectory records.
#include "noise_host.hpp"

#include <cmath>
#include <complex>

#include "common.hpp"
#include "gates.hpp"

namespace aleph {
namespace {

Failure invalid_channel(const std::string& why) {
  Failure f{ALEPH_HIP_ERR_INVALID_ARGUMENT, why};
  f.kind = "invalid-channel";
  return f;
}

void push_complex(std::vector<double>& v, const cplx& z) {
  v.push_back(z.real());
  v.push_back(z.imag());
}

}  // namespace

TrajHost build_trajectories(const std::vector<ProgInstr>& prog, uint32_t n, const aleph_hip_channel* channels,
                            uint32_t n_channels, const double* readout, uint64_t readout_mask) {
  TrajHost h;
  if (n_channels && !channels) throw invalid_channel("null channel array");
  uint32_t next = 0;
  for (uint32_t c = 0; c < n_channels; c++) {
    const aleph_hip_channel& ch = channels[c];
    if (ch.after >= prog.size()) throw invalid_channel("channel attached past the end of the program");
    if (c && ch.after < channels[c - 1].after) throw invalid_channel("channels must be ordered by instruction");
    if (prog[ch.after].type != ProgInstr::GATE) throw invalid_channel("channels attach to gates only");
    if (ch.n_branches == 0) throw invalid_channel("channel without branches");
    for (uint32_t j = 0; j < ch.n_qubits && j < 2; j++)
      if (ch.qubits[j] >= n) throw invalid_channel("channel qubit out of range");
    if (ch.kind == ALEPH_HIP_CHANNEL_PAULI) {
      if (ch.n_qubits < 1 || ch.n_qubits > 2) throw invalid_channel("Pauli channels act on one or two qubits");
      if (ch.n_qubits == 2 && ch.qubits[0] == ch.qubits[1]) throw invalid_channel("duplicate channel qubit");
      if (!ch.weights || !ch.paulis) throw invalid_channel("null Pauli channel data");
      double total = 0.0;
      for (uint32_t b = 0; b < ch.n_branches; b++) {
        const double p = ch.weights[b];
        if (!std::isfinite(p) || p < 0.0) throw invalid_channel("invalid Pauli probability or term arity");
        for (uint32_t j = 0; j < ch.n_qubits; j++)
          if (ch.paulis[b * ch.n_qubits + j] > 3) throw invalid_channel("invalid Pauli code");
        total += p;
      }
      if (!std::isfinite(total) || std::fabs(total - 1.0) > 1e-9)
        throw invalid_channel("Pauli probabilities must sum to one");
    } else if (ch.kind == ALEPH_HIP_CHANNEL_KRAUS) {
      if (ch.n_qubits != 1) throw invalid_channel("Kraus channels act on one qubit");
      if (ch.n_branches > kNoiseMaxKraus) throw invalid_channel("too many Kraus operators");
      if (!ch.kraus) throw invalid_channel("null Kraus channel data");
      cplx comp[2][2] = {{0.0, 0.0}, {0.0, 0.0}};
      for (uint32_t b = 0; b < ch.n_branches; b++) {
        const double* k = ch.kraus + 8 * b;
        for (int e = 0; e < 8; e++)
          if (!std::isfinite(k[e])) throw invalid_channel("non-finite Kraus matrix");
        const cplx K[2][2] = {{cplx(k[0], k[1]), cplx(k[2], k[3])}, {cplx(k[4], k[5]), cplx(k[6], k[7])}};
        for (int i = 0; i < 2; i++)
          for (int j = 0; j < 2; j++)
            for (int r = 0; r < 2; r++) comp[i][j] += std::conj(K[r][i]) * K[r][j];
      }
      for (int i = 0; i < 2; i++)
        for (int j = 0; j < 2; j++) {
          const double dev = std::abs(comp[i][j] - cplx(i == j ? 1.0 : 0.0, 0.0));
          if (!std::isfinite(dev) || dev > 1e-9) throw invalid_channel("Kraus operators must be trace preserving");
        }
    } else {
      throw invalid_channel("unknown channel kind");
    }
  }
  // Readout errors: rows of m[t][o] non-negative and summing to one.
  if (n < 64 && (readout_mask >> n) != 0) throw invalid_channel("invalid readout probability or qubit");
  h.readout.assign(2 * (size_t)n, 0.0);
  if (readout_mask) {
    if (!readout) throw invalid_channel("null readout matrices");
    for (uint32_t q = 0; q < n; q++) {
      if (!((readout_mask >> q) & 1ull)) continue;
      const double* m = readout + 4 * q;
      for (int e = 0; e < 4; e++)
        if (!std::isfinite(m[e]) || m[e] < 0.0) throw invalid_channel("invalid readout probability or qubit");
      if (std::fabs(m[0] + m[1] - 1.0) > 1e-9 || std::fabs(m[2] + m[3] - 1.0) > 1e-9)
        throw invalid_channel("invalid readout probability or qubit");
      h.readout[2 * q] = m[1];       // P(read 1 | true 0)
      h.readout[2 * q + 1] = m[2];   // P(read 0 | true 1)
    }
  }
  h.readout_mask = readout_mask;

  for (uint32_t i = 0; i < prog.size(); i++) {
    const ProgInstr& pi = prog[i];
    if (pi.type == ProgInstr::GATE) {
      const DenseGate& d = pi.gate;
      TrajOp op;
      op.k = (uint32_t)d.qubits.size();
      for (uint32_t t = 0; t < op.k; t++) op.q[t] = d.qubits[t];
      for (uint32_t cq : d.controls) op.cmask |= 1ull << cq;
      op.off = (uint32_t)h.reals.size();
      if (d.diagonal) {
        op.kind = TrajOp::DIAG;
        for (uint32_t j = 0; j < d.dim; j++) push_complex(h.reals, d.m[(size_t)j * d.dim + j]);
      } else {
        if (op.k > 3) {
          Failure f{ALEPH_HIP_ERR_INVALID_ARGUMENT, "dense gates on more than 3 qubits are not supported under noise"};
          f.kind = "unsupported";
          throw f;
        }
        op.kind = TrajOp::DENSE;
        for (const cplx& z : d.m) push_complex(h.reals, z);
      }
      h.ops.push_back(op);
    } else if (pi.type == ProgInstr::DIAG_PHASE) {
      TrajOp op;
      op.kind = TrajOp::PHASE;
      op.count = (uint32_t)pi.angles.size();
      op.off = (uint32_t)h.reals.size();
      op.off2 = (uint32_t)h.masks.size();
      op.off3 = (uint32_t)h.index.size();
      uint32_t at = 0;
      h.index.push_back(0);
      for (size_t t = 0; t < pi.angles.size(); t++) {
        h.reals.push_back(pi.angles[t]);
        for (uint64_t c : pi.conds[t]) h.masks.push_back(c);
        at += (uint32_t)pi.conds[t].size();
        h.index.push_back(at);
      }
      if (op.count) h.ops.push_back(op);
    }
    for (; next < n_channels && channels[next].after == i; next++) {
      const aleph_hip_channel& ch = channels[next];
      TrajOp op;
      op.count = ch.n_branches;
      op.off = (uint32_t)h.reals.size();
      op.k = ch.n_qubits;
      op.q[0] = ch.qubits[0];
      op.q[1] = ch.qubits[1];
      if (ch.kind == ALEPH_HIP_CHANNEL_PAULI) {
        op.kind = TrajOp::PAULI;
        op.off2 = (uint32_t)h.masks.size();
        for (uint32_t b = 0; b < ch.n_branches; b++) {
          h.reals.push_back(ch.weights[b]);
          uint64_t xm = 0, zm = 0;
          for (uint32_t j = 0; j < ch.n_qubits; j++) {
            const uint8_t code = ch.paulis[b * ch.n_qubits + j];
            const uint64_t bit = 1ull << ch.qubits[j];
            if (code == 1 || code == 2) xm |= bit;   // X, Y
            if (code == 2 || code == 3) zm |= bit;   // Y, Z
          }
          h.masks.push_back(xm);
          h.masks.push_back(zm);
        }
      } else {
        op.kind = TrajOp::KRAUS;
        for (uint32_t e = 0; e < 8 * ch.n_branches; e++) h.reals.push_back(ch.kraus[e]);
      }
      h.ops.push_back(op);
    }
  }
  if (h.reals.empty()) h.reals.push_back(0.0);
  if (h.masks.empty()) h.masks.push_back(0);
  if (h.index.empty()) h.index.push_back(0);
  return h;
}

namespace {

// Dense matrix (interleaved, dim 2^k, targets MSB first) that is the identity
// except for a 2x2 block selected by every target but one being 1: the
// remaining target's position, or -1.
int controlled_target(const double* m, uint32_t k) {
  const uint32_t dim = 1u << k;
  for (uint32_t t = 0; t < k; t++) {
    const uint32_t tb = 1u << (k - 1 - t), cb = (dim - 1u) & ~tb;
    bool ok = true;
    for (uint32_t r = 0; r < dim && ok; r++)
      for (uint32_t c = 0; c < dim && ok; c++) {
        if ((r & cb) == cb && (c & cb) == cb) continue;
        ok = m[2 * (r * dim + c)] == (r == c ? 1.0 : 0.0) && m[2 * (r * dim + c) + 1] == 0.0;
      }
    if (ok) return (int)t;
  }
  return -1;
}

// Smallest eigenvalue of K^dagger K.
double min_branch_probability(const double* k) {
  const double a = k[0] * k[0] + k[1] * k[1] + k[4] * k[4] + k[5] * k[5];
  const double d = k[2] * k[2] + k[3] * k[3] + k[6] * k[6] + k[7] * k[7];
  const cplx b = std::conj(cplx(k[0], k[1])) * cplx(k[2], k[3]) + std::conj(cplx(k[4], k[5])) * cplx(k[6], k[7]);
  return 0.5 * ((a + d) - std::sqrt((a - d) * (a - d) + 4.0 * std::norm(b)));
}

void mul2x2(const double* a, const double* b, double* out) {
  for (int r = 0; r < 2; r++)
    for (int c = 0; c < 2; c++) {
      cplx z = 0.0;
      for (int j = 0; j < 2; j++)
        z += cplx(a[2 * (2 * r + j)], a[2 * (2 * r + j) + 1]) * cplx(b[2 * (2 * j + c)], b[2 * (2 * j + c) + 1]);
      out[2 * (2 * r + c)] = z.real();
      out[2 * (2 * r + c) + 1] = z.imag();
    }
}

// Draws within this relative distance of the bound look at the state, so the
// rounding of the computed probability cannot change a decision; channels
// whose bound is small always do (the unnormalised state would shrink fast).
constexpr double kShortcutGuard = 1e-9;
constexpr double kShortcutMin = 1e-3;

}  // namespace

bool build_staged(TrajHost& h, uint32_t n, StagedHost& out) {
  if (n < kStagedMinQubits || n > kStagedMaxQubits) return false;
  const uint32_t G = staged_reg_bits(n);
  std::vector<TOp> ops;
  std::vector<uint32_t> need;   // qubits that must sit in registers, per record
  // `last` is a ONE record that only Pauli channels have followed: a Kraus
  // channel on its qubit is folded into it.
  int64_t last = -1;
  for (const TrajOp& t : h.ops) {
    TOp op;
    op.f0 = op.f1 = (uint32_t)out.chans.size();
    if (t.kind == TrajOp::PAULI) {
      TChan c;
      c.pauli = 1;
      c.count = t.count;
      c.off = t.off;
      c.off2 = t.off2;
      out.chans.push_back(c);
      continue;
    }
    if (t.kind == TrajOp::KRAUS) {
      TChan c;
      c.count = t.count;
      const double* k0 = h.reals.data() + t.off;
      const double lam = min_branch_probability(k0);
      if (lam >= kShortcutMin) c.thr = lam * (1.0 - kShortcutGuard);
      const uint32_t chan = (uint32_t)out.chans.size();
      out.chans.push_back(c);
      if (last >= 0 && ops[(size_t)last].qmask == (1u << t.q[0]) && ops[(size_t)last].chan == ~0u) {
        TOp& g = ops[(size_t)last];
        g.off = (uint32_t)h.reals.size();
        h.reals.insert(h.reals.end(), g.m, g.m + 8);
        double f[8];
        mul2x2(h.reals.data() + t.off, h.reals.data() + g.off, f);
        for (int e = 0; e < 8; e++) g.m[e] = f[e];
        g.f1 = chan;
        g.chan = chan;
        g.koff = t.off;
        g.count = t.count;
        g.lam = lam;
        last = -1;
        continue;
      }
      op.kind = TOp::KRAUS;
      op.qmask = 1u << t.q[0];
      op.chan = chan;
      op.koff = t.off;
      op.count = t.count;
      op.lam = lam;
      for (int e = 0; e < 8; e++) op.m[e] = k0[e];
      ops.push_back(op);
      need.push_back(op.qmask);
      last = -1;
      continue;
    }
    last = -1;
    const double* m = h.reals.data() + t.off;
    if (t.kind == TrajOp::DIAG) {
      const uint32_t dim = 1u << t.k;
      bool sign = true;
      uint32_t targets = 0;
      for (uint32_t j = 0; j < dim; j++) sign &= m[2 * j] == (j + 1 == dim ? -1.0 : 1.0) && m[2 * j + 1] == 0.0;
      for (uint32_t j = 0; j < t.k; j++) targets |= 1u << t.q[j];
      op.kind = sign ? TOp::SIGN : TOp::DIAG;
      op.cmask = (uint32_t)t.cmask | (sign ? targets : 0u);
      op.off = t.off;
      op.qmask2 = t.k;
      for (uint32_t j = 0; j < t.k; j++) op.qmask |= t.q[j] << (4 * j);
      ops.push_back(op);
      need.push_back(0);
      continue;
    }
    if (t.kind != TrajOp::DENSE) return false;
    const int ct = t.k == 1 ? 0 : controlled_target(m, t.k);
    if (ct >= 0) {
      const uint32_t dim = 1u << t.k, tb = 1u << (t.k - 1 - (uint32_t)ct), hi = dim - 1u, lo = hi & ~tb;
      op.kind = TOp::ONE;
      op.qmask = 1u << t.q[ct];
      op.cmask = (uint32_t)t.cmask;
      for (uint32_t j = 0; j < t.k; j++)
        if ((int)j != ct) op.cmask |= 1u << t.q[j];
      const uint32_t e[4] = {lo * dim + lo, lo * dim + hi, hi * dim + lo, hi * dim + hi};
      for (int i = 0; i < 4; i++) {
        op.m[2 * i] = m[2 * e[i]];
        op.m[2 * i + 1] = m[2 * e[i] + 1];
      }
      ops.push_back(op);
      need.push_back(op.qmask);
      if (op.cmask == 0) last = (int64_t)ops.size() - 1;
      continue;
    }
    if (t.k != 2 || t.cmask != 0) return false;
    op.kind = TOp::TWO;
    op.qmask = 1u << t.q[0];
    op.qmask2 = 1u << t.q[1];
    op.off = t.off;
    ops.push_back(op);
    need.push_back(op.qmask | op.qmask2);
  }
  if (out.chans.size() > kStagedMaxChannels || ops.size() > kStagedMaxOps) return false;
  // Stages in program order (the outcome of a Kraus channel depends on the
  // order of the channels): a stage takes records while their targets fit G
  // register qubits.
  const uint32_t all = (1u << n) - 1u;
  for (size_t i = 0; i < ops.size() || out.stages.empty();) {
    TStage st;
    uint32_t reg = 0;
    st.op_begin = (uint32_t)out.ops.size();
    size_t j = i;
    for (; j < ops.size() && (uint32_t)__builtin_popcount(reg | need[j]) <= G; j++) reg |= need[j];
    for (int b = (int)n - 1; b >= 0 && (uint32_t)__builtin_popcount(reg) < G; b--) reg |= 1u << b;
    uint32_t bit_of[32] = {0}, g = 0;
    for (uint32_t q = 0; q < n; q++)
      if ((reg >> q) & 1u) {
        bit_of[q] = g;
        st.rl[g++] = 1u << q;
      }
    // Thread bits: lanes' first five on qubits distinct modulo 5 where the
    // remaining qubits allow it (one bank group each, see traj_swz).
    uint32_t rest = all & ~reg, classes = 0;
    for (int round = 0; round < 2; round++)
      for (uint32_t q = 0; q < n; q++) {
        if (!((rest >> q) & 1u)) continue;
        if (round == 0 && (((classes >> (q % 5)) & 1u) || st.n_tb >= 5)) continue;
        classes |= 1u << (q % 5);
        st.tl[st.n_tb++] = 1u << q;
        rest &= ~(1u << q);
      }
    for (uint32_t t = 0; t < st.n_tb; t++) st.ts[t] = traj_swz(st.tl[t]);
    for (uint32_t r = 0; r < (1u << G); r++)
      for (uint32_t b = 0; b < G; b++)
        if ((r >> b) & 1u) st.ls[r] ^= traj_swz(st.rl[b]);
    for (; i < j; i++) {
      TOp op = ops[i];
      auto bit = [&](uint32_t mask) { return bit_of[__builtin_ctz(mask)]; };
      if (op.kind == TOp::TWO) {
        if (bit(op.qmask) < bit(op.qmask2)) {   // the matrix MSB on the higher register bit
          std::vector<double> sw(32);
          auto x = [](int v) { return ((v & 1) << 1) | (v >> 1); };
          for (int r = 0; r < 4; r++)
            for (int c = 0; c < 4; c++)
              for (int e = 0; e < 2; e++) sw[2 * (4 * r + c) + e] = h.reals[op.off + 2 * (4 * x(r) + x(c)) + e];
          op.off = (uint32_t)h.reals.size();
          h.reals.insert(h.reals.end(), sw.begin(), sw.end());
          std::swap(op.qmask, op.qmask2);
        }
        op.bit = bit(op.qmask) * (bit(op.qmask) - 1) / 2 + bit(op.qmask2);
      } else if (op.kind != TOp::SIGN && op.kind != TOp::DIAG) {
        op.bit = bit(op.qmask);
      }
      out.ops.push_back(op);
    }
    st.op_end = (uint32_t)out.ops.size();
    out.stages.push_back(st);
  }
  out.ops.push_back(TOp{});   // read ahead, never run
  return true;
}

}  // namespace aleph
