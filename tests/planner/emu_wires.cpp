// CPU model of the fused tile pass for programs planned in wires
// (qsim_wire_plan.hpp).  TEST INFRASTRUCTURE ONLY.
//
// Runs the planner's exact headers, ops, relayout constants and coefficients as
// the device interpreter does, with every LDS write checked for range and
// collisions, every LDS read for an unwritten slot and every store for a second
// write to one address.
#include "../../quict_amd/csrc/qsim_fused_plan.hpp"

#include <complex>
#include <stdexcept>
#include <string>

extern "C" int cpu_apply_gates(double* vec, int n, const qs_gate* gates, int ngates, int threads);

namespace qs {
static std::string g_err;
void set_error(const std::string& msg) { g_err = msg; }
using zc = std::complex<double>;

static void dense(zc* A, int NR, const int* pos, int k, const zc* M, const FOp& op) {
  const int D = 1 << k;
  uint32_t pm = 0;
  for (int i = 0; i < k; ++i) pm |= 1u << pos[i];
  auto off = [&](int q) {
    int o = 0;
    for (int i = 0; i < k; ++i)
      if ((q >> (k - 1 - i)) & 1) o |= 1 << pos[i];
    return o;
  };
  for (int r = 0; r < NR; ++r) {
    if ((r & pm) || ((uint32_t)r & op.creg) != op.cregv) continue;
    std::vector<zc> x(D);
    for (int q = 0; q < D; ++q) x[q] = A[r | off(q)];
    for (int i = 0; i < D; ++i) {
      zc y = 0;
      for (int j = 0; j < D; ++j) y += M[i * D + j] * x[j];
      A[r | off(i)] = y;
    }
  }
}

static void wire_pass(zc* v, int n, int RB, int TB, uint32_t S, const PassHdr& H, const FOp* P, const double* Cd,
                      const uint32_t* X) {
  const int NR = 1 << RB, NT = 1 << TB, K = RB + TB;
  std::vector<zc> a((size_t)NT * NR), lds((size_t)NT * NR), out((size_t)NT * NR);
  std::vector<int> written((size_t)NT * NR);
  auto cz = [&](int i) { return zc(Cd[2 * i], Cd[2 * i + 1]); };
  // a register below a tile: the amplitudes it lacks are zeros and not stored
  const uint64_t N = 1ull << n;
  for (uint64_t t = 0; t < (n > K ? 1ull << (n - K) : 1); ++t) {
    const uint64_t tb = insert_zeros(t, H.sorted, K);
    for (int tid = 0; tid < NT; ++tid)
      for (int r = 0; r < NR; ++r) {
        uint64_t g = tb;
        for (int b = 0; b < TB; ++b) g |= (uint64_t)((tid >> b) & 1) << H.tbits[H.ts0[b]];
        for (int b = 0; b < RB; ++b) g |= (uint64_t)((r >> b) & 1) << H.tbits[H.rs0[b]];
        a[(size_t)tid * NR + r] = g < N ? v[g] : zc(0);
      }
    for (int o = 0; o < H.nops; ++o) {
      const FOp& op = P[o];
      if (op.kind == F_RELAYOUT) {
        const uint32_t* x = X + op.coef;
        const int p = (int)x[0];
        const uint32_t *lw = x + 1, *tw = x + 1 + RB, *y = x + 2 + RB + TB, *z = y + RB + TB;
        uint32_t xf = x[1 + RB + TB];
        if (op.pure)
          for (uint32_t i = 0; i < z[0]; ++i)
            if ((t >> z[1 + 2 * i]) & 1) xf ^= z[2 + 2 * i];
        for (int k = 0; k < 2; ++k) {
          std::fill(written.begin(), written.end(), 0);
          for (int dir = 0; dir < 2; ++dir)
            for (int tid = 0; tid < NT; ++tid)
              for (int r = 0; r < NR; ++r) {
                if (((r >> p) & 1) != k) continue;
                uint32_t off = dir ? 0 : xf;
                for (int b = 0; b < TB; ++b)
                  if ((tid >> b) & 1) off ^= dir ? y[RB + b] : tw[b];
                for (int b = 0; b < RB; ++b)
                  if ((r >> b) & 1) off ^= dir ? y[b] : lw[b];
                if (off % S || off / S >= (uint32_t)(NT * NR / 2)) throw std::runtime_error("lds address out of range");
                if (dir == 0) {
                  if (written[off / S]++) throw std::runtime_error("lds write collision");
                  lds[off / S] = a[(size_t)tid * NR + r];
                } else {
                  if (!written[off / S]) throw std::runtime_error("lds read of an unwritten slot");
                  a[(size_t)tid * NR + r] = lds[off / S];
                }
              }
        }
        // the lanes of one 128-byte cycle on distinct banks, on both sides
        for (int dir = 0; dir < 2; ++dir) {
          uint32_t seen = 0;
          for (uint32_t lane = 0; lane < 128 / S; ++lane) {
            uint32_t off = 0;
            for (int b = 0; b < TB; ++b)
              if ((lane >> b) & 1) off ^= dir ? y[RB + b] : tw[b];
            const uint32_t bit = 1u << (off / S % (128 / S));
            if (seen & bit) throw std::runtime_error("lds bank conflict");
            seen |= bit;
          }
        }
        continue;
      }
      if (((uint32_t)t & op.cblk) != op.cblkv) continue;
      for (int tid = 0; tid < NT; ++tid) {
        zc* A = &a[(size_t)tid * NR];
        const bool tok = ((uint32_t)tid & op.cthr) == op.cthrv;
        std::vector<zc> M;
        switch (op.kind) {
          case F_PHASE:
            if (op.pure == 1 && cz(op.coef).imag() != 0.0) throw std::runtime_error("real phase with imaginary part");
            if (tok)
              for (int r = 0; r < NR; ++r) {
                if (((uint32_t)r & op.creg) != op.creg) continue;
                const zc f = cz(op.coef);
                if (op.pure < 2) {
                  A[r] *= f;
                  continue;
                }
                if (std::abs(f.real()) > 1.0 + 1e-12) throw std::runtime_error("shear above 1");
                double re = A[r].real() + f.real() * A[r].imag();
                const double im = A[r].imag() + f.imag() * re;
                re += f.real() * im;
                A[r] = op.pure == 3 ? zc(-re, -im) : zc(re, im);
              }
            break;
          case F_ROT: {
            const int bit = 1 << op.pos[0];
            const zc f = cz(op.coef);
            if (op.creg || op.cthr || std::abs(f.real()) > 1.0 + 1e-12) throw std::runtime_error("bad rotation");
            for (int r = 0; r < NR; ++r) {
              if (r & bit) continue;
              A[r] += f.real() * A[r | bit];
              A[r | bit] += f.imag() * A[r];
              A[r] += f.real() * A[r | bit];
            }
            break;
          }
          case F_DIAG: {
            uint32_t sel = 0;
            for (int k = 0; k < op.ntt; ++k) sel = (sel << 1) | ((tid >> op.tpos[k]) & 1u);
            if (op.coef + (op.pure ? 1 << op.ntt : NR << op.ntt) > H.nstage) throw std::runtime_error("table not staged");
            for (int r = 0; r < NR; ++r) A[r] *= cz(op.coef + (op.pure ? (int)sel : (int)sel * NR + r));
            break;
          }
          case F_PERM1:
            M = {0, op.pure ? zc(1) : cz(op.coef), op.pure ? zc(1) : cz(op.coef + 1), 0};
            if (tok) dense(A, NR, op.pos, 1, M.data(), op);
            break;
          case F_SWAP2:
            M.assign(16, 0);
            M[0] = M[15] = 1;
            M[1 * 4 + 2] = op.pure ? zc(1) : cz(op.coef);
            M[2 * 4 + 1] = op.pure ? zc(1) : cz(op.coef + 1);
            if (tok) dense(A, NR, op.pos, 2, M.data(), op);
            break;
          case F_XX2:
            if (op.creg || op.cthr) throw std::runtime_error("xx2 op with controls");
            M.assign(16, 0);
            for (int s = 0; s < 4; ++s) M[5 * s] = cz(op.coef + s), M[4 * s + (s ^ 3)] = cz(op.coef + 4 + s);
            dense(A, NR, op.pos, 2, M.data(), op);
            break;
          case F_DENSE1:
          case F_DENSE2:
          case F_DENSE3:
          case F_DENSE4: {
            const int k = op.kind == F_DENSE1 ? 1 : op.kind == F_DENSE2 ? 2 : op.kind == F_DENSE3 ? 3 : 4;
            for (int i = 1; i < k; ++i)
              if (op.pos[i - 1] <= op.pos[i]) throw std::runtime_error("positions not descending");
            for (int i = 0; i < (1 << (2 * k)); ++i)
              M.push_back(cz(op.coef + i));
            if (tok) dense(A, NR, op.pos, k, M.data(), op);
            break;
          }
          default:
            throw std::runtime_error("unknown op");
        }
      }
    }
    std::fill(written.begin(), written.end(), 0);
    uint64_t tmask = 0;
    for (int j = 0; j < K; ++j) tmask |= 1ull << H.tbits[j];
    auto compact = [&](uint64_t g) {
      uint32_t k = 0;
      for (int j = 0; j < K; ++j) k |= (uint32_t)((g >> H.sorted[j]) & 1) << j;
      return k;
    };
    uint64_t sx = tb ^ H.sflip;
    for (int i = 0; i < H.nsx; ++i)
      if ((t >> H.sxb[i]) & 1) sx ^= H.sxm[i];
    for (int tid = 0; tid < NT; ++tid)
      for (int r = 0; r < NR; ++r) {
        uint64_t g = sx;
        for (int b = 0; b < TB; ++b)
          if ((tid >> b) & 1) g ^= H.st[b];
        for (int b = 0; b < RB; ++b)
          if ((r >> b) & 1) g ^= H.sr[b];
        if ((g & ~tmask) != tb) throw std::runtime_error("store outside the tile");
        if (written[compact(g)]++) throw std::runtime_error("store collision");
        out[compact(g)] = a[(size_t)tid * NR + r];
      }
    for (uint32_t k = 0; k < (uint32_t)(NT * NR); ++k) {
      uint64_t g = tb;
      for (int j = 0; j < K; ++j) g |= (uint64_t)((k >> j) & 1) << H.sorted[j];
      if (g < N) v[g] = out[k];
      else if (out[k] != zc(0)) throw std::runtime_error("amplitude outside the register");
    }
  }
}
}  // namespace qs

extern "C" const char* wires_last_error() { return qs::g_err.c_str(); }

// Plans and runs `gates` on vec (NULL: plans only), chunk by chunk as the
// streamed launch does.  stats: passes, fused passes, ops, relayouts, ops with a
// tile predicate, phases, exchanges, largest staged table count.
extern "C" int wires_apply(double* vec, int n, const qs_gate* gates, int ngates, int RB, int TB, int L, int amp_bytes,
                           int* stats) {
  using namespace qs;
  try {
    Config c{RB, TB, L};
    c.wires = true;
    FusedProgram prog;
    auto chunk = [&](const FusedProgram& sub, int) -> int {
      for (const PassHdr& H : sub.hdrs)
        if (vec)
          wire_pass(reinterpret_cast<zc*>(vec), n, RB, TB, (uint32_t)amp_bytes, H, sub.ops.data() + H.op0,
                    sub.coef.data() + 2 * (size_t)H.coef0, sub.aux.data());
      return 0;
    };
    auto single = [&](const qs_gate& g) -> int { return vec ? cpu_apply_gates(vec, n, &g, 1, 1) : 0; };
    const int rc = build_streamed(gates, ngates, n, c, (uint32_t)amp_bytes, prog, chunk, single);
    if (rc) return rc;
    std::fill(stats, stats + 8, 0);
    stats[0] = (int)prog.plans.size();
    stats[1] = (int)prog.hdrs.size();
    stats[2] = (int)prog.ops.size();
    for (const FOp& o : prog.ops) {
      stats[3] += o.kind == F_RELAYOUT;
      stats[4] += o.cblk != 0;
      stats[5] += o.kind == F_PHASE;
      stats[6] += o.kind == F_PERM1;
    }
    for (const PassHdr& h : prog.hdrs) stats[7] = std::max(stats[7], h.nstage);
    if (getenv("QS_FUSION_DEBUG")) print_program_stats(prog, n, RB + TB, L, ngates);
    return 0;
  } catch (const std::exception& e) {
    g_err = e.what();
    return -99;
  }
}
