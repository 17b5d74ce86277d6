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
                      const uint32_t* X, const PassStart& known = PassStart{}) {
  const int NR = 1 << RB, NT = 1 << TB, K = RB + TB;
  std::vector<zc> a((size_t)NT * NR), lds((size_t)NT * NR), out((size_t)NT * NR);
  std::vector<int> written((size_t)NT * NR);
  auto cz = [&](int i) { return zc(Cd[2 * i], Cd[2 * i + 1]); };
  // a register below a tile: the amplitudes it lacks are zeros and not stored
  const uint64_t N = 1ull << n;
  const uint64_t tiles = known.fixed ? 1ull << __builtin_popcountll(known.free) : n > K ? 1ull << (n - K) : 1;
  for (uint64_t i = 0; i < tiles; ++i) {
    uint32_t number = (uint32_t)i;
    const uint64_t tb = known.fixed ? start_tile(known, i, H.sorted, K, number) : insert_zeros(i, H.sorted, K);
    const uint64_t t = number;
    for (int tid = 0; tid < NT; ++tid)
      for (int r = 0; r < NR; ++r) {
        uint64_t g = tb;
        for (int b = 0; b < TB; ++b) g |= (uint64_t)((tid >> b) & 1) << H.tbits[H.ts0[b]];
        for (int b = 0; b < RB; ++b) g |= (uint64_t)((r >> b) & 1) << H.tbits[H.rs0[b]];
        const bool zero = ((known.sh ? g ^ (g >> known.sh) : g) & known.fixed) != 0;
        if (!known.fixed) a[(size_t)tid * NR + r] = g >= N ? zc(0) : v[g];  // (wire_load: with nsmall)
        else if (zero || known.fresh) a[(size_t)tid * NR + r] = zero ? 0.0 : 1.0;
        else if (g >= N) throw std::runtime_error("load outside the vector");
        else a[(size_t)tid * NR + r] = v[g];
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

// The program from |0...0> (identity: from the identity matrix on n = 2m bits), vec
// holding anything before: as the launches do, with what is known to be zero neither
// read nor computed.  stats: passes, tiles run, tiles there are.
extern "C" int wires_run(double* vec, int n, int identity, const qs_gate* gates, int ngates, int RB, int TB, int L,
                         int amp_bytes, int64_t* stats) {
  using namespace qs;
  try {
    Config c{RB, TB, L};
    c.wires = true;
    FusedProgram prog;
    const int K = RB + TB;
    KnownZeros z = known_start(n, identity, K);
    std::fill(stats, stats + 3, 0);
    zc* v = reinterpret_cast<zc*>(vec);
    auto rest = [&]() {
      for (uint64_t i = 0; z.fixed && i < 1ull << n; ++i) {
        const bool zero = ((z.sh ? i ^ (i >> z.sh) : i) & z.fixed) != 0;
        if (zero || z.fresh) v[i] = zero ? 0.0 : 1.0;
      }
      z = KnownZeros();
    };
    auto chunk = [&](const FusedProgram& sub, int) -> int {
      for (const PassHdr& H : sub.hdrs) {
        const PassStart S = enter_pass(z, H, K, std::max(n, K));
        ++stats[0];
        stats[1] += S.fixed ? 1ll << __builtin_popcountll(S.free) : n > K ? 1ll << (n - K) : 1;
        stats[2] += n > K ? 1ll << (n - K) : 1;
        wire_pass(v, n, RB, TB, (uint32_t)amp_bytes, H, sub.ops.data() + H.op0, sub.coef.data() + 2 * (size_t)H.coef0,
                  sub.aux.data(), S);
      }
      return 0;
    };
    auto single = [&](const qs_gate& g) -> int {
      rest();
      return cpu_apply_gates(vec, n, &g, 1, 1);
    };
    const int rc = build_streamed(gates, ngates, n, c, (uint32_t)amp_bytes, prog, chunk, single);
    rest();
    return rc;
  } catch (const std::exception& e) {
    g_err = e.what();
    return -99;
  }
}

// Energy-gradient sweep of a variational circuit: psi runs the planned circuit from
// |0...0>, lam = Z on index bit zbit of it, both run the planned inverse.  ops: axis,
// bit, slot per gate and, for fixed gates, records g and their inverses inv.
// grads[slot] receives Im <lam|P|psi> summed over the gates of the slot; psi the
// state swept back to |0...0>; fwd the forward state (up to a phase).  stats: forward
// and backward passes.
extern "C" int wires_gradient(int n, int nops, const int* axis, const int* bit, const int* slot, const qs_gate* g,
                              const qs_gate* inv, const double* theta, int zbit, int amp_bytes, double* fwd,
                              double* psi_out, double* grads, int* stats) {
  using namespace qs;
  try {
    Config c{4, 8, 4};
    c.wires = true;
    std::vector<VarOp> ops(nops);
    for (int i = 0; i < nops; ++i) {
      ops[i].axis = axis[i], ops[i].bit = bit[i], ops[i].slot = slot[i];
      if (axis[i] < 0) ops[i].g = g[i], ops[i].inv = inv[i];
    }
    const uint64_t N = 1ull << n;
    std::vector<zc> psi(N), lam(N);
    psi[0] = 1.0;
    for (int back = 0; back < 2; ++back) {
      FusedProgram prog;
      const int rc = build_var(ops, back, n, c, (uint32_t)amp_bytes, prog);
      if (rc) return rc;
      const int rc2 = check_passes(prog, c, 0, (int)prog.hdrs.size());
      if (rc2) return rc2;
      stats[back] = (int)prog.hdrs.size();
      for (size_t h = 0; h < prog.hdrs.size(); ++h) {
        PassHdr& H = prog.hdrs[h];
        for (int i = 0; i < H.nops; ++i) {
          FOp& o = prog.ops[H.op0 + i];
          if (!o.sym) continue;
          const double t = theta[o.sym - 1];
          double* p = &prog.coef[2 * (size_t)(H.coef0 + o.coef)];
          if (o.kind == F_ROT) rot_payload(std::cos(t / 2), std::sin(t / 2), o.sgn, p);
          else o.pure = phase_payload_sym(std::cos(t), std::sin(t), o.sgn, p);
        }
        std::vector<double> cols(H.ngrad, 0.0);
        const FOp* P = prog.ops.data() + H.op0;
        const double* C = prog.coef.data() + 2 * (size_t)H.coef0;
        if (!back) {
          wire_pass(psi.data(), n, 4, 8, (uint32_t)amp_bytes, H, P, C, prog.aux.data());
        } else {
          // run both vectors op by op up to each measurement: as passes that stop there
          std::vector<zc> a = psi, b = lam;
          for (int i = 0; i <= H.nops; ++i) {
            if (i < H.nops && P[i].kind != F_MEAS) continue;
            if (i == H.nops) break;
            std::vector<zc> x = psi, y = lam;
            PassHdr S = H;  // the ops before i, stored where the layout stands (register bit pos[0] known)
            std::vector<FOp> pre;
            for (int k = 0; k < i; ++k)
              if (P[k].kind != F_MEAS) pre.push_back(P[k]);
            S.nops = (int)pre.size();
            // store register r, thread t at the tile-local index (r | t << RB)
            for (int q = 0; q < 4; ++q) S.sr[q] = 1ull << H.sorted[q];
            for (int q = 0; q < 8; ++q) S.st[q] = 1ull << H.sorted[4 + q];
            S.sflip = 0, S.nsx = 0;
            wire_pass(x.data(), n, 4, 8, (uint32_t)amp_bytes, S, pre.data(), C, prog.aux.data());
            wire_pass(y.data(), n, 4, 8, (uint32_t)amp_bytes, S, pre.data(), C, prog.aux.data());
            const uint64_t m = 1ull << H.sorted[P[i].pos[0]];
            double s = 0;
            for (uint64_t k = 0; k < N; ++k) {
              const zc z = P[i].pure ? ((k & m) ? zc(0, 1) : zc(0, -1)) * x[k ^ m] : ((k & m) ? -1.0 : 1.0) * x[k];
              s += (std::conj(y[k]) * z).imag();
            }
            if (P[i].coef >= H.ngrad) throw std::runtime_error("gradient column out of range");
            cols[P[i].coef] += s;
          }
          std::vector<FOp> all;
          for (int k = 0; k < H.nops; ++k)
            if (P[k].kind != F_MEAS) all.push_back(P[k]);
          PassHdr S = H;
          S.nops = (int)all.size();
          wire_pass(psi.data(), n, 4, 8, (uint32_t)amp_bytes, S, all.data(), C, prog.aux.data());
          wire_pass(lam.data(), n, 4, 8, (uint32_t)amp_bytes, S, all.data(), C, prog.aux.data());
          for (int k = 0; k < H.ngrad; ++k) grads[prog.gcols[h][k].slot] += prog.gcols[h][k].sgn * cols[k];
        }
      }
      if (!back) {
        std::memcpy(fwd, psi.data(), N * sizeof(zc));
        for (uint64_t k = 0; k < N; ++k) lam[k] = ((k >> zbit) & 1) ? -psi[k] : psi[k];
      }
    }
    std::memcpy(psi_out, psi.data(), N * sizeof(zc));
    return 0;
  } catch (const std::exception& e) {
    g_err = e.what();
    return -99;
  }
}
