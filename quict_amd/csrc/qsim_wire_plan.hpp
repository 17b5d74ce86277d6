// Pass planner in wires.  Included by qsim_fused_plan.hpp.
//
// plan_groups (qsim_fused_plan.hpp) wants every bit of a gate in the tile.  Only
// the bits a gate MIXES have to be there: a control or a diagonal bit outside
// the tile is constant over a tile, so it selects whether the tile's workgroup
// runs the op at all.  And a SWAP or an X needs no pass: it renames what the
// later gates act on.  So the circuit is first reduced to gates on "wires"
// (reduce_gates):
//   * uncontrolled SWAPs exchange the wires two circuit bits stand for; each wire
//     ends on the index bit its circuit bit has at the end (`home`);
//   * uncontrolled X / Y become a flip of the wire's frame: later gates are
//     conjugated (a CX with a flipped control also flips the target's frame), and
//     what is left is one X at the end, which joins the wire's last gate or is a
//     flip of a store address;
//   * every diagonal gate on one or two targets (of modulus 1) becomes phases "all these bits
//     are 1: times f" (Rz, S, T, CZ, CRz, Rzz, ...), their common factors one
//     number for the whole program;
//   * one-qubit gates on a wire are multiplied together, past phases that
//     commute with them.
// plan_wires then picks each pass's tile wires, by how many more gates each
// further wire lets run, and every store moves the wires that the next tile
// shares with this one onto the low index bits and the others home where their
// home lies in the tile.
//
// Measured on MI355X against plan_groups and k_fused: the 30-qubit complex128
// 2000-gate 60/40 circuit 556 ms in 73 passes, 191 ms in 23 (157 with known zeros and
// joined ops); 8 layers of the hardware-efficient ansatz on 25 qubits, complex64, 4.98
// ms in 23 passes, 2.70 ms in 8 (1.71); the matrix of a 300-gate 13-qubit circuit 3.84
// against 2.09 ms (1.5); 400 gates on 20 qubits as a captured graph 295 against 193 us
// (118).  Against 80-bit arithmetic the state is closer than the per-gate kernels' (838
// gates on 13 qubits: 2e-15 against 1.2e-14): a factored gate is unitary to the last
// bit, a rounded matrix is not, and a split that does not give the matrix back to that
// rounding is not taken.
//
// schedule_wires turns one pass into ops.  A CX is a GF(2)-linear map of the
// index, so it needs no arithmetic at all when it is left to the addresses of
// the next relayout or of the store: the scheduler keeps the map `A` (logical
// bit j = parity of the base bits in row j, XOR a constant, XOR bits of the tile
// number) and clears it at each relayout.
#pragma once

#include <cmath>

namespace qs {

struct WireProgram {
  std::vector<qs_gate> g;     // bits[] hold wires
  std::vector<char> single;   // a gate the tile kernel cannot take: a pass of its own
  std::vector<int> home;      // wire -> index bit its amplitudes end on
  std::vector<WireSym> sym;   // parallel to g
};

// What the scheduler and the grouping need to know of a gate.
enum WClass : uint8_t { W_REAL, W_PHASE, W_CX, W_FLIP, W_TABLE, W_SINGLE, W_ZMEAS /* phase that is measured */ };

static bool pure_exchange(const qs_gate& g) { return g.m[0] == 1.0 && g.m[1] == 0.0 && g.m[2] == 1.0 && g.m[3] == 0.0; }

static WClass wire_class(const qs_gate& g, bool single, const WireSym& sym) {
  if (single) return W_SINGLE;
  if (g.kind == QS_GATE_PHASE && sym.meas != 0.0) return W_ZMEAS;
  if (g.kind == QS_GATE_PHASE) return W_PHASE;
  if (g.kind == QS_GATE_DIAG) return W_TABLE;
  if (g.kind == QS_GATE_XPERM && g.ncontrols == 0 && pure_exchange(g)) return W_FLIP;
  if (g.kind == QS_GATE_XPERM && g.ncontrols == 1 && pure_exchange(g)) return W_CX;
  return W_REAL;
}

static cplx cdiv_(cplx a, cplx b) {
  const double d = b.first * b.first + b.second * b.second;
  return {(a.first * b.first + a.second * b.second) / d, (a.second * b.first - a.first * b.second) / d};
}

// Whether f may be taken out of a gate as a common factor and divided by.  Entries far
// from modulus 1 stay in their gate: a program's common factor, or the reciprocal of
// one, would leave the range of its precision where no amplitude does.
static bool near_unit(cplx f) { return std::fabs(f.first * f.first + f.second * f.second - 1.0) <= 2e-5; }

struct WireReducer {
  const Config& c;
  WireProgram& W;
  std::vector<char> dead;
  int lab[64];       // circuit bit -> wire
  uint64_t F = 0;    // frame flips: logical value = frame value ^ F
  int last1[64];     // the last one-qubit gate on a wire that further ones may join, or -1
  char touched[64];  // 1: gates diagonal on the wire came after it
  int lastt[64];     // the last gate touching the wire, or -1
  cplx gphase{1.0, 0.0};
  bool keep_phase = true;  // false: the state is wanted up to a common phase

  WireReducer(const Config& cfg, WireProgram& w, int n) : c(cfg), W(w) {
    for (int b = 0; b < 64; ++b) lab[b] = b, last1[b] = -1, touched[b] = 0, lastt[b] = -1;
    W.home.resize(n);
  }

  // Append a gate (bits already wires) and note which wires it touches.
  int put(const qs_gate& g, bool single = false, const WireSym& sym = {}) {
    const int id = (int)W.g.size();
    W.g.push_back(g);
    W.sym.push_back(sym);
    W.single.push_back(single);
    dead.push_back(0);
    const bool diag = !single && gate_diag_like(g);
    for (int i = 0; i < g.ncontrols + g.ntargets; ++i) {
      const int w = g.bits[i];
      lastt[w] = id;
      if (diag || (!single && i < g.ncontrols)) touched[w] = 1;
      else last1[w] = -1;
    }
    return id;
  }

  // One-qubit gate with frame matrix M (row-major) on wire w; diag: a phase (1, f).
  void one_qubit(int w, const double* M, bool diag) {
    const int k = last1[w];
    if (k >= 0) {
      qs_gate& e = W.g[k];
      const bool ediag = e.kind == QS_GATE_PHASE;
      if (!touched[w] || diag || ediag) {
        double B[8], P[8];
        if (ediag) {
          const double d2[4] = {1.0, 0.0, e.m[0], e.m[1]};
          diag_to_dense1(d2, B);
        } else {
          std::memcpy(B, e.m, sizeof(B));
        }
        mat2_mul(M, B, P);
        if (touched[w] && !diag) {
          // a dense gate after phases that share the wire with the waiting phase
          // e: e commutes with them and joins the new gate
          dead[k] = 1;
        } else if (diag && ediag) {
          e.m[0] = P[6], e.m[1] = P[7];
          return;
        } else {
          e.kind = QS_GATE_DENSE;
          std::memset(e.m, 0, sizeof(e.m));
          std::memcpy(e.m, P, sizeof(P));
          return;
        }
        put_one(w, P, false);
        return;
      }
    }
    put_one(w, M, diag);
  }
  void put_one(int w, const double* M, bool diag) {
    qs_gate g;
    std::memset(&g, 0, sizeof(g));
    g.kind = diag ? QS_GATE_PHASE : QS_GATE_DENSE;
    g.ntargets = 1;
    g.bits[0] = w;
    if (diag) g.m[0] = M[6], g.m[1] = M[7];
    else std::memcpy(g.m, M, 8 * sizeof(double));
    last1[w] = put(g);
    touched[w] = 0;
  }

  // Amplitudes whose k bits (circuit-frame wires ws) are all 1, times f.
  void phase(const int* ws, int k, cplx f) {
    if (f.first == 1.0 && f.second == 0.0) return;
    if (k == 0) {
      gphase = cm_(gphase, f);
      return;
    }
    int flipped = 0;
    for (int i = 0; i < k; ++i) flipped += (F >> ws[i]) & 1;
    // Every flipped bit splits the phase in two (below): from two of them on, on more
    // than two bits (whose parts join what is on their wires), the flips become gates.
    const bool split = flipped && (flipped == 1 || k <= 2) && near_unit(f);
    for (int i = 0; i < k; ++i) {
      if (!((F >> ws[i]) & 1)) continue;
      if (!split) {
        materialize(ws[i]);
        continue;
      }
      // bit i is 1 where the frame bit is 0: f where the others are 1, undone
      // where the frame bit is 1 too
      int rest[QS_MAX_GATE_BITS];
      int r = 0;
      for (int j = 0; j < k; ++j)
        if (j != i) rest[r++] = ws[j];
      const uint64_t F0 = F;
      phase(rest, r, f);
      F &= ~(1ull << ws[i]);
      phase(ws, k, cdiv_({1.0, 0.0}, f));
      F = F0;
      return;
    }
    if (k == 1) {
      const double M[8] = {1, 0, 0, 0, 0, 0, f.first, f.second};
      one_qubit(ws[0], M, true);
      return;
    }
    if (k == 2 && lastt[ws[0]] >= 0 && lastt[ws[0]] == lastt[ws[1]] && !dead[lastt[ws[0]]]) {
      qs_gate& e = W.g[lastt[ws[0]]];
      if (e.kind == QS_GATE_PHASE && e.ncontrols + e.ntargets == 2) {
        const cplx p = cm_(f, {e.m[0], e.m[1]});
        e.m[0] = p.first, e.m[1] = p.second;
        return;
      }
    }
    qs_gate g;
    std::memset(&g, 0, sizeof(g));
    g.kind = QS_GATE_PHASE;
    g.ncontrols = k - 1;
    g.ntargets = 1;
    for (int i = 0; i < k; ++i) g.bits[i] = ws[i];
    g.m[0] = f.first, g.m[1] = f.second;
    put(g);
  }

  // exp(-i sgn theta[slot] P / 2), P = X, Y, Z (axis 0, 1, 2) on a circuit bit, up to
  // a common phase; meas: Im <lam|P|psi> is taken before it.
  void param(int axis, int bit, int slot, double sgn, bool meas) {
    const int w = lab[bit];
    const double flip = ((F >> w) & 1) && axis != 0 ? -1.0 : 1.0;  // X Y X = -Y, X Z X = -Z
    qs_gate g;
    std::memset(&g, 0, sizeof(g));
    g.ntargets = 1;
    g.bits[0] = w;
    g.kind = axis == 2 ? QS_GATE_PHASE : QS_GATE_DENSE;
    WireSym s;
    s.slot = slot;
    s.sgn = sgn * flip;
    s.meas = meas ? flip : 0.0;
    const double P[8] = {1, 0, 0, 0, 0, 0, 0, 1}, Q[8] = {1, 0, 0, 0, 0, 0, 0, -1};
    if (axis == 0) one_qubit(w, P, true);  // X = S^dagger Y S
    put(g, false, s);
    if (axis == 0) one_qubit(w, Q, true);
  }

  // Turn a frame flip into an X gate.
  void materialize(int w) {
    if (!((F >> w) & 1)) return;
    F &= ~(1ull << w);
    const double X[8] = {0, 0, 1, 0, 1, 0, 0, 0};
    if (last1[w] >= 0 && !touched[w]) {
      one_qubit(w, X, false);
      return;
    }
    qs_gate g;
    std::memset(&g, 0, sizeof(g));
    g.kind = QS_GATE_XPERM;
    g.ntargets = 1;
    g.bits[0] = w;
    g.m[0] = g.m[2] = 1.0;
    put(g);
  }

  void add(const qs_gate& gin) {
    const int nc = gin.ncontrols, nt = gin.ntargets;
    if (gin.kind == QS_GATE_SWAP && nc == 0) {
      std::swap(lab[gin.bits[0]], lab[gin.bits[1]]);
      if (!pure_exchange(gin)) {  // the phases of an exchange: diag(1, m0, m1, 1) after it
        qs_gate d;
        std::memset(&d, 0, sizeof(d));
        d.kind = QS_GATE_DIAG;
        d.ntargets = 2;
        d.bits[0] = gin.bits[0], d.bits[1] = gin.bits[1];
        d.m[0] = 1.0;
        for (int i = 0; i < 4; ++i) d.m[2 + i] = gin.m[i];
        d.m[6] = 1.0;
        add(d);
      }
      return;
    }
    qs_gate g = gin;
    for (int i = 0; i < nc + nt; ++i) g.bits[i] = lab[gin.bits[i]];
    const int* w = g.bits;
    auto entry = [&](int i) { return cplx{g.m[2 * i], g.m[2 * i + 1]}; };
    auto zero = [&](int i) { return g.m[2 * i] == 0.0 && g.m[2 * i + 1] == 0.0; };
    auto unit = [&](int i) { return near_unit(entry(i)); };
    if (g.kind == QS_GATE_XPERM && nc <= 1 && (pure_exchange(g) || (unit(0) && !zero(1)))) {
      const int t = w[nc];
      if (nc == 0) {
        F ^= 1ull << t;
      } else {
        qs_gate x = g;
        std::memset(x.m, 0, sizeof(x.m));
        x.m[0] = x.m[2] = 1.0;
        put(x);
        if ((F >> w[0]) & 1) F ^= 1ull << t;
      }
      if (!pure_exchange(g)) {  // then diag(m0, m1) on the target under the control
        phase(w, nc, entry(0));
        phase(w, nc + 1, cdiv_(entry(1), entry(0)));
      }
      return;
    }
    if (g.kind == QS_GATE_PHASE) {
      phase(w, nc + nt, entry(0));
      return;
    }
    if (g.kind == QS_GATE_DIAG && nt == 1 && unit(0)) {
      phase(w, nc, entry(0));
      phase(w, nc + 1, cdiv_(entry(1), entry(0)));
      return;
    }
    if (g.kind == QS_GATE_DIAG && nt == 2 && unit(0) && unit(1) && unit(2)) {
      int a[QS_MAX_GATE_BITS];
      for (int i = 0; i < nc; ++i) a[i] = w[i];
      phase(a, nc, entry(0));
      a[nc] = w[nc];
      phase(a, nc + 1, cdiv_(entry(2), entry(0)));
      a[nc] = w[nc + 1];
      phase(a, nc + 1, cdiv_(entry(1), entry(0)));
      phase(w, nc + 2, cdiv_(cm_(entry(3), entry(0)), cm_(entry(1), entry(2))));
      return;
    }
    const bool dense = g.kind == QS_GATE_DENSE;
    if (dense && nt <= 2) {
      for (int i = 0; i < nc; ++i) materialize(w[i]);
      std::vector<double> M(g.m, g.m + (2 << (2 * nt)));
      int x = 0;
      for (int i = 0; i < nt; ++i)
        if ((F >> w[nc + i]) & 1) x |= 1 << (nt - 1 - i);
      xor_conjugate(M, nt, x);
      if (nt == 1 && nc == 0) {
        one_qubit(w[0], M.data(), false);
        return;
      }
      std::copy(M.begin(), M.end(), g.m);
      put(g);
      return;
    }
    for (int i = 0; i < nc + nt; ++i) materialize(w[i]);
    put(g, (dense && nt > std::min(4, c.RB)) || (g.kind == QS_GATE_DIAG && nc + nt > c.RB + 2));
  }

  // After the last gate.  A unitary one-qubit gate becomes
  //   factor * phase(a) * [[c, -s], [s, c]] * phase(b),   c >= 0:
  // the rotation is 3 multiply-adds per component pair in the tile kernel where
  // the complex 2x2 is 8, and the phases wait on their wire, past everything
  // diagonal there, and join the next gate's (or precede the next mixing one).
  void finish(int n, double tol) {
    for (int w = 0; w < n; ++w) materialize(w);
    for (int b = 0; b < n; ++b) W.home[lab[b]] = b;
    std::vector<qs_gate> in;
    std::vector<char> ins;
    std::vector<WireSym> insym;
    in.swap(W.g);
    ins.swap(W.single);
    insym.swap(W.sym);
    W.g.reserve(in.size() + 16);
    cplx pend[64];
    for (int w = 0; w < 64; ++w) pend[w] = {1.0, 0.0};
    const double eps = 5e-16;  // rounding of the factors: not an op
    auto is_one = [&](cplx f) { return std::fabs(f.first - 1.0) <= eps && std::fabs(f.second) <= eps; };
    auto push = [&](const qs_gate& g, bool single, const WireSym& sym = {}) {
      W.g.push_back(g);
      W.single.push_back(single);
      W.sym.push_back(sym);
    };
    auto flush = [&](int w) {
      if (!is_one(pend[w])) {
        qs_gate g;
        std::memset(&g, 0, sizeof(g));
        g.kind = QS_GATE_PHASE;
        g.ntargets = 1;
        g.bits[0] = w;
        g.m[0] = pend[w].first, g.m[1] = pend[w].second;
        push(g, false);
      }
      pend[w] = {1.0, 0.0};
    };
    for (size_t k = 0; k < in.size(); ++k) {
      if (dead[k]) continue;
      const qs_gate& g = in[k];
      const int nb = g.ncontrols + g.ntargets;
      if (insym[k].slot >= 0) {
        if (g.kind == QS_GATE_DENSE) flush(g.bits[0]);
        push(g, false, insym[k]);
        continue;
      }
      if (!ins[k] && g.kind == QS_GATE_PHASE && nb == 1) {
        pend[g.bits[0]] = cm_(pend[g.bits[0]], {g.m[0], g.m[1]});
        continue;
      }
      if (!ins[k] && g.kind == QS_GATE_DENSE && g.ncontrols == 0 && g.ntargets == 1) {
        const int w = g.bits[0];
        cplx f, pa, pb;
        double c_, s_;
        if (factor(g.m, tol, f, pa, pb, c_, s_)) {
          gphase = cm_(gphase, f);
          pend[w] = cm_(pb, pend[w]);
          if (s_ != 0.0) {
            flush(w);
            qs_gate r = g;
            std::memset(r.m, 0, sizeof(r.m));
            r.m[0] = r.m[6] = c_;
            r.m[2] = -s_;
            r.m[4] = s_;
            push(r, false);
          }
          pend[w] = cm_(pa, pend[w]);
          continue;
        }
      }
      if (ins[k] || !gate_diag_like(g))
        for (int i = ins[k] ? 0 : g.ncontrols; i < nb; ++i) flush(g.bits[i]);
      push(g, ins[k]);
    }
    for (int w = 0; w < n; ++w) flush(w);
    if (keep_phase && !is_one(gphase)) {  // the common factor multiplies whole tiles, in one pass
      qs_gate g;
      std::memset(&g, 0, sizeof(g));
      g.kind = QS_GATE_PHASE;
      g.m[0] = gphase.first, g.m[1] = gphase.second;
      push(g, false);
    }
  }

  // m = f diag(1, pa) [[c, -s], [s, c]] diag(1, pb); false if no such product gives m to
  // tol.  Three of the four entries' phases fix f, pa and pb: the larger two are among
  // them.  (Where gates on a wire cancel, the smaller two are rounding, and the phase of
  // a rounding error would go into a large entry.)
  static bool factor(const double* m, double tol, cplx& f, cplx& pa, cplx& pb, double& c_, double& s_) {
    auto e = [&](int i) { return cplx{m[2 * i], m[2 * i + 1]}; };
    auto mag = [](cplx z) { return std::hypot(z.first, z.second); };
    auto unit = [&](cplx z) {
      const double r = mag(z);
      return cplx{z.first / r, z.second / r};
    };
    auto neg = [](cplx z) { return cplx{-z.first, -z.second}; };
    c_ = mag(e(0)), s_ = mag(e(2));
    const double h = std::hypot(c_, s_);
    if (!(std::fabs(h - 1.0) <= tol)) return false;
    c_ /= h, s_ /= h;
    f = c_ == 0.0 ? unit(e(2)) : unit(e(0));
    pa = s_ == 0.0 || c_ == 0.0 ? cplx{1.0, 0.0} : unit(cdiv_(e(2), f));
    if (s_ == 0.0) pa = unit(cdiv_(e(3), f)), pb = {1.0, 0.0};
    else if (c_ >= s_) pb = unit(cdiv_(e(3), cm_(f, pa)));
    else pb = neg(unit(cdiv_(e(1), f)));
    // (written so that a phase of a zero, which is not a number, fails)
    auto gives = [&](int i, cplx z, double r) {
      const double x = m[2 * i] - z.first * r, y = m[2 * i + 1] - z.second * r;
      return x * x + y * y <= tol * tol;
    };
    const cplx fa = cm_(f, pa);
    if (!(gives(0, f, c_) && gives(1, cm_(f, pb), -s_) && gives(2, fa, s_) && gives(3, cm_(fa, pb), c_))) return false;
    // s may have either sign: the one that leaves a factor at 1, else any
    const double d = 1e-15;
    auto neg_one = [&](cplx z) { return std::fabs(z.first + 1.0) <= d && std::fabs(z.second) <= d; };
    if (s_ != 0.0 && c_ != 0.0 && (neg_one(pa) || neg_one(pb))) {
      s_ = -s_;
      pa = neg(pa);
      pb = neg(pb);
    }
    return true;
  }
};

// ---- one pass -------------------------------------------------------------------

// A gate of the pass on tile-local bits.
struct LocalGate {
  int idx;                 // gate index in the program
  WClass cls;
  uint32_t all, mix;       // its bits in the tile; those it mixes
  uint32_t ctl;            // controls in the tile (real gates)
  uint32_t outer;          // tile-number bits (all must be 1)
  std::vector<int> loc;    // bit i of the gate -> tile-local bit, or -1
};

// Payload of a phase f: real, unit (shears, with or without a minus sign) or any.
static void phase_payload(cplx f, double tol, OpBuild& ob) {
  const double r = std::hypot(f.first, f.second);
  if (f.second == 0.0) {
    ob.op.pure = 1;
    ob.coef = {f.first, 0.0};
  } else if (std::fabs(r - 1.0) <= tol) {
    const double sg = f.first < 0.0 ? -1.0 : 1.0;
    const double re = sg * f.first / r, im = sg * f.second / r;
    ob.op.pure = f.first < 0.0 ? 3 : 2;
    ob.coef = {-im / (1.0 + re), im};
  } else {
    ob.op.pure = 0;
    ob.coef = {f.first, f.second};
  }
}

// How far from unitary a gate may be and still be run as a rotation and phases:
// rounding of its matrix (gates of single-precision circuits come rounded to float).
static double unit_tolerance(uint32_t amp_bytes) { return amp_bytes == 16 ? 1e-14 : 1e-6; }

// Schedules gates (prog.pgates, on index bits) of pass p.  allowed: tile-local bits
// that may go to the low index bits at the store (at least L of them); home[j]:
// the index bit where tile-local bit j ends, to be taken where it is free.
static int schedule_wires(const std::vector<WClass>& cls, PassPlan& p, const Config& c, uint32_t amp_bytes,
                          uint32_t allowed, const std::vector<int>& home, PassHdr& H, FusedProgram& prog,
                          std::vector<GradCol>& gcols) {
  const int RB = c.RB, TB = c.TB, K = RB + TB, L = c.L, NR = 1 << RB;
  const uint32_t full = (1u << K) - 1;
  const double tol = unit_tolerance(amp_bytes);
  std::memset(&H, 0, sizeof(H));
  int g2l[64], g2o[64];
  {
    for (int b = 0; b < 64; ++b) g2l[b] = -1, g2o[b] = -1;
    for (int j = 0; j < K; ++j) {
      H.tbits[j] = H.sorted[j] = p.tbits[j];
      g2l[p.tbits[j]] = j;
    }
    int o = 0;
    for (int b = 0; b < 64; ++b)
      if (g2l[b] < 0) g2o[b] = o++;
  }
  std::vector<LocalGate> rem;
  rem.reserve(p.gates.size());
  for (int gi : p.gates) {
    const qs_gate& g = prog.pgates[gi];
    LocalGate l;
    l.idx = gi;
    l.cls = cls[gi];
    l.all = l.mix = l.ctl = l.outer = 0;
    const int nb = g.ncontrols + g.ntargets;
    const bool diag = l.cls == W_PHASE || l.cls == W_TABLE || l.cls == W_ZMEAS;
    l.loc.resize(nb);
    for (int i = 0; i < nb; ++i) {
      const int j = g2l[g.bits[i]];
      l.loc[i] = j;
      if (j < 0) {
        l.outer |= 1u << g2o[g.bits[i]];
        continue;
      }
      l.all |= 1u << j;
      if (!diag) (i < g.ncontrols ? l.ctl : l.mix) |= 1u << j;
    }
    rem.push_back(std::move(l));
  }
  // lanes in the order of the bits the store may write to the low index bits
  std::vector<int> tord;
  for (int j = 0; j < K; ++j)
    if ((allowed >> j) & 1) tord.push_back(j);
  for (int j = 0; j < K; ++j)
    if (!((allowed >> j) & 1)) tord.push_back(j);

  // the linear map of the layout: logical bit j = parity of base bits A[j] ^ aff ^ (tile-number bits outx[j])
  uint32_t A[32], outx[32], aff = 0;
  int cols[32];  // rows that contain base bit j
  auto reset_map = [&]() {
    for (int j = 0; j < K; ++j) A[j] = 1u << j, outx[j] = 0, cols[j] = 1;
    aff = 0;
  };
  reset_map();
  auto row_clean = [&](int j) { return A[j] == (1u << j) && outx[j] == 0; };
  auto mask_row_clean = [&](uint32_t m) {
    for (; m; m &= m - 1)
      if (!row_clean(__builtin_ctz(m))) return false;
    return true;
  };
  auto mask_mix_clean = [&](uint32_t m) {
    for (; m; m &= m - 1) {
      const int j = __builtin_ctz(m);
      if (!row_clean(j) || cols[j] != 1) return false;
    }
    return true;
  };

  Layout cur;
  uint32_t regs = 0;  // register bits of cur
  std::vector<Built> built;
  auto set_flips = [&]() {  // flips of the slots as build_op sees them
    cur.flip = 0;
    for (uint32_t m = aff; m; m &= m - 1) cur.flip |= 1u << slot_of(cur, __builtin_ctz(m));
  };
  auto add_op = [&](OpBuild& ob, const LocalGate& l) {
    Built b;
    b.op = ob.op;
    b.coef = std::move(ob.coef);
    b.op.cblk = b.op.cblkv = l.outer;
    for (uint32_t m = l.all; m; m &= m - 1) b.slots |= 1u << slot_of(cur, __builtin_ctz(m));
    if (b.op.kind == F_DIAG)
      for (int k = 0; k < b.op.ntt; ++k) b.selp.push_back(b.op.tpos[k]);
    const bool two = b.op.kind == F_DENSE2 || b.op.kind == F_XX2 || b.op.kind == F_DIAG;
    if (l.outer != 0 || !two || !try_merge(built, b, NR, RB)) built.push_back(std::move(b));
  };
  // Gradient column before a measured gate, its sign with the wire's pending flip.
  auto emit_meas = [&](const LocalGate& l, int y) {
    const WireSym& sym = prog.psym[l.idx];
    Built b;
    std::memset(&b.op, 0, sizeof(b.op));
    b.op.kind = F_MEAS;
    b.op.pure = y;
    b.op.pos[0] = slot_of(cur, __builtin_ctz(l.all));
    b.op.coef = (int)gcols.size();
    b.slots = 1u << b.op.pos[0];
    gcols.push_back({sym.slot, (l.all & aff) ? -sym.meas : sym.meas});
    built.push_back(std::move(b));
  };
  auto emit_phase = [&](const LocalGate& l) {
    const qs_gate& g = prog.pgates[l.idx];
    const WireSym& sym = prog.psym[l.idx];
    OpBuild ob;
    std::memset(&ob.op, 0, sizeof(ob.op));
    ob.op.kind = F_PHASE;
    if (sym.slot >= 0) {
      ob.op.sym = 1 + sym.slot;
      ob.op.sgn = (l.all & aff) ? -sym.sgn : sym.sgn;
      ob.op.pure = 2;
      ob.coef = {0.0, 0.0};
    } else {
      phase_payload({g.m[0], g.m[1]}, tol, ob);
    }
    for (uint32_t m = l.all; m; m &= m - 1) {
      const int s = slot_of(cur, __builtin_ctz(m));
      if (s < RB) ob.op.creg |= 1u << s;
      else ob.op.cthr |= 1u << (s - RB);
    }
    ob.op.cregv = ob.op.creg;
    ob.op.cthrv = ob.op.cthr;
    add_op(ob, l);
  };
  auto emit_gate = [&](const LocalGate& l) -> int {
    // controls outside the tile are the op's tile predicate: drop them here
    const qs_gate& g = prog.pgates[l.idx];
    const WireSym& sym = prog.psym[l.idx];
    OpBuild ob;
    if (sym.slot >= 0) {  // rotation about Y
      if (sym.meas != 0.0) emit_meas(l, 1);
      std::memset(&ob.op, 0, sizeof(ob.op));
      ob.op.kind = F_ROT;
      ob.op.npos = 1;
      ob.op.pos[0] = slot_of(cur, __builtin_ctz(l.mix));
      ob.op.sym = 1 + sym.slot;
      ob.op.sgn = (l.all & aff) ? -sym.sgn : sym.sgn;
      ob.coef = {0.0, 0.0};
      add_op(ob, l);
      return QS_OK;
    }
    set_flips();
    int rc;
    if (l.outer == 0) {
      rc = build_op(g, l.loc, cur, NR, ob);
    } else {
      qs_gate in = g;
      std::vector<int> loc;
      in.ncontrols = 0;
      for (int i = 0; i < g.ncontrols + g.ntargets; ++i)
        if (l.loc[i] >= 0) {
          in.bits[loc.size()] = g.bits[i];
          loc.push_back(l.loc[i]);
          in.ncontrols += i < g.ncontrols;
        }
      rc = build_op(in, loc, cur, NR, ob);
    }
    if (rc) {
      set_error("fusion planner produced an op the tile kernel cannot encode");
      return rc;
    }
    if (ob.op.kind == F_DENSE1 && uncontrolled_in_tile(ob.op)) {
      const std::vector<double>& m = ob.coef;
      const double cc = m[0], ss = m[4];
      if (m[1] == 0.0 && m[3] == 0.0 && m[5] == 0.0 && m[7] == 0.0 && m[6] == cc && m[2] == -ss && cc >= 0.0 &&
          std::fabs(cc * cc + ss * ss - 1.0) <= 1e-12) {
        ob.op.kind = F_ROT;
        ob.coef = {-ss / (1.0 + cc), ss};
      }
    }
    add_op(ob, l);
    return QS_OK;
  };

  // One scan over the remaining gates in order: those that commute with every
  // gate still waiting and can run in the present layout run now.  `last`: the
  // waiting phases run whatever their slots.
  int scan_rc = QS_OK;
  auto scan = [&](bool last) -> bool {
    const size_t G = rem.size();
    // what the gates after k use and mix (whether a CX's bits are needed again here)
    std::vector<uint32_t> ua(G + 1, 0), um(G + 1, 0);
    for (size_t k = G; k-- > 0;) ua[k] = ua[k + 1] | rem[k].all, um[k] = um[k + 1] | rem[k].mix;
    uint32_t wa = 0, wm = 0;
    size_t o = 0;
    bool any = false;
    for (size_t k = 0; k < G; ++k) {
      LocalGate& l = rem[k];
      bool ran = false;
      if (!((l.all & wm) | (l.mix & wa)) && !scan_rc) {
        switch (l.cls) {
          case W_FLIP: {
            const int t = __builtin_ctz(l.mix);
            if (regs & l.mix) {  // a register bit keeps its value for the half-tile relayouts
              if (mask_mix_clean(l.mix)) scan_rc = emit_gate(l), ran = true;
            } else {
              aff ^= 1u << t;
              ran = true;
            }
            break;
          }
          case W_CX: {
            const int t = __builtin_ctz(l.mix);
            const bool in = l.ctl != 0;
            const bool t_reg = (regs & l.mix) != 0;
            const bool again = ((ua[k + 1] & l.mix) | (um[k + 1] & l.ctl)) != 0;
            const bool can = t_reg && mask_mix_clean(l.mix) && mask_row_clean(l.ctl);
            if (can && again) {
              scan_rc = emit_gate(l);
              ran = true;
              break;
            }
            if (t_reg) {  // one register bit has to stay as it is for the half-tile relayouts
              int clean = 0;
              for (int b : cur.rs) clean += b != t && row_clean(b);
              if (!clean) {
                if (can) scan_rc = emit_gate(l), ran = true;
                break;
              }
            }
            if (in) {
              const int cb = __builtin_ctz(l.ctl);
              A[t] ^= A[cb];
              for (int b = 0; b < K; ++b)
                if ((A[cb] >> b) & 1) cols[b] += ((A[t] >> b) & 1) ? 1 : -1;
              outx[t] ^= outx[cb];
              aff ^= ((aff >> cb) & 1u) << t;
            } else {
              outx[t] ^= l.outer;
            }
            ran = true;
            break;
          }
          case W_PHASE:
            if ((last || (l.all & regs)) && !(l.all & aff) && mask_row_clean(l.all)) emit_phase(l), ran = true;
            break;
          case W_ZMEAS:
            if (!(l.all & ~regs) && mask_row_clean(l.all)) emit_meas(l, 0), emit_phase(l), ran = true;
            break;
          case W_TABLE:
            if (__builtin_popcount(l.all & ~regs) <= 2 && mask_row_clean(l.all)) scan_rc = emit_gate(l), ran = true;
            break;
          default:
            if (!(l.mix & ~regs) && mask_mix_clean(l.mix) && mask_row_clean(l.ctl)) scan_rc = emit_gate(l), ran = true;
        }
      }
      if (ran) {
        any = true;
        continue;
      }
      wa |= l.all;
      wm |= l.mix;
      if (o != k) rem[o] = std::move(l);
      ++o;
    }
    rem.resize(o);
    return any;
  };

  // What would run with the registers `R`: gates that need register bits count
  // most; an exchange can wait for phases that need one of their bits there.
  auto simulate = [&](uint32_t R) -> int {
    uint32_t wa = 0, wm = 0, dm = 0, dv = 0;
    int score = 0;
    for (const LocalGate& l : rem) {
      bool ran = false;
      if (!((l.all & wm) | (l.mix & wa))) {
        switch (l.cls) {
          case W_FLIP:
            ran = true;
            ++score;
            break;
          case W_CX:
            ++score;
            if (!((R & l.mix) && !(l.mix & (dm | dv)) && !(l.ctl & dv))) dv |= l.mix, dm |= l.mix | l.ctl;
            ran = true;
            break;
          case W_PHASE:
            ran = (l.all & R) && !(l.all & dv);
            break;
          case W_ZMEAS:
            ran = !(l.all & ~R) && !(l.all & dv);
            if (ran) score += 4;
            break;
          case W_TABLE:
            ran = __builtin_popcount(l.all & ~R) <= 2 && !(l.all & dv);
            if (ran) score += 4;
            break;
          default:
            ran = !(l.mix & ~R) && !(l.mix & (dm | dv)) && !(l.ctl & dv);
            if (ran) score += 4;
        }
      }
      if (ran) continue;
      wa |= l.all;
      wm |= l.mix;
      if (wm == full) break;
    }
    return score;
  };
  // Register set for the next stretch: bits added one by one (or a gate's targets
  // together), each the one that lets most gates run.
  auto choose = [&](uint32_t banned) -> std::vector<int> {
    uint32_t R = 0;
    std::vector<int> out;
    auto take = [&](uint32_t m) {
      for (m &= ~R; m; m &= m - 1) out.push_back(__builtin_ctz(m));
    };
    int base = simulate(0);
    while ((int)out.size() < RB) {
      const int room = RB - (int)out.size();
      uint32_t best = 0;
      double best_gain = 0;
      uint32_t seen = 0, wa = 0, wm = 0;
      for (const LocalGate& l : rem) {
        // candidates: what the unblocked gates with missing register bits need
        if (!((l.all & wm) | (l.mix & wa))) {
          uint32_t need = 0;
          if (l.cls == W_ZMEAS) need = l.all & ~R;
          else if (l.cls != W_PHASE && l.cls != W_TABLE) need = l.mix & ~R;
          else if (l.cls == W_TABLE) {
            uint32_t m = l.all & ~R;
            for (int k = __builtin_popcount(m); k > 2; --k, m &= m - 1) need |= m & (~m + 1);
          }
          if (need && !(need & banned) && __builtin_popcount(need) <= room &&
              !(__builtin_popcount(need) == 1 && (seen & need))) {
            if (__builtin_popcount(need) == 1) seen |= need;
            const double gain = (double)(simulate(R | need) - base) / __builtin_popcount(need);
            if (gain > best_gain) best_gain = gain, best = need;
          }
          if (l.cls == W_PHASE || l.cls == W_CX || l.cls == W_FLIP || !need) continue;  // (a phase runs as soon as one of its bits is a register bit)
        }
        wa |= l.all;
        wm |= l.mix;
        if (wm == full) break;
      }
      if (!best) break;
      take(best);
      R |= best;
      base = simulate(R);
    }
    // room left: bits that later gates need first, then the present ones, then any
    for (const LocalGate& l : rem) {
      if ((int)out.size() >= RB) break;
      if (l.cls != W_REAL) continue;
      for (uint32_t m = l.mix & ~R & ~banned; m && (int)out.size() < RB; m &= m - 1) {
        out.push_back(__builtin_ctz(m));
        R |= m & (~m + 1);
      }
    }
    for (int pass = 0; pass < 2; ++pass)
      for (int j = K - 1; j >= 0 && (int)out.size() < RB; --j) {
        const uint32_t m = 1u << j;
        if ((R & m) || (banned & m) || (pass == 0 && ((allowed & m) || !(regs & m || !regs)))) continue;
        out.push_back(j);
        R |= m;
      }
    return out;
  };

  const uint32_t low_local = (1u << L) - 1;
  cur = make_layout(choose(low_local), K);
  auto note_regs = [&]() {
    regs = 0;
    for (int b : cur.rs) regs |= 1u << b;
  };
  note_regs();
  for (int b = 0; b < RB; ++b) H.rs0[b] = cur.rs[b];
  for (int b = 0; b < TB; ++b) H.ts0[b] = cur.ts[b];
  const int op_start = (int)prog.ops.size();
  const int coef_start = (int)(prog.coef.size() / 2);

  // Relayout through a half-tile LDS image (see RELAYOUT in qsim_fused_plan.hpp)
  // that also applies the pending linear map.  The bit h that splits it is a
  // register bit of both layouts whose value is its slot's.
  auto relayout_one = [&](std::vector<int> nr) {
    int q = -1;
    for (int flips = 0; flips < 2 && q < 0; ++flips)  // rather one without a pending flip
      for (int i = 0; i < RB && q < 0; ++i)
        if (index_in(nr, cur.rs[i]) >= 0 && row_clean(cur.rs[i]) && (flips || !((aff >> cur.rs[i]) & 1))) q = i;
    const int h = cur.rs[q];
    const uint32_t carry = aff & (1u << h);  // a flip of the slot stays with it
    std::swap(nr[index_in(nr, h)], nr[q]);
    Layout next = make_layout(nr, K, tord);
    // placement: the lanes one 128-byte LDS cycle serves (the first G thread
    // bits) hit distinct banks when their images are independent in the low G
    // index bits.  va: logical images of the writing lanes, vb: of the reading
    // ones; a basis (their intersection, the rest of va, the rest of vb, unit
    // vectors) gets index bits so that both stay independent there.
    int G = 0;
    while ((amp_bytes << G) < 128u) ++G;
    G = std::min(G, TB);
    const uint32_t not_h = full & ~(1u << h);
    auto column = [&](int b) {
      uint32_t v = 0;
      for (int j = 0; j < K; ++j)
        if ((A[j] >> b) & 1) v |= 1u << j;
      return v & not_h;
    };
    std::vector<uint32_t> va(G), basis, image;
    uint32_t wmask = 0;
    for (int i = 0; i < G; ++i) va[i] = column(cur.ts[i]), wmask |= 1u << next.ts[i];
    std::vector<uint32_t> ech;  // echelon form of the basis so far
    auto independent = [&](uint32_t v) {
      for (uint32_t e : ech)
        if ((v ^ e) < v) v ^= e;
      if (!v) return false;
      ech.push_back(v);
      std::sort(ech.rbegin(), ech.rend());
      return true;
    };
    int lowbit = 0, hi = G;
    for (int m = 1; m < (1 << G); ++m) {  // the intersection of the two lane spaces
      uint32_t v = 0;
      for (int i = 0; i < G; ++i)
        if ((m >> i) & 1) v ^= va[i];
      if (!(v & ~wmask) && independent(v)) basis.push_back(v), image.push_back(1u << lowbit++);
    }
    const int first_b = lowbit;
    for (int i = 0; i < G; ++i)
      if (independent(va[i])) basis.push_back(va[i]), image.push_back(1u << lowbit++);
    int share = first_b;
    for (int i = 0; i < G; ++i) {
      const uint32_t v = 1u << next.ts[i];
      if (independent(v)) basis.push_back(v), image.push_back((1u << share++) | (1u << hi++));
    }
    for (int j = 0; j < K; ++j)
      if (j != h && independent(1u << j)) basis.push_back(1u << j), image.push_back(1u << hi++);
    // images of the unit vectors: reduce the basis to them
    std::vector<uint32_t> pl(K, 0);
    std::vector<char> used(basis.size(), 0);
    std::vector<int> pivot(K, -1);
    for (int j = 0; j < K; ++j) {
      if (j == h) continue;
      size_t q1 = 0;
      while (used[q1] || !((basis[q1] >> j) & 1)) ++q1;
      used[q1] = 1;
      pivot[j] = (int)q1;
      for (size_t t = 0; t < basis.size(); ++t)
        if (t != q1 && ((basis[t] >> j) & 1)) basis[t] ^= basis[q1], image[t] ^= image[q1];
    }
    for (int j = 0; j < K; ++j)
      if (j != h) pl[j] = image[pivot[j]];

    Built rl;
    std::memset(&rl.op, 0, sizeof(rl.op));
    rl.op.kind = F_RELAYOUT;
    rl.op.coef = (int)prog.aux.size();
    auto& x = prog.aux;
    x.push_back((uint32_t)q);
    auto woff = [&](int b) {
      uint32_t v = 0;
      for (int j = 0; j < K; ++j)
        if (j != h && ((A[j] >> b) & 1)) v ^= pl[j];
      return v * amp_bytes;
    };
    for (int b : cur.rs) x.push_back(woff(b));
    for (int b : cur.ts) x.push_back(woff(b));
    uint32_t fo = 0, outs = 0;
    for (int j = 0; j < K; ++j) {
      if (j != h && ((aff >> j) & 1)) fo ^= pl[j];
      outs |= outx[j];
    }
    x.push_back(fo * amp_bytes);
    for (int b : next.rs) x.push_back(b == h ? 0u : pl[b] * amp_bytes);
    for (int b : next.ts) x.push_back(pl[b] * amp_bytes);
    if (outs) {
      rl.op.pure = 1;
      x.push_back((uint32_t)__builtin_popcount(outs));
      for (uint32_t m = outs; m; m &= m - 1) {
        const int o = __builtin_ctz(m);
        uint32_t v = 0;
        for (int j = 0; j < K; ++j)
          if ((outx[j] >> o) & 1) v ^= pl[j];
        x.push_back((uint32_t)o);
        x.push_back(v * amp_bytes);
      }
    }
    built.push_back(rl);
    H.uses_lds = 1;
    cur = next;
    reset_map();
    aff = carry;
    note_regs();
  };
  auto relayout_to = [&](const std::vector<int>& nr) {
    int h = -1;
    bool shared = false;
    for (int b : cur.rs)
      if (row_clean(b)) {
        h = b;
        shared = shared || index_in(nr, b) >= 0;
      }
    if (!shared) {  // through a layout that keeps one of the present register bits
      std::vector<int> mid(nr.begin(), nr.end() - 1);
      mid.push_back(h);
      relayout_one(mid);
    }
    relayout_one(nr);
  };

  while (!rem.empty()) {
    scan(false);
    if (scan_rc) return scan_rc;
    if (rem.empty()) break;
    bool phases = true;
    for (const LocalGate& l : rem) phases = phases && l.cls == W_PHASE;
    if (phases) {
      if (scan(true)) continue;
      if (scan_rc) return scan_rc;
      relayout_to(cur.rs);  // their bits are not clean: the same registers, a clean map
      continue;
    }
    std::vector<int> nr = choose(0);
    uint32_t R = 0, keep = 0;
    for (int b : nr) R |= 1u << b;
    for (int b : cur.rs)
      if (row_clean(b)) keep |= 1u << b;
    if (!(R & keep)) {
      // no register bit carries over: one that does in the place of the last one
      // chosen costs one relayout instead of two
      const int s0 = simulate(R);
      int best = -1, best_s = -1;
      const uint32_t R1 = R & ~(1u << nr[RB - 1]);
      for (uint32_t m = keep; m; m &= m - 1) {
        const int s = simulate(R1 | (m & (~m + 1)));
        if (s > best_s) best_s = s, best = __builtin_ctz(m);
      }
      if (best_s > 0 && 2 * best_s >= s0) nr[RB - 1] = best;
    }
    bool same = true;
    for (int b : nr) same = same && ((regs >> b) & 1);
    bool map_clean = aff == 0;
    for (int j = 0; j < K; ++j) map_clean = map_clean && row_clean(j);
    if (same && map_clean) {
      set_error("fusion planner: no schedulable gate");
      return QS_ERR_UNSUPPORTED;
    }
    relayout_to(nr);
  }

  // ---- the store: the first L lanes go to the low index bits
  auto store_ok = [&]() {
    for (int i = 0; i < L; ++i) {
      const int b = cur.ts[i];
      if (!((allowed >> b) & 1) || !row_clean(b) || cols[b] != 1) return false;
    }
    uint32_t outs = 0;
    for (int j = 0; j < K; ++j) outs |= outx[j];
    return __builtin_popcount(outs) <= FMAX_SX;
  };
  if (!store_ok()) {
    std::vector<int> nr;
    uint32_t R = 0;
    int spare = __builtin_popcount(allowed) - L;  // allowed bits that may stay in registers
    auto take = [&](int b) {
      const bool al = (allowed >> b) & 1;
      if ((int)nr.size() >= RB || ((R >> b) & 1) || (al && spare <= 0)) return;
      spare -= al;
      nr.push_back(b);
      R |= 1u << b;
    };
    for (int b : cur.rs)
      if (!((allowed >> b) & 1) && row_clean(b)) take(b);
    for (int b : cur.rs)
      if (!((allowed >> b) & 1)) take(b);
    for (int b : cur.rs)
      if (nr.empty() && row_clean(b)) take(b);
    for (int j = K - 1; j >= 0; --j)
      if (!((allowed >> j) & 1)) take(j);
    for (int j = K - 1; j >= 0; --j) take(j);
    relayout_to(nr);
    if (!store_ok()) {
      set_error("fusion planner: internal error: store layout");
      return QS_ERR_ARG;
    }
  }
  // destinations: lanes 0..L-1 to the low bits (home first), the others home where
  // their home is in the tile, else where they are, else anywhere
  {
    std::vector<int> dest(K, -1);
    std::vector<char> used(64, 0);
    uint32_t lows = 0;
    for (int i = 0; i < L; ++i) lows |= 1u << cur.ts[i];
    auto give = [&](int j, int b) {
      dest[j] = b;
      used[b] = 1;
    };
    auto is_low = [&](int b) { return g2l[b] >= 0 && g2l[b] < L; };
    for (int j = 0; j < K; ++j) {
      const bool lo = (lows >> j) & 1;
      if (g2l[home[j]] >= 0 && is_low(home[j]) == lo) give(j, home[j]);
    }
    for (int i = 0; i < L; ++i)  // lane i to index bit i where that is free
      if (dest[cur.ts[i]] < 0 && !used[p.tbits[i]]) give(cur.ts[i], p.tbits[i]);
    for (int j = 0; j < K; ++j)
      if (dest[j] < 0 && is_low(p.tbits[j]) == (bool)((lows >> j) & 1) && !used[p.tbits[j]]) give(j, p.tbits[j]);
    for (int j = 0; j < K; ++j) {
      if (dest[j] >= 0) continue;
      const bool lo = (lows >> j) & 1;
      for (int k = lo ? 0 : L; k < (lo ? L : K); ++k)
        if (!used[p.tbits[k]]) {
          give(j, p.tbits[k]);
          break;
        }
    }
    p.tbo = dest;
    for (int j = 0; j < K; ++j) H.tbo[j] = dest[j];
  }
  // coefficients: the diagonal tables (staged in LDS) first
  const size_t nb = built.size();
  for (Built& b : built) {
    if (b.op.kind == F_DIAG) finalize_diag(b, NR);
    if (wire_heavy(b.op)) H.has_dk = 1;
  }
  auto put_coef = [&](Built& b) {
    b.op.coef = (int)(prog.coef.size() / 2) - coef_start;
    prog.coef.insert(prog.coef.end(), b.coef.begin(), b.coef.end());
  };
  for (Built& b : built)
    if (b.op.kind == F_DIAG && b.op.creg != 0) put_coef(b);
  H.nstage = (int)(prog.coef.size() / 2) - coef_start;
  for (size_t i = 0; i < nb; ++i) {
    Built& b = built[i];
    if (b.op.kind == F_DIAG && b.op.creg == 0) continue;  // the merged product is the identity
    if (b.op.kind != F_DIAG && b.op.kind != F_RELAYOUT && b.op.kind != F_MEAS) put_coef(b);
    prog.ops.push_back(b.op);
  }
  for (int b = 0; b < RB; ++b) H.rs1[b] = cur.rs[b];
  for (int b = 0; b < TB; ++b) H.ts1[b] = cur.ts[b];
  // store addresses: logical bit j to index bit tbo[j], through the pending map
  auto smask = [&](int b) {
    uint64_t m = 0;
    for (int j = 0; j < K; ++j)
      if ((A[j] >> b) & 1) m ^= 1ull << p.tbo[j];
    return m;
  };
  bool same = aff == 0;
  for (int b = 0; b < RB; ++b) {
    H.sr[b] = smask(cur.rs[b]);
    same = same && H.sr[b] == (1ull << H.tbits[H.rs0[b]]);
  }
  for (int b = 0; b < TB; ++b) {
    H.st[b] = smask(cur.ts[b]);
    same = same && H.st[b] == (1ull << H.tbits[H.ts0[b]]);
  }
  uint32_t outs = 0;
  for (int j = 0; j < K; ++j) {
    if ((aff >> j) & 1) H.sflip |= 1ull << p.tbo[j];
    outs |= outx[j];
  }
  for (; outs; outs &= outs - 1) {
    const int o = __builtin_ctz(outs);
    H.sxb[H.nsx] = o;
    for (int j = 0; j < K; ++j)
      if ((outx[j] >> o) & 1) H.sxm[H.nsx] |= 1ull << p.tbo[j];
    ++H.nsx;
    same = false;
  }
  H.sync_store = (!H.uses_lds && !same) ? 1 : 0;
  H.op0 = op_start;
  H.nops = (int)prog.ops.size() - op_start;
  H.coef0 = coef_start;
  H.ncoef = (int)(prog.coef.size() / 2) - coef_start;
  return QS_OK;
}

// ---- grouping --------------------------------------------------------------------

// Plans the whole program, whose gates fill(reducer) adds; every fused pass goes to done(header, first aux word,
// plan) as soon as it is scheduled and is appended to prog.plans after that.
//
// A register of at most K bits is one tile: wires up to K are idle and every store
// puts all wires home (bits n..K-1 are not there: the kernel neither loads nor
// stores them).
template <typename Fill, typename Done>
static int plan_wires(const Fill& fill, int ngates, int nbits, const Config& c, uint32_t amp_bytes,
                      FusedProgram& prog, const Done& done) {
  const int K = c.RB + c.TB, L = c.L;
  const int n = std::max(nbits, K);
  const bool one_tile = n == K;
  WireProgram W;
  {
    WireReducer red(c, W, n);
    W.g.reserve(ngates + 8);
    fill(red);
    red.finish(n, unit_tolerance(amp_bytes));
  }
  const int G = (int)W.g.size();
  const uint64_t all_wires = n >= 64 ? ~0ull : (1ull << n) - 1;
  std::vector<WClass> cls(G);
  // the remaining gates, in order
  enum { ALONE = 1, TABLE = 2, MEAS = 4 };
  struct Rem {
    uint64_t a, m, need;  // its wires, those it mixes, those it needs in the tile
    int id, w, flags;     // gate, weight
  };
  std::vector<Rem> rem(G);
  for (int i = 0; i < G; ++i) {
    const qs_gate& g = W.g[i];
    const WClass t = cls[i] = wire_class(g, W.single[i], W.sym[i]);
    Rem& r = rem[i];
    r.a = gate_mask(g);
    uint64_t targets = 0;
    for (int k = 0; k < g.ntargets; ++k) targets |= 1ull << g.bits[g.ncontrols + k];
    r.m = t == W_SINGLE ? r.a : t == W_PHASE || t == W_TABLE || t == W_ZMEAS ? 0 : targets;
    r.need = t == W_TABLE || t == W_ZMEAS ? r.a : r.m;
    r.id = i;
    r.w = t == W_PHASE ? 1 : t == W_FLIP ? 0 : 2;
    r.flags = (t == W_SINGLE ? ALONE : 0) | (t == W_TABLE ? TABLE : 0) | (W.sym[i].meas != 0.0 ? MEAS : 0);
  }
  prog.pgates = W.g;
  prog.psym = W.sym;
  std::vector<int> pos(n), at(n);  // wire -> index bit, index bit -> wire
  for (int b = 0; b < n; ++b) pos[b] = at[b] = b;
  auto translate = [&](int gi) {
    qs_gate& g = prog.pgates[gi];
    for (int i = 0; i < g.ncontrols + g.ntargets; ++i) g.bits[i] = pos[W.g[gi].bits[i]];
  };
  auto low_wires = [&]() {
    uint64_t m = 0;
    for (int b = 0; b < L; ++b) m |= 1ull << at[b];
    return m;
  };
  int R = G;
  const int max_tables = FMAX_PASS_COEF / (4 << c.RB);  // staged in LDS
  // Weight of the gates that run with tile wires S; cand: what further unblocked
  // gates need besides (in order, each once); taken: the gates (positions).  from:
  // where the first gate is that does not run, and what was counted before; more wires
  // do not change that part.
  struct From {
    int k = 0, w = 0, tables = 0, meas = 0;
  };
  // Candidates beyond the first 48 (more than there are wires; gates on several wires
  // have more sets than that) cost a scan each and do not make plans shorter: 200
  // three-qubit diagonal gates on 20 qubits 10 passes in 1.9 ms of planning, now 1.5 ms.
  constexpr size_t MAX_CAND = 48;
  auto scan = [&](uint64_t S, From& from, std::vector<uint64_t>* cand, std::vector<int>* taken) -> int {
    uint64_t wa = 0, wm = 0;
    int w = from.w, tables = from.tables, meas = from.meas;
    for (int k = from.k; k < R; ++k) {
      const Rem& r = rem[k];
      if (!((r.a & wm) | (r.m & wa))) {
        const uint64_t need = r.need & ~S;
        bool able = true;
        if (r.flags)
          able = !(r.flags & ALONE) && !((r.flags & TABLE) && tables >= max_tables) &&
                 !((r.flags & MEAS) && meas >= FMAX_GRAD);
        if (!need && able) {
          w += r.w;
          if (r.flags) tables += (r.flags & TABLE) != 0, meas += (r.flags & MEAS) != 0;
          if (taken) taken->push_back(k);
          continue;
        }
        if (cand) {
          if (!wa) from.k = k, from.w = w, from.tables = tables, from.meas = meas;
          if (need && able && cand->size() < MAX_CAND && std::find(cand->begin(), cand->end(), need) == cand->end())
            cand->push_back(need);
        }
      }
      wa |= r.a;
      wm |= r.m;
      if (wm == all_wires) break;
    }
    return w;
  };

  // The pass waiting for its store to be decided by the next one's tile.
  bool have = false;
  uint64_t PS = 0;  // its wires
  std::vector<int> pg_;
  auto finish_pass = [&](uint64_t allowed) -> int {
    PassPlan p;
    p.fused = true;
    p.single = -1;
    p.gates = pg_;
    std::vector<int> home;
    uint32_t al = 0;
    for (int b = 0; b < n; ++b)
      if ((PS >> at[b]) & 1) {
        if ((allowed >> at[b]) & 1) al |= 1u << p.tbits.size();
        p.tbits.push_back(b);
        home.push_back(W.home[at[b]]);
      }
    p.tbo = p.tbits;
    for (int gi : p.gates) translate(gi);
    const int a0 = (int)prog.aux.size();
    PassHdr H;
    std::vector<GradCol> cols;
    int rc = schedule_wires(cls, p, c, amp_bytes, al, home, H, prog, cols);
    if (rc) return rc;
    H.aux0 = a0;
    H.naux = (int)prog.aux.size() - a0;
    H.ngrad = (int)cols.size();
    prog.gcols.push_back(std::move(cols));
    std::vector<int> wires(K);
    for (int j = 0; j < K; ++j) wires[j] = at[p.tbits[j]];
    for (int j = 0; j < K; ++j) {
      at[p.tbo[j]] = wires[j];
      pos[wires[j]] = p.tbo[j];
    }
    rc = done(H, a0, p);
    prog.plans.push_back(std::move(p));
    have = false;
    return rc;
  };
  // the wires of PS that go to the low bits when no further tile shares them:
  // those whose home is there, others to make up L
  auto homing = [&]() {
    uint64_t m = 0;
    int k = 0;
    for (int w = 0; w < n; ++w)
      if (((PS >> w) & 1) && W.home[w] < L) m |= 1ull << w, ++k;
    for (int round = 0; round < 3 && k < L; ++round)
      for (int w = 0; w < n && k < L; ++w) {
        if (!((PS >> w) & 1) || ((m >> w) & 1)) continue;
        // rather those whose home is not in the tile, and those on the low bits now
        const bool out = !((PS >> at[W.home[w]]) & 1);
        if (round == 2 || (out && (round == 1 || pos[w] < L))) m |= 1ull << w, ++k;
      }
    return m;
  };

  std::vector<uint64_t> cand;
  std::vector<int> taken;
  while (R > 0) {
    const uint64_t start = have ? 0 : low_wires();
    auto fits = [&](uint64_t S) {
      return __builtin_popcountll(S) <= K && (!have || __builtin_popcountll(S & ~PS) <= K - L);
    };
    uint64_t S = start;
    From from;
    for (;;) {
      cand.clear();
      const int base = scan(S, from, &cand, nullptr);
      uint64_t best = 0;
      double best_gain = -1;
      int nfit = 0;
      for (uint64_t m : cand) nfit += fits(S | m);
      for (uint64_t m : cand) {
        if (!fits(S | m)) continue;
        const double gain = nfit == 1 ? 0 : (double)(scan(S | m, from, nullptr, nullptr) - base) / __builtin_popcountll(m);
        if (gain > best_gain) best_gain = gain, best = m;
      }
      if (!best) break;
      S |= best;
    }
    taken.clear();
    from = From();
    scan(S, from, nullptr, &taken);
    // Phases that no later gate of the pass waits for stay for a pass that needs
    // them, where one of their bits is a register bit; unless no mixing gate is left.
    std::vector<char> drop(R, 0);
    {
      std::vector<char> in(R, 0);
      for (int k : taken) in[k] = 1;
      bool left = false;
      for (int k = 0; k < R; ++k) left = left || (!in[k] && rem[k].need != 0);
      if (left) {
        uint64_t later = 0;
        for (size_t i = taken.size(); i-- > 0;) {
          const int k = taken[i];
          if (cls[rem[k].id] == W_PHASE && !(rem[k].a & later)) drop[k] = 1;
          else later |= rem[k].m;
        }
      }
      size_t o = 0;
      for (int k : taken) o += !drop[k];
      if (o > 0) {
        taken.erase(std::remove_if(taken.begin(), taken.end(), [&](int k) { return drop[k]; }), taken.end());
      }
    }
    if (taken.empty()) {
      // the head gate runs on its own (nothing precedes it): one the tile kernel
      // cannot take, or one with more bits than a tile has room for
      if (have) {
        const int rc = finish_pass(one_tile ? homing() : PS);
        if (rc) return rc;
        continue;  // its store may have brought bits that let the head gate fit
      }
      PassPlan p;
      p.fused = false;
      p.single = rem[0].id;
      translate(p.single);
      prog.plans.push_back(std::move(p));
      rem.erase(rem.begin());
      --R;
      continue;
    }
    std::vector<int> ids;
    {
      std::vector<char> in(R, 0);
      for (int k : taken) in[k] = 1, ids.push_back(rem[k].id);
      int o = 0;
      for (int k = 0; k < R; ++k)
        if (!in[k]) rem[o++] = rem[k];
      R = o;
    }
    // fill the tile: wires of the pass before (they leave its store a choice of
    // low wires), then those on the lowest index bits
    if (have)
      for (int w = 0; w < n && __builtin_popcountll(S) < K; ++w)
        if ((PS >> w) & 1) S |= 1ull << w;
    for (int b = 0; b < n && __builtin_popcountll(S) < K; ++b) S |= 1ull << at[b];
    if (have) {
      const int rc = finish_pass(one_tile ? homing() : S & PS);
      if (rc) return rc;
    }
    have = true;
    PS = S;
    pg_ = ids;
  }
  if (have) {
    const int rc = finish_pass(homing());
    if (rc) return rc;
  }
  // passes without gates that bring the last wires home
  for (int tries = 0;; ++tries) {
    if (tries > 64) {
      set_error("fusion planner: internal error: qubits do not come home");
      return QS_ERR_ARG;
    }
    bool all_home = true;
    for (int w = 0; w < n; ++w) all_home = all_home && pos[w] == W.home[w];
    if (all_home) break;
    uint64_t S = low_wires();
    while (__builtin_popcountll(S) < K) {
      // a wire on the home of one of the tile's wires, else the first one astray
      uint64_t add = 0;
      for (int w = 0; w < n && !add; ++w)
        if (((S >> w) & 1) && !((S >> at[W.home[w]]) & 1)) add = 1ull << at[W.home[w]];
      for (int w = 0; w < n && !add; ++w)
        if (!((S >> w) & 1) && pos[w] != W.home[w]) add = 1ull << w;
      for (int b = 0; b < n && !add; ++b)
        if (!((S >> at[b]) & 1)) add = 1ull << at[b];
      S |= add;
    }
    PS = S;
    pg_.clear();
    have = true;
    const int rc = finish_pass(homing());
    if (rc) return rc;
  }
  return QS_OK;
}

}  // namespace qs

namespace qs {

// ---- programs with parameters ------------------------------------------------------

// One gate of a variational circuit: a fixed gate with its inverse, or a rotation
// exp(-i theta[slot] P / 2), P = X, Y, Z (axis 0, 1, 2), on a circuit bit.
struct VarOp {
  int axis = -1;  // -1: fixed
  int bit = 0, slot = -1;
  qs_gate g, inv;
};

// Plans the circuit (or, backward: its inverse, with a gradient column before every
// rotation's inverse) without its angles.  QS_ERR_UNSUPPORTED for circuits with a
// gate that needs a pass of its own.
static int build_var(const std::vector<VarOp>& ops, bool backward, int n, const Config& c, uint32_t amp_bytes,
                     FusedProgram& prog) {
  auto fill = [&](WireReducer& red) {
    red.keep_phase = false;
    for (size_t i = 0; i < ops.size(); ++i) {
      const VarOp& o = ops[backward ? ops.size() - 1 - i : i];
      if (o.axis < 0) red.add(backward ? o.inv : o.g);
      else red.param(o.axis, o.bit, o.slot, backward ? -1.0 : 1.0, backward);
    }
  };
  auto done = [&](const PassHdr& H, int a0, PassPlan& p) -> int {
    p.hdr = (int)prog.hdrs.size();
    prog.hdrs.push_back(H);
    prog.aux0.push_back(a0);
    return QS_OK;
  };
  const int rc = plan_wires(fill, (int)ops.size(), n, c, amp_bytes, prog, done);
  if (rc) return rc;
  for (const PassPlan& p : prog.plans)
    if (!p.fused) {
      set_error("a gate of the circuit needs a pass of its own");
      return QS_ERR_UNSUPPORTED;
    }
  return QS_OK;
}

// Shear payload of a rotation by sgn * theta, from cos and sin of theta / 2: |t| <= 1
// (a rotation by more than a half turn is taken with a minus sign, which a
// state known up to a phase does not notice).
static void rot_payload(double ch, double sh, double sgn, double* out) {
  sh *= sgn;
  if (ch < 0.0) ch = -ch, sh = -sh;
  out[0] = -sh / (1.0 + ch);
  out[1] = sh;
}
// The same for the phase exp(i sgn theta); returns the op's `pure`.
static int phase_payload_sym(double c, double s, double sgn, double* out) {
  s *= sgn;
  const bool neg = c < 0.0;
  if (neg) c = -c, s = -s;
  out[0] = -s / (1.0 + c);
  out[1] = s;
  return neg ? 3 : 2;
}

}  // namespace qs
