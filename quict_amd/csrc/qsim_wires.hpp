// Launch of the tile passes planned in wires (kernels in qsim_wires.hip), and their
// op encoding.
#pragma once
#include "qsim_common.hpp"
#include "qsim_fused_plan.hpp"

#include <algorithm>
#include <cstring>
#include <vector>

namespace qs {

// Opcodes of k_wires.  P, C: register positions; M: mask of register positions.
enum WCode : uint32_t {
  // the ops of nearly every circuit: dispatched first
  WC_ROT = 0,        // + P: rotation, payload f = (t, s)
  WC_RP = 4,         // + P: rotation f, then the phase f2 (shears) of P alone
  WC_RPS = 8,        // + P: rotation f, then minus that phase
  WC_PR = 12,        // + P: phase f of P alone, then the rotation f2
  WC_PRS = 16,       // + P: minus the phase, then the rotation
  WC_BW = 20,        // + P: column Z, phase f, column Y, rotation f2 (two vectors)
  WC_BWS = 24,       // + P: the same with minus the phase
  WC_HOT = 28,       // from here on: the others
  WC_EX = 28,        // + P: exchange of the pair, uncontrolled in the tile
  WC_PHR = 32,       // + M: phase as shears (t, s)
  WC_PHS = 48,       // + M: minus that
  WC_PHN = 64,       // + M: real factor
  WC_TABLE = 80,     // diagonal table in LDS, per register
  WC_LANE = 81,      // diagonal table in LDS, one entry per lane
  WC_U2 = 82,        // + P: complex 2x2
  WC_MZ = 86,        // + P: gradient column Im <lam|Z|psi> (two vectors)
  WC_MY = 90,        // + P: Im <lam|Y|psi>
  WC_EXT = 94,       // + P: where the thread predicate holds
  WC_EXC = 98,       // + 4 P + C: where register bit C is 1
  WC_RELAYOUT = 114, // the kernel reads from the payload which position splits the exchange
  WC_HEAVY = 115,    // from here on: only in the HEAVY instance
  WC_PHC = 115,      // + M: factor f that is neither real nor of modulus 1
  WC_U2G = 131,      // + P: complex 2x2 under register and thread controls
  WC_EXG = 135,      // + P: exchange under register and thread controls
  WC_D2 = 139,       // + pair: complex 4x4 under controls
  WC_XX = 145,       // + pair: diagonal + anti-diagonal
  WC_SW = 151,       // + pair: exchange of 01 and 10 under controls
  WC_D3 = 157,       // + missing position: 8x8 (RB = 4)
  WC_D4 = 161,
  WC_END = 162
};
// register pairs (P0 > P1) in the order 10, 20, 21, 30, 31, 32
static int wire_pair(int p0, int p1) { return p0 * (p0 - 1) / 2 + p1; }

// Device encoding, one cache line: words code | creg << 8 | cregv << 16 | ntt << 24;
// tpos[0] | tpos[1] << 8; coef; cthr | cthrv << 16; relayout with tile flips; pure;
// cblk; cblkv; then the payload of a rotation or a phase.  The interpreter loads the
// next op while it runs one: with the payload elsewhere (a second dependent load) and
// nothing fetched ahead an op of a 20-qubit pass, one wave a SIMD, took 0.7 us.
template <typename R> struct WireOp {
  uint32_t w[8];
  cx<R> f[32 / sizeof(cx<R>)];  // f[1]: of an op that stands for several (encode_wire_pass)
};
static_assert(sizeof(WireOp<double>) == 64 && sizeof(WireOp<float>) == 64, "WireOp layout");

// f: the op's first coefficient.
template <typename R> static WireOp<R> encode_wire_op(const FOp& o, const double* f) {
  uint32_t code = WC_END;
  const bool ctl = o.creg != 0 || o.cthr != 0;
  switch (o.kind) {
    case F_RELAYOUT:
      code = WC_RELAYOUT;
      break;
    case F_ROT:
      code = WC_ROT + o.pos[0];
      break;
    case F_MEAS:
      code = (o.pure ? WC_MY : WC_MZ) + o.pos[0];
      break;
    case F_PERM1:
      if (!o.pure) code = WC_EXG + o.pos[0];
      else if (!ctl) code = WC_EX + o.pos[0];
      else if (!o.creg) code = WC_EXT + o.pos[0];
      else if (!o.cthr && __builtin_popcount(o.creg) == 1 && o.cregv == o.creg)
        code = WC_EXC + 4 * o.pos[0] + __builtin_ctz(o.creg);
      else code = WC_EXG + o.pos[0];
      break;
    case F_PHASE:
      code = (o.pure == 3 ? WC_PHS : o.pure == 2 ? WC_PHR : o.pure == 1 ? WC_PHN : WC_PHC) + o.creg;
      break;
    case F_DIAG:
      code = o.pure ? WC_LANE : WC_TABLE;
      break;
    case F_DENSE1:
      code = (ctl ? WC_U2G : WC_U2) + o.pos[0];
      break;
    case F_DENSE2:
      code = WC_D2 + wire_pair(o.pos[0], o.pos[1]);
      break;
    case F_XX2:
      code = WC_XX + wire_pair(o.pos[0], o.pos[1]);
      break;
    case F_SWAP2:
      code = WC_SW + wire_pair(o.pos[0], o.pos[1]);
      break;
    case F_DENSE3:
      code = WC_D3 + (6 - o.pos[0] - o.pos[1] - o.pos[2]);
      break;
    case F_DENSE4:
      code = WC_D4;
      break;
  }
  const bool diag = o.kind == F_DIAG;
  WireOp<R> e;
  std::memset((void*)&e, 0, sizeof(e));
  if (o.kind == F_ROT || o.kind == F_PHASE) e.f[0] = mk<R>((R)f[0], (R)f[1]);
  e.w[0] = code | (diag ? 0 : o.creg) << 8 | (diag ? 0 : o.cregv) << 16 | (uint32_t)o.ntt << 24;
  e.w[1] = (uint32_t)o.tpos[0] | (uint32_t)o.tpos[1] << 8;
  e.w[2] = (uint32_t)o.coef;
  e.w[3] = o.cthr | o.cthrv << 16;
  e.w[4] = (uint32_t)(o.kind == F_RELAYOUT ? o.pure : 0);  // relayout: flips that depend on the tile
  e.w[5] = (uint32_t)o.pure;
  e.w[6] = o.cblk;
  e.w[7] = o.cblkv;
  return e;
}

// Where a rotation or phase went: op `op` of the pass, payload f[which]; a phase's code
// is `code` with its shears, `minus` with minus their result.
struct WirePlace {
  int fop, op, which;
  uint32_t code, minus;
};

// A pass's n ops (payloads coef[2 * op.coef ...]) into out; returns how many they are
// there.  Neighbours on one register bit, under the same tile predicate and no other,
// become one op: rotation and phase, phase and rotation, and in a gradient sweep the four
// of a parameter pair, column Z, phase, column Y, rotation.  An op costs 0.2 us besides
// its arithmetic where one wave a SIMD runs (branches to its code, waiting for the next
// descriptor).  20-qubit gradient 938 -> 770 us, 1024 circuits of 8 to 18 qubits
// 8.5 -> 7.0 ms, 20-qubit graph replay 127 -> 120 us, 30 qubits 161 -> 157 ms.
template <typename R>
static int encode_wire_pass(const FOp* ops, int n, const double* coef, WireOp<R>* out, std::vector<WirePlace>* places) {
  auto payload = [&](const FOp& o) { return coef + 2 * (size_t)o.coef; };
  auto rot = [&](int i) { return i < n && ops[i].kind == F_ROT; };
  auto phase = [&](int i, int p) {  // as shears, of bit p alone
    return i < n && ops[i].kind == F_PHASE && ops[i].pure >= 2 && ops[i].creg == 1u << p && !ops[i].cthr;
  };
  auto meas = [&](int i, int y, int p) { return i < n && ops[i].kind == F_MEAS && ops[i].pure == y && ops[i].pos[0] == p; };
  auto same = [&](int i, int k) {
    for (int j = i + 1; j < i + k; ++j)
      if (ops[j].cblk != ops[i].cblk || ops[j].cblkv != ops[i].cblkv) return false;
    return true;
  };
  int m = 0;
  for (int i = 0; i < n;) {
    int k = 1, ph = -1, ro = -1;  // ops taken, the phase and the rotation among them
    uint32_t code = 0, minus = 0;
    const int p = ops[i].kind == F_PHASE ? __builtin_ctz(ops[i].creg | 16) : ops[i].pos[0];
    if (ops[i].kind == F_MEAS && meas(i, 0, p) && phase(i + 1, p) && meas(i + 2, 1, p) && rot(i + 3) &&
        ops[i + 3].pos[0] == p && same(i, 4)) {
      k = 4, ph = i + 1, ro = i + 3, code = WC_BW + p, minus = WC_BWS + p;
    } else if (rot(i) && phase(i + 1, p) && same(i, 2)) {
      k = 2, ro = i, ph = i + 1, code = WC_RP + p, minus = WC_RPS + p;
    } else if (phase(i, p) && rot(i + 1) && ops[i + 1].pos[0] == p && same(i, 2)) {
      k = 2, ph = i, ro = i + 1, code = WC_PR + p, minus = WC_PRS + p;
    }
    WireOp<R>& e = out[m];
    if (k > 1) {
      const int first = std::min(ph, ro);
      e = encode_wire_op<R>(ops[first], payload(ops[first]));
      const double* f = payload(ops[std::max(ph, ro)]);
      e.f[1] = mk<R>((R)f[0], (R)f[1]);
      e.w[0] = (e.w[0] & ~0xffu) | (ops[ph].pure == 3 ? minus : code);
      if (k == 4) e.w[2] = (uint32_t)ops[i].coef, e.w[5] = (uint32_t)ops[i + 2].coef;
      if (places) {
        places->push_back({ph, m, ph > ro, code, minus});
        places->push_back({ro, m, ro > ph, 0, 0});
      }
    } else {
      const bool f = ops[i].kind == F_ROT || ops[i].kind == F_PHASE;
      e = encode_wire_op<R>(ops[i], f ? payload(ops[i]) : nullptr);
      if (places && f) places->push_back({i, m, 0, WC_PHR + ops[i].creg, WC_PHS + ops[i].creg});
    }
    i += k;
    ++m;
  }
  return m;
}

// One pass of one program in a launch of several (12-bit tiles): byte offsets into
// the images (see VarImage), and where its amplitudes are.
struct WireJob {
  uint32_t hdr, ops, aux, coef;
  uint64_t off;    // first amplitude
  uint64_t part;   // first entry of the gradient rows (tile by tile, ngrad each)
  uint32_t blk0;   // first block; the jobs are in block order
  uint32_t keep;   // two vectors: store psi (1), lam (2)
};
constexpr int WIRE_MAX_JOBS = 20;  // the widths of a QNN batch
struct WireJobs {
  int n;
  WireJob j[WIRE_MAX_JOBS];
};
// lam == nullptr: one vector.  cus: the device's compute units.  The kernel reads the programs through one pointer
// argument, which it never writes: pointers inside the jobs would make every
// descriptor a vector load.
template <typename R>
void launch_jobs(cx<R>* psi, cx<R>* lam, const char* image, const WireJobs& jobs, uint32_t blocks, bool heavy, double* partial,
                 size_t lds, int cus, hipStream_t s);

// One pass over the 2^(n-K) tiles of v: header hd, its device copy dh and the
// program's device arrays; nsmall: amplitudes of a register below a tile, else 0.  The caller checks hipGetLastError().
template <typename R, int RB, int TB>
void launch_wires(cx<R>* v, uint64_t tiles, const PassHdr& hd, const PassHdr* dh, const WireOp<R>* ops, const cx<R>* coef,
                  const uint32_t* aux, uint32_t nsmall, const PassStart& S, size_t lds, hipStream_t s);
// Lets the kernels take their largest LDS allocation (once per process).
template <typename R, int RB, int TB> void wires_lds_attr();

}  // namespace qs
