// Launch of the tile passes planned in wires (kernels in qsim_wires.hip), and their
// op encoding.
#pragma once
#include "qsim_common.hpp"
#include "qsim_fused_plan.hpp"

#include <cstring>

namespace qs {

// Opcodes of k_wires.  P, C: register positions; M: mask of register positions.
enum WCode : uint32_t {
  WC_RELAYOUT = 0,   // + position that splits the exchange
  WC_ROT = 4,        // + P: rotation, payload (t, s)
  WC_EX = 8,         // + P: exchange of the pair, uncontrolled in the tile
  WC_EXT = 12,       // + P: where the thread predicate holds
  WC_EXC = 16,       // + 4 P + C: where register bit C is 1
  WC_PHR = 32,       // + M: phase as shears (t, s)
  WC_PHS = 48,       // + M: minus that
  WC_PHC = 64,       // + M: phase f
  WC_PHN = 80,       // + M: real factor
  WC_TABLE = 96,     // diagonal table in LDS, per register
  WC_LANE = 97,      // diagonal table in LDS, one entry per lane
  WC_U2 = 98,        // + P: complex 2x2
  WC_MZ = 102,       // + P: gradient column Im <lam|Z|psi> (two vectors)
  WC_MY = 106,       // + P: Im <lam|Y|psi>
  WC_HEAVY = 110,    // from here on: only in the HEAVY instance
  WC_U2G = 110,      // + P: complex 2x2 under register and thread controls
  WC_EXG = 114,      // + P: exchange under register and thread controls
  WC_D2 = 118,       // + pair: complex 4x4 under controls
  WC_XX = 124,       // + pair: diagonal + anti-diagonal
  WC_SW = 130,       // + pair: exchange of 01 and 10 under controls
  WC_D3 = 136,       // + missing position: 8x8 (RB = 4)
  WC_D4 = 140,
  WC_END = 141
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
  cx<R> f;
  uint32_t pad[8 - sizeof(cx<R>) / 4];
};
static_assert(sizeof(WireOp<double>) == 64 && sizeof(WireOp<float>) == 64, "WireOp layout");

// f: the op's first coefficient.
template <typename R> static WireOp<R> encode_wire_op(const FOp& o, const double* f) {
  uint32_t code = WC_END;
  const bool ctl = o.creg != 0 || o.cthr != 0;
  switch (o.kind) {
    case F_RELAYOUT:
      code = WC_RELAYOUT;  // the kernel reads the position from the payload
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
  if (o.kind == F_ROT || o.kind == F_PHASE) e.f = mk<R>((R)f[0], (R)f[1]);
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
// lam == nullptr: one vector.  The kernel reads the programs through one pointer
// argument, which it never writes: pointers inside the jobs would make every
// descriptor a vector load.
template <typename R>
void launch_jobs(cx<R>* psi, cx<R>* lam, const char* image, const WireJobs& jobs, uint32_t blocks, bool heavy, double* partial,
                 size_t lds, hipStream_t s);

// One pass over the 2^(n-K) tiles of v: header hd, its device copy dh and the
// program's device arrays; nsmall: amplitudes of a register below a tile, else 0.  The caller checks hipGetLastError().
template <typename R, int RB, int TB>
void launch_wires(cx<R>* v, uint64_t tiles, const PassHdr& hd, const PassHdr* dh, const WireOp<R>* ops, const cx<R>* coef,
                  const uint32_t* aux, uint32_t nsmall, const PassStart& S, size_t lds, hipStream_t s);
// Lets the kernels take their largest LDS allocation (once per process).
template <typename R, int RB, int TB> void wires_lds_attr();

}  // namespace qs
