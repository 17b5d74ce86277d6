// Variational circuits as planned tile passes: a forward program and an inverse
// program with gradient columns (build_var), packed once and refilled with angles.
// Used by the energy gradient (qsim_grad.hip) and the QNN batch (qsim_qnn.hip).
#pragma once
#include "qsim_common.hpp"
#include "qsim_wires.hpp"

#include <cmath>
#include <cstring>
#include <vector>

namespace qs {

// cos, sin of theta / 2 and of theta, per parameter.
struct AngleTable {
  std::vector<double> v;
  void fill(const double* theta, int n) {
    v.resize(4 * (size_t)n);
    for (int i = 0; i < n; ++i) {
      v[4 * i] = std::cos(0.5 * theta[i]);
      v[4 * i + 1] = std::sin(0.5 * theta[i]);
      v[4 * i + 2] = std::cos(theta[i]);
      v[4 * i + 3] = std::sin(theta[i]);
    }
  }
};

// A circuit's two programs in one host image: [headers][ops][relayout constants]
// [coefficients as complex<R>], each part 256-byte aligned.
class VarImage {
 public:
  struct Pass {
    bool heavy;
    size_t lds;    // dynamic LDS bytes
    int ngrad;
  };
  std::vector<char> host;
  uint64_t ob = 0, xb = 0, cb = 0;      // byte offsets of ops, constants, coefficients
  std::vector<Pass> fwd, bwd;           // headers 0..: forward passes, then backward ones
  std::vector<GradCol> cols;            // gradient columns in pass order

  // Plans `ops` on n bits (idle bits up to a tile).  QS_OK or an error code.
  template <typename R> int build(const std::vector<VarOp>& ops, int n) {
    Config c{4, 8, 4};
    c.wires = true;
    FusedProgram prog[2];
    uint64_t nh = 0, no = 0, nx = 0, nc = 0;
    for (int d = 0; d < 2; ++d) {
      int rc = build_var(ops, d == 1, n, c, (uint32_t)sizeof(cx<R>), prog[d]);
      if (!rc) rc = check_program(prog[d], c);
      if (rc) return rc;
      nh += prog[d].hdrs.size(), no += prog[d].ops.size(), nx += prog[d].aux.size(), nc += prog[d].coef.size() / 2;
    }
    auto al = [](uint64_t b) { return (b + 255) & ~255ull; };
    ob = al(nh * sizeof(PassHdr));
    xb = ob + al((no + 1) * sizeof(WireOp<R>));  // (k_jobs fetches one op ahead)
    cb = xb + al(nx * sizeof(uint32_t));
    host.assign(cb + al(nc * sizeof(cx<R>)), 0);
    uint32_t h0 = 0, o0 = 0, x0 = 0, c0 = 0;
    for (int d = 0; d < 2; ++d) {
      const FusedProgram& p = prog[d];
      for (size_t h = 0; h < p.hdrs.size(); ++h) {
        PassHdr H = p.hdrs[h];
        std::vector<FOp> ops(p.ops.begin() + H.op0, p.ops.begin() + H.op0 + H.nops);
        for (FOp& o : ops)
          if (o.kind == F_RELAYOUT) o.coef += (int)x0;
        std::vector<WirePlace> at;
        H.nops = encode_wire_pass<R>(ops.data(), H.nops, p.coef.data() + 2 * (size_t)H.coef0, &op<R>(o0 + (uint64_t)H.op0), &at);
        for (const WirePlace& w : at) {
          const FOp& o = ops[w.fop];
          if (o.sym) refs.push_back({o0 + (uint32_t)(H.op0 + w.op), w.which, o.sym - 1, o.sgn, o.kind == F_ROT, w.code, w.minus});
        }
        const int nv = d + 1;
        const size_t image = (size_t)nv * 2048 * sizeof(cx<R>);
        (d ? bwd : fwd).push_back({H.has_dk != 0, (H.uses_lds ? image : 0) + (size_t)H.nstage * sizeof(cx<R>) +
                                                      (d ? (size_t)H.ngrad * 4 * sizeof(double) : 0), H.ngrad});
        if (d) cols.insert(cols.end(), p.gcols[h].begin(), p.gcols[h].end());
        H.op0 += (int)o0;
        H.coef0 += (int)c0;
        H.aux0 += (int)x0;
        std::memcpy(host.data() + (h0 + h) * sizeof(PassHdr), &H, sizeof(H));
      }
      if (!p.aux.empty()) std::memcpy(host.data() + xb + (uint64_t)x0 * 4, p.aux.data(), p.aux.size() * 4);
      cx<R>* cf = reinterpret_cast<cx<R>*>(host.data() + cb) + c0;
      for (size_t i = 0; i < p.coef.size() / 2; ++i) cf[i] = mk<R>((R)p.coef[2 * i], (R)p.coef[2 * i + 1]);
      h0 += (uint32_t)p.hdrs.size(), o0 += (uint32_t)p.ops.size(), x0 += (uint32_t)p.aux.size();
      c0 += (uint32_t)(p.coef.size() / 2);
    }
    return QS_OK;
  }

  // Payloads of the parameterised ops; at(slot) is the slot's row of the angle table.
  template <typename R, typename At> void bind(const AngleTable& t, const At& at) {
    for (const Ref& r : refs) {
      const double* v = &t.v[4 * (size_t)at(r.slot)];
      double p[2];
      if (r.rot) {
        rot_payload(v[0], v[1], r.sgn, p);
      } else {
        const int pure = phase_payload_sym(v[2], v[3], r.sgn, p);
        uint32_t& w0 = op<R>(r.op).w[0];
        w0 = (w0 & ~0xffu) | (pure == 3 ? r.minus : r.code);
      }
      op<R>(r.op).f[r.which] = mk<R>((R)p[0], (R)p[1]);
    }
  }

 private:
  struct Ref {
    uint32_t op;
    int which, slot;
    double sgn;
    bool rot;
    uint32_t code, minus;
  };
  std::vector<Ref> refs;
  template <typename R> WireOp<R>& op(uint64_t i) { return reinterpret_cast<WireOp<R>*>(host.data() + ob)[i]; }
};

// Column sums of gradient rows: out[i] = sum over rows of partial[off + row * stride].
struct ColSum {
  uint64_t off;
  uint32_t rows, stride;
};
// Enqueues them (fixed order: the same sums for the same rows); cols is device memory.
void column_sums(const double* partial, const ColSum* cols, int ncols, double* out, hipStream_t s);

}  // namespace qs
