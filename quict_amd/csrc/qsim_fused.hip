// Gate fusion: many gates per full-state pass.
//
// The reference applies one kernel per gate (QuICT/simulation/state_vector/
// statevector_simulator.py:155-164); at 30 qubits every gate streams the whole
// 16 GiB state through HBM.  Here a host planner groups gates into passes; a
// pass owns a set of K "tile" bits (the L lowest amplitude bits, always, plus
// up to K-L arbitrary higher bits).  The state splits into 2^(n-K) disjoint
// tiles of 2^K amplitudes; one workgroup loads one tile, applies every gate of
// the pass to it and writes it back: one HBM read+write per pass instead of
// per gate.
//
// Inside a tile the 2^K amplitudes live in registers: thread t of the 2^TB
// threads holds NR = 2^RB amplitudes.  A "layout" names which tile bit each
// register-index bit and each thread-index bit ("slot") carries.  A gate whose
// non-diagonal targets are register bits is applied entirely in registers;
// controls and up to two diagonal bits may sit on thread bits (lane predicates
// / per-lane tables).  When a gate needs a thread bit in registers the tile is
// re-laid-out through LDS (one ds write + one ds read per amplitude) — the
// only LDS traffic besides the pass coefficients.  Loads/stores use a layout
// whose thread bits include the L low bits, so every wavefront touches
// contiguous 2^L-amplitude runs.
//
// Gates that only relabel the amplitudes cost no instructions:
//  * an uncontrolled SWAP exchanges which tile bit two slots carry (the layout
//    changes, the registers do not);
//  * an uncontrolled X / Y flips the logical value of one slot: the planner
//    conjugates later ops by X on that slot, and the flip is folded into the
//    next LDS relayout address or the store address (one XOR per tile).
//
// Two planners fill this scheme.  plan_wires (qsim_wire_plan.hpp, kernels in
// qsim_wires.hip) runs every program but noisy density matrices and complex64
// gradients: it wants only the bits a gate mixes in the tile.  plan_groups (qsim_fused_plan.hpp, k_fused) wants
// all of them; it is greedy with commutation: scanning the remaining gates in
// order, a gate joins the current pass if its bits fit in the tile and it commutes
// with every gate already deferred.
#include "qsim_common.hpp"
#include "qsim_fused_kernel.hpp"
#include "qsim_wires.hpp"
#include "qsim_internal.hpp"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <stdexcept>

namespace qs {

// Device image of a pass program: [hdrs][ops as FOpW][aux][coef in R], each
// part 256-byte aligned.
struct ProgImage {
  std::vector<char> host;
  uint64_t hb = 0, ob = 0, xb = 0, cb = 0;
};

template <typename R> static void pack_program(const FusedProgram& prog, const Config& c, ProgImage& im) {
  auto al = [](uint64_t b) { return (b + 255) & ~255ull; };
  im.hb = al(prog.hdrs.size() * sizeof(PassHdr));
  const uint64_t op_bytes = c.wires ? sizeof(WireOp<R>) : sizeof(FOpW);
  im.ob = al((prog.ops.size() + 1) * op_bytes);  // (k_wires fetches one op ahead)
  im.xb = al(prog.aux.size() * sizeof(uint32_t));
  const uint64_t ncoef = prog.coef.size() / 2;
  im.cb = al(ncoef * sizeof(cx<R>));
  im.host.assign(im.hb + im.ob + im.xb + im.cb, 0);
  char* h = im.host.data();
  PassHdr* hd = reinterpret_cast<PassHdr*>(h);
  for (size_t i = 0; i < prog.hdrs.size(); ++i) std::memcpy(hd + i, &prog.hdrs[i], sizeof(PassHdr));
  if (c.wires) {
    WireOp<R>* w = reinterpret_cast<WireOp<R>*>(h + im.hb);
    for (size_t i = 0; i < prog.hdrs.size(); ++i) {
      const PassHdr& H = prog.hdrs[i];
      hd[i].nops = encode_wire_pass<R>(prog.ops.data() + H.op0, H.nops, prog.coef.data() + 2 * (size_t)H.coef0, w + H.op0,
                                       nullptr);
    }
  } else {
    for (size_t i = 0; i < prog.ops.size(); ++i) {
      const FOpW e = encode_op(prog.ops[i]);
      std::memcpy(h + im.hb + i * sizeof(FOpW), &e, sizeof(FOpW));
    }
  }
  if (!prog.aux.empty()) std::memcpy(h + im.hb + im.ob, prog.aux.data(), prog.aux.size() * sizeof(uint32_t));
  cx<R>* hc = reinterpret_cast<cx<R>*>(h + im.hb + im.ob + im.xb);
  for (uint64_t i = 0; i < ncoef; ++i) hc[i] = mk<R>((R)prog.coef[2 * i], (R)prog.coef[2 * i + 1]);
}

// Device view of an uploaded image.
template <typename R> struct ProgDev {
  const PassHdr* H;
  const FOpW* O;
  const uint32_t* X;
  const cx<R>* C;
  ProgDev(const char* d, const ProgImage& im)
      : H((const PassHdr*)d), O((const FOpW*)(d + im.hb)), X((const uint32_t*)(d + im.hb + im.ob)),
        C((const cx<R>*)(d + im.hb + im.ob + im.xb)) {}
};

// Writes what a vector with known zeros has not had written: its start, or the zeros.
template <typename R>
__global__ __launch_bounds__(256) void k_rest(cx<R>* __restrict__ v, uint64_t N, uint64_t fixed, uint32_t sh,
                                              uint32_t fresh) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += stride) {
    const bool zero = ((sh ? i ^ (i >> sh) : i) & fixed) != 0;
    if (zero || fresh) st(v + i, mk<R>(zero ? (R)0 : (R)1, (R)0));
  }
}
template <typename R> static int write_rest(cx<R>* v, int n, KnownZeros& z, hipStream_t s) {
  if (!z.fixed) return QS_OK;
  const uint64_t N = 1ull << n, blocks = std::min<uint64_t>((N + 255) / 256, 1ull << 20);
  hipLaunchKernelGGL(k_rest<R>, dim3((unsigned)blocks), dim3(256), 0, s, v, N, z.fixed, (uint32_t)z.sh,
                     (uint32_t)z.fresh);
  QS_CHECK_HIP(hipGetLastError());
  z = KnownZeros();
  return QS_OK;
}

// One fused pass: host header hd, its device copy dh.  prof: bracket the
// launch with the context's timing events (never while capturing a graph).
template <typename R, int RB, int TB>
static int launch_fused(qs_ctx* ctx, cx<R>* v, int n, const Config& c, const PassHdr& hd, const PassHdr* dh,
                        const ProgDev<R>& d, KnownZeros& z, hipStream_t s, bool prof) {
  constexpr int K = RB + TB;
  int rc = QS_OK;
  // (the kernel that prefetches tiles takes a vector that is there)
  if (!c.wires && !hd.has_dk && ctx->fused_prefetch && (rc = write_rest(v, n, z, s))) return rc;
  // (of a vector with known zeros the amplitudes that can differ from 0 are read, none
  // of them before the first pass)
  const double reads = z.fresh ? 0.0 : std::ldexp(1.0, n - __builtin_popcountll(z.fixed & ((1ull << n) - 1)));
  const PassStart S = enter_pass(z, hd, K, std::max(n, K));
  const uint64_t tiles = S.fixed ? 1ull << __builtin_popcountll(S.free) : n > K ? 1ull << (n - K) : 1;
  const size_t lds_bytes = (size_t)(1u << (K - 1)) * sizeof(cx<R>);  // half-tile relayout image
  const size_t lds_relayout = hd.uses_lds ? lds_bytes : 0;
  const size_t lds = hd.has_dk && !c.wires ? lds_relayout : lds_relayout + (size_t)hd.nstage * sizeof(cx<R>);
  if (prof && ctx->profile) ctx->prof_bytes += (reads + std::ldexp((double)tiles, std::min(n, K))) * sizeof(cx<R>);
  if (prof && (rc = prof_begin(ctx, PROF_FUSED, s))) return rc;
  if (c.wires) {
    launch_wires<R, RB, TB>(v, tiles, hd, dh, (const WireOp<R>*)d.O, d.C, d.X, n < K ? 1u << n : 0u, S, lds, s);
  } else {
    auto pass = [&](auto kernel, uint64_t grid) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(1 << TB), lds, s, v, dh, d.O, d.C, d.X, tiles, S);
    };
    if (hd.has_dk && S.fixed) pass(k_fused<R, RB, TB, true, false, true>, tiles);
    else if (hd.has_dk) pass(k_fused<R, RB, TB, true, false, false>, tiles);
    else if (S.fixed) pass(k_fused<R, RB, TB, false, false, true>, tiles);
    else if (ctx->fused_prefetch)  // persistent, prefetching: resident workgroups only
      pass(k_fused<R, RB, TB, false, true, false>, std::min<uint64_t>(tiles, (uint64_t)ctx->num_cus * ctx->fused_wg_per_cu));
    else pass(k_fused<R, RB, TB, false, false, false>, tiles);
  }
  QS_CHECK_HIP(hipGetLastError());
  if (prof && (rc = prof_end(ctx, s))) return rc;
  return QS_OK;
}

// A pass the tile kernel cannot take: the gate's own kernel.
template <typename R>
static int launch_single(qs_ctx* ctx, cx<R>* v, int n, const qs_gate& g, KnownZeros& z, hipStream_t s, bool prof) {
  int rc = write_rest(v, n, z, s);
  if (rc) return rc;
  if (prof && (rc = prof_begin(ctx, PROF_GATE, s))) return rc;
  rc = apply_gate(ctx, v, n, sizeof(R) == 8 ? QS_C128 : QS_C64, &g, s);
  if (rc) return rc;
  if (prof && (rc = prof_end(ctx, s))) return rc;
  return QS_OK;
}

// Launch every pass of `prog` (image at dprog) on stream s.
template <typename R, int RB, int TB>
static int launch_passes(qs_ctx* ctx, cx<R>* v, int n, const Config& c, const FusedProgram& prog, const char* dprog,
                         const ProgImage& im, KnownZeros z, hipStream_t s, bool prof, int* npass_out) {
  const ProgDev<R> d(dprog, im);
  int npass = 0, rc = QS_OK;
  for (size_t i = 0; i < prog.plans.size(); ++i) {
    if (!prog.plans[i].fused) {
      rc = launch_single<R>(ctx, v, n, prog.pgates[prog.plans[i].single], z, s, prof);
    } else {
      const int h = prog.hdr_of[i];
      rc = launch_fused<R, RB, TB>(ctx, v, n, c, prog.hdrs[h], d.H + h, d, z, s, prof);
    }
    if (rc) return rc;
    ++npass;
  }
  if (npass_out) *npass_out = npass;
  return write_rest(v, n, z, s);
}

// A gate that does not keep the norm: a noise channel's superoperator.
static bool superoperator(const qs_gate& g) {
  if (g.kind != QS_GATE_DENSE || g.ntargets < 2 || g.ntargets > 4) return false;
  const int D = 1 << g.ntargets;
  const double* m = g.ntargets == 2 ? g.m : g.big;
  for (int j = 0; j < D; ++j) {
    double s = 0;
    for (int i = 0; i < D; ++i) s += m[2 * (i * D + j)] * m[2 * (i * D + j)] + m[2 * (i * D + j) + 1] * m[2 * (i * D + j) + 1];
    if (std::fabs(s - 1.0) > 1e-5) return true;
  }
  return false;
}

// Planner settings.  Programs are planned in wires (qsim_wire_plan.hpp) and run by
// k_wires, except noisy density matrices: their superoperators mix the row and the
// column bit of every qubit a gate touches, so hardly a bit can stay outside the
// tile, and their two-target ops, not the passes, are what they wait for (the
// 14-qubit 300-gate one on MI355X: 56.3 ms in 26 passes planned with whole gates in
// the tile, 56.2 ms in 13 passes planned in wires).  They keep plan_groups and
// k_fused.  QS_FUSION_REMAP=0 / 1 selects that planner for every call, without
// qubit moves / moving whenever that saves a pass.
static Config fused_config(int RB, int TB, int L, const qs_gate* gates, int ngates) {
  Config c{RB, TB, L};
  c.wires = true;
  for (int i = 0; i < ngates && c.wires; ++i) c.wires = !superoperator(gates[i]);
  if (const char* rm = getenv("QS_FUSION_REMAP")) {
    c.wires = false;
    c.remap = rm[0] == '1' ? 2 : 0;
  }
  return c;
}

// Planning overlapped with the passes: each
// chunk of passes is uploaded and launched as soon as it is planned, so the
// device starts after the first pass is planned instead of after the whole
// program.  A planner error after the first chunk leaves the vector partly
// evolved (the planner's errors are internal: a gate the tile kernel takes
// always schedules).
template <typename R, int RB, int TB>
static int run_fused_streamed(qs_ctx* ctx, cx<R>* v, int n, const qs_gate* gates, int ngates, const Config& c,
                              KnownZeros z, int* passes, hipStream_t s) {
  FusedProgram prog;
  int npass = 0;
  auto chunk = [&](const FusedProgram& sub, int) -> int {
    ProgImage im;
    pack_program<R>(sub, c, im);
    std::lock_guard<std::mutex> lock(ctx->slot_mu);
    qs_ctx::ProgSlot* slot = nullptr;
    int rc = acquire_prog_slot(ctx, im.host.size() + 256, &slot);
    if (rc) return rc;
    std::memcpy(slot->host, im.host.data(), im.host.size());
    QS_CHECK_HIP(hipMemcpyAsync(slot->dev, slot->host, im.host.size(), hipMemcpyHostToDevice, s));
    const ProgDev<R> d((const char*)slot->dev, im);
    for (size_t h = 0; h < sub.hdrs.size() && !rc; ++h, ++npass)
      rc = launch_fused<R, RB, TB>(ctx, v, n, c, sub.hdrs[h], d.H + h, d, z, s, true);
    QS_CHECK_HIP(hipEventRecord(slot->done, s));
    slot->pending = true;
    return rc;
  };
  auto single = [&](const qs_gate& g) -> int {
    ++npass;
    return launch_single<R>(ctx, v, n, g, z, s, true);
  };
  int rc = build_streamed(gates, ngates, n, c, (uint32_t)sizeof(cx<R>), prog, chunk, single);
  if (!rc)
    if (const char* dbg = getenv("QS_FUSION_DEBUG"))
      if (dbg[0] == '1') print_program_stats(prog, n, RB + TB, c.L, ngates);
  if (passes) *passes = npass;
  return rc ? rc : write_rest(v, n, z, s);
}

template <typename R, int RB, int TB>
static int run_fused_t(qs_ctx* ctx, cx<R>* v, int n, const qs_gate* gates, int ngates, int L, KnownZeros z, int* passes,
                       hipStream_t s) {
  Config c = fused_config(RB, TB, L, gates, ngates);
  if (z.whole) c.wires = false, c.remap = 0;
  if (c.remap == 0) {  // passes are final as they form: streamed
    const char* st = getenv("QS_FUSION_STREAM");
    if (!(st && st[0] == '0')) return run_fused_streamed<R, RB, TB>(ctx, v, n, gates, ngates, c, z, passes, s);
  }
  FusedProgram prog;
  int rc = build_program(gates, ngates, n, c, (uint32_t)sizeof(cx<R>), prog);
  if (rc) return rc;
  if (const char* dbg = getenv("QS_FUSION_DEBUG"))
    if (dbg[0] == '1') print_program_stats(prog, n, RB + TB, L, ngates);
  ProgImage im;
  pack_program<R>(prog, c, im);
  // upload from a pinned slot that stays untouched until this call's passes
  // have run (its event), so the call returns without waiting for the device
  std::lock_guard<std::mutex> lock(ctx->slot_mu);
  qs_ctx::ProgSlot* slot = nullptr;
  rc = acquire_prog_slot(ctx, im.host.size() + 256, &slot);
  if (rc) return rc;
  char* dprog = (char*)slot->dev;
  if (!im.host.empty()) {
    std::memcpy(slot->host, im.host.data(), im.host.size());
    QS_CHECK_HIP(hipMemcpyAsync(dprog, slot->host, im.host.size(), hipMemcpyHostToDevice, s));
  }
  rc = launch_passes<R, RB, TB>(ctx, v, n, c, prog, dprog, im, z, s, true, passes);
  QS_CHECK_HIP(hipEventRecord(slot->done, s));
  slot->pending = true;
  return rc;
}

}  // namespace qs

// A gate sequence planned and uploaded once, its passes captured in a HIP graph.
struct qs_graph {
  int device = 0;
  int passes = 0;
  void* dprog = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
};

namespace qs {

template <typename R, int RB, int TB>
static int capture_t(qs_ctx* ctx, cx<R>* v, int n, const qs_gate* gates, int ngates, int L, int init_zero,
                     qs_graph* G) {
  const Config c = fused_config(RB, TB, L, gates, ngates);
  FusedProgram prog;
  int rc = build_program(gates, ngates, n, c, (uint32_t)sizeof(cx<R>), prog);
  if (rc) return rc;
  // Refused: what would not fit a tile whole, though the planner in wires runs some
  // of these gates with bits outside the tile.
  bool refuse = false;
  for (int i = 0; i < ngates; ++i)
    refuse = refuse || !fusable(gates[i], c) ||
             __builtin_popcountll(gate_mask(gates[i]) & ~((1ull << L) - 1)) > RB + TB - L;
  for (const PassPlan& p : prog.plans) refuse = refuse || !p.fused;
  if (refuse) {
    set_error("qs_graph_capture: a gate the tile kernel cannot take would run as its own per-gate pass "
              "(a dense gate on more than 4 targets, a diagonal or phase gate on more than 6 bits, or a gate "
              "with more than tile_log2 bits, or more than tile_log2 - low_bits bits above the low bits); "
              "such sequences are not captured");
    return QS_ERR_UNSUPPORTED;
  }
  ProgImage im;
  pack_program<R>(prog, c, im);
  QS_CHECK_HIP(hipMalloc(&G->dprog, std::max<size_t>(im.host.size(), 256)));
  if (!im.host.empty()) QS_CHECK_HIP(hipMemcpy(G->dprog, im.host.data(), im.host.size(), hipMemcpyHostToDevice));
  hipStream_t s = nullptr;
  QS_CHECK_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
  hipError_t e = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
  if (e != hipSuccess) {
    (void)hipStreamDestroy(s);
    set_error(std::string("hipStreamBeginCapture: ") + hipGetErrorString(e));
    return QS_ERR_DEVICE;
  }
  int npass = 0;
  rc = launch_passes<R, RB, TB>(ctx, v, n, c, prog, (const char*)G->dprog, im, init_zero ? known_start(n, false, RB + TB) : KnownZeros(), s, false,
                                &npass);
  hipGraph_t graph = nullptr;
  e = hipStreamEndCapture(s, &graph);
  (void)hipStreamDestroy(s);
  if (rc) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  if (e != hipSuccess) {
    set_error(std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    return QS_ERR_DEVICE;
  }
  G->graph = graph;
  QS_CHECK_HIP(hipGraphInstantiate(&G->exec, graph, nullptr, nullptr, 0));
  G->passes = npass;
  return QS_OK;
}

template <typename R, int RB, int TB> static void set_lds_attr() {
  static bool done = false;
  if (done) return;
  wires_lds_attr<R, RB, TB>();
  const int bytes = (int)((1u << (RB + TB - 1)) * sizeof(cx<R>) + FMAX_PASS_COEF * sizeof(cx<R>));
  for (const void* k : {(const void*)k_fused<R, RB, TB, true, false, true>, (const void*)k_fused<R, RB, TB, true, false, false>,
                        (const void*)k_fused<R, RB, TB, false, false, true>, (const void*)k_fused<R, RB, TB, false, true, false>,
                        (const void*)k_fused<R, RB, TB, false, false, false>})
    (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  done = true;
}

static int apply_gates_fused_impl(qs_ctx* ctx, void* vec, int n, int dtype, const qs_gate* gates, int ngates,
                                  int start, int* passes, hipStream_t s);

// The planner is host C++: no exception may cross the C ABI.
int apply_gates_fused(qs_ctx* ctx, void* vec, int n, int dtype, const qs_gate* gates, int ngates, int start, int* passes,
                      hipStream_t s) {
  try {
    return apply_gates_fused_impl(ctx, vec, n, dtype, gates, ngates, start, passes, s);
  } catch (const std::exception& e) {
    set_error(std::string("fusion planner: ") + e.what());
    return QS_ERR_DEVICE;
  }
}

// Whether a list on a register of at most a tile is faster planned and run in one launch
// than as a kernel a gate.  us a call on MI355X, 10 qubits, kernels / one launch: 6 gates
// on one or two qubits 27 / 26 to 35, 8 of them 40 to 60 / 30 to 40, 40 of them 160 / 39 to
// 114.  The workgroup's dense op on three targets (four in complex128) takes longer than
// the gate's own kernel: 20 such gates 123 / 185 (462 / 539), and pays for it only among
// enough others; on four targets in complex64 it is the faster by far, 3 gates 74 / 45.
static bool one_launch_pays(const qs_gate* gates, int ngates, int dtype) {
  int gain = 0;
  for (int i = 0; i < ngates; ++i) {
    const bool wide = gates[i].kind == QS_GATE_DENSE && (gates[i].ntargets == 3 || gates[i].ntargets == 4);
    gain += !wide ? 1 : gates[i].ntargets == 4 && dtype == QS_C64 ? 3 : -1;
  }
  return gain >= 7;
}

// A program's upload reads a staging slot that later calls use again, and waits for the
// slot's event: neither belongs into a caller's graph.
static bool capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) {
    (void)hipGetLastError();  // (the null stream while another stream captures)
    return true;
  }
  return st != hipStreamCaptureStatusNone;
}

static int apply_gates_fused_impl(qs_ctx* ctx, void* vec, int n, int dtype, const qs_gate* gates, int ngates,
                                  int start, int* passes, hipStream_t s) {
  // Tile shapes (4 register bits per thread, 2^(K-4) threads, a half-tile LDS
  // image for relayouts): K = 12 by default for both precisions (256 threads;
  // 32 KiB of LDS for complex128, 16 KiB for complex64); complex128 also takes
  // 11 or 13, complex64 13.
  const int K = ctx->tile_log2 ? ctx->tile_log2 : 12;
  const int L = ctx->low_bits ? ctx->low_bits : 4;
  if (L > K - 4) {  // tile shape and low bits may be set in either order
    set_error("low_bits must not exceed tile_log2 - 4");
    return QS_ERR_ARG;
  }
  // Registers of at most a tile run programs planned in wires in one launch where that
  // pays (one_launch_pays); into a graph of the caller's they go as a kernel a gate.
  // Programs that keep whole gates in the tile (fused_config) need more than one tile's
  // bits.
  KnownZeros z = start < 0 ? KnownZeros() : known_start(n, start == QS_START_IDENTITY, K);
  z.whole = start == QS_START_ZERO_WHOLE;
  const bool per_gate = ngates == 0 || (n < K + 1 && (!one_launch_pays(gates, ngates, dtype) || z.whole || capturing(s) || !fused_config(4, K - 4, L, gates, ngates).wires));
  if (per_gate) {
    const int rc = dtype == QS_C128 ? write_rest((cx<double>*)vec, n, z, s) : write_rest((cx<float>*)vec, n, z, s);
    if (rc) return rc;
    for (int i = 0; i < ngates; ++i) {
      int rc = apply_gate(ctx, vec, n, dtype, &gates[i], s);
      if (rc) return rc;
    }
    if (passes) *passes = ngates;
    return QS_OK;
  }
  if (dtype == QS_C128) {
    cx<double>* v = (cx<double>*)vec;
    switch (K) {
      case 11:
        set_lds_attr<double, 4, 7>();
        return run_fused_t<double, 4, 7>(ctx, v, n, gates, ngates, L, z, passes, s);
      case 12:
        set_lds_attr<double, 4, 8>();
        return run_fused_t<double, 4, 8>(ctx, v, n, gates, ngates, L, z, passes, s);
      case 13:
        set_lds_attr<double, 4, 9>();
        return run_fused_t<double, 4, 9>(ctx, v, n, gates, ngates, L, z, passes, s);
      default:
        set_error("complex128 fusion tiles: tile_log2 must be 11, 12 or 13");
        return QS_ERR_UNSUPPORTED;
    }
  }
  cx<float>* v = (cx<float>*)vec;
  switch (K) {
    case 12:
      set_lds_attr<float, 4, 8>();
      return run_fused_t<float, 4, 8>(ctx, v, n, gates, ngates, L, z, passes, s);
    case 13:
      set_lds_attr<float, 4, 9>();
      return run_fused_t<float, 4, 9>(ctx, v, n, gates, ngates, L, z, passes, s);
    default:
      set_error("complex64 fusion tiles: tile_log2 must be 12 or 13");
      return QS_ERR_UNSUPPORTED;
  }
}

}  // namespace qs

namespace qs {

static int graph_capture_impl(qs_ctx* ctx, void* vec, int n, int dtype, const qs_gate* gates, int ngates,
                              int init_zero, qs_graph* G);

static int graph_capture(qs_ctx* ctx, void* vec, int n, int dtype, const qs_gate* gates, int ngates, int init_zero,
                         qs_graph* G) {
  try {
    return graph_capture_impl(ctx, vec, n, dtype, gates, ngates, init_zero, G);
  } catch (const std::exception& e) {
    set_error(std::string("fusion planner: ") + e.what());
    return QS_ERR_DEVICE;
  }
}

static int graph_capture_impl(qs_ctx* ctx, void* vec, int n, int dtype, const qs_gate* gates, int ngates,
                              int init_zero, qs_graph* G) {
  const int K = ctx->tile_log2 ? ctx->tile_log2 : 12;
  const int L = ctx->low_bits ? ctx->low_bits : 4;
  if (L > K - 4) {
    set_error("low_bits must not exceed tile_log2 - 4");
    return QS_ERR_ARG;
  }
  if (n < K + 1) {
    set_error("qs_graph_capture: registers below 2^(tile+1) amplitudes run one kernel per gate and are not captured");
    return QS_ERR_UNSUPPORTED;
  }
  if (dtype == QS_C128) {
    cx<double>* v = (cx<double>*)vec;
    switch (K) {
      case 11: set_lds_attr<double, 4, 7>(); return capture_t<double, 4, 7>(ctx, v, n, gates, ngates, L, init_zero, G);
      case 12: set_lds_attr<double, 4, 8>(); return capture_t<double, 4, 8>(ctx, v, n, gates, ngates, L, init_zero, G);
      case 13: set_lds_attr<double, 4, 9>(); return capture_t<double, 4, 9>(ctx, v, n, gates, ngates, L, init_zero, G);
      default: set_error("complex128 fusion tiles: tile_log2 must be 11, 12 or 13"); return QS_ERR_UNSUPPORTED;
    }
  }
  cx<float>* v = (cx<float>*)vec;
  switch (K) {
    case 12: set_lds_attr<float, 4, 8>(); return capture_t<float, 4, 8>(ctx, v, n, gates, ngates, L, init_zero, G);
    case 13: set_lds_attr<float, 4, 9>(); return capture_t<float, 4, 9>(ctx, v, n, gates, ngates, L, init_zero, G);
    default: set_error("complex64 fusion tiles: tile_log2 must be 12 or 13"); return QS_ERR_UNSUPPORTED;
  }
}

}  // namespace qs

using namespace qs;

extern "C" {

int qs_graph_capture(qs_ctx* ctx, void* vec, int n, int dtype, const qs_gate* gates, int ngates, int init_zero,
                     qs_graph** out) {
  QS_REQUIRE(ctx, "null ctx");
  QS_REQUIRE(out != nullptr, "null output handle");
  *out = nullptr;
  int rc = check_state_args(vec, n, dtype);
  if (rc) return rc;
  QS_REQUIRE(ngates >= 0 && (ngates == 0 || gates != nullptr), "bad gate list");
  for (int i = 0; i < ngates; ++i) {
    rc = validate_gate(&gates[i], n);
    if (rc) return rc;
  }
  QS_CHECK_HIP(hipSetDevice(ctx->device));
  qs_graph* G = new qs_graph();
  G->device = ctx->device;
  rc = graph_capture(ctx, vec, n, dtype, gates, ngates, init_zero, G);
  if (rc) {
    qs_graph_destroy(G);
    return rc;
  }
  *out = G;
  return QS_OK;
}

int qs_graph_launch(qs_graph* g, void* stream) {
  QS_REQUIRE(g != nullptr && g->exec != nullptr, "null or empty graph");
  QS_CHECK_HIP(hipGraphLaunch(g->exec, as_stream(stream)));
  return QS_OK;
}

int qs_graph_passes(const qs_graph* g) { return g ? g->passes : -1; }

void qs_graph_destroy(qs_graph* g) {
  if (!g) return;
  if (g->exec) (void)hipGraphExecDestroy(g->exec);
  if (g->graph) (void)hipGraphDestroy(g->graph);
  if (g->dprog) (void)hipFree(g->dprog);
  delete g;
}

}  // extern "C"
