// Energy and gradient of a variational circuit from planned programs (qs_var): the
// forward program, lam = H psi and the energy, then the inverse program on psi and lam
// with the gradient columns, all queued at once, one host wait at the end.
//
// Against the call that takes gate records (qsim_grad.hip): the plan outlives the
// call (it does not depend on the angles), so no planning stands between the passes,
// and the sweep is planned in wires: 20 qubits, 480 parameters 2.50 -> 0.77 ms, a new
// circuit's first call 18.5 -> 2.8 ms.
#include "qsim_internal.hpp"
#include "qsim_sweep.hpp"

#include <algorithm>
#include <cstdlib>
#include <exception>

namespace qs {

// One block a column: the rows in a fixed order.  A column's entries are `stride`
// doubles apart; the blocks of neighbouring columns share the cache lines.
__global__ __launch_bounds__(256) void k_column_sums(const double* __restrict__ partial, const ColSum* __restrict__ cols,
                                                     double* __restrict__ out) {
  __shared__ double red[4];
  const ColSum c = cols[blockIdx.x];
  const double* p = partial + c.off;
  double s = 0;
  for (uint32_t r = threadIdx.x; r < c.rows; r += 256) s += p[(uint64_t)r * c.stride];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_down(s, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

void column_sums(const double* partial, const ColSum* cols, int ncols, double* out, hipStream_t s) {
  if (ncols) hipLaunchKernelGGL(k_column_sums, dim3((unsigned)ncols), dim3(256), 0, s, partial, cols, out);
}

// |0...0> over n amplitudes of psi; lam, when given, zeroed.
template <typename R>
__global__ __launch_bounds__(256) void k_basis(cx<R>* __restrict__ psi, cx<R>* __restrict__ lam, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * 256;
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
    st(psi + i, mk<R>(i == 0 ? (R)1 : (R)0, (R)0));
    if (lam) st(lam + i, mk<R>((R)0, (R)0));
  }
}

}  // namespace qs

struct qs_var {
  qs_ctx* ctx = nullptr;
  int n = 0, dtype = 0, nslots = 0;
  qs::VarImage im;
  qs::AngleTable angles;
  std::vector<qs::ColSum> colsums;
  // per backward pass: first entry of its gradient rows, and the columns summed so far
  // once they have been written (0: not after this pass)
  std::vector<uint64_t> row0;
  std::vector<int> sum_to;
  // device: image, column descriptors, column sums, gradient rows, inner-product partials
  char* dev = nullptr;
  uint64_t col_off = 0, sum_off = 0, part_off = 0, ip_off = 0, dev_bytes = 0;
  char* host = nullptr;  // pinned: image, then the results
  uint64_t res_off = 0;
};

namespace qs {

static uint64_t al256(uint64_t b) { return (b + 255) & ~255ull; }

template <typename R> static int var_build(qs_var* v, const std::vector<VarOp>& ops) {
  const int n = std::max(v->n, 12);
  int rc = v->im.build<R>(ops, n);
  if (rc) return rc;
  // Rows of as many passes as fit, then their sums, then the next ones in their place:
  // 33 qubits and 480 parameters would be 8 GB of rows beside 275 GB of state.
  constexpr uint64_t MAX_ROWS = (64ull << 20) / sizeof(double);
  const uint64_t tiles = 1ull << (n - 12);
  uint64_t part = 0, most = 0;
  for (const VarImage::Pass& p : v->im.bwd) {
    const uint64_t rows = tiles * p.ngrad;
    if (part > 0 && part + rows > MAX_ROWS) {
      v->sum_to.back() = (int)v->colsums.size();
      part = 0;
    }
    v->row0.push_back(part);
    v->sum_to.push_back(0);
    for (int i = 0; i < p.ngrad; ++i) v->colsums.push_back({part + i, (uint32_t)tiles, (uint32_t)p.ngrad});
    part += rows;
    most = std::max(most, part);
  }
  if (!v->sum_to.empty()) v->sum_to.back() = (int)v->colsums.size();
  const uint64_t nc = v->colsums.size();
  v->col_off = al256(v->im.host.size());
  v->sum_off = al256(v->col_off + nc * sizeof(ColSum));
  v->part_off = al256(v->sum_off + nc * sizeof(double));
  v->ip_off = al256(v->part_off + most * sizeof(double));
  v->dev_bytes = v->ip_off + (2 * (uint64_t)inner_partial_blocks() + 64) * sizeof(double);
  v->res_off = al256(v->im.host.size());
  const hipError_t err = hipMalloc((void**)&v->dev, v->dev_bytes);
  if (err != hipSuccess) {  // (the call that takes gate records needs less)
    (void)hipGetLastError();
    v->dev = nullptr;
    set_error(std::string("planned gradient: ") + hipGetErrorString(err));
    return QS_ERR_UNSUPPORTED;
  }
  QS_CHECK_HIP(hipHostMalloc((void**)&v->host, v->res_off + (nc + 2) * sizeof(double), hipHostMallocDefault));
  if (nc) QS_CHECK_HIP(hipMemcpy(v->dev + v->col_off, v->colsums.data(), nc * sizeof(ColSum), hipMemcpyHostToDevice));
  return QS_OK;
}

template <typename R>
static int var_gradient(qs_var* v, cx<R>* psi, cx<R>* lam, const double* theta, const qs_pauli_term* terms, int nterms,
                        double* energy, double* grads, hipStream_t s) {
  qs_ctx* ctx = v->ctx;
  const int n = std::max(v->n, 12);
  const uint64_t N = 1ull << n, tiles = N >> 12;
  v->angles.fill(theta, v->nslots);
  v->im.bind<R>(v->angles, [](int slot) { return slot; });
  std::memcpy(v->host, v->im.host.data(), v->im.host.size());
  WaitOnError wait(s);
  QS_CHECK_HIP(hipMemcpyAsync(v->dev, v->host, v->im.host.size(), hipMemcpyHostToDevice, s));
  hipLaunchKernelGGL(k_basis<R>, dim3((unsigned)std::min<uint64_t>(N / 256, 1u << 16)), dim3(256), 0, s, psi,
                     v->n < 12 ? lam : nullptr, N);
  QS_CHECK_HIP(hipGetLastError());
  double* partial = (double*)(v->dev + v->part_off);
  double* ipart = (double*)(v->dev + v->ip_off);
  double* ires = ipart + 2 * inner_partial_blocks();
  WireJobs J;
  std::memset(&J, 0, sizeof(J));
  J.n = 1;
  WireJob& j = J.j[0];
  j.ops = (uint32_t)v->im.ob, j.aux = (uint32_t)v->im.xb, j.coef = (uint32_t)v->im.cb;
  int rc = QS_OK;
  uint32_t h = 0;
  for (const VarImage::Pass& p : v->im.fwd) {
    if ((rc = prof_begin(ctx, PROF_FUSED, s))) return rc;
    j.hdr = h++ * (uint32_t)sizeof(PassHdr);
    launch_jobs<R>(psi, nullptr, v->dev, J, (uint32_t)tiles, p.heavy, nullptr, p.lds, ctx->num_cus, s);
    QS_CHECK_HIP(hipGetLastError());
    if ((rc = prof_end(ctx, s))) return rc;
  }
  rc = pauli_sum_async(ctx, psi, lam, v->n, v->dtype, terms, nterms, s);
  if (!rc) rc = inner_async(psi, lam, v->n, v->dtype, ipart, ires, s);
  if (rc) return rc;
  if ((rc = prof_begin(ctx, PROF_GRAD, s))) return rc;
  const int nc = (int)v->colsums.size();
  double* sums = (double*)(v->dev + v->sum_off);
  int summed = 0;
  for (size_t i = 0; i < v->im.bwd.size(); ++i) {
    const VarImage::Pass& p = v->im.bwd[i];
    j.hdr = h++ * (uint32_t)sizeof(PassHdr);
    j.keep = i + 1 < v->im.bwd.size() ? 3 : 0;  // nothing reads the vectors after the sweep
    j.part = v->row0[i];
    launch_jobs<R>(psi, lam, v->dev, J, (uint32_t)tiles, p.heavy, partial, p.lds, ctx->num_cus, s);
    QS_CHECK_HIP(hipGetLastError());
    if (v->sum_to[i] > summed) {
      column_sums(partial, (const ColSum*)(v->dev + v->col_off) + summed, v->sum_to[i] - summed, sums + summed, s);
      QS_CHECK_HIP(hipGetLastError());
      summed = v->sum_to[i];
    }
  }
  if ((rc = prof_end(ctx, s))) return rc;
  double* res = (double*)(v->host + v->res_off);
  if (nc) QS_CHECK_HIP(hipMemcpyAsync(res, sums, nc * sizeof(double), hipMemcpyDeviceToHost, s));
  QS_CHECK_HIP(hipMemcpyAsync(res + nc, ires, 2 * sizeof(double), hipMemcpyDeviceToHost, s));
  QS_CHECK_HIP(hipStreamSynchronize(s));
  wait.waited = true;
  *energy = res[nc];
  for (int i = 0; i < nc; ++i) grads[v->im.cols[i].slot] += v->im.cols[i].sgn * res[i];
  return QS_OK;
}

static int var_create(qs_ctx* ctx, int n, int dtype, const qs_gate* gates, const qs_gate* inverses, int ngates,
                      const int32_t* axis, const int32_t* slot, int nslots, qs_var* v) {
  std::vector<VarOp> ops(ngates);
  for (int i = 0; i < ngates; ++i) {
    VarOp& o = ops[i];
    if (slot[i] >= 0) {
      o.axis = axis[i], o.slot = slot[i], o.bit = gates[i].bits[0];
    } else {
      o.g = gates[i], o.inv = inverses[i];
    }
  }
  v->ctx = ctx, v->n = n, v->dtype = dtype, v->nslots = nslots;
  try {
    return dtype == QS_C128 ? var_build<double>(v, ops) : var_build<float>(v, ops);
  } catch (const std::exception& e) {
    set_error(std::string("fusion planner: ") + e.what());
    return QS_ERR_DEVICE;
  }
}

}  // namespace qs

using namespace qs;

extern "C" {

int qs_var_create(qs_ctx* ctx, int n, int dtype, const qs_gate* gates, const qs_gate* inverses, int ngates,
                  const int32_t* axis, const int32_t* param_slot, int nslots, qs_var** out) {
  QS_REQUIRE(ctx && out, "null argument");
  *out = nullptr;
  QS_REQUIRE(n >= 1 && n <= 40 && (dtype == QS_C64 || dtype == QS_C128), "bad register");
  QS_REQUIRE(ngates >= 0 && (ngates == 0 || (gates && inverses && axis && param_slot)), "bad gate list");
  QS_REQUIRE(nslots >= 0, "bad parameter count");
  for (int i = 0; i < ngates; ++i) {
    if (param_slot[i] >= 0) {
      QS_REQUIRE(param_slot[i] < nslots, "parameter slot out of range");
      QS_REQUIRE(axis[i] >= 0 && axis[i] <= 2 && gates[i].bits[0] >= 0 && gates[i].bits[0] < n, "bad rotation");
      continue;
    }
    int rc = validate_gate(&gates[i], n);
    if (!rc) rc = validate_gate(&inverses[i], n);
    if (rc) return rc;
  }
  QS_CHECK_HIP(hipSetDevice(ctx->device));
  qs_var* v = new qs_var();
  const int rc = var_create(ctx, n, dtype, gates, inverses, ngates, axis, param_slot, nslots, v);
  if (rc) {
    qs_var_destroy(v);
    return rc;
  }
  *out = v;
  return QS_OK;
}

int qs_var_gradient(qs_var* v, void* psi, void* lam, const double* theta, const qs_pauli_term* terms, int nterms,
                    double* energy, double* grads, void* stream) {
  QS_REQUIRE(v && psi && lam && psi != lam && energy, "null argument");
  QS_REQUIRE(v->nslots == 0 || (theta && grads), "null parameters");
  QS_REQUIRE(nterms >= 1 && terms, "the Pauli sum needs at least one term");
  for (int k = 0; k < nterms; ++k)
    QS_REQUIRE(((terms[k].xmask | terms[k].zmask) >> v->n) == 0, "Pauli mask outside the register");
  hipStream_t s = as_stream(stream);
  if (v->dtype == QS_C128)
    return var_gradient<double>(v, (cx<double>*)psi, (cx<double>*)lam, theta, terms, nterms, energy, grads, s);
  return var_gradient<float>(v, (cx<float>*)psi, (cx<float>*)lam, theta, terms, nterms, energy, grads, s);
}

int qs_var_passes(const qs_var* v, int backward) {
  return v ? (int)(backward ? v->im.bwd.size() : v->im.fwd.size()) : -1;
}

void qs_var_destroy(qs_var* v) {
  if (!v) return;
  if (v->dev) (void)hipFree(v->dev);
  if (v->host) (void)hipHostFree(v->host);
  delete v;
}

}  // extern "C"
