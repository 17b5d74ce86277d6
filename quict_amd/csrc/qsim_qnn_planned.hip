// Batched variational circuits in complex128, forward + adjoint backward (no reference
// counterpart): the circuit family of qsim_qnn.hip as planned tile passes.
//
// The layers are the same gates for every circuit of a width, so a width has one pair
// of planned programs (forward, and inverse with gradient columns; VarImage), and the
// circuits of a width are one vector: circuit after circuit, padded to whole tiles of
// 2^12 amplitudes, a program running on every 2^w (or, below a tile, 2^12) amplitudes
// of it.  A launch takes one pass of every width.  Ry rotations about one axis add, so
// the encoding is the product state prod_q (cos(phi_q/2)|0> + sin(phi_q/2)|1>) with
// phi_q = sum_{j = q mod w} x_j, written directly; lam = (d loss / d E_c) Z_0 psi, so
// the gradient columns add up over circuits by themselves, and d loss / d phi_q =
// Im <lam|Y_q|psi> at the start of the circuit needs lam alone, psi there being that
// product state.
//
// What bounds it: f64 vector work of the two-vector passes.  1024 circuits of 8..18
// qubits, 6 layers: 78.3 -> 7.0 ms against one persistent workgroup a circuit at a
// time (k_qnn), which swept the state w / 2 times a layer forward and w / 2 back, in LDS
// up to 11 qubits and in memory above; here 18 qubits take 4 passes forward and 3 back.
#include "qsim_internal.hpp"
#include "qsim_qnn.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <vector>

namespace qs {

// The circuits of one width.  Their kernels outside the sweeps take a block of 256
// threads per unit: 2^12 amplitudes of a circuit, or all of a narrower one's.
struct QnnGroup {
  int32_t w;
  uint32_t unit0;   // first block
  uint32_t slot0;   // first circuit, in the order of the batch on the device
  uint32_t nslot;
  uint64_t amp0;    // first amplitude, a multiple of 2^12
};
struct QnnGroups {
  int n;
  QnnGroup g[QNN_MAX_W];
};
struct QnnUnit {
  int w, m;         // width; log2 amplitudes of the unit
  uint32_t slot;    // circuit
  uint32_t sub;     // the unit's number in the circuit: its index bits from 12 up
  uint64_t off;     // first amplitude
  uint32_t pad;     // amplitudes behind it that fill the width's last tile
};

__device__ __forceinline__ QnnUnit qnn_unit(const QnnGroups& G) {
  int j = 0;
  while (j + 1 < G.n && blockIdx.x >= G.g[j + 1].unit0) ++j;
  const QnnGroup& g = G.g[j];
  QnnUnit u;
  u.w = g.w;
  u.m = min(g.w, 12);
  const uint32_t i = blockIdx.x - g.unit0;
  const uint32_t slot = i >> (u.w - u.m);
  u.sub = i & ((1u << (u.w - u.m)) - 1);
  u.slot = g.slot0 + slot;
  u.off = g.amp0 + ((uint64_t)i << u.m);
  const uint64_t end = u.off + (1ull << u.m);
  u.pad = slot + 1 == g.nslot ? (uint32_t)((4096 - (end & 4095)) & 4095) : 0;
  return u;
}

// cos and sin of half the encoding angle of every bit (bit b is qubit w - 1 - b) into
// f[b][0], f[b][1].
__device__ __forceinline__ void qnn_encoding(const QnnUnit& u, const double* __restrict__ x, int nfeat,
                                             double (&f)[QNN_MAX_W][2]) {
  if ((int)threadIdx.x < u.w) {
    const int q = u.w - 1 - (int)threadIdx.x;
    double phi = 0;
    for (int j = q; j < nfeat; j += u.w) phi += x[(uint64_t)u.slot * nfeat + j];
    f[threadIdx.x][0] = cos(0.5 * phi);
    f[threadIdx.x][1] = sin(0.5 * phi);
  }
  __syncthreads();
}

// The encoded product state.  Thread t's amplitudes are t + 256 k.  Memory-bound: one
// write of psi.
__global__ __launch_bounds__(256) void k_qnn_init(const QnnGroups G, const double* __restrict__ x, int nfeat,
                                                  cx<double>* __restrict__ psi) {
  __shared__ double f[QNN_MAX_W][2];
  const QnnUnit u = qnn_unit(G);
  const uint32_t tid = threadIdx.x;
  qnn_encoding(u, x, nfeat, f);
  double p = 1;
  for (int b = 12; b < u.w; ++b) p *= f[b][(u.sub >> (b - 12)) & 1];
  for (int b = 0; b < min(u.m, 8); ++b) p *= f[b][(tid >> b) & 1];
  cx<double>* v = psi + u.off;
  for (uint32_t i = tid; i < 1u << u.m; i += 256) {
    double a = p;
    for (int b = 8; b < u.m; ++b) a *= f[b][(i >> b) & 1];
    st(v + i, mk<double>(a, 0));
  }
  for (uint32_t i = tid; i < u.pad; i += 256) st(v + (1u << u.m) + i, mk<double>(0, 0));
}

// The sum over the block's threads, in all of them; red: 4 doubles.
__device__ __forceinline__ double block_sum(double v, double* red) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return (red[0] + red[1]) + (red[2] + red[3]);
}

// A unit's amplitudes, thread t's at t + 256 k, and its part of <Z_0>: qubit 0 is the
// circuit's highest bit.
__device__ __forceinline__ double qnn_load_z(const QnnUnit& u, const cx<double>* __restrict__ psi, cx<double> (&a)[16]) {
  const uint32_t n = 1u << u.m, top = 1u << (u.m - 1);
  double e = 0;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const uint32_t i = threadIdx.x + 256 * k;
    a[k] = i < n ? ld(psi + u.off + i) : mk<double>(0, 0);
    const double p = (double)a[k].re * a[k].re + (double)a[k].im * a[k].im;
    e += u.w <= 12 && (i & top) ? -p : p;
  }
  return u.w > 12 && (u.sub >> (u.w - 13)) ? -e : e;
}

// <Z_0> of the units of circuits wider than a unit.
__global__ __launch_bounds__(256) void k_qnn_expect(const QnnGroups G, const cx<double>* __restrict__ psi,
                                                    double* __restrict__ epart) {
  __shared__ double red[4];
  const QnnUnit u = qnn_unit(G);
  cx<double> a[16];
  const double e = block_sum(qnn_load_z(u, psi, a), red);
  if (threadIdx.x == 0) epart[blockIdx.x] = e;
}

// E_c (a wide circuit's from its units' parts, the same sum in each of its blocks),
// the loss term, and lam = (d loss / d E_c) Z_0 psi.
__global__ __launch_bounds__(256) void k_qnn_lambda(const QnnGroups G, const cx<double>* __restrict__ psi,
                                                    const double* __restrict__ epart, const double* __restrict__ target,
                                                    double inv_ncirc, cx<double>* __restrict__ lam, double* __restrict__ expval,
                                                    double* __restrict__ loss_terms) {
  __shared__ double red[4];
  const QnnUnit u = qnn_unit(G);
  const uint32_t tid = threadIdx.x;
  cx<double> a[16];
  double e = qnn_load_z(u, psi, a);
  if (u.w > 12) e = tid < 1u << (u.w - 12) ? epart[blockIdx.x - u.sub + tid] : 0.0;
  e = block_sum(e, red);
  const double t = target[u.slot];
  const double dl = 2.0 * (e - t) * inv_ncirc;
  if (u.sub == 0 && tid == 0) {
    expval[u.slot] = e;
    loss_terms[u.slot] = (e - t) * (e - t);
  }
  cx<double>* v = lam + u.off;
  const uint32_t n = 1u << u.m, top = 1u << (u.m - 1);
  const double d = u.w > 12 && (u.sub >> (u.w - 13)) ? -dl : dl;
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const uint32_t i = tid + 256 * k;
    const double s = u.w <= 12 && (i & top) ? -d : d;
    if (i < n) st(v + i, mk<double>((s * a[k].re), (s * a[k].im)));
  }
  for (uint32_t i = tid; i < u.pad; i += 256) st(v + n + i, mk<double>(0, 0));
}

// A unit's part of d loss / d phi_q = Im <lam|Y_q|chi>, chi the encoded product state:
// sum over i of Re lam(i) chi_q(i), chi_q having bit q's factor replaced by -sin where
// the bit is 0 and cos where it is 1.  A thread's eight low bits are the same in all its
// amplitudes: their products are taken once, those of bits 8..11 come from a table.
__global__ __launch_bounds__(256) void k_qnn_gradx(const QnnGroups G, const double* __restrict__ x, int nfeat,
                                                   const cx<double>* __restrict__ lam, double* __restrict__ gpart) {
  __shared__ double f[QNN_MAX_W][2], tab[16][5], red[4][13];
  const QnnUnit u = qnn_unit(G);
  const uint32_t tid = threadIdx.x;
  qnn_encoding(u, x, nfeat, f);
  // tab[k][4]: the product over bits 8..m-1 of k; tab[k][b]: with bit 8 + b replaced
  if (tid < 80) {
    const int k = tid / 5, d = tid % 5;
    double p = 8 + d < u.m || d == 4 ? 1.0 : 0.0;
    for (int b = 8; b < u.m; ++b) {
      const int one = (k >> (b - 8)) & 1;
      p *= b - 8 != d ? f[b][one] : one ? f[b][0] : -f[b][1];
    }
    tab[k][d] = p;
  }
  __syncthreads();
  double v[13];
  double A = 0, H[4] = {0, 0, 0, 0};
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    const uint32_t i = tid + 256 * k;
    const double l = i < 1u << u.m ? (double)lam[u.off + i].re : 0.0;
    A += l * tab[k][4];
#pragma unroll
    for (int b = 0; b < 4; ++b) H[b] += l * tab[k][b];
  }
  double lo = 1;
#pragma unroll
  for (int b = 0; b < 8; ++b) {  // v[b] = product of the bits below b
    v[b] = lo;
    if (b < u.m) lo *= f[b][(tid >> b) & 1];
  }
  double hi = A;
#pragma unroll
  for (int b = 7; b >= 0; --b) {
    const int one = (tid >> b) & 1;
    if (b < u.m) {
      v[b] *= hi * (one ? f[b][0] : -f[b][1]);
      hi *= f[b][one];
    }
  }
#pragma unroll
  for (int b = 0; b < 4; ++b) v[8 + b] = H[b] * lo;
  v[12] = A * lo;
#pragma unroll
  for (int i = 0; i < 13; ++i) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v[i] += __shfl_down(v[i], o, 64);
    if ((tid & 63) == 0) red[tid >> 6][i] = v[i];
  }
  __syncthreads();
  if ((int)tid < u.w) {
    const int b = (int)tid, i = min(b, 12);
    double p = (red[0][i] + red[1][i]) + (red[2][i] + red[3][i]);
    for (int c = 12; c < u.w; ++c) {
      const int one = (u.sub >> (c - 12)) & 1;
      p *= c != b ? f[c][one] : one ? f[c][0] : -f[c][1];
    }
    gpart[(uint64_t)blockIdx.x * QNN_MAX_W + u.w - 1 - b] = p;
  }
}

// A circuit's units in a fixed order; feature j is encoded on qubit j mod w.
__global__ __launch_bounds__(256) void k_qnn_gradx_sum(const QnnGroups G, const double* __restrict__ gpart, int nfeat,
                                                       double* __restrict__ grad_x) {
  __shared__ double red[8][32];
  int j = 0;
  while (j + 1 < G.n && blockIdx.x >= G.g[j + 1].slot0) ++j;
  const QnnGroup& g = G.g[j];
  const uint32_t units = 1u << max(g.w - 12, 0), u0 = g.unit0 + (blockIdx.x - g.slot0) * units;
  const uint32_t q = threadIdx.x & 31, r = threadIdx.x >> 5;
  double s = 0;
  if ((int)q < g.w)
    for (uint32_t i = r; i < units; i += 8) s += gpart[(uint64_t)(u0 + i) * QNN_MAX_W + q];
  red[r][q] = s;
  __syncthreads();
  for (int k = (int)threadIdx.x; k < nfeat; k += 256) {
    const int c = k % g.w;
    grad_x[(uint64_t)blockIdx.x * nfeat + k] = ((red[0][c] + red[1][c]) + (red[2][c] + red[3][c])) +
                                               ((red[4][c] + red[5][c]) + (red[6][c] + red[7][c]));
  }
}

constexpr size_t QNN_MAX_IMAGES = 64;  // planned programs kept, 0.1..0.6 MB each; a batch has at most 19 widths (2..20)

static int qnn_image(QnnState* S, int w, int layers, VarImage** out) {
  const auto key = std::make_pair(w, layers);
  auto it = S->images.find(key);
  if (it == S->images.end()) {
    std::vector<VarOp> ops;
    for (int l = 0; l < layers; ++l) {
      for (int q = 0; q < w; ++q)
        for (int g = 0; g < 2; ++g) {
          VarOp o;
          o.axis = 1 + g;  // Y, then Z
          o.bit = w - 1 - q;
          o.slot = (l * 2 + g) * w + q;
          ops.push_back(o);
        }
      for (int q = 0; q + 1 < w; ++q) {
        VarOp o;
        std::memset((void*)&o.g, 0, sizeof(o.g));
        o.g.kind = QS_GATE_XPERM;
        o.g.ncontrols = o.g.ntargets = 1;
        o.g.bits[0] = w - 1 - q, o.g.bits[1] = w - 2 - q;
        o.g.m[0] = o.g.m[2] = 1.0;
        o.inv = o.g;
        ops.push_back(o);
      }
    }
    VarImage im;
    const int rc = im.build<double>(ops, std::max(w, 12));
    if (rc) return rc;
    it = S->images.emplace(key, std::move(im)).first;
  }
  *out = &it->second;
  return QS_OK;
}

// Runs circuits order[0..n), one width after another, and adds to grad_theta.  Returns
// QS_ERR_UNSUPPORTED, with nothing done, if device memory does not suffice.
static int qnn_part(qs_ctx* ctx, QnnState* S, const int32_t* order, int n, int ncirc, const int32_t* widths,
                    int nfeat, const double* x, const double* target, int layers, int max_width, const AngleTable& angles,
                    double* expval, double* loss_terms, double* grad_theta, double* grad_x) {
  auto al = [](uint64_t b) { return (b + 255) & ~255ull; };
  QnnGroups G;
  std::memset((void*)&G, 0, sizeof(G));
  uint64_t amps = 0, units = 0, wide_units = 0;
  for (int i = 0; i < n;) {
    QnnGroup& g = G.g[G.n++];
    g.w = widths[order[i]];
    int e = i;
    while (e < n && widths[order[e]] == g.w) ++e;
    g.unit0 = (uint32_t)units, g.slot0 = (uint32_t)i, g.nslot = (uint32_t)(e - i);
    g.amp0 = amps;
    units += (uint64_t)g.nslot << std::max(g.w - 12, 0);
    if (g.w > 12) wide_units = units;
    amps += ((((uint64_t)g.nslot << g.w) + 4095) >> 12) << 12;
    i = e;
  }
  // the programs, their places in the image, the gradient rows
  std::vector<VarImage*> im(G.n);
  std::vector<uint64_t> base(G.n);
  std::vector<ColSum> cols;
  uint64_t blob = 0, part = 0;
  for (int j = 0; j < G.n; ++j) {
    const int rc = qnn_image(S, G.g[j].w, layers, &im[j]);
    if (rc) return rc == QS_ERR_UNSUPPORTED ? QS_ERR_DEVICE : rc;
    const int w = G.g[j].w;
    im[j]->bind<double>(angles, [=](int slot) { return (slot / w) * max_width + slot % w; });
    base[j] = blob;
    blob += al(im[j]->host.size());
  }
  auto tiles = [&](int j) { return (((uint64_t)G.g[j].nslot << G.g[j].w) + 4095) >> 12; };
  std::vector<std::vector<uint64_t>> row0(G.n);
  for (int j = 0; j < G.n; ++j)
    for (const VarImage::Pass& p : im[j]->bwd) {
      row0[j].push_back(part);
      for (int i = 0; i < p.ngrad; ++i) cols.push_back({part + i, (uint32_t)tiles(j), (uint32_t)p.ngrad});
      part += tiles(j) * p.ngrad;
    }
  const uint64_t nc = cols.size(), nx = (uint64_t)n * nfeat;
  const uint64_t col_off = blob, x_off = al(col_off + nc * sizeof(ColSum)), t_off = al(x_off + nx * sizeof(double)),
                 up = t_off + n * sizeof(double);
  // results: column sums, <Z_0>, loss terms, grad_x
  const uint64_t res_off = al(up), nres = nc + 2 * (uint64_t)n + (grad_x ? nx : 0);
  const uint64_t e_off = al(res_off + nres * sizeof(double)), g_off = al(e_off + wide_units * sizeof(double)),
                 part_off = al(g_off + (grad_x ? units * QNN_MAX_W * sizeof(double) : 0)),
                 psi_off = al(part_off + part * sizeof(double)), lam_off = al(psi_off + amps * sizeof(cx<double>)),
                 total = lam_off + amps * sizeof(cx<double>);
  int rc = S->room(total, res_off + nres * sizeof(double));
  if (rc) return rc;
  for (int j = 0; j < G.n; ++j) std::memcpy(S->host + base[j], im[j]->host.data(), im[j]->host.size());
  std::memcpy(S->host + col_off, cols.data(), nc * sizeof(ColSum));
  double* hx = (double*)(S->host + x_off);
  double* ht = (double*)(S->host + t_off);
  for (int i = 0; i < n; ++i) {
    if (nfeat) std::memcpy(hx + (uint64_t)i * nfeat, x + (uint64_t)order[i] * nfeat, nfeat * sizeof(double));
    ht[i] = target[order[i]];
  }
  hipStream_t s = S->stream;
  char* d = S->dev;
  cx<double>* psi = (cx<double>*)(d + psi_off);
  cx<double>* lam = (cx<double>*)(d + lam_off);
  double* sums = (double*)(d + res_off);
  double* de = sums + nc;
  double* epart = (double*)(d + e_off);
  const double* dx = (const double*)(d + x_off);
  const double* dt = (const double*)(d + t_off);
  WaitOnError wait(s);
  QS_CHECK_HIP(hipMemcpyAsync(d, S->host, up, hipMemcpyHostToDevice, s));
  if ((rc = prof_begin(ctx, PROF_QNN, s))) return rc;
  const dim3 block(256), all((unsigned)units);
  hipLaunchKernelGGL(k_qnn_init, all, block, 0, s, G, dx, nfeat, psi);
  QS_CHECK_HIP(hipGetLastError());
  for (int back = 0; back < 2; ++back) {
    if (back) {
      if (wide_units) {
        hipLaunchKernelGGL(k_qnn_expect, dim3((unsigned)wide_units), block, 0, s, G, psi, epart);
        QS_CHECK_HIP(hipGetLastError());
      }
      hipLaunchKernelGGL(k_qnn_lambda, all, block, 0, s, G, psi, epart, dt, 1.0 / ncirc, lam, de, de + n);
      QS_CHECK_HIP(hipGetLastError());
    }
    for (size_t p = 0;; ++p) {
      WireJobs J;
      std::memset((void*)&J, 0, sizeof(J));
      uint64_t blocks = 0;
      size_t lds = 0;
      bool heavy = false;
      for (int j = 0; j < G.n; ++j) {
        const std::vector<VarImage::Pass>& P = back ? im[j]->bwd : im[j]->fwd;
        if (p >= P.size()) continue;
        WireJob& w = J.j[J.n++];
        const size_t h = back ? im[j]->fwd.size() + p : p;
        w.hdr = (uint32_t)(base[j] + h * sizeof(PassHdr));
        w.ops = (uint32_t)(base[j] + im[j]->ob), w.aux = (uint32_t)(base[j] + im[j]->xb);
        w.coef = (uint32_t)(base[j] + im[j]->cb);
        w.off = G.g[j].amp0;
        w.part = back ? row0[j][p] : 0;
        w.blk0 = (uint32_t)blocks;
        w.keep = p + 1 < P.size() ? 3 : grad_x ? 2 : 0;
        blocks += tiles(j);
        lds = std::max(lds, P[p].lds);
        heavy = heavy || P[p].heavy;
      }
      if (!J.n) break;
      launch_jobs<double>(psi, back ? lam : nullptr, d, J, (uint32_t)blocks, heavy, (double*)(d + part_off), lds, ctx->num_cus, s);
      QS_CHECK_HIP(hipGetLastError());
    }
  }
  column_sums((const double*)(d + part_off), (const ColSum*)(d + col_off), (int)nc, sums, s);
  QS_CHECK_HIP(hipGetLastError());
  if (grad_x && nfeat) {
    double* gpart = (double*)(d + g_off);
    hipLaunchKernelGGL(k_qnn_gradx, all, block, 0, s, G, dx, nfeat, lam, gpart);
    QS_CHECK_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_qnn_gradx_sum, dim3((unsigned)n), block, 0, s, G, gpart, nfeat, de + 2 * (uint64_t)n);
    QS_CHECK_HIP(hipGetLastError());
  }
  if ((rc = prof_end(ctx, s))) return rc;
  double* res = (double*)(S->host + res_off);
  QS_CHECK_HIP(hipMemcpyAsync(res, sums, nres * sizeof(double), hipMemcpyDeviceToHost, s));
  QS_CHECK_HIP(hipStreamSynchronize(s));
  wait.waited = true;
  const double* r = res;
  for (int j = 0; j < G.n; ++j) {
    const int w = G.g[j].w;
    for (const GradCol& c : im[j]->cols) grad_theta[(c.slot / w) * max_width + c.slot % w] += c.sgn * *r++;
  }
  for (int i = 0; i < n; ++i) {
    expval[order[i]] = r[i];
    loss_terms[order[i]] = r[n + i];
    if (grad_x && nfeat)
      std::memcpy(grad_x + (uint64_t)order[i] * nfeat, r + 2 * (uint64_t)n + (uint64_t)i * nfeat, nfeat * sizeof(double));
  }
  return QS_OK;
}

int qnn_planned(qs_ctx* ctx, int ncirc, const int32_t* widths, int nfeat, const double* x, const double* target, int layers,
                int max_width, const double* theta, double* expval, double* loss, double* grad_theta, double* grad_x) {
  QnnState* S = ctx->qnn;
  std::lock_guard<std::mutex> lock(S->mu);
  int rc0 = S->open(ctx->device);
  if (rc0) return rc0;
  if (S->images.size() > QNN_MAX_IMAGES - QNN_MAX_W) S->images.clear();
  // widest first; as many circuits at a time as two vectors of 4 GiB hold, fewer if
  // the device has less to give
  std::vector<int32_t> order(ncirc);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return widths[a] > widths[b]; });
  const int nth = layers * 2 * max_width;
  AngleTable angles;
  angles.fill(theta, nth);
  std::vector<double> terms(ncirc), gth(nth, 0.0);
  uint64_t cap = (4ull << 30) / sizeof(cx<double>);
  for (int i = 0; i < ncirc;) {
    uint64_t amps = 1ull << widths[order[i]];
    int e = i + 1;
    while (e < ncirc && amps + (1ull << widths[order[e]]) <= cap) amps += 1ull << widths[order[e++]];
    const int rc = qnn_part(ctx, S, order.data() + i, e - i, ncirc, widths, nfeat, x, target, layers, max_width,
                               angles, expval, terms.data(), gth.data(), grad_x);
    if (rc == QS_ERR_UNSUPPORTED && e > i + 1) {
      cap = amps / 2;
      continue;
    }
    if (rc) return rc == QS_ERR_UNSUPPORTED ? QS_ERR_DEVICE : rc;
    i = e;
  }
  std::copy(gth.begin(), gth.end(), grad_theta);
  double L = 0;
  for (int i = 0; i < ncirc; ++i) L += terms[i];
  *loss = L / ncirc;
  return QS_OK;
}

}  // namespace qs
