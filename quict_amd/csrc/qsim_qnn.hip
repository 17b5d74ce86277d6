// Batched variational circuits, forward + adjoint backward (no reference counterpart).
//
// Circuit c (width w = widths[c], qubit 0 = most significant amplitude bit):
//   angle encoding   Ry(x[c, j]) on qubit j mod w, j < nfeat
//   `layers` times   Ry(theta[l,0,q]) Rz(theta[l,1,q]) on every qubit q, then CX(q, q+1), q = 0..w-2
//   readout          E_c = <Z_0>,  loss_c = (E_c - target_c)^2,  loss = mean_c loss_c
//
// complex128 batches run as planned tile passes (qsim_qnn_planned.hip), which apply the
// gates of different qubits in another order.  In 32 bits that would move the results
// by 1e-6, and complex64 callers keep the order they have: k_qnn takes a circuit per
// workgroup and a layer's qubits one after another.
//
// k_qnn.  Ry rotations about one axis add, so the encoding is the product state
// prod_q (cos(phi_q/2)|0> + sin(phi_q/2)|1>) with phi_q = sum_{j = q mod w} x_j: one
// pass.  A CX ladder is the GF(2)-linear permutation "prefix xor" of the qubit bits, so
// no amplitude is moved: every wave keeps, in lane q, the physical index mask c_q =
// P(e_q) and the parity mask r_q (logical bit q of a physical index p is parity(p &
// r_q)), and updates both after every ladder.  A rotation on logical qubit q then pairs
// physical p with p ^ c_q.  The rotations of four consecutive qubits run in one sweep
// over groups of 16 amplitudes (a coset of the span of their masks, enumerated by
// inserting zeros at the masks' elimination pivots).  psi and lam are in LDS up to 13
// qubits (128 KiB), above that in a slot of device memory a workgroup.
//
// What bounds it: one workgroup's chain of sweeps, barriers and LDS round trips.  192
// circuits of 5..13 qubits, 4 layers: the kernel 214 us against 690 us with two qubits
// a sweep, states above 11 qubits in device memory, every thread taking the sines of
// every angle, and two barriers a qubit for its two derivatives; the call
// 841 -> 257 us.  1024 circuits of 8..18 qubits, 6 layers: 46.8 -> 18.7 ms.
// The launch shape follows from the widths (qnn_c64): the caller's is checked only.
#include "qsim_common.hpp"
#include "qsim_internal.hpp"
#include "qsim_qnn.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <exception>
#include <numeric>
#include <vector>

namespace qs {

constexpr int QNN_MAX_LAYERS = 16;

__device__ __forceinline__ int parity64(uint64_t v) { return __popcll(v) & 1; }

template <typename R>
__device__ __forceinline__ double block_reduce(double v, double* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  const int nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0;
  for (int i = 0; i < nw; ++i) s += red[i];
  return s;
}

template <typename R>
__device__ __forceinline__ void block_reduce2(double& a, double& b, double* red) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    a += __shfl_down(a, off, 64);
    b += __shfl_down(b, off, 64);
  }
  const int nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    red[2 * (threadIdx.x >> 6)] = a;
    red[2 * (threadIdx.x >> 6) + 1] = b;
  }
  __syncthreads();
  double sa = 0, sb = 0;
  for (int i = 0; i < nw; ++i) {
    sa += red[2 * i];
    sb += red[2 * i + 1];
  }
  a = sa;
  b = sb;
}

// Pair (p0, p1) of physical indices for logical qubit with column mask m and
// row mask r; h enumerates 2^(w-1) pairs.  Returns p0 with logical bit 0.
__device__ __forceinline__ void pair_of(uint64_t h, uint64_t m, uint64_t r, uint64_t& p0, uint64_t& p1) {
  const int pivot = 63 - __clzll(m);
  uint64_t a = ((h >> pivot) << (pivot + 1)) | (h & ((1ull << pivot) - 1));
  uint64_t b = a ^ m;
  if (parity64(a & r)) {
    p0 = b;
    p1 = a;
  } else {
    p0 = a;
    p1 = b;
  }
}

// ---- one circuit family, complex64 --------------------------------------------
struct QnnArgs {
  int n;                   // circuits of this launch, and the first of them
  int first;
  uint32_t alt;            // qubits with the other order of rounding (prod)
  int nfeat, layers, max_width;
  const int32_t* widths;   // per circuit, widest first
  const double* x;         // nfeat each
  const double* target;
  const double* trig;      // (layer, qubit): cos, sin of half the Ry angle, of half the Rz angle
  double* expval;
  double* loss_terms;
  double* grad_circ;       // layers x 2 x max_width each: the circuit's term of d(loss)/d(theta)
  double* grad_x;          // nfeat each
  cx<float>* slots;        // per workgroup 2 x 2^slot_width amplitudes (states in device memory)
  int slot_width;
  int* counter;
  double inv_ncirc;
};

// The angles' cosines and sines, once for the batch, and the launches' queues.
__global__ void k_qnn_trig(const double* __restrict__ theta, int layers, int max_width, double* __restrict__ trig,
                           int* counters, int ncounters) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < ncounters) counters[i] = 0;
  if (i >= layers * max_width) return;
  const int l = i / max_width, q = i % max_width;
  const double ty = theta[(l * 2 + 0) * max_width + q], tz = theta[(l * 2 + 1) * max_width + q];
  trig[4 * i] = cos(0.5 * ty);
  trig[4 * i + 1] = sin(0.5 * ty);
  trig[4 * i + 2] = cos(0.5 * tz);
  trig[4 * i + 3] = sin(0.5 * tz);
}

// Where amplitude p of a state is.  In LDS, sweeps along the lowest bits would put a
// wave's lanes 128 bytes apart; xor-ing bits 5..9 onto the banks spreads them, and
// being linear it goes through the masks: at(p ^ q) = at(p) ^ at(q).
template <bool INLDS> __device__ __forceinline__ uint32_t at(uint32_t p) { return INLDS ? p ^ ((p >> 5) & 31) : p; }

// D qubits' masks: offsets of a group's members and the pivots, ascending, where a
// group's number gets zeros inserted.
template <int D, bool INLDS> struct Sweep {
  uint32_t off[1 << D], r[D];
  int piv[D];
  __device__ __forceinline__ Sweep(uint32_t cm, uint32_t rm, int q0) {
    uint32_t m[D], red[D];
#pragma unroll
    for (int i = 0; i < D; ++i) {
      m[i] = __builtin_amdgcn_readlane(cm, q0 + i);
      r[i] = __builtin_amdgcn_readlane(rm, q0 + i);
      uint32_t v = m[i];
#pragma unroll
      for (int j = 0; j < i; ++j)
        if ((v >> piv[j]) & 1) v ^= red[j];
      red[i] = v;
      piv[i] = 31 - __clz(v);
    }
#pragma unroll
    for (int i = 0; i < D; ++i)
#pragma unroll
      for (int j = i + 1; j < D; ++j) {
        const int lo = min(piv[i], piv[j]), hi = max(piv[i], piv[j]);
        piv[i] = lo, piv[j] = hi;
      }
#pragma unroll
    for (int s = 0; s < 1 << D; ++s) {
      uint32_t o = 0;
#pragma unroll
      for (int i = 0; i < D; ++i)
        if ((s >> i) & 1) o ^= m[i];
      off[s] = at<INLDS>(o);
    }
  }
  __device__ __forceinline__ uint32_t base(uint32_t h) const {
#pragma unroll
    for (int i = 0; i < D; ++i) h = ((h >> piv[i]) << (piv[i] + 1)) | (h & ((1u << piv[i]) - 1));
    return h;
  }
};

// (By value: a choice between two array elements is a choice between addresses, which
// puts the array into scratch memory.)
__device__ __forceinline__ float pick(bool f, float x, float y) { return f ? x : y; }
__device__ __forceinline__ cx<float> pick(bool f, cx<float> x, cx<float> y) {
  return mk<float>(pick(f, x.re, y.re), pick(f, x.im, y.im));
}

// Products with the order of rounding that complex64 results have had: which of two
// products is rounded and which one the fused multiply-add takes exactly, moves results
// by 1e-7 and is otherwise the compiler's choice.  prod: u x, with the imaginary part's
// products the other way round (ALT) on qubits that are not a multiple of fuse_qubits;
// turn, turn_back: e^{+-i t/2} x; mix: c x + s y.
template <bool ALT> __device__ __forceinline__ cx<float> prod(cx<float> u, cx<float> x) {
  return mk<float>(rfma(u.re, x.re, -(u.im * x.im)),
                   ALT ? rfma(u.im, x.re, u.re * x.im) : rfma(u.re, x.im, u.im * x.re));
}
template <int D, int I, bool ALT>
__device__ __forceinline__ void qnn_rotate(cx<float> (&a)[1 << D], const cx<float>* u, bool flip) {
#pragma unroll
  for (int s = 0; s < 1 << D; ++s) {
    if ((s >> I) & 1) continue;
    const int s1 = s | (1 << I);
    const cx<float> x0 = pick(flip, a[s1], a[s]), x1 = pick(flip, a[s], a[s1]);
    const cx<float> y0 = cfma(prod<ALT>(u[0], x0), u[1], x1), y1 = cfma(prod<ALT>(u[2], x0), u[3], x1);
    a[s] = pick(flip, y1, y0);
    a[s1] = pick(flip, y0, y1);
  }
}
template <int D, int I>
__device__ __forceinline__ void qnn_rotations(cx<float> (&a)[1 << D], const cx<float>* u, const uint32_t* r, uint32_t p,
                                              uint32_t alt) {
  if constexpr (I < D) {
    const bool flip = __popc(p & r[I]) & 1;  // the member with bit I of s set holds logical 0
    if ((alt >> I) & 1) qnn_rotate<D, I, true>(a, u + 4 * I, flip);
    else qnn_rotate<D, I, false>(a, u + 4 * I, flip);
    qnn_rotations<D, I + 1>(a, u, r, p, alt);
  }
}
__device__ __forceinline__ cx<float> turn(float c, float s, cx<float> x) {
  return mk<float>(rfma(c, x.re, -(s * x.im)), rfma(s, x.re, c * x.im));
}
__device__ __forceinline__ cx<float> turn_back(float c, float s, cx<float> x) {
  return mk<float>(rfma(c, x.re, s * x.im), rfma(c, x.im, -(s * x.re)));
}
__device__ __forceinline__ cx<float> mix(float c, cx<float> x, float s, cx<float> y) {
  return mk<float>(rfma(c, x.re, s * y.re), rfma(c, x.im, s * y.im));
}

// Forward: U_i = Rz Ry on logical qubit q0 + i, i < D; t: the qubits' rows of the trig table.
template <int D, bool INLDS>
__device__ __forceinline__ void qnn_fwd(cx<float>* psi, uint32_t N, uint32_t cm, uint32_t rm, int q0,
                                        const double* __restrict__ t, uint32_t alt, int tid, int nt) {
  using R = float;
  constexpr int G = 1 << D;
  const Sweep<D, INLDS> S(cm, rm, q0);
  cx<R> u[4 * D];
#pragma unroll
  for (int i = 0; i < D; ++i) {
    const double cy = t[4 * i], sy = t[4 * i + 1], cz = t[4 * i + 2], sz = t[4 * i + 3];
    // U = Rz(tz) Ry(ty) = [[e^{-i tz/2} cy, -e^{-i tz/2} sy], [e^{i tz/2} sy, e^{i tz/2} cy]]
    u[4 * i] = mk<R>((R)(cz * cy), (R)(-sz * cy));
    u[4 * i + 1] = mk<R>((R)(-cz * sy), (R)(sz * sy));
    u[4 * i + 2] = mk<R>((R)(cz * sy), (R)(sz * sy));
    u[4 * i + 3] = mk<R>((R)(cz * cy), (R)(sz * cy));
  }
#pragma unroll 1
  for (uint32_t h = tid; h < N >> D; h += nt) {
    const uint32_t p = S.base(h), g = at<INLDS>(p);
    cx<R> a[G];
#pragma unroll
    for (int s = 0; s < G; ++s) a[s] = ld(psi + (g ^ S.off[s]));
    qnn_rotations<D, 0>(a, u, S.r, p, alt);
#pragma unroll
    for (int s = 0; s < G; ++s) st(psi + (g ^ S.off[s]), a[s]);
  }
}

// Backward: for each qubit the Rz step (gradient gz = Im <lam|Z|psi>, v[4 + i]; then
// Rz^dagger = diag(e^{i tz/2}, e^{-i tz/2}) on both) and the Ry step (gy = Im <lam|Y|psi>
// with Y psi = (-i a1, i a0), v[i]; then Ry^dagger = [[cy, sy], [-sy, cy]]).  ENC: gy
// alone, nothing is applied.
template <int D, bool INLDS, bool ENC>
__device__ __forceinline__ void qnn_bwd(cx<float>* psi, cx<float>* lam, uint32_t N, uint32_t cm, uint32_t rm, int q0,
                                        const double* __restrict__ t, double (&v)[8], int tid, int nt) {
  using R = float;
  constexpr int G = 1 << D;
  const Sweep<D, INLDS> S(cm, rm, q0);
#pragma unroll 1
  for (uint32_t h = tid; h < N >> D; h += nt) {
    const uint32_t p = S.base(h), g = at<INLDS>(p);
    cx<R> a[G], b[G];
#pragma unroll
    for (int s = 0; s < G; ++s) {
      a[s] = ld(psi + (g ^ S.off[s]));
      b[s] = ld(lam + (g ^ S.off[s]));
    }
#pragma unroll
    for (int i = 0; i < D; ++i) {
      const bool flip = __popc(p & S.r[i]) & 1;
      const R cy = ENC ? (R)0 : (R)t[4 * i], sy = ENC ? (R)0 : (R)t[4 * i + 1];
      const R cz = ENC ? (R)0 : (R)t[4 * i + 2], sz = ENC ? (R)0 : (R)t[4 * i + 3];
#pragma unroll
      for (int s = 0; s < G; ++s) {
        if ((s >> i) & 1) continue;
        const int s1 = s | (1 << i);
        cx<R> a0 = pick(flip, a[s1], a[s]), a1 = pick(flip, a[s], a[s1]);  // logical 0 / 1
        cx<R> b0 = pick(flip, b[s1], b[s]), b1 = pick(flip, b[s], b[s1]);
        if (!ENC) {
          v[4 + i] +=
              ((double)b0.re * a0.im - (double)b0.im * a0.re) - ((double)b1.re * a1.im - (double)b1.im * a1.re);
          a0 = turn(cz, sz, a0);
          b0 = turn(cz, sz, b0);
          a1 = turn_back(cz, sz, a1);
          b1 = turn_back(cz, sz, b1);
        }
        v[i] += -((double)b0.re * a1.re + (double)b0.im * a1.im) + ((double)b1.re * a0.re + (double)b1.im * a0.im);
        if (!ENC) {
          const cx<R> c0 = mix(cy, a0, sy, a1), c1 = mix(cy, a1, -sy, a0);
          const cx<R> d0 = mix(cy, b0, sy, b1), d1 = mix(cy, b1, -sy, b0);
          a[s] = pick(flip, c1, c0);
          a[s1] = pick(flip, c0, c1);
          b[s] = pick(flip, d1, d0);
          b[s1] = pick(flip, d0, d1);
        }
      }
    }
    if (!ENC) {
#pragma unroll
      for (int s = 0; s < G; ++s) {
        st(psi + (g ^ S.off[s]), a[s]);
        st(lam + (g ^ S.off[s]), b[s]);
      }
    }
  }
}

// The wave's sums of eight values, sum k in the lanes 8 k .. 8 k + 7: halves are
// exchanged first, so ten exchanges instead of 48.
__device__ __forceinline__ double wave_sums(double (&v)[8], int lane) {
#pragma unroll
  for (int o = 32, n = 4; n >= 1; o >>= 1, n >>= 1) {
    const bool hi = lane & o;
#pragma unroll
    for (int i = 0; i < n; ++i) {
      const double keep = hi ? v[i + n] : v[i], send = hi ? v[i] : v[i + n];
      v[i] = keep + __shfl_xor(send, o, 64);
    }
  }
  double s = v[0];
  s += __shfl_xor(s, 4, 64);
  s += __shfl_xor(s, 2, 64);
  s += __shfl_xor(s, 1, 64);
  return s;
}

template <int NT, bool INLDS>
__global__ __launch_bounds__(NT) void k_qnn(QnnArgs A) {
  using R = float;
  constexpr int NW = NT / 64;
  extern __shared__ __align__(16) char lds_raw[];
  __shared__ double red[2][8][NW];  // two buffers in turn: one barrier a sweep covers both uses
  __shared__ double enc[QNN_MAX_W][2];
  __shared__ int cur;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int MW = A.max_width, nth = A.layers * 2 * MW;
  for (;;) {
    if (tid == 0) cur = atomicAdd(A.counter, 1);
    __syncthreads();
    const int k = __builtin_amdgcn_readfirstlane(cur);
    __syncthreads();
    if (k >= A.n) break;
    const int c = A.first + k;
    const int w = __builtin_amdgcn_readfirstlane(A.widths[c]);
    const uint32_t N = 1u << w;
    cx<R>*psi, *lam;
    if constexpr (INLDS) {
      psi = reinterpret_cast<cx<R>*>(lds_raw);
      lam = psi + N;
    } else {
      psi = A.slots + ((uint64_t)blockIdx.x << (A.slot_width + 1));
      lam = psi + (1u << A.slot_width);
    }
    // encoding angles and product state
    if (tid < w) {
      double phi = 0;
      for (int j = tid; j < A.nfeat; j += w) phi += A.x[(uint64_t)c * A.nfeat + j];
      enc[tid][0] = cos(0.5 * phi);
      enc[tid][1] = sin(0.5 * phi);
    }
    double* grow = A.grad_circ + (uint64_t)c * nth;
    for (int i = tid; i < nth; i += NT)
      if (i % MW >= w) grow[i] = 0.0;
    __syncthreads();
    for (uint32_t i = tid; i < N; i += NT) {
      double re = 1;
      for (int q = 0; q < w; ++q) re *= enc[q][(i >> (w - 1 - q)) & 1];
      st(psi + at<INLDS>(i), mk<R>((R)re, (R)0));
    }
    uint32_t cm = lane < w ? 1u << (w - 1 - lane) : 0, rm = cm;
    __syncthreads();
    for (int l = 0; l < A.layers; ++l) {
      for (int q0 = 0; q0 < w; q0 += 4) {
        const double* t = A.trig + 4 * (l * MW + q0);
        const uint32_t alt = A.alt >> q0;
        switch (min(4, w - q0)) {
          case 1: qnn_fwd<1, INLDS>(psi, N, cm, rm, q0, t, alt, tid, NT); break;
          case 2: qnn_fwd<2, INLDS>(psi, N, cm, rm, q0, t, alt, tid, NT); break;
          case 3: qnn_fwd<3, INLDS>(psi, N, cm, rm, q0, t, alt, tid, NT); break;
          default: qnn_fwd<4, INLDS>(psi, N, cm, rm, q0, t, alt, tid, NT);
        }
        __syncthreads();
      }
      // CX ladder: r'_q = r_0 ^ .. ^ r_q, c'_q = c_q ^ c_{q+1}
#pragma unroll
      for (int o = 1; o < 32; o <<= 1) {
        const uint32_t v = __shfl_up(rm, o, 64);
        if (lane >= o) rm ^= v;
      }
      if (lane >= w) rm = 0;
      cm ^= __shfl_down(cm, 1, 64);
    }
    // E = <Z_0>, lam = Z_0 psi
    double e = 0;
    {
      const uint32_t r0 = __builtin_amdgcn_readlane(rm, 0);
      for (uint32_t i = tid; i < N; i += NT) {
        const cx<R> a = ld(psi + at<INLDS>(i));
        const double p = (double)a.re * a.re + (double)a.im * a.im;
        const bool one = __popc(i & r0) & 1;
        e += one ? -p : p;
        st(lam + at<INLDS>(i), one ? mk<R>(-a.re, -a.im) : a);
      }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o, 64);
    if (lane == 0) red[0][0][wave] = e;
    __syncthreads();
    e = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) e += red[0][0][i];
    const double tgt = A.target[c];
    const double dl = 2.0 * (e - tgt) * A.inv_ncirc;  // d(mean loss)/dE_c
    if (tid == 0) {
      A.expval[c] = e;
      A.loss_terms[c] = (e - tgt) * (e - tgt);
    }
    int buf = 1;
    // backward; l = -1: the encoding, d E / d phi_q = Im <lam|Y_q|psi> with the identity map again
    for (int l = A.layers - 1; l >= -1; --l) {
      if (l >= 0) {
        const uint32_t v = __shfl_up(rm, 1, 64);
        if (lane >= 1 && lane < w) rm ^= v;
#pragma unroll
        for (int o = 1; o < 32; o <<= 1) cm ^= __shfl_down(cm, o, 64);
      }
      for (int q0 = 0; q0 < w; q0 += 4) {
        const int d = min(4, w - q0);
        const double* t = A.trig + 4 * (max(l, 0) * MW + q0);
        double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        if (l >= 0) {
          switch (d) {
            case 1: qnn_bwd<1, INLDS, false>(psi, lam, N, cm, rm, q0, t, v, tid, NT); break;
            case 2: qnn_bwd<2, INLDS, false>(psi, lam, N, cm, rm, q0, t, v, tid, NT); break;
            case 3: qnn_bwd<3, INLDS, false>(psi, lam, N, cm, rm, q0, t, v, tid, NT); break;
            default: qnn_bwd<4, INLDS, false>(psi, lam, N, cm, rm, q0, t, v, tid, NT);
          }
        } else {
          switch (d) {
            case 1: qnn_bwd<1, INLDS, true>(psi, lam, N, cm, rm, q0, t, v, tid, NT); break;
            case 2: qnn_bwd<2, INLDS, true>(psi, lam, N, cm, rm, q0, t, v, tid, NT); break;
            case 3: qnn_bwd<3, INLDS, true>(psi, lam, N, cm, rm, q0, t, v, tid, NT); break;
            default: qnn_bwd<4, INLDS, true>(psi, lam, N, cm, rm, q0, t, v, tid, NT);
          }
        }
        const double s = wave_sums(v, lane);
        if ((lane & 7) == 0) red[buf][lane >> 3][wave] = s;
        __syncthreads();
        if (tid < 8 && (tid & 3) < d) {
          double g = 0;
#pragma unroll
          for (int i = 0; i < NW; ++i) g += red[buf][tid][i];
          const int q = q0 + (tid & 3);
          if (l >= 0) grow[(l * 2 + (tid >> 2)) * MW + q] = dl * g;
          else if (tid < 4)
            for (int j = q; j < A.nfeat; j += w) A.grad_x[(uint64_t)c * A.nfeat + j] = dl * g;
        }
        buf ^= 1;
      }
    }
    __syncthreads();
  }
}

__global__ void k_qnn_clear(int* counter) {
  if (threadIdx.x == 0) *counter = 0;
}

// grad_theta[i] = sum over circuits of grad_circ[c][i]: 32 columns a block, eight
// threads a column, in a fixed order.  (One thread a column: 43 us for 192 circuits.)
__global__ __launch_bounds__(256) void k_qnn_reduce(const double* __restrict__ grad_circ, int ncirc, int nth,
                                                    double* __restrict__ g) {
  __shared__ double red[8][32];
  const int q = threadIdx.x & 31, r = threadIdx.x >> 5, i = blockIdx.x * 32 + q;
  double s = 0;
  if (i < nth)
    for (int c = r; c < ncirc; c += 8) s += grad_circ[(uint64_t)c * nth + i];
  red[r][q] = s;
  __syncthreads();
  if (r == 0 && i < nth)
    g[i] = ((red[0][q] + red[1][q]) + (red[2][q] + red[3][q])) + ((red[4][q] + red[5][q]) + (red[6][q] + red[7][q]));
}

QnnState* qnn_state_create() { return new QnnState(); }
void qnn_state_destroy(QnnState* S) {
  if (!S) return;
  if (S->dev) (void)hipFree(S->dev);
  if (S->host) (void)hipHostFree(S->host);
  if (S->stream) (void)hipStreamDestroy(S->stream);
  delete S;
}
int QnnState::open(int device) {
  QS_CHECK_HIP(hipSetDevice(device));
  if (!stream) QS_CHECK_HIP(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
  return QS_OK;
}
int QnnState::room(uint64_t dev_need, uint64_t host_need) {
  if (dev_bytes < dev_need) {
    if (dev) QS_CHECK_HIP(hipFree(dev));
    dev = nullptr, dev_bytes = 0;
    const hipError_t err = hipMalloc((void**)&dev, dev_need);
    if (err != hipSuccess) {
      (void)hipGetLastError();
      dev = nullptr;
      set_error(std::string("batch of variational circuits: ") + hipGetErrorString(err));
      return QS_ERR_UNSUPPORTED;
    }
    dev_bytes = dev_need;
  }
  if (host_bytes < host_need) {
    if (host) QS_CHECK_HIP(hipHostFree(host));
    host = nullptr, host_bytes = 0;
    QS_CHECK_HIP(hipHostMalloc((void**)&host, host_need, hipHostMallocDefault));
    host_bytes = host_need;
  }
  return QS_OK;
}

static int qnn_check(const qs_qnn_config* cfg, int dtype) {
  if (!cfg) return QS_OK;
  const int t = cfg->block_threads, w = cfg->lds_max_width;
  QS_REQUIRE(cfg->fuse_qubits >= 0 && cfg->fuse_qubits <= 3, "fuse_qubits must be in [1, 3] (0: 1)");
  QS_REQUIRE(t == 64 || t == 128 || t == 256 || t == 512 || t == 1024,
             "block_threads must be a power of two in [64, 1024]");
  QS_REQUIRE(w >= 0 && w <= 13, "lds_max_width must be in [0, 13]");
  QS_REQUIRE(cfg->blocks_per_cu >= 1 && cfg->blocks_per_cu <= 8, "blocks_per_cu must be in [1, 8]");
  QS_REQUIRE(w == 0 || (2ull << w) * amp_bytes(dtype) <= 150 * 1024, "LDS state too large for one workgroup");
  return QS_OK;
}

// Launch shapes, one launch each, the widest circuits first.  A sweep has 2^(w-4) groups
// and takes 240 registers a thread, eight waves a CU: 512 threads from 14 qubits on (a
// workgroup a CU, each with its slot) and for 12 and 13 (a workgroup's LDS), 128 up to 11
// (32 KiB: four workgroups a CU).  Up to one circuit a CU the last two go as one
// launch: they run side by side, and only the widest counts.
static int qnn_c64(qs_ctx* ctx, int fuse, int ncirc, const int32_t* widths, int nfeat, const double* x, const double* target,
                   int layers, int max_width, const double* theta, double* expval, double* loss, double* grad_theta,
                   double* grad_x) {
  QnnState* S = ctx->qnn;
  std::lock_guard<std::mutex> lock(S->mu);
  int rc = S->open(ctx->device);
  if (rc) return rc;
  std::vector<int32_t> order(ncirc);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return widths[a] > widths[b]; });
  auto wider = [&](int w) {  // circuits of more than w qubits
    return (int)(std::partition_point(order.begin(), order.end(), [&](int c) { return widths[c] > w; }) - order.begin());
  };
  const int cus = ctx->num_cus;
  int end[3] = {wider(13), wider(11), ncirc};
  if (ncirc - end[0] <= cus && end[1] > end[0]) end[1] = ncirc;
  const int wmax = widths[order[0]];
  auto al = [](uint64_t b) { return (b + 255) & ~255ull; };
  const uint64_t n = ncirc, nth = (uint64_t)layers * 2 * max_width, nx = n * nfeat;
  // up: theta, x, target, widths; down: <Z_0>, loss terms, grad_theta, grad_x
  const uint64_t x_off = al(nth * sizeof(double)), t_off = al(x_off + nx * sizeof(double)),
                 w_off = al(t_off + n * sizeof(double)), up = w_off + n * sizeof(int32_t), res_off = al(up),
                 nres = 2 * n + nth + nx, trig_off = al(res_off + nres * sizeof(double)),
                 cnt_off = al(trig_off + 2 * nth * sizeof(double)), gc_off = cnt_off + 256,
                 slot_off = al(gc_off + n * nth * sizeof(double));
  int slots = std::min(end[0], cus);
  for (;;) {  // fewer states in device memory at a time if it has not so much to give
    rc = S->room(slot_off + ((uint64_t)slots << (wmax + 1)) * sizeof(cx<float>), res_off + nres * sizeof(double));
    if (rc != QS_ERR_UNSUPPORTED || slots <= 1) break;
    slots /= 2;
  }
  if (rc) return rc == QS_ERR_UNSUPPORTED ? QS_ERR_DEVICE : rc;
  std::memcpy(S->host, theta, nth * sizeof(double));
  double* hx = (double*)(S->host + x_off);
  double* ht = (double*)(S->host + t_off);
  int32_t* hw = (int32_t*)(S->host + w_off);
  for (int i = 0; i < ncirc; ++i) {
    if (nfeat) std::memcpy(hx + (uint64_t)i * nfeat, x + (uint64_t)order[i] * nfeat, nfeat * sizeof(double));
    ht[i] = target[order[i]];
    hw[i] = widths[order[i]];
  }
  hipStream_t s = S->stream;
  char* d = S->dev;
  WaitOnError wait(s);
  QS_CHECK_HIP(hipMemcpyAsync(d, S->host, up, hipMemcpyHostToDevice, s));
  QnnArgs A;
  A.nfeat = nfeat, A.layers = layers, A.max_width = max_width;
  A.alt = 0;
  for (int q = 0; q < QNN_MAX_W; ++q) A.alt |= (uint32_t)(q % fuse != 0) << q;
  A.widths = (const int32_t*)(d + w_off);
  A.x = (const double*)(d + x_off);
  A.target = (const double*)(d + t_off);
  A.trig = (const double*)(d + trig_off);
  double* res = (double*)(d + res_off);
  A.expval = res, A.loss_terms = res + n, A.grad_x = res + 2 * n + nth;
  A.grad_circ = (double*)(d + gc_off);
  A.slots = (cx<float>*)(d + slot_off);
  A.slot_width = wmax;
  A.inv_ncirc = 1.0 / ncirc;
  int* counters = (int*)(d + cnt_off);
  if ((rc = prof_begin(ctx, PROF_QNN, s))) return rc;
  hipLaunchKernelGGL(k_qnn_trig, dim3((unsigned)((layers * max_width + 63) / 64)), dim3(64), 0, s, (const double*)d, layers,
                     max_width, (double*)(d + trig_off), counters, 3);
  QS_CHECK_HIP(hipGetLastError());
  for (int i = 0, first = 0; i < 3; first = end[i], ++i) {
    A.first = first, A.n = end[i] - first, A.counter = counters + i;
    if (A.n <= 0) continue;
    const size_t lds = (size_t)2 << std::max((int)widths[order[first]], 1) << 3;
    if (i == 0) {
      hipLaunchKernelGGL((k_qnn<512, false>), dim3((unsigned)slots), dim3(512), 0, s, A);
    } else if (i == 1) {
      QS_CHECK_HIP(hipFuncSetAttribute((const void*)k_qnn<512, true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       128 * 1024));
      hipLaunchKernelGGL((k_qnn<512, true>), dim3((unsigned)std::min(A.n, 2 * cus)), dim3(512), lds, s, A);
    } else {
      hipLaunchKernelGGL((k_qnn<128, true>), dim3((unsigned)std::min(A.n, 16 * cus)), dim3(128), lds, s, A);
    }
    QS_CHECK_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(k_qnn_reduce, dim3((unsigned)((nth + 31) / 32)), dim3(256), 0, s, A.grad_circ, ncirc, (int)nth,
                     res + 2 * n);
  QS_CHECK_HIP(hipGetLastError());
  if ((rc = prof_end(ctx, s))) return rc;
  const double* r = (const double*)(S->host + res_off);
  QS_CHECK_HIP(hipMemcpyAsync((void*)r, res, (grad_x ? nres : nres - nx) * sizeof(double), hipMemcpyDeviceToHost, s));
  QS_CHECK_HIP(hipStreamSynchronize(s));
  wait.waited = true;
  std::vector<double> terms(ncirc);
  for (int i = 0; i < ncirc; ++i) {
    expval[order[i]] = r[i];
    terms[order[i]] = r[n + i];
    if (grad_x && nfeat)
      std::memcpy(grad_x + (uint64_t)order[i] * nfeat, r + 2 * n + nth + (uint64_t)i * nfeat, nfeat * sizeof(double));
  }
  std::copy(r + 2 * n, r + 2 * n + nth, grad_theta);
  double L = 0;
  for (int i = 0; i < ncirc; ++i) L += terms[i];
  *loss = L / ncirc;
  return QS_OK;
}

// ---- per-circuit gate programs --------------------------------------------------
// Each circuit runs its own op list (qs_qnn_op): Rx / Ry / Rz on a logical qubit
// with a shared trainable angle theta[param] or a fixed value, Ry(x[c, j])
// encodings, CX (a GF(2) update of the qubit masks, no amplitude moves) and CZ
// (one sign pass).  Forward, E_c = <Z_0>, lam = Z_0 psi, then the ops in reverse:
// a trainable rotation exp(-i t P / 2) contributes Im <lam|P|psi> (both at the
// point after the gate) to d E / d t before its inverse is applied to both;
// an encoding contributes the same to d E / d x[c, j].  One rotation per pass.
struct QnnProgArgs {
  int ncirc, nfeat, nparams, lds_max_width, max_width;
  const int32_t* order;   // circuits, widest first
  const int32_t* widths;
  const int32_t* off;     // ncirc + 1 op offsets
  const qs_qnn_op* ops;
  const double* x;        // ncirc x nfeat
  const double* target;
  const double* theta;    // nparams
  double* expval;
  double* loss_terms;
  double* grad_circ;      // ncirc x nparams
  double* grad_x;         // ncirc x nfeat
  void* slots;
  int* counter;
  double inv_ncirc;
};

// 2x2 rotation exp(-i t P / 2), P = X, Y, Z (kinds QS_QNN_RX, RY / ENC_RY, RZ)
template <typename R> __device__ __forceinline__ void rot_matrix(int axis, double t, cx<R>* u) {
  const double c = cos(0.5 * t), s = sin(0.5 * t);
  if (axis == 0) {  // X: [[c, -i s], [-i s, c]]
    u[0] = mk<R>((R)c, (R)0);
    u[1] = mk<R>((R)0, (R)-s);
    u[2] = mk<R>((R)0, (R)-s);
    u[3] = mk<R>((R)c, (R)0);
  } else if (axis == 1) {  // Y: [[c, -s], [s, c]]
    u[0] = mk<R>((R)c, (R)0);
    u[1] = mk<R>((R)-s, (R)0);
    u[2] = mk<R>((R)s, (R)0);
    u[3] = mk<R>((R)c, (R)0);
  } else {  // Z: diag(e^{-i t/2}, e^{i t/2})
    u[0] = mk<R>((R)c, (R)-s);
    u[1] = mk<R>((R)0, (R)0);
    u[2] = mk<R>((R)0, (R)0);
    u[3] = mk<R>((R)c, (R)s);
  }
}

__device__ __forceinline__ int op_axis(int kind) { return kind == QS_QNN_RX ? 0 : (kind == QS_QNN_RZ ? 2 : 1); }

template <typename R>
__global__ __launch_bounds__(1024) void k_qnn_prog(QnnProgArgs A) {
  extern __shared__ __align__(16) char lds_raw[];
  __shared__ double red[64];
  __shared__ uint64_t cm[QNN_MAX_W], rm[QNN_MAX_W];
  __shared__ int cur;
  const int tid = threadIdx.x, nt = blockDim.x;
  cx<R>* slot_psi = reinterpret_cast<cx<R>*>(A.slots) + (uint64_t)blockIdx.x * 2 * (1ull << A.max_width);
  cx<R>* slot_lam = slot_psi + (1ull << A.max_width);
  for (;;) {
    if (tid == 0) cur = atomicAdd(A.counter, 1);
    __syncthreads();
    const int k = cur;
    __syncthreads();
    if (k >= A.ncirc) break;
    const int c = A.order[k];
    const int w = A.widths[c];
    const uint64_t N = 1ull << w, half = N >> 1;
    cx<R>* psi;
    cx<R>* lam;
    if (w <= A.lds_max_width) {
      psi = reinterpret_cast<cx<R>*>(lds_raw);
      lam = psi + N;
    } else {
      psi = slot_psi;
      lam = slot_lam;
    }
    const qs_qnn_op* ops = A.ops + A.off[c];
    const int nops = A.off[c + 1] - A.off[c];
    if (tid < w) cm[tid] = rm[tid] = 1ull << (w - 1 - tid);
    for (uint64_t i = tid; i < N; i += nt) st(psi + i, mk<R>((R)(i == 0 ? 1 : 0), (R)0));
    __syncthreads();
    // forward
    for (int o = 0; o < nops; ++o) {
      const qs_qnn_op op = ops[o];
      if (op.kind == QS_QNN_CX) {
        if (tid == 0) {
          rm[op.q1] ^= rm[op.q0];
          cm[op.q0] ^= cm[op.q1];
        }
      } else if (op.kind == QS_QNN_CZ) {
        const uint64_t ra = rm[op.q0], rb = rm[op.q1];
        for (uint64_t i = tid; i < N; i += nt)
          if (parity64(i & ra) & parity64(i & rb)) {
            const cx<R> a = ld(psi + i);
            st(psi + i, mk<R>(-a.re, -a.im));
          }
      } else {
        const double t = op.kind == QS_QNN_ENC_RY ? A.x[(uint64_t)c * A.nfeat + op.param]
                                                  : (op.param >= 0 ? A.theta[op.param] : op.value);
        cx<R> u[4];
        rot_matrix<R>(op_axis(op.kind), t, u);
        const uint64_t m = cm[op.q0], r = rm[op.q0];
        for (uint64_t h = tid; h < half; h += nt) {
          uint64_t p0, p1;
          pair_of(h, m, r, p0, p1);
          const cx<R> a0 = ld(psi + p0), a1 = ld(psi + p1);
          st(psi + p0, cfma(mul(u[0], a0), u[1], a1));
          st(psi + p1, cfma(mul(u[2], a0), u[3], a1));
        }
      }
      __syncthreads();
    }
    double e = 0;
    {
      const uint64_t r0 = rm[0];
      for (uint64_t i = tid; i < N; i += nt) {
        const cx<R> a = ld(psi + i);
        const double pr = (double)a.re * a.re + (double)a.im * a.im;
        const bool one = parity64(i & r0);
        e += one ? -pr : pr;
        st(lam + i, one ? mk<R>(-a.re, -a.im) : a);
      }
    }
    e = block_reduce<R>(e, red);
    const double tgt = A.target[c];
    const double dl = 2.0 * (e - tgt) * A.inv_ncirc;
    double* grow = A.grad_circ + (uint64_t)c * A.nparams;
    for (int i = tid; i < A.nparams; i += nt) grow[i] = 0.0;
    for (int j = tid; j < A.nfeat; j += nt) A.grad_x[(uint64_t)c * A.nfeat + j] = 0.0;
    __syncthreads();
    // backward
    for (int o = nops - 1; o >= 0; --o) {
      const qs_qnn_op op = ops[o];
      if (op.kind == QS_QNN_CX) {
        if (tid == 0) {
          rm[op.q1] ^= rm[op.q0];
          cm[op.q0] ^= cm[op.q1];
        }
      } else if (op.kind == QS_QNN_CZ) {
        const uint64_t ra = rm[op.q0], rb = rm[op.q1];
        for (uint64_t i = tid; i < N; i += nt)
          if (parity64(i & ra) & parity64(i & rb)) {
            const cx<R> a = ld(psi + i), b = ld(lam + i);
            st(psi + i, mk<R>(-a.re, -a.im));
            st(lam + i, mk<R>(-b.re, -b.im));
          }
      } else {
        const bool enc = op.kind == QS_QNN_ENC_RY;
        const bool train = enc || op.param >= 0;
        const int axis = op_axis(op.kind);
        const double t = enc ? A.x[(uint64_t)c * A.nfeat + op.param] : (op.param >= 0 ? A.theta[op.param] : op.value);
        cx<R> u[4];
        rot_matrix<R>(axis, -t, u);  // the inverse
        const uint64_t m = cm[op.q0], r = rm[op.q0];
        double g = 0;
        for (uint64_t h = tid; h < half; h += nt) {
          uint64_t p0, p1;
          pair_of(h, m, r, p0, p1);
          const cx<R> a0 = ld(psi + p0), a1 = ld(psi + p1), b0 = ld(lam + p0), b1 = ld(lam + p1);
          if (train) {
            // Im <lam|P|psi>: X psi = (a1, a0); Y psi = (-i a1, i a0); Z psi = (a0, -a1)
            if (axis == 0)
              g += ((double)b0.re * a1.im - (double)b0.im * a1.re) + ((double)b1.re * a0.im - (double)b1.im * a0.re);
            else if (axis == 1)
              g += -((double)b0.re * a1.re + (double)b0.im * a1.im) + ((double)b1.re * a0.re + (double)b1.im * a0.im);
            else
              g += ((double)b0.re * a0.im - (double)b0.im * a0.re) - ((double)b1.re * a1.im - (double)b1.im * a1.re);
          }
          st(psi + p0, cfma(mul(u[0], a0), u[1], a1));
          st(psi + p1, cfma(mul(u[2], a0), u[3], a1));
          st(lam + p0, cfma(mul(u[0], b0), u[1], b1));
          st(lam + p1, cfma(mul(u[2], b0), u[3], b1));
        }
        if (train) {
          double dummy = 0;
          block_reduce2<R>(g, dummy, red);
          if (tid == 0) {
            if (enc) A.grad_x[(uint64_t)c * A.nfeat + op.param] += dl * g;
            else grow[op.param] += dl * g;
          }
        }
      }
      __syncthreads();
    }
    if (tid == 0) {
      A.expval[c] = e;
      A.loss_terms[c] = (e - tgt) * (e - tgt);
    }
    __syncthreads();
  }
}

template <typename R>
static int qnn_prog_t(qs_ctx* ctx, int ncirc, const int32_t* widths, const int32_t* off, const qs_qnn_op* ops,
                      int nparams, int nfeat, const double* x, const double* target, const double* theta,
                      double* expval, double* loss, double* grad_theta, double* grad_x, const qs_qnn_config* cfg,
                      hipStream_t s) {
  const int lds_w = cfg ? cfg->lds_max_width : 11;
  const int threads = cfg ? cfg->block_threads : 256;
  const int per_cu = cfg ? cfg->blocks_per_cu : 2;
  QS_REQUIRE(threads == 64 || threads == 128 || threads == 256 || threads == 512 || threads == 1024,
             "block_threads must be a power of two in [64, 1024]");
  QS_REQUIRE(lds_w >= 0 && lds_w <= 13, "lds_max_width must be in [0, 13]");
  QS_REQUIRE(per_cu >= 1 && per_cu <= 8, "blocks_per_cu must be in [1, 8]");
  const size_t lds_bytes = lds_w > 0 ? (size_t)2 * (1ull << lds_w) * sizeof(cx<R>) : 0;
  QS_REQUIRE(lds_bytes <= 150 * 1024, "LDS state too large for one workgroup");
  int max_width = 1;
  for (int i = 0; i < ncirc; ++i) max_width = std::max(max_width, (int)widths[i]);
  int cus = 0;
  QS_CHECK_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
  const int blocks = std::max(1, cus * per_cu);
  const int nops = off[ncirc];
  auto al = [](uint64_t b) { return (b + 255) & ~255ull; };
  const uint64_t np = std::max(nparams, 1), nf = std::max(nfeat, 1);
  const uint64_t sz_i = al((uint64_t)ncirc * sizeof(int32_t)), sz_o = al((uint64_t)(ncirc + 1) * sizeof(int32_t)),
                 sz_ops = al((uint64_t)std::max(nops, 1) * sizeof(qs_qnn_op)),
                 sz_x = al((uint64_t)ncirc * nf * sizeof(double)), sz_c = al((uint64_t)ncirc * sizeof(double)),
                 sz_t = al(np * sizeof(double)), sz_gc = al((uint64_t)ncirc * np * sizeof(double));
  const uint64_t slot_bytes = max_width > lds_w ? (uint64_t)blocks * 2 * (1ull << max_width) * sizeof(cx<R>) : 0;
  const uint64_t total = 2 * sz_i + sz_o + sz_ops + 2 * sz_x + 3 * sz_c + 2 * sz_t + 256 + sz_gc + slot_bytes;
  int rc = ensure_scratch(ctx, total);
  if (rc) return rc;
  char* b = (char*)ctx->scratch;
  int32_t* d_order = (int32_t*)b;
  b += sz_i;
  int32_t* d_w = (int32_t*)b;
  b += sz_i;
  int32_t* d_off = (int32_t*)b;
  b += sz_o;
  qs_qnn_op* d_ops = (qs_qnn_op*)b;
  b += sz_ops;
  double* d_x = (double*)b;
  b += sz_x;
  double* d_gx = (double*)b;
  b += sz_x;
  double* d_t = (double*)b;
  b += sz_c;
  double* d_e = (double*)b;
  b += sz_c;
  double* d_l = (double*)b;
  b += sz_c;
  double* d_th = (double*)b;
  b += sz_t;
  double* d_gth = (double*)b;
  b += sz_t;
  int* d_cnt = (int*)b;
  b += 256;
  double* d_gc = (double*)b;
  b += sz_gc;
  void* d_slots = b;
  std::vector<int32_t> order(ncirc);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int c2) { return widths[a] > widths[c2]; });
  QS_CHECK_HIP(hipMemcpyAsync(d_order, order.data(), ncirc * sizeof(int32_t), hipMemcpyHostToDevice, s));
  QS_CHECK_HIP(hipMemcpyAsync(d_w, widths, ncirc * sizeof(int32_t), hipMemcpyHostToDevice, s));
  QS_CHECK_HIP(hipMemcpyAsync(d_off, off, (ncirc + 1) * sizeof(int32_t), hipMemcpyHostToDevice, s));
  if (nops) QS_CHECK_HIP(hipMemcpyAsync(d_ops, ops, nops * sizeof(qs_qnn_op), hipMemcpyHostToDevice, s));
  if (nfeat) QS_CHECK_HIP(hipMemcpyAsync(d_x, x, (uint64_t)ncirc * nfeat * sizeof(double), hipMemcpyHostToDevice, s));
  QS_CHECK_HIP(hipMemcpyAsync(d_t, target, ncirc * sizeof(double), hipMemcpyHostToDevice, s));
  if (nparams) QS_CHECK_HIP(hipMemcpyAsync(d_th, theta, nparams * sizeof(double), hipMemcpyHostToDevice, s));
  QnnProgArgs A;
  A.ncirc = ncirc;
  A.nfeat = nfeat;
  A.nparams = nparams;
  A.lds_max_width = lds_w;
  A.max_width = max_width;
  A.order = d_order;
  A.widths = d_w;
  A.off = d_off;
  A.ops = d_ops;
  A.x = d_x;
  A.target = d_t;
  A.theta = d_th;
  A.expval = d_e;
  A.loss_terms = d_l;
  A.grad_circ = d_gc;
  A.grad_x = d_gx;
  A.slots = d_slots;
  A.counter = d_cnt;
  A.inv_ncirc = 1.0 / ncirc;
  if (lds_bytes > 64 * 1024)
    QS_CHECK_HIP(hipFuncSetAttribute((const void*)k_qnn_prog<R>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)lds_bytes));
  rc = prof_begin(ctx, PROF_QNN, s);
  if (rc) return rc;
  hipLaunchKernelGGL(k_qnn_clear, dim3(1), dim3(64), 0, s, d_cnt);
  QS_CHECK_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_qnn_prog<R>, dim3(blocks), dim3(threads), lds_bytes, s, A);
  QS_CHECK_HIP(hipGetLastError());
  if (nparams) {
    hipLaunchKernelGGL(k_qnn_reduce, dim3((unsigned)((nparams + 31) / 32)), dim3(256), 0, s, d_gc, ncirc, nparams,
                       d_gth);
    QS_CHECK_HIP(hipGetLastError());
  }
  rc = prof_end(ctx, s);
  if (rc) return rc;
  std::vector<double> lt(ncirc);
  QS_CHECK_HIP(hipMemcpyAsync(expval, d_e, ncirc * sizeof(double), hipMemcpyDeviceToHost, s));
  QS_CHECK_HIP(hipMemcpyAsync(lt.data(), d_l, ncirc * sizeof(double), hipMemcpyDeviceToHost, s));
  if (nparams) QS_CHECK_HIP(hipMemcpyAsync(grad_theta, d_gth, nparams * sizeof(double), hipMemcpyDeviceToHost, s));
  if (grad_x && nfeat)
    QS_CHECK_HIP(hipMemcpyAsync(grad_x, d_gx, (uint64_t)ncirc * nfeat * sizeof(double), hipMemcpyDeviceToHost, s));
  QS_CHECK_HIP(hipStreamSynchronize(s));
  double L = 0;
  for (int i = 0; i < ncirc; ++i) L += lt[i];
  *loss = L / ncirc;
  return QS_OK;
}

}  // namespace qs

using namespace qs;

extern "C" int qs_qnn_batch(qs_ctx* ctx, int dtype, int ncirc, const int32_t* widths, int nfeat, const double* x,
                            const double* target, int layers, int max_width, const double* theta, double* expval,
                            double* loss, double* grad_theta, double* grad_x, const qs_qnn_config* cfg,
                            void* stream) {
  QS_REQUIRE(ctx && widths && x && target && theta && expval && loss && grad_theta, "null argument");
  QS_REQUIRE(dtype == QS_C64 || dtype == QS_C128, "dtype must be QS_C64 or QS_C128");
  QS_REQUIRE(ncirc >= 1 && nfeat >= 0 && layers >= 1 && layers <= QNN_MAX_LAYERS, "bad batch shape");
  QS_REQUIRE(max_width >= 1 && max_width <= QNN_MAX_W, "max_width must be in [1, 20]");
  for (int i = 0; i < ncirc; ++i) QS_REQUIRE(widths[i] >= 2 && widths[i] <= max_width, "width out of range");
  int rc = qnn_check(cfg, dtype);
  if (rc) return rc;
  try {
    return dtype == QS_C128 ? qnn_planned(ctx, ncirc, widths, nfeat, x, target, layers, max_width, theta, expval, loss,
                                          grad_theta, grad_x)
                            : qnn_c64(ctx, cfg && cfg->fuse_qubits ? cfg->fuse_qubits : 1, ncirc, widths, nfeat, x, target, layers, max_width, theta, expval, loss,
                                      grad_theta, grad_x);
  } catch (const std::exception& e) {
    set_error(std::string("batch of variational circuits: ") + e.what());
    return QS_ERR_DEVICE;
  }
}

extern "C" int qs_qnn_batch_programs(qs_ctx* ctx, int dtype, int ncirc, const int32_t* widths,
                                     const int32_t* prog_offsets, const qs_qnn_op* ops, int nparams, int nfeat,
                                     const double* x, const double* target, const double* theta, double* expval,
                                     double* loss, double* grad_theta, double* grad_x, const qs_qnn_config* cfg,
                                     void* stream) {
  QS_REQUIRE(ctx && widths && prog_offsets && target && expval && loss, "null argument");
  QS_REQUIRE(dtype == QS_C64 || dtype == QS_C128, "dtype must be QS_C64 or QS_C128");
  QS_REQUIRE(ncirc >= 1 && nparams >= 0 && nfeat >= 0, "bad batch shape");
  QS_REQUIRE(nparams == 0 || (theta && grad_theta), "theta / grad_theta missing");
  QS_REQUIRE(nfeat == 0 || x, "x missing");
  QS_REQUIRE(prog_offsets[0] == 0, "prog_offsets[0] must be 0");
  for (int c = 0; c < ncirc; ++c) {
    const int w = widths[c];
    QS_REQUIRE(w >= 1 && w <= QNN_MAX_W, "width out of range [1, 20]");
    QS_REQUIRE(prog_offsets[c + 1] >= prog_offsets[c], "prog_offsets must not decrease");
    QS_REQUIRE(prog_offsets[c + 1] == prog_offsets[c] || ops, "ops missing");
    for (int o = prog_offsets[c]; o < prog_offsets[c + 1]; ++o) {
      const qs_qnn_op& op = ops[o];
      QS_REQUIRE(op.kind >= QS_QNN_RX && op.kind <= QS_QNN_ENC_RY, "unknown op kind");
      QS_REQUIRE(op.q0 >= 0 && op.q0 < w, "op qubit out of range");
      if (op.kind == QS_QNN_CX || op.kind == QS_QNN_CZ)
        QS_REQUIRE(op.q1 >= 0 && op.q1 < w && op.q1 != op.q0, "two-qubit op needs two distinct qubits");
      if (op.kind == QS_QNN_ENC_RY) QS_REQUIRE(op.param >= 0 && op.param < nfeat, "encoding feature out of range");
      else if (op.kind <= QS_QNN_RZ) QS_REQUIRE(op.param < nparams, "parameter index out of range");
    }
  }
  if (dtype == QS_C128)
    return qnn_prog_t<double>(ctx, ncirc, widths, prog_offsets, ops, nparams, nfeat, x, target, theta, expval, loss,
                              grad_theta, grad_x, cfg, as_stream(stream));
  return qnn_prog_t<float>(ctx, ncirc, widths, prog_offsets, ops, nparams, nfeat, x, target, theta, expval, loss,
                           grad_theta, grad_x, cfg, as_stream(stream));
}
