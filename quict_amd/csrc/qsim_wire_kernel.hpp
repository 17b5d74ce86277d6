// The tile pass of programs planned in wires (qsim_wire_plan.hpp): op
// interpreter and kernel.
//
// What bounds it: with 3 to 4 times fewer passes than k_fused each pass carries
// 30 to 60 ops, and a wave's instructions are what a pass waits for.  So the ops are
// written to need few of them and no copies of the tile: 2171 vector and 1839 scalar
// instructions a wave in a 30-qubit pass of about 63 ops, the vector ALU busy 60% of
// the time with four waves a SIMD:
//   * every op changes its registers in place.  A rotation is three shears,
//     x0 += t x1, x1 += s x0, x0 += t x1 (t = -tan(theta / 2), s = sin(theta),
//     |theta| <= pi / 2, so |t| <= 1): 3 fused multiply-adds per component pair
//     instead of 4, and no value outlives its successor, so the compiler keeps one
//     register set.  k_fused's ops read and write two sets and need 162 VGPRs;
//   * a phase touches only the amplitudes it changes, again as shears (of the real
//     and imaginary parts) when its angle is at most pi / 2;
//   * ops that do not apply to the tile are skipped, one opcode selects the op,
//     and ops that few circuits need live in a second instance (HEAVY).
#pragma once
#include "qsim_fused_kernel.hpp"
#include "qsim_wires.hpp"

namespace qs {

// ---- ops, in place -----------------------------------------------------------------

template <typename R, int NR, int P>
__device__ __forceinline__ void wo_rot(cx<R> (&a)[NR], cx<R> ts) {
  const R t = ts.re, s = ts.im;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (r & (1 << P)) continue;
    cx<R>&x0 = a[r], &x1 = a[r | (1 << P)];
    x0.re = rfma(t, x1.re, x0.re);
    x0.im = rfma(t, x1.im, x0.im);
    x1.re = rfma(s, x0.re, x1.re);
    x1.im = rfma(s, x0.im, x1.im);
    x0.re = rfma(t, x1.re, x0.re);
    x0.im = rfma(t, x1.im, x0.im);
  }
}

// Exchange in place (v_swap_b32).  Written as assignments the exchange would make
// the compiler rename the pair's registers in this one arm of the op switch, and
// copy the tile back in all the others.
__device__ __forceinline__ void swap_bits(float& x, float& y) {
  asm volatile("v_swap_b32 %0, %1" : "+v"(x), "+v"(y));
}
__device__ __forceinline__ void swap_bits(double& x, double& y) {
  uint64_t u = __builtin_bit_cast(uint64_t, x), w = __builtin_bit_cast(uint64_t, y);
  uint32_t u0 = (uint32_t)u, u1 = (uint32_t)(u >> 32), w0 = (uint32_t)w, w1 = (uint32_t)(w >> 32);
  asm volatile("v_swap_b32 %0, %2\n\tv_swap_b32 %1, %3" : "+v"(u0), "+v"(u1), "+v"(w0), "+v"(w1));
  x = __builtin_bit_cast(double, (uint64_t)u1 << 32 | u0);
  y = __builtin_bit_cast(double, (uint64_t)w1 << 32 | w0);
}

template <typename R, int NR, int P, int C>
__device__ __forceinline__ void wo_ex(cx<R> (&a)[NR]) {
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if ((r & (1 << P)) || (C >= 0 && !((r >> (C & 31)) & 1))) continue;
    swap_bits(a[r].re, a[r | (1 << P)].re);
    swap_bits(a[r].im, a[r | (1 << P)].im);
  }
}

// x *= f in place: both cross products before either part changes.
template <typename R> __device__ __forceinline__ void mul_in_place(cx<R>& x, cx<R> f) {
  const R u = f.im * x.im, w = f.im * x.re;
  x.re = rfma(f.re, x.re, -u);
  x.im = rfma(f.re, x.im, w);
}

// The amplitudes whose register bits in MASK are all 1 times f (MODE 0), a real
// factor (1), the unit number of the shear pair f (2) or minus that (3: the signs
// are operand modifiers).
template <typename R, int NR, uint32_t MASK, int MODE>
__device__ __forceinline__ void wo_phase(cx<R> (&a)[NR], cx<R> f) {
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (((uint32_t)r & MASK) != MASK) continue;
    cx<R>& x = a[r];
    if constexpr (MODE == 1) {
      x.re = f.re * x.re;
      x.im = f.re * x.im;
    } else if constexpr (MODE == 2) {
      x.re = rfma(f.re, x.im, x.re);
      x.im = rfma(f.im, x.re, x.im);
      x.re = rfma(f.re, x.im, x.re);
    } else if constexpr (MODE == 3) {
      x.re = rfma(f.re, x.im, x.re);
      x.im = rfma(-f.im, x.re, -x.im);
      x.re = rfma(f.re, x.im, -x.re);
    } else {
      mul_in_place(x, f);
    }
  }
}

template <typename R, int NR, int P>
__device__ __forceinline__ void wo_u2(cx<R> (&a)[NR], const cx<R>* m) {
  const cx<R> m00 = m[0], m01 = m[1], m10 = m[2], m11 = m[3];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (r & (1 << P)) continue;
    cx<R>&x0 = a[r], &x1 = a[r | (1 << P)];
    // the parts that need the other three components first, then each component
    // times its real diagonal entry, in place
    R p0r = m01.re * x1.re, p0i = m01.re * x1.im, p1r = m10.re * x0.re, p1i = m10.re * x0.im;
    p0r = rfma(-m01.im, x1.im, p0r);
    p0i = rfma(m01.im, x1.re, p0i);
    p1r = rfma(-m10.im, x0.im, p1r);
    p1i = rfma(m10.im, x0.re, p1i);
    p0r = rfma(-m00.im, x0.im, p0r);
    p0i = rfma(m00.im, x0.re, p0i);
    p1r = rfma(-m11.im, x1.im, p1r);
    p1i = rfma(m11.im, x1.re, p1i);
    x0.re = rfma(m00.re, x0.re, p0r);
    x0.im = rfma(m00.re, x0.im, p0i);
    x1.re = rfma(m11.re, x1.re, p1r);
    x1.im = rfma(m11.re, x1.im, p1i);
  }
}

// Relayout in two rounds (see relayout_half) of NV tiles, each through a half-tile
// image of its own, so that they share the barriers; or (IMAGES = 1) one after another
// through the same image: half the LDS, so that a CU holds three workgroups of two
// complex128 tiles instead of two.
template <typename R, int RB, int TB, int NV, int IMAGES, int P>
__device__ __forceinline__ void wire_relayout(cx<R> (&a)[NV][1 << RB], char* lds, const uint32_t* __restrict__ x,
                                              bool tile_flips, uint32_t tid, uint32_t blk) {
  constexpr int NR = 1 << RB;
  constexpr uint32_t image = (uint32_t)sizeof(cx<R>) << (RB + TB - 1);
  uint32_t lw[RB], lq[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) lw[b] = x[1 + b];
  uint32_t w = thr_off<TB>(x + 1 + RB, tid) ^ x[1 + RB + TB];
  const uint32_t* y = x + 2 + RB + TB;
  if (tile_flips) {
    const uint32_t* z = y + RB + TB;
    const uint32_t nz = z[0];
    uint32_t f = 0;
    for (uint32_t i = 0; i < nz; ++i) f ^= ((blk >> z[1 + 2 * i]) & 1u) ? z[2 + 2 * i] : 0u;
    w ^= f;
  }
#pragma unroll
  for (int b = 0; b < RB; ++b) lq[b] = y[b];
  const uint32_t rd = thr_off<TB>(y + RB, tid);
#pragma unroll
  for (int k = 0; k < 2 * (NV / IMAGES); ++k) {
    const int v0 = IMAGES == NV ? 0 : k >> 1, v1 = IMAGES == NV ? NV : v0 + 1;
    lds_barrier();
#pragma unroll
    for (int r = 0; r < NR; ++r)
      if (((r >> P) & 1) == (k & 1)) {
        const uint32_t o = w ^ reg_off<RB>(r, lw);
#pragma unroll
        for (int v = v0; v < v1; ++v) st_lds<R>(lds + (v - v0) * image, o, a[v][r]);
      }
    lds_barrier();
#pragma unroll
    for (int r = 0; r < NR; ++r)
      if (((r >> P) & 1) == (k & 1)) {
        const uint32_t o = rd ^ reg_off<RB>(r, lq);
#pragma unroll
        for (int v = v0; v < v1; ++v) a[v][r] = ld_lds<R>(lds + (v - v0) * image, o);
      }
  }
}

// Lane moves within the 64 lanes of a wave (DPP): lanes without a source add 0.
template <int CTRL, int ROWS> __device__ __forceinline__ double wave_move(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, CTRL, ROWS, 0xf, false),
                          __builtin_amdgcn_update_dpp(0, lo, CTRL, ROWS, 0xf, false));
}
// The sum over the wave, in lane 63.
__device__ __forceinline__ double wave_total(double v) {
  v += wave_move<0x111, 0xf>(v);  // row_shr:1
  v += wave_move<0x112, 0xf>(v);  // row_shr:2
  v += wave_move<0x114, 0xf>(v);  // row_shr:4
  v += wave_move<0x118, 0xf>(v);  // row_shr:8
  v += wave_move<0x142, 0xa>(v);  // row_bcast:15
  v += wave_move<0x143, 0xc>(v);  // row_bcast:31
  return v;
}

// This lane's part of Im <lam|P|psi>, P = Z (Y false) or Y on register bit PB, in
// double for both precisions.
template <typename R, int NR, int PB, bool Y>
__device__ __forceinline__ double measure(const cx<R> (&psi)[NR], const cx<R> (&lam)[NR]) {
  double s0 = 0, s1 = 0;  // two chains
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (r & (1 << PB)) continue;
    const cx<R> a0 = psi[r], a1 = psi[r | (1 << PB)], b0 = lam[r], b1 = lam[r | (1 << PB)];
    if constexpr (Y) {  // Y psi = (-i a1, i a0)
      s0 = rfma((double)b1.re, (double)a0.re, s0);
      s0 = rfma((double)b1.im, (double)a0.im, s0);
      s1 = rfma((double)b0.re, (double)a1.re, s1);
      s1 = rfma((double)b0.im, (double)a1.im, s1);
    } else {
      s0 = rfma((double)b0.re, (double)a0.im, s0);
      s0 = rfma(-(double)b0.im, (double)a0.re, s0);
      s1 = rfma((double)b1.re, (double)a1.im, s1);
      s1 = rfma(-(double)b1.im, (double)a1.re, s1);
    }
  }
  return s0 - s1;
}
// The wave's part, in lane 63, which writes it to its place in the gradient row.
template <typename R, int NR, int PB, bool Y>
__device__ __forceinline__ void wo_measure(const cx<R> (&psi)[NR], const cx<R> (&lam)[NR], double* slot, uint32_t tid) {
  const double s = wave_total(measure<R, NR, PB, Y>(psi, lam));
  if ((tid & 63) == 63) *slot = s;
}
// Column Z, a phase, column Y, a rotation: a parameter pair of a gradient sweep.  The two
// columns share the steps of their sums: halves of the wave are exchanged first, then
// lanes 0..31 add up one and 32..63 the other.
template <typename R, int NR, int P, int MODE>
__device__ __forceinline__ void wo_back(cx<R> (&psi)[NR], cx<R> (&lam)[NR], cx<R> ph, cx<R> ts, double* slot_z,
                                        double* slot_y, uint32_t tid) {
  const double z = measure<R, NR, P, false>(psi, lam);
  wo_phase<R, NR, 1u << P, MODE>(psi, ph);
  wo_phase<R, NR, 1u << P, MODE>(lam, ph);
  const double y = measure<R, NR, P, true>(psi, lam);
  wo_rot<R, NR, P>(psi, ts);
  wo_rot<R, NR, P>(lam, ts);
  const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)__double2loint(z), (uint32_t)__double2loint(y), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)__double2hiint(z), (uint32_t)__double2hiint(y), false, false);
  double s = __hiloint2double((int)hi[0], (int)lo[0]) + __hiloint2double((int)hi[1], (int)lo[1]);
  s += wave_move<0x111, 0xf>(s);
  s += wave_move<0x112, 0xf>(s);
  s += wave_move<0x114, 0xf>(s);
  s += wave_move<0x118, 0xf>(s);
  s += wave_move<0x142, 0xa>(s);
  if ((tid & 31) == 31) *(tid & 32 ? slot_y : slot_z) = s;
}

// One op on NV vectors (2: psi and lam of a gradient sweep); grad: this wave's column
// 0 of the tile's gradient row.
template <typename R, int RB, int TB, int NV, int IMAGES, bool HEAVY>
__device__ __forceinline__ void wire_op(cx<R> (&a)[NV][1 << RB], char* lds, const WireOp<R>& e, const cx<R>* __restrict__ C,
                                        const cx<R>* __restrict__ G, const uint32_t* __restrict__ X, uint32_t tid,
                                        uint32_t blk, double* grad) {
  static_assert(RB == 4, "opcodes are laid out for four register bits");
  constexpr int NR = 1 << RB;
  const uint32_t code = e.w[0] & 0xff;
  const uint32_t cthr = e.w[3] & 0xffff;
  const bool tok = (tid & cthr) == e.w[3] >> 16;
  const cx<R>* g = G + e.w[2];  // uniform payloads, through scalar loads
#define QS_V(...)                                  \
  _Pragma("unroll") for (int v = 0; v < NV; ++v) { \
    __VA_ARGS__;                                   \
  }
#define QS_4(X) X(0) X(1) X(2) X(3)
  if (code < WC_HOT) {
    switch (code) {
#define QS_ROT(P) case WC_ROT + P: QS_V(wo_rot<R, NR, P>(a[v], e.f[0])) break;
      QS_4(QS_ROT)
#define QS_RP(BASE, MODE, P)                            \
  case BASE + P:                                        \
    QS_V(wo_rot<R, NR, P>(a[v], e.f[0]))                \
    QS_V(wo_phase<R, NR, 1u << P, MODE>(a[v], e.f[1]))  \
    break;
#define QS_PR(BASE, MODE, P)                            \
  case BASE + P:                                        \
    QS_V(wo_phase<R, NR, 1u << P, MODE>(a[v], e.f[0]))  \
    QS_V(wo_rot<R, NR, P>(a[v], e.f[1]))                \
    break;
#define QS_BW(BASE, MODE, P)                                                                                     \
  case BASE + P:                                                                                                 \
    if constexpr (NV == 2)                                                                                       \
      wo_back<R, NR, P, MODE>(a[0], a[1], e.f[0], e.f[1], grad + (e.w[2] << (TB - 6)), grad + (e.w[5] << (TB - 6)), tid); \
    else __builtin_unreachable();                                                                                \
    break;
#define QS_HOT(P) \
  QS_RP(WC_RP, 2, P) QS_RP(WC_RPS, 3, P) QS_PR(WC_PR, 2, P) QS_PR(WC_PRS, 3, P) QS_BW(WC_BW, 2, P) QS_BW(WC_BWS, 3, P)
      QS_4(QS_HOT)
      default: __builtin_unreachable();
    }
    return;
  }
  switch (code) {
    case WC_RELAYOUT: {
      const uint32_t* x = X + e.w[2];
      const bool tf = e.w[4] != 0;
      switch (x[0]) {
        case 0: wire_relayout<R, RB, TB, NV, IMAGES, 0>(a, lds, x, tf, tid, blk); break;
        case 1: wire_relayout<R, RB, TB, NV, IMAGES, 1>(a, lds, x, tf, tid, blk); break;
        case 2: wire_relayout<R, RB, TB, NV, IMAGES, 2>(a, lds, x, tf, tid, blk); break;
        case 3: wire_relayout<R, RB, TB, NV, IMAGES, 3>(a, lds, x, tf, tid, blk); break;
        default: __builtin_unreachable();
      }
      break;
    }
#define QS_16(X) X(0) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14) X(15)
#define QS_EX(P) case WC_EX + P: QS_V(wo_ex<R, NR, P, -1>(a[v])) break;
    QS_4(QS_EX)
#define QS_EXT(P) case WC_EXT + P: if (tok) QS_V(wo_ex<R, NR, P, -1>(a[v])) break;
    QS_4(QS_EXT)
#define QS_EXC(Q)                                                            \
  case WC_EXC + Q:                                                           \
    if constexpr (Q / 4 != Q % 4) QS_V(wo_ex<R, NR, Q / 4, Q % 4>(a[v]))     \
    else __builtin_unreachable();                                            \
    break;
    QS_16(QS_EXC)
// lanes whose thread bits fail sit these out: a wave all of whose lanes do skips the op
#define QS_PH(BASE, MODE, M) case BASE + M: if (tok) QS_V(wo_phase<R, NR, M, MODE>(a[v], e.f[0])) break;
#define QS_PHR(M) QS_PH(WC_PHR, 2, M)
    QS_16(QS_PHR)
#define QS_PHS(M) QS_PH(WC_PHS, 3, M)
    QS_16(QS_PHS)
#define QS_PHN(M) QS_PH(WC_PHN, 1, M)
    QS_16(QS_PHN)
    case WC_TABLE:
    case WC_LANE: {
      const uint32_t s = diag_sel((int)(e.w[0] >> 24), (int)(e.w[1] & 0xff), (int)((e.w[1] >> 8) & 0xff), tid);
      const cx<R>* T = C + e.w[2] + (code == WC_LANE ? s : s * NR);
      const int step = code == WC_LANE ? 0 : 1;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const cx<R> f = ld(T + r * step);
        QS_V(mul_in_place(a[v][r], f))
      }
      break;
    }
#define QS_U2(P) case WC_U2 + P: QS_V(wo_u2<R, NR, P>(a[v], g)) break;
    QS_4(QS_U2)
#define QS_MZ(P)                                                                                        \
  case WC_MZ + P:                                                                                       \
    if constexpr (NV == 2) wo_measure<R, NR, P, false>(a[0], a[1], grad + (e.w[2] << (TB - 6)), tid);   \
    else __builtin_unreachable();                                                                       \
    break;
    QS_4(QS_MZ)
#define QS_MY(P)                                                                                        \
  case WC_MY + P:                                                                                       \
    if constexpr (NV == 2) wo_measure<R, NR, P, true>(a[0], a[1], grad + (e.w[2] << (TB - 6)), tid);    \
    else __builtin_unreachable();                                                                       \
    break;
    QS_4(QS_MY)
    default: {
      if constexpr (HEAVY) {
        const uint32_t creg = (e.w[0] >> 8) & 0xff, cregv = (e.w[0] >> 16) & 0xff;
        const bool pure = e.w[5] != 0;
        switch (code) {
#define QS_PHC(M) QS_PH(WC_PHC, 0, M)
          QS_16(QS_PHC)
#define QS_U2G(P) case WC_U2G + P: QS_V(do_dense1<R, NR, P, 3>(a[v], g, creg, cregv, tok)) break;
          QS_4(QS_U2G)
#define QS_EXG(P)                                                          \
  case WC_EXG + P:                                                         \
    if (pure) QS_V(do_perm1<R, NR, P, 3, true>(a[v], g, creg, cregv, tok)) \
    else QS_V(do_perm1<R, NR, P, 3, false>(a[v], g, creg, cregv, tok))     \
    break;
          QS_4(QS_EXG)
#define QS_PAIR(A, B)                                                                            \
  case WC_D2 + A * (A - 1) / 2 + B: QS_V(do_dense2<R, NR, A, B, 3>(a[v], g, creg, cregv, tok)) break; \
  case WC_XX + A * (A - 1) / 2 + B: QS_V(do_xx2<R, NR, A, B, false>(a[v], g)) break;               \
  case WC_SW + A * (A - 1) / 2 + B:                                                              \
    if (pure) QS_V(do_swap2<R, NR, A, B, 3, true>(a[v], g, creg, cregv, tok))                    \
    else QS_V(do_swap2<R, NR, A, B, 3, false>(a[v], g, creg, cregv, tok))                        \
    break;
          QS_PAIR(1, 0) QS_PAIR(2, 0) QS_PAIR(2, 1) QS_PAIR(3, 0) QS_PAIR(3, 1) QS_PAIR(3, 2)
          case WC_D3 + 0: QS_V(do_densek<R, NR, 3, 14u>(a[v], g, creg, cregv, tok)) break;
          case WC_D3 + 1: QS_V(do_densek<R, NR, 3, 13u>(a[v], g, creg, cregv, tok)) break;
          case WC_D3 + 2: QS_V(do_densek<R, NR, 3, 11u>(a[v], g, creg, cregv, tok)) break;
          case WC_D3 + 3: QS_V(do_densek<R, NR, 3, 7u>(a[v], g, creg, cregv, tok)) break;
          case WC_D4: QS_V(do_densek<R, NR, 4, 15u>(a[v], g, creg, cregv, tok)) break;
          default: __builtin_unreachable();
        }
      } else {
        __builtin_unreachable();
      }
    }
  }
}

// The wave's tiles from v (NV vectors at the same offsets).
template <typename R, int RB, int TB, int NV>
__device__ __forceinline__ void wire_load(cx<R> (&a)[NV][1 << RB], const cx<R>* const (&v)[NV],
                                          const PassHdr* __restrict__ H, uint64_t tb, uint32_t tid, uint32_t nsmall) {
  constexpr int NR = 1 << RB;
  uint64_t gin = 0;
#pragma unroll
  for (int b = 0; b < TB; ++b) gin |= (uint64_t)((tid >> b) & 1u) << H->tbits[H->ts0[b]];
  const uint64_t base = tb | gin;
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      uint64_t g = 0;
#pragma unroll
      for (int b = 0; b < RB; ++b)
        if ((r >> b) & 1) g |= 1ull << H->tbits[H->rs0[b]];
      if (nsmall == 0) a[i][r] = ld_nt(v[i] + (base | g));
      else a[i][r] = (uint32_t)(base | g) < nsmall ? ld(v[i] + (base | g)) : zero<R>();
    }
}

// The same for a vector with known zeros.
template <typename R, int RB, int TB>
__device__ __forceinline__ void wire_load_start(cx<R> (&a)[1 << RB], const cx<R>* v, const PassHdr* __restrict__ H,
                                                const PassStart& S, uint64_t tb, uint32_t tid) {
  uint64_t base = tb;
#pragma unroll
  for (int b = 0; b < TB; ++b) base |= (uint64_t)((tid >> b) & 1u) << H->tbits[H->ts0[b]];
#pragma unroll
  for (int r = 0; r < 1 << RB; ++r) {
    uint64_t g = 0;
#pragma unroll
    for (int b = 0; b < RB; ++b)
      if ((r >> b) & 1) g |= 1ull << H->tbits[H->rs0[b]];
    a[r] = start_load(S, v, base | g);
  }
}

// Store: per-lane and per-register address bits, flips that depend on the tile.
template <typename R, int RB, int TB, int NV>
__device__ __forceinline__ void wire_store(const cx<R> (&a)[NV][1 << RB], cx<R>* const (&v)[NV],
                                           const PassHdr* __restrict__ H, uint64_t tb, uint32_t tid, uint32_t blk,
                                           uint32_t nsmall) {
  constexpr int NR = 1 << RB;
  uint64_t base = tb ^ H->sflip;
#pragma unroll
  for (int b = 0; b < TB; ++b) base ^= ((tid >> b) & 1u) ? H->st[b] : 0ull;
  const int nx = H->nsx;
  for (int i = 0; i < nx; ++i) base ^= ((blk >> H->sxb[i]) & 1u) ? H->sxm[i] : 0ull;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    if (v[i] == nullptr) continue;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      uint64_t g = 0;
#pragma unroll
      for (int b = 0; b < RB; ++b)
        if ((r >> b) & 1) g ^= H->sr[b];
      if (nsmall == 0 || (uint32_t)(base ^ g) < nsmall) st_nt(v[i] + (base ^ g), a[i][r]);
    }
  }
}

// Touches the lines of a pass's ops and relayout constants, a 64-byte line a thread,
// so that they are in this XCD's L2 before the op loop asks for them one by one through
// the scalar cache: the program was written by a copy, a line's first use costs a trip
// to memory, and on a small register no other wave hides it.  Asked for before the tile,
// so that nothing waits for them alone.  20 qubits: graph replay 163 -> 139 us, gradient
// 1.09 -> 0.94 ms; 25 and 30 qubits: no difference.  (Scalar loads of the same lines by
// every wave: 191 us and 1.50 ms, the scalar cache answers them one after another.)
template <typename R, int TB>
__device__ __forceinline__ void touch_pass(const PassHdr* __restrict__ H, const WireOp<R>* __restrict__ ops,
                                           const uint32_t* __restrict__ aux, uint32_t tid, uint32_t& seen) {
  const char* p = reinterpret_cast<const char*>(ops + H->op0);
  const char* q = reinterpret_cast<const char*>(aux + H->aux0);
  const uint32_t np = (uint32_t)H->nops * (uint32_t)sizeof(WireOp<R>), nq = (uint32_t)H->naux * 4u;
  for (uint32_t i = 64 * tid; i < np; i += 64u << TB) seen ^= *reinterpret_cast<const uint32_t*>(p + i);
  for (uint32_t i = 64 * tid; i < nq; i += 64u << TB) seen ^= *reinterpret_cast<const uint32_t*>(q + i);
}

// The ops of a pass on the wave's tiles.  Returns the workgroup's gradient row in LDS
// (NV = 2): per column one entry a wave.
template <typename R, int RB, int TB, int NV, int IMAGES, bool HEAVY>
__device__ __forceinline__ double* wire_ops(cx<R> (&a)[NV][1 << RB], char* lds, const PassHdr* __restrict__ H,
                                            const WireOp<R>* __restrict__ ops, const cx<R>* __restrict__ coef,
                                            const uint32_t* __restrict__ aux, uint32_t tid, uint32_t blk) {
  constexpr int K = RB + TB;
  const WireOp<R>* P = ops + H->op0;
  const cx<R>* G = coef + H->coef0;
  // behind the relayout images: diagonal tables (read per lane), the gradient row
  cx<R>* C = reinterpret_cast<cx<R>*>(lds) + (H->uses_lds ? IMAGES << (K - 1) : 0);
  if (H->nstage) {
    for (int i = (int)tid; i < H->nstage; i += (int)blockDim.x) C[i] = G[i];
    __syncthreads();
  }
  double* row = reinterpret_cast<double*>(C + H->nstage);
  double* grad = row + (tid >> 6);
  const int nops = H->nops;
  WireOp<R> e = P[0];
  for (int o = 0; o < nops; ++o) {
    const WireOp<R> nx = P[o + 1];  // (past the last op: what follows in the program's memory)
    if ((blk & e.w[6]) == e.w[7]) wire_op<R, RB, TB, NV, IMAGES, HEAVY>(a, lds, e, C, G, aux, tid, blk, grad);
    e = nx;
  }
  return row;
}

// One workgroup, one tile: load, ops, store.  nsmall != 0: a register of nsmall
// amplitudes, fewer than a tile has; the rest of the tile is zeros.
template <typename R, int RB, int TB, bool HEAVY>
__global__ __launch_bounds__(1 << TB, HEAVY ? 2 : sizeof(R) == 8 ? 4 : 7) void k_wires(
    cx<R>* __restrict__ v, const PassHdr* __restrict__ H, const WireOp<R>* __restrict__ ops, const cx<R>* __restrict__ coef,
    const uint32_t* __restrict__ aux, uint32_t nsmall, const PassStart S) {
  extern __shared__ __align__(16) char lds_raw[];
  const uint32_t tid = threadIdx.x;
  uint32_t blk = blockIdx.x;
  cx<R> a[1][1 << RB];
  const uint64_t tb =
      S.fixed ? start_tile(S, blockIdx.x, H->sorted, RB + TB, blk) : insert_zeros((uint64_t)blk, H->sorted, RB + TB);
  uint32_t seen = 0;
  touch_pass<R, TB>(H, ops, aux, tid, seen);
  if (S.fixed) wire_load_start<R, RB, TB>(a[0], v, H, S, tb, tid);
  else wire_load<R, RB, TB, 1>(a, {v}, H, tb, tid, nsmall);
  asm volatile("" ::"v"(seen));
  wire_ops<R, RB, TB, 1, 1, HEAVY>(a, lds_raw, H, ops, coef, aux, tid, blk);
  if (H->sync_store) __syncthreads();
  wire_store<R, RB, TB, 1>(a, {v}, H, tb, tid, blk, nsmall);
}

// The same for one pass of several programs (jobs), each on its own part of psi (NV
// = 1) or of psi and lam (NV = 2, with the tile's gradient row).
template <typename R, int NV, int IMAGES, bool HEAVY>
__global__ __launch_bounds__(256, HEAVY || (IMAGES == 2 && sizeof(R) == 8) ? 2 : NV == 2 ? 3 : sizeof(R) == 8 ? 4 : 7) void k_jobs(
    cx<R>* __restrict__ psi, cx<R>* __restrict__ lam, const char* __restrict__ image, const WireJobs J,
    double* __restrict__ partial) {
  extern __shared__ __align__(16) char lds_raw[];
  const uint32_t tid = threadIdx.x;
  int j = 0;
  while (j + 1 < J.n && blockIdx.x >= J.j[j + 1].blk0) ++j;
  const WireJob& job = J.j[j];
  const uint32_t blk = blockIdx.x - job.blk0;
  const PassHdr* H = reinterpret_cast<const PassHdr*>(image + job.hdr);
  const uint64_t tb = insert_zeros((uint64_t)blk, H->sorted, 12);
  const WireOp<R>* ops = reinterpret_cast<const WireOp<R>*>(image + job.ops);
  const uint32_t* aux = reinterpret_cast<const uint32_t*>(image + job.aux);
  cx<R> a[NV][16];
  uint32_t seen = 0;
  touch_pass<R, 8>(H, ops, aux, tid, seen);
  if constexpr (NV == 1) {
    wire_load<R, 4, 8, 1>(a, {psi + job.off}, H, tb, tid, 0);
  } else {
    wire_load<R, 4, 8, 2>(a, {psi + job.off, lam + job.off}, H, tb, tid, 0);
  }
  asm volatile("" ::"v"(seen));
  double* row = wire_ops<R, 4, 8, NV, IMAGES, HEAVY>(a, lds_raw, H, ops, reinterpret_cast<const cx<R>*>(image + job.coef), aux,
                                             tid, blk);
  if (H->sync_store || NV == 2) __syncthreads();
  if constexpr (NV == 1) {
    wire_store<R, 4, 8, 1>(a, {psi + job.off}, H, tb, tid, blk, 0);
  } else {
    wire_store<R, 4, 8, 2>(a, {job.keep & 1 ? psi + job.off : nullptr, job.keep & 2 ? lam + job.off : nullptr}, H, tb,
                           tid, blk, 0);
    const int ng = H->ngrad;
    double* out = partial + job.part + (uint64_t)blk * ng;
    for (int i = (int)tid; i < ng; i += 256) out[i] = (row[4 * i] + row[4 * i + 1]) + (row[4 * i + 2] + row[4 * i + 3]);
  }
}

}  // namespace qs
