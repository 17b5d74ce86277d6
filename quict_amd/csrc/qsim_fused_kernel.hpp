// The fused tile pass on the device: op interpreter and kernel (included by
// qsim_fused.hip, which plans, uploads and launches the programs).
#pragma once
#include "qsim_common.hpp"
#include "qsim_fused_plan.hpp"

namespace qs {

// ---- device helpers ------------------------------------------------------------


// XOR of the register-slot offsets selected by the bits of r (compile-time r, uniform offsets).
template <int RB> __device__ __forceinline__ uint32_t reg_off(int r, const uint32_t (&lr)[RB]) {
  uint32_t o = 0;
#pragma unroll
  for (int b = 0; b < RB; ++b)
    if ((r >> b) & 1) o ^= lr[b];
  return o;
}

template <int TB> __device__ __forceinline__ uint32_t thr_off(const uint32_t* lt, uint32_t tid) {
  uint32_t o = 0;
#pragma unroll
  for (int b = 0; b < TB; ++b) o ^= ((tid >> b) & 1u) ? lt[b] : 0u;
  return o;
}

// Workgroup barrier for LDS traffic only: waits for this wave's LDS (and scalar)
// operations, not for outstanding global loads, so prefetched tile loads stay
// in flight across relayouts.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Non-temporal amplitude loads / stores for the streaming tile traffic.
template <typename R> __device__ __forceinline__ cx<R> ld_nt(const cx<R>* p) {
  return cx<R>{__builtin_nontemporal_load(&p->re), __builtin_nontemporal_load(&p->im)};
}
template <typename R> __device__ __forceinline__ void st_nt(cx<R>* p, cx<R> a) {
  __builtin_nontemporal_store(a.re, &p->re);
  __builtin_nontemporal_store(a.im, &p->im);
}

template <typename R> __device__ __forceinline__ void st_lds(char* lds, uint32_t off, cx<R> a) {
  st(reinterpret_cast<cx<R>*>(lds + off), a);
}
template <typename R> __device__ __forceinline__ cx<R> ld_lds(const char* lds, uint32_t off) {
  return ld(reinterpret_cast<const cx<R>*>(lds + off));
}

// Every op below writes all the registers it may touch without branching on
// data-dependent conditions: controls select coefficients (the identity where a
// control fails) or select between old and new values.  Branches per register
// or lane-predicated regions make the compiler keep a second copy of the whole
// register tile and move it back after every op.
//
// CM (control mode): 0 no controls, 1 register-bit controls only (uniform per
// register pair), 2 thread-bit controls only (per lane), 3 both.

template <typename R> __device__ __forceinline__ cx<R> sel(bool c, cx<R> x, cx<R> y) {
  return cx<R>{c ? x.re : y.re, c ? x.im : y.im};
}
template <typename R> __device__ __forceinline__ cx<R> one() { return mk<R>((R)1, (R)0); }
template <typename R> __device__ __forceinline__ cx<R> zero() { return mk<R>((R)0, (R)0); }

// Uncontrolled dense1 with a real matrix (H, Ry, their products): half the products.
template <typename R, int NR, int P>
__device__ __forceinline__ void do_dense1_real(cx<R> (&a)[NR], const cx<R>* m) {
  const R m00 = m[0].re, m01 = m[1].re, m10 = m[2].re, m11 = m[3].re;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (r & (1 << P)) continue;
    const int r1 = r | (1 << P);
    const cx<R> x0 = a[r], x1 = a[r1];
    a[r] = mk<R>(rfma(m01, x1.re, m00 * x0.re), rfma(m01, x1.im, m00 * x0.im));
    a[r1] = mk<R>(rfma(m11, x1.re, m10 * x0.re), rfma(m11, x1.im, m10 * x0.im));
  }
}

template <typename R, int NR, int P, int CM>
__device__ __forceinline__ void do_dense1(cx<R> (&a)[NR], const cx<R>* m, uint32_t creg, uint32_t cregv, bool tok) {
  cx<R> m00 = m[0], m01 = m[1], m10 = m[2], m11 = m[3];
  if constexpr (CM >= 2) {  // lanes whose thread-bit controls fail apply the identity
    m00 = sel(tok, m00, one<R>());
    m01 = sel(tok, m01, zero<R>());
    m10 = sel(tok, m10, zero<R>());
    m11 = sel(tok, m11, one<R>());
  }
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (r & (1 << P)) continue;
    cx<R> n00 = m00, n01 = m01, n10 = m10, n11 = m11;
    if constexpr (CM == 1 || CM == 3) {
      const bool on = ((uint32_t)r & creg) == cregv;
      n00 = sel(on, n00, one<R>());
      n01 = sel(on, n01, zero<R>());
      n10 = sel(on, n10, zero<R>());
      n11 = sel(on, n11, one<R>());
    }
    const int r1 = r | (1 << P);
    const cx<R> x0 = a[r], x1 = a[r1];
    a[r] = cfma(mul(n00, x0), n01, x1);
    a[r1] = cfma(mul(n10, x0), n11, x1);
  }
}

// a0' = m0 a1, a1' = m1 a0 (pure: plain exchange) where the controls hold.
// PURE: plain exchange (X, CX, ...): no phase products at all
template <typename R, int NR, int P, int CM, bool PURE>
__device__ __forceinline__ void do_perm1(cx<R> (&a)[NR], const cx<R>* m, uint32_t creg, uint32_t cregv, bool tok) {
  const cx<R> m0 = m[0], m1 = m[1];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (r & (1 << P)) continue;
    bool on = true;
    if constexpr (CM == 1 || CM == 3) on = ((uint32_t)r & creg) == cregv;
    if constexpr (CM >= 2) on = on && tok;
    const int r1 = r | (1 << P);
    const cx<R> x0 = a[r], x1 = a[r1];
    cx<R> y0 = x1, y1 = x0;
    if constexpr (!PURE) {
      y0 = mul(m0, x1);
      y1 = mul(m1, x0);
    }
    a[r] = sel(on, y0, x0);
    a[r1] = sel(on, y1, x1);
  }
}

// positions P0 (MSB) > P1 (LSB)
template <typename R, int NR, int P0, int P1, int CM>
__device__ __forceinline__ void do_dense2(cx<R> (&a)[NR], const cx<R>* m, uint32_t creg, uint32_t cregv, bool tok) {
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (r & ((1 << P0) | (1 << P1))) continue;
    bool on = true;
    if constexpr (CM == 1 || CM == 3) on = ((uint32_t)r & creg) == cregv;
    if constexpr (CM >= 2) on = on && tok;
    const int idx[4] = {r, r | (1 << P1), r | (1 << P0), r | (1 << P0) | (1 << P1)};
    cx<R> x[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = a[idx[j]];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      // one matrix row at a time keeps scalar-register pressure low
      cx<R> acc = mul(m[4 * i], x[0]);
#pragma unroll
      for (int j = 1; j < 4; ++j) acc = cfma(acc, m[4 * i + j], x[j]);
      a[idx[i]] = (CM == 0) ? acc : sel(on, acc, x[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Diagonal + anti-diagonal two-target op (positions P0 > P1): per group
// y_s = d_s x_s + o_s x_(s^3), s = (bit P0, bit P1); REAL: real payload.
template <typename R, int NR, int P0, int P1, bool REAL>
__device__ __forceinline__ void do_xx2(cx<R> (&a)[NR], const cx<R>* m) {
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (r & ((1 << P0) | (1 << P1))) continue;
    const int idx[4] = {r, r | (1 << P1), r | (1 << P0), r | (1 << P0) | (1 << P1)};
    cx<R> x[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = a[idx[j]];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      if constexpr (REAL) {
        const R d = m[s].re, o = m[4 + s].re;
        a[idx[s]] = mk<R>(rfma(o, x[s ^ 3].re, d * x[s].re), rfma(o, x[s ^ 3].im, d * x[s].im));
      } else {
        a[idx[s]] = cfma(mul(m[s], x[s]), m[4 + s], x[s ^ 3]);
      }
    }
  }
}

template <typename R, int NR, int P0, int P1, int CM, bool PURE>
__device__ __forceinline__ void do_swap2(cx<R> (&a)[NR], const cx<R>* m, uint32_t creg, uint32_t cregv, bool tok) {
  const cx<R> m0 = m[0], m1 = m[1];
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if (r & ((1 << P0) | (1 << P1))) continue;
    bool on = true;
    if constexpr (CM == 1 || CM == 3) on = ((uint32_t)r & creg) == cregv;
    if constexpr (CM >= 2) on = on && tok;
    const int i01 = r | (1 << P1), i10 = r | (1 << P0);
    const cx<R> x01 = a[i01], x10 = a[i10];
    cx<R> y01 = x10, y10 = x01;
    if constexpr (!PURE) {
      y01 = mul(m0, x10);
      y10 = mul(m1, x01);
    }
    a[i01] = sel(on, y01, x01);
    a[i10] = sel(on, y10, x10);
  }
}

// Offset (register index bits) of matrix index q for targets given by mask PM,
// highest set bit = most significant matrix bit.
template <uint32_t PM, int KB> __host__ __device__ constexpr int densek_off(int q) {
  int o = 0, k = 0;
  for (int b = 31; b >= 0; --b)
    if ((PM >> b) & 1u) {
      if ((q >> (KB - 1 - k)) & 1) o |= 1 << b;
      ++k;
    }
  return o;
}

// dense on KB register bits given by mask PM
template <typename R, int NR, int KB, uint32_t PM>
__device__ __forceinline__ void do_densek(cx<R> (&a)[NR], const cx<R>* m, uint32_t creg, uint32_t cregv, bool tok) {
  constexpr int D = 1 << KB;
  if (!tok) return;
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    if ((uint32_t)r & PM) continue;
    if (((uint32_t)r & creg) != cregv) continue;
    cx<R> x[D];
#pragma unroll
    for (int q = 0; q < D; ++q) x[q] = a[r | densek_off<PM, KB>(q)];
#pragma unroll
    for (int i = 0; i < D; ++i) {
      cx<R> acc = mul(m[i * D], x[0]);
#pragma unroll
      for (int j = 1; j < D; ++j) acc = cfma(acc, m[i * D + j], x[j]);
      a[r | densek_off<PM, KB>(i)] = acc;
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

// Diagonal gate that depends on thread bits only: one complex factor per lane
// (table entry `sel`, up to two thread-index bits t0 (MSB), t1), applied to every
// register at once.  One per-lane LDS read instead of selects between table
// entries: selects of loaded values become lane-divergent branches.
__device__ __forceinline__ uint32_t diag_sel(int ns, int t0, int t1, uint32_t tid) {
  const uint32_t b0 = (tid >> t0) & 1u, b1 = (tid >> t1) & 1u;
  return ns == 0 ? 0u : ns == 1 ? b0 : ((b0 << 1) | b1);
}

template <typename R, int NR>
__device__ __forceinline__ void do_diag_lane(cx<R> (&a)[NR], uint32_t sel, const cx<R>* T) {
  const cx<R> f = ld(T + sel);
#pragma unroll
  for (int r = 0; r < NR; ++r) a[r] = mul(f, a[r]);
}

// Diagonal op: the host resolved every register-bit dependence at plan time, so
// the payload is a table T[sel * NR + r] (sel = up to two thread-index bits, MSB
// first) and `creg` is the mask of registers whose entry is not 1 for some sel.
template <typename R, int NR>
__device__ __forceinline__ void do_diag(cx<R> (&a)[NR], uint32_t sel, const cx<R>* T) {
  // per-lane loads from row `sel` (the address is lane-dependent, so the 16..64
  // table entries never occupy scalar registers); every register is multiplied
  // (entries of untouched registers are 1): no per-register branches
  const cx<R>* Tl = T + sel * NR;
#pragma unroll
  for (int r = 0; r < NR; ++r) a[r] = mul(ld(Tl + r), a[r]);
}

// Relayout in two rounds through a half-tile LDS image (see the RELAYOUT
// payload): round k moves the registers whose bit P is k, writing them with the
// current layout (pending flips included) and reading the same registers back
// with the new layout.
template <typename R, int RB, int TB, int P>
__device__ __forceinline__ void relayout_half(cx<R> (&a)[1 << RB], char* lds, const uint32_t* __restrict__ x,
                                              bool tile_flips, uint32_t tid, uint32_t blk) {
  constexpr int NR = 1 << RB;
  uint32_t lw[RB], lq[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) lw[b] = x[1 + b];
  uint32_t w = thr_off<TB>(x + 1 + RB, tid) ^ x[1 + RB + TB];
  const uint32_t* y = x + 2 + RB + TB;
  if (tile_flips) {  // programs planned in wires: flips that depend on the tile
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
  for (int k = 0; k < 2; ++k) {
    lds_barrier();
#pragma unroll
    for (int r = 0; r < NR; ++r)
      if (((r >> P) & 1) == k) st_lds<R>(lds, w ^ reg_off<RB>(r, lw), a[r]);
    lds_barrier();
#pragma unroll
    for (int r = 0; r < NR; ++r)
      if (((r >> P) & 1) == k) a[r] = ld_lds<R>(lds, rd ^ reg_off<RB>(r, lq));
  }
}

// One op of a pass program applied to the register tile.
template <typename R, int RB, int TB, bool DK>
__device__ __forceinline__ void run_op(cx<R> (&a)[1 << RB], char* lds, const FOpW& e,
                                       const cx<R>* __restrict__ C, const cx<R>* __restrict__ G,
                                       const uint32_t* __restrict__ X, uint32_t tid) {
  constexpr int NR = 1 << RB;
  const int kind = (int)(e.w[0] & 0xff);
  const uint32_t opcoef = e.w[3];
  if (kind == F_RELAYOUT) {
    const uint32_t* x = X + opcoef;
    const uint32_t pk = x[0];
    if (pk == 0) relayout_half<R, RB, TB, 0>(a, lds, x, false, tid, 0);
    else if (pk == 1) relayout_half<R, RB, TB, 1>(a, lds, x, false, tid, 0);
    else if (pk == 2 || RB < 4) relayout_half<R, RB, TB, 2>(a, lds, x, false, tid, 0);
    else relayout_half<R, RB, TB, (RB > 3 ? 3 : 0)>(a, lds, x, false, tid, 0);
    return;
  }
  const int pure = (int)((e.w[0] >> 8) & 0xff);
  const int ntt = (int)(e.w[0] >> 24);
  const int pos0 = (int)(e.w[1] & 0xff), pos1 = (int)((e.w[1] >> 8) & 0xff);
  const int pos2 = (int)((e.w[1] >> 16) & 0xff), pos3 = (int)(e.w[1] >> 24);
  const uint32_t creg = e.w[4], cregv = e.w[5];
  const bool tok = (tid & e.w[6]) == e.w[7];
  // Payloads: diagonal tables are read per lane from the LDS copy (C); the
  // uniform payloads of dense / exchange ops come from global memory through
  // scalar loads (G), so control selects on them are scalar and they never
  // wait behind the tile's vector loads.
  const cx<R>* m = C + opcoef;
  const cx<R>* g = G + opcoef;
  // control mode: bit 0 register-bit controls, bit 1 thread-bit controls
  const int cm = (e.w[6] ? 2 : 0) | (creg ? 1 : 0);
  switch (kind) {
    case F_DENSE1:
      switch (pos0 * 4 + cm) {
#define QS_D1(P, M)                                                   \
  case P * 4 + M:                                                     \
    if constexpr (P < RB) {                                           \
      if (M == 0 && pure) do_dense1_real<R, NR, P>(a, g);              \
      else do_dense1<R, NR, P, M>(a, g, creg, cregv, tok);             \
    } else {                                                          \
      __builtin_unreachable();                                        \
    }                                                                 \
    break;
#define QS_D1P(P) QS_D1(P, 0) QS_D1(P, 1) QS_D1(P, 2) QS_D1(P, 3)
        QS_D1P(0) QS_D1P(1) QS_D1P(2) QS_D1P(3) QS_D1P(4)
#undef QS_D1P
#undef QS_D1
        default:
          __builtin_unreachable();
      }
      break;
    case F_PERM1:
      switch (pos0 * 4 + cm) {
#define QS_P1(P, M)                                                   \
  case P * 4 + M:                                                     \
    if constexpr (P < RB) {                                           \
      if (pure) do_perm1<R, NR, P, M, true>(a, g, creg, cregv, tok);   \
      else do_perm1<R, NR, P, M, false>(a, g, creg, cregv, tok);       \
    } else {                                                          \
      __builtin_unreachable();                                        \
    }                                                                 \
    break;
#define QS_P1P(P) QS_P1(P, 0) QS_P1(P, 1) QS_P1(P, 2) QS_P1(P, 3)
        QS_P1P(0) QS_P1P(1) QS_P1P(2) QS_P1P(3) QS_P1P(4)
#undef QS_P1P
#undef QS_P1
        default:
          __builtin_unreachable();
      }
      break;
    case F_DIAG: {
      const uint32_t sel = diag_sel(ntt, (int)(e.w[2] & 0xff), (int)((e.w[2] >> 8) & 0xff), tid);
      if (pure) do_diag_lane<R, NR>(a, sel, m);
      else do_diag<R, NR>(a, sel, m);
      break;
    }
    case F_DENSE2:
    case F_XX2:
    case F_SWAP2: {
      // controlled two-target ops are rare: one instance per pair, control mode 3
      // (selects) whenever any control is present; XX ops are never controlled
      const bool ctl = cm != 0;
      const int code = pos0 * 8 + pos1;
      const bool sw = kind == F_SWAP2, xx = kind == F_XX2;
      switch (code) {
#define QS_D2(A, B)                                                                  \
  case A * 8 + B:                                                                    \
    if constexpr (A < RB) {                                                          \
      if (sw) {                                                                      \
        if (ctl) {                                                                   \
          if (pure) do_swap2<R, NR, A, B, 3, true>(a, g, creg, cregv, tok);          \
          else do_swap2<R, NR, A, B, 3, false>(a, g, creg, cregv, tok);              \
        } else {                                                                     \
          if (pure) do_swap2<R, NR, A, B, 0, true>(a, g, creg, cregv, tok);          \
          else do_swap2<R, NR, A, B, 0, false>(a, g, creg, cregv, tok);              \
        }                                                                            \
      } else if (xx) {                                                               \
        if (pure) do_xx2<R, NR, A, B, true>(a, g);                                   \
        else do_xx2<R, NR, A, B, false>(a, g);                                       \
      } else {                                                                       \
        if (ctl) do_dense2<R, NR, A, B, 3>(a, g, creg, cregv, tok);                  \
        else do_dense2<R, NR, A, B, 0>(a, g, creg, cregv, tok);                      \
      }                                                                              \
    } else {                                                                         \
      __builtin_unreachable();                                                       \
    }                                                                                \
    break;
        QS_D2(1, 0) QS_D2(2, 0) QS_D2(2, 1) QS_D2(3, 0) QS_D2(3, 1) QS_D2(3, 2)
        QS_D2(4, 0) QS_D2(4, 1) QS_D2(4, 2) QS_D2(4, 3)
#undef QS_D2
        default:
          __builtin_unreachable();
      }
      break;
    }
    case F_DENSE3: {
      if constexpr (DK) {
        const uint32_t pm = (1u << pos0) | (1u << pos1) | (1u << pos2);
        switch (pm) {
#define QS_D3(M) \
case M:        \
  if constexpr ((M >> RB) == 0) do_densek<R, NR, 3, M>(a, m, creg, cregv, tok); \
  break;
          QS_D3(7u) QS_D3(11u) QS_D3(13u) QS_D3(14u) QS_D3(19u) QS_D3(21u) QS_D3(22u) QS_D3(25u) QS_D3(26u)
          QS_D3(28u)
#undef QS_D3
        }
      }
      break;
    }
    case F_DENSE4: {
      if constexpr (DK) {
        const uint32_t pm = (1u << pos0) | (1u << pos1) | (1u << pos2) | (1u << pos3);
        switch (pm) {
#define QS_D4(M) \
case M:        \
  if constexpr ((M >> RB) == 0) do_densek<R, NR, 4, M>(a, m, creg, cregv, tok); \
  break;
          QS_D4(15u) QS_D4(23u) QS_D4(27u) QS_D4(29u) QS_D4(30u)
#undef QS_D4
        }
      }
      break;
    }
    default:
      __builtin_unreachable();
  }
}

// Apply a pass's op list to the register tile `a` (load layout on entry, store
// layout on exit).  DK: include the in-register 3- and 4-target dense ops.
// U2: two ops per loop iteration.  With one op per iteration the tile's value at
// the loop head and after the op switch get different registers (an op writes
// its outputs while its inputs are still live), and the compiler copies the
// whole tile (64 registers at complex128) twice per op; with two ops per
// iteration the first op's outputs form their own register set and neither op
// needs a copy.  Every impossible switch arm is unreachable (the host checks
// each op before launch), so no arm passes the tile through unchanged.
template <typename R, int RB, int TB, bool DK, bool U2>
__device__ __forceinline__ void run_ops(cx<R> (&a)[1 << RB], char* lds, const PassHdr* __restrict__ H,
                                        const FOpW* __restrict__ P, const cx<R>* __restrict__ C,
                                        const cx<R>* __restrict__ G, const uint32_t* __restrict__ X,
                                        uint32_t tid) {
  const int nops = H->nops;
  if constexpr (U2) {
    int o = 0;
    for (; o + 1 < nops; o += 2) {
      run_op<R, RB, TB, DK>(a, lds, P[o], C, G, X, tid);
      run_op<R, RB, TB, DK>(a, lds, P[o + 1], C, G, X, tid);
    }
    if (o < nops) run_op<R, RB, TB, DK>(a, lds, P[o], C, G, X, tid);
  } else {
    for (int o = 0; o < nops; ++o) run_op<R, RB, TB, DK>(a, lds, P[o], C, G, X, tid);
  }
}

// Its amplitude a, 0 or 1 where that is known.
template <typename R>
__device__ __forceinline__ cx<R> start_load(const PassStart& S, const cx<R>* __restrict__ v, uint64_t a) {
  const uint64_t t = S.sh ? a ^ (a >> S.sh) : a;
  if (t & S.fixed) return mk<R>((R)0, (R)0);
  return S.fresh ? mk<R>((R)1, (R)0) : ld_nt(v + a);
}

// One pass over all 2^(n-K) tiles.  PF: persistent workgroups that prefetch
// the next tile into a second register set while the current one is computed
// (grid = resident workgroups); otherwise one tile per workgroup.  START: over the tiles
// of a vector with known zeros that hold anything (S), an instance of its own: with the
// choice in one kernel a full pass of the 14-qubit noisy density matrix took 2.25 ms
// instead of 1.89 ms.
template <typename R, int RB, int TB, bool DK, bool PF, bool START>
__global__ __launch_bounds__(1 << TB) void k_fused(cx<R>* __restrict__ v, const PassHdr* __restrict__ H,
                                                   const FOpW* __restrict__ ops, const cx<R>* __restrict__ coef,
                                                   const uint32_t* __restrict__ aux, uint64_t ntiles, const PassStart S) {
  static_assert(!(PF && START), "the prefetching kernel takes a vector that is there");
  constexpr int NR = 1 << RB;
  constexpr int K = RB + TB;
  extern __shared__ __align__(16) char lds_raw[];
  const uint32_t tid = threadIdx.x;
  const FOpW* P = ops + H->op0;
  const cx<R>* C;
  if constexpr (!DK) {
    // Stage the pass coefficients in LDS once per workgroup: op payload reads are
    // then LDS reads, which never wait on the global tile loads.
    cx<R>* lc = reinterpret_cast<cx<R>*>(lds_raw) + (H->uses_lds ? (1 << (K - 1)) : 0);
    const cx<R>* gc = coef + H->coef0;
    const int nc = H->ncoef;
    for (int i = (int)tid; i < nc; i += (int)blockDim.x) lc[i] = gc[i];
    __syncthreads();
    C = lc;
  } else {
    C = coef + H->coef0;
  }
  cx<R> a[NR];
  if constexpr (!PF) {
    // One tile per workgroup, straight-line: the store address is derived from
    // the header after the ops, so only the tile base stays live across them
    // (the op interpreter needs every scalar register it can get).
    uint64_t tb;
    if constexpr (START) {
      uint32_t number;
      tb = start_tile(S, blockIdx.x, H->sorted, K, number);
    } else {
      tb = insert_zeros((uint64_t)blockIdx.x, H->sorted, K);
    }
    {
      uint64_t gin = 0;
#pragma unroll
      for (int b = 0; b < TB; ++b) gin |= (uint64_t)((tid >> b) & 1u) << H->tbits[H->ts0[b]];
      uint64_t min_[RB];
#pragma unroll
      for (int b = 0; b < RB; ++b) min_[b] = 1ull << H->tbits[H->rs0[b]];
      const uint64_t base = tb | gin;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        uint64_t g = 0;
#pragma unroll
        for (int b = 0; b < RB; ++b)
          if ((r >> b) & 1) g |= min_[b];
        if constexpr (START) a[r] = start_load(S, v, base | g);
        else a[r] = ld_nt(v + (base | g));
      }
    }
    run_ops<R, RB, TB, DK, !DK>(a, lds_raw, H, P, C, coef + H->coef0, aux, tid);
    if (H->sync_store) __syncthreads();
    // store: tile base (uniform) XOR per-lane part (with pending flips) XOR register part
    uint64_t gout = 0;
#pragma unroll
    for (int b = 0; b < TB; ++b) gout |= (uint64_t)((tid >> b) & 1u) << H->tbo[H->ts1[b]];
    const uint64_t base = tb ^ gout ^ H->sflip;
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      uint64_t g = 0;
#pragma unroll
      for (int b = 0; b < RB; ++b)
        if ((r >> b) & 1) g |= 1ull << H->tbo[H->rs1[b]];
      st_nt(v + (base ^ g), a[r]);
    }
    (void)ntiles;
  } else {
    // per-lane parts of the load and store addresses, per-register parts as bit masks
    uint64_t gin = 0, gout = 0;
#pragma unroll
    for (int b = 0; b < TB; ++b) {
      const uint64_t bit = (tid >> b) & 1u;
      gin |= bit << H->tbits[H->ts0[b]];
      gout |= bit << H->tbo[H->ts1[b]];
    }
    gout ^= H->sflip;
    uint64_t min_[RB], mout[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      min_[b] = 1ull << H->tbits[H->rs0[b]];
      mout[b] = 1ull << H->tbo[H->rs1[b]];
    }
    cx<R> nx[NR];
    uint64_t t = blockIdx.x;
    if (t < ntiles) {
      const uint64_t base = insert_zeros(t, H->sorted, K) | gin;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        uint64_t g = 0;
#pragma unroll
        for (int b = 0; b < RB; ++b)
          if ((r >> b) & 1) g |= min_[b];
        a[r] = ld_nt(v + (base | g));
      }
    }
    for (; t < ntiles; t += gridDim.x) {
      const uint64_t tn = t + gridDim.x;
      if (tn < ntiles) {
        const uint64_t base = insert_zeros(tn, H->sorted, K) | gin;
#pragma unroll
        for (int r = 0; r < NR; ++r) {
          uint64_t g = 0;
#pragma unroll
          for (int b = 0; b < RB; ++b)
            if ((r >> b) & 1) g |= min_[b];
          nx[r] = ld_nt(v + (base | g));
        }
      }
      run_ops<R, RB, TB, DK, false>(a, lds_raw, H, P, C, coef + H->coef0, aux, tid);
      if (H->sync_store) __syncthreads();
      const uint64_t base = insert_zeros(t, H->sorted, K) ^ gout;
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        uint64_t g = 0;
#pragma unroll
        for (int b = 0; b < RB; ++b)
          if ((r >> b) & 1) g |= mout[b];
        st_nt(v + (base ^ g), a[r]);
      }
#pragma unroll
      for (int r = 0; r < NR; ++r) a[r] = nx[r];
    }
  }
}

}  // namespace qs
