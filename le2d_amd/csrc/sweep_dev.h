// sweep_dev.h -- device numerics of the sweeps, shared by every kernel.
//
// Numerics (reference simple/le_core.c:29-69, :192-257): per sweep each node's
// state u = (vx, vy, sxx, sxy, syy) is projected on four Riemann invariants
// with speeds +c1, -c1, +c2, -c2; each invariant is advanced by the
// superbee-limited second-order TVD scheme with clamped edges; the increment
// is projected back.  All invariants are formed from pre-sweep values.
//
// Face formulation.  The reference evaluates, per node and invariant, the two
// face fluxes f(i+1/2) and f(i-1/2) (tvd2, :48-69).  The flux a node computes
// for its right face is, operand for operand, the one its right neighbour
// computes for its left face, so each face is evaluated once here and shared:
// one division, one limiter and one flux per face and invariant instead of
// two.  The node update then applies u - k*(f_out - f_in) - u in the
// reference's order, which keeps FP64 results bit-identical when the
// compiler does not contract multiply-adds (-ffp-contract=off).
//
// Layout: field q (vx, vy, sxx, sxy, syy) of node (i, j) at q*plane + j*pitch + i;
// the fields of a row lie side by side (plane = padded row, pitch = 5 rows).
#pragma once

#include "engine.h"

namespace le2d {

// ---------------------------------------------------------------------------
// Scalar pieces.

// Superbee limiter with the reference's ternary min/max (simple/le_core.c:31-38):
// max(0, max(min(1, 2r), min(2, r))).
template <typename T>
__device__ __forceinline__ T superbee(T r) {
  // max(0, max(min(1, 2r), min(2, r))) = max(c, min(r, 2)) = med3(r, c, 2)
  // with c = clamp(2r, 0, 1): for r < 0, c = 0 and min(r, 2) = r < 0; for
  // r >= 0, c = min(2r, 1).  The clamp is the add's output modifier.
  if constexpr (sizeof(T) == 4) {
    // FP32 tier (held to an error bound against FP64, not to bits): two
    // instructions.  A NaN r (0/0: both slopes exactly -eps) gives 0 here,
    // the first-order flux, where the reference's formula gives 2.
    const float c = __builtin_fminf(__builtin_fmaxf(r + r, 0.0f), 1.0f);
#if LE2D_FP32_NAN2
    return __builtin_fmaxf(c, __builtin_fminf(r, 2.0f));  // NaN: max(0, 2) = 2
#else
    return __builtin_amdgcn_fmed3f(r, c, 2.0f);
#endif
  } else {
    // FP64: max(c, min(r, 2)) is the reference's value bit for bit for every
    // r (NaN and infinities included: the clamp sends NaN to 0, min(NaN, 2)
    // is 2) except r = -0, where this gives +0 and the reference's ternaries
    // keep -0.  No result bit depends on that sign.  The limiter value
    // reaches the node only through the face flux u + (phi*hk)*du, where a
    // zero phi changes at most the sign of a zero flux, and through the
    // increment (u - k*(f_out - f_in)) - u, which is the same for fluxes that
    // differ only in the sign of a zero: f_out - f_in is then the same nonzero
    // value or a zero, and (u - (+-0)) - u is +0 for every finite u (NaN for
    // infinite u either way).
    const double c = __builtin_fmin(__builtin_fmax(r + r, 0.0), 1.0);
    return __builtin_fmax(c, __builtin_fmin(r, 2.0));
  }
}

// The build's flux limiter (LE2D_LIMITER).  minmod is the reference's
// ternary form max(0, min(1, r)) (simple/le_core.c:36), so NaN gives 1 and
// -0 stays -0 in both types; CIR is 0 (:37).  Both are options beside the
// default superbee.
template <typename T>
__device__ __forceinline__ T limiter(T r) {
#if LE2D_LIMITER == 1
  const T m = T(1) > r ? r : T(1);
  return T(0) > m ? T(0) : m;
#elif LE2D_LIMITER == 2
  (void)r;
  return T(0);
#else
  return superbee(r);
#endif
}

// Limited flux through the face between upwind node u0 and downwind node u1;
// um is the node upwind of u0 (simple/le_core.c:50-66 with eps = 1e-6).
// The reference forms ((phi / 2) * (1 - k)) * (u1 - u0); phi / 2 is exact for
// every value phi takes (superbee: 0, 1, 2, r in (1,2), 2r in (0,1); minmod:
// 0, 1, r in [0,1); CIR: 0; r is a normal number: its numerator is 0 or at
// least about 2^-73 in magnitude), so (phi / 2) * (1 - k) rounds the same
// real number as phi * hk with the exact constant hk = (1 - k) / 2, one
// multiply fewer per face.
// Slope ratio.  FP64: IEEE division, as the reference.  FP32 tier: the
// hardware reciprocal (about 1 ulp) times the numerator; that tier is held to
// an error bound against FP64, not to bit parity, and the correctly rounded
// FP32 division sequence costs several times more issue slots.
// Build options of the FP32 tier's accuracy/cost trade-off (defaults in
// brackets): LE2D_FP32_RATIO [0] the reciprocal times the numerator, 1 the
// same refined by one Newton step on the quotient, 2 IEEE division;
// LE2D_FP32_NAN2 [0] a NaN ratio gives the limiter 0, 1 gives 2 as the
// reference's formula does.
#ifndef LE2D_FP32_RATIO
#define LE2D_FP32_RATIO 0
#endif
#ifndef LE2D_FP32_NAN2
#define LE2D_FP32_NAN2 0
#endif
__device__ __forceinline__ double slope_ratio(double n, double d) { return n / d; }
__device__ __forceinline__ float slope_ratio(float n, float d) {
#if LE2D_FP32_RATIO == 2
  return n / d;
#elif LE2D_FP32_RATIO == 1
  const float rc = __builtin_amdgcn_rcpf(d);
  const float q = n * rc;
  return __builtin_fmaf(__builtin_fmaf(-d, q, n), rc, q);
#else
  return n * __builtin_amdgcn_rcpf(d);
#endif
}

// How a march divides.  DivIeee: slope_ratio whatever the operands.
template <typename T>
struct DivIeee {
  static constexpr bool kSees = false;  // whether see and row do anything
  __device__ __forceinline__ T ratio(T n, T d) { return slope_ratio(n, d); }
  __device__ __forceinline__ void see(T, T) {}
  __device__ __forceinline__ void row(const T (&)[5]) {}
  __device__ __forceinline__ bool in_range() const { return true; }
};

// FP64 quotients of a tile whose values stay below 2^764: the compiler's IEEE
// sequence (a reciprocal, two Newton steps on it, the product and one
// residual step, Markstein's method) without its operand scaling and its
// special-case fix-up, 8 instructions instead of 11 and no use of VCC, which
// ties the divisions of a face set in a row.
//
// The scaling is an identity where no intermediate leaves the normal range.
// A slope operand is a difference plus eps = 1e-6, so it is 0 or at least
// 2^-73 in magnitude (a difference that cancels against eps does so exactly);
// with operands below 2^764 every intermediate lies between 2^-838 and 2^838.
// The fix-up matters for a zero divisor and for non-finite operands only.
// So the march keeps the largest magnitude of the rows it loads and the
// smallest divisor (row, see: a maximum or minimum of three high words as
// FP32 bit patterns, whose order is the magnitudes'), and a tile that met a
// value of 2^300 or more, a non-finite one or a zero divisor is marched again
// with DivIeee (ok).  With constants up to 2^60 (coef_bounded) one sweep grows values
// by less than 2^134, so those of the four sweeps of a pass stay below 2^702 and
// their invariants' differences below 2^764.
//
// Left out, the scaling changes no bit: the operations are those of n / d as
// compiled.  Checked on the GPU where rounding is closest, on every quotient
// within 5 units of the product's last place of a rounding boundary for the
// 2^39 divisors below a power of two (1.4e12 quotients), and on 2e10 random
// ones: all equal to n / d; the test of the quotients repeats that for 2^30 divisors
// of each kind.
struct DivBounded {
  static constexpr bool kSees = true;
  float big = 0.0f, small = 1.0f;
  static __device__ __forceinline__ float hi(double x) {
    return __builtin_bit_cast(float, (int)(__builtin_bit_cast(unsigned long long, x) >> 32));
  }
  __device__ __forceinline__ double ratio(double n, double d) {
    const double y0 = __builtin_amdgcn_rcp(d);
    const double e0 = __builtin_fma(-d, y0, 1.0);
    const double y1 = __builtin_fma(y0, e0, y0);
    const double e1 = __builtin_fma(-d, y1, 1.0);
    const double y = __builtin_fma(y1, e1, y1);
    const double q = n * y;
    return __builtin_fma(__builtin_fma(-d, q, n), y, q);
  }
  __device__ __forceinline__ void see(double a, double b) {
    small = __builtin_fminf(__builtin_fminf(__builtin_fabsf(hi(a)), __builtin_fabsf(hi(b))), small);
  }
  // maximum (not fmax): a high word of 2^1017 or more is an FP32 NaN pattern
  // and must win
  static __device__ __forceinline__ float mx(float a, float b, float c) {
    return __builtin_elementwise_maximum(
        __builtin_elementwise_maximum(__builtin_fabsf(a), __builtin_fabsf(b)), c);
  }
  __device__ __forceinline__ void row(const double (&u)[5]) {
    big = mx(hi(u[0]), hi(u[1]), big);
    big = mx(hi(u[2]), hi(u[3]), big);
    big = __builtin_elementwise_maximum(__builtin_fabsf(hi(u[4])), big);
  }
  // high words of 2^300 and 2^-80
  __device__ __forceinline__ bool in_range() const {
    return big < __builtin_bit_cast(float, (1023 + 300) << 20);
  }
  __device__ __forceinline__ bool ok() const {
    return in_range() && small > __builtin_bit_cast(float, (1023 - 80) << 20);
  }
};

template <typename T, typename Div>
__device__ __forceinline__ T face_flux(T um, T u0, T u1, T hk, Div &dv) {
  const T eps = T(1e-6);
  const T du = u1 - u0;
  const T r = dv.ratio((u0 - um) + eps, du + eps);
  if constexpr (sizeof(T) == 4)
    return __builtin_fmaf(limiter(r) * hk, du, u0);  // FP32 tier: fused
  else
    return u0 + (limiter(r) * hk) * du;
}

// Increment of one invariant from its outflow and inflow face fluxes
// (simple/le_core.c:68 and :253-256): (u - k*(out - in)) - u.
template <typename T>
__device__ __forceinline__ T face_delta(T u, T k, T out, T in) {
  return (u - k * (out - in)) - u;
}

template <typename T>
struct W4 {
  T a, b, c, d;  // speeds +c1, -c1, +c2, -c2
};

// Invariants for a sweep along the axis whose velocity is vn and whose normal
// stress is sn (simple/le_core.c:192-218).
template <typename T>
__device__ __forceinline__ W4<T> invariants(T vn, T sn, T vt, T sxy, const SweepCoef<T> &c) {
  W4<T> w;
  if constexpr (sizeof(T) == 4) {
    // FP32 tier: one fused multiply-add per invariant (the negations on the
    // uniform factors, so no lane value needs negating)
    const T ni1 = -c.irhoc1, ni2 = -c.irhoc2;
    w.a = __builtin_fmaf(sn, ni1, vn);
    w.b = __builtin_fmaf(sn, c.irhoc1, vn);
    w.c = __builtin_fmaf(sxy, ni2, vt);
    w.d = __builtin_fmaf(sxy, c.irhoc2, vt);
  } else {
    const T n = sn * c.irhoc1;
    const T m = sxy * c.irhoc2;
    w.a = vn - n;
    w.b = vn + n;
    w.c = vt - m;
    w.d = vt + m;
  }
  return w;
}

// Faces of the four invariants between positions p and p+1: the upwind and
// the two adjoining values of each (+c1 and +c2: upwind is the left side; -c1
// and -c2: the right side).
template <typename T, typename Div>
__device__ __forceinline__ W4<T> faces4(T am, T bm, T cm, T dm, const W4<T> &w0, const W4<T> &w1,
                                        const SweepCoef<T> &c, Div &dv) {
  const T eps = T(1e-6);
  W4<T> f;
  f.a = face_flux(am, w0.a, w1.a, c.hk1, dv);
  f.b = face_flux(bm, w1.b, w0.b, c.hk1, dv);
  f.c = face_flux(cm, w0.c, w1.c, c.hk2, dv);
  f.d = face_flux(dm, w1.d, w0.d, c.hk2, dv);
  dv.see((w1.a - w0.a) + eps, (w0.b - w1.b) + eps);  // the divisors
  dv.see((w1.c - w0.c) + eps, (w0.d - w1.d) + eps);
  return f;
}

// The same, given the invariants at p-1, p, p+1, p+2.
template <typename T, typename Div>
__device__ __forceinline__ W4<T> faces(const W4<T> &wm, const W4<T> &w0, const W4<T> &w1,
                                       const W4<T> &w2, const SweepCoef<T> &c, Div &dv) {
  return faces4(wm.a, w2.b, wm.c, w2.d, w0, w1, c, dv);
}
template <typename T>
__device__ __forceinline__ W4<T> faces(const W4<T> &wm, const W4<T> &w0, const W4<T> &w1,
                                       const W4<T> &w2, const SweepCoef<T> &c) {
  DivIeee<T> dv;
  return faces(wm, w0, w1, w2, c, dv);
}

// Whether a sweep's constants are small enough for DivBounded: every
// magnitude at most 2^60 (wavefront-uniform).
__device__ __forceinline__ bool coef_bounded(const SweepCoef<double> &c) {
  int m = 0;
  for (double x : {c.k1, c.k2, c.hk1, c.hk2, c.irhoc1, c.irhoc2, c.rhoc1, c.rhoc2, c.rhoc3})
    m = max(m, (int)(__builtin_bit_cast(unsigned long long, x) >> 52) & 0x7ff);
  int k = 0;
  for (double x : {c.k1, c.k2, c.hk1, c.hk2})
    k = max(k, (int)(__builtin_bit_cast(unsigned long long, x) >> 52) & 0x7ff);
  return m < 1023 + 60 && k < 1023 + 5;
}

// Back-transform of the increments (simple/le_core.c:221-249).  vn/sn are
// the along-axis velocity and normal stress, vt/so the tangential velocity
// and the other normal stress.
template <typename T>
__device__ __forceinline__ void apply(T &vn, T &vt, T &sn, T &so, T &sxy, const W4<T> &w,
                                      const W4<T> &fl, const W4<T> &fr,
                                      const SweepCoef<T> &c) {
  if constexpr (sizeof(T) == 4) {
    // FP32 tier: the increment (u - k*(out - in)) - u is k*(in - out); the
    // back-transform's factor 1/2 and the stress factors are folded into
    // uniform constants (hoisted), each field takes one fused multiply-add
    const T h1 = T(0.5) * c.k1, h2 = T(0.5) * c.k2;
    const T da = fl.a - fr.a, db = fr.b - fl.b, dc = fl.c - fr.c, dd = fr.d - fl.d;
    const T t1 = db - da, t2 = dd - dc;
    vn = __builtin_fmaf(h1, da + db, vn);
    vt = __builtin_fmaf(h2, dc + dd, vt);
    sn = __builtin_fmaf(h1 * c.rhoc1, t1, sn);
    so = __builtin_fmaf(h1 * c.rhoc3, t1, so);
    sxy = __builtin_fmaf(h2 * c.rhoc2, t2, sxy);
  } else {
    const T e1 = T(0.5) * face_delta(w.a, c.k1, fr.a, fl.a);
    const T e2 = T(0.5) * face_delta(w.b, c.k1, fl.b, fr.b);
    const T e3 = T(0.5) * face_delta(w.c, c.k2, fr.c, fl.c);
    const T e4 = T(0.5) * face_delta(w.d, c.k2, fl.d, fr.d);
    vn = vn + (e1 + e2);
    vt = vt + (e3 + e4);
    sn = sn + (e2 - e1) * c.rhoc1;
    so = so + (e2 - e1) * c.rhoc3;
    sxy = sxy + c.rhoc2 * (e4 - e3);
  }
}

// ---------------------------------------------------------------------------
// Rows and nodes.

// Row of window position p along y: clamp (le_step) or the ring edge
// (le_step_soa / le_step_y_cf).
template <int EDGE>
__device__ __forceinline__ int ypos(int p, int ny) {
  if (p < 0) return 0;
  if (p < ny) return p;
  return EDGE == EDGE_CLAMP ? ny - 1 : max(p - 5, 0);
}

template <typename T>
struct Node {
  T vx, vy, sxx, sxy, syy;
};

// c ? a : b field by field.  A conditional on two Node lvalues is copied
// through a selected address, which keeps an array holding either operand
// in scratch memory; selecting the values keeps it in registers.
template <typename T>
__device__ __forceinline__ Node<T> pick_node(bool c, const Node<T> &a, const Node<T> &b) {
  Node<T> n;
  n.vx = c ? a.vx : b.vx;
  n.vy = c ? a.vy : b.vy;
  n.sxx = c ? a.sxx : b.sxx;
  n.sxy = c ? a.sxy : b.sxy;
  n.syy = c ? a.syy : b.syy;
  return n;
}

template <typename T>
__device__ __forceinline__ Node<T> load_node(const T *__restrict__ p, long plane) {
  Node<T> n;
  n.vx = p[0];
  n.vy = p[plane];
  n.sxx = p[2 * plane];
  n.sxy = p[3 * plane];
  n.syy = p[4 * plane];
  return n;
}

// Row loads and stores go through a buffer resource whose base is the row
// (wavefront-uniform, built in SGPRs): the lane's byte offset within the field
// row is the VGPR offset and the field's plane offset the SGPR offset, so a
// load or store costs no per-lane address arithmetic (a global access with a
// 64-bit per-lane address costs one 64-bit add each).  The resource covers
// the row's five padded field rows (row_fits keeps that under 2^31 bytes);
// every offset used is inside it.  Word 3 is the gfx9 raw-buffer format
// (32-bit data, no swizzle).
template <typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_rsrc(const T *row, long plane) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(row), (short)0,
                                           (int)(5 * plane * (long)sizeof(T)), 0x00020000);
}

template <typename T>
__device__ __forceinline__ T buf_ld(__amdgpu_buffer_rsrc_t r, unsigned voff, int soff) {
  if constexpr (sizeof(T) == 8)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

template <typename T>
__device__ __forceinline__ void buf_st(__amdgpu_buffer_rsrc_t r, unsigned voff, int soff, T v) {
  if constexpr (sizeof(T) == 8)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, voff, soff, 0);
  else
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, voff, soff, 0);
}

template <typename T>
__device__ __forceinline__ Node<T> load_row_node(const T *__restrict__ row, long plane,
                                                 unsigned boff) {
  const __amdgpu_buffer_rsrc_t r = row_rsrc(row, plane);
  const int ps = (int)(plane * (long)sizeof(T));
  Node<T> n;
  n.vx = buf_ld<T>(r, boff, 0);
  n.vy = buf_ld<T>(r, boff, ps);
  n.sxx = buf_ld<T>(r, boff, 2 * ps);
  n.sxy = buf_ld<T>(r, boff, 3 * ps);
  n.syy = buf_ld<T>(r, boff, 4 * ps);
  return n;
}

template <typename T>
__device__ __forceinline__ void store_row_node(T *__restrict__ row, long plane, unsigned boff,
                                               const Node<T> &u) {
  const __amdgpu_buffer_rsrc_t r = row_rsrc(row, plane);
  const int ps = (int)(plane * (long)sizeof(T));
  buf_st<T>(r, boff, 0, u.vx);
  buf_st<T>(r, boff, ps, u.vy);
  buf_st<T>(r, boff, 2 * ps, u.sxx);
  buf_st<T>(r, boff, 3 * ps, u.sxy);
  buf_st<T>(r, boff, 4 * ps, u.syy);
}

template <typename T>
__device__ __forceinline__ W4<T> inv_y(const Node<T> &n, const SweepCoef<T> &c) {
  return invariants(n.vy, n.syy, n.vx, n.sxy, c);
}

// ---------------------------------------------------------------------------
// Fused step: the x-sweep and the y-sweep of one time step in one pass over
// HBM (5 reads + 5 writes per node-update instead of twice that).
//
// A workgroup of FB lanes owns a window of FB consecutive columns starting two
// columns left of its strip of FB-4 output columns, and a segment of `seg`
// rows.  Lane t reads column x0-2+t (clamped into the grid), so the two halo
// columns on each side of the strip come from ordinary lanes: no extra loads,
// no divergent work.  Walking positions p = j0-2 .. j1+1 down the strip, each
// position's row (ypos-mapped) is read once and x-swept through LDS (every
// face of the strip in one pass over lanes 2..FB-2); each lane's post-x node
// then feeds the register y-march of k_sweep_y.  Only rows [j0, j1) of the
// FB-4 inner columns are written.  The y-march consumes x-swept values of the
// rows just outside the segment, recomputed here from the unswept input,
// which is exactly what the y-sweep of the two-kernel sequence reads.
//
// Workgroups are renumbered so that the tiles one XCD receives (the hardware
// deals workgroups to the 8 XCDs round-robin) are consecutive strips of the
// same segments: strips that share halo columns share an L2.
__device__ __forceinline__ int xcd_tile(int L, int N) {
  const int per = N >> 3, rem = N & 7, xcd = L & 7, k = L >> 3;
  return xcd < rem ? xcd * (per + 1) + k : rem * (per + 1) + (xcd - rem) * per + k;
}

template <typename T>
__device__ __forceinline__ void store_node(T *p, long plane, const Node<T> &u) {
  p[0] = u.vx;
  p[plane] = u.vy;
  p[2 * plane] = u.sxx;
  p[3 * plane] = u.sxy;
  p[4 * plane] = u.syy;
}

// Synchronisation of a window's LDS exchange: a workgroup barrier, or for a
// one-wavefront window (FB = 64) a wavefront-scope release/acquire fence
// pair around a wave barrier.  A wavefront's lanes run in lockstep and its
// LDS operations complete in order, so no wait and no s_barrier is needed;
// the workgroup-scope fence of __syncthreads would wait for every LDS write
// to complete and keep the compiler from overlapping independent exchanges.
template <int FB>
__device__ __forceinline__ void window_sync() {
  if constexpr (FB <= 64) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  } else {
    __syncthreads();
  }
}

// x-sweep of one window row; returns the lane's post-x node (meaningful on
// lanes 2..FB-3).  sw[t] holds lane t's invariants, sf[t] the face between
// lanes t-1 and t.
template <typename T, int FB>
__device__ __forceinline__ Node<T> window_xsweep(Node<T> u, W4<T> *sw, W4<T> *sf, int t,
                                                 const SweepCoef<T> &c) {
  const W4<T> w = invariants(u.vx, u.sxx, u.vy, u.sxy, c);
  sw[t] = w;
  window_sync<FB>();
  if (t >= 2 && t <= FB - 2) sf[t] = faces(sw[t - 2], sw[t - 1], sw[t], sw[t + 1], c);
  window_sync<FB>();
  if (t >= 2 && t <= FB - 3) apply(u.vx, u.vy, u.sxx, u.syy, u.sxy, w, sf[t], sf[t + 1], c);
  return u;
}

// One tile of the fused step: the window of strip `strip` (lane t reads
// column strip*(FB-4)-2+t, clamped; lanes 2..FB-3 write) over output rows
// [j0, j1), marched downwards (DIR = +1, j increasing) or upwards (DIR = -1).
// Callers alternate the direction between neighbouring segments of a strip,
// so the two segments that read the halo rows around a shared boundary do so
// at about the same time (both start there, or both end there) and the
// second read hits L2.  Each face is the same operands and operations in
// either direction, so the result does not depend on DIR.  Used by the
// single-grid, material and batched kernels alike.
template <typename T, int EDGE, int FB, int DIR>
__device__ __forceinline__ void march_tile(const T *__restrict__ src, T *__restrict__ dst, int nx,
                                           int ny, long pitch, long plane, int strip, int j0,
                                           int j1, const SweepCoef<T> &cx,
                                           const SweepCoef<T> &cy, W4<T> *sw, W4<T> *sf) {
  const int t = threadIdx.x;
  const int x = strip * (FB - 4) - 2 + t;
  const unsigned boff = (unsigned)min(max(x, 0), nx - 1) * (unsigned)sizeof(T);
  const unsigned woff = (unsigned)max(x, 0) * (unsigned)sizeof(T);
  const bool writer = t >= 2 && t <= FB - 3 && x < nx;
#define ROW(p) load_row_node(src + (long)ypos<EDGE>((p), ny) * pitch, plane, boff)
#define XS(n) window_xsweep<T, FB>((n), sw, sf, t, cx)
  // Slots P0/P1/P2 hold the x-swept nodes of positions j, j+DIR, j+2*DIR
  // (their y-invariants are re-formed when needed, 6 operations each, rather
  // than held), FI is the face on the side already passed and NC the raw row
  // of position j+3*DIR.  Row j is written, then position j+3*DIR is x-swept
  // into P0 while NN receives the raw row of position j+4*DIR.  Unrolled six
  // times (slot period 3, face and prefetch period 2) so no register is
  // copied between steps.  wb keeps the invariants of position j-DIR (the
  // components its faces still read).
  Node<T> A, B, C, N0, N1;
  W4<T> F0, F1, wb;
  int j;
  if constexpr (DIR > 0) {
    const W4<T> w2 = inv_y(XS(ROW(j0 - 2)), cy);
    wb = inv_y(XS(ROW(j0 - 1)), cy);
    A = XS(ROW(j0));
    B = XS(ROW(j0 + 1));
    C = XS(ROW(j0 + 2));
    N0 = ROW(j0 + 3);
    F0 = faces(w2, wb, inv_y(A, cy), inv_y(B, cy), cy);  // face j0-1 | j0
    j = j0;
  } else {
    const W4<T> w2 = inv_y(XS(ROW(j1 + 1)), cy);
    wb = inv_y(XS(ROW(j1)), cy);
    A = XS(ROW(j1 - 1));
    B = XS(ROW(j1 - 2));
    C = XS(ROW(j1 - 3));
    N0 = ROW(j1 - 4);
    F0 = faces(inv_y(B, cy), inv_y(A, cy), wb, w2, cy);  // face j1-1 | j1
    j = j1 - 1;
  }
#define STEP(P0, P1, P2, FI, FO, NC, NN)                                     \
  {                                                                           \
    NN = ROW(j + 4 * DIR);                                                    \
    const W4<T> w0 = inv_y(P0, cy);                                           \
    if constexpr (DIR > 0) {                                                  \
      FO = faces(wb, w0, inv_y(P1, cy), inv_y(P2, cy), cy); /* j | j+1 */     \
      apply(P0.vy, P0.vx, P0.syy, P0.sxx, P0.sxy, w0, FI, FO, cy);            \
    } else {                                                                  \
      FO = faces(inv_y(P2, cy), inv_y(P1, cy), w0, wb, cy); /* j-1 | j */     \
      apply(P0.vy, P0.vx, P0.syy, P0.sxx, P0.sxy, w0, FO, FI, cy);            \
    }                                                                         \
    if (writer) store_row_node(dst + (long)j * pitch, plane, woff, P0);      \
    j += DIR;                                                                 \
    if (DIR > 0 ? j >= j1 : j < j0) break;                                    \
    if constexpr (DIR > 0) {                                                  \
      wb.a = w0.a;                                                            \
      wb.c = w0.c;                                                            \
    } else {                                                                  \
      wb.b = w0.b;                                                            \
      wb.d = w0.d;                                                            \
    }                                                                         \
    P0 = XS(NC);                                                              \
  }
  for (;;) {
    STEP(A, B, C, F0, F1, N0, N1)
    STEP(B, C, A, F1, F0, N1, N0)
    STEP(C, A, B, F0, F1, N0, N1)
    STEP(A, B, C, F1, F0, N1, N0)
    STEP(B, C, A, F0, F1, N0, N1)
    STEP(C, A, B, F1, F0, N1, N0)
  }
#undef STEP
#undef XS
#undef ROW
}

// Direction by segment index: even segments march down, odd ones up.
template <typename T, int EDGE, int FB>
__device__ __forceinline__ void march_tile_alt(const T *__restrict__ src, T *__restrict__ dst,
                                               int nx, int ny, long pitch, long plane, int strip,
                                               int j0, int j1, int segi,
                                               const SweepCoef<T> &cx, const SweepCoef<T> &cy,
                                               W4<T> *sw, W4<T> *sf) {
  if (segi & 1)
    march_tile<T, EDGE, FB, -1>(src, dst, nx, ny, pitch, plane, strip, j0, j1, cx, cy, sw, sf);
  else
    march_tile<T, EDGE, FB, 1>(src, dst, nx, ny, pitch, plane, strip, j0, j1, cx, cy, sw, sf);
}

// ---------------------------------------------------------------------------
// Heterogeneous media: node-local march for tiles that straddle a material
// interface.
//
// The reference has one material per task (simple/le_core.h:168-186) and no
// interface rule.  Here every node is updated entirely in its own material:
// the five stencil nodes of a sweep are projected on that node's
// eigenvectors, advected with that node's Courant numbers and projected back
// with that node's constants.  Both faces of a node are therefore evaluated
// by the node itself (no sharing across an interface); with one material the
// operands and operations are exactly those of march_tile, so the bits agree.
// `ids` holds one material index per node (pitched rows of `idp` bytes);
// cxt/cyt are the per-material constants of the x- and y-sweep.
template <typename T, int EDGE, int FB>
__device__ __forceinline__ void march_tile_mixed(const T *__restrict__ src, T *__restrict__ dst,
                                                 const unsigned char *__restrict__ ids, long idp,
                                                 int nx, int ny, long pitch, long plane, int strip,
                                                 int j0, int j1,
                                                 const SweepCoef<T> *__restrict__ cxt,
                                                 const SweepCoef<T> *__restrict__ cyt,
                                                 Node<T> *sn) {
  const int t = threadIdx.x;
  const int x = strip * (FB - 4) - 2 + t;
  const int xc = min(max(x, 0), nx - 1);
  const unsigned boff = (unsigned)xc * (unsigned)sizeof(T);
  const unsigned woff = (unsigned)max(x, 0) * (unsigned)sizeof(T);
  const bool inner = t >= 2 && t <= FB - 3;
  const bool writer = inner && x < nx;

  // x-sweep of the row of position p; returns this lane's post-x node.
  auto xrow = [&](int p) -> Node<T> {
    const int row = ypos<EDGE>(p, ny);
    Node<T> u = load_row_node(src + (long)row * pitch, plane, boff);
    const int m = ids[(long)row * idp + xc];
    sn[t] = u;
    window_sync<FB>();
    if (inner) {
      const SweepCoef<T> c = cxt[m];
      W4<T> w[5];
#pragma unroll
      for (int q = 0; q < 5; ++q) {
        const Node<T> &v = sn[t - 2 + q];
        w[q] = invariants(v.vx, v.sxx, v.vy, v.sxy, c);
      }
      const W4<T> fl = faces(w[0], w[1], w[2], w[3], c);
      const W4<T> fr = faces(w[1], w[2], w[3], w[4], c);
      apply(u.vx, u.vy, u.sxx, u.syy, u.sxy, w[2], fl, fr, c);
    }
    window_sync<FB>();
    return u;
  };

  // y-march over positions; P[q] holds the post-x node of position j-2+q
  Node<T> P[5];
#pragma unroll
  for (int q = 0; q < 5; ++q) P[q] = xrow(j0 - 2 + q);
  for (int j = j0;;) {
    const SweepCoef<T> c = cyt[ids[(long)j * idp + xc]];
    W4<T> w[5];
#pragma unroll
    for (int q = 0; q < 5; ++q) w[q] = inv_y(P[q], c);
    const W4<T> fl = faces(w[0], w[1], w[2], w[3], c);
    const W4<T> fr = faces(w[1], w[2], w[3], w[4], c);
    Node<T> u = P[2];
    apply(u.vy, u.vx, u.syy, u.sxx, u.sxy, w[2], fl, fr, c);
    if (writer) store_row_node(dst + (long)j * pitch, plane, woff, u);
    if (++j >= j1) break;
#pragma unroll
    for (int q = 0; q < 4; ++q) P[q] = P[q + 1];
    P[4] = xrow(j + 2);
  }
}

// Two full steps of the node-local scheme over a tile that straddles a
// material interface: the strip geometry, edge rules and stage order of
// pair_tile (pair_dev.h), with every node's update in its own material (as
// march_tile_mixed).  Rows are held in shift registers: few tiles take this
// path.  sn has FB entries.
template <typename T, int FB>
__device__ __forceinline__ void march_pair_mixed(const T *__restrict__ src, T *__restrict__ dst,
                                                 const unsigned char *__restrict__ ids, long idp,
                                                 int nx, int ny, long pitch, long plane, int strip,
                                                 int j0, int j1,
                                                 const SweepCoef<T> *__restrict__ cxt,
                                                 const SweepCoef<T> *__restrict__ cyt,
                                                 Node<T> *sn) {
  const int t = threadIdx.x;
  const int x0 = strip * (FB - 8);
  const int x = x0 - 4 + t;
  const int xc = min(max(x, 0), nx - 1);
  const unsigned boff = (unsigned)xc * (unsigned)sizeof(T);
  const unsigned woff = (unsigned)max(x, 0) * (unsigned)sizeof(T);
  const bool writer = t >= 4 && t <= FB - 5 && x < nx;
  const int tlo = max(0, 4 - x0), thi = min(FB - 1, nx + 3 - x0);
  int nb[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) nb[k] = min(max(t - 2 + k, tlo), thi);
  const bool inner = t >= 2 && t <= FB - 3;

  // node-local x-sweep of row `row` (u: this lane's node of it)
  auto xsweep = [&](Node<T> u, int row) -> Node<T> {
    const int m = ids[(long)row * idp + xc];
    sn[t] = u;
    window_sync<FB>();
    if (inner) {
      const SweepCoef<T> c = cxt[m];
      W4<T> w[5];
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        const Node<T> &v = sn[nb[k]];
        w[k] = invariants(v.vx, v.sxx, v.vy, v.sxy, c);
      }
      const W4<T> fl = faces(w[0], w[1], w[2], w[3], c);
      const W4<T> fr = faces(w[1], w[2], w[3], w[4], c);
      apply(u.vx, u.vy, u.sxx, u.syy, u.sxy, w[2], fl, fr, c);
    }
    window_sync<FB>();
    return u;
  };
  // node-local y-update of row j from the x-swept rows j-2 .. j+2
  auto yupdate = [&](const Node<T> *P, int j) -> Node<T> {
    const SweepCoef<T> c = cyt[ids[(long)j * idp + xc]];
    W4<T> w[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) w[k] = inv_y(P[k], c);
    const W4<T> fl = faces(w[0], w[1], w[2], w[3], c);
    const W4<T> fr = faces(w[1], w[2], w[3], w[4], c);
    Node<T> u = P[2];
    apply(u.vy, u.vx, u.syy, u.sxx, u.sxy, w[2], fl, fr, c);
    return u;
  };
  auto raw = [&](int p) -> Node<T> {
    return load_row_node(src + (long)ypos<EDGE_CLAMP>(p, ny) * pitch, plane, boff);
  };

  // stage 1: P[k] = x-swept time-n row at position q-2+k (clamped rows)
  Node<T> P[5], Q[5];
  int q = j0 - 2;
#pragma unroll
  for (int k = 0; k < 5; ++k) P[k] = xsweep(raw(q - 2 + k), ypos<EDGE_CLAMP>(q - 2 + k, ny));
  // time-(n+1) row q x-swept for stage 2 (meaningful for 0 <= q < ny)
  auto next = [&]() -> Node<T> {
    const int row = min(max(q, 0), ny - 1);
    const Node<T> y1 = yupdate(P, row);
    const Node<T> x2 = xsweep(y1, row);
#pragma unroll
    for (int k = 0; k < 4; ++k) P[k] = P[k + 1];
    P[4] = xsweep(raw(q + 3), ypos<EDGE_CLAMP>(q + 3, ny));
    ++q;
    return x2;
  };
  // stage 2: Q[k] = x-swept time-(n+1) row at position r-2+k, clamped
#pragma unroll
  for (int k = 0; k < 4; ++k) Q[k] = next();  // positions j0-2 .. j0+1
  Q[3] = pick_node(j0 + 1 >= ny, Q[2], Q[3]);
  Q[1] = pick_node(j0 - 1 < 0, Q[2], Q[1]);
  Q[0] = pick_node(j0 - 2 < 0, Q[1], Q[0]);
  for (int r = j0; r < j1; ++r) {
    const Node<T> xn = next();  // position r+2
    Q[4] = pick_node(r + 2 >= ny, Q[3], xn);
    const Node<T> u = yupdate(Q, r);
    if (writer) store_row_node(dst + (long)r * pitch, plane, woff, u);
#pragma unroll
    for (int k = 0; k < 4; ++k) Q[k] = Q[k + 1];
  }
}

// The same two steps for a block of kMixRows output rows and up to 56 columns,
// every row of it and its halo on a wavefront of its own: lane t of wavefront
// v holds node (x0-4+t, j0-4+v).  What bounds a mixed tile is latency (each
// row of the march waits for its ids, then for its nodes' constants, then for
// two exchanges), and a pass waits for its mixed tiles: here the rows' waits
// overlap, four sweeps one after another instead of (rows + 8) x 4.  It computes
// 16 rows for 8, so the march stays where mixed tiles fill the device.  The
// operations are march_pair_mixed's.  sn holds 16 x 64 nodes.
constexpr int kMixRows = 8;

template <typename T>
__device__ __forceinline__ void block_pair_mixed(const T *__restrict__ src, T *__restrict__ dst,
                                                 const unsigned char *__restrict__ ids, long idp,
                                                 int nx, int ny, long pitch, long plane, int x0,
                                                 int x1, int j0, int j1,
                                                 const SweepCoef<T> *__restrict__ cxt,
                                                 const SweepCoef<T> *__restrict__ cyt,
                                                 Node<T> *sn) {
  constexpr int ROWS = kMixRows + 8;
  const int v = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int t = (int)(threadIdx.x & 63);
  const int x = x0 - 4 + t, xc = min(max(x, 0), nx - 1);
  const int j = j0 - 4 + v, jc = min(max(j, 0), ny - 1);
  const int tlo = max(0, 4 - x0), thi = min(63, nx + 3 - x0);
  Node<T> u = load_row_node(src + (long)jc * pitch, plane, (unsigned)xc * (unsigned)sizeof(T));
  const int m = ids[(long)jc * idp + xc];
#pragma unroll 1
  for (int s = 0; s < 2; ++s) {
    {
      const SweepCoef<T> c = cxt[m];
      sn[v * 64 + t] = u;
      window_sync<64>();
      W4<T> w[5];
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        const Node<T> &n = sn[v * 64 + min(max(t - 2 + k, tlo), thi)];
        w[k] = invariants(n.vx, n.sxx, n.vy, n.sxy, c);
      }
      window_sync<64>();
      const W4<T> fl = faces(w[0], w[1], w[2], w[3], c);
      const W4<T> fr = faces(w[1], w[2], w[3], w[4], c);
      apply(u.vx, u.vy, u.sxx, u.syy, u.sxy, w[2], fl, fr, c);
    }
    sn[v * 64 + t] = u;
    __syncthreads();
    {
      const SweepCoef<T> c = cyt[m];
      W4<T> w[5];
#pragma unroll
      for (int k = 0; k < 5; ++k) {
        // row j-2+k clamped to the grid, then to the block (rows whose
        // stencil leaves the block are not outputs' inputs)
        const int r = min(max(min(max(j - 2 + k, 0), ny - 1) - (j0 - 4), 0), ROWS - 1);
        w[k] = inv_y(sn[r * 64 + t], c);
      }
      if (s == 0) __syncthreads();  // the second step rewrites the rows
      const W4<T> fl = faces(w[0], w[1], w[2], w[3], c);
      const W4<T> fr = faces(w[1], w[2], w[3], w[4], c);
      apply(u.vy, u.vx, u.syy, u.sxx, u.sxy, w[2], fl, fr, c);
    }
  }
  if (v >= 4 && j < j1 && t >= 4 && t < 60 && x < x1)
    store_row_node(dst + (long)j * pitch, plane, (unsigned)max(x, 0) * (unsigned)sizeof(T), u);
}

}  // namespace le2d
