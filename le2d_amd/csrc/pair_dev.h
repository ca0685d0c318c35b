// pair_dev.h -- two full steps per pass over HBM.
//
// Tile.  A workgroup of two wavefronts owns a window of 64*C consecutive
// columns, lane t of each wavefront the C columns C*t .. C*t+C-1 of it, and
// writes the 64*C-8 columns between the 4 halo columns on each side, for the
// rows [j0, j1) of a segment.  Raw rows j0-4 .. j1+5 are read once (clamped at
// the grid edges, as the reference clamps), so a pass moves 5 reads + 5
// writes per node for two steps.
//
// Stages.  Stage 1 (wavefront 0) x-sweeps each raw row and y-marches to time
// n+1, rows j0-2 .. j1+1; stage 2 (wavefront 1) x-sweeps each of them and y-marches
// to time n+2.  Each time-(n+1) row passes through an LDS ring of two slots,
// one workgroup barrier per row: wavefront 0 writes row k into slot k & 1 and
// arrives at barrier k; wavefront 1 passes barrier k before it reads row k and
// arrives at barrier k+1 only after the read, so a slot is rewritten only
// after its row was read.  Both wavefronts pass exactly j1 - j0 + 4 barriers.
// With one stage each, a wavefront holds half the march state, so more of
// them are resident; each x-sweep's LDS exchange stays within its wavefront
// (wavefront-scope ordering).
//
// Columns per lane.  What bounds the pass is VALU issue (FP64 also power, which
// follows the instruction count), and C columns per lane issue fewer
// instructions per node: the window re-computes 8 halo columns of 64*C, one
// lane exchange and one lane shift serve C columns, the limiter's slopes are
// shared between a lane's faces, a row takes one 8- or 16-byte access per field,
// and the columns' independent work hides latency at two wavefronts per
// SIMD.  FP64 8192^2, all fields random: C = 2 issues 580e6 VALU instructions
// per pass against 641e6 with C = 1 and has a seventh of the LDS bank
// conflicts, 1.57-1.59 ms against 1.67-1.70; FP32 C = 4 0.58-0.59 ms
// against 0.61-0.64 for the one-column forms.  C = 2 (FP64) and C = 4 (FP32) fill the
// 256 registers of two wavefronts per SIMD; more columns spill.  Grids that do
// not fill the device with wide windows take fewer columns per lane (2048^2 FP32
// 45 us at C = 1, 58 at C = 4).
//
// The operands and operations of every update are those of two single steps,
// so the result is bit-identical.
#pragma once

#include "sweep_dev.h"

namespace le2d {

// ---------------------------------------------------------------------------
// C neighbouring columns of one row.

template <typename T, int C>
struct alignas(C * sizeof(T)) Vec {
  T v[C];
};
template <typename T, int C>
struct Nodes {
  Node<T> n[C];
};
template <typename T, int C>
struct Ws {  // invariants of C nodes, or C faces
  W4<T> w[C];
};

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// One access of 4, 8 or 16 bytes (buffer accesses need 4-byte alignment only).
template <typename T, int C>
__device__ __forceinline__ Vec<T, C> buf_ldv(__amdgpu_buffer_rsrc_t r, unsigned voff, int soff) {
  using V = Vec<T, C>;
  static_assert(sizeof(V) == 4 || sizeof(V) == 8 || sizeof(V) == 16, "one access");
  if constexpr (sizeof(V) == 16)
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
  else if constexpr (sizeof(V) == 8)
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0));
  else
    return __builtin_bit_cast(V, __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0));
}

template <typename T, int C>
__device__ __forceinline__ void buf_stv(__amdgpu_buffer_rsrc_t r, unsigned voff, int soff,
                                        const Vec<T, C> &v) {
  if constexpr (sizeof(v) == 16)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), r, voff, soff, 0);
  else if constexpr (sizeof(v) == 8)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, voff, soff, 0);
  else
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, voff, soff, 0);
}

template <typename T, int C>
__device__ __forceinline__ Nodes<T, C> unpack(const Vec<T, C> (&f)[5]) {
  Nodes<T, C> u;
#pragma unroll
  for (int k = 0; k < C; ++k) u.n[k] = {f[0].v[k], f[1].v[k], f[2].v[k], f[3].v[k], f[4].v[k]};
  return u;
}

template <typename T, int C>
__device__ __forceinline__ void pack(const Nodes<T, C> &u, Vec<T, C> (&f)[5]) {
#pragma unroll
  for (int k = 0; k < C; ++k) {
    f[0].v[k] = u.n[k].vx;
    f[1].v[k] = u.n[k].vy;
    f[2].v[k] = u.n[k].sxx;
    f[3].v[k] = u.n[k].sxy;
    f[4].v[k] = u.n[k].syy;
  }
}

template <typename T, int C>
__device__ __forceinline__ Nodes<T, C> load_nodes(const T *__restrict__ row, long plane,
                                                  unsigned boff) {
  const __amdgpu_buffer_rsrc_t r = row_rsrc(row, plane);
  const int ps = (int)(plane * (long)sizeof(T));
  Vec<T, C> f[5];
#pragma unroll
  for (int q = 0; q < 5; ++q) f[q] = buf_ldv<T, C>(r, boff, q * ps);
  return unpack(f);
}

// Columns past nx-1 of a lane's access fall in the row's padding to 256 bytes,
// which no output depends on and which may hold anything (see_row).
template <typename T, int C>
__device__ __forceinline__ void store_nodes(T *__restrict__ row, long plane, unsigned boff,
                                            const Nodes<T, C> &u) {
  const __amdgpu_buffer_rsrc_t r = row_rsrc(row, plane);
  const int ps = (int)(plane * (long)sizeof(T));
  Vec<T, C> f[5];
  pack(u, f);
#pragma unroll
  for (int q = 0; q < 5; ++q) buf_stv<T, C>(r, boff, q * ps, f[q]);
}

template <typename T, int C>
__device__ __forceinline__ Nodes<T, C> pick_nodes(bool c, const Nodes<T, C> &a,
                                                  const Nodes<T, C> &b) {
  Nodes<T, C> u;
#pragma unroll
  for (int k = 0; k < C; ++k) u.n[k] = pick_node(c, a.n[k], b.n[k]);
  return u;
}

template <typename T>
__device__ __forceinline__ W4<T> pick_w(bool c, const W4<T> &a, const W4<T> &b) {
  return {c ? a.a : b.a, c ? a.b : b.b, c ? a.c : b.c, c ? a.d : b.d};
}

// Shows the row's values to `dv`.  With several columns per lane the lanes from
// the grid's last column on also hold columns of the padding, which is never
// initialised: they take the last column's values, so that what the memory held
// before cannot send a tile to the IEEE divisions (FP64 2047 x 2048 with NaN in the
// padding 167 us a pass, 121 with zeros or this).
template <typename T, int C, typename Edge, typename Div>
__device__ __forceinline__ void see_row(Nodes<T, C> &u, const Edge &d, int t, Div &dv) {
  if constexpr (C > 1 && Div::kSees) {
    if (d.any) {  // wavefront-uniform
#pragma unroll
      for (int k = 1; k < C; ++k) u.n[k] = pick_node(t >= d.th && k > d.e, u.n[k - 1], u.n[k]);
    }
  }
#pragma unroll
  for (int k = 0; k < C; ++k) {
    const T f[5] = {u.n[k].vx, u.n[k].vy, u.n[k].sxx, u.n[k].sxy, u.n[k].syy};
    dv.row(f);
  }
}

template <typename T, int C>
__device__ __forceinline__ Ws<T, C> inv_y(const Nodes<T, C> &u, const SweepCoef<T> &c) {
  Ws<T, C> w;
#pragma unroll
  for (int k = 0; k < C; ++k) w.w[k] = inv_y(u.n[k], c);
  return w;
}

template <typename T, int C, typename Div>
__device__ __forceinline__ Ws<T, C> faces(const Ws<T, C> &wm, const Ws<T, C> &w0,
                                          const Ws<T, C> &w1, const Ws<T, C> &w2,
                                          const SweepCoef<T> &c, Div &dv) {
  Ws<T, C> f;
#pragma unroll
  for (int k = 0; k < C; ++k) f.w[k] = faces(wm.w[k], w0.w[k], w1.w[k], w2.w[k], c, dv);
  return f;
}

template <typename T, int C>
__device__ __forceinline__ void apply_y(Nodes<T, C> &u, const Ws<T, C> &w, const Ws<T, C> &fl,
                                        const Ws<T, C> &fr, const SweepCoef<T> &c) {
#pragma unroll
  for (int k = 0; k < C; ++k)
    apply(u.n[k].vy, u.n[k].vx, u.n[k].syy, u.n[k].sxx, u.n[k].sxy, w.w[k], fl.w[k], fr.w[k], c);
}

// The components of a row's invariants that the next face's upwind side reads.
template <typename T, int C>
__device__ __forceinline__ void keep_ac(Ws<T, C> &to, const Ws<T, C> &w) {
#pragma unroll
  for (int k = 0; k < C; ++k) {
    to.w[k].a = w.w[k].a;
    to.w[k].c = w.w[k].c;
  }
}

// ---------------------------------------------------------------------------
// Lane shifts.

// Lane t+1's value on lane t (lane 63 receives 0): a wavefront shift of the
// data-parallel primitives (DPP wave_shl:1), no LDS round trip.
__device__ __forceinline__ int lane_next(int v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x130, 0xf, 0xf, true);
}
__device__ __forceinline__ float lane_next(float v) {
  return __builtin_bit_cast(float, lane_next(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double lane_next(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)lane_next((int)(unsigned)b);
  const unsigned hi = (unsigned)lane_next((int)(unsigned)(b >> 32));
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
template <typename T>
__device__ __forceinline__ W4<T> lane_next(const W4<T> &v) {
  W4<T> r;
  r.a = lane_next(v.a);
  r.b = lane_next(v.b);
  r.c = lane_next(v.c);
  r.d = lane_next(v.d);
  return r;
}
// Lane t-1's value on lane t (lane 0 receives 0): DPP wave_shr:1.
__device__ __forceinline__ float lane_prev(float v) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x138, 0xf, 0xf, true));
}

// FP32 one-wavefront x-sweep faces with shared slopes.  The limiter's
// numerator (u0 - um) + eps of a face is, operand for operand, the
// denominator du + eps of the face upwind of it: the face on the left for
// the invariants moving to +x (a, c), the face on the right for those moving
// to -x (b, d).  Lane t forms its face's du and du + eps once from its
// neighbour's invariants and its own (du = w1 - w0 for a, c and w0 - w1 for b, d), and takes the
// numerators from lanes t-1 and t+1 by lane shifts: two subtractions per
// face and invariant instead of four, the same operations on the same
// operands.  Lanes 0 and 63 receive shifted zeros; no output reads their
// faces.
__device__ __forceinline__ W4<float> faces_shared(const W4<float> &w0, const W4<float> &w1,
                                                  const SweepCoef<float> &c) {
  const float eps = 1e-6f;
  const float da = w1.a - w0.a, db = w0.b - w1.b, dc = w1.c - w0.c, dd = w0.d - w1.d;
  const float sa = da + eps, sb = db + eps, sc = dc + eps, sd = dd + eps;
  W4<float> f;
  f.a = __builtin_fmaf(limiter(slope_ratio(lane_prev(sa), sa)) * c.hk1, da, w0.a);
  f.b = __builtin_fmaf(limiter(slope_ratio(lane_next(sb), sb)) * c.hk1, db, w1.b);
  f.c = __builtin_fmaf(limiter(slope_ratio(lane_prev(sc), sc)) * c.hk2, dc, w0.c);
  f.d = __builtin_fmaf(limiter(slope_ratio(lane_next(sd), sd)) * c.hk2, dd, w1.d);
  return f;
}

// ---------------------------------------------------------------------------
// x-sweep of a window row.  The grid's edges clamp as the reference does: the
// columns past an edge take the edge column's invariants, whatever the lanes
// outside the grid hold.  Meaningful on the columns 2 .. 64*C-3.

template <typename T>
struct alignas(2 * sizeof(T)) P2 {
  T p, q;
};

// One column per lane: the right-moving (a, c) and left-moving (b, d) pairs of
// every lane, two 16-byte columns in FP64 (W4 rows of 32 bytes read by component
// had 7 times the bank conflicts).
template <typename T>
struct X1Lds {
  P2<T> ac[64], bd[64];
};
// C columns per lane: what a lane needs of its neighbours, the invariants of
// the last column of the lane on its left, the right-moving pair of the
// column before that, and the left-moving pair of the first column of the
// lane on its right.  Entry t+1 is lane t's.
template <typename T>
struct XnLds {
  W4<T> last[66];
  P2<T> prev[66], first[66];
};
template <typename T, int C>
struct XLdsOf {
  using type = XnLds<T>;
};
template <typename T>
struct XLdsOf<T, 1> {
  using type = X1Lds<T>;
};

// Where the window meets the grid's left and right edge.  One column per lane:
// the lanes t-2, t-1, t and t+1 clamped into those that hold grid columns.
// C columns: the lane whose first column is grid column 0 (-1: none), the
// lane that holds grid column nx-1 (64 or more: none) and that column's place
// in it.  any: the window holds an edge (wavefront-uniform).
struct X1Edge {
  bool any;
  int i2, i1, i0, ir;
};
struct XnEdge {
  bool any;
  int tl, th, e;
};

template <int C, int HALO = 4>  // HALO: halo columns, 4 for two steps, 2 for one
__device__ __forceinline__ auto x_edge(int x0, int nx, int t) {
  const int last = nx - 1 + HALO - x0;  // window column of grid column nx-1
  if constexpr (C == 1) {
    const int lo = x0 == 0 ? HALO : 0, hi = min(63, last);
    return X1Edge{x0 == 0 || last < 63, min(max(t - 2, lo), hi), min(max(t - 1, lo), hi),
                  min(max(t, lo), hi), min(max(t + 1, lo), hi)};
  } else {
    return XnEdge{x0 == 0 || last < 64 * C, x0 == 0 ? HALO / C : -1, last / C, last % C};
  }
}

template <typename T, typename Div>
__device__ __forceinline__ void x_sweep(Nodes<T, 1> &un, X1Lds<T> &x, int t, const X1Edge &d,
                                        const SweepCoef<T> &c, Div &dv) {
  Node<T> &u = un.n[0];
  const W4<T> w = invariants(u.vx, u.sxx, u.vy, u.sxy, c);
  x.ac[t] = {w.a, w.c};
  x.bd[t] = {w.b, w.d};
  window_sync<64>();
  const P2<T> lac = x.ac[d.i1], lbd = x.bd[d.i1];
  const W4<T> wl = {lac.p, lbd.p, lac.q, lbd.q};
  W4<T> we = w, f;
  if (d.any) {  // lanes outside the grid stand for the edge column
    const P2<T> oac = x.ac[d.i0], obd = x.bd[d.i0];
    we = {oac.p, obd.p, oac.q, obd.q};
  }
  if constexpr (sizeof(T) == 4) {
    window_sync<64>();  // the next x-sweep rewrites x only after every lane read it
    f = faces_shared(wl, we, c);
  } else {
    const P2<T> l2 = x.ac[d.i2], r = x.bd[d.ir];
    window_sync<64>();
    f = faces4(l2.p, r.p, l2.q, r.q, wl, we, c, dv);
  }
  // the face on the lane's right is the right neighbour's
  apply(u.vx, u.vy, u.sxx, u.syy, u.sxy, w, f, lane_next(f), c);
}

template <typename T, int C, typename Div>
__device__ __forceinline__ void x_sweep(Nodes<T, C> &u, XnLds<T> &x, int t, const XnEdge &d,
                                        const SweepCoef<T> &c, Div &dv) {
  static_assert(C == 2 || C == 4, "the 4 halo columns are whole lanes");
  Ws<T, C> w;
#pragma unroll
  for (int k = 0; k < C; ++k)
    w.w[k] = invariants(u.n[k].vx, u.n[k].sxx, u.n[k].vy, u.n[k].sxy, c);
  x.last[t + 1] = w.w[C - 1];
  x.prev[t + 1] = {w.w[C - 2].a, w.w[C - 2].c};
  x.first[t + 1] = {w.w[0].b, w.w[0].d};
  if (d.any) {
    window_sync<64>();  // the neighbours' own entries are written first
#pragma unroll
    for (int k = 1; k < C; ++k) w.w[k] = pick_w(t == d.th && k > d.e, w.w[k - 1], w.w[k]);
    if (t == d.th) {
      x.last[t + 1] = w.w[C - 1];
      x.first[t + 2] = {w.w[C - 1].b, w.w[C - 1].d};
    }
    if (t == d.tl) {
      x.last[t] = w.w[0];
      x.prev[t] = {w.w[0].a, w.w[0].c};
    }
  }
  window_sync<64>();
  const W4<T> l = x.last[t];
  const P2<T> l2 = x.prev[t], r = x.first[t + 2];
  window_sync<64>();  // the next x-sweep rewrites x only after every lane read it
  if (d.any) {  // the lane past the last column forms that column's right face
    w.w[0] = pick_w(t == d.th + 1, l, w.w[0]);
    w.w[1] = pick_w(t == d.th + 1, l, w.w[1]);
  }
  Ws<T, C> f;
#pragma unroll
  for (int k = 0; k < C; ++k) {  // the face on the left of column k
    const T am = k > 1 ? w.w[k - 2].a : k ? l.a : l2.p, cm = k > 1 ? w.w[k - 2].c : k ? l.c : l2.q;
    const T bm = k + 1 < C ? w.w[k + 1].b : r.p, dm = k + 1 < C ? w.w[k + 1].d : r.q;
    f.w[k] = faces4(am, bm, cm, dm, k ? w.w[k - 1] : l, w.w[k], c, dv);
  }
  const W4<T> fe = lane_next(f.w[0]);  // the face right of the lane's last column
#pragma unroll
  for (int k = 0; k < C; ++k)
    apply(u.n[k].vx, u.n[k].vy, u.n[k].sxx, u.n[k].syy, u.n[k].sxy, w.w[k], f.w[k],
          k + 1 < C ? f.w[k + 1] : fe, c);
}

// ---------------------------------------------------------------------------
// The march.

__device__ __forceinline__ void split_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// Wavefronts per SIMD that the registers of C columns per lane allow without
// spilling (FP64 150 at C = 1 and 256 at C = 2; FP32 127 and 224 at C = 2 and 4).
template <typename T, int C>
constexpr int pair_waves() { return C == 1 ? 3 : C == 2 && sizeof(T) == 4 ? 4 : 2; }

template <typename T, int C>
struct PairLds {
  typename XLdsOf<T, C>::type x[2];  // one per stage
  Vec<T, C> ring[2][5][64];
  int go;  // the values of stage 1's first rows are in the divisions' range
};

// FP32, which has the registers, keeps each slot's y-invariants (WA.., VA..)
// instead of re-forming them.
template <typename T>
constexpr bool kHoldInv = sizeof(T) == 4;

// One step on `rows` rows from row q on, each handed to `out` with its count; one
// row only if a value of the first five raw rows is out of the divisions' range,
// which `start` is told.
template <typename T, int EDGE, int C, typename XLds, typename XEdge, typename Div,
          typename Start, typename Out>
__device__ __forceinline__ void march_rows(const T *__restrict__ src, int ny, long pitch, long plane,
                                           unsigned boff, int q, int rows, int t, const XEdge &ed,
                                           const SweepCoef<T> &cx, const SweepCoef<T> &cy,
                                           XLds &lds, Div &dv, Start start, Out out) {
  // Slots A/B/D hold the x-swept rows q, q+1, q+2, F the face q-1 | q, wb the
  // invariants of row q-1, N the raw row in flight.  Unrolled three times, so
  // no slot is copied.
  constexpr bool HOLD = kHoldInv<T>;
#define ROW(p) load_nodes<T, C>(src + (long)ypos<EDGE>((p), ny) * pitch, plane, boff)
  Nodes<T, C> A = {}, B = {}, D = {}, N;
  Ws<T, C> F, wb = {}, WA, WB, WD;
  int k = 0;
  {
    // x-sweep rows q-2 .. q+2, a loop so that no more rows are held than
    // the march holds (unrolled, the compiler keeps all five until the end
    // and spills)
    Ws<T, C> w2 = {};
    N = ROW(q - 2);
#pragma unroll 1
    for (int p = q - 1; p <= q + 3; ++p) {
      Nodes<T, C> u = N;
      N = ROW(p);
      see_row(u, ed, t, dv);
      x_sweep(u, lds, t, ed, cx, dv);
      w2 = wb;
      wb = inv_y(A, cy);
      A = B;
      B = D;
      D = u;
    }
    if constexpr (Div::kSees) {
      const bool go = __all(dv.in_range());
      start(go);
      if (!go) rows = 1;
    }
    WA = inv_y(A, cy);
    WB = inv_y(B, cy);
    if constexpr (HOLD) WD = inv_y(D, cy);
    F = faces(w2, wb, WA, WB, cy, dv);
  }
#define ADVANCE(P0, P1, P2, W0, W1, W2)                                              \
  {                                                                                  \
    const Ws<T, C> w0 = HOLD ? W0 : inv_y(P0, cy);                                   \
    const Ws<T, C> fo =                                                              \
        faces(wb, w0, HOLD ? W1 : inv_y(P1, cy), HOLD ? W2 : inv_y(P2, cy), cy, dv); \
    apply_y(P0, w0, F, fo, cy);                                                      \
    F = fo;                                                                          \
    keep_ac(wb, w0);                                                                 \
    out(k, P0);                                                                      \
    if (++k >= rows) break;                                                          \
    P0 = N;                                                                          \
    N = ROW(q + 4);                                                                  \
    see_row(P0, ed, t, dv);                                                          \
    x_sweep(P0, lds, t, ed, cx, dv);                                                 \
    if constexpr (HOLD) W0 = inv_y(P0, cy);                                          \
    ++q;                                                                             \
  }
  for (;;) {
    ADVANCE(A, B, D, WA, WB, WD)
    ADVANCE(B, D, A, WB, WD, WA)
    ADVANCE(D, A, B, WD, WA, WB)
  }
#undef ADVANCE
#undef ROW
}

template <typename T, int C, typename Div>
__device__ __forceinline__ void pair_march(const T *__restrict__ src, T *__restrict__ dst, int nx,
                                           int ny, long pitch, long plane, int strip, int j0, int j1,
                                           const SweepCoef<T> &cx, const SweepCoef<T> &cy,
                                           PairLds<T, C> &lds, Div &dv) {
  constexpr bool HOLD = kHoldInv<T>;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int t = (int)(threadIdx.x & 63);
  const int x0 = strip * (64 * C - 8);
  const int x = x0 - 4 + C * t;  // the lane's first column
  const auto ed = x_edge<C>(x0, nx, t);
  const int rows = j1 - j0 + 4;  // stage-1 rows j0-2 .. j1+1
#define XS(u) x_sweep(u, lds.x[wave], t, ed, cx, dv)
  if (wave == 0) {
    const unsigned boff = (unsigned)min(max(x, 0), (nx - 1) / C * C) * (unsigned)sizeof(T);
    auto start = [&](bool go) { lds.go = go; };  // read behind the first barrier
    auto put = [&](int k, const Nodes<T, C> &u) {
      Vec<T, C> out[5];
      pack(u, out);
#pragma unroll
      for (int f = 0; f < 5; ++f) lds.ring[k & 1][f][t] = out[f];
      split_sync();
    };
    march_rows<T, EDGE_CLAMP, C>(src, ny, pitch, plane, boff, j0 - 2, rows, t, ed, cx, cy,
                                 lds.x[0], dv, start, put);
  } else {
    // Stage 2: slots A/B/D hold the x-swept time-(n+1) rows r, r+1, r+2, G the
    // face r-1 | r, vb the invariants of row r-1.  Positions above row 0 or
    // below row ny-1 take that edge row's value, the reference's row clamp of
    // the time-(n+1) state.
    const unsigned woff = (unsigned)max(x, 0) * (unsigned)sizeof(T);
    const bool writer = t >= 4 / C && t < 64 - 4 / C && x < nx;
    Nodes<T, C> A, B, D, M1, M2;
    Ws<T, C> G, vb, VA, VB, VD;
    int k = 0;
    auto take = [&](Nodes<T, C> &u) {
      Vec<T, C> in[5];
#pragma unroll
      for (int f = 0; f < 5; ++f) in[f] = lds.ring[k & 1][f][t];
      ++k;
      u = unpack(in);
      XS(u);
    };
    auto get = [&](Nodes<T, C> &u) {
      split_sync();
      take(u);
    };
    split_sync();
    if constexpr (Div::kSees)
      if (!__builtin_amdgcn_readfirstlane(lds.go)) return;  // stage 1 ends here too
    take(M2);  // row j0-2
    get(M1);  // row j0-1
    get(A);   // row j0
    get(B);   // row j0+1
    B = pick_nodes(j0 + 1 >= ny, A, B);
    M1 = pick_nodes(j0 - 1 < 0, A, M1);
    M2 = pick_nodes(j0 - 2 < 0, M1, M2);
    vb = inv_y(M1, cy);
    VA = inv_y(A, cy);
    VB = inv_y(B, cy);
    G = faces(inv_y(M2, cy), vb, VA, VB, cy, dv);
    int r = j0;
#define STAGE2(Q0, Q1, Q2, V0, V1, V2)                                                   \
  {                                                                                      \
    get(Q2);                                                                             \
    Q2 = pick_nodes(r + 2 >= ny, Q1, Q2);                                                \
    if constexpr (HOLD) V2 = inv_y(Q2, cy);                                              \
    const Ws<T, C> v0 = HOLD ? V0 : inv_y(Q0, cy);                                       \
    const Ws<T, C> go =                                                                  \
        faces(vb, v0, HOLD ? V1 : inv_y(Q1, cy), HOLD ? V2 : inv_y(Q2, cy), cy, dv);         \
    apply_y(Q0, v0, G, go, cy);                                                          \
    G = go;                                                                              \
    if (writer) store_nodes<T, C>(dst + (long)r * pitch, plane, woff, Q0);               \
    if (++r >= j1) break;                                                                \
    keep_ac(vb, v0);                                                                     \
  }
    for (;;) {
      STAGE2(A, B, D, VA, VB, VD)
      STAGE2(B, D, A, VB, VD, VA)
      STAGE2(D, A, B, VD, VA, VB)
    }
#undef STAGE2
  }
#undef XS
}

// The tile, in FP64 with DivBounded's quotients, and once more with IEEE
// divisions if it does not meet their conditions (the output of the first
// march is overwritten; the input is another buffer).  FP64 8192^2 random field 1.55 ms a
// pass against 1.65, disk 1.24 against 1.34; 2048^2 111 us against 122.
//
// The first march ends after its first rows if a value of them is out of range,
// so a field that is so everywhere costs little more than the IEEE march alone
// (2048^2 with NaN everywhere 118 us a pass against 214 in two full marches); a
// tile whose first such value, or whose only zero divisor, is further down
// costs both.
template <typename T, int C>
__device__ __forceinline__ void pair_tile(const T *__restrict__ src, T *__restrict__ dst, int nx,
                                          int ny, long pitch, long plane, int strip, int j0, int j1,
                                          const SweepCoef<T> &cx, const SweepCoef<T> &cy,
                                          PairLds<T, C> &lds) {
#if LE2D_LIMITER != 2  // CIR forms no ratio
  if constexpr (sizeof(T) == 8) {
    if (coef_bounded(cx) && coef_bounded(cy)) {
      DivBounded dv;
      pair_march<T, C>(src, dst, nx, ny, pitch, plane, strip, j0, j1, cx, cy, lds, dv);
      if (__syncthreads_and(dv.ok())) return;
    }
  }
#endif
  DivIeee<T> dv;
  pair_march<T, C>(src, dst, nx, ny, pitch, plane, strip, j0, j1, cx, cy, lds, dv);
}

// One step on the tile of strip `strip` (60 of 64 columns written) and rows
// [j0, j1), by one wavefront.  Two columns per lane, which leave half as many wavefronts,
// are slower on the grids that take this march (1500 x 1001 30.6 us against 26.0).
template <typename T, int EDGE, typename Div>
__device__ __forceinline__ void step_march(const T *__restrict__ src, T *__restrict__ dst, int nx,
                                           int ny, long pitch, long plane, int strip, int j0, int j1,
                                           const SweepCoef<T> &cx, const SweepCoef<T> &cy,
                                           X1Lds<T> &lds, Div &dv) {
  const int t = (int)threadIdx.x;
  const int x0 = strip * 60, x = x0 - 2 + t;
  const unsigned boff = (unsigned)min(max(x, 0), nx - 1) * (unsigned)sizeof(T);
  const unsigned woff = (unsigned)max(x, 0) * (unsigned)sizeof(T);
  const bool writer = t >= 2 && t < 62 && x < nx;
  auto put = [&](int k, const Nodes<T, 1> &u) {
    if (writer) store_nodes<T, 1>(dst + (long)(j0 + k) * pitch, plane, woff, u);
  };
  march_rows<T, EDGE, 1>(src, ny, pitch, plane, boff, j0, j1 - j0, t, x_edge<1, 2>(x0, nx, t), cx,
                         cy, lds, dv, [](bool) {}, put);
}

template <typename T, int EDGE>
__device__ __forceinline__ void step_tile(const T *__restrict__ src, T *__restrict__ dst, int nx,
                                          int ny, long pitch, long plane, int strip, int j0, int j1,
                                          const SweepCoef<T> &cx, const SweepCoef<T> &cy,
                                          X1Lds<T> &lds) {
#if LE2D_LIMITER != 2
  if constexpr (sizeof(T) == 8) {  // as pair_tile
    if (coef_bounded(cx) && coef_bounded(cy)) {
      DivBounded dv;
      step_march<T, EDGE>(src, dst, nx, ny, pitch, plane, strip, j0, j1, cx, cy, lds, dv);
      if (__syncthreads_and(dv.ok())) return;
    }
  }
#endif
  DivIeee<T> dv;
  step_march<T, EDGE>(src, dst, nx, ny, pitch, plane, strip, j0, j1, cx, cy, lds, dv);
}

}  // namespace le2d
