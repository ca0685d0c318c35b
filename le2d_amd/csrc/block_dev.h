// block_dev.h -- one or two full steps per pass on blocks held in registers.
//
// Two steps, for grids that do not fill the device.  What bounds a pass of
// pair_dev.h's march on a small grid is one workgroup's march: every row waits
// for the row before it, two exchanges and a barrier, and short segments, which
// put more of the device to work, recompute more halo rows.  Here a workgroup
// of WV wavefronts holds a block of 64 columns by R*WV rows, R rows per
// wavefront and one column per lane, and takes each of the four sweeps on all
// of it at once: all loads in flight together, the x-sweeps of a wavefront's
// rows independent of each other, and two exchanges of boundary rows between
// neighbouring wavefronts per y-sweep.  It writes the 56 columns and R*WV-8
// rows between the halos (one step: 60 and R*WV-4).  One block's loads do not
// overlap its own arithmetic, so FP64, whose registers allow one block a compute
// unit (two of the lowest), takes it where every block has a unit to itself, FP32
// up to sixteen for each.
//
// us a pass, block against march: FP64 96 x 80 7.6 against 9.1, 250 x 300 8.5 against
// 12.4, 512^2 14.6 against 19.1, 724^2 21.4 against 25.3, but 900^2 (two rounds
// of blocks) 37 against 34; FP32 250 x 300 4.5 against 6.5, 512^2 7.1 against 9.3, 1031
// x 517 9.5 against 12.1, 900^2 13.4 against 16.1, and past one block a unit 1500 x
// 1001 21.4 against 23.3, 3000^2 95 against 94 to 100 (the march at its default and
// near heights is slower, at the tuner's best the same).
//
// One step.  With half the halo the blocks pay on larger grids too: in FP32,
// where two or more of them share a compute unit and one loads while another computes,
// they beat the march at every size (1500 x 1001 11.7 us against 14.4, 8192 x 4096
// 254 against 266, where the copy rate allows 214), in FP64 on small and on large
// grids (512^2 8.0 us against 10.3, 3000^2 153 against 170, copy rate 115).  Wavefronts
// come in fours, one per SIMD (3 x 6 rows 12.2 us at 512^2, 3 x 8 8.0).
//
// The operands and operations of every update are those of single steps, so the
// result is bit-identical.
#pragma once

#include "pair_dev.h"

namespace le2d {

// A wavefront's exchange: in the x-sweeps its own rows' invariants, in the
// y-sweep what its neighbours need of its rows, then the face below its last row.
template <typename T>
union BlockLds {
  X1Lds<T> x;
  struct {
    W4<T> first[64];   // first row
    P2<T> second[64];  // b and d of the second
    P2<T> last[64];    // a and c of the last
  } y;
  W4<T> face[64];
};

// Keeps a node's computation where it stands: without it the compiler delays the
// ends of a wavefront's x-sweeps until the y-sweep needs them and holds the
// operands of all of them (216 registers at R = 4 in FP64 instead of 184).
template <typename T>
__device__ __forceinline__ void pin(Node<T> &n) {
  asm volatile("" : "+v"(n.vx), "+v"(n.vy), "+v"(n.sxx), "+v"(n.sxy), "+v"(n.syy));
}

template <typename T, int STEPS, int EDGE, int R, int WV, typename Div>
__device__ __forceinline__ void block_march(const T *__restrict__ src, T *__restrict__ dst, int nx,
                                            int ny, long pitch, long plane, int strip, int j0,
                                            const SweepCoef<T> &cx, const SweepCoef<T> &cy,
                                            BlockLds<T> (&lds)[WV], Div &dv) {
  constexpr int H = 2 * STEPS;  // halo columns and rows
  static_assert(R >= 2 && R * WV > 2 * H, "a wavefront's boundary is two rows");
  static_assert(STEPS == 1 || EDGE == EDGE_CLAMP, "the ring edge is for one step");
  const int v = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int t = (int)(threadIdx.x & 63);
  const int x0 = strip * (64 - 2 * H), x = x0 - H + t;
  const int jw = j0 - H + v * R;  // this wavefront's first row
  const unsigned boff = (unsigned)min(max(x, 0), nx - 1) * (unsigned)sizeof(T);
  const X1Edge ed = x_edge<1, H>(x0, nx, t);
  Nodes<T, 1> u[R];
#pragma unroll
  for (int r = 0; r < R; ++r)
    u[r] = load_nodes<T, 1>(src + (long)min(ypos<EDGE>(jw + r, ny), ny - 1) * pitch, plane, boff);
#pragma unroll
  for (int r = 0; r < R; ++r) see_row(u[r], ed, t, dv);
  // A wavefront whose rows are out of the divisions' range only passes the remaining
  // barriers, as block_tile takes the block again.  Where it is asked costs finite
  // fields the least: tall blocks before the first barrier (before the x-sweeps it would
  // wait for every row's load), or before the last x-sweeps where registers are short,
  // low ones between the two steps, the lowest not at all in one step.  FP64 us a pass
  // with NaN everywhere, finite in brackets: 96 x 80 13.7 (10.5), 512^2 23.1 (16.8); with both
  // marches in full 15.8 and 27.9.
  enum { NEVER, IN_X, BEFORE_Y, BETWEEN };
  constexpr int ask = STEPS > 1 ? (R > 4 ? BEFORE_Y : BETWEEN)
                                : (R > 6 ? IN_X : R > 2 ? BEFORE_Y : NEVER);
  auto stand_by = [&](int passed) {
    if (!Div::kSees || __all(dv.in_range())) return false;
#pragma unroll 1
    for (int k = passed; k < 4 * STEPS - 1; ++k) __syncthreads();
    return true;
  };
#pragma unroll 1
  for (int s = 0;; ++s) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      x_sweep(u[r], lds[v].x, t, ed, cx, dv);
      pin(u[r].n[0]);
      if (ask == IN_X && r == R - 3 && stand_by(0)) return;
    }
    // after a step rows outside the grid take the edge row's value (one step's are
    // loaded so)
    if (STEPS > 1 && (jw < 0 || jw + R > ny)) {  // wavefront-uniform
#pragma unroll
      for (int r = R - 2; r >= 0; --r) u[r] = pick_nodes(jw + r < 0, u[r + 1], u[r]);
#pragma unroll
      for (int r = 1; r < R; ++r) u[r] = pick_nodes(jw + r >= ny, u[r - 1], u[r]);
    }
    Ws<T, R> w;
#pragma unroll
    for (int r = 0; r < R; ++r) w.w[r] = inv_y(u[r].n[0], cy);
    window_sync<64>();  // the x-sweeps' exchange shares the memory
    lds[v].y.first[t] = w.w[0];
    lds[v].y.second[t] = {w.w[1].b, w.w[1].d};
    lds[v].y.last[t] = {w.w[R - 1].a, w.w[R - 1].c};
    if (ask == BEFORE_Y && s == 0 && stand_by(0)) return;
    __syncthreads();
    // the row above (a and c) and two rows below; rows past the block's own
    // edge stand for nothing that an output reads, rows past the grid's take its
    // edge row
    const int va = max(v - 1, 0), vb = min(v + 1, WV - 1);
    const P2<T> above = lds[va].y.last[t], below2 = lds[vb].y.second[t];
    W4<T> e = lds[vb].y.first[t], e2 = {}, wm = {};
    __syncthreads();
    e = pick_w(STEPS > 1 && jw + R >= ny, w.w[R - 1], e);
    e2.b = STEPS > 1 && jw + R >= ny - 1 ? e.b : below2.p;
    e2.d = STEPS > 1 && jw + R >= ny - 1 ? e.d : below2.q;
    wm.a = STEPS > 1 && jw <= 0 ? w.w[0].a : above.p;
    wm.c = STEPS > 1 && jw <= 0 ? w.w[0].c : above.q;
    // each wavefront forms the face below its last row, the wavefront below
    // takes it over
    const W4<T> fe = faces(w.w[R - 2], w.w[R - 1], e, e2, cy, dv);
    lds[v].face[t] = fe;
    __syncthreads();
    W4<T> fi = lds[va].face[t];
    if (s + 1 < STEPS) __syncthreads();  // the next x-sweeps reuse the memory
    if (STEPS > 1 && jw == 0)  // the grid's first face
      fi = faces(w.w[0], w.w[0], w.w[0], w.w[1], cy, dv);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const W4<T> fo = r == R - 1 ? fe
                                  : faces(r ? w.w[r - 1] : wm, w.w[r], w.w[r + 1],
                                          r + 2 < R ? w.w[r + 2] : e, cy, dv);
      Node<T> &n = u[r].n[0];
      apply(n.vy, n.vx, n.syy, n.sxx, n.sxy, w.w[r], fi, fo, cy);
      pin(n);
      fi = fo;
    }
    if (s + 1 >= STEPS) break;
    if (ask == BETWEEN && stand_by(4)) return;
  }
  const unsigned woff = (unsigned)max(x, 0) * (unsigned)sizeof(T);
  const bool writer = t >= H && t < 64 - H && x < nx;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int i = v * R + r;  // row of the block
    if (i >= H && i < R * WV - H && jw + r < ny && writer)
      store_nodes<T, 1>(dst + (long)(jw + r) * pitch, plane, woff, u[r]);
  }
}

template <typename T, int STEPS, int EDGE, int R, int WV>
__device__ __forceinline__ void block_tile(const T *__restrict__ src, T *__restrict__ dst, int nx,
                                           int ny, long pitch, long plane, int strip, int j0,
                                           const SweepCoef<T> &cx, const SweepCoef<T> &cy,
                                           BlockLds<T> (&lds)[WV]) {
#if LE2D_LIMITER != 2
  if constexpr (sizeof(T) == 8) {  // as pair_tile
    if (coef_bounded(cx) && coef_bounded(cy)) {
      DivBounded dv;
      block_march<T, STEPS, EDGE, R, WV>(src, dst, nx, ny, pitch, plane, strip, j0, cx, cy, lds, dv);
      if (__syncthreads_and(dv.ok())) return;
    }
  }
#endif
  DivIeee<T> dv;
  block_march<T, STEPS, EDGE, R, WV>(src, dst, nx, ny, pitch, plane, strip, j0, cx, cy, lds, dv);
}

}  // namespace le2d
