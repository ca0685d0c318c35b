// sweep.hip -- the x-sweep, y-sweep and fused-step kernels for gfx950 and
// their launchers.  Numerics and the fused-step tile march: sweep_dev.h.
#include <map>
#include <mutex>
#include <tuple>

#include "block_dev.h"

namespace le2d {

// ---------------------------------------------------------------------------
// x-sweep of grids that leave the last-level cache (FP32; FP64 from 2^24 nodes on, see
// sweep_x), and of a caller who set the rows of a workgroup to other than the
// default.  A workgroup of BX lanes owns BX consecutive nodes of a row and walks
// `rows` rows.  Per row: coalesced loads of the five planes, invariants
// to LDS (with a 2-node clamped halo each side), one face per lane (lane 0
// also the segment's left face) to LDS, then the node update and coalesced
// stores.  LDS is double-buffered by row parity, so a row costs two barriers.
template <typename T, int BX>
__global__ __launch_bounds__(BX) void k_sweep_x(const T *__restrict__ src, T *__restrict__ dst,
                                                int nx, int ny, long pitch, long plane,
                                                int rows, SweepCoef<T> c) {
  __shared__ W4<T> sw[2][BX + 4];
  __shared__ W4<T> sf[2][BX + 1];
  const int t = threadIdx.x;
  const int x0 = blockIdx.x * BX;
  const int x = x0 + t;
  const int xc = min(x, nx - 1);
  // lanes 0..3 also fetch the halo nodes x0-2, x0-1, x0+BX, x0+BX+1 (clamped)
  const int hx = (t < 2) ? max(x0 - 2 + t, 0) : min(x0 + BX + (t - 2), nx - 1);
  const int hs = (t < 2) ? t : BX + t;
  const int j0 = blockIdx.y * rows;
  const int j1 = min(j0 + rows, ny);
  const unsigned boff = (unsigned)xc * (unsigned)sizeof(T);
  const unsigned hoff = (unsigned)hx * (unsigned)sizeof(T);
  const unsigned woff = (unsigned)x * (unsigned)sizeof(T);
  int b = 0;
  for (int j = j0; j < j1; ++j, b ^= 1) {
    const T *r = src + (long)j * pitch;
    Node<T> u = load_row_node(r, plane, boff);
    const W4<T> w = invariants(u.vx, u.sxx, u.vy, u.sxy, c);
    sw[b][t + 2] = w;
    if (t < 4) {
      const Node<T> h = load_row_node(r, plane, hoff);
      sw[b][hs] = invariants(h.vx, h.sxx, h.vy, h.sxy, c);
    }
    __syncthreads();
    // face x+1/2 -> sf[t+1]; lane 0 also face x0-1/2 -> sf[0]
    sf[b][t + 1] = faces(sw[b][t + 1], sw[b][t + 2], sw[b][t + 3], sw[b][t + 4], c);
    if (t == 0) sf[b][0] = faces(sw[b][0], sw[b][1], sw[b][2], sw[b][3], c);
    __syncthreads();
    if (x < nx) {
      apply(u.vx, u.vy, u.sxx, u.syy, u.sxy, w, sf[b][t], sf[b][t + 1], c);
      store_row_node(dst + (long)j * pitch, plane, woff, u);
    }
  }
}

// The x-sweep by wavefronts on their own, one row of a 64-column window each (60
// written, as the fused step's): no barrier, 2 KB of LDS per wavefront and the tiles of
// one XCD side by side, so that a window's halo and the cache lines it shares with
// its neighbour are in that XCD's L2.  What bounds it is memory: FP64 4096 x 2049 116 us
// against 138 above, 1500 x 1001 18.2 against 25.0, 8192 x 4096 460 against 502 (copy
// rate 107, 19 and 427); FP32 1500 x 1001 9.7 against 12.3.
template <typename T>
constexpr int kRowWaves = sizeof(T) == 8 ? 1 : 4;  // FP64 4096 x 2049 118 us with 4

template <typename T>
__global__ __launch_bounds__(64 * kRowWaves<T>) void k_sweep_x_row(
    const T *__restrict__ src, T *__restrict__ dst, int nx, int ny, long pitch, long plane,
    int nstrips, SweepCoef<T> c) {
  __shared__ X1Lds<T> lds[kRowWaves<T>];
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int v = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int t = (int)(threadIdx.x & 63);
  const int x0 = tile % nstrips * 60, x = x0 - 2 + t;
  const int j = tile / nstrips * kRowWaves<T> + v;
  if (j >= ny) return;  // no barriers below
  const unsigned boff = (unsigned)min(max(x, 0), nx - 1) * (unsigned)sizeof(T);
  Nodes<T, 1> u = load_nodes<T, 1>(src + (long)j * pitch, plane, boff);
  DivIeee<T> dv;
  x_sweep(u, lds[v], t, x_edge<1, 2>(x0, nx, t), c, dv);
  if (t >= 2 && t < 62 && x < nx)
    store_nodes<T, 1>(dst + (long)j * pitch, plane, (unsigned)x * (unsigned)sizeof(T), u);
}

// ---------------------------------------------------------------------------
// y-sweep.  Each lane owns one column and takes a segment of `seg` rows in
// groups of kYRows: all the group's rows and the two above and below it are loaded
// before any arithmetic, so a wavefront has 40 accesses in flight where a march that
// reads one row ahead had 5, and no access is strided.  The re-read rows come from
// the caches.  Measured at the default, one group a segment, against the march
// (us): FP32 4096 x 2049 57.8 against 69.3, 512^2 4.1 against 11.1, 8192^2 441 against
// 511; FP64 1500 x 1001 20.2 against 30.1, 8192 x 4096 488 against 511 (copy rate
// 53.5, 1.7, 427, 19 and 427).
//
// by_xcd: the tiles of one XCD are consecutive (xcd_tile), which keeps the re-read rows in
// its L2 and pays where both buffers stay in the last-level cache (FP64 1500 x 1001
// 20.2 us against 25.2); larger grids are walked in order (FP32 8192^2 441 against 456).
constexpr int kYRows = 4;

template <typename T, int EDGE>
__global__ __launch_bounds__(256) void k_sweep_y(const T *__restrict__ src, T *__restrict__ dst,
                                                 int nx, int ny, long pitch, long plane, int seg,
                                                 int nstrips, bool by_xcd, SweepCoef<T> c) {
  const int tile = by_xcd ? xcd_tile(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  const int x = tile % nstrips * (int)blockDim.x + (int)threadIdx.x;
  if (x >= nx) return;  // no barriers below
  const int j0 = tile / nstrips * seg, j1 = min(j0 + seg, ny);
  const unsigned boff = (unsigned)x * (unsigned)sizeof(T);
  for (int j = j0; j < j1; j += kYRows) {
    Node<T> u[kYRows + 4];  // positions j-2 ..
#pragma unroll
    for (int r = 0; r < kYRows + 4; ++r)
      u[r] = load_row_node(src + (long)min(ypos<EDGE>(j + r - 2, ny), ny - 1) * pitch, plane, boff);
    W4<T> wm = inv_y(u[1], c), w0 = inv_y(u[2], c), w1 = inv_y(u[3], c);
    W4<T> fin = faces(inv_y(u[0], c), wm, w0, w1, c);  // face j-1/2
#pragma unroll
    for (int r = 0; r < kYRows; ++r) {
      const W4<T> w2 = inv_y(u[r + 4], c);
      const W4<T> fout = faces(wm, w0, w1, w2, c);
      Node<T> &n = u[r + 2];
      apply(n.vy, n.vx, n.syy, n.sxx, n.sxy, w0, fin, fout, c);
      if (j + r < j1) store_row_node(dst + (long)(j + r) * pitch, plane, boff, n);
      fin = fout;
      wm = w0;
      w0 = w1;
      w1 = w2;
    }
  }
}

// ---------------------------------------------------------------------------
// One step over one grid, marched in windows of FB columns: 64 by one wavefront
// that keeps its own state (step_tile in pair_dev.h; FP64 1500 x 1001 26.0 us against
// 27.9 through march_tile, 2048^2 77 against 82), wider ones, which only a caller
// asks for, through march_tile in sweep_dev.h.
template <typename T, int EDGE, int FB>
__global__ __launch_bounds__(FB, 3) void k_step_xy(const T *__restrict__ src, T *__restrict__ dst,
                                                int nx, int ny, long pitch, long plane, int seg,
                                                int nstrips, SweepCoef<T> cx, SweepCoef<T> cy) {
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int strip = tile % nstrips, segi = tile / nstrips;
  const int j0 = segi * seg;
  const int j1 = min(j0 + seg, ny);
  if constexpr (FB == 64) {
    __shared__ X1Lds<T> lds;
    step_tile<T, EDGE>(src, dst, nx, ny, pitch, plane, strip, j0, j1, cx, cy, lds);
  } else {
    __shared__ W4<T> sw[FB];
    __shared__ W4<T> sf[FB];
    march_tile_alt<T, EDGE, FB>(src, dst, nx, ny, pitch, plane, strip, j0, j1, segi, cx, cy, sw,
                                sf);
  }
}

// One step over one grid in blocks of R rows on each of WV wavefronts (block_tile).
template <typename T, int EDGE, int R, int WV>
__global__ __launch_bounds__(64 * WV, (R > 6 ? 2 : 1)) void k_step_block(
    const T *__restrict__ src, T *__restrict__ dst, int nx, int ny, long pitch, long plane,
    int nstrips, SweepCoef<T> cx, SweepCoef<T> cy) {
  __shared__ BlockLds<T> lds[WV];
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  block_tile<T, 1, EDGE, R, WV>(src, dst, nx, ny, pitch, plane, tile % nstrips,
                                tile / nstrips * (R * WV - 4), cx, cy, lds);
}

// Two steps over one grid (pair_tile in pair_dev.h) in windows of FB columns,
// FB/64 per lane ...
template <typename T, int FB>
__global__ __launch_bounds__(128, (pair_waves<T, FB / 64>())) void k_step2_xy(
    const T *__restrict__ src, T *__restrict__ dst, int nx, int ny, long pitch, long plane,
    int seg, int nstrips, SweepCoef<T> cx, SweepCoef<T> cy) {
  __shared__ PairLds<T, FB / 64> lds;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int strip = tile % nstrips, segi = tile / nstrips;
  const int j0 = segi * seg;
  const int j1 = min(j0 + seg, ny);
  pair_tile<T, FB / 64>(src, dst, nx, ny, pitch, plane, strip, j0, j1, cx, cy, lds);
}

// ... and in windows of 64 columns, one per lane: the same kernel at FB = 64 under the
// name that profiles and the resource report know.  HOLD is part of that name
// (the march goes by kHoldInv).
template <typename T, bool HOLD>
__global__ __launch_bounds__(128, (pair_waves<T, 1>())) void k_step2_split(
    const T *__restrict__ src, T *__restrict__ dst, int nx, int ny, long pitch, long plane,
    int seg, int nstrips, SweepCoef<T> cx, SweepCoef<T> cy) {
  __shared__ PairLds<T, 1> lds;
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int strip = tile % nstrips, segi = tile / nstrips;
  const int j0 = segi * seg;
  const int j1 = min(j0 + seg, ny);
  pair_tile<T, 1>(src, dst, nx, ny, pitch, plane, strip, j0, j1, cx, cy, lds);
}

// Two steps over one grid in blocks of R rows on each of WV wavefronts
// (block_tile).
template <typename T, int R, int WV>
__global__ __launch_bounds__(64 * WV) void k_step2_block(const T *__restrict__ src,
                                                       T *__restrict__ dst, int nx, int ny,
                                                       long pitch, long plane, int nstrips,
                                                       SweepCoef<T> cx, SweepCoef<T> cy) {
  __shared__ BlockLds<T> lds[WV];
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  block_tile<T, 2, EDGE_CLAMP, R, WV>(src, dst, nx, ny, pitch, plane, tile % nstrips,
                       tile / nstrips * (R * WV - 8), cx, cy, lds);
}

// ---------------------------------------------------------------------------
// Launchers.

template <typename T, int FB>
static void launch_step_xy(DevGrid *g, const SweepCoef<T> &cx, const SweepCoef<T> &cy, int edge,
                           int seg, unsigned nblocks, int nstrips) {
  const T *src = static_cast<const T *>(g->buf[g->cur]);
  T *dst = static_cast<T *>(g->buf[g->cur ^ 1]);
  if (edge == EDGE_RING)
    hipLaunchKernelGGL((k_step_xy<T, EDGE_RING, FB>), dim3(nblocks), dim3(FB), 0, g->stream, src,
                       dst, g->nx, g->ny, g->pitch, g->plane, seg, nstrips, cx, cy);
  else
    hipLaunchKernelGGL((k_step_xy<T, EDGE_CLAMP, FB>), dim3(nblocks), dim3(FB), 0, g->stream, src,
                       dst, g->nx, g->ny, g->pitch, g->plane, seg, nstrips, cx, cy);
}

// The two-step kernel of a window of `cols` columns (pair_cols).
template <typename T>
using PairKernel = void (*)(const T *, T *, int, int, long, long, int, int, SweepCoef<T>,
                            SweepCoef<T>);
template <typename T>
static PairKernel<T> pair_kernel(int cols) {
  if (cols == 64) return k_step2_split<T, sizeof(T) == 4>;
  if constexpr (sizeof(T) == 4)
    if (cols == 256) return k_step2_xy<T, 256>;
  return k_step2_xy<T, 128>;
}

// The block kernels by the rows they write, shortest first: two steps ...
template <typename T>
struct BlockKernel {
  int rows, wavefronts;
  void (*kernel)(const T *, T *, int, int, long, long, int, SweepCoef<T>, SweepCoef<T>);
};
template <typename T, int R, int WV>
constexpr BlockKernel<T> block_kernel() {
  return {R * WV - 8, WV, k_step2_block<T, R, WV>};
}
static const BlockKernel<double> kBlocks8[] = {
    block_kernel<double, 2, 6>(), block_kernel<double, 2, 8>(), block_kernel<double, 3, 8>(),
    block_kernel<double, 4, 8>(), block_kernel<double, 5, 8>(), block_kernel<double, 6, 8>()};
static const BlockKernel<float> kBlocks4[] = {
    block_kernel<float, 2, 6>(), block_kernel<float, 2, 8>(),  block_kernel<float, 3, 8>(),
    block_kernel<float, 4, 8>(), block_kernel<float, 4, 12>(), block_kernel<float, 6, 12>()};
static_assert(sizeof kBlocks8 / sizeof *kBlocks8 == kBlockKinds &&
              sizeof kBlocks4 / sizeof *kBlocks4 == kBlockKinds);
template <typename T>
static const BlockKernel<T> *block_kernels() {
  if constexpr (sizeof(T) == 8) return kBlocks8;
  else return kBlocks4;
}

// ... and one, with either edge.
template <typename T, int R, int WV, int EDGE>
constexpr BlockKernel<T> step_block_kernel() {
  return {R * WV - 4, WV, k_step_block<T, EDGE, R, WV>};
}
template <typename T, int EDGE>
static const BlockKernel<T> *step_block_kernels() {
  constexpr int last_r = sizeof(T) == 8 ? 7 : 4, last_wv = sizeof(T) == 8 ? 4 : 12;
  static const BlockKernel<T> kernels[] = {
      step_block_kernel<T, 2, 4, EDGE>(), step_block_kernel<T, 2, 8, EDGE>(),
      step_block_kernel<T, 3, 8, EDGE>(), step_block_kernel<T, last_r, last_wv, EDGE>()};
  static_assert(sizeof kernels / sizeof *kernels == kStepBlockKinds);
  return kernels;
}

int step_block_rows(int elem, int kind) {
  return elem == 8 ? step_block_kernels<double, EDGE_CLAMP>()[kind].rows
                   : step_block_kernels<float, EDGE_CLAMP>()[kind].rows;
}

int block_rows(int elem, int kind) {
  return elem == 8 ? kBlocks8[kind].rows : kBlocks4[kind].rows;
}

int device_cus() {
  int dev = 0, cus = 0;
  if (hipGetDevice(&dev) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
    return 0;
  return cus;
}

// Rows per segment for a launch of `lanes` lanes per segment and strip: `seg`, or
// the lowest height above it at which the launch stays under 2^32 work-items,
// the runtime's limit (one row each on 2^32 nodes of 40 bytes is past it).
static int launch_rows(int seg, int ny, int nstrips, int lanes) {
  while ((long)nstrips * (((long)ny + seg - 1) / seg) * lanes > 0xffffffffL) ++seg;
  return seg;
}

// Launches the kernel of `kinds` that writes `rows` rows (the first if none does)
// on the blocks of `width` columns that cover the grid.
template <typename T>
static int launch_blocks(DevGrid *g, const SweepCoef<T> &cx, const SweepCoef<T> &cy,
                         const BlockKernel<T> *kinds, int count, int rows, int width,
                         const char *what) {
  const BlockKernel<T> *b = kinds;
  for (int k = 1; k < count; ++k)
    if (kinds[k].rows == rows) b = kinds + k;
  const int nstrips = (g->nx + width - 1) / width;
  const long nblocks = (long)nstrips * ((g->ny + b->rows - 1) / b->rows);
  if (nblocks > 0x7fffffffL) return set_error(ERR_ARG, "%s: grid too large", what);
  hipLaunchKernelGGL(b->kernel, dim3((unsigned)nblocks), dim3(64 * b->wavefronts), 0, g->stream,
                     static_cast<const T *>(g->buf[g->cur]), static_cast<T *>(g->buf[g->cur ^ 1]),
                     g->nx, g->ny, g->pitch, g->plane, nstrips, cx, cy);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(ERR_DEVICE, "%s launch: %s", what, hipGetErrorString(e));
  g->cur ^= 1;
  return OK;
}

template <typename T>
int step_xy(DevGrid *g, const SweepCoef<T> &cx, const SweepCoef<T> &cy, int edge) {
  if (g->elem != (int)sizeof(T)) return set_error(ERR_ARG, "step_xy: element size mismatch");
  if (g->tiles.step_rows)
    return launch_blocks<T>(g, cx, cy,
                            edge == EDGE_RING ? step_block_kernels<T, EDGE_RING>()
                                              : step_block_kernels<T, EDGE_CLAMP>(),
                            kStepBlockKinds, g->tiles.step_rows, 60, "step_xy");
  const int fb = g->tiles.xy_block == 64 || g->tiles.xy_block == 256 ? g->tiles.xy_block : 128;
  const int nstrips = (g->nx + fb - 5) / (fb - 4);
  const int seg = max(1, g->tiles.xy_seg);
  const long nsegs = (g->ny + seg - 1) / seg;
  const long nblocks = nsegs * nstrips;
  if (nblocks > 0x7fffffffL) return set_error(ERR_ARG, "step_xy: grid too large");
  if (fb == 64)
    launch_step_xy<T, 64>(g, cx, cy, edge, seg, (unsigned)nblocks, nstrips);
  else if (fb == 128)
    launch_step_xy<T, 128>(g, cx, cy, edge, seg, (unsigned)nblocks, nstrips);
  else
    launch_step_xy<T, 256>(g, cx, cy, edge, seg, (unsigned)nblocks, nstrips);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(ERR_DEVICE, "step_xy launch: %s", hipGetErrorString(e));
  g->cur ^= 1;
  return OK;
}

template <typename T>
int step2_xy(DevGrid *g, const SweepCoef<T> &cx, const SweepCoef<T> &cy) {
  if (g->elem != (int)sizeof(T)) return set_error(ERR_ARG, "step2_xy: element size mismatch");
  if (g->tiles.block_rows)
    return launch_blocks<T>(g, cx, cy, block_kernels<T>(), kBlockKinds, g->tiles.block_rows, 56,
                            "step2_xy");
  if (g->tiles.pair_seg < 1) return set_error(ERR_ARG, "step2_xy: no pair segment height");
  const int cols = pair_cols(g->elem, g->tiles.pair_block);
  const int nstrips = (g->nx + cols - 9) / (cols - 8);
  const int seg = launch_rows(g->tiles.pair_seg, g->ny, nstrips, 128);
  const long nblocks = ((long)g->ny + seg - 1) / seg * nstrips;
  hipLaunchKernelGGL(pair_kernel<T>(cols), dim3((unsigned)nblocks), dim3(128), 0, g->stream,
                     static_cast<const T *>(g->buf[g->cur]), static_cast<T *>(g->buf[g->cur ^ 1]),
                     g->nx, g->ny, g->pitch, g->plane, seg, nstrips, cx, cy);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(ERR_DEVICE, "step2_xy launch: %s", hipGetErrorString(e));
  g->cur ^= 1;
  return OK;
}

template <typename K>
static int occupancy_of(K kernel, int lanes) {
  int n = 0;
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, lanes, 0) == hipSuccess ? n : 0;
}

// Workgroups per CU x CUs of the current device, cached per device.
long pair_resident(int elem, int window) {
  static std::mutex mu;
  static std::map<std::tuple<int, int, int>, long> cache;
  int dev = 0;
  const int cus = device_cus(), cols = pair_cols(elem, window);
  if (!cus || hipGetDevice(&dev) != hipSuccess) return 0;
  std::lock_guard<std::mutex> lk(mu);
  const auto key = std::make_tuple(dev, elem, cols);
  auto it = cache.find(key);
  if (it != cache.end()) return it->second;
  const int per = elem == 8 ? occupancy_of(pair_kernel<double>(cols), 128)
                            : occupancy_of(pair_kernel<float>(cols), 128);
  const long r = (long)min(4, per) * cus;
  cache[key] = r;
  return r;
}

template int step2_xy<double>(DevGrid *, const SweepCoef<double> &, const SweepCoef<double> &);
template int step2_xy<float>(DevGrid *, const SweepCoef<float> &, const SweepCoef<float> &);
template int step_xy<double>(DevGrid *, const SweepCoef<double> &, const SweepCoef<double> &, int);
template int step_xy<float>(DevGrid *, const SweepCoef<float> &, const SweepCoef<float> &, int);

// Both buffers of the grid stay in the 256 MB last-level cache from one sweep to
// the next.
static bool stays_cached(const DevGrid *g) {
  return 2 * g->pitch * (long)g->ny * g->elem <= 256l << 20;
}

template <typename T>
int sweep_x(DevGrid *g, const SweepCoef<T> &c) {
  if (g->elem != (int)sizeof(T)) return set_error(ERR_ARG, "sweep_x: element size mismatch");
  const T *src = static_cast<const T *>(g->buf[g->cur]);
  T *dst = static_cast<T *>(g->buf[g->cur ^ 1]);
  // the wavefront form unless the caller set the rows of a workgroup; grids that leave
  // the cache stay with whole workgroups, whose 1 to 2 KB row pieces need fewer
  // halo lines, in FP32 (4096 x 2049 59 us against 62) and in FP64 from 2^24 nodes on
  // (6000 x 5000 415 against 466, 8192^2 903 against 931; 3900^2 223 against 213)
  if (!g->tiles.x_fixed &&
      (stays_cached(g) || (sizeof(T) == 8 && (long)g->nx * g->ny < 1l << 24))) {
    constexpr int waves = kRowWaves<T>;
    const int nstrips = (g->nx + 59) / 60;
    const long nblocks = (long)nstrips * ((g->ny + waves - 1) / waves);
    if (nblocks > 0x7fffffffL) return set_error(ERR_ARG, "sweep_x: grid too large");
    hipLaunchKernelGGL((k_sweep_x_row<T>), dim3((unsigned)nblocks), dim3(64 * waves), 0, g->stream,
                       src, dst, g->nx, g->ny, g->pitch, g->plane, nstrips, c);
  } else {
    constexpr int BX = 256;
    // gridDim.y is at most 65535
    const int rows = max(max(1, g->tiles.x_rows), (g->ny + 65534) / 65535);
    dim3 grid((g->nx + BX - 1) / BX, (g->ny + rows - 1) / rows);
    hipLaunchKernelGGL((k_sweep_x<T, BX>), grid, dim3(BX), 0, g->stream, src, dst, g->nx, g->ny,
                       g->pitch, g->plane, rows, c);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(ERR_DEVICE, "sweep_x launch: %s", hipGetErrorString(e));
  g->cur ^= 1;
  return OK;
}

template <typename T>
int sweep_y(DevGrid *g, const SweepCoef<T> &c, int edge) {
  if (g->elem != (int)sizeof(T)) return set_error(ERR_ARG, "sweep_y: element size mismatch");
  const int bx = g->tiles.y_block == 64 || g->tiles.y_block == 128 ? g->tiles.y_block : 256;
  const int nstrips = (g->nx + bx - 1) / bx;
  const int seg = launch_rows(max(1, g->tiles.y_seg), g->ny, nstrips, bx);
  const long nblocks = ((long)g->ny + seg - 1) / seg * nstrips;
  const T *src = static_cast<const T *>(g->buf[g->cur]);
  T *dst = static_cast<T *>(g->buf[g->cur ^ 1]);
  const bool by_xcd = stays_cached(g);
  if (edge == EDGE_RING)
    hipLaunchKernelGGL((k_sweep_y<T, EDGE_RING>), dim3((unsigned)nblocks), dim3(bx), 0, g->stream,
                       src, dst, g->nx, g->ny, g->pitch, g->plane, seg, nstrips, by_xcd, c);
  else
    hipLaunchKernelGGL((k_sweep_y<T, EDGE_CLAMP>), dim3((unsigned)nblocks), dim3(bx), 0, g->stream,
                       src, dst, g->nx, g->ny, g->pitch, g->plane, seg, nstrips, by_xcd, c);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return set_error(ERR_DEVICE, "sweep_y launch: %s", hipGetErrorString(e));
  g->cur ^= 1;
  return OK;
}

template int sweep_x<double>(DevGrid *, const SweepCoef<double> &);
template int sweep_x<float>(DevGrid *, const SweepCoef<float> &);
template int sweep_y<double>(DevGrid *, const SweepCoef<double> &, int);
template int sweep_y<float>(DevGrid *, const SweepCoef<float> &, int);

}  // namespace le2d
