// engine.hip -- device memory, host<->device transfers and error state of
// the sweep engine.
#include <algorithm>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include <mutex>
#include <unordered_map>

#include "engine.h"
#include "le2d.h"

namespace le2d {

static thread_local char g_err[512] = "";

int set_error(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
  return code;
}

const char *last_error() { return g_err; }

int require_device() {
  int n = 0;
  hipError_t e = hipGetDeviceCount(&n);
  if (e != hipSuccess || n < 1) {
    fprintf(stderr,
            "le2d: no HIP device is available (%s); this library runs the sweeps on the GPU "
            "only and has no CPU path\n",
            e != hipSuccess ? hipGetErrorString(e) : "device count 0");
    abort();
  }
  return OK;
}

// Device allocator.  Allocations made by an installed allocator are recorded
// with its free function, so each is returned to the allocator that made it.
namespace {
struct Allocator {
  le2d_alloc_fn alloc = nullptr;
  le2d_free_fn release = nullptr;
  void *ctx = nullptr;
};
struct Owner {
  le2d_free_fn release;
  void *ctx;
};
std::mutex g_alloc_mu;
Allocator g_alloc;
std::unordered_map<void *, Owner> g_owned;
}  // namespace

int dev_alloc(void **p, size_t bytes, const char *what) {
  *p = nullptr;
  Allocator a;
  {
    std::lock_guard<std::mutex> lk(g_alloc_mu);
    a = g_alloc;
  }
  if (a.alloc) {
    void *q = nullptr;
    if (a.alloc(&q, bytes, a.ctx) != 0 || !q)
      return set_error(ERR_NOMEM, "%s: the installed allocator refused %zu bytes", what, bytes);
    std::lock_guard<std::mutex> lk(g_alloc_mu);
    g_owned[q] = {a.release, a.ctx};
    *p = q;
    return OK;
  }
  const hipError_t e = hipMalloc(p, bytes);
  if (e != hipSuccess) {
    *p = nullptr;
    return set_error(ERR_NOMEM, "%s: hipMalloc(%zu) failed: %s", what, bytes,
                     hipGetErrorString(e));
  }
  return OK;
}

}  // namespace le2d

extern "C" int le2d_set_device_allocator(le2d_alloc_fn alloc, le2d_free_fn release, void *ctx) {
  if ((alloc == nullptr) != (release == nullptr))
    return le2d::set_error(le2d::ERR_ARG, "set_device_allocator: give both functions or neither");
  std::lock_guard<std::mutex> lk(le2d::g_alloc_mu);
  le2d::g_alloc = {alloc, release, alloc ? ctx : nullptr};
  return le2d::OK;
}

namespace le2d {

void dev_free(void *p) {
  if (!p) return;
  Owner o{nullptr, nullptr};
  {
    std::lock_guard<std::mutex> lk(g_alloc_mu);
    auto it = g_owned.find(p);
    if (it != g_owned.end()) {
      o = it->second;
      g_owned.erase(it);
    }
  }
  if (o.release)
    o.release(p, o.ctx);
  else
    (void)hipFree(p);
}

// One grid row of one field, padded to 256 bytes so every row starts aligned.
static long field_pitch(int nx, int elem) {
  const long per = 256 / elem;
  return ((long)nx + per - 1) / per * per;
}

// Row-interleaved fields: the five fields of grid row j are stored side by
// side (vx, vy, sxx, sxy, syy), each padded to 256 bytes, and the rows follow
// one another.  The workgroups of a sweep that work on the same rows then
// read and write one contiguous region instead of five regions a plane
// apart, which keeps the DRAM access stream local.
void grid_layout(int elem, int nx, int ny, long *pitch, long *plane) {
  (void)ny;
  const long fp = field_pitch(nx, elem);
  *pitch = 5 * fp;
  *plane = fp;
}

bool row_fits(int elem, int nx) {
  return nx >= 1 && 5 * field_pitch(nx, elem) * (long)elem <= 0x7fffffffL;
}

size_t grid_bytes(int elem, int nx, int ny) {
  return (size_t)5 * field_pitch(nx, elem) * ny * elem;
}

int grid_alloc(DevGrid *g, int elem, int nx, int ny, hipStream_t stream) {
  if ((elem != 4 && elem != 8) || nx < 3 || ny < 3)
    return set_error(ERR_ARG, "grid_alloc: need elem 4|8 and nx, ny >= 3 (got %d, %d, %d)", elem,
                     nx, ny);
  if (!row_fits(elem, nx)) return set_error(ERR_ARG, "grid_alloc: row of %d nodes too long", nx);
  g->elem = elem;
  g->nx = nx;
  g->ny = ny;
  grid_layout(elem, nx, ny, &g->pitch, &g->plane);
  g->stream = stream;
  g->cur = 0;
  (void)hipGetDevice(&g->device);
  const size_t bytes = grid_bytes(elem, nx, ny);
  for (int k = 0; k < 2; ++k) {
    const int rc = dev_alloc(&g->buf[k], bytes, "grid_alloc");
    if (rc) {
      grid_free(g);
      return rc;
    }
  }
  g->tiles = default_tiles(elem, nx, ny);
  return OK;
}

void grid_free(DevGrid *g) {
  for (int k = 0; k < 2; ++k) {
    dev_free(g->buf[k]);
    g->buf[k] = nullptr;
  }
}

// AOS (node-contiguous, unpitched) <-> the device layout.  One lane per node;
// the AOS side is read/written as 5 consecutive values per lane.
template <typename T>
__global__ void k_aos_to_planes(const T *__restrict__ aos, T *__restrict__ pl, int nx, int ny,
                                long pitch, long plane) {
  const long n = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (long)nx * ny) return;
  const long j = n / nx, i = n - j * nx;
  const T *s = aos + 5 * n;
  T *d = pl + j * pitch + i;
#pragma unroll
  for (int q = 0; q < 5; ++q) d[q * plane] = s[q];
}

template <typename T>
__global__ void k_planes_to_aos(const T *__restrict__ pl, T *__restrict__ aos, int nx, int ny,
                                long pitch, long plane) {
  const long n = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (n >= (long)nx * ny) return;
  const long j = n / nx, i = n - j * nx;
  const T *s = pl + j * pitch + i;
  T *d = aos + 5 * n;
#pragma unroll
  for (int q = 0; q < 5; ++q) d[q] = s[q * plane];
}

static int check(hipError_t e, const char *what) {
  if (e != hipSuccess) return set_error(ERR_DEVICE, "%s: %s", what, hipGetErrorString(e));
  return OK;
}

// The other ping-pong buffer stages the AOS image (it holds at least 5*nx*ny
// values and carries no state between steps).
int grid_upload(DevGrid *g, const void *host, int soa) {
  const size_t es = g->elem;
  const size_t row = (size_t)g->nx * es;
  void *cur = g->buf[g->cur];
  if (soa) {
    for (int q = 0; q < 5; ++q) {
      const char *h = static_cast<const char *>(host) + (size_t)q * g->nx * g->ny * es;
      char *d = static_cast<char *>(cur) + (size_t)q * g->plane * es;
      int rc = check(hipMemcpy2DAsync(d, g->pitch * es, h, row, row, g->ny, hipMemcpyHostToDevice,
                                      g->stream),
                     "upload planes");
      if (rc) return rc;
    }
    return check(hipStreamSynchronize(g->stream), "upload sync");
  }
  void *stage = g->buf[g->cur ^ 1];
  const size_t bytes = (size_t)g->nx * g->ny * 5 * es;
  int rc = check(hipMemcpyAsync(stage, host, bytes, hipMemcpyHostToDevice, g->stream), "upload");
  if (rc) return rc;
  const long n = (long)g->nx * g->ny;
  const int bs = 256;
  const unsigned nb = (unsigned)((n + bs - 1) / bs);
  if (g->elem == 8)
    hipLaunchKernelGGL(k_aos_to_planes<double>, dim3(nb), dim3(bs), 0, g->stream,
                       static_cast<const double *>(stage), static_cast<double *>(cur), g->nx, g->ny,
                       g->pitch, g->plane);
  else
    hipLaunchKernelGGL(k_aos_to_planes<float>, dim3(nb), dim3(bs), 0, g->stream,
                       static_cast<const float *>(stage), static_cast<float *>(cur), g->nx, g->ny,
                       g->pitch, g->plane);
  rc = check(hipGetLastError(), "aos_to_planes launch");
  if (rc) return rc;
  return check(hipStreamSynchronize(g->stream), "upload sync");
}

int grid_download(DevGrid *g, void *host, int soa) {
  const size_t es = g->elem;
  const size_t row = (size_t)g->nx * es;
  void *cur = g->buf[g->cur];
  if (soa) {
    for (int q = 0; q < 5; ++q) {
      char *h = static_cast<char *>(host) + (size_t)q * g->nx * g->ny * es;
      const char *d = static_cast<const char *>(cur) + (size_t)q * g->plane * es;
      int rc = check(hipMemcpy2DAsync(h, row, d, g->pitch * es, row, g->ny, hipMemcpyDeviceToHost,
                                      g->stream),
                     "download planes");
      if (rc) return rc;
    }
    return check(hipStreamSynchronize(g->stream), "download sync");
  }
  void *stage = nullptr;
  int rc = grid_aos_image(g, &stage);
  if (rc) return rc;
  rc = check(hipMemcpyAsync(host, stage, (size_t)g->nx * g->ny * 5 * es, hipMemcpyDeviceToHost,
                            g->stream),
             "download");
  if (rc) return rc;
  return check(hipStreamSynchronize(g->stream), "download sync");
}

int grid_aos_image(DevGrid *g, void **image) {
  const void *cur = g->buf[g->cur];
  void *stage = *image = g->buf[g->cur ^ 1];
  const long n = (long)g->nx * g->ny;
  const int bs = 256;
  const unsigned nb = (unsigned)((n + bs - 1) / bs);
  if (g->elem == 8)
    hipLaunchKernelGGL(k_planes_to_aos<double>, dim3(nb), dim3(bs), 0, g->stream,
                       static_cast<const double *>(cur), static_cast<double *>(stage), g->nx, g->ny,
                       g->pitch, g->plane);
  else
    hipLaunchKernelGGL(k_planes_to_aos<float>, dim3(nb), dim3(bs), 0, g->stream,
                       static_cast<const float *>(cur), static_cast<float *>(stage), g->nx, g->ny,
                       g->pitch, g->plane);
  return check(hipGetLastError(), "planes_to_aos launch");
}

static int step_blocks(int elem, int nx, int ny);
static int step_segment(int nx, int ny);
static long pair_blocks(int nx, int ny, int rows);

Tiles default_tiles(int elem, int nx, int ny) {
  Tiles t;
  // one row per x-sweep workgroup (the most workgroups in flight): 8192^2
  // FP32 0.426 ms against 0.457 at 4 rows
  t.x_rows = 1;
  t.pair_split = 0;
  t.step_rows = step_blocks(elem, nx, ny);
  if (t.step_rows == 0) {
    t.xy_block = 64;
    t.xy_seg = step_segment(nx, ny);
  } else {
    // the tiles of a material plane's single steps: 256-lane windows from 4096
    // columns on, else one-wave windows, and ~64 workgroups per CU in segments of
    // at least 16 rows (short segments keep the halo rows of neighbouring segments
    // in L2), shorter where that leaves the device idle
    t.xy_block = nx >= 4096 ? 256 : 64;
    const long strips = (nx + t.xy_block - 5) / (t.xy_block - 4);
    const long want = (16384 + strips - 1) / strips;
    t.xy_seg = (int)std::min<long>(std::max<long>(16, (ny + want - 1) / want), ny);
    if (t.xy_block == 64 && strips * ((ny + 15) / 16) < 12 * device_cus())
      t.xy_seg = std::min(16, step_segment(nx, ny));
  }
  // FP64 at most 128 columns: 4096^2 248 us against 260 at 256, 8192^2 1005 against 1036
  // (FP32 460 at 256 against 490)
  t.y_block = elem == 4 && nx >= 8 * 256 ? 256 : (nx >= 8 * 128 ? 128 : 64);
  t.y_seg = std::min(4, ny);  // one group of rows (kYRows in sweep.hip)
  const GridSize size{nx, ny};
  const PairShape p = pick_pair_shape(elem, &size, 1, 0, 192);
  int window = p.window, seg = p.seg;
  // blocks where each has a compute unit to itself, of the fewest rows that give
  // that (block_dev.h has both sides' times); in FP32, where several share one, also
  // blocks of 40 rows on grids of up to 16 for each (us a pass, blocks against the
  // march at its default shape: 2500 x 1500 41.2 and 45.1, 2961 x 2216 64.9 and 70.2,
  // 3500 x 2500, 15.5 for each, 89.8 and 95.5; against the march's fastest shape, which
  // only the tuner finds, 1200^2 21.0 and 23.2, 2048^2 43.5 and 43.0, 3000^2 and 3500
  // x 2500 the same or better: the tuner keeps the blocks)
  int rows = 0;
  for (int k = 0; k < kBlockKinds && !rows; ++k)
    if (pair_blocks(nx, ny, block_rows(elem, k)) <= device_cus()) rows = block_rows(elem, k);
  if (elem == 4 && !rows && pair_blocks(nx, ny, 40) <= 16 * device_cus()) rows = 40;
  if (rows) {
    window = 64;
    seg = rows;
  }
  t.pair_block = window;
  t.pair_seg = seg;
  t.block_rows = pair_block_rows(elem, nx, ny, window, seg);
  return t;
}

static long pair_blocks(int nx, int ny, int rows) {
  return (long)((nx + 55) / 56) * ((ny + rows - 1) / rows);
}

// A block height in the 64-column window, on grids of up to two such blocks for each
// compute unit, in FP32 up to four, of 40 rows up to sixteen: there blocks are no
// slower than a march of that height (us a pass, blocks of so many rows and so
// many for each unit against marches one row lower and higher: FP64 900^2 32, 1.9:
// 37 and 47, 49; FP32 1500 x 1001 24, 4.4: 23.0 and 26.0, 27.1, but 2500 x 1500 24, 11:
// 50 and 45, 44 and 64, 4.2: 55 and 52, 53; 40, 6.7: 43.0 and 43.9, 45.2).
int pair_block_rows(int elem, int nx, int ny, int window, int seg) {
  if (window != 64) return 0;
  for (int k = 0; k < kBlockKinds; ++k)
    if (block_rows(elem, k) == seg) {
      const int each = elem == 8 ? 2 : seg == 40 ? 16 : 4;
      return pair_blocks(nx, ny, seg) <= each * device_cus() ? seg : 0;
    }
  return 0;
}

void set_pair_shape(DevGrid *g, int window, int seg) {
  g->tiles.pair_block = window;
  g->tiles.pair_seg = seg;
  g->tiles.block_rows = pair_block_rows(g->elem, g->nx, g->ny, window, seg);
}

// Rows of the single step's blocks, 0 for the march.  The lowest blocks of which every
// one has a compute unit to itself (us, march against block: FP64 96 x 80 6.0
// against 4.1, 300 x 250 7.5 against 5.5, 512^2 10.3 against 8.0).  Past that FP32
// stays with blocks of 20 rows (900^2 10.5 against 8.2, 1500 x 1001 14.4 against 11.7, 3000^2
// 84 against 73) up to grids far outside the last-level cache, where 44 rows re-read
// fewer halo rows (8192 x 4096 254 against 272 at 20; 3000^2 74.3 against 72.9).  FP64
// blocks hold the registers of two wavefronts per SIMD and last long, so the march
// comes first (900^2 18.4 against 20.4, 1500 x 1001 26.0 against 30.9) until blocks of 24
// rows make several rounds (2048^2 77 both, 3000^2 170 against 153, 8192 x 4096
// 577 against 565; from 2^26 nodes on, against 256-lane windows, the fastest march
// there: 4096 x 17000 1057 against 988, 10000^2 1617 against 1559, 14000^2 3206
// against 3114, but 8192^2 1061 to 1081 against 1080).
static int step_blocks(int elem, int nx, int ny) {
  const long strips = (nx + 59) / 60, cus = device_cus();
  auto blocks = [&](int kind) {
    const int rows = step_block_rows(elem, kind);
    return strips * ((ny + rows - 1) / rows);
  };
  int kind = 0;
  while (kind < kStepBlockKinds - 1 && blocks(kind) > cus) ++kind;
  if (kind < kStepBlockKinds - 1) return step_block_rows(elem, kind);
  if (blocks(kind) >= (elem == 8 ? 12 : 24) * cus) return step_block_rows(elem, kind);
  return elem == 8 ? 0 : step_block_rows(elem, kind - 1);
}

// Segment height of the single step's march in 64-column windows.  A row costs a
// wavefront about the same again for each wavefront that shares its SIMD, and as
// much once more for its own latency, so a launch of w wavefronts per SIMD (at most
// three at once) lasts (rows marched) x (1 + w): FP64 1500 x 1001 26.0 us at 13 rows
// (w = 2), 28.7 at 16 (2), 29.1 at 11 (3), 30.7 at 8 (4); 512^2 10.3 at 6 (1), 11.7
// at 4 (2).
static int step_segment(int nx, int ny) {
  const long strips = (nx + 59) / 60, simds = std::max(4, 4 * device_cus());
  int best = 2;
  long best_cost = 0;
  for (int s = 2; s <= std::max(2, std::min(ny, 64)); ++s) {
    const long n = strips * ((ny + s - 1) / s), full = n / (3 * simds);
    const long last = (n - full * 3 * simds + simds - 1) / simds;
    const long cost = (s + 5) * (full * 4 + (last ? 1 + last : 0));
    if (!best_cost || cost < best_cost) {
      best_cost = cost;
      best = s;
    }
  }
  return best;
}

static long pair_slots(int elem, int window) {
  const long r = pair_resident(elem, window);
  return r > 0 ? r : 1024;
}

std::vector<int> pair_round_segs(int elem, int nx, int ny, int window) {
  const int width = pair_cols(elem, window) - 8;
  const long strips = (nx + width - 1) / width, slots = pair_slots(elem, window);
  std::vector<int> segs;
  for (long k = 1; k <= 8; ++k) {
    const long n = k * slots / strips;
    const int s = n > 0 ? (int)std::max<long>(2, (ny + n - 1) / n) : 0;
    if (s && s <= 192 && (segs.empty() || segs.back() != s)) segs.push_back(s);
  }
  return segs;
}

// Cost of a shape: rounds of workgroups x rows each marches (its segment and
// the 8 re-read halo rows) x columns of its window, per unit of the window's
// rate.  A round is the workgroups that saturate the device, four per CU (two
// wavefronts per SIMD: FP64 1024^2 in 64-column windows 40 us at 20 rows with
// 1.9 wavefronts per SIMD, 44 at 16 with 2.4); a last round that is mostly
// empty costs as much as a full one (FP64 2048^2 in 128-column windows 109 us at
// 37 rows, one full round, 132 at 32 and 138 at 54), and a grid that does not
// fill a round takes the shortest segments that stay in it (FP64 512^2 19 us at
// 6 rows, 20.5 at 8).  Wider windows recompute fewer halo columns but need a
// larger grid (FP64 2048^2 109 us at 128 columns against 120 at 64, 8192^2 1.55
// ms against 1.64, but 1024^2 46 us against 40; FP32 8192^2 0.59 ms at 256
// against 0.64 at 128 and 0.67 at 64, but 2048^2 51 us against 45 at 64).  The rates
// are what wide windows gain beyond their smaller halo.
PairShape pick_pair_shape(int elem, const GridSize *g, size_t n, int only, int cap) {
  // one grid: every height; several: enough of them to meet a round closely
  static const int few[] = {2,  3,  4,  5,  6,  7,  8,  10, 12,  14,  16,  18,  20, 24,
                            28, 32, 37, 42, 48, 56, 64, 72, 80,  96,  112, 128, 144, 160};
  PairShape best{only ? only : 64, 2};
  double best_cost = 1e300;
  for (int w : {64, 128, 256}) {
    const int cols = pair_cols(elem, w), width = cols - 8;
    if (only ? w != only : cols != w) continue;
    const double rate = cols == 64 ? 1.0 : cols == 128 ? (elem == 8 ? 1.08 : 1.0) : 1.05;
    const long slots = pair_slots(elem, w);
    const int count = n == 1 ? 191 : (int)(sizeof few / sizeof *few);
    for (int k = 0; k < count; ++k) {
      const int s = n == 1 ? k + 2 : few[k];
      if (s > cap && k) break;
      long blocks = 0;
      int tall = 0;
      for (size_t i = 0; i < n; ++i) {
        blocks += (long)((g[i].nx + width - 1) / width) * ((g[i].ny + s - 1) / s);
        tall = std::max(tall, g[i].ny);
      }
      const long rounds = (blocks + slots - 1) / slots;
      const double cost = (double)rounds * (std::min(s, tall) + 8) * cols / rate;
      if (cost < best_cost * (1 - 1e-9)) {
        best_cost = cost;
        best = {w, s};
      }
      if (s >= tall) break;
    }
  }
  // Several FP32 grids that this puts into one round of 64-column workgroups: with
  // 75 registers three rounds are resident at once, and r of them last (1 + r) / 2 of
  // one (us a step at the rows of one round and at the rows taken here: 12 instances of
  // 300 to 600 17.8 at 48, 16.0 at 24; 16 of 96 to 500 10.4 at 20, 10.3 at 10; 25 of 128 to
  // 384 12.5 at 28, 12.0 at 14; 40 of 128 to 384 19.6 at 56, 16.0 at 24; 100 of 64 to
  // 200 14.9 at 37, about 13.4 at 16).
  if (n > 1 && elem == 4 && best.window == 64) {
    const long slots = pair_slots(elem, 64);
    double cost = 0;
    for (int k = (int)(sizeof few / sizeof *few) - 1; k >= 0; --k) {
      if (few[k] > best.seg || few[k] > cap) continue;
      long blocks = 0;
      for (size_t i = 0; i < n; ++i)
        blocks += (long)((g[i].nx + 55) / 56) * ((g[i].ny + few[k] - 1) / few[k]);
      const long rounds = (blocks + slots - 1) / slots;
      if (!cost && rounds != 1) break;
      if (rounds > 3) break;
      const double c = (few[k] + 8) * (1.0 + rounds) / 2;
      if (!cost || c < cost) {
        cost = c;
        best.seg = few[k];
      }
    }
  }
  best.seg = std::max(1, std::min(best.seg, cap));
  return best;
}

// One 16-byte vector per lane, one pass: the fastest copy shape measured on
// MI355X (about 6.2 TB/s for 4 GiB), against ~4.7 TB/s for grid-stride loops.
typedef unsigned v4u __attribute__((ext_vector_type(4)));

__global__ void k_copy16(const v4u *__restrict__ src, v4u *__restrict__ dst, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = src[i];
}

int copy_probe(size_t bytes, int iters, double *ms) {
  require_device();
  if (bytes < 16 || iters < 1) return set_error(ERR_ARG, "copy_probe: bytes %zu iters %d", bytes, iters);
  void *a = nullptr, *b = nullptr;
  int rc = dev_alloc(&a, bytes, "copy_probe");
  if (!rc) rc = dev_alloc(&b, bytes, "copy_probe");
  if (rc) {
    dev_free(a);
    return rc;
  }
  (void)hipMemset(a, 1, bytes);
  const long n = (long)(bytes / 16);
  const unsigned blocks = (unsigned)((n + 255) / 256);
  hipEvent_t e0, e1;
  (void)hipEventCreate(&e0);
  (void)hipEventCreate(&e1);
  hipLaunchKernelGGL(k_copy16, dim3(blocks), dim3(256), 0, 0, (const v4u *)a, (v4u *)b, n);
  (void)hipEventRecord(e0, 0);
  for (int k = 0; k < iters; ++k)
    hipLaunchKernelGGL(k_copy16, dim3(blocks), dim3(256), 0, 0, (const v4u *)a, (v4u *)b, n);
  (void)hipEventRecord(e1, 0);
  hipError_t e = hipEventSynchronize(e1);
  float t = 0;
  (void)hipEventElapsedTime(&t, e0, e1);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  dev_free(a);
  dev_free(b);
  if (e != hipSuccess) return set_error(ERR_DEVICE, "copy_probe: %s", hipGetErrorString(e));
  *ms = t / iters;
  return OK;
}

}  // namespace le2d
