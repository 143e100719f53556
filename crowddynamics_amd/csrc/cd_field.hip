// Navigation field construction on the device: the distance map, direction
// map and obstacle blending of crowddynamics' quickest-path navigation
// (crowddynamics/core/steering/quickest_path.py:54-197,
// core/steering/obstacle_handling.py:15-74, cached per target by
// simulation/field.py:131-164).  The reference solves the Eikonal equation
// with scikit-fmm 0.0.9 (distance(phi, dx)) on the host; here it runs on the
// node grid in HBM.
//
// Distance map.  The nodes bordering the zero contour of phi are frozen at
// scikit-fmm's linear-interpolation distance (d_k = dx phi_i / (phi_i -
// phi_j) at the nearest crossing along axis k, combined as
// 1 / sqrt(sum 1 / d_k^2)); every other unmasked node converges to the
// fixed point of the first-order upwind update
//   u = a + dx                                  if b - a >= dx
//   u = (a + b + sqrt(2 dx^2 - (a - b)^2)) / 2   otherwise,
// a <= b the smaller neighbour values along the two axes.  That is the
// solution the fast marching method computes (the CPU oracle marches it in
// order of distance); on the GPU it is reached by relaxation: a workgroup
// takes a 32 x 32 tile with a one-node halo into LDS and sweeps it in
// red-black order until the tile stops changing, and the launches repeat
// until no tile changes.  A tile whose border changed marks the neighbours
// that read it; the next launch visits the marked tiles only.  Values only
// decrease, so every node's final value is the fixed point whatever the
// order of updates.
//
// Direction map: np.gradient (central differences inside, one-sided at the
// edges), normalised with the reference library's hypot; zero length gives
// NaN, and NaN (masked) inputs propagate.  Obstacle blending: within radius
// of the obstacles the target direction is mixed with the direction away
// from them with weight strength^(x / radius), then every node is
// normalised.  Missing directions in the buffer around obstacles take the
// direction of the nearest node that has one (quickest_path.py:152-166).

#include "cd_common.h"

namespace {

constexpr int kFT = 32;                // tile side in nodes
constexpr int kFH = kFT + 2;           // with the halo
constexpr int kFThreads = 512;         // one node of each colour per thread
constexpr int kFSweeps = 4;            // red-black sweeps between two barriers
constexpr int kFRounds = 24;           // rounds of such sweeps per tile visit (bounded)
static_assert(2 * kFThreads == kFT * kFT, "a thread relaxes two nodes of the tile");

// Bookkeeping of the relaxation in the work buffer: three sets of tile
// marks (pass p visits the tiles of set p % 3, marks set p + 1 and clears
// set p + 2), then whether each set holds a mark.
struct FieldMarks {
  int *dirty;  // [3][tiles]
  int *live;   // [3]
  int tiles;
};
inline int64_t field_tiles(int64_t rows, int64_t cols) {
  return ((rows + kFT - 1) / kFT) * ((cols + kFT - 1) / kFT);
}

enum : uint8_t { F_FREE = 0, F_FROZEN = 2, F_MASKED = 3 };

// Minimum and maximum of values that are never NaN.  (The library's take a
// canonicalising instruction for each operand, on the relaxation's chain.)
__device__ __forceinline__ double min_num(double a, double b) {
  double r;
  asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double max_num(double a, double b) {
  double r;
  asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// The square root of x in [2^-760, 2^1000]: the hardware's reciprocal root
// refined by Goldschmidt's iteration and two residual corrections, the steps
// of LLVM's published lowering of the fp64 square root for these targets, here
// without the scaling that it adds for the rest of the range.  Equal to sqrt,
// bit for bit, on 1.7e10 inputs on the device: random ones over the range and
// over one octave, and the neighbours of squares and of the squares of
// midpoints between two doubles.
__device__ __forceinline__ double sqrt_mid(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  const double d0 = __builtin_fma(-g, g, x);
  h = __builtin_fma(h, r, h);
  g = __builtin_fma(d0, h, g);
  const double d1 = __builtin_fma(-g, g, x);
  return __builtin_fma(d1, h, g);
}

// The update from the smaller neighbour values a <= b along the two axes
// (a finite), h2 = 2 h^2.
template <bool MID>
__device__ __forceinline__ double eik_update(double a, double b, double h, double h2) {
  const double d = b - a;
  const double x = h2 - d * d;
  const double two = (a + b + (MID ? sqrt_mid(x) : sqrt(x))) / 2.0;
  return d >= h ? a + h : two;  // (b infinite: d is)
}

// Frozen nodes (on or next to the contour), free nodes at +inf, masked
// nodes excluded.
__global__ void __launch_bounds__(256) k_field_init(const double *phi, const uint8_t *mask,
                                                    int rows, int cols, double dx, double *u,
                                                    uint8_t *state, FieldMarks M) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k < M.tiles) {  // the first pass visits every tile (fewer tiles than nodes)
    M.dirty[k] = 1;
    M.dirty[M.tiles + k] = 0;
  }
  if (k < 2) M.live[k] = k == 0 ? 1 : 0;
  if (k >= (int64_t)rows * cols) return;
  const int r = (int)(k / cols), c = (int)(k - (int64_t)r * cols);
  if (mask && mask[k]) {
    u[k] = __builtin_inf();
    state[k] = F_MASKED;
    return;
  }
  const double p = phi[k];
  if (p == 0.0) {
    u[k] = 0.0;
    state[k] = F_FROZEN;
    return;
  }
  double ld[2] = {0.0, 0.0};
  bool borders = false;
#pragma unroll
  for (int dim = 0; dim < 2; ++dim) {
#pragma unroll
    for (int s = -1; s <= 1; s += 2) {
      const int rr = dim ? r + s : r, cc = dim ? c : c + s;
      if (rr < 0 || rr >= rows || cc < 0 || cc >= cols) continue;
      const int64_t j = (int64_t)rr * cols + cc;
      if (mask && mask[j]) continue;
      const double q = phi[j];
      if (!(p * q < 0.0)) continue;
      borders = true;
      const double d = dx * p / (p - q);
      if (ld[dim] == 0.0 || ld[dim] > d) ld[dim] = d;
    }
  }
  if (!borders) {
    u[k] = __builtin_inf();
    state[k] = F_FREE;
    return;
  }
  double dsum = 0.0;
#pragma unroll
  for (int dim = 0; dim < 2; ++dim)
    if (ld[dim] > 0.0) dsum += 1.0 / ld[dim] / ld[dim];
  u[k] = sqrt(1.0 / dsum);
  state[k] = F_FROZEN;
}

// Pass `pass` visits the marked tiles: load the tile and its halo, relax
// the free nodes in red-black order until none changes (at most kFRounds
// rounds), store what changed, and mark the neighbours that read a changed
// border (or the tile itself, when the rounds ran out).
//
// Bound by the front's serial chain: a sweep moves it two nodes, and half a
// sweep is one LDS round trip and one square root.  Each thread owns one node
// of each colour (with four nodes per thread, half of them of the wrong colour,
// the lanes idled through the other half); a node whose neighbours' minima are
// those of its last update skips the update; and the waves meet at a barrier
// only every fourth sweep.  Between barriers a wave reads its neighbours' rows
// as they are at that moment: values only decrease and are stored whole, so an
// old value is one that a later sweep replaces, and a round in which no thread
// of the block changed a node checked every node against final values.
//
// Two maps, fill and blending of a 1001 x 501 grid with 24 obstacles, host
// work included, each step against the one before it on one card: all tiles
// visited in every pass, four barriers a sweep and a look after each pass 5.9
// ms, marked tiles in batches 1.55 (one, two, four and eight sweeps a barrier
// 1.59, 1.59, 1.54 and 1.61); both branches of the update selected instead of
// taken, minima without canonicalising, a square root without scaling and the
// tile read together with its mark 1.65 to 1.36.  From there shorter visits of
// 5 rounds took 15 % more, tiles of 64 x 32 nodes 32 %, of 16 x 16 28 %, the
// colours in arrays of their own 4 %, skipping waves with nothing new nearby
// 17 %.  Reading a tile before its mark is known streams the map through every
// pass, also for tiles that leave at once: 4001 x 2001 nodes take 4.7 ms a map
// (15.5 with every tile swept in every pass).
template <bool MID>
__global__ void __launch_bounds__(kFThreads) k_field_relax(int rows, int cols, double dx,
                                                           double *u, const uint8_t *state,
                                                           FieldMarks M, int pass) {
  __shared__ double su[kFH * kFH];
  __shared__ int s_change[3];
  const int tile = blockIdx.y * gridDim.x + blockIdx.x;
  const int tid = threadIdx.x;
  const int now = pass % 3, next = (pass + 1) % 3, after = (pass + 2) % 3;
  if (tid == 0) {
    M.dirty[after * M.tiles + tile] = 0;
    if (tile == 0) M.live[after] = 0;
  }
  // the mark, the tile and its nodes' states are read together
  const int marked = M.dirty[now * M.tiles + tile];
  const int r0 = blockIdx.y * kFT, c0 = blockIdx.x * kFT;
  constexpr int kLoads = (kFH * kFH + kFThreads - 1) / kFThreads;
  double v[kLoads];
#pragma unroll
  for (int k = 0; k < kLoads; ++k) {
    const int idx = tid + k * kFThreads;
    const int rr = r0 - 1 + idx / kFH, cc = c0 - 1 + idx % kFH;
    v[k] = __builtin_inf();
    if (idx < kFH * kFH && rr >= 0 && rr < rows && cc >= 0 && cc < cols)
      v[k] = u[(int64_t)rr * cols + cc];
  }
  const int lr = tid / (kFT / 2);
  int lc[2];
  bool free_[2];
  int64_t node[2];
#pragma unroll
  for (int colour = 0; colour < 2; ++colour) {
    lc[colour] = 2 * (tid % (kFT / 2)) + ((lr + colour) & 1);
    const int rr = r0 + lr, cc = c0 + lc[colour];
    node[colour] = (int64_t)rr * cols + cc;
    free_[colour] = rr < rows && cc < cols && state[node[colour]] == F_FREE;
  }
  if (!marked) return;  // the same for the whole block
#pragma unroll
  for (int k = 0; k < kLoads; ++k)
    if (tid + k * kFThreads < kFH * kFH) su[tid + k * kFThreads] = v[k];
  if (tid < 3) s_change[tid] = 0;
  __syncthreads();
  double own[2], first[2], plo[2], phi[2];
#pragma unroll
  for (int colour = 0; colour < 2; ++colour) {
    own[colour] = first[colour] = su[(lr + 1) * kFH + lc[colour] + 1];
    plo[colour] = phi[colour] = -1.0;
  }
  auto at = [&](int idx) {
    return __hip_atomic_load(&su[idx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  const double h2 = 2.0 * dx * dx;
  bool more = true;
  for (int it = 0; it < kFRounds && more; ++it) {
    bool ch = false;
    for (int sweep = 0; sweep < kFSweeps; ++sweep) {
#pragma unroll
      for (int colour = 0; colour < 2; ++colour) {
        const int idx = (lr + 1) * kFH + lc[colour] + 1;
        if (free_[colour]) {
          const double a = min_num(at(idx - 1), at(idx + 1));
          const double b = min_num(at(idx - kFH), at(idx + kFH));
          const double lo = min_num(a, b), hi = max_num(a, b);
          if (lo < own[colour] && (lo != plo[colour] || hi != phi[colour])) {
            plo[colour] = lo;
            phi[colour] = hi;
            const double w = eik_update<MID>(lo, hi, dx, h2);
            if (w < own[colour]) {
              own[colour] = w;
              __hip_atomic_store(&su[idx], w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
              ch = true;
            }
          }
        }
      }
    }
    if (ch) s_change[it % 3] = 1;
    if (tid == 0) s_change[(it + 1) % 3] = 0;
    __syncthreads();
    more = s_change[it % 3] != 0;
  }
  bool mark[5] = {false, false, false, false, false};  // up, down, left, right, itself
#pragma unroll
  for (int colour = 0; colour < 2; ++colour) {
    if (own[colour] == first[colour]) continue;
    u[node[colour]] = own[colour];
    mark[0] = mark[0] || lr == 0;
    mark[1] = mark[1] || lr == kFT - 1;
    mark[2] = mark[2] || lc[colour] == 0;
    mark[3] = mark[3] || lc[colour] == kFT - 1;
  }
  mark[4] = more;
  const int gx = gridDim.x, gy = gridDim.y;
  int *dirty = M.dirty + next * M.tiles;
  bool any = false;
  auto set = [&](bool m, bool inside, int t) {
    if (m && inside) {
      dirty[t] = 1;
      any = true;
    }
  };
  set(mark[0], (int)blockIdx.y > 0, tile - gx);
  set(mark[1], (int)blockIdx.y + 1 < gy, tile + gx);
  set(mark[2], (int)blockIdx.x > 0, tile - 1);
  set(mark[3], (int)blockIdx.x + 1 < gx, tile + 1);
  set(mark[4], true, tile);
  if (any) M.live[next] = 1;
}

// Signed distance: negative where phi < 0; masked and unreached nodes NaN.
__global__ void __launch_bounds__(256) k_field_finish(const double *phi, int64_t n, double *u,
                                                      const uint8_t *state) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= n) return;
  const double v = u[k];
  if (state[k] == F_MASKED || __builtin_isinf(v))
    u[k] = __builtin_nan("");
  else
    u[k] = phi[k] < 0.0 ? -v : v;
}

__global__ void __launch_bounds__(256) k_direction_map(const double *d, int rows, int cols,
                                                       double *ex, double *ey) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= (int64_t)rows * cols) return;
  const int r = (int)(k / cols), c = (int)(k - (int64_t)r * cols);
  double gu, gv;  // along rows (y), along cols (x)
  if (rows < 2)
    gu = 0.0;
  else if (r == 0)
    gu = d[k + cols] - d[k];
  else if (r == rows - 1)
    gu = d[k] - d[k - cols];
  else
    gu = (d[k + cols] - d[k - cols]) / 2.0;
  if (cols < 2)
    gv = 0.0;
  else if (c == 0)
    gv = d[k + 1] - d[k];
  else if (c == cols - 1)
    gv = d[k] - d[k - 1];
  else
    gv = (d[k + 1] - d[k - 1]) / 2.0;
  double l = hypot_ref(gu, gv);
  if (l == 0.0) l = __builtin_nan("");
  ex[k] = gv / l;
  ey[k] = gu / l;
}

__global__ void __launch_bounds__(256) k_obstacle_blend(const double *dobs, const double *ox,
                                                        const double *oy, double *tx,
                                                        double *ty, int64_t n, double radius,
                                                        double strength) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= n) return;
  double x0 = tx[k], y0 = ty[k];
  const double x = -dobs[k];
  if (0.0 < x && x < radius) {
    const double p = pow(strength, x / radius);
    x0 = -p * ox[k] + (1.0 - p) * x0;
    y0 = -p * oy[k] + (1.0 - p) * y0;
  }
  const double l = hypot_ref(x0, y0);
  tx[k] = x0 / l;
  ty[k] = y0 / l;
}

// Missing directions (NaN) at nodes of `fill` take those of the nearest
// node with a direction within `reach` nodes (squared index distance, ties
// to the smaller row, then column); nodes with none in reach stay NaN.
// Reads (sx, sy), writes (dx_, dy_): a separate output, so the search sees
// only the original directions.
__global__ void __launch_bounds__(256) k_fill_nearest(const double *sx, const double *sy,
                                                      const uint8_t *fill, int rows, int cols,
                                                      int reach, double *dx_, double *dy_) {
  const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (k >= (int64_t)rows * cols) return;
  const double x0 = sx[k], y0 = sy[k];
  dx_[k] = x0;
  dy_[k] = y0;
  if (!fill[k] || !(__builtin_isnan(x0) || __builtin_isnan(y0))) return;
  const int r = (int)(k / cols), c = (int)(k - (int64_t)r * cols);
  // First the square of half-width kNear, then, unless the best node is nearer
  // than all outside it, the rest; of each the rows by growing distance and of
  // a row the part inside the grid and the best distance so far, four nodes at
  // a time so that their loads leave together.  Bound by those loads where no
  // direction is near: 1000^2 nodes with a hole of 980^2 and reach 6 take
  // 0.12 ms and with reach 100 15 ms (rings of growing width 0.13 and 24, every
  // node of the square in turn 0.12 and 19), 100 x 100 nodes with no direction
  // and reach 1000 0.70 ms (rings, beyond the grid too, 134; in turn 1.0).  The
  // grown obstacles of a 1001 x 501 grid take 17 us (rings 17; in turn 52).
  constexpr int kNear = 4;
  int best = 0x7fffffff;
  int64_t bj = -1;
  auto scan = [&](int dr, int lo, int hi) {  // columns lo to hi of row r + dr
    const int64_t row = (int64_t)(r + dr) * cols;
    for (int cc = lo; cc <= hi; cc += 4) {
      double v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = sx[row + min(cc + u, hi)];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t j = row + min(cc + u, hi);
        const int dc = min(cc + u, hi) - c, d2 = dr * dr + dc * dc;
        if (__builtin_isnan(v[u]) || d2 > best || (d2 == best && j >= bj)) continue;
        if (__builtin_isnan(sy[j])) continue;  // (row-major order among equals)
        best = d2;
        bj = j;
      }
    }
  };
  for (int h = min(kNear, reach), done = -1;; done = h, h = reach) {  // done: its half-width
    const int last = min(h, max(r, rows - 1 - r));
    for (int m = 0; m <= last && m * m <= best; ++m) {
      const int w = best == 0x7fffffff ? h : min(h, (int)sqrtf((float)(best - m * m)) + 1);
      const int c0 = max(c - w, 0), c1 = min(c + w, cols - 1);
      for (int dr = -m; dr <= m; dr += max(2 * m, 1)) {
        if (r + dr < 0 || r + dr >= rows) continue;
        scan(dr, c0, m <= done ? c - done - 1 : c1);
        if (m <= done) scan(dr, c + done + 1, c1);
      }
    }
    if (h == reach || best < (h + 1) * (h + 1)) break;
  }
  if (bj >= 0) {
    dx_[k] = sx[bj];
    dy_[k] = sy[bj];
  }
}

constexpr int64_t kMaxFieldNodes = (int64_t)1 << 30;

}  // namespace

extern "C" {

int64_t cd_field_work_bytes(int64_t rows, int64_t cols) {
  if (rows < 1 || cols < 1 || rows * cols > kMaxFieldNodes || rows > 0x7fffffff ||
      cols > 0x7fffffff)
    return CD_ERR_ARG;
  return align_up(rows * cols) + align_up(12 * field_tiles(rows, cols)) + 256;
}

int cd_distance_map(const double *phi, const uint8_t *mask, int64_t rows, int64_t cols,
                    double dx, double *out, void *work, int64_t work_bytes,
                    cd_stream_t stream) {
  const int64_t need = cd_field_work_bytes(rows, cols);
  if (need < 0 || !phi || !out || !work || !(dx > 0.0)) return CD_ERR_ARG;
  if (work_bytes < need) return CD_ERR_WORKSPACE;
  hipStream_t s = (hipStream_t)stream;
  const int64_t n = rows * cols;
  uint8_t *state = (uint8_t *)work;
  const dim3 tiles((unsigned)((cols + kFT - 1) / kFT), (unsigned)((rows + kFT - 1) / kFT));
  FieldMarks M;
  M.tiles = (int)field_tiles(rows, cols);
  M.dirty = (int *)((char *)work + align_up(n));
  M.live = (int *)((char *)M.dirty + align_up(12 * (int64_t)M.tiles));
  const unsigned nb = (unsigned)((n + 255) / 256);
  hipLaunchKernelGGL(k_field_init, dim3(nb), dim3(256), 0, s, phi, mask, (int)rows, (int)cols,
                     dx, out, state, M);
  int rc = check_launch();
  if (rc) return rc;
  // every pass settles at least the next node in order of distance
  const int64_t max_passes = n + 64;
  auto relax = (dx >= 0x1p-370 && dx <= 0x1p490) ? k_field_relax<true> : k_field_relax<false>;
  // Passes are sent in batches, with one look at the marks after each: a
  // look waits for the stream (about 40 us), a pass without marks takes 3 us.
  // An open domain takes about as many passes as the front crosses tiles,
  // half of tiles.x + tiles.y; what obstacles add comes in batches of eight, or
  // of fewer where there are few tiles: a lone tile is settled by its first
  // pass (12 x 7 nodes: 72 us with a look after each pass, 88 in eights, 37
  // so).
  int h_live = 1;
  const int64_t least = std::min<int64_t>(8, 2 * (int64_t)M.tiles - 1);
  int64_t batch = std::max(least, ((int64_t)tiles.x + tiles.y) / 2);
  for (int64_t pass = 0; pass < max_passes && h_live; batch = least) {
    const int64_t end = std::min(max_passes, pass + batch);
    for (; pass < end; ++pass)
      hipLaunchKernelGGL(relax, tiles, dim3(kFThreads), 0, s, (int)rows, (int)cols, dx, out,
                         (const uint8_t *)state, M, (int)(pass % 3));
    if ((rc = check_launch())) return rc;
    if (hipMemcpyAsync(&h_live, M.live + pass % 3, sizeof(int), hipMemcpyDeviceToHost, s) !=
            hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
      return CD_ERR_HIP;
  }
  if (h_live) return CD_ERR_HIP;  // not converged within the bound
  hipLaunchKernelGGL(k_field_finish, dim3(nb), dim3(256), 0, s, phi, n, out,
                     (const uint8_t *)state);
  return check_launch();
}

int cd_direction_map(const double *dmap, int64_t rows, int64_t cols, double *ex, double *ey,
                     cd_stream_t stream) {
  if (cd_field_work_bytes(rows, cols) < 0 || !dmap || !ex || !ey) return CD_ERR_ARG;
  const int64_t n = rows * cols;
  hipLaunchKernelGGL(k_direction_map, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, dmap, (int)rows, (int)cols, ex, ey);
  return check_launch();
}

int cd_obstacle_handling(const double *dobs, const double *ox, const double *oy, double *tx,
                         double *ty, int64_t n, double radius, double strength,
                         cd_stream_t stream) {
  if (n < 0 || n > kMaxFieldNodes || (n > 0 && (!dobs || !ox || !oy || !tx || !ty)) ||
      !(radius > 0.0))
    return CD_ERR_ARG;
  if (n == 0) return CD_OK;
  hipLaunchKernelGGL(k_obstacle_blend, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, dobs, ox, oy, tx, ty, n, radius, strength);
  return check_launch();
}

int cd_fill_missing(const double *sx, const double *sy, const uint8_t *fill, int64_t rows,
                    int64_t cols, int32_t reach, double *ex, double *ey, cd_stream_t stream) {
  if (cd_field_work_bytes(rows, cols) < 0 || !sx || !sy || !fill || !ex || !ey || reach < 0 ||
      reach > 1024 || ex == sx || ey == sy)
    return CD_ERR_ARG;
  const int64_t n = rows * cols;
  hipLaunchKernelGGL(k_fill_nearest, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, sx, sy, fill, (int)rows, (int)cols, (int)reach, ex, ey);
  return check_launch();
}

}  // extern "C"
