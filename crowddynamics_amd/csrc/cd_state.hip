// Agent state nodes and the herding neighbours on the device, so that the
// full logic tree keeps its host synchronisation off the step:
//
//   InsideDomain   (crowddynamics/simulation/logic.py:343-358): active =
//                  position inside the domain polygon; data['inactive'] +=
//                  the number of agents whose state changed.
//   TargetReached  (logic.py:361-387): reached_by |= position inside the
//                  target polygon; data['target_i'] = sum(reached_by).
//   herding        (core/steering/collective_motion.py:69-154,240-279): the
//                  size_nearest_other nearest agents within sight whose line
//                  of sight crosses no obstacle (find_nearest_neighbors over
//                  the block list at cell size = sight), and the herding
//                  direction of the followers from the neighbours heading
//                  away (herding_interaction).
//
// Point in polygon is the crossings test (E. Haines, "Point in Polygon
// Strategies", Graphics Gems IV, 1994) that matplotlib's Path.contains_points
// (called by the reference) implements: a ray toward +x from the point
// toggles the state at each edge whose endpoints straddle the point's y
// (y_k >= y on one side only), where the crossing lies at or beyond the
// point; the side is decided by the sign of a cross product, without a
// division, and the polygon closes from its last vertex back to its first.

#include "cd_common.h"

namespace {

__device__ __forceinline__ bool crossings_inside(double tx, double ty, const double2 *v, int V) {
  if (!(__builtin_isfinite(tx) && __builtin_isfinite(ty)) || V < 1) return false;
  bool inside = false;
  double x0 = v[0].x, y0 = v[0].y;
  bool f0 = y0 >= ty;
  for (int k = 1; k <= V; ++k) {
    const double2 w = v[k < V ? k : 0];
    const bool f1 = w.y >= ty;
    if (f0 != f1) {
      if (((w.y - ty) * (x0 - w.x) >= (w.x - tx) * (y0 - w.y)) == f1) inside = !inside;
    }
    f0 = f1;
    x0 = w.x;
    y0 = w.y;
  }
  return inside;
}

__global__ void __launch_bounds__(256) k_inside_domain(const double2 *pos, int n,
                                                       const double2 *v, int V,
                                                       uint8_t *active,
                                                       unsigned long long *changed) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  bool ch = false;
  if (i < n) {
    const double2 p = pos[i];
    const uint8_t now = crossings_inside(p.x, p.y, v, V) ? 1 : 0;
    ch = (active[i] != 0) != (now != 0);
    active[i] = now;
  }
  const unsigned long long b = __ballot(ch);
  if ((threadIdx.x & 63) == 0 && b) atomicAdd(changed, (unsigned long long)__popcll(b));
}

__global__ void k_zero_u64(unsigned long long *x) { *x = 0ull; }

__global__ void __launch_bounds__(256) k_target_reached(const double2 *pos, int n,
                                                        const double2 *v, int V,
                                                        uint8_t *reached,
                                                        unsigned long long *count) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  bool r = false;
  if (i < n) {
    const double2 p = pos[i];
    r = reached[i] != 0 || crossings_inside(p.x, p.y, v, V);
    reached[i] = r ? 1 : 0;
  }
  const unsigned long long b = __ballot(r);
  if ((threadIdx.x & 63) == 0 && b) atomicAdd(count, (unsigned long long)__popcll(b));
}

// line_intersect (core/geom2D.py:38-59): segments x0-x1 and y0-y1 cross
// (parallel segments do not).
__device__ __forceinline__ bool line_intersect(double2 x0, double2 x1, double2 y0, double2 y1) {
  const double ux = x1.x - x0.x, uy = x1.y - x0.y;
  const double vx = y1.x - y0.x, vy = y1.y - y0.y;
  const double bx = y0.x - x0.x, by = y0.y - x0.y;
  const double d = ux * vy - uy * vx;
  if (d == 0.0) return false;
  const double t0 = bx * vy - by * vx;
  const double t1 = bx * uy - by * ux;
  const double a = t0 / d, c = t1 / d;
  return 0.0 <= a && a <= 1.0 && 0.0 <= c && c <= 1.0;
}

// The same answer with the divisions only where they can matter: a or c
// outside [-2, 2] is outside [0, 1] however the quotient is rounded.
__device__ __forceinline__ bool line_blocks(double2 x0, double2 x1, double4 s) {
  const double ux = x1.x - x0.x, uy = x1.y - x0.y;
  const double vx = s.z - s.x, vy = s.w - s.y;
  const double bx = s.x - x0.x, by = s.y - x0.y;
  const double d2 = 2.0 * fabs(ux * vy - uy * vx);
  if (fabs(bx * vy - by * vx) > d2 || fabs(bx * uy - by * ux) > d2) return false;
  return line_intersect(x0, x1, make_double2(s.x, s.y), make_double2(s.z, s.w));
}

constexpr int kMaxNearest = 16;
constexpr int kNearLanes = 16;   // lanes per agent
constexpr int kNearGroups = 256 / kNearLanes;
constexpr int kNearList = 128;   // candidates in sight an agent's list holds
constexpr int kNearQueue = kNearList / kNearLanes;  // or those a lane holds of its own

// (l, j) before (m, k): ascending distance, ties to the smaller index.
__device__ __forceinline__ bool nearer(double l, int j, double m, int k) {
  return l < m || (l == m && j < k);
}

// x^2 times 1 +- kGate, which decides against another square as the lengths
// do; `off` where x^2 may lose bits to the subnormals.
__device__ __forceinline__ double gate2(double x, double side, double off) {
  return x > 0x1p-480 ? (x * x) * (1.0 + side * kGate) : off;
}

// The k nearest neighbours of an agent within sight (strictly closer than
// sight) whose line of sight crosses no segment, over the 3 x 3 cells of
// the block list (cells of side sight); ascending distance, ties to the
// smaller index, missing slots -1.
//
// 16 lanes serve an agent.  They first list the candidates in sight in LDS
// (a row's three cells are one range of the block list; a ballot gives each
// lane its place), then take the nearest one left, round by round: a
// butterfly finds it, and the lanes share the segments that could hide it.
// The order (distance, index) is total, so this is the list that inserting
// the visible candidates one by one builds; only the candidates that would
// enter it are tested against the segments.
//
// Where an agent has more candidates in sight than the list holds, its place
// is shared out: a lane keeps the nearest eight of its own share, in order,
// and a round's butterfly takes the lanes' first ones.  When a lane that met
// more than eight has given all of them away, the lanes walk the cells again
// from the last candidate taken.  (Walking them in every round, 4000 agents
// with 1250 in sight, nearly all hidden, took 49 ms a call and 20000 that see
// 630 took 5.0; now 2.8 and 0.51.  One thread per agent that met each
// candidate once took 43 and 18.  The eights in registers for every agent are
// faster still there, 0.37, but take 92 registers instead of 70: 20000 agents
// with 28 in sight 107 us instead of 99.)
//
// Bound by the latency of its rounds: with one thread per agent, each
// walking 80 candidates and testing all segments with two divisions, the
// lists indexed in scratch memory, 20000 agents at 1 / m^2 with 44 segments
// took 1502 us; this takes 37 us.
__global__ void __launch_bounds__(256) k_nearest(const double2 *pos, int n, double sight, int K,
                                                 const double4 *segs, int W, Work Wk,
                                                 const ScnState *ss, int64_t *nbr) {
  __shared__ double s_l[kNearGroups][kNearList];
  __shared__ int s_j[kNearGroups][kNearList];
  const int g = threadIdx.x / kNearLanes, q = threadIdx.x % kNearLanes;
  const int shift = (threadIdx.x & 63) & ~(kNearLanes - 1);  // the group's lanes in the wave
  const int i = blockIdx.x * kNearGroups + g;
  const bool have = i < n;
  const bool valid = have && ss->valid;
  const int c = valid ? Wk.cell_of[i] : -1;
  const double2 pi = have ? pos[i] : make_double2(0.0, 0.0);
  int row0[3] = {0, 0, 0}, row1[3] = {0, 0, 0};
  if (c >= 0) {
    const int nx = ss->nx, ny = ss->ny;
    const int lx = c / ny, ly = c - lx * ny;
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const int ox = lx + r - 1;
      if (ox < 0 || ox >= nx) continue;
      row0[r] = Wk.offset[ox * ny + max(ly - 1, 0)];
      row1[r] = Wk.offset[ox * ny + min(ly + 1, ny - 1) + 1];
    }
  }
  const double far2 = gate2(sight, 1.0, __builtin_inf());  // the length is not below sight
  int cnt = 0;  // the same in the group's lanes
  for (int r = 0; r < 3; ++r) {
    for (int e0 = row0[r]; e0 < row1[r]; e0 += kNearLanes) {
      const int e = e0 + q;
      int j = -1;
      double l = 0.0;
      if (e < row1[r]) {
        j = Wk.pidx[e];
        const double2 pj = pos[j];
        const double x = pi.x - pj.x, y = pi.y - pj.y;
        if (j == i || x * x + y * y > far2) {
          j = -1;
        } else {
          l = hypot_ref(x, y);
          if (!(l < sight)) j = -1;
        }
      }
      const unsigned m = (unsigned)(__ballot(j >= 0) >> shift) & ((1u << kNearLanes) - 1u);
      const int at = cnt + __popc(m & ((1u << q) - 1u));
      if (j >= 0 && at < kNearList) {
        s_l[g][at] = l;
        s_j[g][at] = j;
      }
      cnt += __popc(m);
    }
  }
  __syncthreads();
  const bool listed = cnt <= kNearList;
  int head = 0, held = 0;  // the lane's own: given away, kept
  bool more = true;        // others of its share lie behind them (or it has not looked yet)
  double last_l = -1.0;
  int last_j = -1;
  int out = -1;  // lane k: the k-th neighbour
  for (int k = 0, round = 0; k < K && round < cnt; ++round) {
    // the nearest candidate after (last_l, last_j)
    double bl = __builtin_inf();
    int bj = 0x7fffffff;
    if (listed) {
      for (int t = q; t < cnt; t += kNearLanes) {
        const double l = s_l[g][t];
        const int j = s_j[g][t];
        if (nearer(last_l, last_j, l, j) && nearer(l, j, bl, bj)) {
          bl = l;
          bj = j;
        }
      }
    } else {
      double *own_l = &s_l[g][q];  // the t-th at t kNearLanes
      int *own_j = &s_j[g][q];
      if (((__ballot(more && head == held) >> shift) & ((1ull << kNearLanes) - 1ull)) != 0ull) {
        const double near2 = gate2(last_l, -1.0, 0.0);
        double hold2 = __builtin_inf();  // farther is behind all eight
        head = held = 0;
        more = false;
        for (int r = 0; r < 3; ++r)
          for (int e = row0[r] + q; e < row1[r]; e += kNearLanes) {
            const int j = Wk.pidx[e];
            const double2 pj = pos[j];
            const double x = pi.x - pj.x, y = pi.y - pj.y;
            const double d2 = x * x + y * y;
            if (j == i || d2 > far2 || d2 < near2) continue;
            if (d2 > hold2) {
              more = true;
              continue;
            }
            const double l = hypot_ref(x, y);
            if (!(l < sight) || !nearer(last_l, last_j, l, j)) continue;
            int t = held;
            if (held < kNearQueue) {
              ++held;
            } else {
              more = true;
              t = kNearQueue - 1;
              if (!nearer(l, j, own_l[t * kNearLanes], own_j[t * kNearLanes])) continue;
            }
            for (; t > 0; --t) {
              const double pl = own_l[(t - 1) * kNearLanes];
              const int pk = own_j[(t - 1) * kNearLanes];
              if (!nearer(l, j, pl, pk)) break;
              own_l[t * kNearLanes] = pl;
              own_j[t * kNearLanes] = pk;
            }
            own_l[t * kNearLanes] = l;
            own_j[t * kNearLanes] = j;
            if (held == kNearQueue)
              hold2 = gate2(own_l[(kNearQueue - 1) * kNearLanes], 1.0, __builtin_inf());
          }
      }
      if (head < held) {
        bl = own_l[head * kNearLanes];
        bj = own_j[head * kNearLanes];
      }
    }
    const int first = bj;
#pragma unroll
    for (int o = 1; o < kNearLanes; o <<= 1) {
      const double l = __shfl_xor(bl, o, 64);
      const int j = __shfl_xor(bj, o, 64);
      if (nearer(l, j, bl, bj)) {
        bl = l;
        bj = j;
      }
    }
    if (bj == first) ++head;
    last_l = bl;
    last_j = bj;
    const double2 pj = pos[bj];
    bool hidden = false;
    for (int w = q; w < W && !hidden; w += kNearLanes) hidden = line_blocks(pi, pj, segs[w]);
    const bool any = ((__ballot(hidden) >> shift) & ((1ull << kNearLanes) - 1ull)) != 0ull;
    if (!any) {
      if (q == k) out = bj;
      ++k;
    }
  }
  if (have && q < K) nbr[(int64_t)i * K + q] = out;
}

__device__ __forceinline__ double2 normalize2(double2 v) {
  const double l = hypot_ref(v.x, v.y);
  return l != 0.0 ? make_double2(v.x / l, v.y / l) : v;
}

// herding_relationship (collective_motion.py:26-58), its first result: j
// is "heading away" from i unless cos(phi) < c_j < 1, c_j = -e_ij . v_j/|v_j|
// (both velocities non-zero), e_ij the unit vector from i to j.
__device__ __forceinline__ bool heading_away(double2 x1, double2 x2, double2 v1, double2 v2,
                                             double cos_phi) {
  if (hypot_ref(v1.x, v1.y) == 0.0 || hypot_ref(v2.x, v2.y) == 0.0) return false;
  const double2 e = normalize2(make_double2(x2.x - x1.x, x2.y - x1.y));
  const double2 n2 = normalize2(v2);
  const double cj = -(e.x * n2.x + e.y * n2.y);
  return !(cos_phi < cj && cj < 1.0);
}

// herding_interaction (collective_motion.py:110-154) of the followers over
// their neighbour lists (nearest first).  Lane k of an agent's 16 tests
// neighbour k; the sums are then taken in the list's order from the lanes.
// Bound by the dependent loads and lengths of one neighbour (one thread per
// agent walked K of them: 15 us for 20000 agents and K = 8).
__global__ void __launch_bounds__(256) k_herding(const double2 *pos, const double2 *vel, int n,
                                                 const uint8_t *is_follower,
                                                 const int64_t *nbr, int K,
                                                 double weight_position, double cos_phi,
                                                 double2 *dir, uint8_t *has) {
  static_assert(kMaxNearest <= kNearLanes, "a lane per neighbour");
  const int q = threadIdx.x % kNearLanes;
  const int shift = (threadIdx.x & 63) & ~(kNearLanes - 1);
  const int i = blockIdx.x * kNearGroups + threadIdx.x / kNearLanes;
  const bool follows = i < n && is_follower[i];
  double2 xi = make_double2(0.0, 0.0), xj = xi, vj = xi;
  bool away = false;
  if (follows) {
    const double2 vi = vel[i];
    xi = pos[i];
    const int64_t j = q < K ? nbr[(int64_t)i * K + q] : -1;
    if (j >= 0) {
      xj = pos[j];
      vj = vel[j];
      away = heading_away(xi, xj, vi, vj, cos_phi);
    }
  }
  const unsigned m = (unsigned)(__ballot(away) >> shift) & ((1u << kNearLanes) - 1u);
  double mpx = 0.0, mpy = 0.0, mvx = 0.0, mvy = 0.0;
  for (int k = 0; k < K; ++k) {
    const double px = __shfl(xj.x, shift + k, 64), py = __shfl(xj.y, shift + k, 64);
    const double vx = __shfl(vj.x, shift + k, 64), vy = __shfl(vj.y, shift + k, 64);
    if (m >> k & 1u) {
      mpx += px;
      mpy += py;
      mvx += vx;
      mvy += vy;
    }
  }
  if (i >= n || q != 0) return;
  double2 d = make_double2(0.0, 0.0);
  const int num = __popc(m);
  if (num > 0) {
    const double2 e0 = normalize2(make_double2(mpx / num - xi.x, mpy / num - xi.y));
    const double2 e1 = normalize2(make_double2(mvx, mvy));
    // weighted_average (core/vector2D.py:206-232), then normalize
    d = normalize2(make_double2(weight_position * e0.x + (1.0 - weight_position) * e1.x,
                                weight_position * e0.y + (1.0 - weight_position) * e1.y));
  }
  dir[i] = d;
  has[i] = num > 0 ? 1 : 0;
}

}  // namespace

extern "C" {

int cd_inside_domain(const double *pos, int64_t n, const double *vertices, int64_t n_vertices,
                     uint8_t *active, uint64_t *inactive, cd_stream_t stream) {
  if (n < 0 || n > 0x7fffffff || n_vertices < 0 || n_vertices > (1 << 20) || !inactive ||
      (n > 0 && (!pos || !active)) || (n_vertices > 0 && !vertices))
    return CD_ERR_ARG;
  if (n == 0) return CD_OK;
  hipLaunchKernelGGL(k_inside_domain, dim3(grid_for(n, kBS)), dim3(kBS), 0, (hipStream_t)stream,
                     (const double2 *)pos, (int)n, (const double2 *)vertices, (int)n_vertices,
                     active, (unsigned long long *)inactive);
  return check_launch();
}

int cd_target_reached(const double *pos, int64_t n, const double *vertices, int64_t n_vertices,
                      uint8_t *reached_by, uint64_t *count, cd_stream_t stream) {
  if (n < 0 || n > 0x7fffffff || n_vertices < 0 || n_vertices > (1 << 20) || !count ||
      (n > 0 && (!pos || !reached_by)) || (n_vertices > 0 && !vertices))
    return CD_ERR_ARG;
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(k_zero_u64, dim3(1), dim3(1), 0, s, (unsigned long long *)count);
  if (n > 0)
    hipLaunchKernelGGL(k_target_reached, dim3(grid_for(n, kBS)), dim3(kBS), 0, s,
                       (const double2 *)pos, (int)n, (const double2 *)vertices, (int)n_vertices,
                       reached_by, (unsigned long long *)count);
  return check_launch();
}

int cd_nearest_neighbors(const cd_agents_t *a, double sight, int32_t k, const double *segments,
                         int64_t n_segments, int64_t *neighbors, const cd_workspace_t *w,
                         cd_stream_t stream) {
  int rc = check_agents(a);
  if (rc) return rc;
  if (!(sight > 0.0) || k < 1 || k > kMaxNearest || n_segments < 0 || n_segments > 0x7fffffff ||
      (n_segments > 0 && !segments) || (a->n > 0 && !neighbors))
    return CD_ERR_ARG;
  if ((rc = check_ws(a, w))) return rc;
  if (a->n == 0) return CD_OK;
  // the block list at cell size = sight (collective_motion.py:250-257)
  if ((rc = cd_add_to_cells(a, sight, w, stream))) return rc;
  const Work W = carve(w);
  const Layout L = make_layout(w);
  hipLaunchKernelGGL(k_nearest, dim3(grid_for(a->n, kNearGroups)), dim3(256), 0, (hipStream_t)stream,
                     (const double2 *)a->position, (int)a->n, sight, (int)k,
                     (const double4 *)segments, (int)n_segments, W,
                     (const ScnState *)((char *)w->ptr + L.scn_state), neighbors);
  return check_launch();
}

int cd_herding_interaction(const double *pos, const double *vel, int64_t n,
                           const uint8_t *is_follower, const int64_t *neighbors, int32_t k,
                           double weight_position, double cos_phi, double *direction,
                           uint8_t *has_direction, cd_stream_t stream) {
  if (n < 0 || n > 0x7fffffff || k < 1 || k > kMaxNearest ||
      (n > 0 && (!pos || !vel || !is_follower || !neighbors || !direction || !has_direction)))
    return CD_ERR_ARG;
  if (n == 0) return CD_OK;
  hipLaunchKernelGGL(k_herding, dim3(grid_for(n, kNearGroups)), dim3(256), 0, (hipStream_t)stream,
                     (const double2 *)pos, (const double2 *)vel, (int)n, is_follower, neighbors,
                     (int)k, weight_position, cos_phi, (double2 *)direction, has_direction);
  return check_launch();
}

}  // extern "C"
