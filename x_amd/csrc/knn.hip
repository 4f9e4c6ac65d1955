// k-nearest-neighbour look-up of MotionPriorCMax's displacement table (atl/objectives/mpcm.py:30-42,56-78): for
// every plane p (batch x time bin) and query q (a look-up-table cell centre), the k nearest of the plane's n points
// (tile-trajectory positions).  The reference computes a dense (Q x n) distance matrix per plane (torch.cdist) and
// a top-k over it; here the points are binned once into a uniform grid of about one point per cell and every query
// searches rings of cells around its own cell, keeping a sorted top-k in registers, until no unvisited cell can
// hold a closer point.
//
// Order: squared distance (qx - px)^2 + (qy - py)^2 with each product and the sum rounded in fp32 (the file is built
// with -ffp-contract=off), ties by the lower point index; the indices are written in that order.  This is the
// exact-distance order of the reference's GPU path (pykeops argKmin on (x_i - y_j)^2); its CPU path (cdist's
// matrix-product form, then topk) selects the same set wherever the k-th and (k+1)-th distances are apart, and
// leaves the order of exact ties open.  Points whose distance is not finite are never selected (their slots,
// possible only if fewer than k finite points exist, hold -1).
#include "common.h"
#include "scan.h"
#include "../../include/atl_hip.h"

#include <cmath>

using namespace atlhip;

namespace {

constexpr int kKnnMaxK = 32;
constexpr int kGeomBlock = 1024;

// Grid of one plane (shared by all planes: the queries define it).  Cell (cx, cy) covers
// [ox + cx * csx, ox + (cx + 1) * csx) x [oy + cy * csy, ...); positions outside the grid are clamped into the border
// cells, whose extent is therefore unbounded on their outer sides.
struct KnnGeom {
  float ox, oy, csx, csy, icx, icy;
  int GX, GY;
};

struct KnnLayout {
  int64_t geom, cnt, start, part, pts, bytes;
};

inline int64_t align256(int64_t v) { return (v + 255) & ~int64_t(255); }

KnnLayout knn_layout(int64_t P, int64_t n) {
  const int64_t ncap = n + 1;                      // cells per plane, at most
  const int64_t ncell = P * ncap;
  KnnLayout L;
  int64_t off = 0;
  L.geom = off;  off += align256(sizeof(KnnGeom));
  L.cnt = off;   off += align256(ncell * 4);
  L.start = off; off += align256((ncell + 1) * 4);
  L.part = off;  off += align256((scan_tiles(ncell) + 1) * 4);
  L.pts = off;   off += align256(P * n * 16);
  L.bytes = off;
  return L;
}

__device__ __forceinline__ int cell_of(float p, float o, float ic, int G) {
  const float c = floorf((p - o) * ic);
  return (int)fminf(fmaxf(c, 0.f), (float)(G - 1));   // NaN -> 0
}

// The queries' bounding box, split into about n cells (at most n + 1) of aspect close to 1.
__global__ void __launch_bounds__(kGeomBlock) k_knn_geom(const float2* __restrict__ q, int64_t Q, int64_t n,
                                                         KnnGeom* __restrict__ geo) {
  __shared__ float red[4][kGeomBlock / kWave];
  float x0 = INFINITY, y0 = INFINITY, x1 = -INFINITY, y1 = -INFINITY;
  for (int64_t i = threadIdx.x; i < Q; i += kGeomBlock) {
    const float2 p = q[i];
    if (isfinite(p.x) && isfinite(p.y)) {
      x0 = fminf(x0, p.x); x1 = fmaxf(x1, p.x);
      y0 = fminf(y0, p.y); y1 = fmaxf(y1, p.y);
    }
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) {
    x0 = fminf(x0, __shfl_xor(x0, d, kWave)); x1 = fmaxf(x1, __shfl_xor(x1, d, kWave));
    y0 = fminf(y0, __shfl_xor(y0, d, kWave)); y1 = fmaxf(y1, __shfl_xor(y1, d, kWave));
  }
  const int w = threadIdx.x / kWave;
  if ((threadIdx.x & (kWave - 1)) == 0) { red[0][w] = x0; red[1][w] = x1; red[2][w] = y0; red[3][w] = y1; }
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int k = 1; k < kGeomBlock / kWave; ++k) {
    x0 = fminf(x0, red[0][k]); x1 = fmaxf(x1, red[1][k]); y0 = fminf(y0, red[2][k]); y1 = fmaxf(y1, red[3][k]);
  }
  if (!(x0 <= x1)) { x0 = 0.f; x1 = 0.f; }       // no finite query: any grid will do
  if (!(y0 <= y1)) { y0 = 0.f; y1 = 0.f; }
  const float w_ = fmaxf(x1 - x0, 1.f), h_ = fmaxf(y1 - y0, 1.f);
  const double ncap = (double)n + 1.0;
  const double cs = sqrt((double)w_ * (double)h_ / (double)(n > 0 ? n : 1));
  int GX = (int)fmin(fmax(ceil((double)w_ / cs), 1.0), ncap);
  int GY = (int)fmin(fmax(ceil((double)h_ / cs), 1.0), floor(ncap / GX));
  GY = GY < 1 ? 1 : GY;
  KnnGeom g;
  g.ox = x0; g.oy = y0;
  g.csx = w_ / (float)GX; g.csy = h_ / (float)GY;
  g.icx = (float)GX / w_; g.icy = (float)GY / h_;
  g.GX = GX; g.GY = GY;
  *geo = g;
}

__global__ void __launch_bounds__(kBlock) k_knn_zero(int* __restrict__ p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i < n) p[i] = 0;
}

// Point counts per cell (plane-major, ncap cells per plane); SCATTER: each point takes a slot of its cell (filled
// from the cell's end: the counts run back to zero) and writes (x, y, index) there.
template <bool SCATTER>
__global__ void __launch_bounds__(kBlock) k_knn_bin(const float2* __restrict__ pts, int64_t P, int64_t n,
                                                    const KnnGeom* __restrict__ geo, int* __restrict__ cnt,
                                                    const int* __restrict__ start, float4* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (i >= P * n) return;
  const KnnGeom g = *geo;
  const int64_t plane = i / n;
  const int j = (int)(i - plane * n);
  const float2 p = pts[i];
  const int64_t c = plane * (n + 1) + (int64_t)cell_of(p.y, g.oy, g.icy, g.GY) * g.GX + cell_of(p.x, g.ox, g.icx, g.GX);
  if (!SCATTER) {
    atomicAdd(cnt + c, 1);
  } else {
    const int slot = start[c] + atomicSub(cnt + c, 1) - 1;
    out[slot] = make_float4(p.x, p.y, __int_as_float(j), 0.f);
  }
}

// (d, j) before (D, J) in the output order
__device__ __forceinline__ bool before(float d, int j, float D, int J) { return d < D || (d == D && j < J); }

// One query per thread: rings of cells around its own cell, each ring's rows read as contiguous cell ranges; the
// search ends when the k-th best distance is below the squared distance to every unvisited cell (with a slack
// that covers the rounding of the binning), or when every cell has been visited.
template <int KC>
__global__ void __launch_bounds__(kBlock) k_knn_query(const float2* __restrict__ qs, int64_t Q, int64_t n, int k,
                                                      const KnnGeom* __restrict__ geo, const int* __restrict__ start,
                                                      const float4* __restrict__ pts, int64_t* __restrict__ out) {
  const int64_t plane = blockIdx.y;
  const int64_t qi = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (qi >= Q) return;
  const KnnGeom g = *geo;
  const float2 q = qs[qi];
  const int* __restrict__ cs = start + plane * (n + 1);
  const int qcx = cell_of(q.x, g.ox, g.icx, g.GX), qcy = cell_of(q.y, g.oy, g.icy, g.GY);
  float D[KC];
  int J[KC];
#pragma unroll
  for (int s = 0; s < KC; ++s) { D[s] = INFINITY; J[s] = 0x7fffffff; }
  float dk = INFINITY;                             // the k-th entry (slot k - 1)
  int jk = 0x7fffffff;
  // slack of the unvisited-cell bounds: a point can be binned one rounding away from its cell's edge
  const float slack = 1e-4f * (g.csx + g.csy) + 1e-5f * (fabsf(g.ox) + fabsf(g.oy) + fabsf(q.x) + fabsf(q.y));
  const int rmax = max(g.GX, g.GY);
  for (int r = 0; r <= rmax; ++r) {
    const int y0 = max(qcy - r, 0), y1 = min(qcy + r, g.GY - 1);
    for (int y = y0; y <= y1; ++y) {
      const bool edge_row = (y == qcy - r) || (y == qcy + r);
      // the ring's cells of row y: the whole span on its top and bottom rows, else its two end cells
      for (int part = 0; part < (edge_row ? 1 : 2); ++part) {
        int x0, x1;
        if (edge_row) { x0 = qcx - r; x1 = qcx + r; }
        else { x0 = part == 0 ? qcx - r : qcx + r; x1 = x0; }
        x0 = max(x0, 0); x1 = min(x1, g.GX - 1);
        if (x0 > x1) continue;
        const int b = cs[y * g.GX + x0], e = cs[y * g.GX + x1 + 1];
        for (int t = b; t < e; ++t) {
          const float4 p = pts[t];
          const float dx = q.x - p.x, dy = q.y - p.y;
          const float d = dx * dx + dy * dy;
          const int j = __float_as_int(p.z);
          if (!before(d, j, dk, jk)) continue;
          float cd = d;
          int cj = j;
#pragma unroll
          for (int s = 0; s < KC; ++s) {           // insertion: the array stays sorted by (d, j)
            const bool lt = before(cd, cj, D[s], J[s]);
            const float td = D[s];
            const int tj = J[s];
            D[s] = lt ? cd : td;
            J[s] = lt ? cj : tj;
            cd = lt ? td : cd;
            cj = lt ? tj : cj;
          }
          dk = D[0];
          jk = J[0];
#pragma unroll
          for (int s = 1; s < KC; ++s) {
            dk = s == k - 1 ? D[s] : dk;
            jk = s == k - 1 ? J[s] : jk;
          }
        }
      }
    }
    // distance from q to the nearest unvisited cell: beyond each side of the (2r + 1)^2 block that is not at the
    // grid's edge (border cells extend to infinity, so a block side at the edge leaves nothing beyond it)
    float lb = INFINITY;
    if (qcx - r > 0) lb = fminf(lb, q.x - (g.ox + (float)(qcx - r) * g.csx));
    if (qcx + r < g.GX - 1) lb = fminf(lb, (g.ox + (float)(qcx + r + 1) * g.csx) - q.x);
    if (qcy - r > 0) lb = fminf(lb, q.y - (g.oy + (float)(qcy - r) * g.csy));
    if (qcy + r < g.GY - 1) lb = fminf(lb, (g.oy + (float)(qcy + r + 1) * g.csy) - q.y);
    if (lb == INFINITY) break;                     // every cell visited
    lb = fmaxf(lb - slack, 0.f);
    if (dk < lb * lb) break;                       // finite and closer than anything unvisited
  }
  int64_t* o = out + (plane * Q + qi) * k;
#pragma unroll
  for (int s = 0; s < KC; ++s)
    if (s < k) o[s] = D[s] < INFINITY ? (int64_t)J[s] : (int64_t)-1;
}

// ------------------------------------------------------------------------------ the displacement table, fused
// table (P, ny * nx, 2): per lattice query and plane, the mean displacement of the plane's k nearest points, and its
// adjoint, without the indices (k_knn_query's order and ties, so the same set).  The mean needs the set and not its
// order: a query first brackets its k-th distance, counting its candidates under seven thresholds at a time (14
// instructions a candidate, nothing kept), then adds up the points under the bracket and picks the few inside it by
// (distance, index).  The sorted insertion of k_knn_query costs 350 instructions a candidate, and took 560 us for 15
// planes of 19200 points, k = 32; with the bracketing the whole forward takes 149 us on an even point set and 211 us
// where trajectories of up to 25 px leave parts of the sensor empty (picking the bracket's points one pass each
// instead of kPick a pass: 190 and 267 us).  One thread per query, a wave on an 8 x 8 patch,
// so that its lanes read the same cells.
//
// The adjoint gathers: a point takes the gradient of every query whose k-th (distance, index) it does not exceed, the
// same fp32 distance giving the same decision.  Queries stand in blocks of 4 x 4 with the largest k-th distance of
// each block, so that a point tests about ten blocks (47 to 61 us; 75 to 88 us with a gradient loaded per taken query; torch's
// scatter of 9.2M rows through atomics took 180 us, and the gather and mean forward another 130).
constexpr int kQB = 4;                           // queries per block side
constexpr int kQStep = 8;                        // candidates a query reads at once (2: 238, 4: 216, 8: 211 us)
constexpr int kPick = 4;                         // points picked from the bracket in one pass
constexpr int kPatch = 16;                       // queries per workgroup side: 4 waves of 8 x 8

struct LutLayout {
  int64_t cnt, pmax, start, part, xy, dv, id, kth, kid, bmax, bytes;   // cnt and pmax are cleared together
};

LutLayout lut_layout(int64_t P, int64_t n, int64_t nx, int64_t ny) {
  const int64_t ncell = P * (n + 1), nb = ((nx + kQB - 1) / kQB) * ((ny + kQB - 1) / kQB);
  LutLayout L;
  int64_t off = 0;
  L.cnt = off;   off += ncell * 4;
  L.pmax = off;  off = align256(off + P * 4);
  L.start = off; off += align256((ncell + 1) * 4);
  L.part = off;  off += align256((scan_tiles(ncell) + 1) * 4);
  L.xy = off;    off += align256(P * n * 8);
  L.dv = off;    off += align256(P * n * 8);
  L.id = off;    off += align256(P * n * 4);
  L.kth = off;   off += align256(P * nb * kQB * kQB * 4);
  L.kid = off;   off += align256(P * nb * kQB * kQB * 4);
  L.bmax = off;  off += align256(P * nb * 4);
  L.bytes = off;
  return L;
}

// k_knn_geom's grid for queries x0 + i * step, y0 + j * step: known on the host.
KnnGeom lattice_geom(float x0, float y0, float step, int64_t nx, int64_t ny, int64_t n) {
  const float w = fmaxf((float)(nx - 1) * step, 1.f), h = fmaxf((float)(ny - 1) * step, 1.f);
  const double ncap = (double)n + 1.0, cs = sqrt((double)w * (double)h / (double)n);
  KnnGeom g;
  g.GX = (int)fmin(fmax(ceil((double)w / cs), 1.0), ncap);
  g.GY = (int)fmin(fmax(ceil((double)h / cs), 1.0), floor(ncap / g.GX));
  g.GY = g.GY < 1 ? 1 : g.GY;
  g.ox = x0; g.oy = y0;
  g.csx = w / (float)g.GX; g.csy = h / (float)g.GY;
  g.icx = (float)g.GX / w; g.icy = (float)g.GY / h;
  return g;
}

// k_knn_bin for the points tr (planes / T, 1 + T, n, 2): plane p = (b, s) holds the positions at time s, row 0 of its
// batch those at the reference time, and a point's displacement is their difference.
template <bool SCATTER>
__global__ void __launch_bounds__(kBlock) k_lut_bin(const float2* __restrict__ tr, int T, int n, KnnGeom g,
                                                    int* __restrict__ cnt, const int* __restrict__ start,
                                                    float2* __restrict__ xy, float2* __restrict__ dv,
                                                    int* __restrict__ id) {
  const int j = blockIdx.x * kBlock + threadIdx.x;
  if (j >= n) return;
  const int plane = blockIdx.y, batch = plane / T;
  const float2 p = tr[((int64_t)plane + batch + 1) * n + j];
  const int64_t c = (int64_t)plane * (n + 1) + (int64_t)cell_of(p.y, g.oy, g.icy, g.GY) * g.GX + cell_of(p.x, g.ox, g.icx, g.GX);
  if (!SCATTER) {
    atomicAdd(cnt + c, 1);
  } else {
    const float2 r = tr[(int64_t)batch * (T + 1) * n + j];
    const int slot = start[c] + atomicSub(cnt + c, 1) - 1;
    xy[slot] = p;
    dv[slot] = make_float2(r.x - p.x, r.y - p.y);
    id[slot] = j;
  }
}

__device__ __forceinline__ uint64_t dist_key(float d, int j) {   // orders (d, j), d >= 0
  return ((uint64_t)__float_as_uint(d) << 32) | (uint32_t)j;
}

__global__ void __launch_bounds__(kBlock) k_lut_query(float x0, float y0, float step, int nx, int ny, int n, int k,
                                                      KnnGeom g, const int* __restrict__ start,
                                                      const float2* __restrict__ xy, const float2* __restrict__ dv,
                                                      const int* __restrict__ id, float2* __restrict__ table,
                                                      float* __restrict__ kth, int* __restrict__ kid,
                                                      float* __restrict__ bmax, unsigned* __restrict__ pmax) {
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
  const int npx = (nx + kPatch - 1) / kPatch;
  const int blk = lane >> 4, l = lane & 15;      // a 16-lane row of the wave is one block of 4 x 4 queries
  const int ix = (int)(blockIdx.x % npx) * kPatch + (wave & 1) * 8 + (blk & 1) * kQB + (l & 3);
  const int iy = (int)(blockIdx.x / npx) * kPatch + (wave >> 1) * 8 + (blk >> 1) * kQB + (l >> 2);
  const int plane = blockIdx.y;
  const bool live = ix < nx && iy < ny;
  const int* __restrict__ cs = start + (int64_t)plane * (n + 1);
  const float qx = (float)ix * step + x0, qy = (float)iy * step + y0;
  float dk = 0.f;                                // the k-th distance, its index, and whether others may share it
  int jk = 0;
  bool tie = false;
  if (live) {
    const int qcx = cell_of(qx, g.ox, g.icx, g.GX), qcy = cell_of(qy, g.oy, g.icy, g.GY);
    const float slack = 1e-4f * (g.csx + g.csy) + 1e-5f * (fabsf(g.ox) + fabsf(g.oy) + fabsf(qx) + fabsf(qy));
    // f(d, slot) over the points of a row range of cells, kQStep loads in flight
    auto row = [&](int b, int e, auto&& f) {
      for (int t = b; t < e; t += kQStep) {
        float2 p[kQStep];
#pragma unroll
        for (int u = 0; u < kQStep; ++u) p[u] = xy[(uint32_t)min(t + u, e - 1)];
#pragma unroll
        for (int u = 0; u < kQStep; ++u) {
          const float dx = qx - p[u].x, dy = qy - p[u].y;
          if (t + u < e) f(dx * dx + dy * dy, t + u);
        }
      }
    };
    // over every cell that can hold a point closer than sqrt(hi): a point can be binned one rounding away
    auto disc = [&](float hi, auto&& f) {
      const float rad = __builtin_amdgcn_sqrtf(hi) + slack;   // ~1 ulp: far inside the slack
      const int ya = cell_of(qy - rad, g.oy, g.icy, g.GY), yb = cell_of(qy + rad, g.oy, g.icy, g.GY);
      for (int y = ya; y <= yb; ++y) {
        const float lo = g.oy + (float)y * g.csy;
        const float off = fmaxf(fmaxf(lo - qy, qy - (lo + g.csy)) - slack, 0.f);
        const float hw = __builtin_amdgcn_sqrtf(fmaxf(rad * rad - off * off, 0.f)) + slack;
        const int xa = cell_of(qx - hw, g.ox, g.icx, g.GX), xb = cell_of(qx + hw, g.ox, g.icx, g.GX);
        row(cs[y * g.GX + xa], cs[y * g.GX + xb + 1], f);
      }
    };
    float th[7];
    int c[7];
    auto count = [&](float d, int) {
#pragma unroll
      for (int i = 0; i < 7; ++i) c[i] += d < th[i] ? 1 : 0;
    };
    // an upper bound of the k-th distance from the smallest block of cells around the query that shows one: the
    // thresholds lie around the distance at which the block's density gives k points, and out to the block's corner
    float hi = INFINITY, lo = 0.f;
    int chi = 0, clo = 0;                        // points under hi and under lo (chi: 0 until counted)
    int r = 0;
    while ((2 * r + 1) * (2 * r + 1) < k) ++r;
    for (;;) {
      const int xa = max(qcx - r, 0), xb = min(qcx + r, g.GX - 1), ya = max(qcy - r, 0), yb = min(qcy + r, g.GY - 1);
      int m = 0;
      for (int y = ya; y <= yb; ++y) m += cs[y * g.GX + xb + 1] - cs[y * g.GX + xa];
      if (m >= k) {
        const float area = (float)((xb - xa + 1) * (yb - ya + 1)) * g.csx * g.csy;
        const float e = area * (float)k / (3.14159265f * (float)m);
        const float ddx = fmaxf(qx - (g.ox + (float)xa * g.csx), g.ox + (float)(xb + 1) * g.csx - qx);
        const float ddy = fmaxf(qy - (g.oy + (float)ya * g.csy), g.oy + (float)(yb + 1) * g.csy - qy);
        const float far = fmaxf(ddx * ddx + ddy * ddy, 1.2f * e);   // the block's corner: all but points beyond the grid
        const float q = cbrtf(far / (1.15f * e));
        th[0] = 0.55f * e; th[1] = 0.8f * e; th[2] = 0.95f * e; th[3] = 1.15f * e; th[4] = th[3] * q; th[5] = th[4] * q;
        th[6] = far;
#pragma unroll
        for (int i = 0; i < 7; ++i) c[i] = 0;
        for (int y = ya; y <= yb; ++y) row(cs[y * g.GX + xa], cs[y * g.GX + xb + 1], count);
#pragma unroll
        for (int i = 6; i >= 0; --i)
          if (c[i] >= k) hi = th[i];
        if (hi < INFINITY) break;
      }
      if (xa == 0 && ya == 0 && xb == g.GX - 1 && yb == g.GY - 1) break;   // every cell seen
      r += 1 + r / 2;
    }
    // narrow (lo, hi] until at most three points of it are taken; the first cuts lie where the bound above usually
    // leaves the distance, so that one round is enough for most waves.  A cut that leaves all of the points in is the
    // last: they may share their distance (all points in one place: 1053 -> 775 ms, as every pass reads them all; the indices path 585)
    for (int it = 0, held = -1; it < 8; ++it) {
      const float w = hi - lo;
      if (it == 0 && hi < INFINITY) {
        th[0] = 0.55f * hi; th[1] = 0.68f * hi; th[2] = 0.76f * hi; th[3] = 0.82f * hi; th[4] = 0.88f * hi;
        th[5] = 0.93f * hi; th[6] = 0.97f * hi;
      } else if (hi < INFINITY) {
#pragma unroll
        for (int i = 0; i < 7; ++i) th[i] = lo + w * (0.125f * (float)(i + 1));
      } else {                                   // no bound: far or few points, cut over their powers of two
        const float e = fmaxf(lo, g.csx * g.csy);
#pragma unroll
        for (int i = 0; i < 7; ++i) th[i] = e * (float)(1 << (2 * i + 2));
      }
#pragma unroll
      for (int i = 0; i < 7; ++i) c[i] = 0;
      int all = 0;
      disc(hi, [&](float d, int s) {
        all += d < hi ? 1 : 0;
        count(d, s);
      });
      chi = all;
      float nlo = lo, nhi = hi;
      int ncl = clo, nch = all;
#pragma unroll
      for (int i = 0; i < 7; ++i)
        if (th[i] > lo && c[i] < k) { nlo = th[i]; ncl = c[i]; }
#pragma unroll
      for (int i = 6; i >= 0; --i)
        if (th[i] < hi && c[i] >= k) { nhi = th[i]; nch = c[i]; }
      const bool same = nlo == lo && nhi == hi;
      lo = nlo; hi = nhi; clo = ncl; chi = nch;
      if (chi < k || k - clo < kPick || same || chi - clo == held) break;
      held = chi - clo;
    }
    // the points under lo, and the k - clo first of those in [lo, hi) by (distance, index), kPick at a time
    float sx = 0.f, sy = 0.f;
    uint64_t last = 0, key[kPick];
    int ks[kPick];
    for (int m = clo; m < k; m += kPick) {
#pragma unroll
      for (int i = 0; i < kPick; ++i) { key[i] = ~(uint64_t)0; ks[i] = -1; }
      const bool first = m == clo;
      disc(hi, [&](float d, int s) {
        if (d < lo) {
          if (first) {
            const float2 v = dv[(uint32_t)s];
            sx += v.x;
            sy += v.y;
          }
        } else if (d < hi) {
          uint64_t ck = dist_key(d, id[(uint32_t)s]);
          if ((first || ck > last) && ck < key[kPick - 1]) {
            int cs_ = s;
#pragma unroll
            for (int i = 0; i < kPick; ++i) {
              const bool lt = ck < key[i];
              const uint64_t tk = key[i];
              const int ts = ks[i];
              key[i] = lt ? ck : tk;
              ks[i] = lt ? cs_ : ts;
              ck = lt ? tk : ck;
              cs_ = lt ? ts : cs_;
            }
          }
        }
      });
#pragma unroll
      for (int i = 0; i < kPick; ++i)
        if (m + i < k) {
          if (ks[i] < 0) {                       // fewer than k finite distances
            sx = sy = NAN;
          } else {
            const float2 v = dv[(uint32_t)ks[i]];
            sx += v.x;
            sy += v.y;
          }
          last = key[i];
          // a point at the same distance may be left out unless the next key is known to lie further
          tie = i + 1 >= kPick || (uint32_t)(key[i + 1 < kPick ? i + 1 : i] >> 32) == (uint32_t)(last >> 32);
        }
      if (ks[kPick - 1] < 0) {
        if (k - m > kPick) { sx = sy = NAN; last = ~(uint64_t)0; }
        break;
      }
    }
    const bool short_ = last == ~(uint64_t)0;    // too few: every finite distance counts
    dk = short_ ? INFINITY : __uint_as_float((uint32_t)(last >> 32));
    jk = (int)(uint32_t)last;
    tie = tie && !short_;
    const float inv = (float)k;
    table[(int64_t)plane * nx * ny + (int64_t)iy * nx + ix] = make_float2(sx / inv, sy / inv);
  }
  const int nbx = (nx + kQB - 1) / kQB, nby = (ny + kQB - 1) / kQB;
  const int bx = ix / kQB, by = iy / kQB;
  const bool block_live = bx < nbx && by < nby;
  const int64_t bi = ((int64_t)plane * nby + by) * nbx + bx;
  if (block_live) {                              // NaN: no query here; negative: ties are decided by the index
    kth[bi * (kQB * kQB) + l] = live ? __uint_as_float(__float_as_uint(dk) | (tie ? 0x80000000u : 0u)) : NAN;
    kid[bi * (kQB * kQB) + l] = jk;
  }
  float m = dk;
#pragma unroll
  for (int d = 8; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, kWave));
  if (block_live && l == 0) bmax[bi] = m;
  m = fmaxf(m, __shfl_xor(m, 16, kWave));
  m = fmaxf(m, __shfl_xor(m, 32, kWave));
  if (lane == 0) atomicMax(pmax + plane, __float_as_uint(m));   // distances are not negative: bits order them
}

// gtr rows 1..T of every batch: minus the point's gradient (its displacement is reference minus position).
__global__ void __launch_bounds__(kBlock) k_lut_adjoint(float x0, float y0, float step, int nx, int ny, int n, int T,
                                                        int k, const float2* __restrict__ xy,
                                                        const int* __restrict__ id, const float4* __restrict__ kth,
                                                        const int* __restrict__ kid, const float* __restrict__ bmax,
                                                        const unsigned* __restrict__ pmax,
                                                        const float2* __restrict__ gtable, float2* __restrict__ gtr) {
  const int i = blockIdx.x * kBlock + threadIdx.x;
  if (i >= n) return;
  const int plane = blockIdx.y;
  const int64_t slot = (int64_t)plane * n + i;
  const float2 p = xy[slot];
  const int j = id[slot];
  const int nbx = (nx + kQB - 1) / kQB, nby = (ny + kQB - 1) / kQB;
  // blocks within the plane's largest k-th distance; the hundredth of a step covers the roundings
  const float R = sqrtf(__uint_as_float(pmax[plane])) + 0.01f * step;
  const float ib = 1.f / ((float)kQB * step), eps = 0.01f * step;
  auto block_of = [&](float v, float o, int nb) { return (int)fminf(fmaxf(floorf((v - o) * ib), 0.f), (float)(nb - 1)); };
  const int xa = block_of(p.x - R, x0, nbx), xb = block_of(p.x + R, x0, nbx);
  const int ya = block_of(p.y - R, y0, nby), yb = block_of(p.y + R, y0, nby);
  const float2* __restrict__ gt = gtable + (int64_t)plane * nx * ny;
  float gx = 0.f, gy = 0.f;
  for (int by = ya; by <= yb; ++by)
    for (int bx = xa; bx <= xb; ++bx) {
      const float lx = (float)(bx * kQB) * step + x0, ly = (float)(by * kQB) * step + y0;
      const float ex = fmaxf(fmaxf(lx - p.x, p.x - (lx + 3.f * step)) - eps, 0.f);
      const float ey = fmaxf(fmaxf(ly - p.y, p.y - (ly + 3.f * step)) - eps, 0.f);
      const int64_t bi = ((int64_t)plane * nby + by) * nbx + bx;
      if (!(ex * ex + ey * ey <= bmax[bi])) continue;
      // a row of four queries at a time; their gradients are loaded whether or not they are taken (a load under a
      // condition of its own was a wait per query)
#pragma unroll
      for (int ly = 0; ly < kQB; ++ly) {
        const int iy = by * kQB + ly;
        const float4 kq = kth[bi * kQB + ly];
        const float dks[kQB] = {kq.x, kq.y, kq.z, kq.w};
        const float dy = ((float)iy * step + y0) - p.y;
        const float2* gr = gt + (uint32_t)(min(iy, ny - 1) * nx);
        float2 gv[kQB];
#pragma unroll
        for (int lx = 0; lx < kQB; ++lx) gv[lx] = gr[(uint32_t)min(bx * kQB + lx, nx - 1)];
#pragma unroll
        for (int lx = 0; lx < kQB; ++lx) {
          const float dx = ((float)(bx * kQB + lx) * step + x0) - p.x;
          const float d = dx * dx + dy * dy, dk = fabsf(dks[lx]);
          bool take = d <= dk;                   // false for NaN
          if (d == dk && __float_as_uint(dks[lx]) >> 31) take = j <= kid[bi * (kQB * kQB) + ly * kQB + lx];
          gx += take ? gv[lx].x : 0.f;
          gy += take ? gv[lx].y : 0.f;
        }
      }
    }
  const float inv = (float)k;
  gtr[((int64_t)plane + plane / T + 1) * n + j] = make_float2(-gx / inv, -gy / inv);
}

// gtr row 0 of every batch: minus the sum of the other rows (every displacement starts at the reference position).
__global__ void __launch_bounds__(kBlock) k_lut_ref_grad(int n, int T, float2* __restrict__ gtr) {
  const int j = blockIdx.x * kBlock + threadIdx.x;
  if (j >= n) return;
  float2* g = gtr + (int64_t)blockIdx.y * (T + 1) * n + j;
  float x = 0.f, y = 0.f;
#pragma unroll 4
  for (int s = 1; s <= T; ++s) {
    const float2 v = g[(int64_t)s * n];
    x -= v.x;
    y -= v.y;
  }
  g[0] = make_float2(x, y);
}

int lut_bad(const char* what, int64_t B, int64_t T, int64_t n, double step, int64_t nx, int64_t ny, int64_t k) {
  const int64_t lim = (int64_t)1 << 31;
  if (B < 0 || T < 1 || n < 1 || nx < 0 || ny < 0 || !(step > 0) || B > 65535 || T > 65535 || B * T > 65535 ||
      n >= lim || nx >= lim || ny >= lim || nx * ny > ((int64_t)1 << 30) || (B * T + B) * (n + 1) >= lim || k < 1 ||
      k > kKnnMaxK || k > n) {
    set_error("%s: bad sizes B=%lld T=%lld n=%lld nx=%lld ny=%lld k=%lld (1 <= k <= min(n, %d))", what, (long long)B,
              (long long)T, (long long)n, (long long)nx, (long long)ny, (long long)k, kKnnMaxK);
    return 1;
  }
  return 0;
}

}  // namespace

extern "C" {

int64_t atl_lut_table_ws_bytes(int64_t B, int64_t T, int64_t n, int64_t nx, int64_t ny) {
  if (lut_bad("lut_table", B, T, n, 1.0, nx, ny, 1)) return -1;
  return lut_layout(B * T, n, nx, ny).bytes;
}

int atl_lut_table_fwd(const float* tr, int64_t B, int64_t T, int64_t n, double x0, double y0, double step, int64_t nx,
                      int64_t ny, int64_t k, float* table, void* ws, int64_t ws_bytes, hipStream_t stream) {
  if (lut_bad("lut_table_fwd", B, T, n, step, nx, ny, k)) return 1;
  if (B == 0 || nx * ny == 0) return 0;
  const int64_t P = B * T, ncell = P * (n + 1);
  const LutLayout L = lut_layout(P, n, nx, ny);
  if (!tr || !table || !ws || ws_bytes < L.bytes) {
    set_error("lut_table_fwd: null argument or a workspace of %lld bytes, need %lld", (long long)ws_bytes, (long long)L.bytes);
    return 1;
  }
  char* w = (char*)ws;
  int *cnt = (int*)(w + L.cnt), *start = (int*)(w + L.start), *id = (int*)(w + L.id);
  float2 *xy = (float2*)(w + L.xy), *dv = (float2*)(w + L.dv);
  const KnnGeom g = lattice_geom((float)x0, (float)y0, (float)step, nx, ny, n);
  const int64_t clear = ncell + P;               // the counts and the planes' largest distances behind them
  hipLaunchKernelGGL(k_knn_zero, dim3(grid_for(clear)), dim3(kBlock), 0, stream, cnt, clear);
  const dim3 pgrid(grid_for(n), (unsigned)P);
  hipLaunchKernelGGL((k_lut_bin<false>), pgrid, dim3(kBlock), 0, stream, (const float2*)tr, (int)T, (int)n, g, cnt,
                     (const int*)nullptr, (float2*)nullptr, (float2*)nullptr, (int*)nullptr);
  scan32(cnt, ncell, (int*)(w + L.part), start, stream);
  hipLaunchKernelGGL((k_lut_bin<true>), pgrid, dim3(kBlock), 0, stream, (const float2*)tr, (int)T, (int)n, g, cnt,
                     (const int*)start, xy, dv, id);
  const dim3 qgrid((unsigned)(((nx + kPatch - 1) / kPatch) * ((ny + kPatch - 1) / kPatch)), (unsigned)P);
  hipLaunchKernelGGL(k_lut_query, qgrid, dim3(kBlock), 0, stream, (float)x0, (float)y0, (float)step, (int)nx, (int)ny,
                     (int)n, (int)k, g, (const int*)start, (const float2*)xy, (const float2*)dv, (const int*)id,
                     (float2*)table, (float*)(w + L.kth), (int*)(w + L.kid), (float*)(w + L.bmax), (unsigned*)(w + L.pmax));
  return check_launch("lut_table_fwd");
}

int atl_lut_table_bwd(const float* gtable, int64_t B, int64_t T, int64_t n, double x0, double y0, double step,
                      int64_t nx, int64_t ny, int64_t k, const void* ws, int64_t ws_bytes, float* gtr,
                      hipStream_t stream) {
  if (lut_bad("lut_table_bwd", B, T, n, step, nx, ny, k)) return 1;
  if (B == 0) return 0;
  const int64_t P = B * T;
  const LutLayout L = lut_layout(P, n, nx, ny);
  if (nx * ny == 0 || !gtable || !gtr || !ws || ws_bytes < L.bytes) {
    set_error("lut_table_bwd: no query, null argument or a workspace of %lld bytes, need %lld", (long long)ws_bytes, (long long)L.bytes);
    return 1;
  }
  const char* w = (const char*)ws;
  const dim3 pgrid(grid_for(n), (unsigned)P);
  hipLaunchKernelGGL(k_lut_adjoint, pgrid, dim3(kBlock), 0, stream, (float)x0, (float)y0, (float)step, (int)nx,
                     (int)ny, (int)n, (int)T, (int)k, (const float2*)(w + L.xy), (const int*)(w + L.id),
                     (const float4*)(w + L.kth), (const int*)(w + L.kid), (const float*)(w + L.bmax), (const unsigned*)(w + L.pmax),
                     (const float2*)gtable, (float2*)gtr);
  hipLaunchKernelGGL(k_lut_ref_grad, dim3(grid_for(n), (unsigned)B), dim3(kBlock), 0, stream, (int)n, (int)T,
                     (float2*)gtr);
  return check_launch("lut_table_bwd");
}

int64_t atl_knn_ws_bytes(int64_t P, int64_t n) {
  if (P < 0 || n < 0 || P * (n + 1) >= (int64_t)1 << 31) return -1;
  return knn_layout(P, n).bytes;
}

int atl_knn_indices(const float* queries, int64_t Q, const float* points, int64_t P, int64_t n, int64_t k,
                    int64_t* idx, void* ws, int64_t ws_bytes, hipStream_t stream) {
  if (Q < 0 || P < 0 || n < 0 || k < 1 || k > kKnnMaxK || k > n || P * (n + 1) >= (int64_t)1 << 31 ||
      Q > (int64_t)1 << 30 || P > 65535) {
    set_error("knn_indices: bad sizes Q=%lld P=%lld n=%lld k=%lld (1 <= k <= min(n, %d))", (long long)Q, (long long)P,
              (long long)n, (long long)k, kKnnMaxK);
    return 1;
  }
  if (Q == 0 || P == 0) return 0;
  const KnnLayout L = knn_layout(P, n);
  if (!ws || ws_bytes < L.bytes) { set_error("knn_indices: workspace of %lld bytes, need %lld", (long long)ws_bytes, (long long)L.bytes); return 1; }
  if (!queries || !points || !idx) { set_error("knn_indices: null argument"); return 1; }
  char* w = (char*)ws;
  KnnGeom* geo = (KnnGeom*)(w + L.geom);
  int* cnt = (int*)(w + L.cnt);
  int* start = (int*)(w + L.start);
  float4* pts = (float4*)(w + L.pts);
  const int64_t ncell = P * (n + 1), np = P * n;
  hipLaunchKernelGGL(k_knn_geom, dim3(1), dim3(kGeomBlock), 0, stream, (const float2*)queries, Q, n, geo);
  hipLaunchKernelGGL(k_knn_zero, dim3(grid_for(ncell)), dim3(kBlock), 0, stream, cnt, ncell);
  hipLaunchKernelGGL((k_knn_bin<false>), dim3(grid_for(np)), dim3(kBlock), 0, stream, (const float2*)points, P, n,
                     (const KnnGeom*)geo, cnt, (const int*)nullptr, (float4*)nullptr);
  scan32(cnt, ncell, (int*)(w + L.part), start, stream);
  hipLaunchKernelGGL((k_knn_bin<true>), dim3(grid_for(np)), dim3(kBlock), 0, stream, (const float2*)points, P, n,
                     (const KnnGeom*)geo, cnt, (const int*)start, pts);
  const dim3 grid(grid_for(Q), (unsigned)P);
  if (k <= 8)
    hipLaunchKernelGGL((k_knn_query<8>), grid, dim3(kBlock), 0, stream, (const float2*)queries, Q, n, (int)k,
                       (const KnnGeom*)geo, (const int*)start, (const float4*)pts, idx);
  else if (k <= 16)
    hipLaunchKernelGGL((k_knn_query<16>), grid, dim3(kBlock), 0, stream, (const float2*)queries, Q, n, (int)k,
                       (const KnnGeom*)geo, (const int*)start, (const float4*)pts, idx);
  else
    hipLaunchKernelGGL((k_knn_query<32>), grid, dim3(kBlock), 0, stream, (const float2*)queries, Q, n, (int)k,
                       (const KnnGeom*)geo, (const int*)start, (const float4*)pts, idx);
  return check_launch("knn_indices");
}

}  // extern "C"
