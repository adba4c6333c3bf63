// MI355X (gfx950) voxelizer: triangle soup -> MaterialKind of every cell of
// a forest, the device form of voxelize_part (part_voxelizer.cpp:71-114)
// over CgalSurfaceMesh (cgal_surface_mesh.cpp).
//
// Per cell (box = CellBounds of the block, centre = mid-point):
//   intersects = some triangle of the part (degenerate ones included, as
//                intersects_box does) meets the closed cell box;
//   inside(m)  = ray parity of mesh m at the centre: along +x, +y and +z,
//                count the non-degenerate triangles the closed ray meets
//                (shared edges and vertices count once per triangle, as
//                RayParityInsideDirectionAabb does), inside when at least
//                two of the three counts are odd;
//   external obstacle: boundary if intersects, else solid if inside, else
//                fluid (MapExternal); internal channel: boundary if
//                intersects, fluid in the lumen (inner mesh), solid in the
//                wall (outer mesh minus lumen), else fluid
//                (MapInternalChannel).
// The reference evaluates these with exact predicates (CGAL's
// Exact_predicates_inexact_constructions_kernel), so the tests are written
// as signs of determinants of the input doubles (exact.h): the box test as
// separating axes (box axes, triangle normal, the nine edge x axis
// products), the ray test as the projected-triangle orientations plus the
// side of the plane, with the ray-in-plane case solved in that plane.
//
// Passes: (1) per triangle its box, exact normal signs and degeneracy, and a
// box per 64 triangles; (2) one workgroup per 8^3 tile of cells picks the
// triangles that can matter to the tile (group boxes, then triangle boxes)
// and, triangle by triangle, tests the few cells each one can reach,
// collecting hits, parities and undecided filters as bits per cell (few
// triangles and many blocks: a thread per cell instead); (3) one
// wave per cell whose filters could not decide repeats its classification with
// exact fallbacks, its lanes a candidate triangle each.
//
// What bounds it: the filters' FP64 arithmetic and the dependent loads of the
// triangles.  The earlier form gave each cell a thread that walked the block's
// candidate lists one triangle after another (and needed the lists, counted and
// emitted with a copy to the host between): 2.85 ms + 2 x 0.24 ms for 8,192
// triangles on 1,152 blocks.  Going by triangle, a sliver costs the cells under
// its box instead of a step for every cell: 0.30 ms for the whole pass.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <string>
#include <vector>

#include "exact.h"
#include "launch.h"
#include "octlb_gpu.h"
#include "octlb_internal.h"
#include "voxelize_queue.h"

namespace octlb {
namespace {

using exact::kUnsure;
using exact::Sign2;
using exact::Sign3;

#define VOX_CHECK(expr)                                                                       \
  do {                                                                                        \
    hipError_t _e = (expr);                                                                   \
    if (_e != hipSuccess)                                                                     \
      throw std::runtime_error(std::string(#expr) + ": " + hipGetErrorString(_e) +           \
                               " (voxelize.hip:" + std::to_string(__LINE__) + ")");          \
  } while (0)

constexpr uint8_t kFluid = 0, kSolid = 1, kBoundary = 2;
constexpr int kVoxThreads = 256;

// One triangle of a part, with what every test needs of it.
struct VTri {
  double v[3][3];
  double lo[3], hi[3];
  int nsign[3];  // exact signs of the normal (B - A) x (C - A)
  int degenerate;
  int mesh;      // 0 outer, 1 inner (lumen) surface
};

// ---------------------------------------------------------------- ray test
// Does the closed ray p + t e_a (t >= 0) meet the closed non-degenerate
// triangle?  1, 0, or kUnsure (filters only).
template <bool kExact>
__host__ __device__ int RayHit(const double* p, int a, const VTri& t) {
  const double* A = t.v[0];
  const double* B = t.v[1];
  const double* C = t.v[2];
  const int u = (a + 1) % 3, w = (a + 2) % 3;
  const int na = t.nsign[a];
  const int s = Sign3<kExact>(B, C, p, A);  // normal . (p - A)
  if (s == kUnsure) return kUnsure;
  if (na != 0) {
    // the plane is met at t = -s / n_a: behind the origin when s and n_a agree
    if (s != 0 && s == na) return 0;
    // p's projection along a in the closed projected triangle
    const int e[3] = {Sign2<kExact>(B[u], B[w], A[u], A[w], p[u], p[w], A[u], A[w]),
                      Sign2<kExact>(C[u], C[w], B[u], B[w], p[u], p[w], B[u], B[w]),
                      Sign2<kExact>(A[u], A[w], C[u], C[w], p[u], p[w], C[u], C[w])};
    bool unsure = false;
    for (int k = 0; k < 3; ++k) {
      if (e[k] == -na) return 0;
      if (e[k] == kUnsure) unsure = true;
    }
    return unsure ? kUnsure : 1;
  }
  if (s != 0) return 0;  // parallel plane off the ray
  // the ray lies in the triangle's plane: solve in the coordinate plane
  // (a, q) onto which the triangle projects without collapsing
  const int q = t.nsign[w] != 0 ? u : w;
  bool unsure = false;
  for (int k = 0; k < 3; ++k) {
    const double* X = t.v[k];
    const double* Y = t.v[(k + 1) % 3];
    const double pq = p[q];
    if ((X[q] > pq && Y[q] > pq) || (X[q] < pq && Y[q] < pq)) continue;
    if (X[q] == pq && Y[q] == pq) {
      if (fmax(X[a], Y[a]) >= p[a]) return 1;
      continue;
    }
    // the edge crosses the line through p at a*: (a* - p_a)(Y_q - X_q) has
    // the sign of (X_a - p_a)(Y_q - X_q) - (X_q - p_q)(Y_a - X_a)
    const int num = Sign2<kExact>(X[a], X[q], p[a], pq, Y[a], Y[q], X[a], X[q]);
    if (num == kUnsure) {
      unsure = true;
      continue;
    }
    const int dq = Y[q] > X[q] ? 1 : -1;
    if (num == 0 || num == dq) return 1;
  }
  return unsure ? kUnsure : 0;
}

// ---------------------------------------------------------------- box test
// Does the closed triangle (degenerate ones too) meet the closed box?
template <bool kExact>
__host__ __device__ int BoxHit(const double* lo, const double* hi, const VTri& t) {
  for (int k = 0; k < 3; ++k)
    if (t.hi[k] < lo[k] || t.lo[k] > hi[k]) return 0;
  const double* A = t.v[0];
  const double* B = t.v[1];
  const double* C = t.v[2];
  bool unsure = false;
  if (t.nsign[0] != 0 || t.nsign[1] != 0 || t.nsign[2] != 0) {
    // triangle plane: the box corners nearest and farthest along the normal
    double cmin[3], cmax[3];
    for (int k = 0; k < 3; ++k) {
      cmin[k] = t.nsign[k] > 0 ? lo[k] : hi[k];
      cmax[k] = t.nsign[k] > 0 ? hi[k] : lo[k];
    }
    const int s1 = Sign3<kExact>(B, C, cmin, A);
    if (s1 == 1) return 0;
    const int s2 = Sign3<kExact>(B, C, cmax, A);
    if (s2 == -1) return 0;
    if (s1 == kUnsure || s2 == kUnsure) unsure = true;
  }
  // axes e_k x (Y - X) for the three edges
  for (int e = 0; e < 3; ++e) {
    const double* X = t.v[e];
    const double* Y = t.v[(e + 1) % 3];
    const double* Z = t.v[(e + 2) % 3];
    for (int k = 0; k < 3; ++k) {
      const int i1 = (k + 1) % 3, i2 = (k + 2) % 3;
      if (Y[i1] == X[i1] && Y[i2] == X[i2]) continue;  // edge along e_k: no axis
      // L = (L_i1, L_i2) = (-(Y - X)_i2, (Y - X)_i1); the box's extreme corners along L
      const int l1 = Y[i2] > X[i2] ? -1 : (Y[i2] < X[i2] ? 1 : 0);
      const int l2 = Y[i1] > X[i1] ? 1 : (Y[i1] < X[i1] ? -1 : 0);
      const double mn1 = l1 > 0 ? lo[i1] : hi[i1], mx1 = l1 > 0 ? hi[i1] : lo[i1];
      const double mn2 = l2 > 0 ? lo[i2] : hi[i2], mx2 = l2 > 0 ? hi[i2] : lo[i2];
      // L . (V - c) = (Y - X)_i1 (V - c)_i2 - (Y - X)_i2 (V - c)_i1
      const int xa = Sign2<kExact>(Y[i1], Y[i2], X[i1], X[i2], X[i1], X[i2], mn1, mn2);
      const int za = Sign2<kExact>(Y[i1], Y[i2], X[i1], X[i2], Z[i1], Z[i2], mn1, mn2);
      if (xa == -1 && za == -1) return 0;  // triangle entirely below the box
      const int xb = Sign2<kExact>(Y[i1], Y[i2], X[i1], X[i2], X[i1], X[i2], mx1, mx2);
      const int zb = Sign2<kExact>(Y[i1], Y[i2], X[i1], X[i2], Z[i1], Z[i2], mx1, mx2);
      if (xb == 1 && zb == 1) return 0;  // entirely above
      if ((xa == kUnsure || za == kUnsure) && xa != 0 && xa != 1 && za != 0 && za != 1) unsure = true;
      if ((xb == kUnsure || zb == kUnsure) && xb != 0 && xb != -1 && zb != 0 && zb != -1) unsure = true;
    }
  }
  return unsure ? kUnsure : 1;
}

// ------------------------------------------------------------ per-triangle
constexpr int kGroup = 64;  // triangles per group box: one wave's

// box / gbox: lo[3], hi[3] of every triangle / group, one array per bound
__global__ __launch_bounds__(kVoxThreads) void KTriPrep(const double* tri, int64_t ntri, int64_t nouter, VTri* out,
                                                        double* box, double* gbox, int64_t ngroup) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const bool live = i < ntri;
  double b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
  if (live) {
    VTri t;
    for (int k = 0; k < 3; ++k)
      for (int d = 0; d < 3; ++d) t.v[k][d] = tri[i * 9 + k * 3 + d];
    for (int d = 0; d < 3; ++d) {
      t.lo[d] = fmin(fmin(t.v[0][d], t.v[1][d]), t.v[2][d]);
      t.hi[d] = fmax(fmax(t.v[0][d], t.v[1][d]), t.v[2][d]);
    }
    for (int a = 0; a < 3; ++a) {
      const int u = (a + 1) % 3, w = (a + 2) % 3;
      t.nsign[a] = Sign2<true>(t.v[1][u], t.v[1][w], t.v[0][u], t.v[0][w], t.v[2][u], t.v[2][w], t.v[0][u],
                               t.v[0][w]);
    }
    t.degenerate = (t.nsign[0] == 0 && t.nsign[1] == 0 && t.nsign[2] == 0) ? 1 : 0;
    t.mesh = i < nouter ? 0 : 1;
    out[i] = t;
    for (int d = 0; d < 3; ++d) {
      box[d * ntri + i] = t.lo[d];
      box[(3 + d) * ntri + i] = t.hi[d];
      // a coordinate that is no number excludes nothing, here as in InList
      b[d] = t.lo[d] == t.lo[d] ? t.lo[d] : -INFINITY;
      b[3 + d] = t.hi[d] == t.hi[d] ? t.hi[d] : INFINITY;
    }
  }
  for (int w = kGroup / 2; w > 0; w >>= 1)
    for (int d = 0; d < 3; ++d) {
      b[d] = fmin(b[d], __shfl_xor(b[d], w));
      b[3 + d] = fmax(b[3 + d], __shfl_xor(b[3 + d], w));
    }
  if ((threadIdx.x & 63) == 0 && i / kGroup < ngroup)
    for (int d = 0; d < 6; ++d) gbox[d * ngroup + i / kGroup] = b[d];
}

// ------------------------------------------------------------ classification
constexpr int kVoxTile = 8;
constexpr int kVoxCells = kVoxTile * kVoxTile * kVoxTile;
constexpr int kVoxLanes = 3;      // log2 of the fewest lanes per candidate triangle
constexpr int kVoxQueue = 2048;   // candidates staged in LDS; one round of the waves adds at most 1,024

// state bits of a cell
constexpr uint32_t kBitHit = 1u, kBitOpen = 2u;
__device__ inline uint32_t OddBit(int mesh, int ax) { return 4u << (mesh * 3 + ax); }
__device__ inline uint32_t UnsureBit(int mesh, int ax) { return 256u << (mesh * 3 + ax); }

// The material of a cell with these bits, or -1 if the filters left it open.
__device__ inline int Decide(uint32_t s, int channel) {
  if (s & kBitHit) return kBoundary;
  if (s & kBitOpen) return -1;
  // inside votes: decided when the certain axes settle the majority
  int inside[2];
  for (int q = 0; q < 2; ++q) {
    int yes = 0, no = 0;
    for (int ax = 0; ax < 3; ++ax) {
      if (s & UnsureBit(q, ax)) continue;
      if (s & OddBit(q, ax)) ++yes; else ++no;
    }
    inside[q] = yes >= 2 ? 1 : (no >= 2 ? 0 : -1);
  }
  if (channel && inside[1] != 0) return inside[1] < 0 ? -1 : kFluid;  // lumen
  return inside[0] < 0 ? -1 : (inside[0] ? kSolid : kFluid);
}

struct VoxArgs {
  const VTri* tris;
  const double* box;    // [6][ntri]
  const double* gbox;   // [6][ngroup]
  int64_t ntri;
  int ngroup;
  const double* bounds;
  int nb;
  int n;
  int te;               // tiles per block edge (KClassifyFew: runs per block)
  int first;            // the launch's first tile (workgroup, queue entry)
  int channel;          // internal channel (else external obstacle)
  uint8_t* material;
  int* queue;           // cells the filters left open: index into material
  unsigned int room;    // how many the queue holds
  unsigned int* queued; // how many there are
};

// Lists a box [lo, hi] (of a triangle or of a group) belongs to for the tile
// bounds tb: bit 0 the box list, bit 1 + a the rays along axis a.
__device__ inline int Lists(const double* bx, const double* tb) {
  bool below[3], above[3];  // wholly below / above the tile along an axis
  for (int d = 0; d < 3; ++d) {
    below[d] = bx[3 + d] < tb[d];
    above[d] = bx[d] > tb[3 + d];
  }
  int m = 0;
  if (!(below[0] || above[0] || below[1] || above[1] || below[2] || above[2])) m |= 1;
  for (int a = 0; a < 3; ++a) {
    const int u = (a + 1) % 3, w = (a + 2) % 3;
    if (!(below[u] || above[u] || below[w] || above[w] || below[a])) m |= 2 << a;
  }
  return m;
}

// First index of the ascending v[0 .. n) with v >= x (kStrict: v > x); a
// guess from the spacing, corrected by comparisons.
template <bool kStrict>
__device__ inline int FirstAt(const double* v, int n, double x, double inv) {
  const double g = (x - v[0]) * inv;
  int i = g > 0.0 ? (g < static_cast<double>(n) ? static_cast<int>(g) : n) : 0;
  while (i > 0 && (kStrict ? v[i - 1] > x : v[i - 1] >= x)) --i;
  while (i < n && (kStrict ? v[i] <= x : v[i] < x)) ++i;
  return i;
}

__global__ __launch_bounds__(kVoxThreads) void KClassify(VoxArgs a) {
  __shared__ uint32_t st[kVoxCells];
  __shared__ double cl[3][kVoxTile], ch[3][kVoxTile], cc[3][kVoxTile], inv[3];
  __shared__ VoxEntry queue[kVoxQueue];
  __shared__ int groups[kVoxThreads];
  __shared__ int nq, ng;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int n = a.n;
  const int tile = a.first + static_cast<int>(blockIdx.x);
  // the same tile of all blocks, then the next: with a block's tiles side by
  // side, those of the same size would all fall to one XCD
  const int b = tile % a.nb, tt = tile / a.nb;
  // tiles in MaterialField order: x fastest
  const int org[3] = {tt % a.te * kVoxTile, tt / a.te % a.te * kVoxTile, tt / (a.te * a.te) * kVoxTile};
  int ext[3];
  for (int d = 0; d < 3; ++d) ext[d] = min(kVoxTile, n - org[d]);
  const double* ob = a.bounds + static_cast<size_t>(b) * 6;
  if (tid < 3 * kVoxTile) {
    // CellBounds (part_voxelizer.cpp:33-47) and the centre, in the
    // reference's operation order
    const int d = tid / kVoxTile, i = tid % kVoxTile;
    const double dx = (ob[3 + d] - ob[d]) / static_cast<double>(n);
    cl[d][i] = ob[d] + static_cast<double>(org[d] + i) * dx;
    ch[d][i] = cl[d][i] + dx;
    cc[d][i] = 0.5 * (cl[d][i] + ch[d][i]);
    if (i == 0) inv[d] = 1.0 / dx;
  }
  if (tid == 0) nq = 0;
  const size_t mbase = static_cast<size_t>(b) * n * n * n;
  auto material_at = [&](int c) {  // tile cell c = (k * 8 + j) * 8 + i
    return mbase + (static_cast<size_t>(org[2] + (c >> 6)) * n + org[1] + ((c >> 3) & 7)) * n + org[0] + (c & 7);
  };
  auto in_block = [&](int c) { return (c & 7) < ext[0] && ((c >> 3) & 7) < ext[1] && (c >> 6) < ext[2]; };
  for (int c = tid; c < kVoxCells; c += kVoxThreads) st[c] = 0u;
  __syncthreads();
  const double tb[6] = {cl[0][0], cl[1][0], cl[2][0], ch[0][ext[0] - 1], ch[1][ext[1] - 1], ch[2][ext[2] - 1]};

  // The lanes of a candidate, 8 to 64, go over the cells in its reach: as many as
  // leave none idle where few candidates with long reaches (the faces of a box)
  // meet the tile.
  auto work = [&](int count) {
    int ls = kVoxLanes;  // log2 of them
    while (ls < 6 && (count << ls) * 2 <= kVoxThreads) ++ls;
    const int lanes = 1 << ls, w0 = tid & (lanes - 1);
    for (int q = tid >> ls; q < count; q += kVoxThreads >> ls) {
      const VTri& t = a.tris[VoxTriangle(queue[q])];
      const int l = VoxList(queue[q]);
      int lo[3], hi[3];  // the cells in reach, per axis
      if (l == 0) {
        for (int d = 0; d < 3; ++d) {
          const bool num = t.lo[d] <= t.hi[d];
          lo[d] = num ? FirstAt<false>(ch[d], ext[d], t.lo[d], inv[d]) : 0;
          hi[d] = num ? FirstAt<true>(cl[d], ext[d], t.hi[d], inv[d]) : ext[d];
        }
      } else {
        if (t.degenerate) continue;
        // a ray from a centre can only meet a triangle whose box holds the
        // centre's projection and reaches it along the axis
        for (int d = 0; d < 3; ++d) {
          const bool num = t.lo[d] <= t.hi[d];
          lo[d] = num && d != l - 1 ? FirstAt<false>(cc[d], ext[d], t.lo[d], inv[d]) : 0;
          hi[d] = num ? FirstAt<true>(cc[d], ext[d], t.hi[d], inv[d]) : ext[d];
        }
      }
      const int ni = hi[0] - lo[0], nj = hi[1] - lo[1], nk = hi[2] - lo[2];
      if (ni <= 0 || nj <= 0 || nk <= 0) continue;
      // cells w0, w0 + lanes, ... of the reach, x fastest: stepped with carries
      const int si = lanes % ni, sj = lanes / ni % nj, sk = lanes / (ni * nj);
      int ri = w0 % ni - si, rj = w0 / ni % nj - sj, rk = w0 / (ni * nj) - sk;
      for (;;) {
        ri += si;
        rj += sj;
        rk += sk;
        if (ri >= ni) {
          ri -= ni;
          ++rj;
        }
        if (rj >= nj) {
          rj -= nj;
          ++rk;
        }
        if (rk >= nk) break;
        const int i = lo[0] + ri, j = lo[1] + rj, k = lo[2] + rk;
        const int c = (k * kVoxTile + j) * kVoxTile + i;
        if (st[c] & kBitHit) continue;  // a boundary cell already
        if (l == 0) {
          const double blo[3] = {cl[0][i], cl[1][j], cl[2][k]}, bhi[3] = {ch[0][i], ch[1][j], ch[2][k]};
          const int h = BoxHit<false>(blo, bhi, t);
          if (h != 0) atomicOr(&st[c], h == 1 ? kBitHit : kBitOpen);
        } else {
          const double p[3] = {cc[0][i], cc[1][j], cc[2][k]};
          const int h = RayHit<false>(p, l - 1, t);
          if (h == 1) atomicXor(&st[c], OddBit(t.mesh, l - 1));
          if (h == kUnsure) atomicOr(&st[c], UnsureBit(t.mesh, l - 1));
        }
      }
    }
  };

  for (int g0 = 0; g0 < a.ngroup; g0 += kVoxThreads) {
    if (tid == 0) ng = 0;
    __syncthreads();
    const int g = g0 + tid;
    if (g < a.ngroup) {
      double bx[6];
      for (int d = 0; d < 6; ++d) bx[d] = a.gbox[static_cast<size_t>(d) * a.ngroup + g];
      if (Lists(bx, tb)) groups[atomicAdd(&ng, 1)] = g;
    }
    __syncthreads();
    const int m = ng;
    for (int w0 = 0; w0 < m; w0 += kVoxThreads / 64) {
      if (w0 + wave < m) {
        const int64_t t = static_cast<int64_t>(groups[w0 + wave]) * kGroup + lane;
        if (t < a.ntri) {
          double bx[6];
          for (int d = 0; d < 6; ++d) bx[d] = a.box[static_cast<size_t>(d) * a.ntri + t];
          const int in = Lists(bx, tb);
          for (int l = 0; l < 4; ++l)
            if (in >> l & 1) queue[atomicAdd(&nq, 1)] = MakeVoxEntry(t, l);
        }
      }
      __syncthreads();
      const int count = nq;
      if (count > kVoxQueue - 4 * kVoxThreads) {
        work(count);
        __syncthreads();
        if (tid == 0) nq = 0;
      }
      __syncthreads();
    }
  }
  work(nq);
  __syncthreads();

  for (int c = tid; c < kVoxCells; c += kVoxThreads) {
    const uint32_t s = st[c];
    if (!in_block(c)) continue;
    const int m = Decide(s, a.channel);
    if (m >= 0) {
      a.material[material_at(c)] = static_cast<uint8_t>(m);
    } else {
      const unsigned int slot = atomicAdd(a.queued, 1u);
      if (slot < a.room) a.queue[slot] = static_cast<int>(material_at(c));
    }
  }
}

// Few triangles and many blocks.  A wave takes kFewCells cells of a block, finds
// the triangles (a lane each, so at most 64) that can matter to the layers they
// are in, and goes through these with a thread per cell and the triangle in scalar
// registers.  Few triangles are large ones: most tiles meet none or whole faces,
// and a tile of KClassify pays about 5 ns for its barriers and its queue whatever it
// finds.  A box of 12 triangles over 64,000 blocks, against KClassify: 4^3 cells
// 0.20 / 0.99 ms, 8^3 1.34 / 3.02, 9^3 1.92 / 8.56, 16^3 9.4 / 20.8.
//
// Where all triangles lie in one block its waves go through them one after another,
// some 3.6 us each (50 in one of 1,000 blocks: 0.18 ms, KClassify 0.04), so the
// tiles must outweigh that: kFewTiles of them per triangle.
constexpr int kVoxFew = 64;
constexpr int kFewTiles = 512;
constexpr int kFewCells = 256;
__global__ __launch_bounds__(kVoxThreads) void KClassifyFew(VoxArgs a) {
  const int lane = threadIdx.x & 63, n = a.n, cells = n * n * n;
  const int64_t task =
      (static_cast<int64_t>(a.first) + blockIdx.x) * (kVoxThreads / 64) +
      __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  if (task / a.te >= a.nb) return;
  const int b = static_cast<int>(task / a.te);
  const int c0 = static_cast<int>(task % a.te) * kFewCells, c1 = c0 + min(kFewCells, cells - c0);
  const double* ob = a.bounds + static_cast<size_t>(b) * 6;
  double dx[3];
  for (int d = 0; d < 3; ++d) dx[d] = (ob[3 + d] - ob[d]) / static_cast<double>(n);
  // CellBounds (part_voxelizer.cpp:33-47), in the reference's operation order
  auto low = [&](int d, int i) { return ob[d] + static_cast<double>(i) * dx[d]; };
  const double rb[6] = {low(0, 0), low(1, 0), low(2, c0 / (n * n)),
                        low(0, n - 1) + dx[0], low(1, n - 1) + dx[1], low(2, (c1 - 1) / (n * n)) + dx[2]};
  int in = 0;
  if (lane < a.ntri) {
    double bx[6];
    for (int d = 0; d < 6; ++d) bx[d] = a.box[d * a.ntri + lane];
    in = Lists(bx, rb);
  }
  const uint64_t near = __ballot(in & 1), rays = __ballot(in & 14);
  for (int c = c0 + lane; c < c1; c += 64) {
    const int ijk[3] = {c % n, c / n % n, c / (n * n)};
    double lo[3], hi[3], p[3];
    for (int d = 0; d < 3; ++d) {
      lo[d] = low(d, ijk[d]);
      hi[d] = lo[d] + dx[d];
      p[d] = 0.5 * (lo[d] + hi[d]);
    }
    uint32_t s = 0;
    for (uint64_t todo = near; todo; todo &= todo - 1) {
      const VTri& t = a.tris[__builtin_ctzll(todo)];
      bool reach = true;
      for (int d = 0; d < 3; ++d) reach = reach && (!(t.lo[d] <= t.hi[d]) || (hi[d] >= t.lo[d] && lo[d] <= t.hi[d]));
      if (!reach || (s & kBitHit)) continue;
      const int h = BoxHit<false>(lo, hi, t);
      if (h != 0) s |= h == 1 ? kBitHit : kBitOpen;
    }
    if (!(s & (kBitHit | kBitOpen))) {
      for (uint64_t todo = rays; todo; todo &= todo - 1) {
        const VTri& t = a.tris[__builtin_ctzll(todo)];
        if (t.degenerate) continue;
        bool below[3], above[3];  // the centre, of the triangle's box
        for (int d = 0; d < 3; ++d) {
          const bool num = t.lo[d] <= t.hi[d];
          below[d] = num && !(p[d] >= t.lo[d]);
          above[d] = num && !(p[d] <= t.hi[d]);
        }
#pragma unroll
        for (int ax = 0; ax < 3; ++ax) {
          const int u = (ax + 1) % 3, w = (ax + 2) % 3;
          if (above[ax] || below[u] || above[u] || below[w] || above[w]) continue;
          const int h = RayHit<false>(p, ax, t);
          if (h == 1) s ^= OddBit(t.mesh, ax);
          if (h == kUnsure) s |= UnsureBit(t.mesh, ax);
        }
      }
    }
    const int m = Decide(s, a.channel);
    const size_t at = static_cast<size_t>(b) * cells + c;
    if (m >= 0) {
      a.material[at] = static_cast<uint8_t>(m);
    } else {
      const unsigned int slot = atomicAdd(a.queued, 1u);
      if (slot < a.room) a.queue[slot] = static_cast<int>(at);
    }
  }
}

// One wave per cell that the filters left open; every predicate is decided
// exactly.  The wave walks the groups and queues the triangles that can matter
// to the cell, so that its lanes take one exact test each: such a test is a
// chain of expansions, long beside everything else here.  Taken by tiles as in
// KClassify (a triangle's lanes over its cells) the chains of a tile's open
// cells follow each other: 148 ms for 1,728 blocks and a sphere of 32 triangles
// centred on cell faces, 15.6 ms this way.
constexpr int kExactQueue = 256;  // 63 left over and at most 192 of one group
__global__ __launch_bounds__(64) void KClassifyExact(VoxArgs a) {
  __shared__ VoxEntry queue[kExactQueue];
  __shared__ int nq;
  const int lane = threadIdx.x, n = a.n, cells = n * n * n;
  const int at = a.queue[a.first + static_cast<int>(blockIdx.x)];
  const int b = at / cells, cell = at % cells;
  const int ijk[3] = {cell % n, cell / n % n, cell / (n * n)};
  const double* ob = a.bounds + static_cast<size_t>(b) * 6;
  double box[6], p[6];  // the cell's bounds; its centre as a box
  for (int d = 0; d < 3; ++d) {
    const double dx = (ob[3 + d] - ob[d]) / static_cast<double>(n);
    box[d] = ob[d] + static_cast<double>(ijk[d]) * dx;
    box[3 + d] = box[d] + dx;
    p[d] = p[3 + d] = 0.5 * (box[d] + box[3 + d]);
  }
  // test(entry) for every triangle of the lists in `want` that reach the cell,
  // up to 64 at a time, until one returns true
  auto walk = [&](int want, auto&& test) {
    auto lists = [&](const double* from, int64_t stride) {
      double bx[6];
      for (int d = 0; d < 6; ++d) bx[d] = from[d * stride];
      return want & ((Lists(bx, box) & 1) | (Lists(bx, p) & 14));
    };
    if (lane == 0) nq = 0;
    __syncthreads();
    auto drain = [&](int least) {
      for (int left; (left = nq) >= least;) {
        const int first = left > 64 ? left - 64 : 0;
        const bool found = first + lane < left && test(queue[first + lane]);
        __syncthreads();  // the entries are read before the next are put in
        if (lane == 0) nq = first;
        __syncthreads();
        if (__any(found)) return true;
      }
      return false;
    };
    for (int g0 = 0; g0 < a.ngroup; g0 += 64) {
      uint64_t todo = __ballot(g0 + lane < a.ngroup && lists(a.gbox + min(g0 + lane, a.ngroup - 1), a.ngroup) != 0);
      while (todo) {
        const int64_t t = (static_cast<int64_t>(g0) + __builtin_ctzll(todo)) * kGroup + lane;
        todo &= todo - 1;
        if (t < a.ntri) {
          const int in = lists(a.box + t, a.ntri);
          for (int l = 0; l < 4; ++l)
            if (in >> l & 1) queue[atomicAdd(&nq, 1)] = MakeVoxEntry(t, l);
        }
        __syncthreads();
        if (drain(64)) return true;
      }
    }
    return drain(1);
  };
  if (walk(1, [&](VoxEntry e) { return BoxHit<true>(box, box + 3, a.tris[VoxTriangle(e)]) == 1; })) {
    if (lane == 0) a.material[at] = kBoundary;
    return;
  }
  uint32_t odd = 0;  // this lane's share of the parities
  walk(14, [&](VoxEntry e) {
    const VTri& t = a.tris[VoxTriangle(e)];
    const int ax = VoxList(e) - 1;
    if (!t.degenerate && RayHit<true>(p, ax, t) == 1) odd ^= OddBit(t.mesh, ax);
    return false;
  });
  for (int w = 32; w > 0; w >>= 1) odd ^= __shfl_xor(odd, w);
  int inside[2];
  for (int m = 0; m < 2; ++m) {
    int votes = 0;
    for (int ax = 0; ax < 3; ++ax) votes += (odd & OddBit(m, ax)) ? 1 : 0;
    inside[m] = votes >= 2;
  }
  if (lane == 0) a.material[at] = !(a.channel && inside[1]) && inside[0] ? kSolid : kFluid;
}

// outside_sample_fraction (cgal_surface_mesh.cpp): s^3 points over the
// outer soup's box, inside by ray parity against every outer triangle.
__global__ void KSampleInside(const VTri* tris, int64_t nouter, const double* box, int s, int* inside) {
  const int q = static_cast<int>(blockIdx.x * blockDim.x + threadIdx.x);
  if (q >= s * s * s) return;
  const int ix = q % s, iy = (q / s) % s, iz = q / (s * s);
  const double p[3] = {box[0] + static_cast<double>(ix) * ((box[3] - box[0]) / static_cast<double>(s - 1)),
                       box[1] + static_cast<double>(iy) * ((box[4] - box[1]) / static_cast<double>(s - 1)),
                       box[2] + static_cast<double>(iz) * ((box[5] - box[2]) / static_cast<double>(s - 1))};
  int votes = 0;
  for (int ax = 0; ax < 3; ++ax) {
    int odd = 0;
    for (int64_t e = 0; e < nouter; ++e)
      if (!tris[e].degenerate && RayHit<true>(p, ax, tris[e]) == 1) odd ^= 1;
    votes += odd;
  }
  inside[q] = votes >= 2 ? 1 : 0;
}

// Device memory of one call, an allocation per array.  One for all of them is
// beyond the 2 MB that the runtime hands out of blocks it keeps: freed by every
// call, it left the copies of pageable memory slow, here and in the calls that
// follow (290 KB: 118 instead of 17 us; voxelizer and link build of 1,152 blocks
// 2.1 ms that way, 1.0 ms this way).
class VoxBuffer {
 public:
  template <typename P>
  P* Get(size_t count) {
    void* p = nullptr;
    VOX_CHECK(hipMalloc(&p, std::max<size_t>(count, 1) * sizeof(P)));
    ptrs_.push_back(p);
    return static_cast<P*>(p);
  }
  ~VoxBuffer() {
    for (void* p : ptrs_) (void)hipFree(p);  // teardown
  }

 private:
  std::vector<void*> ptrs_;
};

// Open cells that a call keeps room for; where there are more, the filters run
// again with room for all.
constexpr size_t kOpenRoom = 131072;

constexpr double kMinLumenOutsideFraction = 0.05;  // part_voxelizer.cpp:10-11
constexpr int kWatertightSampleResolution = 5;

}  // namespace

int VoxelizePart(int32_t num_blocks, int32_t n, const double* bounds, int64_t num_triangles,
                 const double* triangles, int64_t num_inner, const double* inner, int32_t role, uint8_t* material,
                 int64_t* num_exact) {
  if (num_blocks <= 0 || n <= 0 || !bounds || !material) throw std::invalid_argument("bad forest arguments");
  if (role != OCTLB_PART_INTERNAL_CHANNEL && role != OCTLB_PART_EXTERNAL_OBSTACLE)
    throw std::invalid_argument("unknown part role");
  // validate_geometry_part (part_voxelizer.cpp:51-69)
  if (num_triangles <= 0 || !triangles) throw std::invalid_argument("geometry part has no triangles");
  const bool channel = role == OCTLB_PART_INTERNAL_CHANNEL;
  if (channel && (num_inner <= 0 || !inner)) throw std::invalid_argument("kInternalChannel requires inner_cavity_soup");
  if (!channel) num_inner = 0;
  const int64_t ntri = num_triangles + num_inner;
  if (ntri > static_cast<int64_t>(INT32_MAX)) throw std::invalid_argument("too many triangles (> 2^31 - 1)");
  const size_t cells = static_cast<size_t>(n) * n * n;
  const size_t total = static_cast<size_t>(num_blocks) * cells;
  if (total > static_cast<size_t>(INT32_MAX)) throw std::invalid_argument("forest too large (cells > 2^31)");

  const int te = (n + kVoxTile - 1) / kVoxTile;
  const int64_t ntile = static_cast<int64_t>(num_blocks) * te * te * te;
  const int64_t ngroup = (ntri + kGroup - 1) / kGroup;
  VoxBuffer buf;
  double* d_raw = buf.Get<double>(static_cast<size_t>(ntri) * 9);
  VOX_CHECK(hipMemcpy(d_raw, triangles, static_cast<size_t>(num_triangles) * 9 * sizeof(double),
                      hipMemcpyHostToDevice));
  if (num_inner > 0)
    VOX_CHECK(hipMemcpy(d_raw + num_triangles * 9, inner, static_cast<size_t>(num_inner) * 9 * sizeof(double),
                        hipMemcpyHostToDevice));
  VTri* d_tri = buf.Get<VTri>(static_cast<size_t>(ntri));
  double* d_tribox = buf.Get<double>(static_cast<size_t>(ntri) * 6);
  double* d_gbox = buf.Get<double>(static_cast<size_t>(ngroup) * 6);
  hipLaunchKernelGGL(KTriPrep, dim3(static_cast<unsigned>((ntri + kVoxThreads - 1) / kVoxThreads)), dim3(kVoxThreads),
                     0, nullptr, d_raw, ntri, num_triangles, d_tri, d_tribox, d_gbox, ngroup);
  VOX_CHECK(hipGetLastError());

  if (channel) {
    // the outer mesh must leave lumen/exterior volume (outside fraction)
    double box[6] = {triangles[0], triangles[1], triangles[2], triangles[0], triangles[1], triangles[2]};
    for (int64_t t = 0; t < num_triangles * 3; ++t)
      for (int d = 0; d < 3; ++d) {
        box[d] = std::min(box[d], triangles[t * 3 + d]);
        box[3 + d] = std::max(box[3 + d], triangles[t * 3 + d]);
      }
    const int s = kWatertightSampleResolution;
    const int pts = s * s * s;
    double* d_box = buf.Get<double>(6);
    int* d_in = buf.Get<int>(pts);
    VOX_CHECK(hipMemcpy(d_box, box, sizeof(box), hipMemcpyHostToDevice));
    hipLaunchKernelGGL(KSampleInside, dim3((pts + 63) / 64), dim3(64), 0, nullptr, d_tri, num_triangles, d_box, s,
                       d_in);
    VOX_CHECK(hipGetLastError());
    std::vector<int> in(pts);
    VOX_CHECK(hipMemcpy(in.data(), d_in, pts * sizeof(int), hipMemcpyDeviceToHost));
    int outside = 0;
    for (int v : in) outside += v ? 0 : 1;
    if (static_cast<double>(outside) / static_cast<double>(pts) < kMinLumenOutsideFraction)
      throw std::invalid_argument(
          "kInternalChannel mesh has insufficient exterior/lumen volume (solid-wall channel expected)");
  }

  VoxArgs a{};
  a.tris = d_tri;
  a.box = d_tribox;
  a.gbox = d_gbox;
  a.ntri = ntri;
  a.ngroup = static_cast<int>(ngroup);
  double* d_bounds = buf.Get<double>(static_cast<size_t>(num_blocks) * 6);
  a.bounds = d_bounds;
  a.nb = num_blocks;
  a.n = n;
  const bool few = ntri <= kVoxFew && ntile >= kFewTiles * ntri;
  constexpr int waves = kVoxThreads / 64;
  a.te = few ? static_cast<int>((cells + kFewCells - 1) / kFewCells) : te;
  a.channel = channel ? 1 : 0;
  a.material = buf.Get<uint8_t>(total);
  a.room = static_cast<unsigned int>(std::min(total, kOpenRoom));
  a.queue = buf.Get<int>(a.room);
  a.queued = buf.Get<unsigned int>(1);
  VOX_CHECK(hipMemcpy(d_bounds, bounds, static_cast<size_t>(num_blocks) * 6 * sizeof(double),
                      hipMemcpyHostToDevice));
  // blocks of 9^3 or 10^3 cells have eight tiles, most of their cells idle:
  // 1.6e9 cells are 17.6 million workgroups
  auto launch = [&](auto kernel, int64_t groups, int threads) {
    ForLaunches(groups, threads, [&](int64_t first, int64_t count) {
      a.first = static_cast<int>(first);
      hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(count)), dim3(threads), 0, nullptr, a);
      VOX_CHECK(hipGetLastError());
    });
  };
  unsigned int queued = 0;
  auto classify = [&] {
    VOX_CHECK(hipMemset(a.queued, 0, sizeof(unsigned int)));
    if (few)
      launch(KClassifyFew, (num_blocks * static_cast<int64_t>(a.te) + waves - 1) / waves, kVoxThreads);
    else
      launch(KClassify, ntile, kVoxThreads);
    VOX_CHECK(hipMemcpy(&queued, a.queued, sizeof(queued), hipMemcpyDeviceToHost));
  };
  classify();
  if (queued > a.room) {
    a.room = queued;
    a.queue = buf.Get<int>(queued);
    classify();
  }
  launch(KClassifyExact, queued, 64);
  VOX_CHECK(hipMemcpy(material, a.material, total, hipMemcpyDeviceToHost));
  if (num_exact) *num_exact = queued;
  return OCTLB_OK;
}

}  // namespace octlb

extern "C" int octlb_voxelize_part(int32_t num_blocks, int32_t n, const double* bounds, int64_t num_triangles,
                                   const double* triangles, int64_t num_inner_triangles,
                                   const double* inner_triangles, int32_t role, uint8_t* material,
                                   int64_t* num_exact) {
  try {
    return octlb::VoxelizePart(num_blocks, n, bounds, num_triangles, triangles, num_inner_triangles,
                               inner_triangles, role, material, num_exact);
  } catch (const std::invalid_argument& e) {
    return octlb::SetError(OCTLB_EINVAL, e.what());
  } catch (const std::exception& e) {
    return octlb::SetError(OCTLB_EHIP, e.what());
  }
}
