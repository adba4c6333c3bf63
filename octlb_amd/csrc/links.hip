// Bouzidi wall fractions from a triangle soup on the GPU: the device form of
// BouzidiLinkData::Build (bouzidi_link_data.cpp:139-233).
//
// The reference visits every fluid cell, finds the nearest point of the soup
// (closest point over the three edges of every triangle, first minimum kept)
// and, for each population whose in-block pull-source neighbour x + c_opp(i)
// is solid-like, stores q = ((w - x) . c dx) / |c dx|^2 when it lies in
// (1e-8, 1 - 1e-8).  Only cells with a solid-like in-block neighbour can
// produce a link, so the device pass
//   1. compacts those candidate cells per block with wave ballots and
//      prefix counts (KCandidates, then a single-workgroup scan),
//   2. gives each candidate one wave: it searches the group of consecutive
//      triangles whose box lies nearest, then the groups whose box is not
//      strictly farther than the best point; lanes keep their first minimum
//      and a butterfly reduction picks the smallest distance, ties to the
//      lowest triangle index -- the sequential first minimum (KNearest);
//      lanes 0..17 then evaluate the 18 populations,
//   3. compacts the links in (block, cell, population) order, the dense
//      q_frac order (KEmit).
// Every floating-point expression keeps the reference's operand order and
// the file is built without FMA contraction, so q is bit-identical.
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "d3q19.h"
#include "octlb_gpu.h"
#include "octlb_internal.h"

namespace octlb {
namespace {

#define LINK_CHECK(expr)                                                                      \
  do {                                                                                        \
    hipError_t _e = (expr);                                                                   \
    if (_e != hipSuccess)                                                                     \
      throw std::runtime_error(std::string(#expr) + ": " + hipGetErrorString(_e) +           \
                               " (links.hip:" + std::to_string(__LINE__) + ")");             \
  } while (0)

constexpr int kLinkThreads = 256;      // 4 waves
constexpr int64_t kMaxGroups = 16384;  // group boxes kept per call

// Consecutive triangles per group: a wave's 64, more where the soup would
// otherwise have more than kMaxGroups groups.
__host__ __device__ inline int64_t GroupSize(int64_t ntri) {
  return 64 * ((ntri + 64 * kMaxGroups - 1) / (64 * kMaxGroups));
}

// Groups of a soup; none where a workgroup shares the whole soup in one go.
int64_t GroupCount(int64_t ntri) { return ntri > kLinkThreads ? (ntri + GroupSize(ntri) - 1) / GroupSize(ntri) : 0; }

__device__ __forceinline__ bool SolidLike(uint8_t m) { return m == 1 || m == 2; }  // kSolid, kBoundary

// Material of cell (i, j, k) in MaterialField order (material_field.cpp:16-31).
__device__ __forceinline__ uint8_t Mat(const uint8_t* mat, int n, int i, int j, int k) {
  return mat[(static_cast<size_t>(k) * n + j) * n + i];
}

// A fluid cell with a solid-like in-block neighbour at x + c_opp(i) for some
// i (NeighborMaterial: outside the block counts as fluid).
__device__ bool IsCandidate(const uint8_t* mat, int n, int i, int j, int k) {
  if (Mat(mat, n, i, j, k) != 0) return false;
  bool any = false;
#pragma unroll
  for (int ip = 1; ip < kQ; ++ip) {
    const int o = Opp(ip);
    const int ni = i + Cx(o), nj = j + Cy(o), nk = k + Cz(o);
    if (ni < 0 || ni >= n || nj < 0 || nj >= n || nk < 0 || nk >= n) continue;
    any = any || SolidLike(Mat(mat, n, ni, nj, nk));
  }
  return any;
}

// Per block: count (WRITE = false) or write (WRITE = true) the candidate
// cells in increasing cell index (i*n + j)*n + k.
template <bool WRITE>
__global__ __launch_bounds__(kLinkThreads) void KCandidates(int n, const uint8_t* material, int* counts,
                                                             const int64_t* offsets, int2* cand) {
  __shared__ int wave_sum[kLinkThreads / 64];
  const int b = blockIdx.x;
  const int ncell = n * n * n;
  const uint8_t* mat = material + static_cast<size_t>(b) * ncell;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int64_t run = WRITE ? offsets[b] : 0;
  for (int base = 0; base < ncell; base += kLinkThreads) {
    const int c = base + static_cast<int>(threadIdx.x);
    bool flag = false;
    if (c < ncell) flag = IsCandidate(mat, n, c / (n * n), (c / n) % n, c % n);
    const uint64_t m = __ballot(flag);
    if (lane == 0) wave_sum[wave] = __popcll(m);
    __syncthreads();
    int before = 0, total = 0;
    for (int w = 0; w < kLinkThreads / 64; ++w) {
      before += w < wave ? wave_sum[w] : 0;
      total += wave_sum[w];
    }
    if (WRITE && flag) {
      const int rank = __popcll(m & ((uint64_t(1) << lane) - 1));
      cand[run + before + rank] = make_int2(b, c);
    }
    run += total;
    __syncthreads();  // wave_sum is rewritten by the next chunk
  }
  if (!WRITE && threadIdx.x == 0) counts[b] = static_cast<int>(run);
}

// Exclusive prefix sum of count ints into int64 offsets, total appended:
// one workgroup, chunks of 1024 in order (deterministic).
__global__ __launch_bounds__(1024) void KScan(const int* in, int64_t count, int64_t* out) {
  __shared__ int64_t part[1024];
  __shared__ int64_t carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  for (int64_t base = 0; base < count; base += 1024) {
    const int64_t i = base + threadIdx.x;
    const int64_t v = i < count ? in[i] : 0;
    part[threadIdx.x] = v;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
      const int64_t add = threadIdx.x >= static_cast<unsigned>(off) ? part[threadIdx.x - off] : 0;
      __syncthreads();
      part[threadIdx.x] += add;
      __syncthreads();
    }
    if (i < count) out[i] = carry + part[threadIdx.x] - v;
    __syncthreads();
    if (threadIdx.x == 1023) carry += part[1023];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[count] = carry;
}

// ClosestPointOnSegment (bouzidi_link_data.cpp:19-40), std::clamp(t, 0, 1).
__device__ __forceinline__ void SegClosest(const double* p, double ax, double ay, double az, double bx, double by,
                                           double bz, double* o) {
  const double abx = bx - ax, aby = by - ay, abz = bz - az;
  const double apx = p[0] - ax, apy = p[1] - ay, apz = p[2] - az;
  const double ab2 = abx * abx + aby * aby + abz * abz;
  double t = 0.0;
  if (ab2 > 0.0) {
    t = (apx * abx + apy * aby + apz * abz) / ab2;
    t = t < 0.0 ? 0.0 : (1.0 < t ? 1.0 : t);
  }
  o[0] = ax + t * abx;
  o[1] = ay + t * aby;
  o[2] = az + t * abz;
}

// ClosestPointOnTriangle (bouzidi_link_data.cpp:42-76): nearest of the three
// edge points in edge order v0v1, v1v2, v2v0, first kept on ties; v0 when no
// distance is below DBL_MAX.
__device__ __forceinline__ void TriClosest(const double* t, const double* p, double* o) {
  double best = DBL_MAX;
  o[0] = t[0];
  o[1] = t[1];
  o[2] = t[2];
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    const int a = 3 * e, b = 3 * ((e + 1) % 3);
    double c[3];
    SegClosest(p, t[a], t[a + 1], t[a + 2], t[b], t[b + 1], t[b + 2], c);
    const double dx = p[0] - c[0], dy = p[1] - c[1], dz = p[2] - c[2];
    const double d2 = dx * dx + dy * dy + dz * dz;
    if (d2 < best) {
      best = d2;
      o[0] = c[0];
      o[1] = c[1];
      o[2] = c[2];
    }
  }
}

// A box (lo[3], hi[3]) that holds every computed point of the edges inside bx.  A
// point a + t (b - a), 0 <= t <= 1, may come out up to 5 2^-53 M beyond the box
// along an axis, M the box's largest coordinate there: 2 M for each rounding of
// b - a and of its product with t, M for the sum.  Widened by 8 2^-53 M, less one
// for this sum's own rounding.
__device__ __forceinline__ void Widen(double* bx) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double m = 0x1p-50 * fmax(fabs(bx[d]), fabs(bx[3 + d]));
    bx[d] -= m;
    bx[3 + d] += m;
  }
}

// Widened box of a triangle.
__device__ __forceinline__ void TriBox(const double* v, double* bx) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    bx[d] = fmin(v[d], fmin(v[3 + d], v[6 + d]));
    bx[3 + d] = fmax(v[d], fmax(v[3 + d], v[6 + d]));
  }
  Widen(bx);
}

// No computed point of an edge inside the widened box bx is at a smaller computed
// squared distance from p: the roundings of p - q, the squares and the sum stay far
// below 1e-12 relative.
__device__ __forceinline__ double BoxDistance2(const double* bx, const double* p) {
  double lb = 0.0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double h = fmax(fmax(bx[d] - p[d], p[d] - bx[3 + d]), 0.0);
    lb += h * h;
  }
  return lb * (1.0 - 1.0e-12);
}

// Widened box (lo[3], hi[3]) of each group of consecutive triangles, one
// array per bound; one wave per group.  A coordinate that is no number is left
// out: the edges that hold it are at no distance from anything.
__global__ __launch_bounds__(kLinkThreads) void KGroupBox(const double* tris, int64_t ntri, int64_t ngroup,
                                                          double* gbox) {
  const int lane = threadIdx.x & 63;
  const int64_t g = static_cast<int64_t>(blockIdx.x) * (kLinkThreads / 64) + (threadIdx.x >> 6);
  if (g >= ngroup) return;
  const int64_t gs = GroupSize(ntri);
  const int64_t v0 = 3 * g * gs, v1 = 3 * (ntri < (g + 1) * gs ? ntri : (g + 1) * gs);  // vertices
  double b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
  for (int64_t v = v0 + lane; v < v1; v += 64)
    for (int d = 0; d < 3; ++d) {
      b[d] = fmin(b[d], tris[3 * v + d]);
      b[3 + d] = fmax(b[3 + d], tris[3 * v + d]);
    }
  for (int w = 32; w > 0; w >>= 1)
    for (int d = 0; d < 3; ++d) {
      b[d] = fmin(b[d], __shfl_xor(b[d], w));
      b[3 + d] = fmax(b[3 + d], __shfl_xor(b[3 + d], w));
    }
  Widen(b);
  if (lane < 6) {
    double out = b[0];
#pragma unroll
    for (int d = 1; d < 6; ++d) out = lane == d ? b[d] : out;
    gbox[lane * ngroup + g] = out;
  }
}

// One wave per candidate cell: nearest soup point, then the 18 populations.
// The search goes by groups: a group whose box is farther (BoxDistance2) than
// the best point so far holds neither a closer nor an equal minimum, and the first
// group searched is the nearest one, so few are left where consecutive triangles
// near each other: 14.7 us for 3,328 cells and 8,192 triangles in the order of
// their surface (257 us when every triangle's box was tested).
//
// Groups of triangles in any order, or of slivers across the domain, span it all
// and none drops out.  Then a wave reads the whole soup, which L2 has to deliver
// once per cell: the four waves of a workgroup share it instead, 256 triangles at a
// time in LDS.  They do where three quarters of the groups hold the cell's centre,
// or of a sample of the groups are left after the nearest one.  A sphere's
// triangles shuffled, whole calls for 8,192 / 131,072 of them: 0.50 / 4.0 ms shared,
// 0.80 / 9.0 ms each wave for itself (0.32 / 0.68 ms in surface order).
// qd[cand][i-1] = q or -1; cnt[cand] = number of links of the cell.
__global__ __launch_bounds__(kLinkThreads) void KNearest(const int2* cand, int64_t ncand, int n, const double* bounds,
                                                         const uint8_t* material, const double* tris, int64_t ntri,
                                                         const double* gbox, int64_t ngroup, double* qd, int* cnt) {
  constexpr int kWaves = kLinkThreads / 64;
  __shared__ double staged[kLinkThreads * 9];
  __shared__ double sbox[6][kLinkThreads];
  __shared__ int left[kWaves];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t ci = static_cast<int64_t>(blockIdx.x) * kWaves + wave;
  const bool live = ci < ncand;  // waves without a cell only help to share triangles
  const int2 ce = cand[live ? ci : ncand - 1];
  const int b = ce.x, c = ce.y;
  const int i = c / (n * n), j = (c / n) % n, k = c % n;
  const double* bb = bounds + 6 * static_cast<size_t>(b);
  const double dx = (bb[3] - bb[0]) / static_cast<double>(n);
  const double dy = (bb[4] - bb[1]) / static_cast<double>(n);
  const double dz = (bb[5] - bb[2]) / static_cast<double>(n);
  // CellCenter (bouzidi_link_data.cpp:85-94)
  const double p[3] = {bb[0] + (static_cast<double>(i) + 0.5) * dx, bb[1] + (static_cast<double>(j) + 0.5) * dy,
                       bb[2] + (static_cast<double>(k) + 0.5) * dz};
  double bd = DBL_MAX;      // this lane's best
  double pb = DBL_MAX;      // the wave's best
  int64_t bt = INT64_MAX;
  double w[3] = {p[0], p[1], p[2]};
  const int64_t gs = GroupSize(ntri);
  auto lower = [&](int64_t g) {
    double bx[6];
#pragma unroll
    for (int d = 0; d < 6; ++d) bx[d] = gbox[d * ngroup + g];
    return BoxDistance2(bx, p);
  };
  // tests triangle t (v[9]); true where it is nearer than the wave's best
  auto test = [&](const double* v, int64_t t) {
    double q[3];
    TriClosest(v, p, q);
    const double d2 = (p[0] - q[0]) * (p[0] - q[0]) + (p[1] - q[1]) * (p[1] - q[1]) +
                      (p[2] - q[2]) * (p[2] - q[2]);
    if (!(d2 < bd || (d2 == bd && t < bt && bt != INT64_MAX))) return false;  // the first of equals
    bd = d2;
    bt = t;
    w[0] = q[0];
    w[1] = q[1];
    w[2] = q[2];
    return d2 < pb;
  };
  auto lower_best = [&]() {
    pb = bd;
    for (int off = 32; off > 0; off >>= 1) pb = fmin(pb, __shfl_xor(pb, off));
  };
  // tests the groups whose bits are set from group g0 on; lb: the box distance of
  // group g0 + lane, by which groups drop out as the best point gets nearer
  auto search = [&](int64_t g0, uint64_t todo, double lb) {
    while (todo) {
      const int64_t t0 = (g0 + __builtin_ctzll(todo)) * gs, t1 = ntri < t0 + gs ? ntri : t0 + gs;
      todo &= todo - 1;
      bool nearer = false;
      for (int64_t t = t0 + lane; t < t1; t += 64) {
        double v[9], bx[6];
#pragma unroll
        for (int e = 0; e < 9; ++e) v[e] = tris[9 * t + e];
        TriBox(v, bx);
        if (!(BoxDistance2(bx, p) > fmin(bd, pb))) nearer = test(v, t) || nearer;
      }
      if (__any(nearer)) {
        lower_best();
        todo &= __ballot(!(lb > pb));
      }
    }
  };
  int64_t first = -1;  // the group searched first
  int kept = 64;       // of 64 groups, how many are still to be searched
  if (ngroup > 0) {
    double near = INFINITY;
    int64_t inside = 0;  // groups whose box holds p, which never drop out
    for (int64_t g0 = 0; g0 < ngroup; g0 += 64) {
      const int64_t g = g0 + lane;
      const double lb = g < ngroup ? lower(g) : INFINITY;
      inside += __popcll(__ballot(lb == 0.0));
      if (lb < near) {
        near = lb;
        first = g;
      }
    }
    if (4 * inside > 3 * ngroup) {
      first = -1;
    } else {
      if (first < 0) first = 0;
      for (int off = 32; off > 0; off >>= 1) {
        const double od = __shfl_xor(near, off);
        const int64_t og = __shfl_xor(first, off);
        if (od < near || (od == near && og < first)) {
          near = od;
          first = og;
        }
      }
      search(first, 1, 0.0);
      kept = ngroup > 8 ? __popcll(__ballot(!(lower(lane * ngroup / 64) > pb))) : 0;
    }
  }
  bool share = ngroup == 0;
  if (!share) {
    if (lane == 0) left[wave] = live ? kept : 0;
    __syncthreads();
    int sum = 0;
    for (int k = 0; k < kWaves; ++k) sum += left[k];
    share = sum > 48 * static_cast<int>(ncand - (ci - wave) < kWaves ? ncand - (ci - wave) : kWaves);
  }
  if (share) {
    for (int64_t base = 0; base < ntri; base += kLinkThreads) {
      const int nt = static_cast<int>(ntri - base < kLinkThreads ? ntri - base : kLinkThreads);
      __syncthreads();  // the triangles before are no longer read
      for (int e = threadIdx.x; e < 9 * nt; e += kLinkThreads) staged[e] = tris[9 * base + e];
      if (static_cast<int>(threadIdx.x) < nt) {
        double bx[6];
        TriBox(tris + 9 * (base + threadIdx.x), bx);
#pragma unroll
        for (int d = 0; d < 6; ++d) sbox[d][threadIdx.x] = bx[d];
      }
      __syncthreads();
      bool nearer = false;
      for (int r = lane; r < nt; r += 64) {
        double bx[6];
#pragma unroll
        for (int d = 0; d < 6; ++d) bx[d] = sbox[d][r];
        if (!(BoxDistance2(bx, p) > fmin(bd, pb))) nearer = test(staged + 9 * r, base + r) || nearer;
      }
      if (__any(nearer)) lower_best();
    }
  } else if (live) {
    for (int64_t g0 = 0; g0 < ngroup; g0 += 64) {
      const int64_t g = g0 + lane;
      const double lb = lower(g < ngroup ? g : 0);
      const uint64_t todo = __ballot(g < ngroup && g != first && !(lb > pb));
      if (todo) search(g0, todo, lb);
    }
  }
  if (!live) return;
  // smallest distance over the wave, ties to the lowest triangle index
  for (int off = 32; off > 0; off >>= 1) {
    const double od = __shfl_xor(bd, off);
    const int64_t ot = __shfl_xor(bt, off);
    const double o0 = __shfl_xor(w[0], off), o1 = __shfl_xor(w[1], off), o2 = __shfl_xor(w[2], off);
    if (od < bd || (od == bd && ot < bt)) {
      bd = od;
      bt = ot;
      w[0] = o0;
      w[1] = o1;
      w[2] = o2;
    }
  }
  bool valid = false;
  double qv = -1.0;
  if (lane < kQ - 1) {
    const int ip = lane + 1;
    const int o = Opp(ip);
    const int ex = Cx(o), ey = Cy(o), ez = Cz(o);
    const int ni = i + ex, nj = j + ey, nk = k + ez;
    const uint8_t* mat = material + static_cast<size_t>(b) * n * n * n;
    if (ni >= 0 && ni < n && nj >= 0 && nj < n && nk >= 0 && nk < n && SolidLike(Mat(mat, n, ni, nj, nk))) {
      const double dir_x = static_cast<double>(ex) * dx;
      const double dir_y = static_cast<double>(ey) * dx;
      const double dir_z = static_cast<double>(ez) * dx;
      const double dn2 = dir_x * dir_x + dir_y * dir_y + dir_z * dir_z;
      if (dn2 > 1.0e-30) {
        const double tx = w[0] - p[0], ty = w[1] - p[1], tz = w[2] - p[2];
        const double proj = (tx * dir_x + ty * dir_y + tz * dir_z) / dn2;
        if (proj > 1.0e-8 && proj < 1.0 - 1.0e-8) {
          valid = true;
          qv = proj;
        }
      }
    }
    qd[ci * (kQ - 1) + lane] = qv;
  }
  const uint64_t m = __ballot(valid);
  if (lane == 0) cnt[ci] = __popcll(m);
}

// One wave per candidate: its links at offset[cand], population order.
__global__ __launch_bounds__(kLinkThreads) void KEmit(const int2* cand, int64_t ncand, const double* qd,
                                                      const int64_t* offset, int32_t* links, double* q) {
  const int lane = threadIdx.x & 63;
  const int64_t ci = static_cast<int64_t>(blockIdx.x) * (kLinkThreads / 64) + (threadIdx.x >> 6);
  if (ci >= ncand) return;
  const double v = lane < kQ - 1 ? qd[ci * (kQ - 1) + lane] : -1.0;
  const bool valid = v >= 0.0;
  const uint64_t m = __ballot(valid);
  if (!valid) return;
  const int64_t at = offset[ci] + __popcll(m & ((uint64_t(1) << lane) - 1));
  const int2 e = cand[ci];
  links[3 * at] = e.x;
  links[3 * at + 1] = e.y;
  links[3 * at + 2] = lane + 1;
  q[at] = v;
}

void GroupBoxes(const double* tris, int64_t ntri, int64_t ngroup, double* gbox, hipStream_t s) {
  if (ngroup == 0) return;
  constexpr int kWaves = kLinkThreads / 64;
  KGroupBox<<<static_cast<unsigned>((ngroup + kWaves - 1) / kWaves), kLinkThreads, 0, s>>>(tris, ntri, ngroup, gbox);
  LINK_CHECK(hipGetLastError());
}

struct DevBuf {
  std::vector<void*> ptrs;
  template <typename P>
  P* Get(size_t count) {
    void* p = nullptr;
    LINK_CHECK(hipMalloc(&p, (count == 0 ? 1 : count) * sizeof(P)));
    ptrs.push_back(p);
    return static_cast<P*>(p);
  }
  // Teardown: a failed release cannot be reported from here.
  ~DevBuf() {
    for (void* p : ptrs) (void)hipFree(p);
  }
};

struct Stream {
  hipStream_t s = nullptr;
  Stream() { LINK_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking)); }
  ~Stream() {
    if (s) (void)hipStreamDestroy(s);  // teardown
  }
};

void BuildLinks(int32_t nb, int32_t n, const double* bounds, const uint8_t* material, int64_t ntri,
                const double* tris, int64_t capacity, int64_t* num_links, int32_t* links, double* q) {
  *num_links = 0;
  if (ntri == 0 || nb == 0) return;  // soup.empty(): no links (bouzidi_link_data.cpp:147-149)
  const size_t ncell = static_cast<size_t>(n) * n * n;
  Stream st;
  DevBuf mem;
  double* d_bounds = mem.Get<double>(6 * static_cast<size_t>(nb));
  uint8_t* d_mat = mem.Get<uint8_t>(ncell * nb);
  double* d_tris = mem.Get<double>(9 * static_cast<size_t>(ntri));
  int* d_counts = mem.Get<int>(nb);
  int64_t* d_boff = mem.Get<int64_t>(static_cast<size_t>(nb) + 1);
  LINK_CHECK(hipMemcpyAsync(d_bounds, bounds, 6 * sizeof(double) * nb, hipMemcpyHostToDevice, st.s));
  LINK_CHECK(hipMemcpyAsync(d_mat, material, ncell * nb, hipMemcpyHostToDevice, st.s));
  LINK_CHECK(hipMemcpyAsync(d_tris, tris, 9 * sizeof(double) * ntri, hipMemcpyHostToDevice, st.s));
  KCandidates<false><<<nb, kLinkThreads, 0, st.s>>>(n, d_mat, d_counts, nullptr, nullptr);
  LINK_CHECK(hipGetLastError());
  KScan<<<1, 1024, 0, st.s>>>(d_counts, nb, d_boff);
  LINK_CHECK(hipGetLastError());
  int64_t ncand = 0;
  LINK_CHECK(hipMemcpyAsync(&ncand, d_boff + nb, sizeof(int64_t), hipMemcpyDeviceToHost, st.s));
  LINK_CHECK(hipStreamSynchronize(st.s));
  if (ncand == 0) return;
  const int64_t ngroup = GroupCount(ntri);
  double* d_gbox = mem.Get<double>(6 * static_cast<size_t>(ngroup) + ncand);  // and the candidates
  int2* d_cand = reinterpret_cast<int2*>(d_gbox + 6 * ngroup);
  GroupBoxes(d_tris, ntri, ngroup, d_gbox, st.s);
  KCandidates<true><<<nb, kLinkThreads, 0, st.s>>>(n, d_mat, nullptr, d_boff, d_cand);
  LINK_CHECK(hipGetLastError());
  double* d_qd = mem.Get<double>(static_cast<size_t>(ncand) * (kQ - 1));
  int* d_cnt = mem.Get<int>(ncand);
  int64_t* d_loff = mem.Get<int64_t>(static_cast<size_t>(ncand) + 1);
  const int64_t waves_per_wg = kLinkThreads / 64;
  const unsigned grid = static_cast<unsigned>((ncand + waves_per_wg - 1) / waves_per_wg);
  KNearest<<<grid, kLinkThreads, 0, st.s>>>(d_cand, ncand, n, d_bounds, d_mat, d_tris, ntri, d_gbox, ngroup, d_qd,
                                            d_cnt);
  LINK_CHECK(hipGetLastError());
  KScan<<<1, 1024, 0, st.s>>>(d_cnt, ncand, d_loff);
  LINK_CHECK(hipGetLastError());
  int64_t total = 0;
  LINK_CHECK(hipMemcpyAsync(&total, d_loff + ncand, sizeof(int64_t), hipMemcpyDeviceToHost, st.s));
  LINK_CHECK(hipStreamSynchronize(st.s));
  *num_links = total;
  if (links == nullptr && q == nullptr) return;  // count query
  if (capacity < total) throw std::invalid_argument("link capacity smaller than the number of links");
  if (total == 0) return;
  int32_t* d_links = mem.Get<int32_t>(3 * static_cast<size_t>(total));
  double* d_q = mem.Get<double>(total);
  KEmit<<<grid, kLinkThreads, 0, st.s>>>(d_cand, ncand, d_qd, d_loff, d_links, d_q);
  LINK_CHECK(hipGetLastError());
  LINK_CHECK(hipMemcpyAsync(links, d_links, 3 * sizeof(int32_t) * total, hipMemcpyDeviceToHost, st.s));
  LINK_CHECK(hipMemcpyAsync(q, d_q, sizeof(double) * total, hipMemcpyDeviceToHost, st.s));
  LINK_CHECK(hipStreamSynchronize(st.s));
}

// ---- no-allocation form: every scratch buffer of the build lives in one
// file-scope device array per GPU, sized for at most kNoAllocMaxBlocks
// blocks and kNoAllocMaxCandidates candidate cells.
constexpr int64_t kNoAllocMaxBlocks = 16384;
constexpr int64_t kNoAllocMaxCandidates = 65536;

constexpr size_t Align256(size_t b) { return (b + 255) & ~static_cast<size_t>(255); }
constexpr size_t kScrCounts = 0;
constexpr size_t kScrBoff = kScrCounts + Align256(sizeof(int) * kNoAllocMaxBlocks);
constexpr size_t kScrCand = kScrBoff + Align256(sizeof(int64_t) * (kNoAllocMaxBlocks + 1));
constexpr size_t kScrQd = kScrCand + Align256(sizeof(int2) * kNoAllocMaxCandidates);
constexpr size_t kScrCnt = kScrQd + Align256(sizeof(double) * (kQ - 1) * kNoAllocMaxCandidates);
constexpr size_t kScrLoff = kScrCnt + Align256(sizeof(int) * kNoAllocMaxCandidates);
constexpr size_t kScrGbox = kScrLoff + Align256(sizeof(int64_t) * (kNoAllocMaxCandidates + 1));
constexpr size_t kScratchBytes = kScrGbox + Align256(6 * sizeof(double) * kMaxGroups);

}  // namespace

// ~11.7 MB per GPU, held until the process ends.  In host code this name is
// only a symbol handle: its device address comes from hipGetSymbolAddress.
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned char* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current GPU, looked up once per device.
unsigned char* ScratchOnCurrentDevice() {
  int dev = 0;
  LINK_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) throw std::runtime_error("device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    LINK_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    g_scratch_ptr[dev] = static_cast<unsigned char*>(p);
  }
  return g_scratch_ptr[dev];
}

void BuildLinksNoAlloc(int32_t nb, int32_t n, const double* d_bounds, const uint8_t* d_mat, int64_t ntri,
                       const double* d_tris, int64_t capacity, int64_t* num_links, int32_t* d_links, double* d_q,
                       hipStream_t s) {
  *num_links = 0;
  if (nb > kNoAllocMaxBlocks) throw std::invalid_argument("more blocks than the no-allocation scratch holds (16384)");
  if (ntri == 0 || nb == 0) return;  // soup.empty(): no links (bouzidi_link_data.cpp:147-149)
  unsigned char* base = ScratchOnCurrentDevice();
  int* d_counts = reinterpret_cast<int*>(base + kScrCounts);
  int64_t* d_boff = reinterpret_cast<int64_t*>(base + kScrBoff);
  int2* d_cand = reinterpret_cast<int2*>(base + kScrCand);
  double* d_qd = reinterpret_cast<double*>(base + kScrQd);
  int* d_cnt = reinterpret_cast<int*>(base + kScrCnt);
  int64_t* d_loff = reinterpret_cast<int64_t*>(base + kScrLoff);
  // every scratch word read below is written first in this call
  KCandidates<false><<<nb, kLinkThreads, 0, s>>>(n, d_mat, d_counts, nullptr, nullptr);
  LINK_CHECK(hipGetLastError());
  KScan<<<1, 1024, 0, s>>>(d_counts, nb, d_boff);
  LINK_CHECK(hipGetLastError());
  int64_t ncand = 0;
  LINK_CHECK(hipMemcpyAsync(&ncand, d_boff + nb, sizeof(int64_t), hipMemcpyDeviceToHost, s));
  LINK_CHECK(hipStreamSynchronize(s));
  if (ncand == 0) return;
  if (ncand > kNoAllocMaxCandidates)
    throw std::invalid_argument("more candidate cells than the no-allocation scratch holds (65536)");
  KCandidates<true><<<nb, kLinkThreads, 0, s>>>(n, d_mat, nullptr, d_boff, d_cand);
  LINK_CHECK(hipGetLastError());
  const int64_t waves_per_wg = kLinkThreads / 64;
  const unsigned grid = static_cast<unsigned>((ncand + waves_per_wg - 1) / waves_per_wg);
  const int64_t ngroup = GroupCount(ntri);
  double* d_gbox = reinterpret_cast<double*>(base + kScrGbox);
  GroupBoxes(d_tris, ntri, ngroup, d_gbox, s);
  KNearest<<<grid, kLinkThreads, 0, s>>>(d_cand, ncand, n, d_bounds, d_mat, d_tris, ntri, d_gbox, ngroup, d_qd, d_cnt);
  LINK_CHECK(hipGetLastError());
  KScan<<<1, 1024, 0, s>>>(d_cnt, ncand, d_loff);
  LINK_CHECK(hipGetLastError());
  int64_t total = 0;
  LINK_CHECK(hipMemcpyAsync(&total, d_loff + ncand, sizeof(int64_t), hipMemcpyDeviceToHost, s));
  LINK_CHECK(hipStreamSynchronize(s));
  *num_links = total;
  if (d_links == nullptr && d_q == nullptr) return;  // count query
  if (capacity < total) throw std::invalid_argument("link capacity smaller than the number of links");
  if (total == 0) return;
  KEmit<<<grid, kLinkThreads, 0, s>>>(d_cand, ncand, d_qd, d_loff, d_links, d_q);
  LINK_CHECK(hipGetLastError());
  LINK_CHECK(hipStreamSynchronize(s));
}

}  // namespace
}  // namespace octlb

extern "C" int octlb_build_links_noalloc(int32_t num_blocks, int32_t n, const double* bounds,
                                         const uint8_t* material, int64_t num_triangles, const double* triangles,
                                         int64_t capacity, int64_t* num_links, int32_t* links, double* q,
                                         void* stream) {
  using namespace octlb;
  if (!num_links) return SetError(OCTLB_EINVAL, "null num_links");
  *num_links = 0;
  if (num_blocks < 0 || n < 1 || n > 1024 || num_triangles < 0 || capacity < 0)
    return SetError(OCTLB_EINVAL, "bad link-build sizes");
  if ((num_blocks > 0 && (!bounds || !material)) || (num_triangles > 0 && !triangles))
    return SetError(OCTLB_EINVAL, "null link-build input");
  if ((links == nullptr) != (q == nullptr)) return SetError(OCTLB_EINVAL, "links and q must both be given");
  try {
    BuildLinksNoAlloc(num_blocks, n, bounds, material, num_triangles, triangles, capacity, num_links, links, q,
                      static_cast<hipStream_t>(stream));
  } catch (const std::invalid_argument& e) {
    return SetError(OCTLB_EINVAL, e.what());
  } catch (const std::exception& e) {
    return SetError(OCTLB_EHIP, e.what());
  }
  return OCTLB_OK;
}

extern "C" int octlb_build_links(int32_t num_blocks, int32_t n, const double* bounds, const uint8_t* material,
                                 int64_t num_triangles, const double* triangles, int64_t capacity,
                                 int64_t* num_links, int32_t* links, double* q) {
  using namespace octlb;
  if (!num_links) return SetError(OCTLB_EINVAL, "null num_links");
  *num_links = 0;
  if (num_blocks < 0 || n < 1 || n > 1024 || num_triangles < 0 || capacity < 0)
    return SetError(OCTLB_EINVAL, "bad link-build sizes");
  if ((num_blocks > 0 && (!bounds || !material)) || (num_triangles > 0 && !triangles))
    return SetError(OCTLB_EINVAL, "null link-build input");
  if ((links == nullptr) != (q == nullptr)) return SetError(OCTLB_EINVAL, "links and q must both be given");
  try {
    BuildLinks(num_blocks, n, bounds, material, num_triangles, triangles, capacity, num_links, links, q);
  } catch (const std::invalid_argument& e) {
    return SetError(OCTLB_EINVAL, e.what());
  } catch (const std::bad_alloc&) {
    return SetError(OCTLB_ENOMEM, "host allocation failed");
  } catch (const std::exception& e) {
    return SetError(OCTLB_EHIP, e.what());
  }
  return OCTLB_OK;
}
