// shortrange.hip -- TreePM short-range force by direct summation over a
// chaining mesh.
//
// Reference: crates/gadget-ng-treepm/src/short_range.rs (pair law :384-398,
// minimum image :53-63, periodic walk :232-330).  The reference walks an
// octree and replaces small nodes by their monopole; here every pair inside
// r_cut is summed exactly, which is the quantity that walk approximates.
//
// Method:
//   1. every particle gets its cell in a chaining mesh of nc^3 cells of side
//      L/nc >= r_cut (nc >= 3); a stable radix sort by cell (sort.hpp) puts
//      them in cell order with ascending particle index inside each cell; the
//      cell offsets are looked up in the sorted cells (a binary search per
//      cell: no atomics, which a clump's particles would all aim at one
//      counter); the particles are gathered as float4 (position relative to
//      the corner of their unwrapped cell, m) plus the original index.  The
//      order of every sum is then fixed, so the result is bit-identical from
//      call to call.  Lengths are divided by r_u, the power of two next to
//      r_cut, and masses by a power of two just above the largest one: both
//      are exact, so nothing is rounded differently, and whatever the caller's
//      units no FP32 intermediate leaves its range (m in kg, g or solar masses
//      times 1 / r^3 in m or cm does);
//   2. the work list is (cell, chunk of 64 particles).  A chunk with more than
//      kHeavy particles in reach is heavy: its workgroup's four wavefronts
//      each take a quarter of every neighbour cell and their sums are added in
//      order; these come first in the grid.  The other chunks are one
//      wavefront each.  The lengths stay on the device and the grid covers the
//      most there can be;
//   3. one wavefront takes a chunk, one particle per lane, and walks the
//      particles of the 27 neighbour cells: FP32 inside 256 of them, FP64
//      across.  The neighbours are wave-uniform, so they come through the
//      scalar cache into scalar registers and the loop needs no LDS staging,
//      barrier or per-pair vector load.  A neighbour cell at offset d (cells,
//      each component -1, 0 or 1) holds its particles at rel + d * side from
//      the lane's cell corner, so the displacement needs no per-pair minimum
//      image: every pair within r_cut <= L/nc <= L/3 is its own minimum image
//      in that form, and no pair outside the cut comes inside it.
//
// The pair law is bound by VALU issue, a transcendental counting as four.
// With r in units of r_u and u = r^2 / (2 r_s^2), S(r) / r^3 is
//   u < 2:  1/r^3 - L(r^2),  L = (1 - S) / r^3 analytic in r^2 (the reference
//           factor, u < 1.25: 1/r^2 (1/r - E(r^2)), E = erf / r),
//   else:   F(r^2) itself, smooth there and free of cancellation,
// with L, E and F from a table of 1025 quadratics over r^2 in LDS (FP64
// coefficients at Chebyshev nodes, relative error below 1e-7): one rsq, one
// 16-byte LDS read and 16 other operations per accepted pair, against rsq,
// rcp, exp and 24 others for a rational erfc of absolute error 1.5e-7.
// 96^3 particles (30 % in Plummer spheres), r_cut = 5 r_s = 6.25 cells:
// 17.0 ms with LDS-staged neighbours, that erfc and one workgroup per 256
// particles; 13.3 with scalar neighbours and the table; 6.3 with heavy chunks
// spread over four wavefronts (8.1 with the erfc formula there).
// Beyond u = 16 (r_cut above 5.6 r_s) a table uniform in r^2 would be too coarse
// where F is steep, below u = 4; there it has 2049 entries uniform in r, for five
// operations a pair more, and ends at the latest where F leaves FP32, at x = 9.3.
// 2e5 particles at r_cut = 6 r_s: 1.64 ms with the device library's erfc in the
// place of a table, 0.91 so (at 5.6 r_s 0.87).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>
#include <new>
#include <string>
#include <type_traits>

#include "../../include/gng_learned.h"
#include "sort.hpp"
#include "status.hpp"

namespace gng {
namespace sr {

constexpr int kChunk = 64;          // particles per work item: one wavefront
constexpr unsigned kHeavy = 8192;   // particles in the 27 cells above which a chunk takes a workgroup
constexpr int kAhead = 8;           // entries past the last particle that may be loaded (never used)

// Workgroups per row of the force launch.  A launch dimension is cut, without
// an error, at 2^32 work items, 2^24 of these workgroups, which 7e8 particles
// can make.
constexpr long long kRow = 1 << 16;

// The unwrapped chaining-mesh cell floor(v nc / L) of one coordinate, in FP64
// (cs = nc / L), and its index wrapped into [0, nc); a non-finite coordinate
// lands in cell 0.  k_cells and k_gather both start from cell_floor, so a
// particle's cell and its in-cell offset always agree.
__device__ __forceinline__ double cell_floor(float v, double cs) { return floor((double)v * cs); }

__device__ __forceinline__ int wrap_cell(double fl, int nc) {
  double c = fmod(fl, (double)nc);
  if (c < 0.0) c += (double)nc;
  return c >= 0.0 && c < (double)nc ? (int)c : 0;
}

__global__ __launch_bounds__(256) void k_cells(const float* __restrict__ x, const float* __restrict__ y,
                                               const float* __restrict__ z, long long n, int nc, double cs,
                                               unsigned* __restrict__ cell_of) {
  const long long p = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= n) return;
  const int cx = wrap_cell(cell_floor(x[p], cs), nc), cy = wrap_cell(cell_floor(y[p], cs), nc),
            cz = wrap_cell(cell_floor(z[p], cs), nc);
  cell_of[p] = (unsigned)(((long long)cz * nc + cy) * nc + cx);
}

struct Counters {
  unsigned long long pairs;  // evaluated pairs
  unsigned heavy, light;     // work items of each kind
  unsigned mmax;             // float bits of the largest finite |m|
  unsigned odd;              // 1: a mass is infinite or NaN
};

// The masses' power of two: m / 2^mass_exponent lies in (-1, 1).
__device__ __forceinline__ int mass_exponent(const Counters* cnt) {
  int e = 0;
  (void)frexpf(__uint_as_float(cnt->mmax), &e);
  return e;
}

// off[c] = first particle of cell c in the sorted cells (off[ncell] = n), and
// the counters reset.
__global__ __launch_bounds__(256) void k_offsets(const unsigned* __restrict__ cells, unsigned n, long long ncell,
                                                 unsigned* __restrict__ off, Counters* __restrict__ cnt) {
  const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
  if (c == 0) *cnt = Counters{0ull, 0u, 0u, 0u, 0u};
  if (c > ncell) return;
  unsigned lo = 0, hi = n;  // the first index whose cell is >= c
  while (lo < hi) {
    const unsigned mid = (lo + hi) >> 1;
    if (cells[mid] < (unsigned)c) lo = mid + 1;
    else hi = mid;
  }
  off[c] = lo;
}

// Most heavy and light work items n particles in ncell cells can make.  The
// particles in reach add up to 27 n over the cells, so at most 27 n / kHeavy
// cells are heavy.
inline long long max_heavy(long long n) { return n / kChunk + 27 * n / kHeavy + 1; }
inline long long max_light(long long n, long long ncell) { return n / kChunk + (n < ncell ? n : ncell); }

// The work items (cell, chunk): heavy ones' from the front of items, the
// others' from its back.  One atomic per wavefront and kind; the places are
// arbitrary, but no result depends on them.  The first workgroups also look
// through the n masses for the largest: one atomic each, since all of them go
// to one word, some 10 ns apart.
constexpr unsigned kMassGroups = 256;
__global__ __launch_bounds__(256) void k_items(const unsigned* __restrict__ off, int nc, long long ncell,
                                               const float* __restrict__ m, long long n, uint2* __restrict__ items,
                                               unsigned cap, Counters* __restrict__ cnt) {
  if (blockIdx.x < kMassGroups) {
    __shared__ unsigned tops[4];
    unsigned top = 0, odd = 0;
    const unsigned groups = min(gridDim.x, kMassGroups);
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += groups * 256LL) {
      const unsigned b = __float_as_uint(fabsf(m[i]));
      if (b >= 0x7F800000u) odd = 1u;
      else top = max(top, b);
    }
    if (odd) cnt->odd = 1u;
    for (int d = 32; d > 0; d >>= 1) top = max(top, __shfl_xor(top, d));
    if ((threadIdx.x & 63) == 0) tops[threadIdx.x >> 6] = top;
    __syncthreads();
    if (threadIdx.x == 0) {
      top = max(max(tops[0], tops[1]), max(tops[2], tops[3]));
      if (top) atomicMax(&cnt->mmax, top);
    }
  }
  const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const unsigned k = c < ncell ? off[c + 1] - off[c] : 0u;
  const unsigned chunks = (k + kChunk - 1) / kChunk;
  unsigned reach = 0;
  if (k) {
    const int cx = (int)(c % nc), cy = (int)((c / nc) % nc), cz = (int)(c / ((long long)nc * nc));
    for (int nb = 0; nb < 27; ++nb) {
      const int ux = (cx + nb % 3 + nc - 1) % nc, uy = (cy + nb / 3 % 3 + nc - 1) % nc, uz = (cz + nb / 9 + nc - 1) % nc;
      const long long u = ((long long)uz * nc + uy) * nc + ux;
      reach += off[u + 1] - off[u];
    }
  }
  for (int kind = 0; kind < 2; ++kind) {
    const unsigned mine = (reach > kHeavy) == (kind == 0) ? chunks : 0u;
    unsigned incl = mine;
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned t = __shfl_up(incl, d);
      if (lane >= d) incl += t;
    }
    unsigned base = 0;
    if (lane == 63 && incl != 0u) base = atomicAdd(kind == 0 ? &cnt->heavy : &cnt->light, incl);
    base = __shfl(base, 63) + incl - mine;
    for (unsigned q = 0; q < mine; ++q)
      items[kind == 0 ? base + q : cap - 1u - (base + q)] = make_uint2((unsigned)c, q);
  }
}

// sorted[i] = particle order[i] (the cell-sorted permutation): its position
// relative to the corner of its unwrapped cell, v - floor(v nc / L) L / nc,
// formed in FP64 from the same floor as k_cells' (so it is also the offset
// from the wrapped cell's corner, whatever image of the box v lies in), over
// r_u, and m over its power of two.  Powers of two keep the caller's own
// roundings: neighbours' are mostly the same one, and cancel in their
// displacement.
__global__ __launch_bounds__(256) void k_gather(const float* __restrict__ x, const float* __restrict__ y,
                                                const float* __restrict__ z, const float* __restrict__ m, long long n,
                                                const unsigned* __restrict__ order, double cs, double cside,
                                                double inv_ru, const Counters* __restrict__ cnt,
                                                float4* __restrict__ sorted, unsigned* __restrict__ sidx) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const unsigned p = order[i];
  const float vx = x[p], vy = y[p], vz = z[p];
  sorted[i] = make_float4((float)(((double)vx - cell_floor(vx, cs) * cside) * inv_ru),
                          (float)(((double)vy - cell_floor(vy, cs) * cside) * inv_ru),
                          (float)(((double)vz - cell_floor(vz, cs) * cside) * inv_ru),
                          ldexpf(m[p], -mass_exponent(cnt)));
  sidx[i] = p;
}

// Lengths in units of r_u.
struct Params {
  float csize;     // chaining cell side
  float rc2;       // r_cut^2
  double g;        // G / r_u^2, taken into the sums with the masses' power of two
  float eps2;
  float tscale;    // table entries per unit of r^2, or of r
  int nc;
  unsigned items;  // capacity of the work list
};

// Entries 0 .. kTable, entry i around r^2 = i / tscale up to u = kTableU, else
// around r = i / tscale, and the last one, 0, for all r from kWideX on.
template <bool WIDE>
constexpr int kTable = WIDE ? 2048 : 1024;
constexpr double kTableU = 16.0, kWideX = 9.3;
// where the law passes from the subtraction to F: the subtraction loses 1 / S of
// a rounding (4 at u = 2 for the exact split; erfc falls faster: 9 at 1.25, 22
// at 2), the quadratics of F get worse as u^-3 (6e-8 at 1.25 with u to 12.5)
template <int KERNEL>
constexpr double kNearU = KERNEL == GNG_SR_EXACT ? 2.0 : 1.25;

// The smooth part of the pair law at r^2 = v (see the head of this file): -L
// or E below u = kNearU (near), F above.  1 - S and erf by their power series
// in u, which also continue them to the v < 0 of entry 0's left node.
template <int KERNEL>
__device__ double smooth_part(double v, double kappa2, bool near) {
  const double u = kappa2 * v, k1 = sqrt(kappa2);
  if (near) {
    double term = 1.0, sum = 0.0;
    for (int m = 0; m < 40; ++m) {
      sum += term / (double)(2 * m + (KERNEL == GNG_SR_EXACT ? 3 : 1));
      term *= -u / (double)(m + 1);
    }
    // 2 / sqrt(pi); the exact split's is negated, so that it is only added
    return KERNEL == GNG_SR_EXACT ? -2.0 * 1.1283791670955126 * sum * k1 * kappa2 : 1.1283791670955126 * sum * k1;
  }
  const double x = sqrt(u);
  const double S = erfc(x) + (KERNEL == GNG_SR_EXACT ? 1.1283791670955126 * x * exp(-u) : 0.0);
  return S / (v * sqrt(v));
}

// Entry i: c0 + d (c1 + d c2) with d = r^2 tscale - i (WIDE: r tscale - i) in
// [-1/2, 1/2], through the Chebyshev nodes of that interval, and 1 where the
// entry is near, else 0.
template <int KERNEL, bool WIDE>
__global__ __launch_bounds__(256) void k_table(double kappa2, double tscale, float4* __restrict__ table) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i > kTable<WIDE>) return;
  const double c = (double)i / tscale, d0 = 0.43301270189221932;  // sqrt(3) / 4
  const auto square = [](double t) { return WIDE ? t * t : t; };
  const bool near = kappa2 * square(c) < kNearU<KERNEL>;
  const double f0 = smooth_part<KERNEL>(square(c), kappa2, near),
               fp = smooth_part<KERNEL>(square(c + d0 / tscale), kappa2, near),
               fm = smooth_part<KERNEL>(square(c - d0 / tscale), kappa2, near);
  if (WIDE && i == kTable<WIDE>) {
    table[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    return;
  }
  table[i] = make_float4((float)f0, (float)((fp - fm) / (2.0 * d0)), (float)((fp + fm - 2.0 * f0) / (2.0 * d0 * d0)),
                         near ? 1.0f : 0.0f);
}

// SOFT: the softening and the masses' unit keep a coincident pair's factor
// below 1e18, so that its zero displacement alone makes it vanish, unless a
// mass is not finite.  The comparison this saves is 4 % of the kernel (96^3
// clustered particles: 6.78 against 6.46 ms).
template <int KERNEL, bool WIDE, bool SOFT>
__global__ __launch_bounds__(256) void k_force(const float4* __restrict__ sorted, const unsigned* __restrict__ sidx,
                                               const unsigned* __restrict__ off, const uint2* __restrict__ items,
                                               const float4* __restrict__ table, const Params pr,
                                               float* __restrict__ ax, float* __restrict__ ay, float* __restrict__ az,
                                               Counters* __restrict__ cnt) {
  constexpr int kSums = 3 * 3 * kChunk;  // doubles: three wavefronts' sums of a heavy chunk
  __shared__ float4 tab[kTable<WIDE> + 1];
  static_assert(kSums / 2 <= kTable<WIDE>, "the sums reuse the table's LDS");
  const unsigned heavy = cnt->heavy, light = cnt->light, group = blockIdx.y * gridDim.x + blockIdx.x;
  const bool whole = group < heavy;  // uniform: the workgroup is one heavy chunk
  if (!whole && (group - heavy) * 4u >= light) return;
  for (int e = threadIdx.x; e <= kTable<WIDE>; e += 256) tab[e] = table[e];
  __syncthreads();
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned w = whole ? group : (group - heavy) * 4u + wave;
  if (!whole && w >= light) return;
  const uint2 item = items[whole ? w : pr.items - 1u - w];
  const unsigned cell = __builtin_amdgcn_readfirstlane(item.x), i0 = off[cell] + item.y * kChunk;
  const unsigned i = i0 + (threadIdx.x & 63u), iend = off[cell + 1];
  const bool live = i < iend;
  const float4 pi = live ? sorted[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const int nc = pr.nc;
  const int cx = (int)(cell % (unsigned)nc), cy = (int)((cell / (unsigned)nc) % (unsigned)nc),
            cz = (int)(cell / ((unsigned)nc * (unsigned)nc));
  double sx = 0.0, sy = 0.0, sz = 0.0;
  unsigned long long seen = 0;
  // keep: coincident pairs need no test
  const auto walk = [&](auto keep) {
    for (int nb = 0; nb < 27; ++nb) {
      const int ox = nb % 3 - 1, oy = (nb / 3) % 3 - 1, oz = nb / 9 - 1;
      // the lane's particle relative to this neighbour cell's corner
      const float px = pi.x - (float)ox * pr.csize, py = pi.y - (float)oy * pr.csize, pz = pi.z - (float)oz * pr.csize;
      int ux = cx + ox, uy = cy + oy, uz = cz + oz;
      ux += ux < 0 ? nc : 0;
      ux -= ux >= nc ? nc : 0;
      uy += uy < 0 ? nc : 0;
      uy -= uy >= nc ? nc : 0;
      uz += uz < 0 ? nc : 0;
      uz -= uz >= nc ? nc : 0;
      const unsigned nbc = ((unsigned)uz * (unsigned)nc + (unsigned)uy) * (unsigned)nc + (unsigned)ux;
      unsigned j0 = off[nbc], j1 = off[nbc + 1];
      seen += j1 - j0;
      if (whole) {
        const unsigned q = (j1 - j0 + 3u) / 4u;
        j0 = min(j1, j0 + wave * q);
        j1 = min(j1, j0 + q);
      }
      float fx = 0.0f, fy = 0.0f, fz = 0.0f;
      auto pair = [&](const float4 pj) {
        const float dx = pj.x - px, dy = pj.y - py, dz = pj.z - pz;
        const float r2b = dx * dx + dy * dy + dz * dz;
        // r2b > 0 skips coincident pairs and the particle itself (for the
        // lane's own cell the offset is 0 * csize = 0, so its displacement
        // is exactly zero)
        if (r2b <= pr.rc2 && (decltype(keep)::value || r2b > 0.0f)) {
          const float r2 = r2b + pr.eps2;
          const float rinv = __builtin_amdgcn_rsqf(r2);
          float at = r2;
          if constexpr (WIDE) {
            at = r2 * rinv;
            at = fmaf(fmaf(-at, at, r2), 0.5f * rinv, at);  // rsq's last bits count 2 u times in F
          }
          // adding 1.5 * 2^23 leaves rint(t) in the low mantissa bits
          float tb = fmaf(at, pr.tscale, 12582912.0f);
          if constexpr (WIDE) tb = fminf(tb, 12582912.0f + (float)kTable<WIDE>);
          const float d = fmaf(at, pr.tscale, -(tb - 12582912.0f));
          const float4 q = tab[__float_as_uint(tb) - 0x4B400000u];
          const float smooth = fmaf(d, fmaf(d, q.z, q.y), q.x);
          float f;
          if constexpr (KERNEL == GNG_SR_EXACT)
            f = fmaf(q.w, rinv * rinv * rinv, smooth);
          else
            f = q.w != 0.0f ? rinv * rinv * (rinv - smooth) : smooth;
          f *= pj.w;
          fx += f * dx;
          fy += f * dy;
          fz += f * dz;
        }
      };
      // four particles at a time, the next four's scalar loads in flight
      // (sorted has kAhead entries past the last particle)
      unsigned j = j0;
      float4 n0 = sorted[j], n1 = sorted[j + 1], n2 = sorted[j + 2], n3 = sorted[j + 3];
      while (j < j1) {
        const unsigned stop = j1 - j > 256u ? j + 256u : j1;
        for (; j + 4 <= stop; j += 4) {
          const float4 p0 = n0, p1 = n1, p2 = n2, p3 = n3;
          n0 = sorted[j + 4];
          n1 = sorted[j + 5];
          n2 = sorted[j + 6];
          n3 = sorted[j + 7];
          pair(p0);
          pair(p1);
          pair(p2);
          pair(p3);
        }
        for (; j < stop; ++j) pair(sorted[j]);  // only before the end of the cell
        sx += fx;
        sy += fy;
        sz += fz;
        fx = fy = fz = 0.0f;
      }
    }
  };
  if (SOFT && cnt->odd == 0u) walk(std::true_type());
  else walk(std::false_type());
  if (whole) {
    double* sums = reinterpret_cast<double*>(tab);
    __syncthreads();
    if (wave != 0u) {
      double* q = sums + (wave - 1u) * 3 * kChunk + (threadIdx.x & 63u);
      q[0] = sx;
      q[kChunk] = sy;
      q[2 * kChunk] = sz;
    }
    __syncthreads();
    if (wave != 0u) return;
    for (int k = 0; k < 3; ++k) {
      const double* q = sums + k * 3 * kChunk + threadIdx.x;
      sx += q[0];
      sy += q[kChunk];
      sz += q[2 * kChunk];
    }
  }
  if (live) {
    const unsigned o = sidx[i];
    const double g = ldexp(pr.g, mass_exponent(cnt));
    ax[o] = (float)(sx * g);
    ay[o] = (float)(sy * g);
    az[o] = (float)(sz * g);
  }
  // evaluated pairs: live lanes x particles seen
  if ((threadIdx.x & 63u) == 0u)
    atomicAdd(&cnt->pairs, (unsigned long long)(iend - i0 < kChunk ? iend - i0 : kChunk) * seen);
}

}  // namespace sr
}  // namespace gng

using namespace gng::sr;
using gng::fail;

struct gng_sr {
  int device = 0;
  long long cap_n = 0;
  float4* d_sorted = nullptr;
  unsigned* d_sidx = nullptr;
  unsigned* d_cell_of = nullptr;
  unsigned* d_cell_sorted = nullptr;  // radix-sort outputs
  unsigned* d_order = nullptr;
  void* d_temp = nullptr;  // radix-sort work space (sized for cap_n)
  size_t temp_bytes = 0;
  long long cap_cells = 0;
  unsigned* d_off = nullptr;
  long long cap_items = 0;
  uint2* d_items = nullptr;
  float4* d_table = nullptr;
  Counters* d_count = nullptr;
  long long last_pairs = -1;
  bool pairs_pending = false;
  std::mutex mu;
  hipEvent_t done_ev = nullptr;  // end of the last call's work, on done_stream
  hipStream_t done_stream = nullptr;
  bool done_valid = false;
};

namespace {

void free_sr(gng_sr* s) {
  (void)hipFree(s->d_sorted);
  (void)hipFree(s->d_sidx);
  (void)hipFree(s->d_cell_of);
  (void)hipFree(s->d_cell_sorted);
  (void)hipFree(s->d_order);
  (void)hipFree(s->d_temp);
  (void)hipFree(s->d_off);
  (void)hipFree(s->d_items);
  (void)hipFree(s->d_table);
  (void)hipFree(s->d_count);
  if (s->done_ev) (void)hipEventDestroy(s->done_ev);
}

// Stream order for one call's work in the context's buffers: construction
// makes s wait for the previous call's work when that ran on another stream,
// destruction records the point the next call waits for.  Construct it under
// the context's lock.  A stream that is being captured cannot wait for work
// outside its graph: the caller orders the graph's launches.
struct SrOrder {
  gng_sr* sr;
  hipStream_t s;
  bool eager = true;
  hipError_t e = hipSuccess;
  SrOrder(gng_sr* sr_, hipStream_t s_) : sr(sr_), s(s_) {
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (s && hipStreamIsCapturing(s, &st) == hipSuccess) eager = st == hipStreamCaptureStatusNone;
    if (eager && sr->done_valid && sr->done_stream != s) e = hipStreamWaitEvent(s, sr->done_ev, 0);
  }
  ~SrOrder() {
    if (!eager || hipEventRecord(sr->done_ev, s) != hipSuccess) return;
    sr->done_valid = true;
    sr->done_stream = s;
  }
};

}  // namespace

namespace {

// Chaining-mesh bookkeeping shared by the entry points: cell of every particle
// and the stable cell-sorted permutation d_order (cells in d_cell_sorted).  Returns nc through *nc_out.
int cell_sort(gng_sr* sr, const float* d_x, const float* d_y, const float* d_z, int64_t n, double box_size,
              double r_cut, hipStream_t s, int* nc_out) {
  int nc = (int)std::floor(box_size / r_cut);
  if (nc > 256) nc = 256;
  const long long ncell = (long long)nc * nc * nc;
  if (n > sr->cap_n) {
    (void)hipFree(sr->d_sorted);
    (void)hipFree(sr->d_sidx);
    (void)hipFree(sr->d_cell_of);
    (void)hipFree(sr->d_cell_sorted);
    (void)hipFree(sr->d_order);
    (void)hipFree(sr->d_temp);
    sr->d_sorted = nullptr;
    sr->d_sidx = sr->d_cell_of = sr->d_cell_sorted = sr->d_order = nullptr;
    sr->d_temp = nullptr;
    sr->cap_n = 0;
    GNG_HIP(hipMalloc(&sr->d_sorted, sizeof(float4) * ((size_t)n + kAhead)));
    GNG_HIP(hipMalloc(&sr->d_sidx, sizeof(unsigned) * (size_t)n));
    GNG_HIP(hipMalloc(&sr->d_cell_of, sizeof(unsigned) * (size_t)n));
    GNG_HIP(hipMalloc(&sr->d_cell_sorted, sizeof(unsigned) * (size_t)n));
    GNG_HIP(hipMalloc(&sr->d_order, sizeof(unsigned) * (size_t)n));
    GNG_HIP(hipMalloc(&sr->d_temp, gng::radix::sort_workspace(n)));
    sr->cap_n = n;
  }
  if (ncell > sr->cap_cells) {
    (void)hipFree(sr->d_off);
    sr->d_off = nullptr;
    sr->cap_cells = 0;
    GNG_HIP(hipMalloc(&sr->d_off, sizeof(unsigned) * (size_t)(ncell + 1)));
    sr->cap_cells = ncell;
  }
  hipLaunchKernelGGL(k_cells, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, d_x, d_y, d_z, (long long)n, nc,
                     (double)nc / box_size, sr->d_cell_of);
  GNG_HIP(hipGetLastError());
  // stable LSD radix sort over the bits a cell index needs
  int end_bit = 1;
  while ((1LL << end_bit) < ncell) ++end_bit;
  GNG_HIP(gng::radix::sort_pairs(sr->d_cell_of, n, end_bit, sr->d_cell_sorted, sr->d_order, sr->d_temp, s));
  *nc_out = nc;
  return GNG_OK;
}

int check_geometry(int64_t n, double box_size, double r_cut) {
  if (n < 0) return fail(GNG_ERR_INVALID, "negative particle count");
  if (n >= (1LL << 31)) return fail(GNG_ERR_INVALID, "n of 2^31 or more is not supported");
  if (!(box_size > 0.0) || !(r_cut > 0.0)) return fail(GNG_ERR_INVALID, "box_size and r_cut must be positive");
  if (box_size < 3.0 * r_cut) return fail(GNG_ERR_INVALID, "box_size must be at least 3 r_cut");
  return GNG_OK;
}

}  // namespace

extern "C" {

int gng_sr_create(int32_t device, gng_sr** out) {
  if (!out) return fail(GNG_ERR_INVALID, "out is NULL");
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return fail(GNG_ERR_NO_DEVICE, "no HIP device");
  if (device < 0 || device >= ndev) return fail(GNG_ERR_INVALID, "device index out of range");
  GNG_HIP(hipSetDevice(device));
  gng_sr* s = new (std::nothrow) gng_sr();
  if (!s) return fail(GNG_ERR_OOM, "host allocation failed");
  s->device = device;
  if (hipEventCreateWithFlags(&s->done_ev, hipEventDisableTiming | hipEventDisableSystemFence) != hipSuccess ||
      hipMalloc(&s->d_count, sizeof(Counters)) != hipSuccess ||
      hipMalloc(&s->d_table, sizeof(float4) * (kTable<true> + 1)) != hipSuccess) {
    free_sr(s);
    delete s;
    return fail(GNG_ERR_OOM, "short-range counters");
  }
  *out = s;
  return GNG_OK;
}

void gng_sr_destroy(gng_sr* sr) {
  if (!sr) return;
  (void)hipSetDevice(sr->device);
  (void)hipDeviceSynchronize();
  free_sr(sr);
  delete sr;
}


int gng_sr_cell_order(gng_sr* sr, const float* d_x, const float* d_y, const float* d_z, int64_t n,
                      double box_size, double r_cut, uint32_t* d_order, void* stream) {
  if (!sr) return fail(GNG_ERR_INVALID, "null short-range context");
  if (int e = check_geometry(n, box_size, r_cut)) return e;
  if (n == 0) return GNG_OK;
  if (!d_x || !d_y || !d_z || !d_order) return fail(GNG_ERR_INVALID, "null array");
  std::lock_guard<std::mutex> lk(sr->mu);
  GNG_HIP(hipSetDevice(sr->device));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  SrOrder order(sr, s);
  GNG_HIP(order.e);
  int nc = 0;
  if (int e = cell_sort(sr, d_x, d_y, d_z, n, box_size, r_cut, s, &nc)) return e;
  GNG_HIP(hipMemcpyAsync(d_order, sr->d_order, sizeof(unsigned) * (size_t)n, hipMemcpyDeviceToDevice, s));
  return GNG_OK;
}

int gng_sr_accelerations(gng_sr* sr, const float* d_x, const float* d_y, const float* d_z, const float* d_m,
                         int64_t n, double box_size, double r_split, double r_cut, double eps2, double g,
                         int32_t kernel, float* d_ax, float* d_ay, float* d_az, void* stream) {
  if (!sr) return fail(GNG_ERR_INVALID, "null short-range context");
  if (int e = check_geometry(n, box_size, r_cut)) return e;
  if (!(r_split > 0.0) || !(eps2 >= 0.0)) return fail(GNG_ERR_INVALID, "r_split must be positive and eps2 non-negative");
  if (kernel != GNG_SR_EXACT && kernel != GNG_SR_REFERENCE) return fail(GNG_ERR_INVALID, "unknown split kernel");
  if (n == 0) return GNG_OK;
  if (!d_x || !d_y || !d_z || !d_m || !d_ax || !d_ay || !d_az) return fail(GNG_ERR_INVALID, "null array");
  std::lock_guard<std::mutex> lk(sr->mu);
  GNG_HIP(hipSetDevice(sr->device));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  SrOrder order(sr, s);
  GNG_HIP(order.e);
  int nc = 0;
  if (int e = cell_sort(sr, d_x, d_y, d_z, n, box_size, r_cut, s, &nc)) return e;
  const long long ncell = (long long)nc * nc * nc;
  const long long cap = max_heavy(n) + max_light(n, ncell);
  if (cap > sr->cap_items) {
    (void)hipFree(sr->d_items);
    sr->d_items = nullptr;
    sr->cap_items = 0;
    GNG_HIP(hipMalloc(&sr->d_items, sizeof(uint2) * (size_t)cap));
    sr->cap_items = cap;
  }
  // the same cs as the cell lookup (cell_sort), and the cell side
  const double cs = (double)nc / box_size, cside = box_size / (double)nc;
  const double inv_ru = std::exp2(-std::round(std::log2(r_cut)));
  hipLaunchKernelGGL(k_offsets, dim3((unsigned)((ncell + 256) / 256)), dim3(256), 0, s, sr->d_cell_sorted, (unsigned)n,
                     ncell, sr->d_off, sr->d_count);
  // a workgroup for every 256 cells, and enough of them for the masses
  const long long item_groups = std::max((ncell + 255) / 256, std::min<long long>((n + 2047) / 2048, kMassGroups));
  hipLaunchKernelGGL(k_items, dim3((unsigned)item_groups), dim3(256), 0, s, sr->d_off, nc, ncell, d_m, (long long)n,
                     sr->d_items, (unsigned)cap, sr->d_count);
  hipLaunchKernelGGL(k_gather, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, d_x, d_y, d_z, d_m, (long long)n,
                     sr->d_order, cs, cside, inv_ru, sr->d_count, sr->d_sorted, sr->d_sidx);
  const double rc = r_cut * inv_ru, rs = r_split * inv_ru, kappa2 = 0.5 / (rs * rs), e2 = eps2 * inv_ru * inv_ru;
  // the table covers r^2 <= r_cut^2 + eps^2, with room for rounding at its end
  const double r2max = rc * rc + e2;
  const bool wide = kappa2 * r2max > kTableU;
  const double tend = wide ? std::min(std::sqrt(r2max), kWideX / std::sqrt(kappa2)) : r2max;
  Params pr;
  pr.csize = (float)(cside * inv_ru);
  pr.rc2 = (float)(rc * rc);
  pr.g = g * inv_ru * inv_ru;
  pr.eps2 = (float)e2;
  pr.tscale = (float)std::min(((wide ? kTable<true> : kTable<false>) - 0.6) / tend, 1e30);  // finite however small r_s is
  pr.nc = nc;
  pr.items = (unsigned)cap;
  // 1 / r^3 stays below 1e18
  const bool soft = e2 >= 1e-12;
  const auto launch = [&](auto k, auto w) {
    constexpr int K = decltype(k)::value;
    constexpr bool W = decltype(w)::value;
    hipLaunchKernelGGL((k_table<K, W>), dim3((kTable<W> + 256) / 256), dim3(256), 0, s, kappa2, (double)pr.tscale,
                       sr->d_table);
    const long long groups = max_heavy(n) + (max_light(n, ncell) + 3) / 4;
    const dim3 grid((unsigned)std::min(groups, kRow), (unsigned)((groups + kRow - 1) / kRow));
    const auto force = soft ? k_force<K, W, true> : k_force<K, W, false>;
    hipLaunchKernelGGL(force, grid, dim3(256), 0, s, sr->d_sorted, sr->d_sidx, sr->d_off, sr->d_items, sr->d_table, pr,
                       d_ax, d_ay, d_az, sr->d_count);
  };
  const auto with_width = [&](auto k) { wide ? launch(k, std::true_type()) : launch(k, std::false_type()); };
  if (kernel == GNG_SR_EXACT) with_width(std::integral_constant<int, GNG_SR_EXACT>());
  else with_width(std::integral_constant<int, GNG_SR_REFERENCE>());
  GNG_HIP(hipGetLastError());
  sr->pairs_pending = true;
  return GNG_OK;
}

int64_t gng_sr_last_pair_count(const gng_sr* sr) {
  if (!sr) return -1;
  gng_sr* m = const_cast<gng_sr*>(sr);
  std::lock_guard<std::mutex> lk(m->mu);
  if (m->pairs_pending) {
    unsigned long long v = 0;
    if (hipSetDevice(m->device) != hipSuccess || hipDeviceSynchronize() != hipSuccess ||
        hipMemcpy(&v, &m->d_count->pairs, sizeof(v), hipMemcpyDeviceToHost) != hipSuccess)
      return -1;
    m->last_pairs = (long long)v;
    m->pairs_pending = false;
  }
  return m->last_pairs;
}

}  // extern "C"
