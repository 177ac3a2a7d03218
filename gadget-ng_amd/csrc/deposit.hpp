// deposit.hpp -- deterministic tiled CIC deposit for gfx950.
//
// Reference semantics: crates/gadget-ng-pm/src/cic.rs:37-93 (mass per cell,
// node-centred trilinear weights, periodic wrap of all 8 indices).
//
// Positions enter as FP32 or FP64 (any stride); every kernel forms the cell
// coordinate c = (x * nm / L) rem_euclid nm in FP64, as cic.rs:50-52 does,
// so FP64 inputs keep their accuracy (cell_fix in pm_kernels.hpp).
//
// Method:
//   1. k_bucket_count  each particle's base cell (i0,j0,k0) gives a tile of
//      T^3 cells and a class: bit a is set when the base cell is on the tile's
//      last layer along axis a, i.e. when the particle also feeds the next
//      tile along that axis.  Bucket = Hilbert rank of the tile * 8 + class.  Counts use one
//      atomic per run of equal buckets within a wavefront (particles that
//      arrive in spatial order share buckets in runs), which also yields each
//      particle's rank inside its bucket.  The max |m| for the fixed-point
//      scale is reduced in the same pass.
//   2. k_scan_*        exclusive scan of the bucket counts.
//   3. k_scatter       particles to bucket order as 24-byte cell records
//      (PartRec: per axis the cell index and a 43-bit in-cell fraction, plus
//      the FP32 mass), and the sum of the fixed-point masses.
//   4. k_deposit       one workgroup per tile owns its T^3 cells outright.  It
//      reads its own particles and, from the 7 lower neighbour tiles, only the
//      classes that reach into it, and adds each of the 8 CIC targets exactly
//      once over all tiles (target offset a lands in tile t + (a & class)).
//      Weights are formed in FP64 from the fractions and become 64-bit fixed
//      point (w * m * 2^s, N max|m| 2^s < 2^62); they accumulate with LDS
//      integer atomics, so the sum is exact and order-independent.  The tile
//      is then written as FP32 mass per cell minus the mean mass per cell
//      (an integer subtracted before the conversion, so a nearly uniform
//      density keeps its contrast to FP32 precision; the constant only
//      touches the k = 0 mode, which the Green's function drops).  No global
//      atomics touch the mesh and no mesh clearing pass is needed.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pm_kernels.hpp"
#include "scan.hpp"

namespace gng {

// Tiles are numbered along a 3-D Hilbert curve: rank[t] is the curve
// position of the tile with linear index t = (tz*nt + ty)*nt + tx and
// order[] the inverse, so bucket order (and the sorted particle order) walks
// the box tile by face-adjacent tile, and the deposit launches its
// workgroups in the same order.
struct TileMap {
  int T;   // tile side in cells
  int nt;  // tiles per axis (nm / T)
  const unsigned* rank;
  const unsigned* order;
  // src[8r + d]: first bucket (rank * 8) of source tile d of the tile of rank
  // r, the tile u - d (bit 0 x, bit 1 y, bit 2 z, periodic), so a deposit
  // workgroup finds its 72 bucket offsets after one table load
  const unsigned* src;
  // per tile rank, kRangeWords words of the flattened layout of its 14
  // bucket ranges, filled by k_tile_ranges for each solve
  unsigned* ranges;
};

// Fill tm.src from rank[] for the tiles t = t0, t0 + step, ...
__device__ __host__ inline void fill_tile_src(int nt, const unsigned* rank, unsigned* src, int t0, int step) {
  const int nt3 = nt * nt * nt;
  for (int t = t0; t < nt3; t += step) {
    const int ux = t % nt, uy = (t / nt) % nt, uz = t / (nt * nt);
    for (int d = 0; d < 8; ++d) {
      const int sx = (d & 1) ? (ux == 0 ? nt - 1 : ux - 1) : ux;
      const int sy = (d & 2) ? (uy == 0 ? nt - 1 : uy - 1) : uy;
      const int sz = (d & 4) ? (uz == 0 ? nt - 1 : uz - 1) : uz;
      src[(size_t)rank[t] * 8 + d] = rank[(sz * nt + sy) * nt + sx] * 8u;
    }
  }
}

// Zero a buffer with vector stores (a fill kernel rather than a memset, so the
// sequence stays safe to capture in a graph).
__device__ __forceinline__ void zero_body(uint4* __restrict__ p, long long n16) {
  const uint4 z = make_uint4(0u, 0u, 0u, 0u);
  for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (long long)gridDim.x * blockDim.x)
    p[i] = z;
}

// The bucket counts cleared and, by the first workgroup, the solve's scalars
// reset: the two clears before a sort in one launch.
__global__ __launch_bounds__(256) void k_sort_reset(uint4* __restrict__ p, long long n16, SolveScalars* sc) {
  if (blockIdx.x == 0) reset_scalars_body(sc);
  zero_body(p, n16);
}

__global__ __launch_bounds__(256) void k_sort_reset_box(const BoxArgs* __restrict__ bx, long long n16) {
  const BoxArgs& b = bx[blockIdx.z];
  if (blockIdx.x == 0) reset_scalars_body(b.sc);
  zero_body(reinterpret_cast<uint4*>(b.count), n16);
}

__device__ __forceinline__ unsigned bucket_of_cell(int ix, int iy, int iz, const TileMap tm) {
  const int tx = ix / tm.T, ty = iy / tm.T, tz = iz / tm.T;
  const unsigned cls = (unsigned)(ix - tx * tm.T == tm.T - 1) | ((unsigned)(iy - ty * tm.T == tm.T - 1) << 1) |
                       ((unsigned)(iz - tz * tm.T == tm.T - 1) << 2);
  return tm.rank[((unsigned)tz * tm.nt + ty) * tm.nt + tx] * 8u + cls;
}

// Each thread classifies kBucketPer particles (block stride 256, so every
// wavefront still sees 64 consecutive particles).  Counting is two-level:
// runs of equal buckets within a wavefront take one slot of a block-local
// hash table in LDS and one LDS atomic; then each distinct bucket of the
// block takes one global atomic, which returns the block's base rank in that
// bucket.  A block of clustered particles thus costs a few global atomics
// instead of one per run.  Ranks within a bucket stay unique; their order
// differs from call to call, which no result depends on (the deposit sums
// integers).
constexpr int kBucketPer = 4;
constexpr int kBucketSlots = 2048;  // > 256 * kBucketPer keys: probing always ends
constexpr unsigned kEmptyKey = 0xffffffffu;

template <typename T, typename M>
__device__ __forceinline__ void bucket_count_body(const PosSrc<T> src, const M* __restrict__ m, long long n,
                                                      const CellMap cm, const TileMap tm,
                                                      unsigned* __restrict__ count, unsigned* __restrict__ bucket,
                                                      unsigned* __restrict__ rank, SolveScalars* sc) {
  __shared__ unsigned hkey[kBucketSlots], hcnt[kBucketSlots];
  for (int e = threadIdx.x; e < kBucketSlots; e += 256) {
    hkey[e] = kEmptyKey;
    hcnt[e] = 0u;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const long long i0 = (long long)blockIdx.x * (256 * kBucketPer) + threadIdx.x;
  unsigned b[kBucketPer], local[kBucketPer];
  int slot[kBucketPer];
  float am = 0.0f;
#pragma unroll
  for (int k = 0; k < kBucketPer; ++k) {
    const long long i = i0 + 256LL * k;
    const bool live = i < n;
    b[k] = kEmptyKey;
    if (live) {
      const long long o = i * src.stride;
      const double px = (double)src.x[o], py = (double)src.y[o], pz = (double)src.z[o];
      am = fmaxf(am, fabsf((float)m[i]));
      int ix, iy, iz;
      unsigned long long f;
      cell_fix(px, cm, ix, f);
      cell_fix(py, cm, iy, f);
      cell_fix(pz, cm, iz, f);
      b[k] = bucket_of_cell(ix, iy, iz, tm);
    }
    // runs of equal buckets: a lane heads a run when its bucket differs from the previous lane's
    const unsigned prev = __shfl_up(b[k], 1);
    const bool head = live && (lane == 0 || prev != b[k]);
    const unsigned long long heads = __ballot(head);
    const unsigned long long below = lane == 63 ? ~0ull : ((1ull << (lane + 1)) - 1);
    const int my_head = 63 - __clzll(heads & below);  // highest head at or below this lane
    const unsigned long long above = heads & ~below;
    const unsigned long long live_mask = __ballot(live);
    const int next_head = above ? __ffsll((long long)above) - 1 : 64 - __clzll(live_mask);
    int hs = 0;
    unsigned hb = 0;
    if (head) {
      // insert or find the bucket in the block's table (linear probing)
      hs = (int)((b[k] * 2654435761u) >> 21);  // 11 bits: kBucketSlots = 2048
      for (;;) {
        const unsigned old = atomicCAS(&hkey[hs], kEmptyKey, b[k]);
        if (old == kEmptyKey || old == b[k]) break;
        hs = (hs + 1) & (kBucketSlots - 1);
      }
      hb = atomicAdd(&hcnt[hs], (unsigned)(next_head - lane));
    }
    const int src = my_head < 0 ? 0 : my_head;
    slot[k] = __shfl(hs, src);
    local[k] = __shfl(hb, src) + (unsigned)(lane - my_head);
  }
  __syncthreads();
  // one global atomic per distinct bucket of the block; hcnt becomes the base
#pragma unroll
  for (int e = threadIdx.x; e < kBucketSlots; e += 256) {
    const unsigned key = hkey[e];
    if (key != kEmptyKey) hcnt[e] = atomicAdd(count + key, hcnt[e]);
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kBucketPer; ++k) {
    const long long i = i0 + 256LL * k;
    if (i < n) {
      bucket[i] = b[k];
      rank[i] = hcnt[slot[k]] + local[k];
    }
  }
  // max |m|: wave, then block, then one atomic per block only when it raises
  // the running maximum (a plain read filters the common equal-mass case)
  for (int off = 32; off > 0; off >>= 1) am = fmaxf(am, __shfl_xor(am, off));
  __shared__ float wmax[4];
  if (lane == 0) wmax[threadIdx.x >> 6] = am;
  __syncthreads();
  if (threadIdx.x == 0) {
    const float bm = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
    const unsigned bits = __float_as_uint(bm);
    if (bm > 0.0f && bits > __atomic_load_n(&sc->mmax_bits, __ATOMIC_RELAXED)) atomicMax(&sc->mmax_bits, bits);
  }
}

template <typename T, typename M>
__global__ __launch_bounds__(256) void k_bucket_count(const PosSrc<T> src, const M* __restrict__ m, long long n,
                                                      const CellMap cm, const TileMap tm,
                                                      unsigned* __restrict__ count, unsigned* __restrict__ bucket,
                                                      unsigned* __restrict__ rank, SolveScalars* sc) {
  bucket_count_body<T, M>(src, m, n, cm, tm, count, bucket, rank, sc);
}

__global__ __launch_bounds__(256) void k_bucket_count_box(const BoxArgs* __restrict__ bx, const PosSrc<float> src, const float* __restrict__ m, const TileMap tm) {
  const BoxArgs& b = bx[blockIdx.z];
  bucket_count_body<float, float>(PosSrc<float>{src.x + b.p0, src.y + b.p0, src.z + b.p0, 1}, m + b.p0, b.n, b.cm, tm, b.count, b.bucket, b.rank,
                                  b.sc);
}

// Exclusive scan of `count` (nb entries) into `offset` (nb + 1 entries),
// in the two launches of scan.hpp (the second adds each workgroup's prefix).
__global__ __launch_bounds__(256) void k_scan_local(const unsigned* __restrict__ count, unsigned* __restrict__ offset,
                                                    unsigned* __restrict__ partial, long long nb) {
  scan_local_body(count, offset, partial, nb);
}

__global__ __launch_bounds__(256) void k_scan_local_box(const BoxArgs* __restrict__ bx, long long nb) {
  const BoxArgs& b = bx[blockIdx.z];
  scan_local_body(b.count, b.offset, b.partial, nb);
}

__global__ __launch_bounds__(256) void k_scan_add_prefix(unsigned* __restrict__ offset,
                                                         const unsigned* __restrict__ partial, int nblocks,
                                                         long long nb) {
  scan_add_prefix_body(offset, partial, nblocks, nb);
}

__global__ __launch_bounds__(256) void k_scan_add_prefix_box(const BoxArgs* __restrict__ bx, int nblocks, long long nb) {
  const BoxArgs& b = bx[blockIdx.z];
  scan_add_prefix_body(b.offset, b.partial, nblocks, nb);
}

// Particle i to its bucket slot as a cell record, and the sum of the
// particles' fixed-point masses round(m 2^s) (one integer atomic per block,
// so the total does not depend on the order): the deposit subtracts the mean
// per cell before it converts to FP32.  Each thread moves kScatterPer
// particles (block stride 256, so a wavefront still reads 64 consecutive
// particles); all of their loads are issued before the dependent offset
// loads, and those before any store, so a thread waits for two memory
// latencies however many particles it moves.
constexpr int kScatterPer = 4;

template <typename T, typename M>
__device__ __forceinline__ void scatter_body(const PosSrc<T> src, const M* __restrict__ m, long long n,
                                                 const CellMap cm, const unsigned* __restrict__ bucket,
                                                 const unsigned* __restrict__ rank,
                                                 const unsigned* __restrict__ offset, PartRec* __restrict__ sorted,
                                                 unsigned* __restrict__ perm, SolveScalars* sc) {
  const long long i0 = (long long)blockIdx.x * (256 * kScatterPer) + threadIdx.x;
  double px[kScatterPer], py[kScatterPer], pz[kScatterPer];
  float mf[kScatterPer];
  unsigned slot[kScatterPer];
#pragma unroll
  for (int k = 0; k < kScatterPer; ++k) {
    const long long i = i0 + 256LL * k;
    if (i < n) {
      const long long o = i * src.stride;
      px[k] = (double)src.x[o];
      py[k] = (double)src.y[o];
      pz[k] = (double)src.z[o];
      mf[k] = (float)m[i];
      slot[k] = bucket[i];
    }
  }
#pragma unroll
  for (int k = 0; k < kScatterPer; ++k) {
    const long long i = i0 + 256LL * k;
    if (i < n) slot[k] = offset[slot[k]] + rank[i];
  }
  const int shift = fixed_shift(sc, n);
  long long q = 0;
#pragma unroll
  for (int k = 0; k < kScatterPer; ++k) {
    const long long i = i0 + 256LL * k;
    if (i < n) {
      int c[3];
      unsigned long long f[3];
      cell_fix(px[k], cm, c[0], f[0]);
      cell_fix(py[k], cm, c[1], f[1]);
      cell_fix(pz[k], cm, c[2], f[2]);
      sorted[slot[k]] = encode_rec(c, f, mf[k]);
      if (perm) perm[slot[k]] = (unsigned)i;  // only for the sorted-order interpolation
      q += rint_small(ldexp((double)mf[k], shift));
    }
  }
  for (int off = 32; off > 0; off >>= 1) q += __shfl_xor(q, off);
  __shared__ long long wsum[4];
  if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = q;
  __syncthreads();
  if (threadIdx.x == 0) {
    const long long t = (wsum[0] + wsum[1]) + (wsum[2] + wsum[3]);
    if (t) atomicAdd(&sc->qsum[(blockIdx.x % kQSlots) * kQStride], (unsigned long long)t);
  }
}

template <typename T, typename M>
__global__ __launch_bounds__(256) void k_scatter(const PosSrc<T> src, const M* __restrict__ m, long long n,
                                                 const CellMap cm, const unsigned* __restrict__ bucket,
                                                 const unsigned* __restrict__ rank,
                                                 const unsigned* __restrict__ offset, PartRec* __restrict__ sorted,
                                                 unsigned* __restrict__ perm, SolveScalars* sc) {
  scatter_body<T, M>(src, m, n, cm, bucket, rank, offset, sorted, perm, sc);
}

__global__ __launch_bounds__(256) void k_scatter_box(const BoxArgs* __restrict__ bx, const PosSrc<float> src, const float* __restrict__ m) {
  const BoxArgs& b = bx[blockIdx.z];
  scatter_body<float, float>(PosSrc<float>{src.x + b.p0, src.y + b.p0, src.z + b.p0, 1}, m + b.p0, b.n, b.cm, b.bucket, b.rank, b.offset, b.sorted,
                             nullptr, b.sc);
}

// The 14 bucket ranges a tile reads: (d, first class, end class).  d is the
// neighbour offset (bit 0 x, bit 1 y, bit 2 z: the source tile is u - d) and
// the classes are those containing every bit of d, merged where adjacent.
// d of range r is (kRangeD >> 3r) & 7 (packed, so a per-lane r needs no load)
constexpr unsigned char kRangeDList[14] = {0, 1, 1, 1, 1, 2, 2, 3, 3, 4, 5, 5, 6, 7};
constexpr unsigned long long pack_range_d() {
  unsigned long long v = 0;
  for (int i = 0; i < 14; ++i) v |= (unsigned long long)kRangeDList[i] << (3 * i);
  return v;
}
constexpr unsigned long long kRangeD = pack_range_d();
__constant__ unsigned char kRangeLo[14] = {0, 1, 3, 5, 7, 2, 6, 3, 7, 4, 5, 7, 6, 7};
__constant__ unsigned char kRangeHi[14] = {8, 2, 4, 6, 8, 4, 8, 4, 8, 8, 6, 8, 8, 8};

// Heavy tiles over several workgroups.  A tile whose 14 ranges hold more than
// `items` particles gets S = ceil(count / items) slices (at most kMaxSlices):
// S workgroups of their own, in front of those of the ordinary tiles so that
// the longest work starts first, each depositing an equal share of the ranges
// into its own LDS tile.  The slices add their int64 tiles into a scratch
// tile with global atomics (integer sums: the result does not depend on the
// order or on how a tile is split) and the last slice to finish converts the
// scratch tile and clears it for the next solve.  Clustered inputs otherwise
// leave a few Plummer-core tiles running hundreds of rounds on one workgroup
// each while the chip idles.
constexpr unsigned kMaxSlices = 1024;
constexpr unsigned kNoSlice = 0xffffffffu;

// Slice workgroups (and half as many scratch tiles) that particles counted once
// can need: a tile is split only above `items`, so S <= 2 count / items.  The
// deposit's table has twice as many.  Its tiles count a particle up to eight
// times, so the first half, where a tile takes S = ceil(count / items), can run
// out: when most particles sit at tile edges.  A tile that finds it so counts a
// particle that m tiles read as 1 / m, which adds up to n over the tiles, and
// takes ceil(that / items) slices of the second half, which cannot run out; its
// slices are up to eight times as long.  Workgroup e of the table runs entry e
// of both halves, so the second costs no empty workgroups.  A solve of 10^6 particles about a tile
// corner (sigma 0.7 cells) on 48^3: 414 us, 2256 where such tiles ran unsplit.
inline unsigned deposit_slots(long long n, unsigned items) { return (unsigned)((2 * n / items + 16) & ~7LL); }

// The flattened range layout of every tile rank r, written after the scatter
// so that a deposit workgroup reads its whole prologue with scalar loads:
// ranges[kRangeWords r + k] is, for k < 13, the end of range k when the 14
// ranges are laid end to end; word 13 is their total, word 14 the slot delta
// of range 0 (sorted slot = flattened index + delta) and word 15 + k the
// change of that delta from range k to k + 1.  Word 28 is the tile's slice
// count (1: not split) and word 29 its scratch tile: a tile above sp.items
// particles reserves S slice workgroups with one atomic and writes their table
// entries; S >= 2, so the first one's half names a scratch tile that no other
// tile has.  A tile that finds the table's first half spent marks what it
// reserved there unused.  The first wavefront also
// sums the scatter's fixed-point mass slots into the integer part of the mean
// mass per cell (sc->qmean) and keeps the fixed-point exponent (sc->shift).
constexpr int kRangeWords = 32;
__device__ __forceinline__ void tile_ranges_body(const unsigned* __restrict__ offset, const TileMap& tm,
                                                 SolveScalars* sc, long long ntot, const DepositSplit& sp) {
  const unsigned ntiles = (unsigned)tm.nt * tm.nt * tm.nt;
  const unsigned r = blockIdx.x * blockDim.x + threadIdx.x;
  if (blockIdx.x == 0 && threadIdx.x < 64) {
    static_assert(kQSlots == 64, "one mass slot per lane");
    unsigned long long q = sc->qsum[threadIdx.x * kQStride];
    for (int off = 32; off > 0; off >>= 1) q += __shfl_xor(q, off);
    if (threadIdx.x == 0) {
      const long long nm = (long long)tm.T * tm.nt;
      sc->qmean = (long long)(q / (unsigned long long)(nm * nm * nm));
      sc->shift = fixed_shift(sc, ntot);
    }
  }
  if (r >= ntiles) return;
  unsigned w[kRangeWords];
  unsigned pre = 0, prev = 0;
#pragma unroll
  for (int k = 0; k < 14; ++k) {
    const int d = (int)((kRangeD >> (3 * k)) & 7ull);
    const unsigned b = tm.src[(size_t)r * 8 + d];
    const unsigned beg = offset[b + kRangeLo[k]];
    const unsigned len = offset[b + kRangeHi[k]] - beg;
    const unsigned delta = beg - pre;
    pre += len;
    if (k < 13) w[k] = pre;
    if (k == 0) w[14] = delta;
    else w[14 + k] = delta - prev;
    prev = delta;
  }
  w[13] = pre;
  unsigned S = 1u, slot = 0u;
  if (sp.slots != 0u && pre > sp.items) {
    const unsigned half = sp.slots / 2u;
    S = min((pre + sp.items - 1u) / sp.items, kMaxSlices);
    unsigned base = atomicAdd(&sc->split_budget, S);
    if (base + S > half) {
      for (unsigned e = base; e < half; ++e) sp.extra[e] = kNoSlice;
      unsigned long long eighths = 0;
      for (int d = 0; d < 8; ++d) {
        const unsigned b = tm.src[(size_t)r * 8 + d];
        for (int c = d; c < 8; ++c)
          if ((c & d) == d) eighths += (unsigned long long)(offset[b + c + 1] - offset[b + c]) << (3 - __popc(c));
      }
      S = min((unsigned)((eighths + 8ull * sp.items - 1ull) / (8ull * sp.items)), kMaxSlices);
      if (S > 1u) base = half + atomicAdd(&sc->split_rest, S);
    }
    if (S > 1u) {
      slot = base / 2u;
      for (unsigned k = 0; k < S; ++k) sp.extra[base + k] = r | (k << 20);
    }
  }
  w[28] = S;
  w[29] = slot;
  w[30] = w[31] = 0u;
  uint4* dst = reinterpret_cast<uint4*>(tm.ranges + (size_t)r * kRangeWords);
#pragma unroll
  for (int k = 0; k < kRangeWords / 4; ++k) dst[k] = make_uint4(w[4 * k], w[4 * k + 1], w[4 * k + 2], w[4 * k + 3]);
}

__global__ __launch_bounds__(256) void k_tile_ranges(const unsigned* __restrict__ offset, const TileMap tm,
                                                     SolveScalars* sc, long long ntot, const DepositSplit sp) {
  tile_ranges_body(offset, tm, sc, ntot, sp);
}

__global__ __launch_bounds__(256) void k_tile_ranges_box(const BoxArgs* __restrict__ bx, const TileMap tm) {
  const BoxArgs& b = bx[blockIdx.z];
  TileMap t = tm;
  t.ranges = b.ranges;
  tile_ranges_body(b.offset, t, b.sc, b.n, b.split);
}

// The 8 CIC targets of one cell record of source range r (d = the range's
// neighbour offset) into the LDS tile acc of T^3 int64 accumulators: FP64
// weights (the 43-bit fractions convert exactly, 1 - f is exact, and the
// products round far below the fixed-point unit) times m 2^s (scale), as
// 64-bit fixed point; live marks the lanes with a record.  Every lane adds
// directly, also where a clump puts much of a wavefront into one cell: lanes
// on one LDS word take turns, but summing them with shuffles first costs as
// many LDS turns (deposit of 512^3 particles, 30 % in Plummer spheres of 0.4
// cells, on 1024^3: 3.42 ms with a shuffle reduction of the most common cell,
// 2.78 ms without; 2^22 particles in one cell: 0.32 ms either way).
template <int T>
__device__ __forceinline__ void deposit_record(unsigned long long* acc, const PartRec& p, int r, bool live,
                                               double scale) {
  const int d = (int)((kRangeD >> (3 * r)) & 7ull);
  const double fx = rec_frac(p, 0), fy = rec_frac(p, 1), fz = rec_frac(p, 2);
  const double ms = (double)rec_mass(p) * scale;
  const double wx[2] = {1.0 - fx, fx}, wy[2] = {1.0 - fy, fy};
  const double wz[2] = {(1.0 - fz) * ms, fz * ms};
  // local base index in the particle's own tile; its class follows from it
  const int lx0 = rec_cell(p, 0) % T, ly0 = rec_cell(p, 1) % T, lz0 = rec_cell(p, 2) % T;
  const int cx = lx0 == T - 1, cy = ly0 == T - 1, cz = lz0 == T - 1;
  const int dx = d & 1, dy = (d >> 1) & 1, dz = (d >> 2) & 1;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int lz = dz ? 0 : lz0 + a;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int ly = dy ? 0 : ly0 + b;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int lx = dx ? 0 : lx0 + c;
        const bool valid = live && (a & cz) == dz && (b & cy) == dy && (c & cx) == dx;
        if (valid) atomicAdd(acc + (lz * T + ly) * T + lx, (unsigned long long)rint_small(wx[c] * (wy[b] * wz[a])));
      }
    }
  }
}

// Record of flattened item q of the tile whose range row is w (uniform, so
// its words come from the scalar cache), for q < limit: the sorted slot is q
// plus the delta of its range, summed as masked steps over the range ends at
// or below q (range ends never decrease; written as arithmetic so that it
// stays in registers).  Range 0, the tile's own bucket, holds most of its
// particles: a wavefront whose 64 items all lie in it (the items of a
// wavefront are consecutive, lane 0's first) skips the per-lane search.
__device__ __forceinline__ PartRec fetch_record(const PartRec* __restrict__ sorted, const unsigned* __restrict__ w,
                                                unsigned q, unsigned limit, int& r, bool& live) {
  const unsigned qw = __builtin_amdgcn_readfirstlane(q);
  unsigned dl = w[14];
  r = 0;
  if (qw + 63u >= w[0]) {
#pragma unroll
    for (int k = 0; k < 13; ++k) {
      const bool ge = q >= w[k];
      r += ge ? 1 : 0;
      dl += w[15 + k] & (0u - (unsigned)ge);
    }
  }
  live = q < limit;
  PartRec v;
  if (live) {
    v = sorted[q + dl];
  } else {
    v.a[0] = v.a[1] = v.a[2] = 0ull;
  }
  return v;
}

// Rounds of records in flight at once: a tile of the uniform headline holds
// about 2.5 rounds at 256 threads, so all of its loads share one memory
// latency.  Slot j holds the record of round it + j; the round loops are
// unrolled by kPrefetch so every slot index is static.
constexpr int kPrefetch = 3;

// Workgroup index b of n to item index so that each XCD (workgroups are dealt
// to the eight round robin) works on one contiguous eighth of the items.
__device__ __forceinline__ unsigned xcd_item(unsigned b, unsigned n) {
  const unsigned per = (n + 7u) / 8u;
  return (b & 7u) * per + (b >> 3);
}
constexpr unsigned xcd_grid(unsigned n) { return (n + 7u) / 8u * 8u; }

// Table entry v, one slice of a heavy tile (sp): its share of the flattened ranges into the
// LDS tile, the LDS tile into the scratch tile, and the last slice of the
// tile converts.
template <int T, int NT>
__device__ __forceinline__ void deposit_slice(unsigned long long* acc, const PartRec* __restrict__ sorted,
                                              const CellMap& cm, const TileMap& tm, const SolveScalars* sc,
                                              float* __restrict__ rho, long long rho_plane, float* __restrict__ keep,
                                              const DepositSplit& sp, unsigned v) {
  constexpr int T3 = T * T * T;
  const int tid = threadIdx.x, nt = tm.nt;
  const unsigned rank = v & 0xfffffu;
  const unsigned* __restrict__ w = tm.ranges + (size_t)rank * kRangeWords;
  const unsigned all = w[13], S = w[28], slot = w[29];
  const unsigned share = (all + S - 1u) / S;
  const unsigned q0 = min(all, (v >> 20) * share), total = min(all, q0 + share);
  const unsigned rounds = (total - q0 + NT - 1u) / NT;
  const double scale = ldexp(1.0, sc->shift), unit = ldexp(1.0, -sc->shift);
  PartRec buf[kPrefetch];
  int rbuf[kPrefetch];
  bool lbuf[kPrefetch];
#pragma unroll
  for (int j = 0; j < kPrefetch; ++j) {
    rbuf[j] = 0;
    lbuf[j] = false;
    if ((unsigned)j < rounds) buf[j] = fetch_record(sorted, w, q0 + j * NT + tid, total, rbuf[j], lbuf[j]);
  }
  for (int c = tid; c < T3; c += NT) acc[c] = 0ull;
  __syncthreads();
  for (unsigned it = 0; it < rounds; it += kPrefetch) {
#pragma unroll
    for (int j = 0; j < kPrefetch; ++j) {
      const unsigned g = it + (unsigned)j;
      if (g < rounds) {  // uniform over the workgroup
        const PartRec p = buf[j];
        const int r = rbuf[j];
        const bool live = lbuf[j];
        if (g + kPrefetch < rounds)
          buf[j] = fetch_record(sorted, w, q0 + (g + kPrefetch) * NT + tid, total, rbuf[j], lbuf[j]);
        deposit_record<T>(acc, p, r, live, scale);
      }
    }
  }
  __syncthreads();
  unsigned long long* part = sp.scratch + (size_t)slot * T3;
  for (int c = tid; c < T3; c += NT) {
    const unsigned long long x = acc[c];
    if (x) atomicAdd(part + c, x);
  }
  __threadfence();
  __syncthreads();
  // the accumulators have been read: their first word holds the flag
  unsigned* const last = reinterpret_cast<unsigned*>(acc);
  if (tid == 0) *last = atomicAdd(sp.done + slot, 1u) == S - 1u;
  __syncthreads();
  if (!*last) return;
  __threadfence();
  const int tile = (int)tm.order[rank];
  const int ux = tile % nt, uy = (tile / nt) % nt, uz = tile / (nt * nt);
  const long long qmean = sc->qmean;
  for (int c = tid; c < T3; c += NT) {
    const int lx = c % T, ly = (c / T) % T, lz = c / (T * T);
    const size_t row = (size_t)(uy * T + ly) * cm.nm + (ux * T + lx);
    const long long x = (long long)__hip_atomic_load(part + c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    part[c] = 0ull;
    rho[(size_t)(uz * T + lz) * rho_plane + row] = (float)((double)(x - qmean) * unit);
    if (keep) keep[(size_t)(uz * T + lz) * cm.nm * cm.nm + row] = (float)((double)x * unit);
  }
  if (tid == 0) sp.done[slot] = 0u;
}

// One workgroup per group of TILES tiles (1 or 2, neighbours along the
// Hilbert curve); T is the tile side (T^3 int64 accumulators in LDS).  Cell
// (x, y, z) of the shifted mass mesh is rho[z*rho_plane + y*nm + x]; keep
// (when not null) receives the unshifted mass per cell, unpadded.  The first
// `lead` workgroups of the grid (at least sp.slots / 2) are the slices of the
// heavy tiles, which the others skip.
// With two tiles, their rounds of records form one sequence, so the prefetch
// ring runs across the tile boundary: the second tile's records load while
// the first tile is converted and written.
template <int T, int NT, int TILES>
__device__ __forceinline__ void deposit_body(const PartRec* __restrict__ sorted, const CellMap& cm, const TileMap& tm,
                                             const SolveScalars* sc, float* __restrict__ rho, long long rho_plane,
                                             float* __restrict__ keep, const DepositSplit& sp, unsigned lead) {
  constexpr int T3 = T * T * T;
  __shared__ unsigned long long acc[T3];
  const int tid = threadIdx.x;
  const int nt = tm.nt;
  if (blockIdx.x < lead) {
    // (uniform) the entries of this workgroup in either half of the table, through
    // one copy of the slice code (24307 particles on 64^3: 85.9 us, 86.4 with two)
    const unsigned e = blockIdx.x, half = sp.slots / 2u;
    const unsigned first = min(sc->split_budget, half), rest = sc->split_rest;
#pragma unroll 1
    for (unsigned h = 0; h < 2u; ++h) {
      if (e >= (h ? rest : first)) continue;
      const unsigned v = sp.extra[h ? half + e : e];
      if (v == kNoSlice) continue;
      __syncthreads();  // the first entry's tile is read
      deposit_slice<T, NT>(acc, sorted, cm, tm, sc, rho, rho_plane, keep, sp, v);
    }
    return;
  }
  const unsigned ntiles = (unsigned)(nt * nt * nt), groups = (ntiles + TILES - 1u) / TILES;
  const unsigned grp = xcd_item(blockIdx.x - lead, groups);
  if (grp >= groups) return;  // uniform: padding of the last eighth
  const unsigned ra = TILES * grp, rb = ra + 1u;
  const bool has_b = TILES == 2 && rb < ntiles;  // uniform: the last workgroup may hold one tile
  const unsigned* __restrict__ wa = tm.ranges + (size_t)ra * kRangeWords;
  const unsigned* __restrict__ wb = tm.ranges + (size_t)(has_b ? rb : ra) * kRangeWords;
  const bool own_a = wa[28] == 1u, own_b = has_b && wb[28] == 1u;  // not left to slices
  const unsigned tot_a = own_a ? wa[13] : 0u, tot_b = own_b ? wb[13] : 0u;
  const unsigned rounds_a = (tot_a + NT - 1u) / NT, rounds = rounds_a + (tot_b + NT - 1u) / NT;
  const int tile_a = (int)tm.order[ra], tile_b = has_b ? (int)tm.order[rb] : 0;
  const double scale = ldexp(1.0, sc->shift), unit = ldexp(1.0, -sc->shift);
  const long long qmean = sc->qmean;
  // record of concatenated round g: tile a below rounds_a, then tile b
  auto fetch = [&](unsigned g, int& r, bool& live) {
    if (TILES == 1) return fetch_record(sorted, wa, g * NT + (unsigned)tid, tot_a, r, live);
    const bool in_b = g >= rounds_a;  // uniform
    return fetch_record(sorted, in_b ? wb : wa, (in_b ? g - rounds_a : g) * NT + (unsigned)tid, in_b ? tot_b : tot_a,
                        r, live);
  };
  // the accumulated tile as FP32 mass per cell minus the mean (and, with
  // keep, unshifted); clears the accumulators behind itself for a next tile
  auto write_tile = [&](int tile, bool clear) {
    const int ux = tile % nt, uy = (tile / nt) % nt, uz = tile / (nt * nt);
    for (int c = tid; c < T3; c += NT) {
      const int lx = c % T, ly = (c / T) % T, lz = c / (T * T);
      const size_t row = (size_t)(uy * T + ly) * cm.nm + (ux * T + lx);
      const long long v = (long long)acc[c];
      if (clear) acc[c] = 0ull;
      rho[(size_t)(uz * T + lz) * rho_plane + row] = (float)((double)(v - qmean) * unit);
      if (keep) keep[(size_t)(uz * T + lz) * cm.nm * cm.nm + row] = (float)((double)v * unit);
    }
  };
  PartRec buf[kPrefetch];
  int rbuf[kPrefetch];
  bool lbuf[kPrefetch];
#pragma unroll
  for (int j = 0; j < kPrefetch; ++j) {
    rbuf[j] = 0;
    lbuf[j] = false;
    if ((unsigned)j < rounds) buf[j] = fetch((unsigned)j, rbuf[j], lbuf[j]);
  }
  // the accumulators are cleared while the first records load
  for (int c = tid; c < T3; c += NT) acc[c] = 0ull;
  __syncthreads();
  if (TILES == 2 && rounds_a == 0u && own_a) {  // an empty tile a: zeros
    write_tile(tile_a, false);
    __syncthreads();
  }
  for (unsigned it = 0; it < rounds; it += kPrefetch) {
#pragma unroll
    for (int j = 0; j < kPrefetch; ++j) {
      const unsigned g = it + (unsigned)j;
      if (g < rounds) {  // uniform over the workgroup
        if (TILES == 2 && g == rounds_a && g != 0u) {
          // tile a is complete: write it and start tile b from zero
          __syncthreads();
          write_tile(tile_a, true);
          __syncthreads();
        }
        const PartRec p = buf[j];
        const int r = rbuf[j];
        const bool live = lbuf[j];
        if (g + kPrefetch < rounds) buf[j] = fetch(g + kPrefetch, rbuf[j], lbuf[j]);
        deposit_record<T>(acc, p, r, live, scale);
      }
    }
  }
  __syncthreads();
  if (TILES == 1) {
    if (own_a) write_tile(tile_a, false);
    return;
  }
  if (rounds == rounds_a && rounds_a != 0u) {
    // tile b had no records (or is not this workgroup's): tile a is still in acc
    write_tile(tile_a, true);
    __syncthreads();
  }
  if (own_b) write_tile(tile_b, false);
}

// At most 96 VGPRs, so five 256-thread workgroups (the LDS limit of a 16^3
// tile) fit a CU.
template <int T, int NT, int TILES>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(5))) void k_deposit(
    const PartRec* __restrict__ sorted, const CellMap cm, const TileMap tm, const SolveScalars* sc,
    float* __restrict__ rho, long long rho_plane, float* __restrict__ keep, const DepositSplit sp) {
  deposit_body<T, NT, TILES>(sorted, cm, tm, sc, rho, rho_plane, keep, sp, sp.slots / 2u);
}

// Every box has its own slices; `lead` is the most of the group.  Four boxes of
// 128^3 with 262144 particles, 30 % of them in one cell: 1.38 ms without slices,
// 0.43 with; without clumps 0.42 either way.
template <int T, int NT>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(5))) void k_deposit_box(
    const BoxArgs* __restrict__ bx, const TileMap tm, unsigned lead) {
  const BoxArgs& b = bx[blockIdx.z];
  TileMap t = tm;
  t.ranges = b.ranges;
  deposit_body<T, NT, 1>(b.sorted, b.cm, t, b.sc, reinterpret_cast<float*>(b.P), 2 * mesh_plane(b.cm.nm),
                         nullptr, b.split, lead);
}

// Particle moments per cell from the sorted cell records of the last sort: for
// the particles whose base cell is c, mom[5c + a] = sum m (f_a - 1/2)
// (a = x, y, z), mom[5c + 3] = sum m |f - 1/2|^2, mom[5c + 4] = sum m, with f
// the 43-bit in-cell fraction of the record.  The sums are 64-bit fixed point
// (the deposit's scale), so they do not depend on the particle order.
//
// kCellMomParts workgroups per tile, one for each part of its z layers (5
// int64 LDS accumulators per cell of the part), write every cell of the tile
// once (zero for an empty cell), so no clearing pass and no global atomics are
// needed.  A tile above sp.items particles (a Plummer core holds 10^5) is
// shared by slices as in the deposit: they add their sums into the tile's own
// words of mom as int64, which k_moments_plan has cleared, and the last of
// them converts the words in place.  256^3 particles, 30 % in 250 Plummer
// spheres: 1.38 ms with one workgroup a part and a shuffle reduction of the
// most common cell, 0.54 so (0.30 for a plain lattice).
constexpr int kCellMoments = 5;
constexpr int kCellMomThreads = 512;
constexpr int kCellMomParts = 2;

// Linear index of cell c of tile (ux, uy, uz).
template <int T>
__device__ __forceinline__ size_t tile_cell(int c, int ux, int uy, int uz, int nm) {
  return ((size_t)(uz * T + c / (T * T)) * nm + (uy * T + (c / T) % T)) * nm + (ux * T + c % T);
}

__global__ void k_moments_reset(SolveScalars* sc) { sc->moment_budget = 0u; }

// One workgroup per tile: words 30 (slices, 1: not split) and 31 (finished
// counter) of its range row, the slice table, and the cleared words of a split
// tile.
template <int T>
__global__ __launch_bounds__(256) void k_moments_plan(const unsigned* __restrict__ offset, const TileMap tm, int nm,
                                                      SolveScalars* sc, const DepositSplit sp,
                                                      double* __restrict__ mom) {
  __shared__ unsigned slices;
  const int tile = blockIdx.x, nt = tm.nt;
  const bool plain = sc->plain != 0u;  // no offsets, and never split: at most kSmallN records
  const unsigned rank = tm.rank[tile], w = plain ? 0u : offset[rank * 8u + 8u] - offset[rank * 8u];
  if (threadIdx.x == 0) {
    unsigned S = 1u, slot = 0u;
    if (sp.slots != 0u && w > sp.items) {
      // (a particle counts in one tile here, so the slots last)
      S = min((w + sp.items - 1u) / sp.items, kMaxSlices);
      const unsigned base = atomicAdd(&sc->moment_budget, S);
      slot = base / 2u;
      for (unsigned k = 0; k < S; ++k) sp.extra[base + k] = (unsigned)tile | (k << 20);
    }
    tm.ranges[(size_t)rank * kRangeWords + 30] = S;
    tm.ranges[(size_t)rank * kRangeWords + 31] = slot;
    slices = S;
  }
  __syncthreads();
  if (slices == 1u) return;
  const int ux = tile % nt, uy = (tile / nt) % nt, uz = tile / (nt * nt);
  for (int c = threadIdx.x; c < T * T * T; c += 256)
#pragma unroll
    for (int k = 0; k < kCellMoments; ++k) mom[tile_cell<T>(c, ux, uy, uz, nm) * kCellMoments + k] = 0.0;
}

template <int T>
__global__ __launch_bounds__(kCellMomThreads) void k_cell_moments(const PartRec* __restrict__ sorted,
                                                                  const unsigned* __restrict__ offset,
                                                                  const CellMap cm, const TileMap tm,
                                                                  const SolveScalars* sc, long long ntot,
                                                                  const DepositSplit sp, double* __restrict__ mom) {
  constexpr int HL = T / kCellMomParts, HC = T * T * HL, NT = kCellMomThreads;
  static_assert(T % kCellMomParts == 0, "tiles split into parts of whole layers");
  __shared__ unsigned long long acc[kCellMoments][HC];
  const int tid = threadIdx.x;
  const int nt = tm.nt;
  const int part = blockIdx.y;
  // the first sp.slots workgroups of a part are slices, the others whole tiles
  const bool slice = blockIdx.x < sp.slots;
  unsigned tile = blockIdx.x - sp.slots, k_slice = 0;
  if (slice) {
    if (blockIdx.x >= sc->moment_budget) return;  // uniform
    const unsigned v = sp.extra[blockIdx.x];
    tile = v & 0xfffffu;
    k_slice = v >> 20;
  }
  const int ux = (int)tile % nt, uy = ((int)tile / nt) % nt, uz = (int)tile / (nt * nt);
  const unsigned rank = tm.rank[tile], b0 = rank * 8u;
  const unsigned S = tm.ranges[(size_t)rank * kRangeWords + 30], slot = tm.ranges[(size_t)rank * kRangeWords + 31];
  if (!slice && S > 1u) return;
  // records in the caller's order (a small problem's deposit does not sort):
  // every tile looks through all of them
  const unsigned plain = sc->plain;
  unsigned beg = plain ? 0u : offset[b0], end = plain ? plain : offset[b0 + 8];
  if (slice) {
    const unsigned share = (end - beg + S - 1u) / S;
    beg = min(end, beg + k_slice * share);
    end = min(end, beg + share);
  }
  const int s = fixed_shift(sc, ntot);
  const double scale = ldexp(1.0, s), unit = ldexp(1.0, -s);
  for (int c = tid; c < HC; c += NT)
#pragma unroll
    for (int k = 0; k < kCellMoments; ++k) acc[k][c] = 0ull;
  __syncthreads();
  // two records in flight per thread
  PartRec next;
  if (beg + (unsigned)tid < end) next = sorted[beg + (unsigned)tid];
  for (unsigned q = beg + (unsigned)tid; q < end; q += NT) {
    const PartRec p = next;
    if (end - q > NT) next = sorted[q + NT];
    const int lx = rec_cell(p, 0) % T, ly = rec_cell(p, 1) % T, lz = rec_cell(p, 2) % T;
    if (lz / HL != part) continue;
    if (plain && (rec_cell(p, 0) / T != ux || rec_cell(p, 1) / T != uy || rec_cell(p, 2) / T != uz)) continue;
    const int c = ((lz - part * HL) * T + ly) * T + lx;
    const double fx = rec_frac(p, 0) - 0.5, fy = rec_frac(p, 1) - 0.5, fz = rec_frac(p, 2) - 0.5;
    const double ms = (double)rec_mass(p) * scale;
    const long long v[kCellMoments] = {rint_small(ms * fx), rint_small(ms * fy), rint_small(ms * fz),
                                        rint_small(ms * (fx * fx + fy * fy + fz * fz)), rint_small(ms)};
#pragma unroll
    for (int k = 0; k < kCellMoments; ++k) atomicAdd(&acc[k][c], (unsigned long long)v[k]);
  }
  __syncthreads();
  // consecutive threads take consecutive words of a cell row
  constexpr int W = HC * kCellMoments;
  if (!slice) {
    for (int e = tid; e < W; e += NT) {
      const int c = e / kCellMoments, k = e % kCellMoments;
      mom[tile_cell<T>(c + part * HC, ux, uy, uz, cm.nm) * kCellMoments + k] = (double)(long long)acc[k][c] * unit;
    }
    return;
  }
  unsigned long long* sums = reinterpret_cast<unsigned long long*>(mom);
  for (int e = tid; e < W; e += NT) {
    const int c = e / kCellMoments, k = e % kCellMoments;
    const unsigned long long v = acc[k][c];
    if (v) atomicAdd(sums + tile_cell<T>(c + part * HC, ux, uy, uz, cm.nm) * kCellMoments + k, v);
  }
  __threadfence();
  __syncthreads();
  unsigned* const last = reinterpret_cast<unsigned*>(&acc[0][0]);  // read above
  if (tid == 0) *last = atomicAdd(sp.done + slot, 1u) == S * kCellMomParts - 1u;
  __syncthreads();
  if (!*last) return;
  __threadfence();
  for (int e = tid; e < W * kCellMomParts; e += NT) {
    const int c = e / kCellMoments, k = e % kCellMoments;
    unsigned long long* p = sums + tile_cell<T>(c, ux, uy, uz, cm.nm) * kCellMoments + k;
    const long long v = (long long)__hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *reinterpret_cast<double*>(p) = (double)v * unit;
  }
  if (tid == 0) sp.done[slot] = 0u;
}

}  // namespace gng
