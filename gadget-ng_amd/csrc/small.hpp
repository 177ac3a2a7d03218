// small.hpp -- the pipeline of small problems in few launches.
//
// At a 64^3 mesh and 32^3 particles the fourteen launches of the general
// pipeline take 2.5 to 11 us each, none of it work: every launch waits for
// the one before it to drain and then for its own first loads.  Two changes
// cut their number to six.
//
// * The deposit of few particles needs no sort: k_cells_small forms every
//   particle's cell record once, and one workgroup per tile (k_deposit_small)
//   looks through all of their packed cells (4 bytes each, from L2) for those
//   that reach its tile.  Six launches become two: 41 to 22 us for 2048
//   particles on 32^3, 41 to 25 us for 8192 on 64^3, 52 to 34 us for 8192 on
//   128^3.
// * Up to N = 128 a z plane of the half spectrum fits a workgroup's LDS (66 KB
//   at 128), so one kernel does both transforms of a plane: k_plane_fwd
//   (x then y) and k_plane_inv (y then x).  k_z_small does the z pass and the
//   packed column in one launch and stores phi over P besides A, so that the
//   three fields of k_plane_inv are separate workgroups, each in place.
//   Transforms of a solve: 45 to 31 us at 32^3, 54 to 34 us at 64^3, 57 to
//   50 us at 96^3, 66 to 61 us at 128^3.
//
// The deposit's sums are the general kernels' integers, so its meshes and
// records are the same bit for bit; the transforms run the same radix plans on
// the same values, rounded alike up to the compiler's choice of fused products.
#pragma once
#include "deposit.hpp"

namespace gng {

constexpr int kPlaneMax = 128;          // largest mesh with plane kernels
// Most particles of the sort-free deposit, whose tiles have one workgroup each
// whatever they hold.  All of them in one clump, against the sorted deposit and
// its slices: 46 against 58 us for 8192 on 48^3, 64 against 66 for 13824, 121
// against 70 for 32768; spread evenly it would stay ahead (38 against 44 us for
// 32768 on 64^3).  On 128^3 (512 tiles) 34 against 53 us for 8192, equal at 32768.
constexpr long long kSmallN = 16384;
constexpr int kSmallBlock = 256;        // particles per workgroup of k_cells_small
constexpr int kSmallThreads = 1024;     // per tile of k_deposit_small
constexpr int kLooksAhead = 8;          // packed cells a thread loads at a time
static_assert(kSmallN <= 65536, "the list of a tile keeps 16-bit indices");

// Cell record, packed cell (10 bits an axis) and FP32 mass of every particle,
// and each workgroup's max |m|.
template <typename T, typename M>
__global__ __launch_bounds__(kSmallBlock) void k_cells_small(const PosSrc<T> src, const M* __restrict__ m, int n,
                                                             const CellMap cm, PartRec* __restrict__ rec,
                                                             unsigned* __restrict__ cell, float* __restrict__ mass,
                                                             float* __restrict__ mpart) {
  __shared__ float wmax[kSmallBlock / 64];
  const int i = blockIdx.x * kSmallBlock + threadIdx.x;
  float mf = 0.0f;
  if (i < n) {
    const long long o = (long long)i * src.stride;
    const double p[3] = {(double)src.x[o], (double)src.y[o], (double)src.z[o]};
    mf = (float)m[i];
    int c[3];
    unsigned long long f[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) cell_fix(p[a], cm, c[a], f[a]);
    rec[i] = encode_rec(c, f, mf);
    cell[i] = (unsigned)c[0] | ((unsigned)c[1] << 10) | ((unsigned)c[2] << 20);
    mass[i] = mf;
  }
  float am = fabsf(mf);
  for (int off = 32; off > 0; off >>= 1) am = fmaxf(am, __shfl_xor(am, off));
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = am;
  __syncthreads();
  if (threadIdx.x == 0) mpart[blockIdx.x] = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
}

// One workgroup per tile of T^3 cells: the fixed-point scale from the partial
// maxima, the total fixed-point mass, and the CIC targets inside the tile.
// Workgroup 0 leaves the scale and the mean in sc for the readers of records.
template <int T>
__global__ __launch_bounds__(kSmallThreads) void k_deposit_small(const PartRec* __restrict__ rec,
                                                                 const unsigned* __restrict__ cell,
                                                                 const float* __restrict__ mass,
                                                                 const float* __restrict__ mpart, int n,
                                                                 const CellMap cm, int nt, SolveScalars* sc,
                                                                 float* __restrict__ rho, long long rho_plane,
                                                                 float* __restrict__ keep) {
  constexpr int T3 = T * T * T, NT = kSmallThreads, WAVES = NT / 64;
  __shared__ unsigned long long acc[T3];
  __shared__ float wmax[WAVES];
  __shared__ long long wsum[WAVES];
  __shared__ unsigned short list[kSmallN];
  __shared__ unsigned hits;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nm = cm.nm;
  const int ux = (int)blockIdx.x % nt, uy = ((int)blockIdx.x / nt) % nt, uz = (int)blockIdx.x / (nt * nt);
  for (int c = tid; c < T3; c += NT) acc[c] = 0ull;
  if (tid == 0) hits = 0u;
  float am = 0.0f;
  const int parts = (n + kSmallBlock - 1) / kSmallBlock;
  for (int k = tid; k < parts; k += NT) am = fmaxf(am, mpart[k]);
  for (int off = 32; off > 0; off >>= 1) am = fmaxf(am, __shfl_xor(am, off));
  if (lane == 0) wmax[wave] = am;
  __syncthreads();
  am = wmax[0];
#pragma unroll
  for (int k = 1; k < WAVES; ++k) am = fmaxf(am, wmax[k]);
  const int shift = fixed_shift(am, n);
  const double scale = ldexp(1.0, shift);
  // All packed cells, eight a thread and round (the loads of a round are in
  // flight together); those that reach the tile join the list, so that the
  // work on them is spread over all threads whatever their order.
  long long q = 0;
  const int u[3] = {ux * T, uy * T, uz * T};
  for (int i0 = tid; i0 < n; i0 += NT * kLooksAhead) {
    unsigned c[kLooksAhead];
    float mf[kLooksAhead];
#pragma unroll
    for (int k = 0; k < kLooksAhead; ++k) {
      const int i = i0 + k * NT;
      c[k] = i < n ? cell[i] : 0xffffffffu;
      mf[k] = i < n ? mass[i] : 0.0f;
    }
#pragma unroll
    for (int k = 0; k < kLooksAhead; ++k) {
      q += rint_small((double)mf[k] * scale);
      bool reach = c[k] != 0xffffffffu;
#pragma unroll
      for (int a = 0; a < 3; ++a) {
        const int l = (int)((c[k] >> (10 * a)) & 1023u) - u[a];
        // the cell itself or the next one, which wraps to 0
        reach = reach && ((unsigned)(l + 1) <= (unsigned)T || (l == nm - 1 && u[a] == 0));
      }
      const unsigned long long any = __ballot(reach);
      if (any) {
        const int first = __ffsll((long long)any) - 1;
        unsigned at = 0u;
        if (lane == first) at = atomicAdd(&hits, (unsigned)__popcll(any));
        at = __shfl(at, first) + (unsigned)__popcll(any & ((1ull << lane) - 1ull));
        if (reach) list[at] = (unsigned short)(i0 + k * NT);
      }
    }
  }
  __syncthreads();
  const int nhits = (int)hits;
  for (int e = tid; e < nhits; e += NT) {
    const PartRec p = rec[list[e]];
    const double fx = rec_frac(p, 0), fy = rec_frac(p, 1), fz = rec_frac(p, 2);
    const double ms = (double)rec_mass(p) * scale;
    const double wx[2] = {1.0 - fx, fx}, wy[2] = {1.0 - fy, fy};
    const double wz[2] = {(1.0 - fz) * ms, fz * ms};
    int l[3][2];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int b = rec_cell(p, a);
      l[a][0] = b - u[a];
      l[a][1] = (b + 1 == nm ? 0 : b + 1) - u[a];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int cx = l[0][k & 1], cy = l[1][(k >> 1) & 1], cz = l[2][k >> 2];
      if ((unsigned)cx < (unsigned)T && (unsigned)cy < (unsigned)T && (unsigned)cz < (unsigned)T)
        atomicAdd(acc + (cz * T + cy) * T + cx,
                  (unsigned long long)rint_small(wx[k & 1] * (wy[(k >> 1) & 1] * wz[k >> 2])));
    }
  }
  for (int off = 32; off > 0; off >>= 1) q += __shfl_xor(q, off);
  if (lane == 0) wsum[wave] = q;
  __syncthreads();
  q = 0;
#pragma unroll
  for (int k = 0; k < WAVES; ++k) q += wsum[k];
  const long long qmean = (long long)((unsigned long long)q / (unsigned long long)((long long)nm * nm * nm));
  const double unit = ldexp(1.0, -shift);
  for (int c = tid; c < T3; c += NT) {
    const int lx = c % T, ly = (c / T) % T, lz = c / (T * T);
    const size_t row = (size_t)(uy * T + ly) * nm + (ux * T + lx);
    const long long v = (long long)acc[c];
    rho[(size_t)(uz * T + lz) * rho_plane + row] = (float)((double)(v - qmean) * unit);
    if (keep) keep[(size_t)(uz * T + lz) * nm * nm + row] = (float)((double)v * unit);
  }
  if (blockIdx.x == 0 && tid == 0) {
    sc->mmax_bits = __float_as_uint(am);
    sc->qmean = qmean;
    sc->shift = shift;
    sc->plain = (unsigned)n;
  }
}

// Threads of the plane kernels: one radix-8 butterfly each.
template <int N>
struct PlaneCfg {
  static constexpr int H = N / 2, LS = H + 1;
  static constexpr int T = N <= 64 ? 256 : 1024;
};

// x then y transform of one z plane (rho: its N rows of N reals, in P's own
// memory).
template <int N>
__device__ __forceinline__ void plane_fwd_body(float2* __restrict__ P, const float2* __restrict__ tw_g) {
  constexpr int H = PlaneCfg<N>::H, LS = PlaneCfg<N>::LS, T = PlaneCfg<N>::T;
  using FX = RegFft<H, false, false, N, T, LS, 1, false, N>;
  using FY = RegFft<N, false, false, H, T, 1, LS, true, N>;
  __shared__ float2 buf[N * LS];
  __shared__ float2 tw[N];
  const int tid = threadIdx.x;
  for (int e = tid; e < N; e += T) tw[e] = tw_g[e];
  float2* plane = P + (size_t)blockIdx.x * mesh_plane(N);
  {
    float2 vin[FX::PER0][FX::R0], vout[FX::PERL][FX::RL];
    for_edge<H, FX::R0, N, T, false>(tid, [&](int p, int r, int l, int i, bool ok) {
      if (ok) vin[p][r] = plane[l * H + i];
    });
    FX::run(vin, vout, buf, tw, tid);
    __syncthreads();
    for_edge<H, FX::RL, N, T, false>(tid, [&](int p, int r, int l, int i, bool ok) {
      if (ok) buf[l * LS + i] = vout[p][r];
    });
  }
  __syncthreads();
  constexpr int TOT = N * H, PER = (TOT + T - 1) / T;
  float2 x[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int e = tid + p * T;
    if ((TOT % T == 0) || e < TOT) {
      const int r = e / H, k = e % H;
      const float2 zk = buf[r * LS + k];
      if (k == 0) {
        x[p] = make_float2(zk.x + zk.y, zk.x - zk.y);
      } else {
        const float2 zc = cconj(buf[r * LS + (H - k)]);
        const float2 E = make_float2(0.5f * (zk.x + zc.x), 0.5f * (zk.y + zc.y));
        // O = (zk - zc) / (2i)
        const float2 O = make_float2(0.5f * (zk.y - zc.y), -0.5f * (zk.x - zc.x));
        x[p] = cadd(E, cmul(tw[k], O));
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int p = 0; p < PER; ++p) {
    const int e = tid + p * T;
    if ((TOT % T == 0) || e < TOT) buf[(e / H) * LS + e % H] = x[p];
  }
  __syncthreads();
  float2 vin[FY::PER0][FY::R0], vout[FY::PERL][FY::RL];
  for_edge<N, FY::R0, H, T, true>(tid, [&](int p, int r, int l, int i, bool ok) {
    if (ok) vin[p][r] = buf[i * LS + l];
  });
  // begins with a barrier: every thread has its values
  FY::run(vin, vout, buf, tw, tid);
  for_edge<N, FY::RL, H, T, true>(tid, [&](int p, int r, int l, int i, bool ok) {
    if (ok) plane[i * H + l] = vout[p][r];
  });
}

template <int N>
__global__ __launch_bounds__(PlaneCfg<N>::T) void k_plane_fwd(float2* __restrict__ P, const float2* __restrict__ tw) {
  plane_fwd_body<N>(P, tw);
}
template <int N>
__global__ __launch_bounds__(PlaneCfg<N>::T) void k_plane_fwd_box(const BoxArgs* __restrict__ bx,
                                                                  const float2* __restrict__ tw) {
  plane_fwd_body<N>(bx[blockIdx.z].P, tw);
}

// The z pass of fft_z_green_body for whole ky rows (workgroups [0, N)), and
// the packed column of fft_z_green_col0_body (workgroups N ..): A = phi,
// B = -i n_z phi after the inverse z transform, and P = A.
template <int N>
__device__ __forceinline__ void z_small_body(float2* P, float2* A, float2* B, const float2* __restrict__ tw_g,
                                             const GreenParams& gp) {
  constexpr int T = PlaneCfg<N>::T;
  if (blockIdx.x >= N) {
    fft_z_green_col0_body<N, T>(P, A, B, tw_g, gp, (int)blockIdx.x - N, P);
    return;
  }
  fft_z_green_body<N, N / 2, T>(P, A, B, tw_g, gp, 0, (int)blockIdx.x, P);
}
template <int N>
__global__ __launch_bounds__(PlaneCfg<N>::T) void k_z_small(float2* P, float2* A, float2* B,
                                                            const float2* __restrict__ tw, const GreenParams gp) {
  z_small_body<N>(P, A, B, tw, gp);
}
template <int N>
__global__ __launch_bounds__(PlaneCfg<N>::T) void k_z_small_box(const BoxArgs* __restrict__ bx,
                                                                const float2* __restrict__ tw) {
  const BoxArgs& b = bx[blockIdx.z];
  z_small_body<N>(b.P, b.A, b.B, tw, b.gp);
}

// y then x inverse transform of plane blockIdx.x of field blockIdx.y + field0
// (0: A times -i n_x, 1: P times -i n_y, 2: B, in place; 3: the potential from A into pot,
// scaled, which runs before the others overwrite A).
template <int N>
__device__ __forceinline__ void plane_inv_body(float2* A, float2* P, float2* B, float2* pot,
                                               const float2* __restrict__ tw_g, int field0, float pot_scale) {
  constexpr int H = PlaneCfg<N>::H, LS = PlaneCfg<N>::LS, T = PlaneCfg<N>::T;
  using FY = RegFft<N, true, false, H, T, 1, LS, true, N>;
  using FX = RegFft<H, true, false, N, T, LS, 1, false, N>;
  __shared__ float2 buf[N * LS];
  __shared__ float2 tw[N];
  const int tid = threadIdx.x;
  for (int e = tid; e < N; e += T) tw[e] = tw_g[e];
  const int field = blockIdx.y + field0;
  float2* plane = (field == 1 ? P : field == 2 ? B : A) + (size_t)blockIdx.x * mesh_plane(N);
  {
    float2 vin[FY::PER0][FY::R0], vout[FY::PERL][FY::RL];
    for_edge<N, FY::R0, H, T, true>(tid, [&](int p, int r, int l, int i, bool ok) {
      vin[p][r] = ok ? plane[i * H + l] : make_float2(0.f, 0.f);
    });
    // two calls, so that the product contracts into the first butterfly as it
    // does in k_fft_y_inv
    if (field == 1) {
      for_edge<N, FY::R0, H, T, true>(tid, [&](int p, int r, int l, int i, bool ok) {
        const float nye = (i == N / 2) ? 0.0f : (float)freq_of(i, N);
        vin[p][r] = make_float2(nye * vin[p][r].y, -nye * vin[p][r].x);
      });
      FY::run(vin, vout, buf, tw, tid);
    } else {
      FY::run(vin, vout, buf, tw, tid);
    }
    __syncthreads();
    for_edge<N, FY::RL, H, T, true>(tid, [&](int p, int r, int l, int i, bool ok) {
      float2 v = vout[p][r];
      // -i n_x; slot 0 holds DC (n=0) and Nyquist (n_eff=0): both vanish
      if (field == 0) v = make_float2((float)l * v.y, -(float)l * v.x);
      if (ok) buf[i * LS + l] = v;
    });
  }
  __syncthreads();
  float2 vin[FX::PER0][FX::R0], vout[FX::PERL][FX::RL];
  for_edge<H, FX::R0, N, T, false>(tid, [&](int p, int r, int l, int k, bool ok) {
    if (!ok) return;
    const float2 y = buf[l * LS + k];
    if (k == 0) {
      vin[p][r] = make_float2(y.x + y.y, y.x - y.y);
    } else {
      const float2 xc = cconj(buf[l * LS + (H - k)]);
      const float2 sm = cadd(y, xc);
      // Z = (X_k + conj X_{H-k}) + i (X_k - conj X_{H-k}) e^{+2 pi i k/N}
      const float2 t = cmul(csub(y, xc), cconj(tw[k]));
      vin[p][r] = make_float2(sm.x - t.y, sm.y + t.x);
    }
  });
  FX::run(vin, vout, buf, tw, tid);
  float2* dst = field == 3 ? pot + (size_t)blockIdx.x * N * H : plane;
  const float sc = field == 3 ? pot_scale : 1.0f;
  for_edge<H, FX::RL, N, T, false>(tid, [&](int p, int r, int l, int i, bool ok) {
    if (ok) dst[l * H + i] = make_float2(vout[p][r].x * sc, vout[p][r].y * sc);
  });
}

template <int N>
__global__ __launch_bounds__(PlaneCfg<N>::T) void k_plane_inv(float2* A, float2* P, float2* B, float2* pot,
                                                              const float2* __restrict__ tw, int field0,
                                                              float pot_scale) {
  plane_inv_body<N>(A, P, B, pot, tw, field0, pot_scale);
}
template <int N>
__global__ __launch_bounds__(PlaneCfg<N>::T) void k_plane_inv_box(const BoxArgs* __restrict__ bx,
                                                                  const float2* __restrict__ tw) {
  const BoxArgs& b = bx[blockIdx.z];
  plane_inv_body<N>(b.A, b.P, b.B, nullptr, tw, 0, 1.0f);
}

}  // namespace gng
