// Fixed-field steps of real walkers between two orthonormalisations, a walker per workgroup (see
// ff_fused.hpp; the formulas are those of adjoint.cpp).
//
// At lattice sizes a walker's block is a few tens of KB and a step some 0.2 to 1 MFLOP, so a step by
// step launch is bound by launch latency and by passes over the walkers: scale, product, copy in the
// forward sweep; two scalings, two transposes, two products, row sums and their reduction in the
// reverse one.  Here the block stays in LDS for all the steps, each wave keeps its rows of B (or B^T)
// in registers as MFMA fragments, the HS factors come from two values per site and the field's
// hash, and only the stored W of each step passes through memory, as real numbers.  The reverse
// kernel accumulates its share of Bbar and Ubar in registers over steps and walkers and adds it to
// its own slot once.
//
// 512 walkers of 64 x 28, per step and spin: forward 7.5 us, reverse 13.3 us; step by step the launches
// took 26 and 215 us (117 of it a serial sum over walkers).
#include "ff_fused.hpp"

#include <algorithm>

namespace {

constexpr int M_MAX = 112, N_MAX = 64, NT = 256;

// LDS stride of a column: 20 mod 32 doubles, so that both fragment reads (16 rows of four columns,
// four rows of 16 columns) spread over the banks
constexpr __host__ __device__ int lds_ld(int fm) { return 16 * fm + (52 - (16 * fm) % 32) % 32; }
static_assert(lds_ld(4) % 32 == 20 && lds_ld(7) % 32 == 20 && lds_ld(5) >= 80, "column stride");

__device__ __forceinline__ double field_sign(unsigned long long key, int s, int nw, int M, int w, int i) {
  const unsigned long long k = ((unsigned long long)s * nw + w) * (unsigned long long)M + i;
  return afqmc_uniform_dev(key, k) < 0.5 ? -1.0 : 1.0;
}

// the HS factor of a site for x = +1 and x = -1
__device__ __forceinline__ void site_factors(const FfFusedArgs& p, int i, double* plus, double* minus) {
  const zd g = cscale(p.gamma[i], p.sigma);
  *plus = cmul(cexp_d(g), p.cdiag[i]).re;
  *minus = cmul(cexp_d(cmk<double>(-g.re, -g.im)), p.cdiag[i]).re;
}

template <int FM, int FN>
__device__ __forceinline__ void load_block(const FfFusedArgs& p, int w, double* Wl) {
  constexpr int LD = lds_ld(FM);
  const zd* W = p.W + (long long)w * p.M * p.N;
  for (int n = threadIdx.x >> 6; n < 16 * FN; n += NT / 64)
    for (int m = threadIdx.x & 63; m < 16 * FM; m += 64)
      Wl[n * LD + m] = m < p.M && n < p.N ? W[m + (long long)n * p.M].re : 0.0;
}
template <int FM, int FN>
__device__ __forceinline__ void store_block(const FfFusedArgs& p, int w, const double* Wl) {
  constexpr int LD = lds_ld(FM);
  zd* W = p.W + (long long)w * p.M * p.N;
  for (int n = threadIdx.x >> 6; n < p.N; n += NT / 64)
    for (int m = threadIdx.x & 63; m < p.M; m += 64) W[m + (long long)n * p.M] = cmk<double>(Wl[n * LD + m], 0.0);
}

template <int FM, int FN>
__global__ __launch_bounds__(NT) void ff_forward_kernel(FfFusedArgs p) {
  constexpr int RT = (FM + 3) / 4, LD = lds_ld(FM);  // row tiles wave, wave + 4, ... are the wave's
  typedef mfma_traits<double> mt;
  extern __shared__ __align__(16) double lds[];
  double *Wl = lds, *plus = Wl + 16 * FN * LD, *minus = plus + 16 * FM, *ds = minus + 16 * FM;
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = p.M, N = p.N, w = blockIdx.x;
  double a[RT][4 * FM];  // B(row, k); past M: any valid element (k there meets a zero, rows are not stored)
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int k = 0; k < 4 * FM; ++k)
      a[t][k] = p.B[min(16 * (wave + 4 * t) + lr, M - 1) + (long long)min(4 * k + lk, M - 1) * M];
  load_block<FM, FN>(p, w, Wl);
  for (int i = tid; i < 16 * FM; i += NT) {
    plus[i] = minus[i] = 0.0;
    if (i < M) site_factors(p, i, &plus[i], &minus[i]);
  }
  __syncthreads();
  for (int st = p.s0; st < p.s1; ++st) {
    if (p.Q) {
      double* q = p.Q + ((long long)(st - p.q0) * p.nw + w) * M * N;
      for (int n = wave; n < N; n += NT / 64)
        for (int m = lane; m < M; m += 64) q[m + (long long)n * M] = Wl[n * LD + m];
    }
    if (tid < 16 * FM) ds[tid] = field_sign(p.key, st, p.nw, M, w, tid) < 0.0 ? minus[tid] : plus[tid];
    __syncthreads();
    typename mt::acc_t acc[RT][FN];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[t][j] = typename mt::acc_t{0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < 4 * FM; ++k) {
      const double d = ds[4 * k + lk];
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const double b = d * Wl[(16 * j + lr) * LD + 4 * k + lk];
#pragma unroll
        for (int t = 0; t < RT; ++t)
          if (wave + 4 * t < FM) acc[t][j] = mt::mma(a[t][k], b, acc[t][j]);
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = 16 * (wave + 4 * t) + mt::row(lk, r);
          if (m < M) Wl[(16 * j + lr) * LD + m] = acc[t][j][r];
        }
    __syncthreads();
  }
  store_block<FM, FN>(p, w, Wl);
}

template <int FM, int FN>
__global__ __launch_bounds__(NT) void ff_reverse_kernel(FfFusedArgs p) {
  constexpr int RT = (FM + 3) / 4, LD = lds_ld(FM);
  typedef mfma_traits<double> mt;
  extern __shared__ __align__(16) double lds[];
  double *Wl = lds, *Dq = Wl + 16 * FN * LD, *plus = Dq + 16 * FN * LD, *minus = plus + 16 * FM;
  double *ds = minus + 16 * FM, *dl = ds + 16 * FM;
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int M = p.M, N = p.N;
  double a[RT][4 * FM];  // B^T(row, k)
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int k = 0; k < 4 * FM; ++k)
      a[t][k] = p.B[min(4 * k + lk, M - 1) + (long long)min(16 * (wave + 4 * t) + lr, M - 1) * M];
  for (int i = tid; i < 16 * FM; i += NT) {
    plus[i] = minus[i] = 0.0;
    if (i < M) site_factors(p, i, &plus[i], &minus[i]);
  }
  for (int e = tid; e < 16 * FN * LD; e += NT) Dq[e] = 0.0;
  typename mt::acc_t bb[RT][FM];
  double ub[RT][4];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
#pragma unroll
    for (int j = 0; j < FM; ++j) bb[t][j] = typename mt::acc_t{0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < 4; ++r) ub[t][r] = 0.0;
  }
  for (int w = blockIdx.x; w < p.nw; w += gridDim.x) {
    load_block<FM, FN>(p, w, Wl);
    __syncthreads();
    for (int st = p.s1 - 1; st >= p.s0; --st) {
      const double* q = p.Q + ((long long)(st - p.q0) * p.nw + w) * M * N;
      for (int m = lane; m < M; m += 64) {
        const double x = field_sign(p.key, st, p.nw, M, w, m), d = x < 0.0 ? minus[m] : plus[m];
        if (wave == 0) {
          ds[m] = d;
          dl[m] = p.sigma * x * p.gprime[m].re - 0.5 * p.dt;
        }
        for (int n = wave; n < N; n += NT / 64) Dq[n * LD + m] = d * q[m + (long long)n * M];
      }
      __syncthreads();
      for (int k = 0; k < N; k += 4) {  // Bbar += Wbar (D Q)^T; columns past N are zero
        const double* v = Dq + (k + lk) * LD + lr;
        const double* u = Wl + (k + lk) * LD + lr;
        double b[FM];
#pragma unroll
        for (int j = 0; j < FM; ++j) b[j] = v[16 * j];
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          if (wave + 4 * t >= FM) continue;
          const double c = u[16 * (wave + 4 * t)];
#pragma unroll
          for (int j = 0; j < FM; ++j) bb[t][j] = mt::mma(c, b[j], bb[t][j]);
        }
      }
      typename mt::acc_t acc[RT][FN];  // Ybar = B^T Wbar
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[t][j] = typename mt::acc_t{0, 0, 0, 0};
#pragma unroll
      for (int k = 0; k < 4 * FM; ++k)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const double b = Wl[(16 * j + lr) * LD + 4 * k + lk];
#pragma unroll
          for (int t = 0; t < RT; ++t)
            if (wave + 4 * t < FM) acc[t][j] = mt::mma(a[t][k], b, acc[t][j]);
        }
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = 16 * (wave + 4 * t) + mt::row(lk, r);
          if (m >= M) continue;
          double u = 0.0;
#pragma unroll
          for (int j = 0; j < FN; ++j) u += acc[t][j][r] * Dq[(16 * j + lr) * LD + m];
          ub[t][r] += u * dl[m];
        }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = 16 * (wave + 4 * t) + mt::row(lk, r);
          if (m >= M) continue;
          const double d = ds[m];
#pragma unroll
          for (int j = 0; j < FN; ++j) Wl[(16 * j + lr) * LD + m] = d * acc[t][j][r];
        }
      __syncthreads();
    }
    store_block<FM, FN>(p, w, Wl);
    __syncthreads();
  }
  double* bo = p.bpart + (long long)blockIdx.x * M * M;
  double* uo = p.upart + (long long)blockIdx.x * M;
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * (wave + 4 * t) + mt::row(lk, r);
      double u = ub[t][r];
#pragma unroll
      for (int o = 8; o > 0; o >>= 1) u += __shfl_xor(u, o, 64);
      if (m >= M) continue;
      if (lr == 0) uo[m] += u;
#pragma unroll
      for (int j = 0; j < FM; ++j) {
        const int n = 16 * j + lr;
        if (n < M) bo[m + (long long)n * M] += bb[t][j][r];
      }
    }
}

// 16 elements by 16 segments of slots a workgroup, the segments added in order
__global__ __launch_bounds__(256) void ff_sum_kernel(int slots, int per, const double* part, zd* out, int accumulate) {
  __shared__ double sh[16][16];
  const int el = threadIdx.x & 15, seg = threadIdx.x >> 4, e = blockIdx.x * 16 + el;
  double s = 0.0;
  if (e < per)
    for (int k = seg; k < slots; k += 16) s += part[(long long)k * per + e];
  sh[seg][el] = s;
  __syncthreads();
  if (seg != 0 || e >= per) return;
  for (int k = 1; k < 16; ++k) s += sh[k][el];
  out[e] = accumulate ? cadd(out[e], cmk<double>(s, 0.0)) : cmk<double>(s, 0.0);
}

template <int FM, int FN, bool REV>
int run(const FfFusedArgs& a, hipStream_t s) {
  auto kernel = REV ? ff_reverse_kernel<FM, FN> : ff_forward_kernel<FM, FN>;
  const int lds = (int)sizeof(double) * ((REV ? 2 : 1) * 16 * FN * lds_ld(FM) + (REV ? 4 : 3) * 16 * FM);
  HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  hipLaunchKernelGGL(kernel, dim3(REV ? std::min(a.nw, FF_SLOTS) : a.nw), dim3(NT), lds, s, a);
  HIP_LAUNCH_CHECK();
  return 0;
}

template <int FM, bool REV>
int pick_cols(const FfFusedArgs& a, hipStream_t s) {
  if (a.N <= 16) return run<FM, 1, REV>(a, s);
  return a.N <= 32 ? run<FM, 2, REV>(a, s) : run<FM, 4, REV>(a, s);
}

template <bool REV>
int pick(const FfFusedArgs& a, hipStream_t s) {
  if (a.nw <= 0 || a.s1 <= a.s0) return 0;
  REQUIRE(ff_fused_ok(a.M, a.N), "fused fixed-field steps: %d x %d blocks not supported", a.M, a.N);
  switch ((a.M + 15) / 16) {
    case 1: return pick_cols<1, REV>(a, s);
    case 2: return pick_cols<2, REV>(a, s);
    case 3: return pick_cols<3, REV>(a, s);
    case 4: return pick_cols<4, REV>(a, s);
    case 5: return pick_cols<5, REV>(a, s);
    case 6: return pick_cols<6, REV>(a, s);
    default: return pick_cols<7, REV>(a, s);
  }
}

}  // namespace

bool ff_fused_ok(int M, int N) { return M >= 1 && M <= M_MAX && N >= 1 && N <= N_MAX; }
int launch_ff_forward(const FfFusedArgs& a, hipStream_t s) { return pick<false>(a, s); }
int launch_ff_reverse(const FfFusedArgs& a, hipStream_t s) { return pick<true>(a, s); }
int launch_ff_sum(int slots, int per, const double* part, zd* out, int accumulate, hipStream_t s) {
  hipLaunchKernelGGL(ff_sum_kernel, dim3((per + 15) / 16), dim3(256), 0, s, slots, per, part, out, accumulate);
  HIP_LAUNCH_CHECK();
  return 0;
}
