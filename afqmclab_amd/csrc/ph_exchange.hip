// tr(A_g^T X_w A_g^T X_w) and tr(A_g^T X_w) (see ph_exchange.hpp).
//
// The product is 4 L Ns^2 operations per walker and vector and only its two traces are wanted, so it
// is bound by the matrix cores as long as D stays on the chip.  A workgroup keeps one walker's X in
// LDS as 2 Ns real columns (re, im interleaved) and runs over the vectors; a wave takes batches of gb
// vectors whose Ns gb columns are the rows of one MFMA tile (16 FM x 16 FN accumulators cover all
// of D for the batch), reads A straight from global memory into fragments (all workgroups pass over
// the vectors in the same order, so A comes from the caches) and needs no barrier: the waves of a
// workgroup draw their batches from a counter in LDS.  K is permuted, the same way on both sides,
// so that a lane reads four consecutive elements at a time.  The traces need D transposed: the wave
// writes gc vectors' blocks at a time to its own part of LDS and sums the products in FP64.
//
// 1024 walkers, 1600 vectors, L = 200, Ns = 40, FP32, per spin: 18.9 ms, 111 TFLOP/s of the 147 that a
// large FP32 matrix product reaches; the complex product with D in memory and a separate trace took
// 32.0 + 6.4 ms.  Seven waves fit the LDS there, so one of the four matrix cores has a single wave and
// idles during its traces.  Measured without gain: whole 128-byte lines of A per load step.
#include "ph_exchange.hpp"

#include <algorithm>
#include <cstring>

namespace {

constexpr int LDS_MAX = 160 * 1024;
constexpr int NS_MAX = 48;

struct KArgs {
  PhExchangeArgs p;
  int gb, gc, slice;  // vectors per batch, per trace pass; batches per workgroup
  int xbytes, sbytes; // LDS of X, of a wave's trace block
};

template <typename T> struct vec4;
template <> struct vec4<float> { typedef float4 type; };
template <> struct vec4<double> { typedef double4 type; };

constexpr __host__ __device__ int trace_ld(int fn) { return 16 * fn + 4; }  // four rows apart: 16 banks apart

// orders the wave's own LDS writes before its lanes' reads of each other's
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// VEC: L is a multiple of 4, so that a lane's four elements of A are aligned
template <typename T, int FM, int FN, int NT, bool VEC>
__global__ __launch_bounds__(NT, 1) void exchange_traces_kernel(KArgs q) {
  typedef typename mfma_traits<T>::acc_t acc_t;
  typedef cplx<T> ct;
  constexpr int COLS = 16 * FN;
  const PhExchangeArgs& p = q.p;
  const int w = blockIdx.x, L = p.L, Ns = p.Ns;
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  extern __shared__ __align__(16) unsigned char lds[];
  T* Xs = reinterpret_cast<T*>(lds);  // (k, c) at ((k / 4) COLS + c) 4 + k % 4, zero past L and 2 Ns
  T* Dw = reinterpret_cast<T*>(lds + q.xbytes + wave * q.sbytes);
  int* next = reinterpret_cast<int*>(lds + q.xbytes + (blockDim.x >> 6) * q.sbytes);

  const ct* X = reinterpret_cast<const ct*>(p.X) + (long long)w * L * Ns;
  const int quads = (L + 3) / 4;
  for (int e = tid; e < quads * 4 * (COLS / 2); e += blockDim.x) {
    const int k = e % (quads * 4), j = e / (quads * 4);
    const ct v = k < L && j < Ns ? X[k + (long long)j * L] : cmk<T>((T)0, (T)0);
    T* o = Xs + ((long long)(k >> 2) * COLS + 2 * j) * 4 + (k & 3);
    o[0] = v.re;
    o[4] = v.im;
  }
  const int nb = (p.G + q.gb - 1) / q.gb;
  const int b_end = min(nb, ((int)blockIdx.y + 1) * q.slice);
  if (tid == 0) *next = blockIdx.y * q.slice;
  __syncthreads();

  constexpr int ldd = trace_ld(FN);
  for (;;) {
    int b = 0;
    if (lane == 0) b = atomicAdd(next, 1);
    b = __builtin_amdgcn_readfirstlane(b);
    if (b >= b_end) break;
    const int g0 = b * q.gb, ng = min(q.gb, p.G - g0), rows = ng * Ns;
    const T* A = reinterpret_cast<const T*>(p.A) + (long long)g0 * Ns * L;
    unsigned ao[FM];  // rows past the batch repeat its last one; nothing reads their results
#pragma unroll
    for (int i = 0; i < FM; ++i) ao[i] = (unsigned)(min(16 * i + lr, rows - 1) * L);
    acc_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int c = 0; c < FN; ++c) acc[i][c] = acc_t{0, 0, 0, 0};

    auto load = [&](int k0, T (*r)[4]) {
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const T* s = A + (ao[i] + (unsigned)(k0 + 4 * lk));
        if constexpr (VEC) {
          const typename vec4<T>::type v = *reinterpret_cast<const typename vec4<T>::type*>(s);
          r[i][0] = v.x; r[i][1] = v.y; r[i][2] = v.z; r[i][3] = v.w;
        } else {
#pragma unroll
          for (int j = 0; j < 4; ++j) r[i][j] = s[j];
        }
      }
    };
    auto multiply = [&](int quad, T (*r)[4]) {
      T x[FN][4];
#pragma unroll
      for (int c = 0; c < FN; ++c) {
        const typename vec4<T>::type v =
            *reinterpret_cast<const typename vec4<T>::type*>(Xs + (quad * COLS + 16 * c + lr) * 4);
        x[c][0] = v.x; x[c][1] = v.y; x[c][2] = v.z; x[c][3] = v.w;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int c = 0; c < FN; ++c) acc[i][c] = mfma_traits<T>::mma(r[i][j], x[c][j], acc[i][c]);
    };
    T a[FM][4], an[FM][4];
    const int nk = L / 16, k0 = 16 * nk;
    if (nk > 0) load(0, an);
    for (int kk = 0; kk < nk; ++kk) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) a[i][j] = an[i][j];
      if (kk + 1 < nk) load(16 * (kk + 1), an);
      multiply(4 * kk + lk, a);
    }
    if (k0 < L) {  // the last L % 16 rows of K, four at a time
      T at[4][FM];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          const int k = k0 + 4 * t + lk;
          const T v = A[ao[i] + (unsigned)(k < L ? k : 0)];
          at[t][i] = k < L ? v : (T)0;
        }
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        if (k0 + 4 * t >= L) break;
        T xt[FN];
#pragma unroll
        for (int c = 0; c < FN; ++c) xt[c] = Xs[((k0 / 4 + t) * COLS + 16 * c + lr) * 4 + lk];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int c = 0; c < FN; ++c) acc[i][c] = mfma_traits<T>::mma(at[t][i], xt[c], acc[i][c]);
      }
    }

    for (int p0 = 0; p0 < ng; p0 += q.gc) {
      const int pg = min(q.gc, ng - p0), r0 = p0 * Ns, nr = pg * Ns;
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        if (16 * i + 15 < r0 || 16 * i >= r0 + nr) continue;
        // rows of other vectors go to a spare last row, so no write depends on a branch
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = 16 * i + mfma_traits<T>::row(lk, r) - r0;
          T* o = Dw + ((unsigned)row < (unsigned)nr ? row : q.gc * Ns) * ldd + lr;
#pragma unroll
          for (int c = 0; c < FN; ++c) o[16 * c] = acc[i][c][r];
        }
      }
      wave_sync();
      // LPG lanes per vector, a lane per column; a row and a column of D per turn, both read from LDS
      constexpr int LPG = FN <= 2 ? 16 : FN <= 4 ? 32 : 64;
      const int sub = lane % LPG, col = min(sub, Ns - 1);
      for (int gi = lane / LPG; gi - lane / LPG < pg; gi += 64 / LPG) {
        const bool in = gi < pg;
        const T* D = Dw + (in ? gi : 0) * Ns * ldd;
        const T *Dr = D + 2 * col, *Dc = D + col * ldd;
        double er = 0, ei = 0;
#pragma unroll 8
        for (int i = 0; i < Ns; ++i) {
          const zd u = to_zd(*reinterpret_cast<const ct*>(Dr + i * ldd));
          const zd v = to_zd(*reinterpret_cast<const ct*>(Dc + 2 * i));
          er += u.re * v.re - u.im * v.im;
          ei += u.re * v.im + u.im * v.re;
        }
        const zd dg = to_zd(*reinterpret_cast<const ct*>(Dc + 2 * col));
        double tr = dg.re, ti = dg.im;
        if (sub >= Ns) er = ei = tr = ti = 0;
#pragma unroll
        for (int o = LPG / 2; o > 0; o >>= 1) {
          er += __shfl_xor(er, o, 64);
          ei += __shfl_xor(ei, o, 64);
          tr += __shfl_xor(tr, o, 64);
          ti += __shfl_xor(ti, o, 64);
        }
        if (in && sub == 0) {
          const long long at = (long long)w * p.G + g0 + p0 + gi;
          ct* bg = reinterpret_cast<ct*>(p.bg) + at;
          zd ev = cmk<double>(er, ei);
          ct bv = cmk<T>((T)tr, (T)ti);
          if (p.accumulate) {
            ev = cadd(p.ex[at], ev);
            bv = cadd(*bg, bv);
          }
          p.ex[at] = ev;
          *bg = bv;
        }
      }
      wave_sync();
    }
  }
}

// Tiles: FN column tiles hold 2 Ns columns; FM row tiles are those that gb whole vectors fill best at
// the largest Ns of each FN: 128, 128, 96, 64, 80, 96 rows in FP32.  FP64 accumulators take twice the
// registers, so one vector (48 rows) a batch above 32 columns.
template <typename T>
constexpr int tile_rows(int fn) {
  return fn <= 2 ? 8 : fn == 3 ? 6 : fn == 4 ? 4 : sizeof(T) == 8 ? 3 : fn;
}

struct Plan {
  int fn, gb, gc, waves, xbytes, sbytes, lds;
};
template <typename T>
bool plan(int L, int Ns, Plan* o) {
  if (Ns < 1 || Ns > NS_MAX || L > (1 << 20)) return false;
  o->fn = (2 * Ns + 15) / 16;
  o->gb = 16 * tile_rows<T>(o->fn) / Ns;
  o->xbytes = (L + 3) / 4 * 4 * 16 * o->fn * (int)sizeof(T);
  const int row = trace_ld(o->fn) * (int)sizeof(T);
  // FP32: up to eight waves (256 registers each), FP64: four (512, for twice the accumulators);
  // fewer, and one vector per trace pass, where the LDS is short.  A single wave would leave three
  // of a compute unit's four matrix cores idle: the caller's other path is faster then.
  for (o->waves = sizeof(T) == 4 ? 8 : 4; o->waves >= 2; --o->waves) {
    const int left = LDS_MAX - 16 - o->xbytes;
    o->gc = std::min(o->gb, (left / o->waves / row - 1) / Ns);
    if (left > 0 && o->gc >= 1) {
      o->sbytes = (o->gc * Ns + 1) * row;
      o->lds = o->xbytes + o->waves * o->sbytes + 16;
      return true;
    }
  }
  return false;
}

template <typename T, int FN, bool VEC>
int run(const PhExchangeArgs& a, const Plan& pl, hipStream_t s) {
  constexpr int NT = sizeof(T) == 4 ? 512 : 256;
  KArgs q;
  memset(&q, 0, sizeof(q));
  q.p = a;
  q.gb = pl.gb; q.gc = pl.gc; q.xbytes = pl.xbytes; q.sbytes = pl.sbytes;
  // a workgroup per walker, and enough slices of the vectors for about eight workgroups per compute
  // unit (an even load at any walker count), as long as a wave has two batches
  const int nb = (a.G + pl.gb - 1) / pl.gb;
  const int want = std::max(1, 2048 / a.nw), most = std::max(1, nb / (2 * pl.waves));
  const int slices = std::min(want, most);
  q.slice = (nb + slices - 1) / slices;
  auto kernel = exchange_traces_kernel<T, tile_rows<T>(FN), FN, NT, VEC>;
  HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, LDS_MAX));
  hipLaunchKernelGGL(kernel, dim3(a.nw, (nb + q.slice - 1) / q.slice), dim3(64 * pl.waves), pl.lds, s, q);
  HIP_LAUNCH_CHECK();
  return 0;
}

template <typename T, bool VEC>
int pick(const PhExchangeArgs& a, const Plan& pl, hipStream_t s) {
  switch (pl.fn) {
    case 1: return run<T, 1, VEC>(a, pl, s);
    case 2: return run<T, 2, VEC>(a, pl, s);
    case 3: return run<T, 3, VEC>(a, pl, s);
    case 4: return run<T, 4, VEC>(a, pl, s);
    case 5: return run<T, 5, VEC>(a, pl, s);
    default: return run<T, 6, VEC>(a, pl, s);
  }
}

}  // namespace

template <typename T>
bool ph_exchange_ok(int L, int Ns) {
  Plan pl;
  return plan<T>(L, Ns, &pl);
}

template <typename T>
int launch_ph_exchange(const PhExchangeArgs& a, hipStream_t s) {
  Plan pl;
  if (a.nw <= 0 || a.G <= 0) return 0;
  REQUIRE(plan<T>(a.L, a.Ns, &pl), "exchange traces: %d orbitals with %d electrons not supported", a.L, a.Ns);
  const bool vec = a.L % 4 == 0 && (reinterpret_cast<uintptr_t>(a.A) % (4 * sizeof(T))) == 0;
  return vec ? pick<T, true>(a, pl, s) : pick<T, false>(a, pl, s);
}

template bool ph_exchange_ok<double>(int, int);
template bool ph_exchange_ok<float>(int, int);
template int launch_ph_exchange<double>(const PhExchangeArgs&, hipStream_t);
template int launch_ph_exchange<float>(const PhExchangeArgs&, hipStream_t);
