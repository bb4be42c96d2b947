// Real-A GEMM (see real_gemm.hpp).
//
// A complex B is 2 N real columns, so the product takes two real MFMAs per 16 x 16 x 4 block (one
// when B is real) where the general complex kernel takes three in FP32 and four in FP64.  Four
// waves share a tile of 16 FM rows and 64 FN columns, each wave 16 FM x 16 FN: all waves read the
// same A fragments, so M pads to 16 rows only.  K tiles of 16 are prefetched into registers and
// double-buffered in LDS (one barrier per K tile).  LDS rows have a stride of 17 mod 32 elements:
// both the stores (16 consecutive k per column) and the fragment reads (16 consecutive columns of
// four k) then spread over the banks.
//
// Measured on MI355X (kernel trace, 2048 walkers of 256 x 112 per launch): propagation with the
// fused HS scale 0.352 ms in FP32 and 0.971 ms in FP64 for real walkers, against 0.922 and 2.227 ms
// for the complex kernel; overlap 0.156 and 0.401 against 0.458 and 1.075 ms.  The floor of the
// FP32 propagation is its 0.94 GB of walkers, read and written once: 0.20 ms at the 4.75 TB/s of a
// large copy (0.97 GB by the counters; matrix cores busy 0.54 of the time).  Multiplying the scale and masking at the load instead of at the store cost 0.28 ms
// (every K tile then waited for its loads before its MFMAs).
#include "real_gemm.hpp"

#include "group.hpp"

#include <algorithm>
#include <type_traits>

namespace {

template <typename T, bool OPT, int NC, int FM, int FN, bool SCALE>
struct RgemmK {
  static constexpr int NT = 256, WPE = 1;
  __device__ static void run(const BlockIdx3& bk, const RealGemmArgs& p);
};
template <typename T, bool OPT, int NC, int FM, int FN, bool SCALE>
__device__ __forceinline__ void RgemmK<T, OPT, NC, FM, FN, SCALE>::run(const BlockIdx3& bk, const RealGemmArgs& p) {
  constexpr int BM = 16 * FM, BN = 64 * FN, BK = 16;
  constexpr int LA = BM + (FM % 2 ? 1 : 17), LB = BN + 17;
  constexpr int AE = FM, BE = 4 * FN;  // elements of A and B a thread loads per K tile
  typedef cplx<T> ct;
  typedef typename mfma_traits<T>::acc_t acc_t;
  __shared__ T As[2][BK][LA];
  __shared__ T Bs[2][NC][BK][LB];

  // contiguous tile ranges per XCD, M tiles (or N tiles) fastest, as in the complex kernel
  int bx, by;
  {
    const unsigned gx = (p.M + BM - 1) / BM, gy = (p.N + BN - 1) / BN;
    const unsigned total = gx * gy, L = bk.x, per = total / 8;
    const unsigned lg = (L < per * 8) ? (L % 8) * per + L / 8 : L;
    if (p.n_fastest) { by = lg % gy; bx = lg / gy; }
    else { bx = lg % gx; by = lg / gx; }
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lk = lane >> 4;
  const int m0 = bx * BM, n0 = by * BN;

  // byte offsets of the thread's elements from the tile's K position, fixed over the K loop (the
  // launcher checks that they fit 32 bits); rows and columns past M and N read element 0 of the
  // tile: they feed only results that are not stored
  const char* Ab = reinterpret_cast<const char*>(reinterpret_cast<const T*>(p.A) + (OPT ? (long long)m0 * p.lda : m0));
  const char* Bb = reinterpret_cast<const char*>(reinterpret_cast<const ct*>(p.B) + (long long)n0 * p.ldb);
  const char* Sb = reinterpret_cast<const char*>(p.scale);
  unsigned ao[AE], bo[BE], so[SCALE ? BE : 1];
  int am[AE], ak[AE];
#pragma unroll
  for (int e = 0; e < AE; ++e) {
    const int idx = tid + 256 * e;
    am[e] = OPT ? idx / BK : idx % BM;
    ak[e] = OPT ? idx % BK : idx / BM;
    const long long o = OPT ? ak[e] + (long long)am[e] * p.lda : am[e] + (long long)ak[e] * p.lda;
    ao[e] = m0 + am[e] < p.M ? (unsigned)(o * sizeof(T)) : 0u;
  }
  const int bk_ = tid % BK, bn = tid / BK;  // element e: column bn + 16 e
#pragma unroll
  for (int e = 0; e < BE; ++e) {
    const int n = n0 + bn + 16 * e;
    const bool in = n < p.N;
    bo[e] = in ? (unsigned)((bk_ + (long long)(bn + 16 * e) * p.ldb) * sizeof(ct)) : 0u;
    if (SCALE) so[e] = in ? (unsigned)(((long long)(n / p.scale_group) * p.scale_strideG + bk_) * sizeof(ct)) : 0u;
  }
  // The loads of a K tile are left alone until they are stored to LDS (the scale and the mask of a
  // partial last K tile are applied there), so nothing waits for them before the MFMAs.
  typedef std::conditional_t<NC == 2, ct, T> bt;  // what is read of a B or scale element
  T ra[AE];
  bt rb[BE], rs[SCALE ? BE : 1];
  auto load = [&](int k0) {
    const char* a = Ab + (OPT ? (long long)k0 : (long long)k0 * p.lda) * (long long)sizeof(T);
    const char* b = Bb + (long long)k0 * (long long)sizeof(ct);
    const char* s = SCALE ? Sb + (long long)k0 * (long long)sizeof(ct) : nullptr;
    if (k0 + BK <= p.K) {
#pragma unroll
      for (int e = 0; e < AE; ++e) ra[e] = *reinterpret_cast<const T*>(a + ao[e]);
#pragma unroll
      for (int e = 0; e < BE; ++e) {
        rb[e] = *reinterpret_cast<const bt*>(b + bo[e]);
        if (SCALE) rs[e] = *reinterpret_cast<const bt*>(s + so[e]);
      }
    } else {  // k past K reads element 0 of the tile
#pragma unroll
      for (int e = 0; e < AE; ++e) ra[e] = *reinterpret_cast<const T*>(a + (k0 + ak[e] < p.K ? ao[e] : 0u));
      const bool in = k0 + bk_ < p.K;
#pragma unroll
      for (int e = 0; e < BE; ++e) {
        rb[e] = *reinterpret_cast<const bt*>(b + (in ? bo[e] : 0u));
        if (SCALE) rs[e] = *reinterpret_cast<const bt*>(s + (in ? so[e] : 0u));
      }
    }
  };
  auto store = [&](int st, int k0) {
    const bool whole = k0 + BK <= p.K, inb = whole || k0 + bk_ < p.K;
#pragma unroll
    for (int e = 0; e < AE; ++e) As[st][ak[e]][am[e]] = (whole || k0 + ak[e] < p.K) ? ra[e] : (T)0;
#pragma unroll
    for (int e = 0; e < BE; ++e) {
      if constexpr (NC == 2) {
        const ct v = SCALE ? cmul(rs[e], rb[e]) : rb[e];
        Bs[st][0][bk_][bn + 16 * e] = inb ? v.re : (T)0;
        Bs[st][NC - 1][bk_][bn + 16 * e] = inb ? v.im : (T)0;
      } else {
        const T v = SCALE ? rs[e] * rb[e] : rb[e];
        Bs[st][0][bk_][bn + 16 * e] = inb ? v : (T)0;
      }
    }
  };

  acc_t acc[NC][FM][FN];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[c][i][j] = acc_t{0, 0, 0, 0};
  const int nk = (p.K + BK - 1) / BK;
  load(0);
  store(0, 0);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int st = kt & 1;
    if (kt + 1 < nk) load((kt + 1) * BK);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      T a[FM], b[NC][FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) a[i] = As[st][kk + lk][16 * i + lr];
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int j = 0; j < FN; ++j) b[c][j] = Bs[st][c][kk + lk][16 * (FN * wave + j) + lr];
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int c = 0; c < NC; ++c) acc[c][i][j] = mfma_traits<T>::mma(a[i], b[c][j], acc[c][i][j]);
    }
    if (kt + 1 < nk) store(st ^ 1, (kt + 1) * BK);
    __syncthreads();
  }

  const T alpha = (T)p.alpha;
  ct* C = reinterpret_cast<ct*>(p.C);
  // FP32: a lane's four rows are contiguous, 32 bytes: two 16-byte stores where they are aligned
  const bool vec = sizeof(T) == 4 && p.ldc % 2 == 0 && (reinterpret_cast<uintptr_t>(p.C) & 15) == 0 && !p.beta_one;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int gn = n0 + 16 * (FN * wave + j) + lr;
      if (gn >= p.N) continue;
      if constexpr (sizeof(T) == 4) {
        const int gm = m0 + 16 * i + 4 * lk;
        if (vec && gm + 3 < p.M) {
          float4* o = reinterpret_cast<float4*>(C + gm + (long long)gn * p.ldc);
          float v[8];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            v[2 * r] = alpha * acc[0][i][j][r];
            v[2 * r + 1] = NC == 2 ? alpha * acc[NC - 1][i][j][r] : 0.f;
          }
          o[0] = make_float4(v[0], v[1], v[2], v[3]);
          o[1] = make_float4(v[4], v[5], v[6], v[7]);
          continue;
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gm = m0 + 16 * i + mfma_traits<T>::row(lk, r);
        if (gm >= p.M) continue;
        ct v = cmk<T>(alpha * acc[0][i][j][r], NC == 2 ? alpha * acc[NC - 1][i][j][r] : (T)0);
        ct* o = C + gm + (long long)gn * p.ldc;
        if (p.beta_one) v = cadd(v, *o);
        *o = v;
      }
    }
}

template <typename T, bool OPT, int NC, int FM, bool SCALE>
int run(const RealGemmArgs& a, hipStream_t s) {
  // two column fragments per wave, one where two FP64 planes would take 256 accumulator registers
  constexpr int FN = (sizeof(T) == 8 && NC == 2) ? 1 : 2;
  const long long tiles = (long long)((a.M + 16 * FM - 1) / (16 * FM)) * ((a.N + 64 * FN - 1) / (64 * FN));
  REQUIRE(tiles < (1ll << 31), "real gemm grid too large (%lld tiles)", tiles);
  return glaunch<RgemmK<T, OPT, NC, FM, FN, SCALE>>(a, dim3((unsigned)tiles), dim3(256), 0, s);
}

template <typename T, bool OPT, int NC, bool SCALE>
int pick_rows(const RealGemmArgs& a, hipStream_t s) {
  // The row fragments of a tile: as few padded rows as possible, then as many rows as possible (B
  // is read once per row tile), but small tiles while the launch would leave compute units idle
  // (a grouped call launches the members' tiles together).  Every choice sums in the same order.
  // Weighing padded rows above everything is right only where a tile of several fragments pads nothing.
  // Real walkers, us per launch with 8 / 7 / 4 / 3 / 2 / 1 fragments, the chosen one in brackets:
  //   propagation FP32, 2048 walkers of 100 x 44: 43 / [41] / 46 / 52 / 54 / 79
  //                     1024 of 144 x 64:         67 / 62 / 56 / [47] / 57 / 86
  //                     2048 of 80 x 36:          32 / 30 / 33 / 27 / 29 / [38]
  //                     1024 of 196 x 86:         125 / 114 / 128 / 133 / 153 / [244]
  //   propagation FP64, 1024 of 196 x 86:         345 / 315 / 276 / 280 / 253 / [346]
  //   overlap FP32,     1024 of 256 x 112:        97 / [89] / 88 / 100 / 105 / 143
  // 5, 11 and 13 fragments (65-80, 161-176, 193-208 rows) thus take single fragments where 16 to 22 %
  // of padding in larger tiles would be up to twice as fast.
  constexpr int opts[6] = {8, 7, 4, 3, 2, 1};
  const long long cols = (a.N + 127) / 128;
  int best = 1;
  long long cost = -1;
  for (int f : opts) {
    const long long tiles = (a.M + 16 * f - 1) / (16 * f);
    const long long rows = tiles * f;
    if (f > 1 && !grouping() && tiles * cols < 256) continue;
    const long long c = rows * 16 + tiles;  // padded rows first
    if (cost < 0 || c < cost) { cost = c; best = f; }
  }
  switch (best) {
    case 8: return run<T, OPT, NC, 8, SCALE>(a, s);
    case 7: return run<T, OPT, NC, 7, SCALE>(a, s);
    case 4: return run<T, OPT, NC, 4, SCALE>(a, s);
    case 3: return run<T, OPT, NC, 3, SCALE>(a, s);
    case 2: return run<T, OPT, NC, 2, SCALE>(a, s);
    default: return run<T, OPT, NC, 1, SCALE>(a, s);
  }
}

}  // namespace

template <typename T>
bool real_gemm_ok(const RealGemmArgs& a) {
  if (a.K <= 0 || (a.scale && (a.op_t || a.scale_group <= 0))) return false;
  const long long lim = 0xffffffffll, ce = sizeof(cplx<T>), ae = sizeof(T);
  return (a.op_t ? 128 * a.lda + 16 : 16 * a.lda + 128) * ae < lim && (128 * a.ldb + 16) * ce < lim &&
         (!a.scale || ((long long)(a.N / a.scale_group + 1) * a.scale_strideG + 16) * ce < lim);
}

template <typename T>
int launch_real_gemm(const RealGemmArgs& a, hipStream_t s) {
  if (a.M <= 0 || a.N <= 0) return 0;
  REQUIRE(real_gemm_ok<T>(a), "real gemm: operand not supported (K %d, lda %lld, ldb %lld, N %d)", a.K, a.lda, a.ldb, a.N);
  if (a.op_t) return a.b_real ? pick_rows<T, true, 1, false>(a, s) : pick_rows<T, true, 2, false>(a, s);
  if (a.scale) return a.b_real ? pick_rows<T, false, 1, true>(a, s) : pick_rows<T, false, 2, true>(a, s);
  return a.b_real ? pick_rows<T, false, 1, false>(a, s) : pick_rows<T, false, 2, false>(a, s);
}

template bool real_gemm_ok<double>(const RealGemmArgs&);
template bool real_gemm_ok<float>(const RealGemmArgs&);
template int launch_real_gemm<double>(const RealGemmArgs&, hipStream_t);
template int launch_real_gemm<float>(const RealGemmArgs&, hipStream_t);
