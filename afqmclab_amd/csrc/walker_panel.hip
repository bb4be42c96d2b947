// Per-walker products of real walkers (see walker_panel.hpp).
//
// walker_green and walker_times: the N x N factor B goes to LDS once per workgroup and is the B
// operand of every wave; a wave takes 16 rows of W at a time against all columns, reading its A
// operand straight from global memory (16 consecutive rows per instruction and k, no sharing
// between waves, so LDS and barriers would add nothing).  The K loop has no barrier, and the row
// dots of a wave need no reduction across waves.  A wave has read all of its rows before it stores
// them, so the product may overwrite W.
//
// walker_gram: one workgroup per walker; K tiles of 16 rows are staged in LDS and serve as both
// operands.  Only the 16 x 16 blocks on or above the diagonal are computed, dealt out to the waves
// in turn (at 112 columns 28 of 49), and written twice.
//
// Measured on MI355X (kernel trace, 2048 walkers of 256 x 112): green 0.19 ms in FP32 and 0.34 ms in
// FP64, against 0.52 and 1.07 ms for the complex kernel's Green epilogue (matrix cores busy 0.43 and 0.50 of the
// time).  32 rows per wave spilled or halved the waves in flight (0.27-0.36 and 0.35-0.48 ms).
#include "walker_panel.hpp"

#include "group.hpp"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int lds_ld(int fn) { return 16 * fn + (fn % 2 ? 1 : 17); }  // row stride, 17 mod 32: see real_gemm.hip

// element at a 32-bit byte offset from a wave-uniform base (one vector register of address; the
// launcher checks that the offsets fit)
template <typename V>
__device__ __forceinline__ V at(const void* base, unsigned byte) {
  return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(base) + byte);
}

// row dots: with the trial, also with its partner rows (bit 0), also with the kinetic partner (bit 1)
enum { PANEL_GREEN = 0, PANEL_HALF = 1, PANEL_KIN = 2, PANEL_TIMES = 4 };

template <typename TS, typename TB, int FN, int WHAT>
struct WalkerPanelK {
  static constexpr int NT = 512, WPE = sizeof(TB) == 4 ? 4 : 2;
  __device__ static void run(const BlockIdx3& bk, const WalkerPanelArgs& p);
};
template <typename TS, typename TB, int FN, int WHAT>
__device__ __forceinline__ void WalkerPanelK<TS, TB, FN, WHAT>::run(const BlockIdx3& bk, const WalkerPanelArgs& p) {
  constexpr int FM = 1, LD = lds_ld(FN), U = 4;  // row fragments, LDS row stride, K steps of four per prefetch
  typedef TB TC;
  typedef typename mfma_traits<TC>::acc_t acc_t;
  const int w = bk.x;
  if ((p.alive && !p.alive[w]) || (p.skip && p.skip[w])) return;
  const int M = p.M, N = p.N;
  const int nt = blockDim.x, tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), nwave = nt >> 6;
  const cplx<TS>* __restrict__ W = reinterpret_cast<const cplx<TS>*>(p.W) + (long long)w * p.strideW;
  const cplx<TB>* __restrict__ B = reinterpret_cast<const cplx<TB>*>(p.B) + (long long)w * p.strideB;

  constexpr int N16 = 16 * FN;
  __shared__ TC Bs[N16 * LD];  // [k][n], zero outside N x N
  constexpr int LU = 8;  // loads in flight per thread
  for (int e0 = tid; e0 < N16 * N16; e0 += LU * nt) {
    TB v[LU];
#pragma unroll
    for (int u = 0; u < LU; ++u) {
      const int e = e0 + u * nt, k = e % N16, n = e / N16;
      v[u] = at<TB>(B, k < N && n < N ? (unsigned)(k + n * N) * (unsigned)sizeof(cplx<TB>) : 0u);
    }
#pragma unroll
    for (int u = 0; u < LU; ++u) {
      const int e = e0 + u * nt, k = e % N16, n = e / N16;
      if (e < N16 * N16) Bs[k * LD + n] = (k < N && n < N) ? (TC)v[u] : (TC)0;
    }
  }
  __syncthreads();

  const int nkb = N16 / (4 * U);  // blocks of U K steps
  for (int m0 = 16 * FM * (wave + nwave * bk.y); m0 < M; m0 += 16 * FM * nwave * bk.gy) {
    acc_t acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
    // rows past M read row M - 1 (their results are not stored), columns past N read column N - 1
    // (their rows of B are zero)
    // (FP64: rows dealt to the fragment so that a lane's four results are consecutive rows, as in FP32)
    const int ra = sizeof(TC) == 8 ? 4 * (lr & 3) + (lr >> 2) : lr;
    unsigned row[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) row[i] = (unsigned)min(m0 + 16 * i + ra, M - 1) * (unsigned)sizeof(cplx<TS>);
    const unsigned colb = (unsigned)M * (unsigned)sizeof(cplx<TS>);
    TS nxt[U][FM];
    auto load = [&](int kb) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = 4 * (U * kb + u) + lk;
#pragma unroll
        for (int i = 0; i < FM; ++i) nxt[u][i] = at<TS>(W, row[i] + (unsigned)min(k, N - 1) * colb);
      }
    };
    load(0);
    for (int kb = 0; kb < nkb; ++kb) {
      TC a[U][FM];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int i = 0; i < FM; ++i) a[u][i] = (TC)nxt[u][i];
      if (kb + 1 < nkb) load(kb + 1);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const TC* b = Bs + (4 * (U * kb + u) + lk) * LD + lr;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          // upper-triangular B: rows 16 kb .. below column block j are zero
          if (WHAT == PANEL_TIMES && p.b_upper && kb > j) continue;
          const TC bj = b[16 * j];
#pragma unroll
          for (int i = 0; i < FM; ++i) acc[i][j] = mfma_traits<TC>::mma(a[u][i], bj, acc[i][j]);
        }
        // one K step's LDS reads at a time: all of them ahead would take the registers of more waves
        asm volatile("" ::: "memory");
      }
    }
    if constexpr (WHAT == PANEL_TIMES) {
      cplx<TS>* out = reinterpret_cast<cplx<TS>*>(p.out) + (long long)w * p.stride_out;
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const int n = 16 * j + lr;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int m = m0 + 16 * i + 4 * lk + r;
            if (m < M && n < N) out[m + (long long)n * M] = cmk<TS>((TS)acc[i][j][r], (TS)0);
          }
        }
    } else {
      // row dots in FP64, summed over the wave's columns and then over the 16 lanes of a row; the
      // whole sum goes to the first 64-column group, zero to the second
      constexpr bool HALF = (WHAT & PANEL_HALF) != 0, KIN = (WHAT & PANEL_KIN) != 0;
      constexpr int NQ = 1 + HALF + KIN;
      const int half = p.partner_half, groups = (N + 63) / 64;
      double d[NQ][FM][4];
#pragma unroll
      for (int q = 0; q < NQ; ++q)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) d[q][i][r] = 0.0;
      typedef TS v4 __attribute__((ext_vector_type(4)));
      // VEC: four rows of a partner as one vector (M and the half a multiple of four: the rows and
      // their partners are aligned, and all inside or all outside M)
      auto dots = [&](auto vecc) {
        constexpr bool VEC = decltype(vecc)::value;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const unsigned c = (unsigned)min(16 * j + lr, N - 1) * (unsigned)M;  // columns past N hold zero (B's are zero)
#pragma unroll
          for (int i = 0; i < FM; ++i) {
            const int m = m0 + 16 * i + 4 * lk;
            v4 q[NQ];
            if constexpr (VEC) {
              const int mc = min(m, M - 4);
              constexpr unsigned es = sizeof(TS);
              q[0] = at<v4>(p.P0, (c + mc) * es);
              if constexpr (HALF) q[1] = at<v4>(p.P0, (c + (mc < half ? mc + half : mc - half)) * es);
              if constexpr (KIN) q[NQ - 1] = at<v4>(p.P2, (c + mc) * es);
            } else {
#pragma unroll
              for (int r = 0; r < 4; ++r) {
                const int k = min(m + r, M - 1);
                constexpr unsigned es = sizeof(TS);
                q[0][r] = at<TS>(p.P0, (c + k) * es);
                if constexpr (HALF) q[1][r] = at<TS>(p.P0, (c + (k < half ? k + half : k - half)) * es);
                if constexpr (KIN) q[NQ - 1][r] = at<TS>(p.P2, (c + k) * es);
              }
            }
#pragma unroll
            for (int t = 0; t < NQ; ++t)
#pragma unroll
              for (int r = 0; r < 4; ++r) d[t][i][r] = fma((double)acc[i][j][r], (double)q[t][r], d[t][i][r]);
          }
          // one column's partner loads at a time: all of them in flight would spill the accumulators
          asm volatile("" ::: "memory");
        }
      };
      if (M % 4 == 0 && half % 4 == 0) dots(std::true_type{});
      else dots(std::false_type{});
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + 16 * i + 4 * lk + r;
#pragma unroll
          for (int t = 0; t < NQ; ++t)
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) d[t][i][r] += __shfl_xor(d[t][i][r], o, 64);
          const double d0 = d[0][i][r], d1 = HALF ? d[NQ > 1 ? 1 : 0][i][r] : 0.0, d2 = KIN ? d[NQ - 1][i][r] : 0.0;
          if (m < M && lr < groups) {
            const long long off = ((long long)w * groups + lr) * M + m;
            p.out0[off] = cmk<double>(lr == 0 ? d0 : 0.0, 0.0);
            if (p.out1) p.out1[off] = cmk<double>(lr == 0 ? d1 : 0.0, 0.0);
            if (p.out2) p.out2[off] = cmk<double>(lr == 0 ? d2 : 0.0, 0.0);
          }
        }
    }
  }
}

template <typename TS, typename TC, int NF>
struct WalkerGramK {
  static constexpr int NT = 256, WPE = 2;
  __device__ static void run(const BlockIdx3& bk, const WalkerPanelArgs& p);
};
template <typename TS, typename TC, int NF>
__device__ __forceinline__ void WalkerGramK<TS, TC, NF>::run(const BlockIdx3& bk, const WalkerPanelArgs& p) {
  constexpr int BK = 16, LD = lds_ld(NF), P = NF * (NF + 1) / 2, Q = (P + 3) / 4;
  typedef typename mfma_traits<TC>::acc_t acc_t;
  const int w = bk.x;
  if ((p.alive && !p.alive[w]) || (p.skip && p.skip[w])) return;
  const int M = p.M, N = p.N;
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const cplx<TS>* __restrict__ W = reinterpret_cast<const cplx<TS>*>(p.W) + (long long)w * p.strideW;
  __shared__ TC Ws[2][BK][LD];
  // the wave's blocks (bi[q], bj[q]), bi <= bj: blocks wave, wave + 4, ... of the upper triangle
  int bi[Q], bj[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    int f = min(wave + 4 * q, P - 1), i = 0;
    while (f >= NF - i) { f -= NF - i; ++i; }
    bi[q] = i;
    bj[q] = i + f;
  }
  const int k_ = tid % BK, n_ = tid / BK;  // element e: column n_ + 16 e
  TS rv[NF];
  auto load = [&](int k0) {  // elements past M or N read element 0 and are zeroed at the store
#pragma unroll
    for (int e = 0; e < NF; ++e) {
      const int k = k0 + k_, n = n_ + 16 * e;
      rv[e] = W[k < M && n < N ? k + n * M : 0].re;
    }
  };
  auto store = [&](int st, int k0) {
#pragma unroll
    for (int e = 0; e < NF; ++e)
      Ws[st][k_][n_ + 16 * e] = (k0 + k_ < M && n_ + 16 * e < N) ? (TC)rv[e] : (TC)0;
  };
  acc_t acc[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) acc[q] = acc_t{0, 0, 0, 0};
  const int nk = (M + BK - 1) / BK;
  load(0);
  store(0, 0);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    if (kt + 1 < nk) load((kt + 1) * BK);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      const TC* v = &Ws[kt & 1][kk + lk][lr];
#pragma unroll
      for (int q = 0; q < Q; ++q) acc[q] = mfma_traits<TC>::mma(v[16 * bi[q]], v[16 * bj[q]], acc[q]);
    }
    if (kt + 1 < nk) store((kt + 1) & 1, (kt + 1) * BK);
    __syncthreads();
  }
  cplx<TC>* S = reinterpret_cast<cplx<TC>*>(p.out) + (long long)w * p.stride_out;
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    if (wave + 4 * q >= P) continue;
    const int n = 16 * bj[q] + lr;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = 16 * bi[q] + mfma_traits<TC>::row(lk, r);
      if (m >= N || n >= N) continue;
      const cplx<TC> v = cmk<TC>(acc[q][r], (TC)0);
      S[n + (long long)m * N] = v;
      if (bi[q] != bj[q]) S[m + (long long)n * N] = v;
    }
  }
}

// f(integral_constant<int, F>) for the fragment count F = ceil(N / 16)
template <typename F>
int for_frags(int N, F&& f) {
  switch ((N + 15) / 16) {
    case 1: return f(std::integral_constant<int, 1>{});
    case 2: return f(std::integral_constant<int, 2>{});
    case 3: return f(std::integral_constant<int, 3>{});
    case 4: return f(std::integral_constant<int, 4>{});
    case 5: return f(std::integral_constant<int, 5>{});
    case 6: return f(std::integral_constant<int, 6>{});
    case 7: return f(std::integral_constant<int, 7>{});
    default: return f(std::integral_constant<int, 8>{});
  }
}

template <typename TS, typename TB, int WHAT>
int panel(const WalkerPanelArgs& a, hipStream_t s) {
  if (a.nw <= 0) return 0;
  REQUIRE(a.N >= 1 && a.N <= WALKER_PANEL_NMAX && a.M >= 1, "walker panel: %d x %d walkers not supported", a.M, a.N);
  REQUIRE((long long)a.M * a.N * (long long)sizeof(cplx<TS>) < (1ll << 32), "walker panel: walkers of %d x %d too large", a.M, a.N);
  // a wave per 16 rows, up to eight; more workgroups per walker only where the walkers alone leave
  // compute units idle (each loads B again)
  const int blocks = (a.M + 15) / 16, waves = std::min(8, blocks);
  const int gy = std::max(1, std::min((blocks + waves - 1) / waves, 512 / std::max(a.nw, 1)));
  return for_frags(a.N, [&](auto f) {
    constexpr int FN = decltype(f)::value;
    return glaunch<WalkerPanelK<TS, TB, FN, WHAT>>(a, dim3(a.nw, gy), dim3(64 * waves), 0, s);
  });
}

}  // namespace

template <typename T> int launch_walker_green(const WalkerPanelArgs& a, hipStream_t s) {
  if (a.partner_half)
    return a.P2 ? panel<T, T, PANEL_HALF | PANEL_KIN>(a, s) : panel<T, T, PANEL_HALF>(a, s);
  return a.P2 ? panel<T, T, PANEL_KIN>(a, s) : panel<T, T, PANEL_GREEN>(a, s);
}
template <typename TS, typename TB> int launch_walker_times(const WalkerPanelArgs& a, hipStream_t s) {
  return panel<TS, TB, PANEL_TIMES>(a, s);
}
template <typename TS, typename TC> int launch_walker_gram(const WalkerPanelArgs& a, hipStream_t s) {
  if (a.nw <= 0) return 0;
  REQUIRE(a.N >= 1 && a.N <= WALKER_PANEL_NMAX && a.M >= 1 && a.M < (1 << 24), "walker gram: %d x %d walkers not supported", a.M, a.N);
  return for_frags(a.N, [&](auto f) {
    return glaunch<WalkerGramK<TS, TC, decltype(f)::value>>(a, dim3(a.nw), dim3(256), 0, s);
  });
}

template int launch_walker_green<double>(const WalkerPanelArgs&, hipStream_t);
template int launch_walker_green<float>(const WalkerPanelArgs&, hipStream_t);
template int launch_walker_times<double, double>(const WalkerPanelArgs&, hipStream_t);
template int launch_walker_times<float, double>(const WalkerPanelArgs&, hipStream_t);
template int launch_walker_gram<double, double>(const WalkerPanelArgs&, hipStream_t);
template int launch_walker_gram<float, double>(const WalkerPanelArgs&, hipStream_t);
template int launch_walker_gram<float, float>(const WalkerPanelArgs&, hipStream_t);
