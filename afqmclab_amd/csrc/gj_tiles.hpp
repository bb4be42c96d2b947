// Gauss-Jordan of real matrices of up to 112 columns on the FP64 matrix cores (included by the real
// small dense translation units after small_dense_kernels.hpp).
//
// The panel scheme of GjBK: the exchange steps of four columns compose to A <- A - M A[P, :] outside the
// panel (P its pivot rows, M = S + I[:, P], S the panel's own columns after its in-place steps); one
// wave factorises panel j+1 while the others apply panel j.  Here update wave v holds columns 16 v ..
// 16 v + 15 as RT accumulator tiles of 16 x 16, and applying a panel is one rank-4 MFMA per tile: the
// multipliers are its A operand (one LDS read per tile instead of four per lane and row), the wave's
// pivot rows its B operand, passed through a 64-element LDS buffer.  A panel's own columns come out of
// the same products: their tiles are preset to -I[:, P] and their part of B to -I.
//
// What bounds it is the pivoting wave's serial chain (search, reciprocal, three eliminations, four times
// a panel: some 9800 cycles at 112 columns with three matrices on a compute unit, against 2350 of
// its matrix cores; which part of the chain takes them was not measured); the tiles take 2 RT registers a lane and little else, so that three matrices
// share a compute unit at 112 columns where the vector form fitted two.
// FP32 storage, against GjBK with real elements: 2048 inversions of 112 columns 341 us, 364; in a group
// of 24 x 256 matrices of mixed sizes those of 65-80 columns 240, 260; 49-64: 281, 353; 33-48: 128,
// 137; 17-32: 103, 109.
#pragma once

template <typename T, int RT, int WPEV>
struct GjTK {
  static constexpr int NT = 64 * (RT + 1), WPE = WPEV, WPE_MAX = WPEV;
  __device__ static void run(const BlockIdx3& bk, const SmallDenseArgs& p);
};
template <typename T, int RT, int WPEV>
__device__ __forceinline__ void GjTK<T, RT, WPEV>::run(const BlockIdx3& bk, const SmallDenseArgs& p) {
  constexpr int NB = 4, NRF = RT <= 4 ? 1 : 2, FROWS = 64 * NRF;
  constexpr int ST = FROWS + 16;  // consecutive columns of a panel start half the banks apart
  typedef mfma_traits<double> mt;
  typedef cplx<T> ct;
  const int bidx = bk.x, N = p.N, NP = (N + NB - 1) / NB;
  if (p.alive && !p.alive[bidx / p.alive_div]) return;
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 15, lk = lane >> 4;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const ct* __restrict__ in = reinterpret_cast<const ct*>(p.in) + (long long)bidx * p.stride_in;
  ct* __restrict__ out = reinterpret_cast<ct*>(p.out) + (long long)bidx * p.stride_out;

  __shared__ double pc[2][NB][ST];  // panel columns handed to the pivoting wave
  __shared__ double mm[2][NB][ST];  // -M of a factorised panel
  __shared__ double rb[RT][NB][16]; // each update wave's pivot rows of its own columns
  __shared__ double pivs[16 * RT], rowscale[FROWS];
  __shared__ int pp[2][NB], perm[16 * RT], qinv[FROWS];
  __shared__ int singular, parity;

  auto epilogue = [&]() __attribute__((always_inline)) {
    for (int i = tid; i < N; i += NT) qinv[perm[i]] = i;
    {  // sign of the row permutation: parity of its inversions
      int odd = 0;
      const int di = NT / N, dj = NT - di * N;
      int i = tid / N, j = tid - (tid / N) * N;
      for (int e = tid; e < N * N; e += NT) {
        odd ^= (i < j && perm[i] > perm[j]) ? 1 : 0;
        i += di;
        j += dj;
        if (j >= N) { j -= N; ++i; }
      }
      if (odd) __hip_atomic_fetch_xor(&parity, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
  };

  if (tid == 0) { singular = 0; parity = 0; }
  // The two roles share only the barriers, so that the tiles hold no registers in the pivoting wave.
  if (wv < RT) {
    typename mt::acc_t x[RT];  // x[R][r] = element (16 R + 4 r + lk, 16 wv + lr), the MFMA result layout
    auto hand_over = [&](int b, int buf) __attribute__((always_inline)) {
      if (b / 4 != wv || (lr >> 2) != (b & 3)) return;
      double* o = &pc[buf][lr & 3][0];
#pragma unroll
      for (int R = 0; R < RT; ++R)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[16 * R + 4 * r + lk] = x[R][r];
    };
    {
      // one 32-bit offset per lane and constant ones per row; padding (columns past N, rows past N in
      // the last tile) reads element 0 of the column or matrix, so that all loads are in flight together
      const int j = 16 * wv + lr;
      const char* base = reinterpret_cast<const char*>(in);
      const unsigned col = j < N ? (unsigned)(j * p.ld_in * sizeof(ct)) : 0u;
      const unsigned off = col + (unsigned)(lk * sizeof(ct));
#pragma unroll
      for (int R = 0; R < RT; ++R)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool ok = R < RT - 1 || 16 * R + 4 * r + lk < N;
          const unsigned o = ok ? off + (unsigned)((16 * R + 4 * r) * sizeof(ct)) : col;
          const double v = load_e<double>(*reinterpret_cast<const ct*>(base + o));
          x[R][r] = ok && j < N ? v : 0.0;
        }
    }
    hand_over(0, 0);
    if (NP > 1) hand_over(1, 1);
    lds_barrier();
    lds_barrier();
    for (int j = 0; j < NP; ++j) {
      const int buf = j & 1;
      // the pivot rows of the wave's columns: the tile by a branch on a bit the compiler cannot see
      // through (it would turn a comparison into a read through a run-time pointer)
#pragma unroll
      for (int k = 0; k < NB; ++k) {
        const int P = __builtin_amdgcn_readfirstlane(pp[buf][k]);
        unsigned tile = 1u << (P >> 4);
        asm volatile("" : "+s"(tile));
        const int in_tile = P & 15;
        static_for<RT>([&](auto rc) __attribute__((always_inline)) {
          constexpr int R = decltype(rc)::value;
          if (tile & (1u << R)) {
            const int ri = in_tile >> 2;
            const double lo = ri & 1 ? x[R][1] : x[R][0], hi = ri & 1 ? x[R][3] : x[R][2];
            const double v = ri & 2 ? hi : lo;
            if (lk == (in_tile & 3)) rb[wv][k][lr] = v;
          }
        });
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      double b = rb[wv][lk][lr];
      if (j / 4 == wv && (lr >> 2) == (j & 3)) {  // the panel's own columns become S = M - I[:, P]
        const int q = lr & 3, pq = NB * j + q < N ? pp[buf][q] : -1;
        b = lk == q ? -1.0 : 0.0;
#pragma unroll
        for (int R = 0; R < RT; ++R)
#pragma unroll
          for (int r = 0; r < 4; ++r) x[R][r] = 16 * R + 4 * r + lk == pq ? -1.0 : 0.0;
      }
#pragma unroll
      for (int R = 0; R < RT; ++R) x[R] = mt::mma(mm[buf][lk][16 * R + lr], b, x[R]);
      if (j + 2 < NP) hand_over(j + 2, buf);
      // this phase's reads of the row buffer before the next phase's writes
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      lds_barrier();
    }
    epilogue();
    lds_barrier();
    // inverse: O^{-1}[qinv[i]][perm[j]] = x(i, j) / (-pivot of row i)
    if (p.write_inverse && 16 * wv + lr < N) {
      ct* oc = out + (long long)perm[16 * wv + lr] * p.ld_out;
#pragma unroll
      for (int R = 0; R < RT; ++R)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int i = 16 * R + 4 * r + lk;
          if (R < RT - 1 || i < N) oc[qinv[i]] = store_e<T>(mul_e(x[R][r], rowscale[i]));
        }
    }
  } else {
    __builtin_amdgcn_s_setprio(2);  // the chain's instructions go first on its SIMD
    double fm[NRF][NB];  // the pivoting wave's M of the last panel, its pivot rows, and used rows
    int pk[NB];
    unsigned used = 0u;
    auto factor = [&](int jn, bool pre) __attribute__((always_inline)) {
      const int buf = jn & 1;
      double y[NRF][NB];
#pragma unroll
      for (int r = 0; r < NRF; ++r)
#pragma unroll
        for (int q = 0; q < NB; ++q) y[r][q] = pc[buf][q][lane + 64 * r];
      if (pre) {  // y -= M_{jn-1} y[P_{jn-1}, :]; the pivot rows come from the unmodified copy in LDS
#pragma unroll
        for (int k = 0; k < NB; ++k) {
          double rv[NB];
#pragma unroll
          for (int q = 0; q < NB; ++q) rv[q] = pc[buf][q][pk[k]];
#pragma unroll
          for (int r = 0; r < NRF; ++r)
#pragma unroll
            for (int q = 0; q < NB; ++q) y[r][q] = cfms(y[r][q], fm[r][k], rv[q]);
        }
      }
      int pkn[NB];
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        const int col = NB * jn + q;
        pkn[q] = 0;
        if (col >= N) continue;
        unsigned key = 0u;
#pragma unroll
        for (int r = 0; r < NRF; ++r) {
          const int i = lane + 64 * r;
          const unsigned kk = (i < N && !((used >> r) & 1u)) ? pivot_key32(y[r][q], i) : 0u;
          key = kk > key ? kk : key;
        }
        const int bi = 255 - (int)(wave_max_u32(key) & 0xFFu);
        const int pr = (bi >= 0 && bi < N) ? bi : 0, rr = pr >> 6, pl = pr & 63;
        double prv[NB];
#pragma unroll
        for (int q2 = 0; q2 < NB; ++q2) {
          prv[q2] = readlane_e(y[0][q2], pl);
          if constexpr (NRF > 1) {
            const double v = readlane_e(y[NRF - 1][q2], pl);
            prv[q2] = rr ? v : prv[q2];
          }
        }
        const double piv = prv[q];
        const bool nz = abs1(piv) > 0.0;
        const double inv = nz ? inverse_e(piv) : 0.0;
        double m[NRF];
#pragma unroll
        for (int r = 0; r < NRF; ++r) m[r] = (lane + 64 * r == pr) ? 0.0 : mul_e(y[r][q], inv);
#pragma unroll
        for (int q2 = 0; q2 < NB; ++q2) {
          if (q2 == q) continue;
#pragma unroll
          for (int r = 0; r < NRF; ++r) y[r][q2] = cfms(y[r][q2], m[r], prv[q2]);
        }
#pragma unroll
        for (int r = 0; r < NRF; ++r) y[r][q] = (lane + 64 * r == pr) ? -1.0 : m[r];
        if (lane == pl) used |= 1u << rr;
        if (lane == 0) {
          pivs[col] = piv;
          perm[col] = pr;
          rowscale[pr] = -inv;
          if (!nz) singular = 1;
        }
        pkn[q] = pr;
      }
#pragma unroll
      for (int q = 0; q < NB; ++q) {  // zero columns past N
        const bool live = NB * jn + q < N;
#pragma unroll
        for (int r = 0; r < NRF; ++r) {
          const int i = lane + 64 * r;
          double v = live ? y[r][q] : 0.0;
          if (live && i == pkn[q]) v += 1.0;
          fm[r][q] = v;
          mm[buf][q][i] = -v;
        }
        pk[q] = pkn[q];
        if (lane == 0) pp[buf][q] = pkn[q];
      }
    };
#pragma unroll
    for (int q = 0; q < NB; ++q) pk[q] = 0;
    lds_barrier();
    factor(0, false);
    lds_barrier();
    for (int j = 0; j < NP; ++j) {
      if (j + 1 < NP) factor(j + 1, true);
      lds_barrier();
    }
    __builtin_amdgcn_s_setprio(0);
    epilogue();
    // det = +-(product of the pivots) = z 2^ez, |z| in [1/2, 1)
    double z = 1.0;
    int ez = 0;
      auto times = [&](double v, int ev) __attribute__((always_inline)) {
        int e;
        z = frexp(z * v, &e);
        ez += e + ev;
      };
#pragma unroll
      for (int q = 0; q < NRF; ++q)
        if (lane + 64 * q < N) times(pivs[lane + 64 * q], 0);
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const double zo = __shfl_xor(z, o, 64);
        const int eo = __shfl_xor(ez, o, 64);
        times(zo, eo);
      }
    lds_barrier();
    if (tid == 64 * RT) {
      // the zero of the phase keeps the sign of the complex kernels' -z
      if (parity) z = -z;
      if (p.info) p.info[bidx] = singular;
      p.logdet[bidx] = singular ? cmk<double>(-1e300, 0.0)
                                : cmk<double>(fma((double)ez, M_LN2, log(fabs(z))), atan2(parity ? -0.0 : 0.0, z));
    }
  }
}

template <typename T, int RT, int WPE>
int run_gjt(const SmallDenseArgs& a, hipStream_t s) {
  return glaunch<GjTK<T, RT, WPE>>(a, dim3(a.batch), dim3(64 * (RT + 1)), 0, s);
}
