// FFT passes of lengths up to 1024 (all but the few that any_plan refuses): the grids
// whose sizes come out of a box and a resolution (104, 90, 208, 106 = 2 x 53 ...)
// rather than powers of two.
//
// A block takes P pencils.  The first stage reads its butterflies' inputs straight
// from global memory and leaves them in LDS, the last one stores (or accumulates)
// straight to global memory, the stages between work in LDS in place; radices 2 to
// 16 are register butterflies, so that most lengths up to 256 take two stages: one
// LDS round trip.  A prime factor above 13 goes first, as a direct DFT on the sums
// and differences of its mirrored inputs (a quarter of the multiplications).
//
// The LDS-staged pass these lengths took (every stage LDS to LDS, a division per
// element, odd primes as full direct sums with their twiddles from L2) ran the x
// pass of a 208 x 180 x 160 grid in 163 us, y in 62 and z in 36, where their bytes
// take 15, 10 and 10 at the card's copy rate.
#include <algorithm>

#include "fft_core.h"

namespace mdsf {
namespace fft {

namespace {

constexpr int kAnyMax = 1024;       // lengths (their twiddles stay in LDS)
constexpr int kAnyStages = 6;
constexpr int kAnyThreads = kFftThreads;
constexpr size_t kAnyLds = 80 * 1024;   // two blocks per CU

// Radices of the stages in order (a byte each: an array indexed at run time would
// put the kernel argument in scratch), after an optional prime first stage q, and
// the multipliers of the divisions the kernels need (b / d = mulhi(b, m), b d < 2^32).
struct AnyPlan {
  int n, q, nst;
  unsigned long long rads;
  unsigned m_first, m_last, m_q;    // divide by n / first radix, n / last radix, n / q
  int lp;                           // log2 of the pencils per block
  int pitch;
  __host__ __device__ int rad(int i) const { return (int)((rads >> (8 * i)) & 255); }
};

__host__ __device__ inline int any_pos(int i) { return i + (i >> 4); }
__device__ __forceinline__ int fdiv(int b, unsigned m) { return (int)__umulhi((unsigned)b, m); }

// --- DFTs of the other radices ----------------------------------------------------
// odd prime P with c[k] = cos(2 pi k / P), s[k] = sin(2 pi k / P), k < (P + 1) / 2
template <int P>
struct Roots;
template <>
struct Roots<7> {
  static constexpr double c[4] = {1.0, 0.6234898018587335, -0.2225209339563144, -0.9009688679024191};
  static constexpr double s[4] = {0.0, 0.7818314824680298, 0.9749279121818236, 0.4338837391175581};
};
template <>
struct Roots<11> {
  static constexpr double c[6] = {1.0, 0.8412535328311812, 0.41541501300188644, -0.14231483827328514,
                                  -0.6548607339452851, -0.9594929736144974};
  static constexpr double s[6] = {0.0, 0.5406408174555976, 0.9096319953545183, 0.9898214418809327,
                                  0.7557495743542583, 0.28173255684142967};
};
template <>
struct Roots<13> {
  static constexpr double c[7] = {1.0, 0.8854560256532099, 0.5680647467311558, 0.12053668025532305,
                                  -0.3546048870425356, -0.7485107481711011, -0.970941817426052};
  static constexpr double s[7] = {0.0, 0.46472317204376856, 0.8229838658936564, 0.992708874098054,
                                  0.9350162426854148, 0.6631226582407952, 0.23931566428755777};
};

template <int P, bool INV>
__device__ __forceinline__ void dft_prime(Cx* v) {
  constexpr int h = (P - 1) / 2;
  Cx a[h], b[h], x0 = v[0], sum = v[0];
#pragma unroll
  for (int r = 1; r <= h; ++r) {
    a[r - 1] = cadd(v[r], v[P - r]);
    b[r - 1] = csub(v[r], v[P - r]);
    sum = cadd(sum, a[r - 1]);
  }
#pragma unroll
  for (int m = 1; m <= h; ++m) {
    Cx C = x0, S = mk(0, 0);
#pragma unroll
    for (int r = 1; r <= h; ++r) {
      const int k = (r * m) % P, kk = k <= h ? k : P - k;
      const double c = Roots<P>::c[kk], s = k <= h ? Roots<P>::s[kk] : -Roots<P>::s[kk];
      C = mk(fma(c, a[r - 1].x, C.x), fma(c, a[r - 1].y, C.y));
      S = mk(fma(s, b[r - 1].x, S.x), fma(s, b[r - 1].y, S.y));
    }
    const Cx t = mul_mi<INV>(S);   // -i S forward
    v[m] = cadd(C, t);
    v[P - m] = csub(C, t);
  }
  v[0] = sum;
}

// coprime A B: the index maps of the prime-factor algorithm leave no twiddles
template <int A, int B, bool INV>
__device__ __forceinline__ void dft_pfa(Cx* v);

template <bool INV>
__device__ __forceinline__ void dft9(Cx* v) {
  // W_9^1, W_9^2, W_9^4
  const double c1 = 0.766044443118978, s1 = 0.6427876096865394,
               c2 = 0.17364817766693036, s2 = 0.984807753012208,
               c4 = -0.9396926207859084, s4 = 0.3420201433256687;
  const double g = INV ? 1.0 : -1.0;
  Cx t[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    t[i][0] = v[i];
    t[i][1] = v[i + 3];
    t[i][2] = v[i + 6];
    dft3<INV>(t[i]);
  }
  t[1][1] = cmul(t[1][1], mk(c1, g * s1));
  t[1][2] = cmul(t[1][2], mk(c2, g * s2));
  t[2][1] = cmul(t[2][1], mk(c2, g * s2));
  t[2][2] = cmul(t[2][2], mk(c4, g * s4));
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    Cx u[3] = {t[0][k], t[1][k], t[2][k]};
    dft3<INV>(u);
    v[k] = u[0];
    v[k + 3] = u[1];
    v[k + 6] = u[2];
  }
}

template <int RAD, bool INV>
__device__ __forceinline__ void dft_any(Cx* v) {
  if constexpr (RAD == 1) return;
  else if constexpr (RAD == 6) dft_pfa<2, 3, INV>(v);
  else if constexpr (RAD == 7 || RAD == 11 || RAD == 13) dft_prime<RAD, INV>(v);
  else if constexpr (RAD == 9) dft9<INV>(v);
  else if constexpr (RAD == 10) dft_pfa<2, 5, INV>(v);
  else if constexpr (RAD == 12) dft_pfa<4, 3, INV>(v);
  else if constexpr (RAD == 14) dft_pfa<2, 7, INV>(v);
  else if constexpr (RAD == 15) dft_pfa<3, 5, INV>(v);
  else dft<RAD, INV>(v);
}

constexpr int inv_mod(int a, int m) {
  for (int i = 1; i < m; ++i)
    if ((a * i) % m == 1) return i;
  return 1;
}

template <int A, int B, bool INV>
__device__ __forceinline__ void dft_pfa(Cx* v) {
  constexpr int N = A * B;
  Cx t[B][A];
#pragma unroll
  for (int j = 0; j < B; ++j) {
#pragma unroll
    for (int i = 0; i < A; ++i) t[j][i] = v[(B * i + A * j) % N];
    dft_any<A, INV>(t[j]);
  }
  constexpr int ea = B * inv_mod(B % A, A), eb = A * inv_mod(A % B, B);
#pragma unroll
  for (int i = 0; i < A; ++i) {
    Cx u[B];
#pragma unroll
    for (int j = 0; j < B; ++j) u[j] = t[j][i];
    dft_any<B, INV>(u);
#pragma unroll
    for (int j = 0; j < B; ++j) v[(i * ea + j * eb) % N] = u[j];
  }
}

// --- stages ------------------------------------------------------------------------
__device__ __forceinline__ Cx ld_lds(const double2* b, int i) {
  const double2 v = b[i];
  return mk(v.x, v.y);
}
__device__ __forceinline__ void st_lds(double2* b, int i, Cx v) { b[i] = make_double2(v.x, v.y); }

// Calls f(integral constant of the radix).
template <int RAD>
struct Int {
  static constexpr int value = RAD;
};
template <typename F>
__device__ __forceinline__ void by_radix(int rad, F f) {
  switch (rad) {
    case 1: f(Int<1>()); break;
    case 2: f(Int<2>()); break;
    case 3: f(Int<3>()); break;
    case 4: f(Int<4>()); break;
    case 5: f(Int<5>()); break;
    case 6: f(Int<6>()); break;
    case 7: f(Int<7>()); break;
    case 8: f(Int<8>()); break;
    case 9: f(Int<9>()); break;
    case 10: f(Int<10>()); break;
    case 11: f(Int<11>()); break;
    case 12: f(Int<12>()); break;
    case 13: f(Int<13>()); break;
    case 14: f(Int<14>()); break;
    case 15: f(Int<15>()); break;
    default: f(Int<16>()); break;
  }
}

// First stage: load(pencil, element) -> LDS.  elem: lanes along the elements of a
// pencil (else along the pencils).
template <bool INV, typename Load>
__device__ __forceinline__ void any_first(const AnyPlan& pl, double2* buf, bool elem, Load load) {
  const int P = 1 << pl.lp;
  by_radix(pl.rad(0), [&](auto rc) {
    constexpr int RAD = decltype(rc)::value;
    const int nq = pl.n / RAD;
#pragma unroll 1
    for (int i = threadIdx.x; i < P * nq; i += kAnyThreads) {
      const int b = opaque(i);   // (no address per butterfly input kept across iterations)
      int p, j;
      if (elem && nq > 1) {
        p = fdiv(b, pl.m_first);
        j = b - p * nq;
      } else {
        p = b & (P - 1);
        j = b >> pl.lp;
      }
      Cx v[RAD];
#pragma unroll
      for (int r = 0; r < RAD; ++r) v[r] = load(p, j + r * nq);
      dft_any<RAD, INV>(v);
      double2* row = buf + p * pl.pitch;
#pragma unroll
      for (int r = 0; r < RAD; ++r) st_lds(row, any_pos(j * RAD + r), v[r]);
    }
  });
}

// First stage of a prime q: the outputs X_m, X_{q-m} of a column from its sums
// a_r = x_r + x_{q-r} and differences b_r, r <= h = (q - 1) / 2,
//   X = x_0 + sum_r a_r cos(2 pi r m / q) -+ i sum_r b_r sin(2 pi r m / q).
// The sums and differences go to `tmp`; each wave then takes 4 values of m of 64
// columns, whose roots are the same for all its lanes (scalar loads of tw).
template <bool INV, typename Load>
__device__ __forceinline__ void any_first_prime(const AnyPlan& pl, double2* tmp, double2* buf,
                                                bool elem, const double2* __restrict__ tw,
                                                Load load) {
  const int P = 1 << pl.lp, q = pl.q, nq = pl.n / q, h = (q - 1) / 2;
#pragma unroll 1
  for (int r = 0; r <= h; ++r)
    for (int i = threadIdx.x; i < P * nq; i += kAnyThreads) {
      const int b = opaque(i);
      int p, j;
      if (elem && nq > 1) {
        p = fdiv(b, pl.m_q);
        j = b - p * nq;
      } else {
        p = b & (P - 1);
        j = b >> pl.lp;
      }
      double2* row = tmp + p * pl.pitch;
      const Cx x = load(p, j + r * nq);
      if (r == 0) {
        st_lds(row, any_pos(j), x);
      } else {
        const Cx y = load(p, j + (q - r) * nq);
        st_lds(row, any_pos(j + r * nq), cadd(x, y));
        st_lds(row, any_pos(j + (q - r) * nq), csub(x, y));
      }
    }
  __syncthreads();
  const int lane = threadIdx.x & 63, cols = P * nq, chunks = (cols + 63) / 64;
  const int blocks = (h + 4) / 4;   // outputs 0 .. h, four at a time
#pragma unroll 1
  for (int it = threadIdx.x >> 6; it < blocks * chunks; it += kAnyThreads / 64) {
    const int itu = __builtin_amdgcn_readfirstlane(it);
    const int mb = itu % blocks, b = (itu / blocks) * 64 + lane;
    const bool on = b < cols;
    const int bb = on ? b : 0;
    const int j = bb >> pl.lp, p = bb & (P - 1);
    const double2* row = tmp + p * pl.pitch;
    const Cx x0 = ld_lds(row, any_pos(j));
    Cx C[4], S[4];
    int idx[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      C[i] = x0;
      S[i] = mk(0, 0);
      idx[i] = 0;
    }
#pragma unroll 2
    for (int r = 1; r <= h; ++r) {
      const Cx a = ld_lds(row, any_pos(j + r * nq)), d = ld_lds(row, any_pos(j + (q - r) * nq));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        idx[i] += 4 * mb + i;   // r m mod q
        idx[i] = idx[i] >= q ? idx[i] - q : idx[i];
        const double2 w = tw[idx[i] * nq];   // (cos, -sin)
        C[i] = mk(fma(w.x, a.x, C[i].x), fma(w.x, a.y, C[i].y));
        S[i] = mk(fma(-w.y, d.x, S[i].x), fma(-w.y, d.y, S[i].y));
      }
    }
    if (!on) continue;
    double2* out = buf + p * pl.pitch;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = 4 * mb + i;
      if (m > h) break;
      const Cx t = mul_mi<INV>(S[i]);
      st_lds(out, any_pos(j * q + m), cadd(C[i], t));
      if (m > 0) st_lds(out, any_pos(j * q + q - m), csub(C[i], t));
    }
  }
}

// A stage in LDS, in place: every butterfly's inputs are read before any output
// is written (at most NIT butterflies per thread, P n <= 4096).
template <bool INV>
__device__ __forceinline__ void any_middle(const AnyPlan& pl, int st, int ns, double2* buf,
                                           const double2* tw) {
  const int P = 1 << pl.lp;
  __syncthreads();
  by_radix(pl.rad(st), [&](auto rc) {
    constexpr int RAD = decltype(rc)::value;
    constexpr int NIT = RAD >= 9 ? 1 : (RAD == 1 ? 1 : (4096 + 256 * RAD - 1) / (256 * RAD));
    if constexpr (RAD == 1) return;
    const int nq = pl.n / RAD, step = pl.n / (ns * RAD);
    const float rns = 1.f / (float)ns;
    Cx v[NIT][RAD];
    int dst[NIT];
#pragma unroll
    for (int t = 0; t < NIT; ++t) {
      const int b = opaque((int)threadIdx.x) + t * kAnyThreads;
      dst[t] = -1;
      if (b < P * nq) {
        const int p = b & (P - 1), j = b >> pl.lp;
        const int jd = (int)(((float)j + 0.5f) * rns), k = j - jd * ns;   // exact: j < 2^10
        const double2* row = buf + p * pl.pitch;
#pragma unroll
        for (int r = 0; r < RAD; ++r) v[t][r] = ld_lds(row, any_pos(j + r * nq));
        twiddle_in<RAD, INV>(v[t], k, step, tw);
        dft_any<RAD, INV>(v[t]);
        dst[t] = (p << 20) | (jd * ns * RAD + k);
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NIT; ++t) {
      if (dst[t] < 0) continue;
      double2* row = buf + (dst[t] >> 20) * pl.pitch;
      const int d0 = dst[t] & 0xfffff;
#pragma unroll
      for (int r = 0; r < RAD; ++r) st_lds(row, any_pos(d0 + r * ns), v[t][r]);
    }
  });
}

// Last stage: LDS -> store(pencil, element, value, ...).  elem as above.
template <bool INV, typename Store>
__device__ __forceinline__ void any_last(const AnyPlan& pl, const double2* buf, bool elem,
                                         const double2* tw, Store store) {
  const int P = 1 << pl.lp;
  __syncthreads();
  by_radix(pl.rad(pl.nst - 1), [&](auto rc) {
    constexpr int RAD = decltype(rc)::value;
    const int ns = pl.n / RAD;
#pragma unroll 1
    for (int i = threadIdx.x; i < P * ns; i += kAnyThreads) {
      const int b = opaque(i);
      int p, k;
      if (elem && ns > 1) {
        p = fdiv(b, pl.m_last);
        k = b - p * ns;
      } else {
        p = b & (P - 1);
        k = b >> pl.lp;
      }
      const double2* row = buf + p * pl.pitch;
      Cx v[RAD];
#pragma unroll
      for (int r = 0; r < RAD; ++r) v[r] = ld_lds(row, any_pos(k + r * ns));
      twiddle_in<RAD, INV>(v, k, 1, tw);
      dft_any<RAD, INV>(v);
#pragma unroll
      for (int r = 0; r < RAD; ++r) store(p, k + r * ns, v[r]);
    }
  });
}

// The stages up to (not including) the last `tail` ones, from load() into LDS;
// returns the buffer that holds the result.  buf2 is used with a prime first stage.
template <bool INV, typename Load>
__device__ __forceinline__ double2* any_head(const AnyPlan& pl, double2* buf, double2* buf2,
                                             const double2* twg, double2* twl, bool elem, int tail,
                                             Load load) {
  double2* cur = buf;
  int st, ns;
  if (pl.q) {
    any_first_prime<INV>(pl, buf, buf2, elem, twg, load);
    cur = buf2;
    st = 0;
    ns = pl.q;
  } else {
    any_first<INV>(pl, buf, elem, load);
    st = 1;
    ns = pl.rad(0);
  }
#pragma unroll 1
  for (; st < pl.nst - tail; ++st) {
    any_middle<INV>(pl, st, ns, cur, twl);
    ns *= pl.rad(st);
  }
  return cur;
}

// LDS of a block: the P pencils (twice with a prime first stage), the twiddles.
__host__ __device__ inline size_t any_buf(const AnyPlan& pl) {
  return (size_t)(1 << pl.lp) * pl.pitch;
}
inline size_t any_lds(const AnyPlan& pl) {
  return (any_buf(pl) * (pl.q ? 2 : 1) + pl.n) * sizeof(double2);
}

// --- kernels -----------------------------------------------------------------------
// (3 waves per SIMD: 168 VGPRs, up to 10 of them spilled)
template <typename R, bool INV, int EPI, int RES>
__global__ __launch_bounds__(kAnyThreads) __attribute__((amdgpu_waves_per_eu(3)))
void k_pass_any(PassArgs<R> a, AnyPlan pl) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  double2* buf = reinterpret_cast<double2*>(lds_raw);
  double2* buf2 = buf + any_buf(pl);
  double2* twl = buf + any_buf(pl) * (pl.q ? 2 : 1);
  const Geom& g = a.g;
  const int n = pl.n, P = 1 << pl.lp;
  for (int i = threadIdx.x; i < n; i += kAnyThreads) twl[i] = a.ax.tw64[i];
  const int h0 = EPI == EPI_ACC ? 0 : blockIdx.y, h1 = EPI == EPI_ACC ? a.nfr : h0 + 1;
  const long long blk = blockIdx.x;
  if (blk >= g.blocks) {
    // P pencils of the Nyquist plane (FP64, in place or into its sums)
    const int p0 = (int)(blk - g.blocks) * P, pc = min(P, a.nq_pencils - p0);
    const bool elem = a.nq_e == 1;
    for (int h = h0; h < h1; ++h) {
      double2* nyq = a.nyq + h * a.nq_F;
      if (h > h0) __syncthreads();
      double2* res = any_head<INV>(pl, buf, buf2, a.ax.tw64, twl, elem, 1, [&](int p, int e) {
        p = p < pc ? p : pc - 1;
        const long long i = (long long)(p0 + p) * a.nq_p + (long long)e * a.nq_e;
        const double2 v = nyq[i];
        const double w = a.nyq_w ? a.nyq_w[i] : 1.0;
        return mk(v.x * w, v.y * w);
      });
      any_last<INV>(pl, res, elem, twl, [&](int p, int e, Cx v) {
        if (p >= pc) return;
        const long long i = (long long)(p0 + p) * a.nq_p + (long long)e * a.nq_e;
        if constexpr (EPI == EPI_ACC) a.nyq_acc[i] += v.x * v.x + v.y * v.y;
        else nyq[i] = make_double2(v.x, v.y);
      });
    }
    return;
  }
  const int s = (int)(blk / g.tiles_f);
  const int f0 = (int)(blk - (long long)s * g.tiles_f) * P;
  const int pc = min(P, g.nf - f0);
  const long long ib = (long long)s * g.in_s + (long long)f0 * g.in_f;
  const long long ob = (long long)s * g.out_s + (long long)f0 * g.out_f;
  for (int h = h0; h < h1; ++h) {
    if (h > h0) __syncthreads();   // the previous frame's pencils are read
    const auto* in = a.in + h * g.in_F + ib;
    const unsigned char* rin = (RES & RES_IN) ? a.res_in + h * a.res_F + ib : nullptr;
    double2* res = any_head<INV>(pl, buf, buf2, a.ax.tw64, twl, g.in_e == 1, 1, [&](int p, int e) {
      p = p < pc ? p : pc - 1;   // pencils past a partial tile read the last one
      const unsigned i = (unsigned)p * (unsigned)g.in_f + (unsigned)e * (unsigned)g.in_e;
      const auto v = in[i];
      Cx x = mk((double)v.x, (double)v.y);
      if constexpr ((RES & RES_IN) != 0) {
        const unsigned b = rin[i];
        x.x += res_value(b & 15u, (float)v.x);
        x.y += res_value(b >> 4, (float)v.y);
      }
      if (INV && a.w) x = cscale(a.w[ib + i], x);
      return x;
    });
    auto* out = a.out + h * g.out_F + ob;
    unsigned char* rout = (RES & RES_OUT) ? a.res_out + h * a.res_F + ob : nullptr;
    any_last<INV>(pl, res, g.out_e == 1, twl, [&](int p, int e, Cx v) {
      if (p >= pc) return;
      const unsigned i = (unsigned)p * (unsigned)g.out_f + (unsigned)e * (unsigned)g.out_e;
      if constexpr (EPI == EPI_ACC) {
        a.acc[ob + i] += v.x * v.x + v.y * v.y;
      } else {
        typename V2<R>::T o;
        o.x = (R)v.x;
        o.y = (R)v.y;
        out[i] = o;
        if constexpr ((RES & RES_OUT) != 0)
          rout[i] = (unsigned char)(res_nibble(v.x, (float)o.x) | (res_nibble(v.y, (float)o.y) << 4));
      }
    });
  }
}

// z pass: rows of 2 m reals as m complex values, all stages into LDS, then the
// real-pair split.
template <typename R>
__global__ __launch_bounds__(kAnyThreads) void k_r2c_z_any(ZArgs<R> a, AnyPlan pl) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  double2* buf = reinterpret_cast<double2*>(lds_raw);
  double2* buf2 = buf + any_buf(pl);
  double2* twl = buf + any_buf(pl) * (pl.q ? 2 : 1);
  const int m = pl.n, P = 1 << pl.lp;
  for (int i = threadIdx.x; i < m; i += kAnyThreads) twl[i] = a.ax.tw64[i];
  const int x = (int)(blockIdx.x / (unsigned)a.tiles_y);
  const int y0 = (int)(blockIdx.x - (unsigned)x * (unsigned)a.tiles_y) * P;
  const int pc = min(P, a.ny - y0);
  const auto* src = reinterpret_cast<const typename V2<R>::T*>(a.in) + ((long long)x * a.ny + y0) * m;
  const double2* Z = any_head<false>(pl, buf, buf2, a.ax.tw64, twl, true, 0, [&](int p, int e) {
    p = p < pc ? p : pc - 1;
    const auto v = src[p * m + e];
    return mk((double)v.x, (double)v.y);
  });
  __syncthreads();
  auto* dst = a.out + (long long)x * m * a.ny + y0;
  // bins k and m - k from the same two values (k = 0 with the Nyquist bin)
  const int half = m / 2 + 1;
  for (int b = threadIdx.x; b < (half << pl.lp); b += kAnyThreads) {
    const int p = b & (P - 1), k = b >> pl.lp;
    if (p >= pc) continue;
    const double2* row = Z + p * pl.pitch;
    const int kk = k == 0 ? 0 : m - k;
    const Cx z = ld_lds(row, any_pos(k)), zm = ld_lds(row, any_pos(kk));
    const Cx u = split_bin(z, zm, a.tw2, k);
    typename V2<R>::T o;
    o.x = (R)u.x;
    o.y = (R)u.y;
    dst[(unsigned)(k * a.ny + p)] = o;
    if (k == 0) {
      a.nyq[(long long)x * a.ny + y0 + p] = make_double2(z.x - z.y, 0.0);
    } else if (kk != k) {
      const Cx w = split_bin(zm, z, a.tw2, kk);
      o.x = (R)w.x;
      o.y = (R)w.y;
      dst[(unsigned)(kk * a.ny + p)] = o;
    }
  }
}

// inverse z pass: half spectrum -> rows of 2 m reals
template <typename R>
__global__ __launch_bounds__(kAnyThreads) void k_c2r_z_any(CArgs<R> a, AnyPlan pl) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  double2* buf = reinterpret_cast<double2*>(lds_raw);
  double2* buf2 = buf + any_buf(pl);
  double2* twl = buf + any_buf(pl) * (pl.q ? 2 : 1);
  const int m = pl.n, P = 1 << pl.lp;
  for (int i = threadIdx.x; i < m; i += kAnyThreads) twl[i] = a.ax.tw64[i];
  const int x = (int)(blockIdx.x / (unsigned)a.tiles_y);
  const int y0 = (int)(blockIdx.x - (unsigned)x * (unsigned)a.tiles_y) * P;
  const int pc = min(P, a.ny - y0);
  const double2* Z = any_head<true>(pl, buf, buf2, a.ax.tw64, twl, false, 1, [&](int p, int e) {
    p = p < pc ? p : pc - 1;
    return c2r_input<R>(a, x, y0 + p, e);
  });
  auto* dst = reinterpret_cast<typename V2<R>::T*>(a.out) + ((long long)x * a.ny + y0) * m;
  any_last<true>(pl, Z, true, twl, [&](int p, int e, Cx v) {
    if (p >= pc) return;
    typename V2<R>::T o;
    o.x = (R)v.x;
    o.y = (R)v.y;
    dst[p * m + e] = o;
  });
}

// --- plans (host) --------------------------------------------------------------------
unsigned magic(int d) { return (unsigned)(((1ULL << 32) + d - 1) / d); }   // d > 1

// Fewest stages of radices 2 to 16 with product s, the largest radix as small as can
// be.  Radices in ascending order in `best`.
void search(int s, int lo, int* cur, int depth, int* best, int* nbest) {
  if (s == 1) {
    if (depth < *nbest || (depth == *nbest && cur[depth - 1] < best[depth - 1])) {
      *nbest = depth;
      for (int i = 0; i < depth; ++i) best[i] = cur[i];
    }
    return;
  }
  if (depth >= kAnyStages || depth >= *nbest) return;
  for (int r = lo; r <= 16; ++r)
    if (s % r == 0) {
      cur[depth] = r;
      search(s / r, r, cur, depth + 1, best, nbest);
    }
}

// Stages of length n: false if n has two prime factors above 13, or if the radices
// found put one above 8 in a middle stage, where a thread holds its butterflies across
// the in-place exchange (of the even lengths 810, 900, 972, 990 and 1000; splits with
// more stages or a larger last radix are not looked for).
bool any_plan(int n, AnyPlan* pl) {
  if (n < 2 || n > kAnyMax) return false;
  pl->n = n;
  int s = n, q = 0;
  for (int p = 2; p <= 13; ++p)
    while (s % p == 0) s /= p;
  if (s > 1) {
    for (int d = 17; d * d <= s; d += 2)
      if (s % d == 0) return false;
    q = s;
    s = n / q;
  } else {
    s = n;
  }
  pl->q = q;
  int cur[kAnyStages], best[kAnyStages], nb = kAnyStages + 1;
  if (s > 1) search(s, 2, cur, 0, best, &nb);
  else nb = 0;
  if (nb > kAnyStages) return false;
  // ascending order in best: the two largest take the ends, the rest the middle
  int k = 0;
  pl->rads = 0;
  auto put = [&](int r) { pl->rads |= (unsigned long long)r << (8 * k++); };
  if (nb == 0) {
    put(1);   // the prime alone: the last stage copies
  } else if (q) {
    if (nb >= 2 && best[nb - 2] > 8) return false;
    for (int i = 0; i < nb; ++i) put(best[i]);   // largest last
  } else {
    if (nb >= 3 && best[nb - 3] > 8) return false;
    if (nb >= 2) put(best[nb - 2]);
    for (int i = 0; i + 2 < nb; ++i) put(best[i]);
    put(best[nb - 1]);
    if (nb == 1) put(1);   // one stage: the last one copies
  }
  pl->nst = k;
  auto over = [&](int d) { return d > 1 ? magic(d) : 0; };
  pl->m_first = over(n / pl->rad(0));
  pl->m_last = over(n / pl->rad(k - 1));
  pl->m_q = q ? over(n / q) : 0;
  pl->lp = 0;
  pl->pitch = (any_pos(n - 1) + 1) | 1;
  return true;
}

// Whether P = 2^lp pencils fit LDS and the in-place stages (all_lds: the last
// stage is one of them, as in the z pass).
bool any_fits(AnyPlan pl, int lp, bool all_lds) {
  pl.lp = lp;
  const int P = 1 << lp;
  if (P * pl.n > 4096 || any_lds(pl) > kAnyLds) return false;
  const int end = all_lds ? pl.nst : pl.nst - 1;
  for (int i = pl.q ? 0 : 1; i < end; ++i)
    if (pl.rad(i) >= 9 && P * (pl.n / pl.rad(i)) > kAnyThreads) return false;
  return true;
}

// Pencils per block: `want` (a power of two) or fewer.
bool any_pencils(AnyPlan* pl, int want, bool all_lds) {
  int lp = 0;
  while ((2 << lp) <= want) ++lp;
  while (lp > 0 && !any_fits(*pl, lp, all_lds)) --lp;
  if (!any_fits(*pl, lp, all_lds)) return false;
  pl->lp = lp;
  return true;
}

}  // namespace

bool any_ok(int n) {
  AnyPlan pl;
  return any_plan(n, &pl) && any_pencils(&pl, 1, true);
}

template <typename R>
hipError_t any_pass(PassArgs<R> a, PassKind kind, int choice, hipStream_t s) {
  AnyPlan pl;
  // passes that read or write pencil-fastest: 16 pencils (runs of 128 bytes of
  // FP32); along the rows, about 2048 values a block
  const bool across = a.g.in_e != 1 || a.g.out_e != 1;
  const int want = choice >= 1 && choice <= 16 ? choice : (across ? 16 : std::max(1, 2048 / a.n));
  if (!any_plan(a.n, &pl) || !any_pencils(&pl, want, false)) return hipErrorInvalidValue;
  const int P = 1 << pl.lp;
  a.P = P;
  a.g.tiles_f = (a.g.nf + P - 1) / P;
  a.g.blocks = (long long)a.g.ns * a.g.tiles_f;
  const long long total = a.g.blocks + (a.nyq ? (a.nq_pencils + P - 1) / P : 0);
  if (total == 0) return hipSuccess;
  const dim3 g((unsigned)total, kind == PK_X_ACC ? 1 : a.nfr), t(kAnyThreads);
  const size_t lds = any_lds(pl);
  constexpr int RO = sizeof(R) == 4 ? RES_OUT : RES_NONE, RI = sizeof(R) == 4 ? RES_IN : RES_NONE;
  switch (kind) {
    case PK_Y: hipLaunchKernelGGL((k_pass_any<R, false, EPI_STORE, RO>), g, t, lds, s, a, pl); break;
    case PK_X_ACC: hipLaunchKernelGGL((k_pass_any<R, false, EPI_ACC, RI>), g, t, lds, s, a, pl); break;
    case PK_X_STORE: hipLaunchKernelGGL((k_pass_any<R, false, EPI_STORE, RI>), g, t, lds, s, a, pl); break;
    default: hipLaunchKernelGGL((k_pass_any<R, true, EPI_STORE, RES_NONE>), g, t, lds, s, a, pl); break;
  }
  return hipGetLastError();
}

template <typename R>
hipError_t any_r2c(ZArgs<R> a, int choice, hipStream_t s) {
  AnyPlan pl;
  if (!any_plan(a.m, &pl) || !any_pencils(&pl, choice >= 1 && choice <= 16 ? choice : 16, true))
    return hipErrorInvalidValue;
  a.P = 1 << pl.lp;
  a.tiles_y = (a.ny + a.P - 1) / a.P;
  hipLaunchKernelGGL(k_r2c_z_any<R>, dim3((unsigned)((long long)a.nx * a.tiles_y)),
                     dim3(kAnyThreads), any_lds(pl), s, a, pl);
  return hipGetLastError();
}

template <typename R>
hipError_t any_c2r(CArgs<R> a, hipStream_t s) {
  AnyPlan pl;
  if (!any_plan(a.m, &pl) || !any_pencils(&pl, 16, false)) return hipErrorInvalidValue;
  a.P = 1 << pl.lp;
  a.tiles_y = (a.ny + a.P - 1) / a.P;
  hipLaunchKernelGGL(k_c2r_z_any<R>, dim3((unsigned)((long long)a.nx * a.tiles_y)),
                     dim3(kAnyThreads), any_lds(pl), s, a, pl);
  return hipGetLastError();
}

template hipError_t any_pass<float>(PassArgs<float>, PassKind, int, hipStream_t);
template hipError_t any_pass<double>(PassArgs<double>, PassKind, int, hipStream_t);
template hipError_t any_r2c<float>(ZArgs<float>, int, hipStream_t);
template hipError_t any_r2c<double>(ZArgs<double>, int, hipStream_t);
template hipError_t any_c2r<float>(CArgs<float>, hipStream_t);
template hipError_t any_c2r<double>(CArgs<double>, hipStream_t);

}  // namespace fft
}  // namespace mdsf
