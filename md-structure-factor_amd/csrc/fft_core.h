// What the FFT translation units share: FP64 complex arithmetic, small DFTs,
// storage conversions, the pass arguments and the LDS-staged stages.
#pragma once

#include "mdsf_internal.h"

namespace mdsf {
namespace fft {

constexpr int kFftThreads = 256;
constexpr int kRegElems = 4096;  // values per block of the register-staged passes
constexpr int kZRegElems = 2048; // of the register-staged z pass (room beside the deposition)

template <typename R> struct V2;
template <> struct V2<float> { using T = float2; };
template <> struct V2<double> { using T = double2; };

struct Cx {
  double x, y;
};

__device__ __forceinline__ Cx mk(double a, double b) {
  Cx c;
  c.x = a;
  c.y = b;
  return c;
}
__device__ __forceinline__ Cx cmul(Cx a, Cx b) { return mk(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ __forceinline__ Cx cmulc(Cx a, Cx b) { return mk(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y); }
__device__ __forceinline__ Cx cadd(Cx a, Cx b) { return mk(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ Cx csub(Cx a, Cx b) { return mk(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ Cx cscale(double s, Cx a) { return mk(s * a.x, s * a.y); }
__device__ __forceinline__ Cx csel(bool c, Cx a, Cx b) { return mk(c ? a.x : b.x, c ? a.y : b.y); }
// multiply by -i (forward) or +i (inverse)
template <bool INV>
__device__ __forceinline__ Cx mul_mi(Cx a) {
  return INV ? mk(-a.y, a.x) : mk(a.y, -a.x);
}
__device__ __forceinline__ Cx ld_tw(const double2* tw, int k) {
  const double2 v = tw[k];
  return mk(v.x, v.y);
}

// --- small DFTs in registers -------------------------------------------------
template <bool INV>
__device__ __forceinline__ void dft2(Cx* v) {
  const Cx a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}

template <bool INV>
__device__ __forceinline__ void dft3(Cx* v) {
  const double s = 0.86602540378443864676;  // sin(2 pi / 3)
  const Cx t1 = cadd(v[1], v[2]);
  const Cx t2 = mk(v[0].x - 0.5 * t1.x, v[0].y - 0.5 * t1.y);
  const Cx t3 = mul_mi<INV>(cscale(s, csub(v[1], v[2])));
  v[0] = cadd(v[0], t1);
  v[1] = cadd(t2, t3);
  v[2] = csub(t2, t3);
}

template <bool INV>
__device__ __forceinline__ void dft4(Cx* v) {
  const Cx t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
  const Cx t2 = cadd(v[1], v[3]), t3 = mul_mi<INV>(csub(v[1], v[3]));
  v[0] = cadd(t0, t2);
  v[2] = csub(t0, t2);
  v[1] = cadd(t1, t3);
  v[3] = csub(t1, t3);
}

template <bool INV>
__device__ __forceinline__ void dft5(Cx* v) {
  const double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
  const double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;
  const Cx t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]);
  const Cx t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
  const Cx x0 = v[0];
  const Cx a1 = mk(x0.x + c1 * t1.x + c2 * t2.x, x0.y + c1 * t1.y + c2 * t2.y);
  const Cx a2 = mk(x0.x + c2 * t1.x + c1 * t2.x, x0.y + c2 * t1.y + c1 * t2.y);
  const Cx b1 = mul_mi<INV>(mk(s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y));
  const Cx b2 = mul_mi<INV>(mk(s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y));
  v[0] = mk(x0.x + t1.x + t2.x, x0.y + t1.y + t2.y);
  v[1] = cadd(a1, b1);
  v[4] = csub(a1, b1);
  v[2] = cadd(a2, b2);
  v[3] = csub(a2, b2);
}

template <bool INV>
__device__ __forceinline__ void dft8(Cx* v) {
  const double h = 0.70710678118654752440;
  Cx e[4] = {v[0], v[2], v[4], v[6]};
  Cx o[4] = {v[1], v[3], v[5], v[7]};
  dft4<INV>(e);
  dft4<INV>(o);
  const Cx w1 = mk(h, INV ? h : -h);
  const Cx w3 = mk(-h, INV ? h : -h);
  const Cx o1 = cmul(o[1], w1);
  const Cx o2 = mul_mi<INV>(o[2]);
  const Cx o3 = cmul(o[3], w3);
  v[0] = cadd(e[0], o[0]);
  v[4] = csub(e[0], o[0]);
  v[1] = cadd(e[1], o1);
  v[5] = csub(e[1], o1);
  v[2] = cadd(e[2], o2);
  v[6] = csub(e[2], o2);
  v[3] = cadd(e[3], o3);
  v[7] = csub(e[3], o3);
}

template <bool INV>
__device__ __forceinline__ void dft16(Cx* v) {
  Cx e[8], o[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    e[i] = v[2 * i];
    o[i] = v[2 * i + 1];
  }
  dft8<INV>(e);
  dft8<INV>(o);
  const double c1 = 0.92387953251128675613, s1 = 0.38268343236508977173;
  const double h = 0.70710678118654752440;
  const double sg = INV ? 1.0 : -1.0;
  const Cx w[8] = {mk(1, 0),        mk(c1, sg * s1),  mk(h, sg * h),  mk(s1, sg * c1),
                   mk(0, sg),       mk(-s1, sg * c1), mk(-h, sg * h), mk(-c1, sg * s1)};
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const Cx t = k == 0 ? o[0] : cmul(o[k], w[k]);
    v[k] = cadd(e[k], t);
    v[k + 8] = csub(e[k], t);
  }
}

template <int RAD, bool INV>
__device__ __forceinline__ void dft(Cx* v) {
  if constexpr (RAD == 2) dft2<INV>(v);
  else if constexpr (RAD == 3) dft3<INV>(v);
  else if constexpr (RAD == 4) dft4<INV>(v);
  else if constexpr (RAD == 5) dft5<INV>(v);
  else if constexpr (RAD == 8) dft8<INV>(v);
  else dft16<INV>(v);
}

// inputs r >= 1 of a butterfly at k times W^(k r step)
template <int RAD, bool INV>
__device__ __forceinline__ void twiddle_in(Cx* v, int k, int step, const double2* tw) {
  // k = 0 multiplies by the table's exact 1 (no divergent branch)
#pragma unroll
  for (int r = 1; r < RAD; ++r) {
    const Cx w = ld_tw(tw, k * r * step);
    v[r] = INV ? cmulc(v[r], w) : cmul(v[r], w);
  }
}

// --- storage conversions ---------------------------------------------------------
template <typename R>
__device__ __forceinline__ Cx load_cx(const typename V2<R>::T* p, long long i) {
  const auto v = p[i];
  return mk((double)v.x, (double)v.y);
}
template <typename R>
__device__ __forceinline__ void store_cx(typename V2<R>::T* p, long long i, Cx v) {
  typename V2<R>::T o;
  o.x = (R)v.x;
  o.y = (R)v.y;
  p[i] = o;
}

// 4-bit residual of an FP32 rounding: round((v - (float)v) * 16 / ulp) in
// [-8, 7], ulp = 2^(max(e, 1) - 150) the FP32 spacing at (float)v (biased
// exponent e).  Both scalings are exact powers of two (ldexp), so encoding
// and decoding take a few instructions and no division.
__device__ __forceinline__ int res_exp(float h) {
  const int e = (int)((__float_as_uint(h) >> 23) & 0xffu);
  return e > 1 ? e : 1;
}
__device__ __forceinline__ unsigned res_nibble(double v, float h) {
  const double q = rint(ldexp(v - (double)h, 154 - res_exp(h)));
  const double c = fmin(fmax(q, -8.0), 7.0);
  return (unsigned)(int)c & 15u;
}
__device__ __forceinline__ double res_value(unsigned nib, float h) {
  const int qi = (int)((nib ^ 8u) & 15u) - 8;
  return ldexp((double)qi, res_exp(h) - 154);
}

// --- LDS-staged stages (any radix), pencil-fastest, FP64 planes --------------------
template <int RAD, bool INV>
__device__ void stage_fixed(const double* __restrict__ ire, const double* __restrict__ iim,
                            double* __restrict__ ore, double* __restrict__ oim, int n, int P,
                            int pitch, int ns, const double2* __restrict__ tw) {
  const int nq = n / RAD;
  const int nbf = P * nq;
  const int twstep = n / (ns * RAD);
  for (int b = threadIdx.x; b < nbf; b += kFftThreads) {
    const int p = b % P, j = b / P;
    const int k = j % ns;
    const int row = p * pitch;
    Cx v[RAD];
#pragma unroll
    for (int r = 0; r < RAD; ++r) {
      const int a = row + j + r * nq;
      v[r] = mk(ire[a], iim[a]);
    }
    twiddle_in<RAD, INV>(v, k, twstep, tw);
    dft<RAD, INV>(v);
    const int d0 = row + (j / ns) * ns * RAD + k;
#pragma unroll
    for (int r = 0; r < RAD; ++r) {
      ore[d0 + r * ns] = v[r].x;
      oim[d0 + r * ns] = v[r].y;
    }
  }
  __syncthreads();
}

// Any other radix (odd primes): one output element per thread iteration,
// direct DFT with W_RAD^m = W_n^(m n / RAD) from the twiddle table.
template <bool INV>
__device__ void stage_generic(const double* __restrict__ ire, const double* __restrict__ iim,
                              double* __restrict__ ore, double* __restrict__ oim, int n, int P,
                              int pitch, int ns, int RAD, const double2* __restrict__ tw) {
  const int nq = n / RAD;
  const int twstep = n / (ns * RAD);
  const int step = n / RAD;
  for (int o = threadIdx.x; o < P * n; o += kFftThreads) {
    const int p = o % P, rest = o / P;
    const int j = rest % nq, m = rest / nq;
    const int k = j % ns;
    const int row = p * pitch;
    Cx acc = mk(0, 0);
    int wm = 0;  // (r * m) mod RAD
    for (int r = 0; r < RAD; ++r) {
      const int a = row + j + r * nq;
      Cx x = mk(ire[a], iim[a]);
      if (r > 0 && k > 0) {
        const Cx w = ld_tw(tw, k * r * twstep);
        x = INV ? cmulc(x, w) : cmul(x, w);
      }
      const Cx w = ld_tw(tw, wm * step);
      acc = cadd(acc, INV ? cmulc(x, w) : cmul(x, w));
      wm += m;
      if (wm >= RAD) wm -= RAD;
    }
    const int d = row + (j / ns) * ns * RAD + k + m * ns;
    ore[d] = acc.x;
    oim[d] = acc.y;
  }
  __syncthreads();
}

// Every stage of `ax` on P pencils in LDS, ping-ponging between plane pairs
// 0 and 1 of `lds` ([re0 | im0 | re1 | im1], P * pitch values each).
// Returns the plane pair holding the result.  A radix-16 stage runs as two
// radix-4 stages (the same factorisation of n): a 16-point butterfly held
// with its twiddles would set the register budget of every kernel that
// contains this loop.
template <bool INV>
__device__ int run_stages(double* lds, int n, int P, int pitch, const FftAxis& ax) {
  const int plane = P * pitch;
  int ns = 1, cur = 0;
  for (int s = 0; s < ax.nstages; ++s) {
    const int RAD0 = ax.radix[s];
    const int sub = RAD0 == 16 ? 2 : 1;
    const int RAD = RAD0 == 16 ? 4 : RAD0;
    for (int h = 0; h < sub; ++h) {
      const double* ire = lds + (2 * cur) * plane;
      const double* iim = ire + plane;
      double* ore = lds + (2 * (cur ^ 1)) * plane;
      double* oim = ore + plane;
      switch (RAD) {
        case 2: stage_fixed<2, INV>(ire, iim, ore, oim, n, P, pitch, ns, ax.tw64); break;
        case 3: stage_fixed<3, INV>(ire, iim, ore, oim, n, P, pitch, ns, ax.tw64); break;
        case 4: stage_fixed<4, INV>(ire, iim, ore, oim, n, P, pitch, ns, ax.tw64); break;
        case 5: stage_fixed<5, INV>(ire, iim, ore, oim, n, P, pitch, ns, ax.tw64); break;
        case 8: stage_fixed<8, INV>(ire, iim, ore, oim, n, P, pitch, ns, ax.tw64); break;
        default: stage_generic<INV>(ire, iim, ore, oim, n, P, pitch, ns, RAD, ax.tw64); break;
      }
      ns *= RAD;
      cur ^= 1;
    }
  }
  return cur;
}

__host__ __device__ inline int lds_pitch(int n) { return (n % 2 == 0) ? n + 1 : n; }

// --- pencil passes -----------------------------------------------------------------
// Pencil p of a block at slow index s and first fast index f0 reads its element
// e at in + s*in_s + (f0+p)*in_f + e*in_e and writes its element k to
// out + s*out_s + (f0+p)*out_f + k*out_e.  Blocks run over (s, f-tile), and over
// the frames of the group as blockIdx.y, except in accumulating passes (which
// have one slow index), whose blocks take the frames in turn.  in_F, out_F:
// elements from one frame to the next.
struct Geom {
  int in_s, in_f, in_e, out_s, out_f, out_e;   // at most a plane of 4096^2
  long long in_F, out_F;
  int nf;            // fast indices per slow index
  int ns;            // slow indices
  int tiles_f;       // ceil(nf / P)
  long long blocks;  // ns * tiles_f
};

enum Epilogue { EPI_STORE = 0, EPI_ACC = 1 };
// residual nibbles read with the input (RES_IN) and / or written with the output (RES_OUT)
enum Residual { RES_NONE = 0, RES_OUT = 1, RES_IN = 2 };

template <typename R>
struct PassArgs {
  const typename V2<R>::T* in;
  typename V2<R>::T* out;
  double* acc;                  // EPI_ACC: |X|^2 added at the output index
  const double* w;              // X *= w[input index] before the transform (inverse x pass)
  const unsigned char* res_in;  // RES_IN: residual nibbles at the input index
  unsigned char* res_out;       // RES_OUT: residual nibbles at the output index
  Geom g;
  int P;
  int n;
  FftAxis ax;
  // Nyquist plane (FP64, in place): blocks from g.blocks on take one pencil
  // each: element e of frame h's pencil at nyq + h*nq_F + pencil*nq_p + e*nq_e
  double2* nyq;
  double* nyq_acc;
  const double* nyq_w;
  int nq_p, nq_e;
  long long nq_F;
  int nq_pencils;               // per frame
  int tpb;                      // tiles per block of the register-staged pass
  // frames of the launch.  EPI_ACC: the same blocks transform every frame's
  // spectrum (and residuals, Nyquist plane) in turn and add its |X|^2, so that
  // the FP64 sums are read and written once for all of them; res_F: residual
  // bytes from one frame to the next
  int nfr;
  long long res_F;
  // log2 of the width B of the residuals' x blocks (their layout is
  // [kz][x / B][ky][x % B]: fft.hip, res_block), 0: rows [kz][ky][x]; ny
  int res_lb, res_ny;
};

// One Nyquist-plane pencil per block, every stage in LDS (FP64): of the block's
// frame, or (accumulating passes) of every frame in turn.
template <bool INV, int EPI, typename A>
__device__ void nyq_pencil(const A& a, int pencil, double* lds) {
  const int n = a.n, pitch = lds_pitch(n);
  const int h0 = EPI == EPI_ACC ? 0 : blockIdx.y, h1 = EPI == EPI_ACC ? a.nfr : h0 + 1;
  const long long base = (long long)pencil * a.nq_p;
  for (int h = h0; h < h1; ++h) {
    double2* nyq = a.nyq + h * a.nq_F;
    double* re = lds;
    double* im = lds + pitch;
    __syncthreads();  // the LDS may still be read for the previous pencil or tile
    for (int e = threadIdx.x; e < n; e += kFftThreads) {
      const long long g = base + (long long)e * a.nq_e;
      const double2 v = nyq[g];
      const double sc = a.nyq_w ? a.nyq_w[g] : 1.0;
      re[e] = v.x * sc;
      im[e] = v.y * sc;
    }
    __syncthreads();
    const int cur = run_stages<INV>(lds, n, 1, pitch, a.ax);
    re = lds + 2 * cur * pitch;
    im = re + pitch;
    for (int e = threadIdx.x; e < n; e += kFftThreads) {
      const long long g = base + (long long)e * a.nq_e;
      if (EPI == EPI_STORE) nyq[g] = make_double2(re[e], im[e]);
      else a.nyq_acc[g] += re[e] * re[e] + im[e] * im[e];
    }
  }
}

// Global element access of a pass: load with the optional weight and
// residual, store / accumulate with the optional residual.  in, res_in, out and
// res_out are the frame's (the weights are every frame's).
template <typename R, int RES>
__device__ __forceinline__ Cx pass_load(const PassArgs<R>& a, const typename V2<R>::T* in,
                                        const unsigned char* res_in, long long gi) {
  Cx x = load_cx<R>(in, gi);
  if constexpr ((RES & RES_IN) != 0) {
    const unsigned b = res_in[gi];
    x.x += res_value(b & 15u, (float)x.x);
    x.y += res_value(b >> 4, (float)x.y);
  }
  if (a.w) x = cscale(a.w[gi], x);
  return x;
}
template <typename R, int EPI, int RES>
__device__ __forceinline__ void pass_store(const PassArgs<R>& a, typename V2<R>::T* out,
                                           unsigned char* res_out, long long go, Cx v) {
  if constexpr (EPI == EPI_ACC) {
    a.acc[go] += v.x * v.x + v.y * v.y;
  } else {
    store_cx<R>(out, go, v);
    if constexpr ((RES & RES_OUT) != 0)
      res_out[go] = (unsigned char)(res_nibble(v.x, (float)v.x) | (res_nibble(v.y, (float)v.y) << 4));
  }
}

// Workgroup barrier that orders LDS accesses only: global loads issued
// before it (the next tile's inputs) stay in flight across it.  The empty
// asm statements keep the compiler from moving memory accesses (twiddle
// loads in particular) across it, which would hold them in registers
// through the exchange.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  asm volatile("" ::: "memory");
}

// x, hidden from the optimiser: per-lane LDS positions derived from it are
// recomputed in each tile iteration instead of being hoisted out of the tile
// loop and held in registers for the whole kernel.
__device__ __forceinline__ int opaque(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// --- z pass: real rows -> half spectrum --------------------------------------------
// Rows (x, y) of nz reals are read as m = nz/2 complex values Z and
// transformed; the half spectrum follows from the real-pair split
//   X_k = A_k + W_nz^k B_k,  A = (Z_k + conj Z_{m-k}) / 2,  B = (Z_k - conj Z_{m-k}) / 2i,
//   X_m = Re Z_0 - Im Z_0.
// Block = P rows y0..y0+P-1 of one x; output spec[(x m + k) Ny + y] in runs
// of P, nyq[x Ny + y] (FP64).
template <typename R>
struct ZArgs {
  const R* in;                       // density rows (x, y) of nz reals
  typename V2<R>::T* out;            // spec[x][kz][y]
  double2* nyq;                      // nyq[x][y]
  int nx, ny, m;
  int P, tiles_y;
  FftAxis ax;                        // length m
  const double2* tw2;                // W_nz^k, k < nz
  int tpb;                           // tiles per block of the register-staged pass
};

__device__ __forceinline__ Cx split_bin(Cx z, Cx zc_conj_src, const double2* tw2, int k) {
  // zc_conj_src = Z_{m-k} (Z_0 for k = 0)
  const Cx zc = mk(zc_conj_src.x, -zc_conj_src.y);
  const Cx A = cscale(0.5, cadd(z, zc));
  const Cx d = cscale(0.5, csub(z, zc));
  const Cx B = mk(d.y, -d.x);  // d / i
  return cadd(A, cmul(B, ld_tw(tw2, k)));
}

// --- inverse z pass: half spectrum -> real rows ---------------------------------------
// Real adjoint of the R2C along z: x_n = Re sum_{k=0..m} X_k e^{+2 pi i k n / nz}.
// With X'_0 = Re X_0, X'_m = Re X_m and X'_k = X_k / 2 inside, this is the
// Hermitian inverse of X': Z_k = (X'_k + conj X'_{m-k}) + i W^{-k} (X'_k - conj X'_{m-k})
// and x_{2j} + i x_{2j+1} = sum_k Z_k e^{+2 pi i jk/m}.  Reads spec[x][kz][y]
// in runs of P (pencils y), writes density rows.
template <typename R>
struct CArgs {
  const typename V2<R>::T* spec;  // spec[x][kz][y]
  const double2* nyq;              // nyq[x][y]
  R* out;                          // rows (x, y) of nz reals
  int nx, ny, m;
  int P, tiles_y;
  FftAxis ax;
  const double2* tw2;
};

template <typename R>
__device__ __forceinline__ Cx c2r_input(const CArgs<R>& a, int x, int y, int k) {
  const long long base = (long long)x * a.m * a.ny + y;
  Cx xk, xc;
  if (k == 0) {
    xk = mk(load_cx<R>(a.spec, base).x, 0.0);
    xc = mk(a.nyq[(long long)x * a.ny + y].x, 0.0);
  } else {
    const Cx u = load_cx<R>(a.spec, base + (long long)k * a.ny);
    const Cx w = load_cx<R>(a.spec, base + (long long)(a.m - k) * a.ny);
    xk = cscale(0.5, u);
    xc = mk(0.5 * w.x, -0.5 * w.y);
  }
  const Cx e = cadd(xk, xc);
  const Cx o = cmulc(csub(xk, xc), ld_tw(a.tw2, k));  // (X - conj X') W^{-k}
  return mk(e.x - o.y, e.y + o.x);                    // e + i o
}

// LDS bytes one workgroup may allocate on the current device (queried once per device).
inline size_t max_lds_per_block() {
  static int cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 65536;
  if (cached[dev] == 0) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess ||
        v <= 0)
      v = 65536;
    cached[dev] = v;
  }
  return (size_t)cached[dev];
}

// pencils per block of the LDS-staged passes (4 FP64 planes of P * pitch)
inline int lds_pencils(int n) {
  int P = 2048 / (n > 0 ? n : 1);
  if (P > 16) P = 16;
  if (P < 1) P = 1;
  return P;
}
inline size_t lds_bytes(int n, int P) { return (size_t)P * lds_pitch(n) * 4 * sizeof(double); }

// The pass kinds the transform uses (forward z is separate):
enum PassKind {
  PK_Y = 0,       // forward y: spec[x][kz][:] -> rho[kz][:][x]
  PK_X_ACC,       // forward x, |X|^2 into sf
  PK_X_STORE,     // forward x, X in place
  PK_X_INV,       // inverse x (weights), in place
  PK_Y_INV,       // inverse y: rho[kz][:][x] -> spec[x][kz][:]
};


// --- any length (fft_any.hip) ----------------------------------------------------
// Whether the any-length passes take length n, and the passes (choice: pencils
// per block, 0 for the default).
bool any_ok(int n);
template <typename R>
hipError_t any_pass(PassArgs<R> a, PassKind kind, int choice, hipStream_t s);
template <typename R>
hipError_t any_r2c(ZArgs<R> a, int choice, hipStream_t s);
template <typename R>
hipError_t any_c2r(CArgs<R> a, hipStream_t s);

}  // namespace fft
}  // namespace mdsf
