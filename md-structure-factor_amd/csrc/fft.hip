// 3-D real-to-complex FFT for gfx950: Stockham autosort stages, FP64 arithmetic.
//
// Replaces np.fft.rfftn (dens.py:313) and the |F|^2 frame sum
// (dens.py:315-318): unnormalised forward transform, exponent -2 pi i k n / N.
//
// Precision.  Storage is the plan precision R (float or double); every
// butterfly, twiddle product and the real-to-complex split is evaluated in
// FP64, with FP64 twiddles generated on the device.  An FP32 plan rounds to
// FP32 only where values are stored between passes, and the y pass's output,
// whose rounding error the x pass would spread along whole rows of the
// spectrum (the error that dominates faint bins next to bright ones), keeps a
// 4-bit residual per value: the rounding error in units of 1/16 of the FP32
// ulp, so that the x pass reads it back 16 times more precisely.
//
// Layout.  Three passes, each reading whole contiguous rows and writing P
// pencils side by side (runs of P values):
//   z  rho[x][y][0..Nz) (density, R)  ->  spec[x][kz][y] (kz < Nz/2), nyq[x][y] (kz = Nz/2)
//   y  spec[x][kz][0..Ny)             ->  rho[kz][ky][x] (the density buffer, free by then)
//                                         + res, one byte per value (FP32 plans; res_block)
//   x  rho[kz][ky][0..Nx)             ->  F in place, or |F|^2 added into sf[kz][ky][kx] (FP64)
// The Nyquist plane nyq (FP64 complex) is transformed in FP64 by a few extra
// blocks of the y and x launches (sf_nyq[x][y]).  The inverse passes of the
// adjoint run the same kernels backwards: x in place (weights applied on
// load), y from rho[kz][ky][x] back to spec[x][kz][y], the complex-to-real z
// pass from spec to density rows.
//
// Register-staged passes (n = R1 R2 or R1 R2 R3, n a power of two up to
// 1024): a block holds 4096 values (16 per thread); the first stage reads its
// inputs straight from global memory, each later stage takes its inputs from
// the previous one through LDS (real and imaginary parts in turn, one FP64
// plane), and the last stage stores straight to global memory or folds |X|^2
// into the accumulator.  Other lengths take the any-length passes of
// fft_any.hip, and those that do not fit them (above 1024, two prime factors above
// 13, or a split with a middle radix above 8: any_plan) the LDS-staged pass (every
// stage in LDS, radices 2/3/4/5/8/16 and generic odd primes).
#include <map>
#include <mutex>

#include <hip/hip_ext.h>

#include "fft_core.h"
#include "halfgrid.h"
#include "mdsf_internal.h"

namespace mdsf {

using namespace fft;

namespace {

// --- twiddles: W_n^k = exp(-2 pi i k / n), generated in FP64 ----------------------
__global__ void k_twiddles(float2* __restrict__ tw, double2* __restrict__ tw64, int n) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= n) return;
  double s, c;
  sincospi(-2.0 * (double)k / (double)n, &s, &c);
  if (tw) tw[k] = make_float2((float)c, (float)s);
  tw64[k] = make_double2(c, s);
}

// The register-staged pass for n = R1 R2 R3 (R3 = 1: two stages).  A tile is
// P = 4096 / n pencils; each thread holds 16 values per stage (16 / R
// butterflies of radix R).  IN_E / OUT_E: the input / output elements of a
// pencil are adjacent in memory (lanes element-fastest, and in_e / out_e = 1),
// else the pencils are (lanes pencil-fastest).
template <int n>
constexpr int reg_pencils() { return kRegElems / n; }

template <int n>
__host__ __device__ constexpr int reg_pitch() { return n + n / 16 + 1; }
constexpr int ilog2(int v) { return v < 2 ? 0 : 1 + ilog2(v / 2); }
__device__ __forceinline__ int reg_pos(int i) { return i + (i >> 4); }

// Element `off` (a 32-bit offset) of an array at a wave-uniform base.
template <typename T>
__device__ __forceinline__ const T& at(const T* base, unsigned off) {
  return *reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + off * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ T& at(T* base, unsigned off) {
  return *reinterpret_cast<T*>(reinterpret_cast<char*>(base) + off * (unsigned)sizeof(T));
}

// Moves each thread's values v[i] (slot i at LDS position pos_out(i) of the
// pencil plane, negative: unused) to its next-stage inputs, v[i] read back
// from pos_in(i), real and imaginary parts in turn through one FP64 plane.
// Positions are recomputed per slot rather than kept in registers.
template <int CNT, typename PO, typename PI>
__device__ __forceinline__ void lds_exchange(double* plane, Cx* v, PO pos_out, PI pos_in) {
  lds_barrier();
#pragma unroll
  for (int i = 0; i < CNT; ++i) {
    const int q = pos_out(i);
    if (q >= 0) plane[q] = v[i].x;
  }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < CNT; ++i) {
    const int q = pos_in(i);
    if (q >= 0) v[i].x = plane[q];
  }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < CNT; ++i) {
    const int q = pos_out(i);
    if (q >= 0) plane[q] = v[i].y;
  }
  lds_barrier();
#pragma unroll
  for (int i = 0; i < CNT; ++i) {
    const int q = pos_in(i);
    if (q >= 0) v[i].y = plane[q];
  }
}

// Tiles per block of the register-staged passes: about `rounds` blocks per
// resident slot on the device (blocks resident at once: occupancy of this
// kernel times the CU count, cached per kernel and device), at most 8.  A
// block transforms its tiles in turn and loads the next one's inputs while it
// transforms the current one; the block scheduler still balances the load
// when the pass shares the GPU with the deposition.
inline int stream_tpb(const void* kernel, size_t lds, long long ntiles, int rounds = 2) {
  static std::mutex mu;
  static std::map<std::pair<const void*, int>, long long> cap;
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = 0;
  long long c;
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = cap.find({kernel, dev});
    if (it != cap.end()) {
      c = it->second;
    } else {
      int nb = 0, cus = 0;
      if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, kernel, kFftThreads, lds) != hipSuccess ||
          nb <= 0)
        nb = 1;
      if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
          cus <= 0)
        cus = 1;
      c = (long long)nb * cus;
      cap[{kernel, dev}] = c;
    }
  }
  const long long t = ntiles / (rounds * c);
  return (int)(t < 1 ? 1 : (t > 8 ? 8 : t));
}

template <typename R, int R1, int R2, int R3, bool INV, bool IN_E, bool OUT_E, int EPI, int RES,
          bool WGT>
__global__ __launch_bounds__(kFftThreads) void k_pass_stream(PassArgs<R> a) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  double* plane = reinterpret_cast<double*>(lds_raw);
  constexpr int n = R1 * R2 * R3;
  constexpr int P = reg_pencils<n>();
  constexpr int pitch = reg_pitch<n>();
  constexpr int RL = R3 > 1 ? R3 : R2;  // radix of the last stage
  constexpr int nq1 = n / R1, nsL = n / RL;
  constexpr bool PF = sizeof(R) == 4;   // prefetch (FP32 storage)
  using T2 = typename V2<R>::T;
  const Geom& g = a.g;
  int tid = threadIdx.x;
  const unsigned in_e = IN_E ? 1u : (unsigned)g.in_e, out_e = OUT_E ? 1u : (unsigned)g.out_e;
  const unsigned in_f = (unsigned)g.in_f, out_f = (unsigned)g.out_f;
  // the axis twiddles, copied to LDS after the exchange plane (read after an
  // exchange barrier, at LDS rather than L2 latency), then the tile's 4096
  // residual bytes: they move between global memory and LDS 16 contiguous
  // bytes per lane, and between LDS and the lanes' strided elements a byte
  // at a time
  double2* twl = reinterpret_cast<double2*>(plane + ((P * pitch + 1) & ~1));
  const double2* tw = twl;
  unsigned char* resl = reinterpret_cast<unsigned char*>(twl + n);
  static_assert((RES & RES_IN) == 0 || IN_E, "input residuals: tiles of whole contiguous rows");
  static_assert((RES & RES_OUT) == 0 || !OUT_E, "output residuals: pencil-fastest stores");
  const long long ntiles = g.blocks;
  const unsigned tiles_f = (unsigned)g.tiles_f;
  // stage-1 slot i = t R1 + r: pencil p, element j + r nq1
  auto in_pos = [&](int t, int pc, unsigned* o) __attribute__((always_inline)) {
    const int b = tid + t * kFftThreads;
    int p = IN_E ? b / nq1 : b % P;
    const int j = IN_E ? b % nq1 : b / P;
    p = p < pc ? p : pc - 1;  // pencils past a partial tile read the last one
    *o = (unsigned)p * in_f + (unsigned)j * in_e;
  };
  T2 raw[16];
  uint4 rq;  // RES_IN: bytes 16 tid .. 16 tid + 15 of the tile's residuals (P whole rows)
  // EPI_ACC: each tile is transformed once per frame (sub), into the same
  // accumulator values; else the block's frame
  const int nsub = EPI == EPI_ACC ? a.nfr : 1;
  const T2* in = a.in;
  T2* out = a.out;
  unsigned char* res_out = a.res_out;
  if constexpr (EPI != EPI_ACC) {
    in += blockIdx.y * g.in_F;
    out += blockIdx.y * g.out_F;
    if constexpr ((RES & RES_OUT) != 0) res_out += blockIdx.y * a.res_F;
  }
  auto load = [&](long long tile, int sub) __attribute__((always_inline)) {
    const unsigned s = (unsigned)(tile / tiles_f);
    const int f0 = (int)((unsigned)tile - s * tiles_f) * P;
    const int pc = min(P, g.nf - f0);
    const long long ib = (long long)s * g.in_s + (long long)f0 * g.in_f;
    const T2* src = in + ib;
    if constexpr (EPI == EPI_ACC) src += sub * g.in_F;
#pragma unroll
    for (int t = 0; t < 16 / R1; ++t) {
      unsigned o;
      in_pos(t, pc, &o);
#pragma unroll
      for (int r = 0; r < R1; ++r) raw[t * R1 + r] = at(src, o + (unsigned)(r * nq1) * in_e);
    }
    if constexpr ((RES & RES_IN) != 0) {
      // past a partial tile's rows: the tile's first bytes (never used)
      const unsigned q = 16u * (unsigned)tid < (unsigned)(pc * n) ? (unsigned)tid : 0u;
      const int hr = EPI == EPI_ACC ? sub : (int)blockIdx.y;
      long long rb = ib;
      unsigned ro = q;
      if (a.res_lb) {
        // P rows of one kz: P B bytes of each x block (all powers of two)
        const unsigned ky = (unsigned)f0 & (unsigned)(a.res_ny - 1);
        const unsigned run = (unsigned)(P << a.res_lb) / 16u;
        rb = (long long)(f0 - (int)ky) * n + ((long long)ky << a.res_lb);
        ro = ((unsigned)tid & ~(run - 1u)) * ((unsigned)a.res_ny / P) + ((unsigned)tid & (run - 1u));
      }
      rq = at(reinterpret_cast<const uint4*>(a.res_in + hr * a.res_F + rb), ro);
    }
  };
  const long long nblk = (ntiles + a.tpb - 1) / a.tpb;
  if ((long long)blockIdx.x >= nblk) {
    // the Nyquist-plane pencils: one per block after the tile blocks
    if (a.nyq) nyq_pencil<INV, EPI>(a, (int)((long long)blockIdx.x - nblk), plane);
    return;
  }
  const long long tend = min(ntiles, (long long)(blockIdx.x + 1) * a.tpb);
  long long tile = (long long)blockIdx.x * a.tpb;
  if (PF) load(tile, 0);
  for (int i = threadIdx.x; i < n; i += kFftThreads) twl[i] = a.ax.tw64[i];
  double accv[EPI == EPI_ACC ? 16 : 1];  // this tile's accumulator values (EPI_ACC)
  for (; tile < tend; ++tile) {
    const unsigned s = (unsigned)(tile / tiles_f);
    const int f0 = (int)((unsigned)tile - s * tiles_f) * P;
    const int pc = min(P, g.nf - f0);
    const long long ib = (long long)s * g.in_s + (long long)f0 * g.in_f;
    const long long ob = (long long)s * g.out_s + (long long)f0 * g.out_f;
    // the accumulator values this tile adds to, loaded now so that their
    // latency passes during the transform (pencils past a partial tile read
    // the last one and are not stored), kept in registers through the frames
    if constexpr (EPI == EPI_ACC) {
#pragma unroll
      for (int t = 0; t < 16 / RL; ++t) {
        const int b = tid + t * kFftThreads;
        int p = OUT_E ? b / nsL : b % P;
        const int k = OUT_E ? b % nsL : b / P;
        p = p < pc ? p : pc - 1;
        const unsigned o = (unsigned)p * out_f + (unsigned)k * out_e;
#pragma unroll
        for (int r = 0; r < RL; ++r) accv[t * RL + r] = at(a.acc + ob, o + (unsigned)(r * nsL) * out_e);
      }
    }
    for (int sub = 0; sub < nsub; ++sub) {
      tid = opaque(tid);
      if (!PF) load(tile, sub);
      Cx v[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) v[i] = mk((double)raw[i].x, (double)raw[i].y);
      if constexpr ((RES & RES_IN) != 0) {
        // the previous tile's last reads of resl preceded its exchange barriers
        // x blocks: 16 bytes after each, so that a wave's reads of 64 adjacent
        // elements spread over the banks
        const int lb = a.res_lb, lpt = lb + ilog2(P);
        reinterpret_cast<uint4*>(resl)[lb ? tid + (16 * tid >> lpt) : tid] = rq;
        lds_barrier();
#pragma unroll
        for (int t = 0; t < 16 / R1; ++t) {
          const int b = tid + t * kFftThreads;
          const int p = b / nq1, j = b % nq1;     // row p, element j (in_f = n, in_e = 1)
          // nq1 is a multiple of the block width (res_block)
          const int xb = j >> lb;
          const int q = lb ? (xb << lpt) + 16 * xb + (p << lb) + (j & ((1 << lb) - 1)) : p * n + j;
          const int dq = lb ? (nq1 >> lb << lpt) + 16 * (nq1 >> lb) : nq1;
#pragma unroll
          for (int r = 0; r < R1; ++r) {
            const unsigned rb = resl[q + r * dq];
            const int i = t * R1 + r;
            v[i].x += res_value(rb & 15u, raw[i].x);
            v[i].y += res_value(rb >> 4, raw[i].y);
          }
        }
      }
      if constexpr (WGT) {
#pragma unroll
        for (int t = 0; t < 16 / R1; ++t) {
          unsigned o;
          in_pos(t, pc, &o);
#pragma unroll
          for (int r = 0; r < R1; ++r) v[t * R1 + r] = cscale(at(a.w + ib, o + (unsigned)(r * nq1) * in_e), v[t * R1 + r]);
        }
      }
      if (PF) {
        if (sub + 1 < nsub) load(tile, sub + 1);
        else if (tile + 1 < tend) load(tile + 1, 0);
      }
      // stage 1 (span 1): DFT_R1; output position j R1 + r
#pragma unroll
      for (int t = 0; t < 16 / R1; ++t) dft<R1, INV>(v + t * R1);
      auto out1 = [&](int i) __attribute__((always_inline)) {
        const int b = tid + (i / R1) * kFftThreads, r = i % R1;
        const int p = IN_E ? b / nq1 : b % P, j = IN_E ? b % nq1 : b / P;
        return p * pitch + reg_pos(j * R1 + r);
      };
      // last stage inputs: element k + r nsL of pencil p
      auto inL = [&](int i) __attribute__((always_inline)) {
        const int b = tid + (i / RL) * kFftThreads, r = i % RL;
        const int p = OUT_E ? b / nsL : b % P, k = OUT_E ? b % nsL : b / P;
        return p * pitch + reg_pos(k + r * nsL);
      };
      if constexpr (R3 > 1) {
        // middle stage (span R1, radix R2): LDS -> DFT_R2 -> LDS
        constexpr int nq2 = n / R2, ns2 = R1;
        auto in2 = [&](int i) __attribute__((always_inline)) {
          const int b = tid + (i / R2) * kFftThreads, r = i % R2;
          return (b % P) * pitch + reg_pos(b / P + r * nq2);
        };
        auto out2 = [&](int i) __attribute__((always_inline)) {
          const int b = tid + (i / R2) * kFftThreads, r = i % R2;
          const int j = b / P, k = j % ns2;
          return (b % P) * pitch + reg_pos((j / ns2) * ns2 * R2 + k + r * ns2);
        };
        lds_exchange<16>(plane, v, out1, in2);
#pragma unroll
        for (int t = 0; t < 16 / R2; ++t) {
          const int b = tid + t * kFftThreads;
          twiddle_in<R2, INV>(v + t * R2, (b / P) % ns2, n / (ns2 * R2), tw);
          dft<R2, INV>(v + t * R2);
        }
        lds_exchange<16>(plane, v, out2, inL);
      } else {
        lds_exchange<16>(plane, v, out1, inL);
      }
#pragma unroll
      for (int t = 0; t < 16 / RL; ++t) {
        const int b = tid + t * kFftThreads;
        const int p = OUT_E ? b / nsL : b % P, k = OUT_E ? b % nsL : b / P;
        Cx* x = v + t * RL;
        twiddle_in<RL, INV>(x, k, 1, tw);
        dft<RL, INV>(x);
        if constexpr (EPI == EPI_ACC) {
#pragma unroll
          for (int r = 0; r < RL; ++r)
            accv[t * RL + r] = accv[t * RL + r] + (x[r].x * x[r].x + x[r].y * x[r].y);
        } else if (p < pc) {
          const unsigned o = (unsigned)p * out_f + (unsigned)k * out_e;
#pragma unroll
          for (int r = 0; r < RL; ++r) {
            const unsigned oe = o + (unsigned)(r * nsL) * out_e;
            T2 st;
            st.x = (R)x[r].x;
            st.y = (R)x[r].y;
            at(out + ob, oe) = st;
            if constexpr ((RES & RES_OUT) != 0)  // element k + r nsL of pencil p
              resl[(k + r * nsL) * P + p] =
                  (unsigned char)(res_nibble(x[r].x, st.x) | (res_nibble(x[r].y, st.y) << 4));
          }
        }
      }
    }
    if constexpr (EPI == EPI_ACC) {
#pragma unroll
      for (int t = 0; t < 16 / RL; ++t) {
        const int b = tid + t * kFftThreads;
        const int p = OUT_E ? b / nsL : b % P, k = OUT_E ? b % nsL : b / P;
        if (p < pc) {
          const unsigned o = (unsigned)p * out_f + (unsigned)k * out_e;
#pragma unroll
          for (int r = 0; r < RL; ++r) at(a.acc + ob, o + (unsigned)(r * nsL) * out_e) = accv[t * RL + r];
        }
      }
    }
    if constexpr ((RES & RES_OUT) != 0) {
      // the tile's residuals: n rows (elements) of P bytes (pencils), stored
      // at ob + element out_e + pencil (out_f = 1); the next tile writes resl
      // only after its exchange barriers
      lds_barrier();
      const unsigned q = 16u * (unsigned)tid;
      const int row = (int)(q / P), col = (int)(q % P);
      unsigned char* dst = res_out + ob;
      if (a.res_lb) {
        // x block f0 / P of this kz: its n rows of P bytes lie one after the other
        at(reinterpret_cast<uint4*>(res_out + (long long)s * g.out_s + (long long)f0 * n),
           (unsigned)tid) = *reinterpret_cast<const uint4*>(resl + q);
      } else if (P >= 16 && (out_e & 15u) == 0 && col + 16 <= pc) {
        at(reinterpret_cast<uint4*>(dst + (size_t)row * out_e + col), 0u) =
            *reinterpret_cast<const uint4*>(resl + q);
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int rw = (int)((q + i) / P), cl = (int)((q + i) % P);
          if (cl < pc) dst[(size_t)rw * out_e + cl] = resl[q + i];
        }
      }
    }
  }
}

// The LDS-staged pass (any n): P pencils loaded into LDS, every stage there.
template <typename R, bool INV, int EPI, int RES>
__global__ __launch_bounds__(kFftThreads) void k_pass_lds(PassArgs<R> a) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  double* lds = reinterpret_cast<double*>(lds_raw);
  const long long blk = blockIdx.x;
  if (blk >= a.g.blocks) {
    nyq_pencil<INV, EPI>(a, (int)(blk - a.g.blocks), lds);
    return;
  }
  const Geom& g = a.g;
  const int n = a.n, P = a.P, pitch = lds_pitch(n);
  const long long s = blk / g.tiles_f;
  const int f0 = (int)(blk - s * g.tiles_f) * P;
  const int pc = min(P, g.nf - f0);
  const long long ib = s * g.in_s + (long long)f0 * g.in_f;
  const long long ob = s * g.out_s + (long long)f0 * g.out_f;
  const bool in_e = g.in_e == 1, out_e = g.out_e == 1;
  const int h0 = EPI == EPI_ACC ? 0 : blockIdx.y, h1 = EPI == EPI_ACC ? a.nfr : h0 + 1;
  for (int h = h0; h < h1; ++h) {
    double* re = lds;
    double* im = lds + P * pitch;
    if (h > h0) __syncthreads();   // the previous frame's results are read
    for (int idx = threadIdx.x; idx < pc * n; idx += kFftThreads) {
      const int p = in_e ? idx / n : idx % pc, e = in_e ? idx % n : idx / pc;
      const Cx x = pass_load<R, RES>(a, a.in + h * g.in_F, a.res_in + h * a.res_F,
                                     ib + (long long)p * g.in_f + (long long)e * g.in_e);
      re[p * pitch + e] = x.x;
      im[p * pitch + e] = x.y;
    }
    __syncthreads();
    const int cur = run_stages<INV>(lds, n, P, pitch, a.ax);
    re = lds + 2 * cur * P * pitch;
    im = re + P * pitch;
    for (int idx = threadIdx.x; idx < pc * n; idx += kFftThreads) {
      const int p = out_e ? idx / n : idx % pc, k = out_e ? idx % n : idx / pc;
      pass_store<R, EPI, RES>(a, a.out + h * g.out_F, a.res_out + h * a.res_F,
                              ob + (long long)p * g.out_f + (long long)k * g.out_e,
                              mk(re[p * pitch + k], im[p * pitch + k]));
    }
  }
}

template <typename R>
__device__ __forceinline__ void z_store(const ZArgs<R>& a, int x, int y, int k, Cx v) {
  const long long o = ((long long)x * a.m + k) * a.ny + y;
  store_cx<R>(a.out, o, v);
}

// Register-staged z pass (c2r form below keeps 2048 values per block).
template <int m>
constexpr int zreg_rows() { return kZRegElems / m; }

// Persistent register-staged z pass, m = R1 R2 R3: a tile is P = 4096 / m rows
// y0..y0+P-1 of one x, 16 values per thread and stage.  The last stage pairs
// its butterflies k and ns - k (0 with ns/2) in one thread, which then holds
// Z_k and Z_{m-k} for each of its bins and applies the real-pair split in
// registers.  Block b takes tiles b, b + gridDim.x, ... and loads the next
// tile's rows while it transforms the current one (FP32 storage).
template <typename R, int R1, int R2, int R3>
__global__ __launch_bounds__(kFftThreads) void k_r2c_z_stream(ZArgs<R> a) {
  constexpr int m = R1 * R2 * R3;
  constexpr int P = kRegElems / m;
  constexpr int pitch = reg_pitch<m>();
  constexpr int RL = R3 > 1 ? R3 : R2;
  constexpr int nq1 = m / R1, ns = m / RL, NB = 16 / RL;
  static_assert(NB % 2 == 0, "the last stage pairs butterflies within a thread");
  constexpr bool PF = sizeof(R) == 4;
  using T2 = typename V2<R>::T;
  __shared__ double plane[P * pitch];
  // the axis twiddles W_m^k and the split's W_nz^k (k < m) in LDS, read after
  // an exchange barrier
  __shared__ double2 twl[m], tw2l[m];
  int tid = threadIdx.x;
  const double2* tw = twl;
  const long long ntiles = (long long)a.nx * a.tiles_y;
  T2 raw[16];
  auto load = [&](long long tile) __attribute__((always_inline)) {
    const int x = (int)(tile / a.tiles_y);
    const int y0 = (int)(tile - (long long)x * a.tiles_y) * P;
    const int pc = min(P, a.ny - y0);
    const T2* src = reinterpret_cast<const T2*>(a.in) + ((long long)x * a.ny + y0) * m;
#pragma unroll
    for (int t = 0; t < 16 / R1; ++t) {
      const int b = tid + t * kFftThreads;
      int p = b / nq1;
      const int j = b % nq1;
      p = p < pc ? p : pc - 1;
#pragma unroll
      for (int r = 0; r < R1; ++r) raw[t * R1 + r] = at(src, (unsigned)(p * m + j + r * nq1));
    }
  };
  long long tile = (long long)blockIdx.x * a.tpb;
  const long long tend = min(ntiles, tile + a.tpb);
  if (PF && tile < tend) load(tile);
  for (int i = threadIdx.x; i < m; i += kFftThreads) {
    twl[i] = a.ax.tw64[i];
    tw2l[i] = a.tw2[i];
  }
  for (; tile < tend; ++tile) {
    tid = opaque(tid);
    if (!PF) load(tile);
    const int x = (int)(tile / a.tiles_y);
    const int y0 = (int)(tile - (long long)x * a.tiles_y) * P;
    const int pc = min(P, a.ny - y0);
    Cx v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = mk((double)raw[i].x, (double)raw[i].y);
    if (PF && tile + 1 < tend) load(tile + 1);
    // stage 1: rows along the lanes; output position j R1 + r
#pragma unroll
    for (int t = 0; t < 16 / R1; ++t) dft<R1, false>(v + t * R1);
    auto out1 = [&](int i) __attribute__((always_inline)) {
      const int b = tid + (i / R1) * kFftThreads, r = i % R1;
      return (b / nq1) * pitch + reg_pos((b % nq1) * R1 + r);
    };
    // last stage: slot i = (2u + h) RL + r, pair c = tid + u 256 of row c % P,
    // butterfly kA = c / P (h = 0) or its partner kB (h = 1), bin k + r ns
    auto kpair = [&](int u, int h) __attribute__((always_inline)) {
      const int kp = (tid + u * kFftThreads) / P;
      return h == 0 ? kp : (kp == 0 ? ns / 2 : ns - kp);
    };
    auto inL = [&](int i) __attribute__((always_inline)) {
      const int r = i % RL, h = (i / RL) & 1, u = i / (2 * RL);
      const int p = (tid + u * kFftThreads) % P;
      return p * pitch + reg_pos(kpair(u, h) + r * ns);
    };
    if constexpr (R3 > 1) {
      constexpr int nq2 = m / R2, ns2 = R1;
      auto in2 = [&](int i) __attribute__((always_inline)) {
        const int b = tid + (i / R2) * kFftThreads, r = i % R2;
        return (b % P) * pitch + reg_pos(b / P + r * nq2);
      };
      auto out2 = [&](int i) __attribute__((always_inline)) {
        const int b = tid + (i / R2) * kFftThreads, r = i % R2;
        const int j = b / P, k = j % ns2;
        return (b % P) * pitch + reg_pos((j / ns2) * ns2 * R2 + k + r * ns2);
      };
      lds_exchange<16>(plane, v, out1, in2);
#pragma unroll
      for (int t = 0; t < 16 / R2; ++t) {
        const int b = tid + t * kFftThreads;
        twiddle_in<R2, false>(v + t * R2, (b / P) % ns2, m / (ns2 * R2), tw);
        dft<R2, false>(v + t * R2);
      }
      lds_exchange<16>(plane, v, out2, inL);
    } else {
      lds_exchange<16>(plane, v, out1, inL);
    }
#pragma unroll
    for (int u = 0; u < NB / 2; ++u) {
      const int c = tid + u * kFftThreads;
      const int p = c % P, kA = kpair(u, 0), kB = kpair(u, 1);
      Cx* za = v + (2 * u) * RL;
      Cx* zb = v + (2 * u + 1) * RL;
      twiddle_in<RL, false>(za, kA, 1, tw);
      dft<RL, false>(za);
      twiddle_in<RL, false>(zb, kB, 1, tw);
      dft<RL, false>(zb);
      if (p >= pc) continue;
      T2* dst = a.out + (long long)x * m * a.ny + y0 + p;
      // bin k of this row at dst[k Ny]; Z_{m-k} of bin kA + r ns is za[RL - r]
      // (kA = 0, r > 0), za[0] (kA = r = 0) or zb[RL - 1 - r]; of bin kB + r ns
      // it is zb[RL - 1 - r] (kA = 0) or za[RL - 1 - r]
      const bool self = kA == 0;
#pragma unroll
      for (int r = 0; r < RL; ++r) {
        const int k1 = kA + r * ns, k2 = kB + r * ns;
        const Cx m1 = csel(self, za[r == 0 ? 0 : RL - r], zb[RL - 1 - r]);
        const Cx m2 = csel(self, zb[RL - 1 - r], za[RL - 1 - r]);
        const Cx x1 = split_bin(za[r], m1, tw2l, k1);
        const Cx x2 = split_bin(zb[r], m2, tw2l, k2);
        T2 s1, s2;
        s1.x = (R)x1.x;
        s1.y = (R)x1.y;
        s2.x = (R)x2.x;
        s2.y = (R)x2.y;
        at(dst, (unsigned)(k1 * a.ny)) = s1;
        at(dst, (unsigned)(k2 * a.ny)) = s2;
      }
      if (self) a.nyq[(long long)x * a.ny + y0 + p] = make_double2(za[0].x - za[0].y, 0.0);
    }
  }
}

// LDS-staged z pass (any m): P rows per block, every stage in LDS.
template <typename R>
__global__ __launch_bounds__(kFftThreads) void k_r2c_z(ZArgs<R> a) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  double* lds = reinterpret_cast<double*>(lds_raw);
  const int m = a.m, P = a.P, pitch = lds_pitch(m);
  const int x = blockIdx.x / a.tiles_y;
  const int y0 = (blockIdx.x - x * a.tiles_y) * P;
  const int pc = min(P, a.ny - y0);
  const auto* src = reinterpret_cast<const typename V2<R>::T*>(a.in) + ((long long)x * a.ny + y0) * m;
  double* re = lds;
  double* im = lds + P * pitch;
  for (int idx = threadIdx.x; idx < pc * m; idx += kFftThreads) {
    const int p = idx / m, e = idx - p * m;
    const Cx v = load_cx<R>(src, idx);
    re[p * pitch + e] = v.x;
    im[p * pitch + e] = v.y;
  }
  __syncthreads();
  const int cur = run_stages<false>(lds, m, P, pitch, a.ax);
  re = lds + 2 * cur * P * pitch;
  im = re + P * pitch;
  for (int idx = threadIdx.x; idx < pc * m; idx += kFftThreads) {
    const int p = idx % pc, k = idx / pc;
    const int kk = k == 0 ? 0 : m - k;
    const Cx z = mk(re[p * pitch + k], im[p * pitch + k]);
    const Cx zm = mk(re[p * pitch + kk], im[p * pitch + kk]);
    z_store<R>(a, x, y0 + p, k, split_bin(z, zm, a.tw2, k));
  }
  for (int p = threadIdx.x; p < pc; p += kFftThreads)
    a.nyq[(long long)x * a.ny + y0 + p] = make_double2(re[p * pitch] - im[p * pitch], 0.0);
}

template <typename R, int R1, int R2>
__global__ __launch_bounds__(kFftThreads) void k_c2r_z_reg(CArgs<R> a) {
  constexpr int m = R1 * R2;
  constexpr int P = zreg_rows<m>();
  constexpr int pitch = reg_pitch<m>();
  constexpr int nq1 = m / R1, ns = m / R2;
  constexpr int T1 = (P * nq1 + kFftThreads - 1) / kFftThreads;
  constexpr int T2 = (P * ns + kFftThreads - 1) / kFftThreads;
  constexpr int VPT = T1 * R1 > T2 * R2 ? T1 * R1 : T2 * R2;
  __shared__ double plane[P * pitch];
  const int x = blockIdx.x / a.tiles_y;
  const int y0 = (blockIdx.x - x * a.tiles_y) * P;
  const int pc = min(P, a.ny - y0);
  const double2* tw = a.ax.tw64;
  const int tid = threadIdx.x;
  Cx v[VPT];
  // stage 1: inputs Z_k built from spec runs (pencil-fastest lanes)
  auto out1 = [&](int i) __attribute__((always_inline)) {
    const int b = tid + (i / R1) * kFftThreads, r = i % R1;
    if (i >= T1 * R1 || b >= P * nq1) return -1;
    return (b % P) * pitch + reg_pos((b / P) * R1 + r);
  };
  auto in2 = [&](int i) __attribute__((always_inline)) {
    const int b = tid + (i / R2) * kFftThreads, r = i % R2;
    if (i >= T2 * R2 || b >= P * ns) return -1;
    return (b / ns) * pitch + reg_pos(b % ns + r * ns);
  };
#pragma unroll
  for (int t = 0; t < T1; ++t) {
    const int b = tid + t * kFftThreads;
    if (b >= P * nq1) break;
    const int p = b % P, j = b / P;
    Cx* xv = v + t * R1;
#pragma unroll
    for (int r = 0; r < R1; ++r) xv[r] = p < pc ? c2r_input<R>(a, x, y0 + p, j + r * nq1) : mk(0, 0);
    dft<R1, true>(xv);
  }
  lds_exchange<VPT>(plane, v, out1, in2);
  R* dst = a.out + ((long long)x * a.ny + y0) * (2LL * m);
#pragma unroll
  for (int t = 0; t < T2; ++t) {
    const int b = tid + t * kFftThreads;
    if (b >= P * ns) break;
    const int p = b / ns, k = b % ns;
    Cx* xv = v + t * R2;
    twiddle_in<R2, true>(xv, k, 1, tw);
    dft<R2, true>(xv);
    if (p < pc) {
#pragma unroll
      for (int r = 0; r < R2; ++r) {
        const long long o = 2 * ((long long)p * m + k + r * ns);
        dst[o] = (R)xv[r].x;
        dst[o + 1] = (R)xv[r].y;
      }
    }
  }
}

template <typename R>
__global__ __launch_bounds__(kFftThreads) void k_c2r_z(CArgs<R> a) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  double* lds = reinterpret_cast<double*>(lds_raw);
  const int m = a.m, P = a.P, pitch = lds_pitch(m);
  const int x = blockIdx.x / a.tiles_y;
  const int y0 = (blockIdx.x - x * a.tiles_y) * P;
  const int pc = min(P, a.ny - y0);
  double* re = lds;
  double* im = lds + P * pitch;
  for (int idx = threadIdx.x; idx < pc * m; idx += kFftThreads) {
    const int p = idx % pc, k = idx / pc;
    const Cx z = c2r_input<R>(a, x, y0 + p, k);
    re[p * pitch + k] = z.x;
    im[p * pitch + k] = z.y;
  }
  __syncthreads();
  const int cur = run_stages<true>(lds, m, P, pitch, a.ax);
  re = lds + 2 * cur * P * pitch;
  im = re + P * pitch;
  R* dst = a.out + ((long long)x * a.ny + y0) * (2LL * m);
  for (int idx = threadIdx.x; idx < pc * m; idx += kFftThreads) {
    const int p = idx / m, j = idx - p * m;
    dst[2 * (long long)idx] = (R)re[p * pitch + j];
    dst[2 * (long long)idx + 1] = (R)im[p * pitch + j];
  }
}

// --- launch helpers --------------------------------------------------------------------
// Events the next stream-kernel launch of a pass records with its own
// dispatch (its begin and end: the frame loop's stage timing), or null.
thread_local hipEvent_t t_pass_ev[2] = {nullptr, nullptr};
thread_local bool t_pass_ev_used = false;

template <typename K, typename A>
void pass_launch(K kernel, dim3 grid, size_t lds, hipStream_t s, const A& a) {
  if (t_pass_ev[0]) {
    hipExtLaunchKernelGGL(kernel, grid, dim3(kFftThreads), lds, s, t_pass_ev[0], t_pass_ev[1], 0,
                          a);
    t_pass_ev_used = true;
  } else {
    hipLaunchKernelGGL(kernel, grid, dim3(kFftThreads), lds, s, a);
  }
}

// Radix split of the register-staged passes for n, or 0.
inline int reg_split(int n, int* r1, int* r2, int* r3) {
  switch (n) {
    case 16: *r1 = 4; *r2 = 4; *r3 = 1; return 1;
    case 32: *r1 = 8; *r2 = 4; *r3 = 1; return 1;
    case 64: *r1 = 8; *r2 = 8; *r3 = 1; return 1;
    case 128: *r1 = 16; *r2 = 8; *r3 = 1; return 1;
    case 256: *r1 = 16; *r2 = 16; *r3 = 1; return 1;
    case 512: *r1 = 8; *r2 = 8; *r3 = 8; return 1;
    case 1024: *r1 = 16; *r2 = 8; *r3 = 8; return 1;
    default: return 0;
  }
}

template <typename R, int R1, int R2, int R3, bool INV, bool IN_E, bool OUT_E, int EPI, int RES,
          bool WGT>
void launch_stream(size_t lds, hipStream_t s, PassArgs<R> a) {
  const void* k =
      reinterpret_cast<const void*>(&k_pass_stream<R, R1, R2, R3, INV, IN_E, OUT_E, EPI, RES, WGT>);
  const unsigned ny = EPI == EPI_ACC ? 1 : a.nfr;   // frames as grid y
  a.tpb = stream_tpb(k, lds, a.g.blocks * ny);
  const long long grid = (a.g.blocks + a.tpb - 1) / a.tpb + (a.nyq ? a.nq_pencils : 0);
  if (grid == 0) return;
  pass_launch(k_pass_stream<R, R1, R2, R3, INV, IN_E, OUT_E, EPI, RES, WGT>,
              dim3((unsigned)grid, ny), lds, s, a);
}

template <typename R, bool INV, bool IN_E, bool OUT_E, int EPI, int RES, bool WGT>
void launch_reg_n(int n, size_t lds, hipStream_t s, const PassArgs<R>& a) {
  switch (n) {
    case 16: launch_stream<R, 4, 4, 1, INV, IN_E, OUT_E, EPI, RES, WGT>(lds, s, a); break;
    case 32: launch_stream<R, 8, 4, 1, INV, IN_E, OUT_E, EPI, RES, WGT>(lds, s, a); break;
    case 64: launch_stream<R, 8, 8, 1, INV, IN_E, OUT_E, EPI, RES, WGT>(lds, s, a); break;
    case 128: launch_stream<R, 16, 8, 1, INV, IN_E, OUT_E, EPI, RES, WGT>(lds, s, a); break;
    case 256: launch_stream<R, 16, 16, 1, INV, IN_E, OUT_E, EPI, RES, WGT>(lds, s, a); break;
    case 512: launch_stream<R, 8, 8, 8, INV, IN_E, OUT_E, EPI, RES, WGT>(lds, s, a); break;
    default: launch_stream<R, 16, 8, 8, INV, IN_E, OUT_E, EPI, RES, WGT>(lds, s, a); break;
  }
}

// log2 of the width of the residuals' x blocks, 0 for rows [kz][ky][x].  A register-staged y pass
// stores P = 4096 / ny pencils (x) side by side: in rows its residuals would be runs
// of P bytes, ny of them nx bytes apart (16 bytes each at 256, 8 at 512).  In the
// layout [kz][x / P][ky][x % P] a tile's residuals are one run of 4096 bytes, and the
// x pass, whose tile is 4096 / nx rows, reads runs of P (4096 / nx) bytes.  Needs both
// passes register-staged, whole blocks, an x tile within one kz and blocks within the
// x pass's first-stage stride (nx / 16 or more).  The y pass of a 512^3 frame takes
// 321 us against 534 with rows (1.15 GB, 3.6 TB/s), a frame of the loop at 256^3 243
// us against 246.
int res_block(const Plan& p) {
  if (p.fft64) return 0;
  int r1, r2, r3;
  const int nx = p.sys.n[0], ny = p.sys.n[1];
  if ((p.tune_y != 0 && p.tune_y != kTuneReg) || (p.tune_x != 0 && p.tune_x != kTuneReg)) return 0;
  if (!reg_split(ny, &r1, &r2, &r3) || !reg_split(nx, &r1, &r2, &r3)) return 0;
  const int b = kRegElems / ny;
  return kRegElems / nx <= ny && (nx / r1) % b == 0 ? ilog2(b) : 0;
}

// choice: 0 = default (register-staged when n has a split, else the any-length
// pass), kTuneReg = register-staged, 1..16 = the any-length pass with that many
// pencils.  Lengths neither takes (any_plan) run the LDS-staged pass.
template <typename R>
hipError_t run_pass(PassArgs<R> a, PassKind kind, hipStream_t s, int choice) {
  int r1, r2, r3;
  const int n = a.n;
  const size_t nyq_lds = (size_t)4 * lds_pitch(n) * sizeof(double);
  bool reg = (choice == 0 || choice == kTuneReg) && reg_split(n, &r1, &r2, &r3);
  if (!reg && any_ok(n)) return any_pass<R>(a, kind, choice, s);
  size_t lds = 0;
  if (reg) {
    a.P = kRegElems / n;
    // exchange plane (rounded to whole double2), the n axis twiddles, the
    // tile's residual bytes
    lds = (((size_t)a.P * (n + n / 16 + 1) + 1) & ~(size_t)1) * sizeof(double) +
          (size_t)n * sizeof(double2) + (size_t)kRegElems;
    if (a.res_lb && a.res_in) lds += (size_t)16 * (n >> a.res_lb);
  } else {
    a.P = (choice >= 1 && choice <= 16) ? choice : lds_pencils(n);
    while (a.P > 1 && lds_bytes(n, a.P) > max_lds_per_block()) a.P /= 2;
    lds = lds_bytes(n, a.P);
  }
  if (nyq_lds > lds) lds = nyq_lds;
  if (lds > max_lds_per_block()) return hipErrorInvalidValue;
  a.g.tiles_f = (a.g.nf + a.P - 1) / a.P;
  a.g.blocks = (long long)a.g.ns * a.g.tiles_f;
  const long long total = a.g.blocks + (a.nyq ? a.nq_pencils : 0);
  if (total == 0) return hipSuccess;
  const dim3 g((unsigned)total, kind == PK_X_ACC ? 1 : a.nfr);   // frames as grid y
  const bool f32 = sizeof(R) == 4;
  switch (kind) {
    case PK_Y:
      if (reg) {
        if (f32) launch_reg_n<R, false, true, false, EPI_STORE, RES_OUT, false>(n, lds, s, a);
        else launch_reg_n<R, false, true, false, EPI_STORE, RES_NONE, false>(n, lds, s, a);
      } else {
        if (f32) hipLaunchKernelGGL((k_pass_lds<R, false, EPI_STORE, RES_OUT>), g, dim3(kFftThreads), lds, s, a);
        else hipLaunchKernelGGL((k_pass_lds<R, false, EPI_STORE, RES_NONE>), g, dim3(kFftThreads), lds, s, a);
      }
      break;
    case PK_X_ACC:
      if (reg) {
        if (f32) launch_reg_n<R, false, true, true, EPI_ACC, RES_IN, false>(n, lds, s, a);
        else launch_reg_n<R, false, true, true, EPI_ACC, RES_NONE, false>(n, lds, s, a);
      } else {
        if (f32) hipLaunchKernelGGL((k_pass_lds<R, false, EPI_ACC, RES_IN>), g, dim3(kFftThreads), lds, s, a);
        else hipLaunchKernelGGL((k_pass_lds<R, false, EPI_ACC, RES_NONE>), g, dim3(kFftThreads), lds, s, a);
      }
      break;
    case PK_X_STORE:
      if (reg) {
        if (f32) launch_reg_n<R, false, true, true, EPI_STORE, RES_IN, false>(n, lds, s, a);
        else launch_reg_n<R, false, true, true, EPI_STORE, RES_NONE, false>(n, lds, s, a);
      } else {
        if (f32) hipLaunchKernelGGL((k_pass_lds<R, false, EPI_STORE, RES_IN>), g, dim3(kFftThreads), lds, s, a);
        else hipLaunchKernelGGL((k_pass_lds<R, false, EPI_STORE, RES_NONE>), g, dim3(kFftThreads), lds, s, a);
      }
      break;
    case PK_X_INV:
      if (reg) launch_reg_n<R, true, true, true, EPI_STORE, RES_NONE, true>(n, lds, s, a);
      else hipLaunchKernelGGL((k_pass_lds<R, true, EPI_STORE, RES_NONE>), g, dim3(kFftThreads), lds, s, a);
      break;
    default:  // PK_Y_INV
      if (reg) launch_reg_n<R, true, false, true, EPI_STORE, RES_NONE, false>(n, lds, s, a);
      else hipLaunchKernelGGL((k_pass_lds<R, true, EPI_STORE, RES_NONE>), g, dim3(kFftThreads), lds, s, a);
      break;
  }
  return hipGetLastError();
}

template <typename R>
typename V2<R>::T* cx(void* p) {
  return static_cast<typename V2<R>::T*>(p);
}

// Register-staged z pass rows per block for half-length m, 0 without a split.
inline int z_reg_rows(int m) {
  switch (m) {
    case 32: return zreg_rows<32>();
    case 64: return zreg_rows<64>();
    case 128: return zreg_rows<128>();
    case 256: return zreg_rows<256>();
    default: return 0;
  }
}

// Half lengths m the persistent z pass handles (the others take k_r2c_z).
inline bool z_stream_ok(int m) {
  return m == 16 || m == 32 || m == 64 || m == 128 || m == 256 || m == 512 || m == 1024;
}

template <typename R, int R1, int R2, int R3>
void launch_z_stream(long long ntiles, hipStream_t s, ZArgs<R> a) {
  // one round of blocks: at 256^3 the z pass alone takes 27.8 us against
  // 30.0 with two, and the pipelined frame loop is unchanged (the y and x
  // passes lose in the frame loop with one round, so they keep two)
  a.tpb = stream_tpb(reinterpret_cast<const void*>(&k_r2c_z_stream<R, R1, R2, R3>), 0, ntiles, 1);
  const long long grid = (ntiles + a.tpb - 1) / a.tpb;
  if (grid == 0) return;
  pass_launch(k_r2c_z_stream<R, R1, R2, R3>, dim3((unsigned)grid), 0, s, a);
}

template <typename R>
hipError_t pass_z(Plan& p, const void* density, hipStream_t s) {
  // the group's frames lie one after the other: nx rows of planes each
  const int nx = p.sys.n[0] * p.nfr, ny = p.sys.n[1], m = p.sys.n[2] / 2;
  ZArgs<R> a;
  a.in = static_cast<const R*>(density);
  a.out = cx<R>(p.spec);
  a.nyq = static_cast<double2*>(p.spec_nyq);
  a.nx = nx;
  a.ny = ny;
  a.m = m;
  a.ax = p.ax_zc;
  a.tw2 = p.tw_r2c64;
  if (z_stream_ok(m) && (p.tune_z == 0 || p.tune_z == kTuneReg)) {
    a.P = kRegElems / m;
    a.tiles_y = (ny + a.P - 1) / a.P;
    const long long ntiles = (long long)nx * a.tiles_y;
    switch (m) {
      case 16: launch_z_stream<R, 4, 4, 1>(ntiles, s, a); break;
      case 32: launch_z_stream<R, 8, 4, 1>(ntiles, s, a); break;
      case 64: launch_z_stream<R, 8, 8, 1>(ntiles, s, a); break;
      case 128: launch_z_stream<R, 16, 8, 1>(ntiles, s, a); break;
      case 256: launch_z_stream<R, 16, 4, 4>(ntiles, s, a); break;
      case 512: launch_z_stream<R, 16, 8, 4>(ntiles, s, a); break;
      default: launch_z_stream<R, 16, 8, 8>(ntiles, s, a); break;
    }
    return hipGetLastError();
  }
  if (any_ok(m)) return any_r2c<R>(a, p.tune_z, s);
  a.P = (p.tune_z >= 1 && p.tune_z <= 16) ? p.tune_z : lds_pencils(m);
  while (a.P > 1 && lds_bytes(m, a.P) > max_lds_per_block()) a.P /= 2;
  a.tiles_y = (ny + a.P - 1) / a.P;
  hipLaunchKernelGGL((k_r2c_z<R>), dim3((unsigned)((long long)nx * a.tiles_y)), dim3(kFftThreads),
                     lds_bytes(m, a.P), s, a);
  return hipGetLastError();
}

template <typename R>
PassArgs<R> base_args(Plan& p, int n, const FftAxis& ax) {
  PassArgs<R> a{};
  a.n = n;
  a.ax = ax;
  a.nfr = p.nfr;
  // the group's frames one after the other: half spectrum (also in the density
  // buffer), residuals, Nyquist plane
  a.g.in_F = a.g.out_F = a.res_F = (long long)p.sys.n[0] * p.sys.n[1] * (p.sys.n[2] / 2);
  a.nq_F = (long long)p.sys.n[0] * p.sys.n[1];
  return a;
}

// y pass: spec[x][kz][0..Ny) -> rho[kz][ky][x]; Nyquist plane nyq[x][:] in place
template <typename R>
hipError_t pass_y(Plan& p, hipStream_t s) {
  const int nx = p.sys.n[0], ny = p.sys.n[1], m = p.sys.n[2] / 2;
  PassArgs<R> a = base_args<R>(p, ny, p.ax_y);
  a.in = cx<R>(p.spec);
  a.out = cx<R>(p.rho);
  a.res_out = static_cast<unsigned char*>(p.res);
  a.res_lb = res_block(p);
  a.g.in_s = ny;                         // slow = kz
  a.g.in_f = (long long)m * ny;          // fast = x
  a.g.in_e = 1;
  a.g.out_s = (long long)ny * nx;
  a.g.out_f = 1;
  a.g.out_e = nx;
  a.g.nf = nx;
  a.g.ns = m;
  a.nyq = static_cast<double2*>(p.spec_nyq);
  a.nq_p = ny;
  a.nq_e = 1;
  a.nq_pencils = nx;
  return run_pass<R>(a, PK_Y, s, p.tune_y);
}

// x pass: rho[kz][ky][0..Nx) in place (F) or |F|^2 into sf_main; the Nyquist
// plane nyq[:][y] in place or into sf_nyq
template <typename R>
PassArgs<R> x_args(Plan& p, void* rho, void* res, void* nyq) {
  const int nx = p.sys.n[0], ny = p.sys.n[1], m = p.sys.n[2] / 2;
  PassArgs<R> a = base_args<R>(p, nx, p.ax_x);
  a.in = cx<R>(rho);
  a.out = cx<R>(rho);
  a.acc = p.sf_main;
  a.res_in = static_cast<const unsigned char*>(res);
  a.res_lb = res_block(p);
  a.res_ny = ny;
  a.g.in_s = 0;
  a.g.in_f = nx;                         // fast = row kz * Ny + ky
  a.g.in_e = 1;
  a.g.out_s = 0;
  a.g.out_f = nx;
  a.g.out_e = 1;
  a.g.nf = m * ny;
  a.g.ns = 1;
  a.nyq = static_cast<double2*>(nyq);
  a.nyq_acc = p.sf_nyq;
  a.nq_p = 1;
  a.nq_e = ny;
  a.nq_pencils = ny;
  return a;
}

template <typename R>
hipError_t pass_x(Plan& p, bool accumulate, hipStream_t s) {
  return run_pass<R>(x_args<R>(p, p.rho, p.res, p.spec_nyq), accumulate ? PK_X_ACC : PK_X_STORE, s,
                     p.tune_x);
}

// Both frames' x passes with |F|^2 into sf_main / sf_nyq, the frame in slot
// sa first: one read and one write of the FP64 sums for the two frames, the
// same additions in the same order as two single passes.
template <typename R>
hipError_t pass_x_pair(Plan& p, int sa, int sb, hipStream_t s) {
  PassArgs<R> a = x_args<R>(p, p.rho_buf[sa], p.res_buf[sa], p.nyq_buf[sa]);
  a.nfr = 2;   // "frames" a slot's buffers apart
  a.g.in_F = cx<R>(p.rho_buf[sb]) - a.in;
  a.res_F = static_cast<const unsigned char*>(p.res_buf[sb]) - a.res_in;
  a.nq_F = static_cast<double2*>(p.nyq_buf[sb]) - a.nyq;
  return run_pass<R>(a, PK_X_ACC, s, p.tune_x);
}

template <typename R>
hipError_t forward_impl(Plan& p, const void* density, bool accumulate, hipStream_t s) {
  hipError_t e = pass_z<R>(p, density, s);
  if (e != hipSuccess) return e;
  e = pass_y<R>(p, s);
  if (e != hipSuccess) return e;
  return pass_x<R>(p, accumulate, s);
}

// Real adjoint of the forward transform applied to the stored spectrum
// (rho[kz][ky][kx] + nyq after a storing forward pass), each bin first
// multiplied by the FP64 weight w (w_main[kz][ky][kx], w_nyq[x][y]):
//   out(r) = Re sum_{kx, ky, kz in [0, Nz/2]} w(q) X(q) e^{+i q.r}.
template <typename R>
hipError_t inverse_impl(Plan& p, const double* w_main, const double* w_nyq, void* out,
                        hipStream_t s) {
  const int nx = p.sys.n[0], ny = p.sys.n[1], m = p.sys.n[2] / 2;
  {  // x: in place, weights on load
    PassArgs<R> a = base_args<R>(p, nx, p.ax_x);
    a.in = cx<R>(p.rho);
    a.out = cx<R>(p.rho);
    a.w = w_main;
    a.g.in_s = 0;
    a.g.in_f = nx;
    a.g.in_e = 1;
    a.g.out_s = 0;
    a.g.out_f = nx;
    a.g.out_e = 1;
    a.g.nf = m * ny;
    a.g.ns = 1;
    a.nyq = static_cast<double2*>(p.spec_nyq);
    a.nyq_w = w_nyq;
    a.nq_p = 1;
    a.nq_e = ny;
    a.nq_pencils = ny;
    const hipError_t e = run_pass<R>(a, PK_X_INV, s, 0);
    if (e != hipSuccess) return e;
  }
  {  // y: rho[kz][:][x] -> spec[x][kz][:]
    PassArgs<R> a = base_args<R>(p, ny, p.ax_y);
    a.in = cx<R>(p.rho);
    a.out = cx<R>(p.spec);
    a.g.in_s = (long long)ny * nx;       // slow = kz
    a.g.in_f = 1;                        // fast = x
    a.g.in_e = nx;
    a.g.out_s = ny;
    a.g.out_f = (long long)m * ny;
    a.g.out_e = 1;
    a.g.nf = nx;
    a.g.ns = m;
    a.nyq = static_cast<double2*>(p.spec_nyq);
    a.nq_p = ny;
    a.nq_e = 1;
    a.nq_pencils = nx;
    const hipError_t e = run_pass<R>(a, PK_Y_INV, s, 0);
    if (e != hipSuccess) return e;
  }
  CArgs<R> c;
  c.spec = cx<R>(p.spec);
  c.nyq = static_cast<const double2*>(p.spec_nyq);
  c.out = static_cast<R*>(out);
  c.nx = nx * p.nfr;   // the group's frames one after the other
  c.ny = ny;
  c.m = m;
  c.ax = p.ax_zc;
  c.tw2 = p.tw_r2c64;
  if (z_reg_rows(m) > 0) {
    c.P = z_reg_rows(m);
    c.tiles_y = (ny + c.P - 1) / c.P;
    const dim3 g((unsigned)((long long)c.nx * c.tiles_y)), b(kFftThreads);
    switch (m) {
      case 32: hipLaunchKernelGGL((k_c2r_z_reg<R, 8, 4>), g, b, 0, s, c); break;
      case 64: hipLaunchKernelGGL((k_c2r_z_reg<R, 8, 8>), g, b, 0, s, c); break;
      case 128: hipLaunchKernelGGL((k_c2r_z_reg<R, 16, 8>), g, b, 0, s, c); break;
      default: hipLaunchKernelGGL((k_c2r_z_reg<R, 16, 16>), g, b, 0, s, c); break;
    }
    return hipGetLastError();
  }
  if (any_ok(m)) return any_c2r<R>(c, s);
  c.P = lds_pencils(m);
  while (c.P > 1 && lds_bytes(m, c.P) > max_lds_per_block()) c.P /= 2;
  c.tiles_y = (ny + c.P - 1) / c.P;
  hipLaunchKernelGGL((k_c2r_z<R>), dim3((unsigned)((long long)c.nx * c.tiles_y)), dim3(kFftThreads),
                     lds_bytes(m, c.P), s, c);
  return hipGetLastError();
}

// stored spectrum (rho[kz][ky][kx] complex, nyq[x][y] FP64) -> complex128 (Nx, Ny, Nz/2+1)
template <typename R>
__global__ __launch_bounds__(kHalfThreads) void k_spec_read(
    const typename V2<R>::T* __restrict__ main, const double2* __restrict__ nyq,
    double2* __restrict__ out, int nx, int ny, int m) {
  half_to_rows<double2>(
      nx, ny, m,
      [&](int kz, int y, int x) {
        const auto v = main[((long long)kz * ny + y) * nx + x];
        return make_double2((double)v.x, (double)v.y);
      },
      [&](int x, int y) { return nyq[(long long)x * ny + y]; },
      [&](int x, int y, int kz, double2 v) { out[((long long)x * ny + y) * (m + 1) + kz] = v; });
}

}  // namespace

bool fft_factor(int n, int* radix, int* nstages) {
  int k = 0;
  int m = n;
  static const int pref[] = {16, 8, 4, 2, 3, 5};
  for (int r : pref) {
    while (m % r == 0 && m > 1) {
      if (k >= kMaxStages) return false;
      radix[k++] = r;
      m /= r;
    }
  }
  for (int r = 7; m > 1; r += 2) {  // remaining odd primes: generic stage
    while (m % r == 0) {
      if (k >= kMaxStages) return false;
      radix[k++] = r;
      m /= r;
    }
  }
  *nstages = k;
  return true;
}

hipError_t fft_make_twiddles(float2* tw, double2* tw64, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_twiddles, dim3((n + 255) / 256), dim3(256), 0, s, tw, tw64, n);
  return hipGetLastError();
}

hipError_t fft_forward(Plan& p, const void* density, bool accumulate, hipStream_t s) {
  return p.fft64 ? forward_impl<double>(p, density, accumulate, s)
                 : forward_impl<float>(p, density, accumulate, s);
}

namespace {

struct TuneKey {
  int n[3];
  int fft64;
  bool operator<(const TuneKey& o) const {
    for (int d = 0; d < 3; ++d)
      if (n[d] != o.n[d]) return n[d] < o.n[d];
    return fft64 < o.fft64;
  }
};
struct TuneVal {
  int z, y, x;
};
std::mutex g_tune_mu;
std::map<TuneKey, TuneVal> g_tune_cache;

// Best of 3 timed launches (after one warm-up) of `run` on stream s, in ms.
template <typename F>
float time_best(F&& run, hipStream_t s, hipEvent_t e0, hipEvent_t e1, hipError_t* err) {
  float best = 1e30f;
  for (int it = 0; it < 4; ++it) {
    (void)hipEventRecord(e0, s);
    const hipError_t e = run();
    (void)hipEventRecord(e1, s);
    if (e != hipSuccess) {
      *err = e;
      return best;
    }
    if ((*err = hipEventSynchronize(e1)) != hipSuccess) return best;
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    if (it > 0 && ms < best) best = ms;
  }
  return best;
}

template <typename R>
hipError_t autotune_impl(Plan& p, hipStream_t s) {
  const int m = p.sys.n[2] / 2;
  hipEvent_t e0, e1;
  hipError_t err = hipEventCreate(&e0);
  if (err != hipSuccess) return err;
  if ((err = hipEventCreate(&e1)) != hipSuccess) {
    (void)hipEventDestroy(e0);
    return err;
  }
  const int cand[5] = {kTuneReg, 2, 4, 8, 16};
  // z pass: the register-staged kernel (m with a two-stage split) or the any-length
  // pass (else the LDS-staged one) with that many rows.  Tiles too large for the
  // LDS-staged pass are left out for both: the any-length pass holds fewer values in
  // LDS, but at most 4,096 a block, and would halve such a tile to one already timed.
  float best = 1e30f;
  int pick = 0;
  for (int c : cand) {
    if (c == kTuneReg && !z_stream_ok(m)) continue;
    if (c != kTuneReg && lds_bytes(m, c) > max_lds_per_block()) continue;
    p.tune_z = c;
    const float t = time_best([&] { return pass_z<R>(p, p.rho, s); }, s, e0, e1, &err);
    if (err != hipSuccess) break;
    if (t < best) {
      best = t;
      pick = c;
    }
  }
  p.tune_z = pick;
  // y and x passes: the same choice
  for (int axis = 0; axis < 2 && err == hipSuccess; ++axis) {
    int& slot = axis == 0 ? p.tune_y : p.tune_x;
    const int n = p.sys.n[axis == 0 ? 1 : 0];
    int r1, r2, r3;
    best = 1e30f;
    pick = 0;
    for (int c : cand) {
      if (c == kTuneReg && !reg_split(n, &r1, &r2, &r3)) continue;
      if (c != kTuneReg && lds_bytes(n, c) > max_lds_per_block()) continue;
      slot = c;
      const float t = time_best(
          [&] { return axis == 0 ? pass_y<R>(p, s) : pass_x<R>(p, true, s); }, s, e0, e1, &err);
      if (err != hipSuccess) break;
      if (t < best) {
        best = t;
        pick = c;
      }
    }
    slot = pick;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return err;
}

}  // namespace

// Picks the z tile height and the y / x pass kernels for this grid by timing
// the candidates on the plan's own buffers (results cached per grid shape and
// precision).  Clobbers the density, spectrum and S(q) accumulators.
hipError_t fft_autotune(Plan& p, hipStream_t s) {
  const TuneKey key{{p.sys.n[0], p.sys.n[1], p.sys.n[2]}, p.fft64};
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tune_cache.find(key);
    if (it != g_tune_cache.end()) {
      p.tune_z = it->second.z;
      p.tune_y = it->second.y;
      p.tune_x = it->second.x;
      return hipSuccess;
    }
  }
  const hipError_t e = p.fft64 ? autotune_impl<double>(p, s) : autotune_impl<float>(p, s);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_tune_cache[key] = TuneVal{p.tune_z, p.tune_y, p.tune_x};
  return hipSuccess;
}

hipError_t fft_inverse(Plan& p, const double* w_main, const double* w_nyq, void* out,
                       hipStream_t s) {
  return p.fft64 ? inverse_impl<double>(p, w_main, w_nyq, out, s)
                 : inverse_impl<float>(p, w_main, w_nyq, out, s);
}

void fft_pass_events(hipEvent_t begin, hipEvent_t end) {
  t_pass_ev[0] = begin;
  t_pass_ev[1] = end;
  t_pass_ev_used = false;
}

bool fft_pass_events_used() { return t_pass_ev_used; }

bool fft_x_pairs(const Plan& p) { return p.group == 1; }

hipError_t fft_x_pair(Plan& p, int slot_a, int slot_b, hipStream_t s) {
  return p.fft64 ? pass_x_pair<double>(p, slot_a, slot_b, s)
                 : pass_x_pair<float>(p, slot_a, slot_b, s);
}

hipError_t fft_pass(Plan& p, int pass, const void* density, hipStream_t s) {
  switch (pass) {
    case 0: return p.fft64 ? pass_z<double>(p, density, s) : pass_z<float>(p, density, s);
    case 1: return p.fft64 ? pass_y<double>(p, s) : pass_y<float>(p, s);
    default: return p.fft64 ? pass_x<double>(p, true, s) : pass_x<float>(p, true, s);
  }
}

hipError_t fft_spectrum_read(Plan& p, double* out, hipStream_t s) {
  const int nx = p.sys.n[0], ny = p.sys.n[1], m = p.sys.n[2] / 2;
  const dim3 grid(half_tiles(nx, ny, m)), block(kHalfThreads);
  if (p.fft64)
    hipLaunchKernelGGL(k_spec_read<double>, grid, block, 0, s, cx<double>(p.rho), static_cast<const double2*>(p.spec_nyq),
                       reinterpret_cast<double2*>(out), nx, ny, m);
  else
    hipLaunchKernelGGL(k_spec_read<float>, grid, block, 0, s, cx<float>(p.rho), static_cast<const double2*>(p.spec_nyq),
                       reinterpret_cast<double2*>(out), nx, ny, m);
  return hipGetLastError();
}

size_t fft_spec_bytes(const int n[3], int fft64) {
  return (size_t)n[0] * n[1] * (n[2] / 2) * (fft64 ? 16 : 8);
}

size_t fft_res_bytes(const int n[3], int fft64) {
  return fft64 ? 0 : (size_t)n[0] * n[1] * (n[2] / 2);
}

// --- plan-free transform for callers that cannot allocate -----------------------
// The working set of mdsf_rfft3_noalloc (twiddles, the z and y pass outputs,
// the y pass residuals, Nyquist plane) lives in this fixed device array, one copy per GPU, held until the
// process ends.  Host code never passes the array's name to a kernel: it is a
// host-side stand-in.  The device address of each GPU's copy comes from
// hipGetSymbolAddress on the first call on that device and is kept per device.
namespace {

constexpr size_t kScratchBytes = (size_t)144 << 20;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned char* g_scratch_ptr[kMaxDevices] = {};

// Device address of the current device's scratch array (resolved once per device).
hipError_t scratch_address(unsigned char** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_ptr[dev] = static_cast<unsigned char*>(ptr);
  }
  *out = g_scratch_ptr[dev];
  return hipSuccess;
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

}  // namespace

}  // namespace mdsf

extern "C" int mdsf_rfft3_noalloc(const int32_t n[3], int precision, const void* d_density,
                                  double* d_spectrum, mdsf_stream stream) {
  using namespace mdsf;
  if (!n || !d_density || !d_spectrum) return fail(MDSF_ERR_ARG, "null argument");
  if (precision != MDSF_F32 && precision != MDSF_F64)
    return fail(MDSF_ERR_ARG, "precision must be MDSF_F32 or MDSF_F64");
  for (int d = 0; d < 3; ++d)
    if (n[d] < 2 || n[d] % 2 != 0 || n[d] > 4096)
      return fail(MDSF_ERR_ARG, "grid sizes must be even and in [2, 4096]");
  const int fft64 = precision == MDSF_F64 ? 1 : 0;
  const int nn[3] = {n[0], n[1], n[2]};
  const size_t nx = n[0], ny = n[1], nz = n[2], m = nz / 2;
  // layout: the spectrum buffer (the y pass output, transformed in place by
  // the x pass), the z pass output, the y pass residuals (FP32), the Nyquist
  // plane (FP64 complex), then the FP64 twiddles of the x, y, z/2 axes and
  // of the R2C split (length nz)
  const size_t lens[4] = {nx, ny, m, nz};
  size_t off = 0;
  const size_t off_rho = off;
  off = align256(off + fft_spec_bytes(nn, fft64));
  const size_t off_spec = off;
  off = align256(off + fft_spec_bytes(nn, fft64));
  const size_t off_res = off;
  off = align256(off + fft_res_bytes(nn, fft64));
  const size_t off_nyq = off;
  off = align256(off + sizeof(double2) * nx * ny);
  size_t off_tw64[4];
  for (int k = 0; k < 4; ++k) {
    off_tw64[k] = off;
    off = align256(off + sizeof(double2) * lens[k]);
  }
  if (off > kScratchBytes)
    return fail(MDSF_ERR_ARG, "grid too large for mdsf_rfft3_noalloc: it needs " +
                                  std::to_string(off) + " bytes of its " +
                                  std::to_string(kScratchBytes) +
                                  "-byte device scratch array (use a plan and mdsf_rfft3)");
  unsigned char* base = nullptr;
  MDSF_HIP(scratch_address(&base));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  Plan p;  // host-side description only: every device pointer is into `base`
  for (int d = 0; d < 3; ++d) p.sys.n[d] = n[d];
  p.fft64 = fft64;
  p.rho = base + off_rho;
  p.spec = base + off_spec;
  p.res = fft_res_bytes(nn, fft64) > 0 ? base + off_res : nullptr;
  p.spec_nyq = base + off_nyq;
  FftAxis* axes[3] = {&p.ax_x, &p.ax_y, &p.ax_zc};
  for (int k = 0; k < 4; ++k) {
    double2* tw64 = reinterpret_cast<double2*>(base + off_tw64[k]);
    if (k < 3) {
      FftAxis& ax = *axes[k];
      ax.n = (int)lens[k];
      if (!fft_factor(ax.n, ax.radix, &ax.nstages))
        return fail(MDSF_ERR_UNSUPPORTED,
                    "FFT length " + std::to_string(ax.n) + " needs too many stages");
      ax.tw = nullptr;
      ax.tw64 = tw64;
    } else {
      p.tw_r2c = nullptr;
      p.tw_r2c64 = tw64;
    }
    MDSF_HIP(fft_make_twiddles(nullptr, tw64, (int)lens[k], s));
  }
  MDSF_HIP(fft_forward(p, d_density, false, s));
  MDSF_HIP(fft_spectrum_read(p, d_spectrum, s));
  return MDSF_OK;
}
