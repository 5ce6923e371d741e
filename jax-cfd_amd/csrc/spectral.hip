// Pseudospectral vorticity step (NavierStokes2D + a low-storage Runge-Kutta /
// Crank-Nicolson stepper: crank_nicolson_rk4, _rk3 or any tableau) for gfx950.
//
// State: the complex64 rfft2 of the vorticity, (n, n/2+1) per instance
// (jax_cfd/spectral/equations.py:129-190).  One step
// (spectral/time_stepping.py:117-170; CN-RK4, 186-197, has five) is stages of
//   F = explicit_terms(u);  h = F + beta_k h;
//   u = (u + gamma_k dt h + mu_k L u) / (1 - mu_k L),  L = nu lap - drag,
// where explicit_terms = filter * rfftn(-(d_x w * v_x + d_y w * v_y)) + forcing
// curl, with v from vorticity_to_velocity (spectral/utils.py:154-189).
//
// Kernels (all launched with blockIdx.y = instance of a same-size batch):
//   ns_cols_inverse   column tile of W packed columns: build the four spectra
//                     d_x w, d_y w, v_x, v_y (scaled by 1/n^2), inverse column
//                     FFT each, write them packed -> G[4].
//   ns_rows           RB rows: four inverse packed real row FFTs, the
//                     product -(gx vx + gy vy), forward packed real row FFT -> P.
//   ns_cols_forward   column tile: forward column FFT of P, unpack the DC/
//                     Nyquist word, 2/3 filter, forcing curl, then the RK/CN
//                     update of (u, h), optionally followed directly by the
//                     next stage's ns_cols_inverse work on the same tile.
//   rows_r2c, ns_cols_out and ns_cols_in, rows_c2r   rfft2 and irfft2; the
//                     explicit-terms seam ends in ns_cols_out.
//
// Packed half spectra: word 0 of a row holds (X[0], X[n/2]) of a real row;
// the column pass of word 0 therefore carries two Hermitian columns, which
// are separated with Y(p) = A(p) + i B(p), A = (Y(p) + conj Y(-p))/2,
// B = (Y(p) - conj Y(-p))/(2i).  On the way in, (A, B) are symmetrised the
// same way, which reproduces irfftn's dropping of the imaginary parts of the
// DC and Nyquist columns after the axis-0 inverse transform.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "jcfd_fft.h"
#include "jcfd_internal.h"

#pragma clang fp contract(off)

namespace jcfd {
namespace {

constexpr int kThreads = 256;

// Internal layout of packed half spectra (n rows x n/2 words: the four
// derivative spectra G and the product spectrum P): column tiles of kTw<N>
// words, each tile one contiguous block of n rows x kTw words.  kTw is the
// number of columns a column kernel's wavefront holds side by side, up to 4:
// its loads and stores are then whole contiguous runs (at 64 x 512^2 the
// update-and-inverse kernel took 123 / 146 / 185 us with tiles of 1 / 2 / 4
// words), while the row kernel's pieces are its rows x kTw words.
template <int N>
constexpr int kTw = N == 512 ? 1 : N == 1024 || N == 256 ? 2 : 4;
template <int N>
__device__ __forceinline__ int tix(int p, int c) {
  return ((c / kTw<N>) * N + p) * kTw<N> + (c % kTw<N>);
}
// Internal state layout (n rows x (n/2 + 1) words, the same size as the
// external rfft2 layout): columns 0 .. n/2 - 1 tiled as above, then column
// n/2 (the Nyquist column) as n consecutive words.
template <int N>
__device__ __forceinline__ int six(int p, int c) {
  return c < N / 2 ? tix<N>(p, c) : (N / 2) * N + p;
}

// Per-element multipliers of the four derivative spectra, following the
// reference's fp32/complex64 operation order.
struct NsMult {
  float ax;   // 2 pi kx  (d_x multiplier is i ax)
  float ay;   // 2 pi ky
  float psi;  // -1 / laplace'  (laplace' = (2 pi i)^2 (kx^2 + ky^2), [0,0] := 1)
};

__device__ __forceinline__ NsMult ns_mult(const NsParams& q, float kx, float ky, bool origin) {
  NsMult m;
  m.ax = q.two_pi * kx;
  m.ay = q.two_pi * ky;
  const float s = kx * kx + ky * ky;
  const float lap = origin ? 1.0f : q.neg_four_pi_sq * s;
  m.psi = -1.0f / lap;
  return m;
}

// i a * z
__device__ __forceinline__ float2 mul_i(float a, float2 z) { return make_float2(-a * z.y, a * z.x); }

// ---- column kernels ----------------------------------------------------------
// A column transform is held in the registers of one wavefront's lanes
// (reg_fft): N / E lanes per column, T columns side by side, neighbouring
// lanes on neighbouring columns.  E = 8 words per lane (16 for N = 1024), so a
// wavefront's tile is 512 (1024) words.  Everything a lane needs between the
// forward transform, the update and the inverse transforms of the four
// spectra sits at the same rows p = j + e L, so the tile never leaves its
// registers: LDS carries two exchanges per 512-point transform, and no
// workgroup barrier exists; the wavefronts of a workgroup are independent.
// What bounds them is the stream of u, h, P and G: 16 x 512^2
// update-and-inverse 30 us (5.0 TB/s) where the staged kernel takes 39,
// 64 x 256^2 30 (35), 8 x 1024^2 68 (97).  Steps: 64 x 256^2 336 -> 277 us,
// 256 x 128^2 364 -> 256, 32 x 512^2 599 -> 548, 8 x 1024^2 759 -> 645
// (staged kernels at their best shapes -> these).
template <int N>
struct ColShape {
  static constexpr int E = N == 1024 ? 16 : 8;
  static constexpr int L = N / E;  // lanes per column
  static constexpr int T = 64 / L;  // columns per wavefront
};
template <int N>
constexpr int col_waves(int w) {  // wavefronts of a workgroup of w columns
  return (w + ColShape<N>::T - 1) / ColShape<N>::T;
}
// LDS of a workgroup of `waves` wavefronts: their exchange buffers, then
// vorticity columns 0 and N/2 of tile 0.
template <int N>
constexpr int col_lds(int waves) {
  return (waves * kRegFftWords<N, ColShape<N>::T> + 2 * N) * static_cast<int>(sizeof(float2));
}
template <int N>
struct ColLds {
  float2 *x, *w0, *wn;
  __device__ __forceinline__ ColLds(char* smem, int waves, int wave) {
    float2* f = reinterpret_cast<float2*>(smem);
    x = f + wave * kRegFftWords<N, ColShape<N>::T>;
    w0 = f + waves * kRegFftWords<N, ColShape<N>::T>;
    wn = w0 + N;
  }
};

// One lane's place in its wavefront's tile of columns from c0, of which the
// workgroup owns the first w.
template <int N>
struct ColLane {
  static constexpr int E = ColShape<N>::E, L = ColShape<N>::L, T = ColShape<N>::T;
  int j;     // rows j + e L
  int c;     // column
  int t;     // its index in the wavefront
  bool own;  // whether the column is this workgroup's (false: a surplus lane, which works on column c0 and stores nothing)
  __device__ __forceinline__ ColLane(int c0, int w, int lane) : j(lane / T), c(c0), t(lane % T), own(lane % T < w) {
    if (own) c = c0 + t;
  }
};

// kx at row p = j + e L (e a compile-time number once unrolled): the table
// entry fp32(index) / fp32(dx n), by over_step's correctly rounded quotient,
// so neither loads nor registers are spent on the table.
template <int N>
__device__ __forceinline__ float lane_kx(const NsParams& q, float jf, int e) {
  constexpr int E = ColShape<N>::E, L = ColShape<N>::L;
  return over_step(jf + static_cast<float>(e < E / 2 ? e * L : e * L - N), q.dnx, q.rcp_dnx);
}

// x, as a value the compiler has to take as new: what is computed from it is
// recomputed where it is used instead of being kept in registers from an
// earlier use (a loop's invariants and the values shared by its halves cost
// the column kernels the fourth wavefront per SIMD).
__device__ __forceinline__ float recompute(float x) {
  asm volatile("" : "+v"(x));
  return x;
}

// Inverse column transforms of the tile -> G[0..4): the four derivative
// spectra (d_x w, d_y w, v_x, v_y), scaled by 1/n^2.  w becomes psi w, psi = -1/laplacian, for the last two, so
// no second array is held.  Column 0 is the symmetrised pair of the DC and
// Nyquist columns, s0 + i sh with s(p) = (a(p) + conj a(-p)) / 2, from the two
// columns in LDS (w0, wn): kx(-p) = -kx(p) (but at 0 and N/2), psi(-p) = psi(p).
template <int N, int R, typename TW>
__device__ __forceinline__ void cols_inverse_body(float2 (&w)[ColShape<N>::E], const TW& tw, const ColLane<N>& ln,
                                                  const ColLds<N>& lds, const NsParams& q,
                                                  float2* __restrict__ g) {
  using S = ColShape<N>;
  constexpr int E = S::E, L = S::L, H = N / 2;
  const size_t gstride = static_cast<size_t>(N) * H;
  const float ky = q.ky[ln.c], kyh = q.ky[H];
  const float ay = q.two_pi * ky, ayh = q.two_pi * kyh;
#pragma unroll 1
  for (int m = 0; m < 4; ++m) {
    const float jf = recompute(static_cast<float>(ln.j));
    if (m == 2) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const float psi = ns_mult(q, lane_kx<N>(q, jf, e), ky, ln.c == 0 && ln.j + e * L == 0).psi;
        w[e] = make_float2(psi * w[e].x, psi * w[e].y);
      }
      if (ln.c == 0 && ln.own) {  // the two columns in LDS likewise
        wave_lds_sync();
#pragma unroll
        for (int e = 0; e < E; ++e) {
          __builtin_amdgcn_sched_barrier(0);
          const int p = ln.j + e * L;
          const float psih = ns_mult(q, lane_kx<N>(q, jf, e), kyh, false).psi;
          lds.w0[p] = w[e];
          lds.wn[p] = make_float2(psih * lds.wn[p].x, psih * lds.wn[p].y);
        }
        wave_lds_sync();
      }
    }
    // the spectrum's multiplier is i times kx or ky; v_y's is -i kx
    const bool along_y = m == 1 || m == 2;
    const float sign = m == 3 ? -1.0f : 1.0f;
    float2 v[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const float k = along_y ? ay : q.two_pi * lane_kx<N>(q, jf, e);
      v[e] = mul_i(sign * k, w[e]);
    }
    if (ln.c == 0 && ln.own) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        __builtin_amdgcn_sched_barrier(0);  // one element's temporaries at a time
        const int p = ln.j + e * L, pm = (N - p) & (N - 1);
        const float2 z0 = lds.w0[pm], zp = lds.wn[p], zm = lds.wn[pm];
        const float kx1 = lane_kx<N>(q, jf, e);
        const float kp = sign * (q.two_pi * kx1), km = pm == p ? kp : -kp;
        const float2 a0 = v[e];
        const float2 b0 = mul_i(along_y ? ay : km, z0);
        const float2 ah = mul_i(along_y ? ayh : kp, zp);
        const float2 bh = mul_i(along_y ? ayh : km, zm);
        const float2 s0 = make_float2(0.5f * (a0.x + b0.x), 0.5f * (a0.y - b0.y));
        const float2 sh = make_float2(0.5f * (ah.x + bh.x), 0.5f * (ah.y - bh.y));
        v[e] = make_float2(s0.x - sh.y, s0.y + sh.x);  // s0 + i sh
      }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) v[e] = make_float2(v[e].x * q.inv_nn, v[e].y * q.inv_nn);
    reg_fft<N, E, S::T, true, R>(v, tw, lds.x + ln.t, ln.j);
    if (ln.own) {
      float2* gm = g + m * gstride + tix<N>(ln.j, ln.c);
#pragma unroll
      for (int e = 0; e < E; ++e) gm[e * (L * kTw<N>)] = v[e];
    }
  }
}

// Minimum waves per SIMD asked of the column kernels: 128 registers hold an E =
// 8 tile with its old (u, h) and twiddles, 256 an E = 16 one.
template <int N>
struct NsColOcc {
  static constexpr int value = N == 1024 ? 2 : 4;
};

// One wavefront's columns from c0: the state (internal layout) -> the inverse
// transforms of the four spectra; w and g already point at the instance.
template <int N, int R>
__device__ __forceinline__ void cols_inverse_tile(const ColLds<N>& lds, const NsParams& q,
                                                  const float2* __restrict__ w, float2* __restrict__ g,
                                                  int c0, int width, int lane) {
  using S = ColShape<N>;
  constexpr int E = S::E, L = S::L, H = N / 2;
  const ColLane<N> ln(c0, width, lane);
  float2 wt[E];
#pragma unroll
  for (int e = 0; e < E; ++e) wt[e] = w[six<N>(ln.j + e * L, ln.c)];
  RegTwiddles<N, E, R> tw;
  tw.template load<1>(q.tw, ln.j);
  if (c0 == 0) {
    if (ln.c == 0 && ln.own) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        lds.w0[ln.j + e * L] = wt[e];
        lds.wn[ln.j + e * L] = w[six<N>(ln.j + e * L, H)];
      }
    }
    wave_lds_sync();
  }
  cols_inverse_body<N, R>(wt, tw, ln, lds, q, g);
}

template <int N, int R>
__global__ __launch_bounds__(1024 / ColShape<N>::E * 8, (NsColOcc<N>::value)) void ns_cols_inverse(
    NsParams q, const float2* __restrict__ w, float2* __restrict__ g, int width) {
  extern __shared__ float4 ns_smem[];
  const int wave = threadIdx.x / 64;
  const ColLds<N> lds(reinterpret_cast<char*>(ns_smem), blockDim.x / 64, wave);
  const int c0 = xcd_tile(blockIdx.x, gridDim.x) * width + wave * ColShape<N>::T;
  const size_t inst = q.slots ? static_cast<size_t>(q.slots[blockIdx.y]) : blockIdx.y;
  cols_inverse_tile<N, R>(lds, q, w + inst * static_cast<size_t>(N) * (N / 2 + 1),
                          g + inst * 4 * static_cast<size_t>(N) * (N / 2), c0, width, threadIdx.x % 64);
}

// Packed real row transforms of a batch of real (N, N) fields.  Between the
// passes of rfft2 and irfft2 the packed words lie row by row: both passes then
// read and write runs of a row (in the step's column tiles, one word wide at
// 512^2, the row pass stores single words; rfft2 and irfft2 of 64 x 512^2 in
// those tiles 110 and 103 us, row by row 63 and 64).
template <int N, int RB>
__global__ __launch_bounds__(kThreads) void rows_r2c(NsParams q, const float* __restrict__ x,
                                                     float2* __restrict__ pout) {
  constexpr int H = N / 2;
  __shared__ float2 zb[RB * H];
  __shared__ float2 twn[N];
  __shared__ float2 twh[H];
  const int tid = threadIdx.x;
  const int i0 = xcd_tile(blockIdx.x, gridDim.x) * RB;
  const size_t inst = q.slots ? static_cast<size_t>(q.slots[blockIdx.y]) : blockIdx.y;
  x += inst * static_cast<size_t>(N) * N;
  pout += inst * static_cast<size_t>(N) * H;
  TwiddleStage<N, 1, kThreads> ta;
  TwiddleStage<H, 2, kThreads> tb;
  ta.load(q.tw, tid);
  tb.load(q.tw, tid);
  const float* xr = x + static_cast<size_t>(i0) * N;
  float* zf = reinterpret_cast<float*>(zb);
  staged<RB * N, 16, kThreads>(tid, [&](int e) { return xr[e]; }, [&](int e, float v) { zf[e] = v; });
  ta.store(twn, tid);
  tb.store(twh, tid);
  __syncthreads();
  lds_fft_waves<H, RB, kThreads, 1, H, false>(zb, twh, tid);
  for (int e = tid; e < RB * H; e += kThreads) {
    const int r = e / H, k = e % H;
    pout[(i0 + r) * H + k] = r2c_combine(zb + r * H, k, H, twn[k]);
  }
}

template <int N, int RB>
__global__ __launch_bounds__(kThreads) void rows_c2r(NsParams q, const float2* __restrict__ pin,
                                                     float* __restrict__ x) {
  constexpr int H = N / 2;
  __shared__ float2 zb[RB * H];
  __shared__ float2 twh[H];
  const int tid = threadIdx.x;
  const int i0 = xcd_tile(blockIdx.x, gridDim.x) * RB;
  const size_t inst = q.slots ? static_cast<size_t>(q.slots[blockIdx.y]) : blockIdx.y;
  x += inst * static_cast<size_t>(N) * N;
  pin += inst * static_cast<size_t>(N) * H;
  TwiddleStage<H, 2, kThreads> tb;
  tb.load(q.tw, tid);
  staged<RB * H, 8, kThreads>(
      tid,
      [&](int e) {
        const int r = e / H, k = e % H;
        return F2Triple{pin[(i0 + r) * H + k], pin[(i0 + r) * H + ((H - k) & (H - 1))], q.tw[k]};
      },
      [&](int e, F2Triple v) { zb[e] = c2r_combine(v.a, v.b, e % H, v.t); });
  tb.store(twh, tid);
  __syncthreads();
  lds_fft_waves<H, RB, kThreads, 1, H, true>(zb, twh, tid);
  const float* zf = reinterpret_cast<const float*>(zb);
  for (int e = tid; e < RB * N; e += kThreads) x[static_cast<size_t>(i0) * N + e] = zf[e];
}

// ---- row kernel -----------------------------------------------------------
// A wavefront transforms RS rows of one spectrum in registers (512 words, E =
// 8 per lane); the four wavefronts of a group take the four spectra of the
// same rows, wavefront 0 then forms the product and transforms it forward
// (64 x 256^2: 31 us with every pass staged in LDS, 22 us so).
// RB rows per workgroup: RB / RS groups, or one group with surplus lanes.
template <int N>
struct RowShape {
  static constexpr int H = N / 2, E = 8;
  static constexpr int L = H / E;      // lanes per row
  static constexpr int RS = 64 / L;    // rows per wavefront
};
template <int N>
constexpr int row_groups(int rb) {
  return rb > RowShape<N>::RS ? rb / RowShape<N>::RS : 1;
}
template <int N>
constexpr int kRowBuffer = kRegFftWords<N / 2, RowShape<N>::RS>;  // words per wavefront
template <int N>
constexpr int row_lds(int rb) {
  return row_groups<N>(rb) * 4 * kRowBuffer<N> * static_cast<int>(sizeof(float2));
}

// NR rows per group from i0: spectrum m = wave % 4 of G -> the product
// spectrum rows of P; g and pout already point at the instance.
template <int N, int NR, int R>
__device__ __forceinline__ void rows_tile(float2* smem, const NsParams& q, const float2* __restrict__ g,
                                          float2* __restrict__ pout, int i0, int tid) {
  using S = RowShape<N>;
  constexpr int H = S::H, E = S::E, L = S::L, RS = S::RS, HH = H / 2, TW = kTw<N>;
  static_assert(NR <= RS, "rows per wavefront");
  const int wave = tid / 64, lane = tid % 64, m = wave % 4;
  i0 += (wave / 4) * NR;
  float2* xb = smem + wave * kRowBuffer<N>;
  const float2* gm = g + m * static_cast<size_t>(N) * H;
  // Loads in the tiled layout's memory order (word of the tile, row, tile),
  // in mirror pairs (kk, H - kk), kk < H/2: both outputs of a pair need both
  // words, so each word is read once; word H/2 (its own mirror) goes alone.
  // Element k of row r goes to LDS word fft_pad(k) RS + r, where the
  // transform's lanes pick it up.
  constexpr int TOT = NR * HH, PER = (TOT + 63) / 64;
  auto row_of = [](int e) { return (e / TW) % NR; };
  auto word_of = [](int e) { return (e / (TW * NR)) * TW + e % TW; };
  float2 a[PER], b[PER], ta[PER], tb[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e0 = lane + 64 * k, e = TOT % 64 == 0 || e0 < TOT ? e0 : TOT - 1;
    const int r = row_of(e), kk = word_of(e);
    a[k] = gm[tix<N>(i0 + r, kk)];
    b[k] = gm[tix<N>(i0 + r, (H - kk) & (H - 1))];
    ta[k] = q.tw[kk];
    tb[k] = q.tw[(H - kk) & (N - 1)];
  }
  float2 mid = make_float2(0.f, 0.f);
  const float2 tmid = q.tw[HH];
  if (lane < NR) mid = gm[tix<N>(i0 + lane, HH)];
  const int j = lane / RS, t = lane % RS;
  RegTwiddles<H, E, R> tw;
  tw.template load<2>(q.tw, j);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e = lane + 64 * k;
    if (TOT % 64 == 0 || e < TOT) {
      const int r = row_of(e), kk = word_of(e);
      xb[fft_pad(kk) * RS + r] = c2r_combine(a[k], b[k], kk, ta[k]);
      if (kk != 0) xb[fft_pad(H - kk) * RS + r] = c2r_combine(b[k], a[k], H - kk, tb[k]);
    }
  }
  if (lane < NR) xb[fft_pad(HH) * RS + lane] = c2r_combine(mid, mid, HH, tmid);
  wave_lds_sync();
  float2 v[E];
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = xb[fft_pad(j) * RS + fft_pad(e * L) * RS + t];
  reg_fft<H, E, RS, true, R>(v, tw, xb + t, j);
  // advection = -(grad_x * vx + grad_y * vy)  (spectral/equations.py:170):
  // each wavefront leaves its field in its own buffer, wavefront 0 of the
  // group reads the other three
  if (m != 0) {
    wave_lds_sync();
#pragma unroll
    for (int e = 0; e < E; ++e) xb[lane + 64 * e] = v[e];
  }
  __syncthreads();
  if (m != 0) return;
  const float2* gy = xb + kRowBuffer<N>;
  const float2* vx = gy + kRowBuffer<N>;
  const float2* vy = vx + kRowBuffer<N>;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const float2 y = gy[lane + 64 * e], cx = vx[lane + 64 * e], cy = vy[lane + 64 * e];
    v[e] = make_float2(-(v[e].x * cx.x + y.x * cy.x), -(v[e].y * cx.y + y.y * cy.y));
  }
  reg_fft<H, E, RS, false, R>(v, tw, xb + t, j);
  wave_lds_sync();
#pragma unroll
  for (int e = 0; e < E; ++e) xb[fft_pad(j) * RS + fft_pad(e * L) * RS + t] = v[e];
  wave_lds_sync();
  constexpr int OUT = NR * H, POUT = (OUT + 63) / 64;
#pragma unroll
  for (int k = 0; k < POUT; ++k) {
    const int e = lane + 64 * k;
    if (OUT % 64 == 0 || e < OUT) {
      const int r = row_of(e), kk = word_of(e);
      pout[tix<N>(i0 + r, kk)] = r2c_pair(xb[fft_pad(kk) * RS + r], xb[fft_pad((H - kk) & (H - 1)) * RS + r], kk, q.tw[kk]);
    }
  }
}

template <int N, int NR, int R>
__global__ __launch_bounds__(1024) void ns_rows(NsParams q, const float2* __restrict__ g,
                                                float2* __restrict__ pout) {
  extern __shared__ float4 ns_smem[];
  const size_t inst = q.slots ? static_cast<size_t>(q.slots[blockIdx.y]) : blockIdx.y;
  const size_t gstride = static_cast<size_t>(N) * (N / 2);
  rows_tile<N, NR, R>(reinterpret_cast<float2*>(ns_smem), q, g + inst * 4 * gstride, pout + inst * gstride,
                      xcd_tile(blockIdx.x, gridDim.x) * (blockDim.x / 256) * NR, threadIdx.x);
}

// The row kernel of launches that fill the chip: four wavefronts take 4 RS
// rows, each wavefront its RS rows of the four spectra one after the other
// (the next spectrum's words on their way meanwhile), so every wavefront
// works to the end and the workgroup's global pieces are 4 RS rows x kTw
// words long.  The words come in through one of two staging buffers; a
// wavefront's part of a buffer then serves as its exchange buffer.
template <int N, int R>
__device__ __forceinline__ void rows_seq_tile(float2* smem, const NsParams& q, const float2* __restrict__ g,
                                              float2* __restrict__ pout, int i0, int tid) {
  using S = RowShape<N>;
  constexpr int H = S::H, E = S::E, L = S::L, RS = S::RS, RB = 4 * RS, HH = H / 2, TW = kTw<N>;
  constexpr int PER = RB * HH / 256, OUT = RB * H / 256, BUF = 4 * kRowBuffer<N>;
  static_assert(RB * HH % 256 == 0 && HH % TW == 0, "whole chunks");
  const int wave = tid / 64, lane = tid % 64;
  auto row_of = [](int e) { return (e / TW) % RB; };
  auto word_of = [](int e) { return (e / (TW * RB)) * TW + e % TW; };
  // word k of row r of the block
  auto slot = [](int r, int k) { return (r / RS) * kRowBuffer<N> + fft_pad(k) * RS + r % RS; };
  const size_t gstride = static_cast<size_t>(N) * H;
  float2 a[PER], b[PER], mid = make_float2(0.f, 0.f);
  auto load = [&](int m) {
    const float2* gm = g + m * gstride;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = tid + 256 * k, r = row_of(e), kk = word_of(e);
      a[k] = gm[tix<N>(i0 + r, kk)];
      b[k] = gm[tix<N>(i0 + r, (H - kk) & (H - 1))];
    }
    if (tid < RB) mid = gm[tix<N>(i0 + tid, HH)];
  };
  load(0);
  const float2 tmid = q.tw[HH];
  const int j = lane / RS, t = lane % RS;
  RegTwiddles<H, E, R> tw;
  tw.template load<2>(q.tw, j);
  // advection = -(grad_x * vx + grad_y * vy)  (spectral/equations.py:170)
  float2 v[E], prod[E];
#pragma unroll
  for (int step = 0; step < 4; ++step) {
    constexpr int order[4] = {0, 2, 1, 3};  // grad_x, vx, grad_y, vy
    float2* buf = smem + (step & 1) * BUF;
    const float2* tab = q.tw;  // the combine's twiddles are read again for each spectrum: registers are scarcer
    asm volatile("" : "+s"(tab));
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = tid + 256 * k, r = row_of(e), kk = word_of(e);
      buf[slot(r, kk)] = c2r_combine(a[k], b[k], kk, as_global(tab)[kk]);
      if (kk != 0) buf[slot(r, H - kk)] = c2r_combine(b[k], a[k], H - kk, as_global(tab)[H - kk]);
    }
    if (tid < RB) buf[slot(tid, HH)] = c2r_combine(mid, mid, HH, tmid);
    if (step < 3) load(order[step < 3 ? step + 1 : 3]);
    // also orders the rewriting of a buffer after every wavefront's last
    // exchange in it, two steps before
    __syncthreads();
    float2* xb = buf + wave * kRowBuffer<N> + t;
    float2 f[E];
#pragma unroll
    for (int e = 0; e < E; ++e) f[e] = xb[(fft_pad(j) + fft_pad(e * L)) * RS];
    reg_fft<H, E, RS, true, R>(f, tw, xb, j);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if (step == 0) prod[e] = f[e];
      else if (step == 1) prod[e] = make_float2(prod[e].x * f[e].x, prod[e].y * f[e].y);
      else if (step == 2) v[e] = f[e];
      else v[e] = make_float2(-(prod[e].x + v[e].x * f[e].x), -(prod[e].y + v[e].y * f[e].y));
    }
  }
  float2* xw = smem + BUF + wave * kRowBuffer<N> + t;
  reg_fft<H, E, RS, false, R>(v, tw, xw, j);
  wave_lds_sync();
#pragma unroll
  for (int e = 0; e < E; ++e) xw[(fft_pad(j) + fft_pad(e * L)) * RS] = v[e];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < OUT; ++k) {
    const int e = tid + 256 * k, r = row_of(e), kk = word_of(e);
    const float2* z = smem + BUF;
    pout[tix<N>(i0 + r, kk)] = r2c_pair(z[slot(r, kk)], z[slot(r, (H - kk) & (H - 1))], kk, q.tw[kk]);
  }
}
template <int N>
constexpr int row_seq_lds() {
  return 2 * 4 * kRowBuffer<N> * static_cast<int>(sizeof(float2));
}

template <int N, int R>
__global__ __launch_bounds__(256, 4) void ns_rows_seq(NsParams q, const float2* __restrict__ g,
                                                      float2* __restrict__ pout) {
  extern __shared__ float4 ns_smem[];
  const size_t inst = q.slots ? static_cast<size_t>(q.slots[blockIdx.y]) : blockIdx.y;
  const size_t gstride = static_cast<size_t>(N) * (N / 2);
  rows_seq_tile<N, R>(reinterpret_cast<float2*>(ns_smem), q, g + inst * 4 * gstride, pout + inst * gstride,
                      xcd_tile(blockIdx.x, gridDim.x) * 4 * RowShape<N>::RS, threadIdx.x);
}

// External rfft2 layout <-> internal state layout of one instance per
// blockIdx.y (slots[blockIdx.y] when given); one word per thread, walked in
// the internal order (contiguous internal side).
template <int N, bool TO_INTERNAL>
__global__ __launch_bounds__(kThreads) void ns_state_convert(const float2* __restrict__ src,
                                                             float2* __restrict__ dst,
                                                             const int* __restrict__ slots) {
  constexpr int H = N / 2, H1 = H + 1, TOT = N * H1;
  const int t = blockIdx.x * kThreads + threadIdx.x;
  if (t >= TOT) return;
  const size_t inst = slots ? static_cast<size_t>(slots[blockIdx.y]) : blockIdx.y;
  int p, c;
  if (t < N * H) {
    constexpr int TW = kTw<N>;
    const int tile = t / (N * TW), r = t % (N * TW);
    p = r / TW;
    c = tile * TW + r % TW;
  } else {
    p = t - N * H;
    c = H;
  }
  const size_t base = inst * TOT;
  if (TO_INTERNAL)
    dst[base + t] = src[base + static_cast<size_t>(p) * H1 + c];
  else
    dst[base + static_cast<size_t>(p) * H1 + c] = src[base + t];
}

// 2/3 rule mask (spectral/utils.py:128-134).
__device__ __forceinline__ float ns_filter(const NsParams& q, int p, int c) {
  if (!q.smooth) return 1.0f;
  const bool row = (p < q.filt_row_lo) || (p >= q.filt_row_hi);
  return (row && c < q.filt_cols) ? 1.0f : 0.0f;
}

// One wavefront's columns from c0 of the forward column pass: P's columns ->
// the RK/CN update of (u, h) in the internal state layout (MODE 1), or the
// update followed by the next stage's inverse work on the new columns (MODE 2);
// all pointers already point at the instance.
template <int N, int MODE, int R>
__device__ __forceinline__ void cols_forward_tile(const ColLds<N>& lds, const NsParams& q,
                                                  const float2* __restrict__ pin, const float2* u_in,
                                                  float2* u_out, float2* h, float2* __restrict__ g,
                                                  int c0, int width, int lane) {
  using S = ColShape<N>;
  constexpr int E = S::E, L = S::L, T = S::T, H = N / 2;
  constexpr int ES = L * kTw<N>;  // words between a lane's elements, in P, G, u and h
  const ColLane<N> ln(c0, width, lane);
  const int at0 = tix<N>(ln.j, ln.c);  // the lane's element 0 (u and h: six = tix for c < N/2)
  // Every global load up front, in the order of use: P and the twiddles,
  // then the state (each element is read and written by its owner only, so
  // reading u and h before the transform is safe also when u_in == u_out).
  float2 v[E];
  const float2* pl = pin + at0;
#pragma unroll
  for (int e = 0; e < E; ++e) v[e] = pl[e * ES];
  RegTwiddles<N, E, R> tw;
  tw.template load<1>(q.tw, ln.j);
  float2 uo[E], ho[E];
  const float2* ul = u_in + at0;
  const float2* hl = h + at0;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    uo[e] = ul[e * ES];
    ho[e] = q.read_h ? hl[e * ES] : make_float2(0.f, 0.f);
  }
  const float ky = q.ky[ln.c];
  if (ln.c == 0 && ln.own) {  // (u, h) of the Nyquist column, parked in LDS
    const float2* uh = u_in + six<N>(ln.j, H);
    const float2* hh = h + six<N>(ln.j, H);
#pragma unroll
    for (int e = 0; e < E; ++e) {
      lds.wn[ln.j + e * L] = uh[e * L];
      if (q.read_h) lds.w0[ln.j + e * L] = hh[e * L];
    }
  }
  float2* x = lds.x;
  reg_fft<N, E, T, false, R>(v, tw, x + ln.t, ln.j);

  // h = F + beta h;  u = (u + g h + mu L u) / (1 - mu L), with the old
  // (u, h) at wavenumber (kx, ky) given; returns u and leaves h in fv.
  auto update = [&](float kxp, float kyc, float2& fv, float2 u0, float2 h0) -> float2 {
    if (q.read_h) fv = make_float2(fv.x + q.beta * h0.x, fv.y + q.beta * h0.y);
    const float lap = q.neg_four_pi_sq * (kxp * kxp + kyc * kyc);
    const float Lc = q.nu * lap - q.drag;
    const float2 lu = make_float2(Lc * u0.x, Lc * u0.y);
    const float2 xx = make_float2((u0.x + q.g * fv.x) + q.mu * lu.x, (u0.y + q.g * fv.y) + q.mu * lu.y);
    const float inv = 1.0f / (1.0f - q.mu * Lc);
    return make_float2(inv * xx.x, inv * xx.y);
  };
  const float jf = recompute(static_cast<float>(ln.j));

  if (c0 == 0) {
    // column 0 of tile 0 carries the DC (A) and Nyquist (B) columns:
    // A = (Y(p) + conj Y(-p))/2, B = (Y(p) - conj Y(-p))/(2i)
    float2* xt = x + ln.t;
    wave_lds_sync();
#pragma unroll
    for (int e = 0; e < E; ++e) xt[fft_pad(ln.j + e * L) * T] = v[e];
    wave_lds_sync();
    if (ln.c == 0 && ln.own) {
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const float2 ym = cconj(xt[fft_pad((N - ln.j - e * L) & (N - 1)) * T]);
        v[e] = make_float2(0.5f * (v[e].x + ym.x), 0.5f * (v[e].y + ym.y));
      }
      bool forced = false;  // entries in the Nyquist column
      for (int t = 0; t < q.n_force; ++t) forced |= q.force_idx[2 * t + 1] == H;
      // F at (p, H), from the transform left in the exchange buffer
      auto nyquist = [&](int p) -> float2 {
        const float2 d = csub(xt[fft_pad(p) * T], cconj(xt[fft_pad((N - p) & (N - 1)) * T]));
        const float m = ns_filter(q, p, H);
        float2 f = make_float2((0.5f * d.y) * m, (-0.5f * d.x) * m);
        if (forced)
          for (int t = 0; t < q.n_force; ++t)
            if (q.force_idx[2 * t] == p && q.force_idx[2 * t + 1] == H) f = cadd(f, q.force_val[t]);
        return f;
      };
      const float kyh = q.ky[H];
      float2* hn = h + six<N>(ln.j, H);
      float2* un = u_out + six<N>(ln.j, H);
#pragma unroll
      for (int e = 0; e < E; ++e) {
        if (e % 2 == 0) __builtin_amdgcn_sched_barrier(0);
        const int p = ln.j + e * L;
        const float2 h0 = q.read_h ? lds.w0[p] : make_float2(0.f, 0.f);
        float2 f = nyquist(p);
        const float2 w = update(lane_kx<N>(q, jf, e), kyh, f, lds.wn[p], h0);
        hn[e * L] = f;
        un[e * L] = w;
        if constexpr (MODE == 2) lds.wn[p] = w;
      }
    }
  }
  // F: the filter, then the sparse, time-constant forcing curl entries (the
  // list is the same for every lane; row p belongs to lane p % L, element p / L)
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const float m = ns_filter(q, ln.j + e * L, ln.c);
    v[e] = make_float2(v[e].x * m, v[e].y * m);
  }
  for (int t = 0; t < q.n_force; ++t) {
    const int fp = q.force_idx[2 * t], fc = q.force_idx[2 * t + 1], se = fp / L;
    if (fc == ln.c && fp % L == ln.j) {
      const float2 f = q.force_val[t];
#pragma unroll
      for (int e = 0; e < E; ++e)
        if (e == se) v[e] = cadd(v[e], f);
    }
  }
#pragma unroll
  for (int e = 0; e < E; ++e) {
    if (e % 2 == 0) __builtin_amdgcn_sched_barrier(0);  // two elements' updates in registers at a time
    uo[e] = update(lane_kx<N>(q, jf, e), ky, v[e], uo[e], ho[e]);
  }
  if (ln.own) {
    float2* hs = h + at0;
    float2* us = u_out + at0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      hs[e * ES] = v[e];
      us[e * ES] = uo[e];
    }
  }
  if constexpr (MODE == 2) {
    if (c0 == 0) {
      if (ln.c == 0 && ln.own) {
#pragma unroll
        for (int e = 0; e < E; ++e) lds.w0[ln.j + e * L] = uo[e];
      }
      wave_lds_sync();
    }
    cols_inverse_body<N, R>(uo, tw, ln, lds, q, g);
  }
}

template <int N, int MODE, int R>
__global__ __launch_bounds__(1024 / ColShape<N>::E * 8, (NsColOcc<N>::value)) void ns_cols_forward(
    NsParams q, const float2* __restrict__ pin, const float2* u_in, float2* u_out, float2* h,
    float2* __restrict__ g, int width) {
  extern __shared__ float4 ns_smem[];
  const int wave = threadIdx.x / 64;
  const ColLds<N> lds(reinterpret_cast<char*>(ns_smem), blockDim.x / 64, wave);
  const int c0 = xcd_tile(blockIdx.x, gridDim.x) * width + wave * ColShape<N>::T;
  const size_t inst = q.slots ? static_cast<size_t>(q.slots[blockIdx.y]) : blockIdx.y;
  const size_t ext = static_cast<size_t>(N) * (N / 2 + 1);
  cols_forward_tile<N, MODE, R>(lds, q, pin + inst * static_cast<size_t>(N) * (N / 2),
                                u_in + inst * ext, u_out + inst * ext, h + inst * ext,
                                g ? g + inst * 4 * static_cast<size_t>(N) * (N / 2) : nullptr, c0, width,
                                threadIdx.x % 64);
}

// ---- staged column kernels: launches too small to fill the chip -----------
// A workgroup of 256 threads per tile of W columns, the tile in LDS around
// every pass: a lone 512-word column keeps four wavefronts busy, where a
// register transform is one wavefront's serial work (1 x 256^2
// update-and-inverse 6.1 us against 12.7; at 64 x 256^2, where wavefronts
// abound, 35 against 30, at 16 x 512^2 39 against 30).
constexpr int kForceRegs = 4;  // forcing-curl entries kept in registers
// Widest tile the staged kernels serve; wider ones are for large launches.
template <int N>
constexpr int kStagedMaxW = N == 32 ? 16 : N == 64 ? 8 : N == 128 ? 4 : N == 256 ? 2 : 1;

// Spectrum m in {0: d_x w, 1: d_y w, 2: v_x, 3: v_y} at (p, c).
__device__ __forceinline__ float2 ns_spectrum(int m, const NsMult& k, float2 w) {
  switch (m) {
    case 0: return mul_i(k.ax, w);
    case 1: return mul_i(k.ay, w);
    case 2: return mul_i(k.ay, make_float2(k.psi * w.x, k.psi * w.y));
    default: return mul_i(-k.ax, make_float2(k.psi * w.x, k.psi * w.y));
  }
}

// Spectra built and inverse-transformed per round of the inverse column
// work: a round's spectra sit side by side as NSP * W columns of one LDS
// tile, so one set of FFT passes (and barriers) serves all of them.  NSP is
// the largest of 4, 2, 1 whose round fits kNsRoundWords complex words.
constexpr int kNsMaxSpectraPerRound = 4;
constexpr int kNsRoundWords = 2048;
template <int N, int W>
struct NsRound {
  static constexpr int value = (kNsMaxSpectraPerRound >= 4 && 4 * N * W <= kNsRoundWords) ? 4
                               : (kNsMaxSpectraPerRound >= 2 && 2 * N * W <= kNsRoundWords) ? 2
                                                                                            : 1;
};

template <int N, int W>
struct StagedCols {
  float2 buf[N * W * NsRound<N, W>::value];  // work tile [p][c] (inverse rounds: [p][spectrum][c])
  float2 w0[N];       // tile 0: vorticity column 0
  float2 wn[N];       // tile 0: vorticity column N/2
  float2 tw[N];
  float kx[N];        // fftfreq
  float ky[N / 2 + 1];  // rfftfreq
};

// Elements of a column tile are owned by threads as e = tid + k * kThreads;
// each thread keeps its vorticity values in registers across the four spectra
// (only tile 0's DC/Nyquist columns, which pair rows p and -p, also go through
// LDS).
template <int N, int W>
struct WTile {
  static constexpr int PER = (N * W + kThreads - 1) / kThreads;
  float2 w[PER];
};

// Build spectrum m of the tile into sm.buf (scaled by 1/n^2), symmetrising and
// packing the DC/Nyquist pair into local column 0 of tile 0.  psi[k] is
// -1/laplacian at this thread's element k (columns other than 0; one
// division per element for all four spectra); 2 pi kx, 2 pi ky come from
// the LDS wavenumber tables.
template <int N, int W, int NSP = 1>
__device__ __forceinline__ void staged_spectrum(StagedCols<N, W>& sm, const WTile<N, W>& wt,
                                               const float (&psi)[WTile<N, W>::PER],
                                               const NsParams& q, int m, int slot, int c0, int tid) {
  constexpr int H = N / 2;
#pragma unroll
  for (int k = 0; k < WTile<N, W>::PER; ++k) {
    const int e = tid + k * kThreads;
    if (e >= N * W) break;
    const int p = e / W, c = e % W, cg = c0 + c;
    float2 out;
    if (cg != 0) {
      NsMult mk;
      mk.ax = q.two_pi * sm.kx[p];
      mk.ay = q.two_pi * sm.ky[cg];
      mk.psi = psi[k];
      out = ns_spectrum(m, mk, wt.w[k]);
    } else {
      const int pm = (N - p) & (N - 1);
      const float2 a0 = ns_spectrum(m, ns_mult(q, sm.kx[p], sm.ky[0], p == 0), sm.w0[p]);
      const float2 b0 = ns_spectrum(m, ns_mult(q, sm.kx[pm], sm.ky[0], pm == 0), sm.w0[pm]);
      const float2 ah = ns_spectrum(m, ns_mult(q, sm.kx[p], sm.ky[H], false), sm.wn[p]);
      const float2 bh = ns_spectrum(m, ns_mult(q, sm.kx[pm], sm.ky[H], false), sm.wn[pm]);
      const float2 s0 = make_float2(0.5f * (a0.x + b0.x), 0.5f * (a0.y - b0.y));
      const float2 sh = make_float2(0.5f * (ah.x + bh.x), 0.5f * (ah.y - bh.y));
      out = make_float2(s0.x - sh.y, s0.y + sh.x);  // s0 + i sh
    }
    sm.buf[p * (NSP * W) + slot * W + c] = make_float2(out.x * q.inv_nn, out.y * q.inv_nn);
  }
}

// Inverse column transforms of the tile -> G[0..4).  sm.w0 / sm.wn must be
// visible (barrier) before the call.
template <int N, int W, int R>
__device__ __forceinline__ void staged_inverse_body(StagedCols<N, W>& sm, const WTile<N, W>& wt,
                                                  const NsParams& q, float2* __restrict__ g,
                                                  int c0, int tid) {
  constexpr int H = N / 2;
  constexpr int PER = WTile<N, W>::PER;
  const size_t gstride = static_cast<size_t>(N) * H;
  float psi[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e = tid + k * kThreads;
    const int p = (e < N * W ? e : N * W - 1) / W, cg = c0 + e % W;
    psi[k] = cg != 0 ? ns_mult(q, sm.kx[p], sm.ky[cg], false).psi : 0.f;
  }
  constexpr int NSP = NsRound<N, W>::value;
#pragma unroll 1
  for (int m0 = 0; m0 < 4; m0 += NSP) {
#pragma unroll
    for (int j = 0; j < NSP; ++j)
      staged_spectrum<N, W, NSP>(sm, wt, psi, q, m0 + j, j, c0, tid);
    __syncthreads();
    lds_fft<N, NSP * W, kThreads, NSP * W, 1, true, true, R>(sm.buf, sm.tw, tid);
#pragma unroll
    for (int j = 0; j < NSP; ++j) {
      float2* gm = g + (m0 + j) * gstride;
      float2 o[PER];
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int e = tid + k * kThreads;
        if ((N * W) % kThreads == 0 || e < N * W) o[k] = sm.buf[(e / W) * (NSP * W) + j * W + e % W];
      }
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int e = tid + k * kThreads;
        if ((N * W) % kThreads == 0 || e < N * W) gm[tix<N>(e / W, c0 + e % W)] = o[k];
      }
    }
    __syncthreads();
  }
}

// The state tile into registers; tile 0 also stages columns 0 and N/2 in LDS.
template <int N, int W>
__device__ __forceinline__ void staged_load(StagedCols<N, W>& sm, WTile<N, W>& wt, const NsParams& q,
                                            const float2* __restrict__ w, int c0, int tid) {
#pragma unroll
  for (int k = 0; k < WTile<N, W>::PER; ++k) {
    const int e = tid + k * kThreads;
    if (e >= N * W) break;
    const int p = e / W, c = e % W;
    wt.w[k] = w[six<N>(p, c0 + c)];
  }
  if (c0 == 0) {
    constexpr int PN = (N + kThreads - 1) / kThreads;
    float2 a[PN], b[PN];
#pragma unroll
    for (int k = 0; k < PN; ++k) {
      const int p = tid + k * kThreads;
      if (N % kThreads == 0 || p < N) {
        a[k] = w[six<N>(p, 0)];
        b[k] = w[six<N>(p, N / 2)];
      }
    }
#pragma unroll
    for (int k = 0; k < PN; ++k) {
      const int p = tid + k * kThreads;
      if (N % kThreads == 0 || p < N) {
        sm.w0[p] = a[k];
        sm.wn[p] = b[k];
      }
    }
  }
}

// Wavenumber tables staged through registers (load() issues the global
// loads, store() writes LDS), like TwiddleStage.
template <int N>
struct WavenumberStage {
  static constexpr int PX = (N + kThreads - 1) / kThreads;
  static constexpr int PY = (N / 2 + 1 + kThreads - 1) / kThreads;
  float x[PX], y[PY];
  __device__ __forceinline__ void load(const NsParams& q, int tid) {
#pragma unroll
    for (int k = 0; k < PX; ++k) {
      const int i = tid + k * kThreads;
      x[k] = q.kx[N % kThreads == 0 || i < N ? i : N - 1];
    }
#pragma unroll
    for (int k = 0; k < PY; ++k) {
      const int i = tid + k * kThreads;
      y[k] = q.ky[i <= N / 2 ? i : N / 2];
    }
  }
  __device__ __forceinline__ void store(float* kx, float* ky, int tid) const {
#pragma unroll
    for (int k = 0; k < PX; ++k) {
      const int i = tid + k * kThreads;
      if (N % kThreads == 0 || i < N) kx[i] = x[k];
    }
#pragma unroll
    for (int k = 0; k < PY; ++k) {
      const int i = tid + k * kThreads;
      if (i <= N / 2) ky[i] = y[k];
    }
  }
};


// Minimum waves per SIMD asked of the column kernels: 5 for the 512-point
// tiles of one or two columns, the most their LDS (inverse rounds of two or
// four spectra) allows; other shapes keep the compiler's choice (wider
// tiles would spill).
template <int N, int W>
struct StagedWaves {
  static constexpr int value = (N == 512 && W <= 2) ? 5 : 1;
};

template <int N, int W, int R>
__global__ __launch_bounds__(kThreads, (StagedWaves<N, W>::value)) void ns_cols_inverse_staged(
    NsParams q, const float2* __restrict__ w, float2* __restrict__ g) {
  __shared__ StagedCols<N, W> sm;
  const int tid = threadIdx.x;
  const int c0 = xcd_tile(blockIdx.x, gridDim.x) * W;
  const size_t inst = q.slots ? static_cast<size_t>(q.slots[blockIdx.y]) : blockIdx.y;
  WTile<N, W> wt;
  TwiddleStage<N, 1, kThreads> tw;
  WavenumberStage<N> wn;
  tw.load(q.tw, tid);
  wn.load(q, tid);
  staged_load<N, W>(sm, wt, q, w + inst * static_cast<size_t>(N) * (N / 2 + 1), c0, tid);
  tw.store(sm.tw, tid);
  wn.store(sm.kx, sm.ky, tid);
  __syncthreads();
  staged_inverse_body<N, W, R>(sm, wt, q, g + inst * 4 * static_cast<size_t>(N) * (N / 2), c0, tid);
}

// As cols_forward_tile: the update (MODE 1), or the update and the next
// stage's inverse work on the same tile (MODE 2).
template <int N, int W, int MODE, int R>
__device__ __forceinline__ void staged_forward_tile(StagedCols<N, W>& sm, const NsParams& q,
                                                  const float2* __restrict__ pin, const float2* u_in,
                                                  float2* u_out, float2* h, float2* __restrict__ g,
                                                  int c0, int tid) {
  constexpr int H = N / 2;
  constexpr int PER = (N * W + kThreads - 1) / kThreads;

  // Every global load of the kernel's first half is issued up front: the
  // tile of P, the state (u, h) at this thread's elements for the update
  // (each element is read and written by its owner only, so reading u and h
  // before the transform is safe also when u_in == u_out), the twiddles.
  // Issue order matters: a wait for a load also waits for every load issued
  // before it, so the tables (needed first) go first and (u, h) (needed
  // after the transform) last.
  TwiddleStage<N, 1, kThreads> tws;
  WavenumberStage<N> wns;
  tws.load(q.tw, tid);
  wns.load(q, tid);
  float2 pv[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e = tid + k * kThreads;
    if ((N * W) % kThreads == 0 || e < N * W) pv[k] = pin[tix<N>(e / W, c0 + e % W)];
  }
  float2 u_pre[PER], h_pre[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e = tid + k * kThreads;
    if ((N * W) % kThreads == 0 || e < N * W) {
      const int idx = six<N>(e / W, c0 + e % W);
      u_pre[k] = u_in[idx];
      h_pre[k] = q.read_h ? h[idx] : make_float2(0.f, 0.f);
    }
  }
  tws.store(sm.tw, tid);
  wns.store(sm.kx, sm.ky, tid);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e = tid + k * kThreads;
    if ((N * W) % kThreads == 0 || e < N * W) sm.buf[e] = pv[k];
  }
  __syncthreads();
  lds_fft<N, W, kThreads, W, 1, true, false, R>(sm.buf, sm.tw, tid);

  // h = F + beta h;  u = (u + g h + mu L u) / (1 - mu L), with the old
  // (u, h) at (p, cg) given.
  auto update_with = [&](int p, int cg, float2 fv, float2 uo, float2 ho) -> float2 {
    const int idx = six<N>(p, cg);
    float2 hv = fv;
    if (q.read_h) hv = make_float2(fv.x + q.beta * ho.x, fv.y + q.beta * ho.y);
    h[idx] = hv;
    const float kx = sm.kx[p], ky = sm.ky[cg];
    const float lap = q.neg_four_pi_sq * (kx * kx + ky * ky);
    const float L = q.nu * lap - q.drag;
    const float2 lu = make_float2(L * uo.x, L * uo.y);
    const float2 x = make_float2((uo.x + q.g * hv.x) + q.mu * lu.x, (uo.y + q.g * hv.y) + q.mu * lu.y);
    const float inv = 1.0f / (1.0f - q.mu * L);
    const float2 un = make_float2(inv * x.x, inv * x.y);
    u_out[idx] = un;
    return un;
  };
  // Column N/2 (tile 0 only): (u, h) read here.
  auto update_nyquist = [&](int p, float2 fv) -> float2 {
    const int idx = six<N>(p, H);
    const float2 ho = q.read_h ? h[idx] : make_float2(0.f, 0.f);
    return update_with(p, H, fv, u_in[idx], ho);
  };

  // The forcing-curl entries, read once (the element loop's stores could
  // alias them as far as the compiler knows, so it would reload them for
  // every element); longer lists are read from memory in the loop.
  int fpr[kForceRegs], fcr[kForceRegs];
  float2 fvr[kForceRegs];
#pragma unroll
  for (int t = 0; t < kForceRegs; ++t) {
    const int tt = t < q.n_force ? t : 0;
    fpr[t] = q.n_force > 0 ? q.force_idx[2 * tt] : -1;
    fcr[t] = q.n_force > 0 ? q.force_idx[2 * tt + 1] : -1;
    fvr[t] = q.n_force > 0 ? q.force_val[tt] : make_float2(0.f, 0.f);
  }

  // Per element: F at (p, cg) (filter, then the sparse, time-constant forcing
  // curl entries), then the update; tile 0 also
  // handles column N/2.  One pass, so no array of F values stays live.
  [[maybe_unused]] WTile<N, W> wt;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e = tid + k * kThreads;
    if (e < N * W) {
      const int p = e / W, c = e % W, cg = c0 + c;
      const float2 y = sm.buf[e];
      float2 f, fh = make_float2(0.f, 0.f);
      if (cg == 0) {
        const float2 ym = cconj(sm.buf[((N - p) & (N - 1)) * W]);
        const float2 a = make_float2(0.5f * (y.x + ym.x), 0.5f * (y.y + ym.y));
        const float2 d = csub(y, ym);
        const float2 b = make_float2(0.5f * d.y, -0.5f * d.x);
        const float m0 = ns_filter(q, p, 0), mh = ns_filter(q, p, H);
        f = make_float2(a.x * m0, a.y * m0);
        fh = make_float2(b.x * mh, b.y * mh);
      } else {
        const float m = ns_filter(q, p, cg);
        f = make_float2(y.x * m, y.y * m);
      }
      if (q.n_force <= kForceRegs) {
#pragma unroll
        for (int t = 0; t < kForceRegs; ++t) {
          if (t < q.n_force && fpr[t] == p && fcr[t] == cg) f = cadd(f, fvr[t]);
          if (t < q.n_force && cg == 0 && fpr[t] == p && fcr[t] == H) fh = cadd(fh, fvr[t]);
        }
      } else {
        for (int t = 0; t < q.n_force; ++t) {
          const int fp = q.force_idx[2 * t], fc = q.force_idx[2 * t + 1];
          if (fp == p && fc == cg) f = cadd(f, q.force_val[t]);
          if (cg == 0 && fp == p && fc == H) fh = cadd(fh, q.force_val[t]);
        }
      }
      const float2 un = update_with(p, cg, f, u_pre[k], h_pre[k]);
      if constexpr (MODE == 2) {
        wt.w[k] = un;
        if (cg == 0) {
          sm.w0[p] = un;
          sm.wn[p] = update_nyquist(p, fh);
        }
      } else {
        if (cg == 0) update_nyquist(p, fh);
      }
    }
  }
  if constexpr (MODE == 2) {
    __syncthreads();  // sm.buf read by all; sm.w0 / sm.wn written
    staged_inverse_body<N, W, R>(sm, wt, q, g, c0, tid);
  }
}


template <int N, int W, int MODE, int R>
__global__ __launch_bounds__(kThreads, (StagedWaves<N, W>::value)) void ns_cols_forward_staged(NsParams q, const float2* __restrict__ pin,
                                                            const float2* u_in, float2* u_out,
                                                            float2* h, float2* __restrict__ g) {
  __shared__ StagedCols<N, W> sm;
  const size_t inst = q.slots ? static_cast<size_t>(q.slots[blockIdx.y]) : blockIdx.y;
  const size_t ext = static_cast<size_t>(N) * (N / 2 + 1);
  staged_forward_tile<N, W, MODE, R>(sm, q, pin + inst * static_cast<size_t>(N) * (N / 2),
                                   u_in + inst * ext, u_out + inst * ext, h + inst * ext,
                                   g ? g + inst * 4 * static_cast<size_t>(N) * (N / 2) : nullptr,
                                   xcd_tile(blockIdx.x, gridDim.x) * W, threadIdx.x);
}


// ---- column kernels of the transforms and the explicit terms -----------------
// Their external side (rows of n/2 + 1 words) is read and written column by
// column, so W columns share a workgroup and its cache lines.

// Columns of P -> out in the external layout: the filter and the forcing curl
// entries of explicit_terms (rfft2 passes neither).  P in the step's column
// tiles (TILED) or row by row.
template <int N, int W, bool TILED>
__global__ __launch_bounds__(kThreads) void ns_cols_out(NsParams q, const float2* __restrict__ pin,
                                                        float2* __restrict__ out) {
  constexpr int H = N / 2, H1 = H + 1, PER = (N * W + kThreads - 1) / kThreads;
  __shared__ float2 buf[N * W];
  __shared__ float2 tw[N];
  const int tid = threadIdx.x, c0 = xcd_tile(blockIdx.x, gridDim.x) * W;
  const size_t inst = q.slots ? static_cast<size_t>(q.slots[blockIdx.y]) : blockIdx.y;
  pin += inst * static_cast<size_t>(N) * H;
  out += inst * static_cast<size_t>(N) * H1;
  TwiddleStage<N, 1, kThreads> tws;
  tws.load(q.tw, tid);
  staged<N * W, PER, kThreads>(
      tid, [&](int e) { return pin[TILED ? tix<N>(e / W, c0 + e % W) : (e / W) * H + c0 + e % W]; },
      [&](int e, float2 x) { buf[e] = x; });
  tws.store(tw, tid);
  __syncthreads();
  lds_fft<N, W, kThreads, W, 1, true, false, 8>(buf, tw, tid);
  // F at (p, c) from its transform: the filter, then the forcing entries
  auto put = [&](int p, int c, float2 f) {
    const float m = ns_filter(q, p, c);
    f = make_float2(f.x * m, f.y * m);
    for (int t = 0; t < q.n_force; ++t)
      if (q.force_idx[2 * t] == p && q.force_idx[2 * t + 1] == c) f = cadd(f, q.force_val[t]);
    out[p * H1 + c] = f;
  };
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e = tid + k * kThreads;
    if (e >= N * W) break;
    const int p = e / W, c = c0 + e % W;
    const float2 y = buf[e];
    if (c != 0) {
      put(p, c, y);
    } else {  // the DC (A) and Nyquist (B) columns
      const float2 ym = cconj(buf[((N - p) & (N - 1)) * W]);
      const float2 d = csub(y, ym);
      put(p, 0, make_float2(0.5f * (y.x + ym.x), 0.5f * (y.y + ym.y)));
      put(p, H, make_float2(0.5f * d.y, -0.5f * d.x));
    }
  }
}

// Columns of a spectrum in the external layout, scaled by 1/n^2 -> inverse
// transforms, row by row.
template <int N, int W>
__global__ __launch_bounds__(kThreads) void ns_cols_in(NsParams q, const float2* __restrict__ in,
                                                       float2* __restrict__ pout) {
  constexpr int H = N / 2, H1 = H + 1, PER = (N * W + kThreads - 1) / kThreads;
  __shared__ float2 buf[N * W];
  __shared__ float2 tw[N];
  __shared__ float2 w0[N], wn[N];  // tile 0: columns 0 and N/2
  const int tid = threadIdx.x, c0 = xcd_tile(blockIdx.x, gridDim.x) * W;
  const size_t inst = q.slots ? static_cast<size_t>(q.slots[blockIdx.y]) : blockIdx.y;
  in += inst * static_cast<size_t>(N) * H1;
  pout += inst * static_cast<size_t>(N) * H;
  TwiddleStage<N, 1, kThreads> tws;
  tws.load(q.tw, tid);
  staged<N * W, PER, kThreads>(
      tid, [&](int e) { return in[(e / W) * H1 + c0 + e % W]; },
      [&](int e, float2 x) {
        if (c0 + e % W == 0) w0[e / W] = x;
        else buf[e] = make_float2(x.x * q.inv_nn, x.y * q.inv_nn);
      });
  if (c0 == 0)
    for (int p = tid; p < N; p += kThreads) wn[p] = in[p * H1 + H];
  tws.store(tw, tid);
  if (c0 == 0) {
    __syncthreads();
    for (int p = tid; p < N; p += kThreads) {
      const int pm = (N - p) & (N - 1);
      const float2 s0 = make_float2(0.5f * (w0[p].x + w0[pm].x), 0.5f * (w0[p].y - w0[pm].y));
      const float2 sh = make_float2(0.5f * (wn[p].x + wn[pm].x), 0.5f * (wn[p].y - wn[pm].y));
      const float2 s = make_float2(s0.x - sh.y, s0.y + sh.x);  // s0 + i sh
      buf[p * W] = make_float2(s.x * q.inv_nn, s.y * q.inv_nn);
    }
  }
  __syncthreads();
  lds_fft<N, W, kThreads, W, 1, true, true, 8>(buf, tw, tid);
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const int e = tid + k * kThreads;
    if (e < N * W) pout[(e / W) * H + c0 + e % W] = buf[e];
  }
}

// ---- mixed-size group step ---------------------------------------------------
// Every item is 1024 complex words of work whatever its grid size (column
// tiles of W = 1024 / n columns, row blocks of 1024 / n rows; capped by the
// sizes' limits), so workgroups of every size take about the same time.  Tile shapes regroup the same per-column and
// per-row arithmetic: results are bit-identical to the per-size kernels'.
template <int N>
struct NsGroupShape {
  static constexpr int W = (1024 / N < N / 2) ? 1024 / N : N / 2;
  static constexpr bool kSeq = N >= 256;  // rows by rows_seq_tile
  static constexpr int RB = kSeq ? 4 * RowShape<N>::RS : ((1024 / N < N / 4) ? 1024 / N : N / 4);
};

// Threads of a group launch: two wavefronts of columns, or the four of a row
// block.
constexpr int ns_group_threads(int cls) { return cls == 1 ? 256 : 128; }

template <int N, int CLS>
__device__ __forceinline__ void ns_group_tile(const NsGroupDesc& d, int tile, int tid, char* smem) {
  using S = NsGroupShape<N>;
  if constexpr (CLS == 1) {
    if constexpr (S::kSeq)
      rows_seq_tile<N, 8>(reinterpret_cast<float2*>(smem), d.q, d.g, d.pbuf, tile * S::RB, tid);
    else
      rows_tile<N, S::RB, 8>(reinterpret_cast<float2*>(smem), d.q, d.g, d.pbuf, tile * S::RB, tid);
  } else {
    const int wave = tid / 64;
    constexpr int waves = col_waves<N>(S::W);
    if (wave >= waves) return;
    const ColLds<N> lds(smem, waves, wave);
    const int c0 = tile * S::W + wave * ColShape<N>::T;
    if constexpr (CLS == 0)
      cols_inverse_tile<N, 8>(lds, d.q, d.ws, d.g, c0, S::W, tid % 64);
    else
      cols_forward_tile<N, CLS == 2 ? 2 : 1, 8>(lds, d.q, d.pbuf, d.ws, d.ws, d.h, d.g, c0, S::W, tid % 64);
  }
}

// One workgroup per item (the host launches exactly the list's item count):
// the hardware's workgroup dispatch keeps the CUs full, as for the per-size
// kernels, with no loop state held in registers.  Groups with 1024^2
// instances have a build of their own (BIG): its 16 words per lane would
// cost every other size registers.
template <int CLS, bool BIG>
__global__ __launch_bounds__(ns_group_threads(CLS), BIG ? 2 : 4) void ns_group_phase(
    const NsGroupDesc* __restrict__ descs, const NsGroupItem* __restrict__ items,
    const int* __restrict__ n_items, int stage) {
  extern __shared__ float4 ns_group_smem[];
  char* smem = reinterpret_cast<char*>(ns_group_smem);
  const int it = blockIdx.x;
  if (it >= *n_items) return;
  const NsGroupItem w = items[it];
  // the descriptor's pointers are all global memory
  NsGroupDesc d = descs[static_cast<size_t>(w.desc) * JCFD_MAX_RK_STAGES + stage];
  d.ws = as_global(d.ws);
  d.h = as_global(d.h);
  d.g = as_global(d.g);
  d.pbuf = as_global(d.pbuf);
  d.q.kx = as_global(d.q.kx);
  d.q.ky = as_global(d.q.ky);
  d.q.tw = as_global(d.q.tw);
  d.q.force_idx = as_global(d.q.force_idx);
  d.q.force_val = as_global(d.q.force_val);
  const int t = threadIdx.x;
  switch (d.n) {
    case 32: ns_group_tile<32, CLS>(d, w.tile, t, smem); break;
    case 64: ns_group_tile<64, CLS>(d, w.tile, t, smem); break;
    case 128: ns_group_tile<128, CLS>(d, w.tile, t, smem); break;
    case 256: ns_group_tile<256, CLS>(d, w.tile, t, smem); break;
    case 512: ns_group_tile<512, CLS>(d, w.tile, t, smem); break;
    case 1024:
      if constexpr (BIG) ns_group_tile<1024, CLS>(d, w.tile, t, smem);
      break;
    default: break;  // rejected on the host
  }
}

template <int N>
constexpr int ns_group_lds_n(int cls) {
  using S = NsGroupShape<N>;
  return cls == 1 ? (S::kSeq ? row_seq_lds<N>() : row_lds<N>(S::RB)) : col_lds<N>(col_waves<N>(S::W));
}

// dynamic LDS stays within the 64 KiB a launch gets without raising the
// kernel's limit
static_assert(ns_group_lds_n<1024>(0) <= 65536 && ns_group_lds_n<1024>(1) <= 65536 &&
                  ns_group_lds_n<512>(0) <= 65536 && ns_group_lds_n<512>(1) <= 65536 &&
                  ns_group_lds_n<64>(0) <= 65536 && ns_group_lds_n<64>(1) <= 65536,
              "group LDS");

int ns_group_lds(int cls, int max_n) {
  int bytes = 0;
  if (max_n >= 32) bytes = std::max(bytes, ns_group_lds_n<32>(cls));
  if (max_n >= 64) bytes = std::max(bytes, ns_group_lds_n<64>(cls));
  if (max_n >= 128) bytes = std::max(bytes, ns_group_lds_n<128>(cls));
  if (max_n >= 256) bytes = std::max(bytes, ns_group_lds_n<256>(cls));
  if (max_n >= 512) bytes = std::max(bytes, ns_group_lds_n<512>(cls));
  if (max_n >= 1024) bytes = std::max(bytes, ns_group_lds_n<1024>(cls));
  return bytes;
}


template <int N> struct NsTiles;
template <> struct NsTiles<32> { static constexpr int W = 8, RB = 2; };
template <> struct NsTiles<64> { static constexpr int W = 8, RB = 2; };
template <> struct NsTiles<128> { static constexpr int W = 8, RB = 2; };
template <> struct NsTiles<256> { static constexpr int W = 8, RB = 2; };
template <> struct NsTiles<512> { static constexpr int W = 8, RB = 1; };
template <> struct NsTiles<1024> { static constexpr int W = 4, RB = 1; };

template <int N, int R>
void launch_cols_inverse(int w, const NsParams& q, const float2* in, float2* g, int batch, hipStream_t s) {
  const int waves = col_waves<N>(w);
  hipLaunchKernelGGL((ns_cols_inverse<N, R>), dim3(N / 2 / w, batch), dim3(64 * waves), col_lds<N>(waves), s,
                     q, in, g, w);
}
template <int N, int MODE, int R>
void launch_cols_forward(int w, const NsParams& q, const float2* pbuf, const float2* u_in, float2* u_out, float2* h,
                         float2* g, int batch, hipStream_t s) {
  const int waves = col_waves<N>(w);
  hipLaunchKernelGGL((ns_cols_forward<N, MODE, R>), dim3(N / 2 / w, batch), dim3(64 * waves), col_lds<N>(waves), s, q,
                     pbuf, u_in, u_out, h, g, w);
}
template <int N, int RB, int R>
void launch_rows(const NsParams& q, const float2* g, float2* pbuf, int batch, hipStream_t s) {
  constexpr int RS = RowShape<N>::RS, NR = RB < RS ? RB : RS;
  if constexpr (RB == 4 * RS)
    hipLaunchKernelGGL((ns_rows_seq<N, R>), dim3(N / RB, batch), dim3(256), row_seq_lds<N>(), s, q, g, pbuf);
  else
    hipLaunchKernelGGL((ns_rows<N, NR, R>), dim3(N / RB, batch), dim3(256 * row_groups<N>(RB)), row_lds<N>(RB), s, q,
                       g, pbuf);
}

template <int N>
struct NsOps {
  static constexpr int W = NsTiles<N>::W, RB = NsTiles<N>::RB;
  static int rfft2(const NsParams& q, const float* x, float2* out, float2* pbuf, int batch,
                   hipStream_t s) {
    NsParams plain = q;
    plain.smooth = 0;
    plain.n_force = 0;
    hipLaunchKernelGGL((rows_r2c<N, RB>), dim3(N / RB, batch), dim3(kThreads), 0, s, q, x, pbuf);
    hipLaunchKernelGGL((ns_cols_out<N, W, false>), dim3(N / 2 / W, batch), dim3(kThreads), 0, s, plain, pbuf, out);
    return check_hip(hipGetLastError(), "rfft2");
  }
  static int irfft2(const NsParams& q, const float2* in, float* x, float2* pbuf, int batch,
                    hipStream_t s) {
    hipLaunchKernelGGL((ns_cols_in<N, W>), dim3(N / 2 / W, batch), dim3(kThreads), 0, s, q, in, pbuf);
    hipLaunchKernelGGL((rows_c2r<N, RB>), dim3(N / RB, batch), dim3(kThreads), 0, s, q, pbuf, x);
    return check_hip(hipGetLastError(), "irfft2");
  }
  // Forward column transforms of P -> explicit terms F (no update).
  static int explicit_cols(const NsParams& q, const float2* pbuf, float2* out, int batch, hipStream_t s) {
    hipLaunchKernelGGL((ns_cols_out<N, W, true>), dim3(N / 2 / W, batch), dim3(kThreads), 0, s, q, pbuf, out);
    return check_hip(hipGetLastError(), "explicit terms");
  }
};

// ---- tunable step kernels ---------------------------------------------------
// The step's column kernels are built for a menu of tile widths W and its row
// kernel for a menu of rows per workgroup RB, each with both radix schedules;
// NsParams carries a plan's choice (w_cols, rb_rows, radix).  Tile shapes
// regroup the same per-column / per-row arithmetic and never change results.
constexpr int kNsLdsMax = 96 * 1024;

template <int N>
constexpr bool ns_cols_ok(int w) {
  return w <= N / 2 && N * w <= 16 * kThreads && col_lds<N>(col_waves<N>(w)) <= kNsLdsMax;
}
template <int N>
constexpr bool ns_rows_ok(int rb) {
  return rb <= N / 4 && row_groups<N>(rb) <= 4 && row_lds<N>(rb) <= kNsLdsMax;
}

// which: 0 cols-inverse, 1 rows, 2 cols-forward + update + next inverse,
// 3 cols-forward + final update.  JCFD_ERR_UNSUPPORTED off the menu.
template <int N, int T, int R>
int ns_variant(int which, const NsParams& q, const float2* a, const float2* u_in, float2* u_out,
               float2* h, float2* g, int batch, hipStream_t s) {
  if (which == 1) {
    if constexpr (ns_rows_ok<N>(T)) {
      launch_rows<N, T, R>(q, a, g, batch, s);
      return JCFD_OK;
    }
    return JCFD_ERR_UNSUPPORTED;
  }
  if (!ns_cols_ok<N>(T)) return JCFD_ERR_UNSUPPORTED;
  if constexpr (T <= kStagedMaxW<N>) {
    const dim3 grid(N / 2 / T, batch);
    if (which == 0)
      hipLaunchKernelGGL((ns_cols_inverse_staged<N, T, R>), grid, dim3(kThreads), 0, s, q, a, g);
    else if (which == 2)
      hipLaunchKernelGGL((ns_cols_forward_staged<N, T, 2, R>), grid, dim3(kThreads), 0, s, q, a, u_in, u_out, h, g);
    else
      hipLaunchKernelGGL((ns_cols_forward_staged<N, T, 1, R>), grid, dim3(kThreads), 0, s, q, a, u_in, u_out, h, g);
    return JCFD_OK;
  }
  if (which == 0)
    launch_cols_inverse<N, R>(T, q, a, g, batch, s);
  else if (which == 2)
    launch_cols_forward<N, 2, R>(T, q, a, u_in, u_out, h, g, batch, s);
  else
    launch_cols_forward<N, 1, R>(T, q, a, u_in, u_out, h, g, batch, s);
  return JCFD_OK;
}

template <int N, int R>
int ns_tile(int which, int tile, const NsParams& q, const float2* a, const float2* u_in, float2* u_out,
            float2* h, float2* g, int batch, hipStream_t s) {
  switch (tile) {
    case 1: return ns_variant<N, 1, R>(which, q, a, u_in, u_out, h, g, batch, s);
    case 2: return ns_variant<N, 2, R>(which, q, a, u_in, u_out, h, g, batch, s);
    case 4: return ns_variant<N, 4, R>(which, q, a, u_in, u_out, h, g, batch, s);
    case 8: return ns_variant<N, 8, R>(which, q, a, u_in, u_out, h, g, batch, s);
    case 16: return ns_variant<N, 16, R>(which, q, a, u_in, u_out, h, g, batch, s);
    default: return JCFD_ERR_UNSUPPORTED;
  }
}

// One tuned launch.  For rows (which 1) `a` is G and the product spectrum is
// written to g; for the column kernels `a` is the state (0) or P (2, 3).
template <int N>
int ns_launch(int which, const NsParams& q, const float2* a, const float2* u_in, float2* u_out,
              float2* h, float2* g, int batch, hipStream_t s) {
  const int tile = which == 1 ? q.rb_rows : q.w_cols;
  const int rc = q.radix == 4 ? ns_tile<N, 4>(which, tile, q, a, u_in, u_out, h, g, batch, s)
                              : ns_tile<N, 8>(which, tile, q, a, u_in, u_out, h, g, batch, s);
  if (rc) return fail(rc, "spectral tile shape not built for n = " + std::to_string(N));
  return check_hip(hipGetLastError(), "spectral step launch");
}

template <int N>
int ns_step_impl(const NsParams* stages, int nstages, const NsBuffers& b, int batch, hipStream_t s) {
  int rc = ns_launch<N>(0, stages[0], b.u_in, nullptr, nullptr, nullptr, b.g, batch, s);
  for (int k = 0; k < nstages && rc == JCFD_OK; ++k) {
    rc = ns_launch<N>(1, stages[k], b.g, nullptr, nullptr, nullptr, b.pbuf, batch, s);
    if (rc) break;
    const float2* u_src = (k == 0) ? b.u_in : b.u_out;
    rc = ns_launch<N>(k + 1 < nstages ? 2 : 3, stages[k], b.pbuf, u_src, b.u_out, b.h, b.g, batch, s);
  }
  return rc;
}

template <int N>
bool ns_tile_on_menu(int which, int tile) {
  switch (tile) {
    case 1: return which == 1 ? ns_rows_ok<N>(1) : ns_cols_ok<N>(1);
    case 2: return which == 1 ? ns_rows_ok<N>(2) : ns_cols_ok<N>(2);
    case 4: return which == 1 ? ns_rows_ok<N>(4) : ns_cols_ok<N>(4);
    case 8: return which == 1 ? ns_rows_ok<N>(8) : ns_cols_ok<N>(8);
    case 16: return which == 1 ? ns_rows_ok<N>(16) : ns_cols_ok<N>(16);
    default: return false;
  }
}

// The step's kernels of the plan's shapes, in the radix-8 schedule.
template <int N>
int ns_explicit_impl(const NsParams& plan, const float2* w, float2* out, float2* g, float2* pbuf,
                     int batch, hipStream_t s) {
  NsParams q = plan;
  q.radix = 8;
  int rc = ns_launch<N>(0, q, w, nullptr, nullptr, nullptr, g, batch, s);
  if (!rc) rc = ns_launch<N>(1, q, g, nullptr, nullptr, nullptr, pbuf, batch, s);
  if (!rc) rc = NsOps<N>::explicit_cols(q, pbuf, out, batch, s);
  return rc;
}

}  // namespace

bool ns_group_size_supported(int n) { return ns_size_supported(n); }

int ns_group_tiles(int n, int list) {
  switch (n) {
    case 32: return list == 0 ? 16 / NsGroupShape<32>::W : 32 / NsGroupShape<32>::RB;
    case 64: return list == 0 ? 32 / NsGroupShape<64>::W : 64 / NsGroupShape<64>::RB;
    case 128: return list == 0 ? 64 / NsGroupShape<128>::W : 128 / NsGroupShape<128>::RB;
    case 256: return list == 0 ? 128 / NsGroupShape<256>::W : 256 / NsGroupShape<256>::RB;
    case 512: return list == 0 ? 256 / NsGroupShape<512>::W : 512 / NsGroupShape<512>::RB;
    case 1024: return list == 0 ? 512 / NsGroupShape<1024>::W : 1024 / NsGroupShape<1024>::RB;
    default: return 0;
  }
}

namespace {
template <bool BIG>
int ns_group_dispatch(int cls, int max_n, const NsGroupQueue& q, int stage, int grid, hipStream_t s) {
  const size_t lds = static_cast<size_t>(ns_group_lds(cls, max_n));
  const dim3 g(grid), t(ns_group_threads(cls));
  switch (cls) {
    case 0: hipLaunchKernelGGL((ns_group_phase<0, BIG>), g, t, lds, s, q.descs, q.items[0], q.n_items, stage); break;
    case 1: hipLaunchKernelGGL((ns_group_phase<1, BIG>), g, t, lds, s, q.descs, q.items[1], q.n_items + 1, stage); break;
    case 2: hipLaunchKernelGGL((ns_group_phase<2, BIG>), g, t, lds, s, q.descs, q.items[0], q.n_items, stage); break;
    default: hipLaunchKernelGGL((ns_group_phase<3, BIG>), g, t, lds, s, q.descs, q.items[0], q.n_items, stage);
  }
  return check_hip(hipGetLastError(), "spectral group launch");
}
}  // namespace

int ns_group_launch(int cls, int max_n, const NsGroupQueue& q, int stage, int grid, hipStream_t s) {
  if (!ns_group_size_supported(max_n))
    return fail(JCFD_ERR_UNSUPPORTED, "spectral group grid size not supported: " + std::to_string(max_n));
  return max_n > 512 ? ns_group_dispatch<true>(cls, max_n, q, stage, grid, s)
                     : ns_group_dispatch<false>(cls, max_n, q, stage, grid, s);
}

bool ns_size_supported(int n) {
  return n == 32 || n == 64 || n == 128 || n == 256 || n == 512 || n == 1024;
}

namespace {
template <int N>
int ns_one_impl(int which, const NsParams* stages, int nstages, const NsBuffers& b, int batch,
                hipStream_t s) {
  switch (which) {
    case 0: return ns_launch<N>(0, stages[0], b.u_in, nullptr, nullptr, nullptr, b.g, batch, s);
    case 1: return ns_launch<N>(1, stages[0], b.g, nullptr, nullptr, nullptr, b.pbuf, batch, s);
    case 2: return ns_launch<N>(2, stages[nstages > 1 ? 1 : 0], b.pbuf, b.u_out, b.u_out, b.h, b.g,
                                batch, s);
    default: return ns_launch<N>(3, stages[nstages - 1], b.pbuf, b.u_out, b.u_out, b.h, b.g, batch, s);
  }
}

}  // namespace

// Tile shapes of plans whose shapes were not set, from the launch's columns
// and rows over all instances.  Narrow tiles (W <= kStagedMaxW, the staged
// kernels) while the launch leaves the chip idle, the register kernels' wider
// ones beyond.  us per launch of the update-and-inverse kernel, W = 1 / 4 / 8:
// 1 x 256^2 5.9 / 12.9 / 13.7, 8 x 256^2 9.4 / 13.9 / 14.9, 32 x 256^2
// 22.0 / 21.1 / 20.7, 64 x 256^2 39 / 31.5 / 30.4; W = 1 / 4: 4 x 512^2
// 14.7 / 15.7, 8 x 512^2 22.4 / 21.4, 64 x 512^2 139 / 128, 1 x 1024^2
// 20.6 / 27.9, 8 x 1024^2 97 / 68.  Row kernel, small / large shape: 1 x 256^2
// 4.3 / 5.9 (RB 1 / 8), 64 x 256^2 50 / 22 (RB 1 / 4), 8 x 512^2 20.6 / 17.9
// (RB 2 / 8), 32 x 512^2 63 / 49, 8 x 1024^2 86 / 59 (RB 1 / 4).
int ns_default_tiles(NsParams* q, int n, int count) {
  if (!ns_size_supported(n)) return fail(JCFD_ERR_UNSUPPORTED, "spectral grid size not built");
  const long long rows = static_cast<long long>(n) * count, cols = rows / 2;
  switch (n) {
    case 32:
      q->w_cols = cols < 1024 ? 1 : cols < 4096 ? 4 : 8;
      q->rb_rows = 8;
      break;
    case 64:
      q->w_cols = cols < 1024 ? 1 : cols < 8192 ? 4 : 8;
      q->rb_rows = rows < 2048 ? 4 : 16;
      break;
    case 128:
      q->w_cols = cols < 1024 ? 1 : cols < 4096 ? 2 : cols < 8192 ? 4 : 8;
      q->rb_rows = rows < 1024 ? 2 : rows < 4096 ? 4 : 8;
      break;
    case 256:
      q->w_cols = cols < 2048 ? 1 : cols < 4096 ? 2 : 8;
      q->rb_rows = rows < 512 ? 1 : rows < 1024 ? 2 : 4;
      break;
    case 512:
      q->w_cols = cols < 2048 ? 1 : 8;
      q->rb_rows = rows < 4096 ? 2 : 8;
      break;
    default:
      q->w_cols = cols < 2048 ? 1 : 4;
      q->rb_rows = rows < 2048 ? 1 : 4;
  }
  q->radix = 8;
  return JCFD_OK;
}

bool ns_tile_supported(int n, int which, int tile) {
  switch (n) {
    case 32: return ns_tile_on_menu<32>(which, tile);
    case 64: return ns_tile_on_menu<64>(which, tile);
    case 128: return ns_tile_on_menu<128>(which, tile);
    case 256: return ns_tile_on_menu<256>(which, tile);
    case 512: return ns_tile_on_menu<512>(which, tile);
    case 1024: return ns_tile_on_menu<1024>(which, tile);
    default: return false;
  }
}

int ns_launch_kernel(int n, int which, const NsParams* stages, int nstages, const NsBuffers& b,
                     int batch, hipStream_t s) {
  if (nstages < 1) return fail(JCFD_ERR_INVALID_ARGUMENT, "at least one stage");
  switch (n) {
    case 32: return ns_one_impl<32>(which, stages, nstages, b, batch, s);
    case 64: return ns_one_impl<64>(which, stages, nstages, b, batch, s);
    case 128: return ns_one_impl<128>(which, stages, nstages, b, batch, s);
    case 256: return ns_one_impl<256>(which, stages, nstages, b, batch, s);
    case 512: return ns_one_impl<512>(which, stages, nstages, b, batch, s);
    case 1024: return ns_one_impl<1024>(which, stages, nstages, b, batch, s);
    default: return fail(JCFD_ERR_UNSUPPORTED, "spectral grid size not built");
  }
}

int ns_launch_step(int n, const NsParams* stages, int nstages, const NsBuffers& b, int batch,
                   hipStream_t s) {
  if (nstages < 1) return fail(JCFD_ERR_INVALID_ARGUMENT, "at least one stage");
  switch (n) {
    case 32: return ns_step_impl<32>(stages, nstages, b, batch, s);
    case 64: return ns_step_impl<64>(stages, nstages, b, batch, s);
    case 128: return ns_step_impl<128>(stages, nstages, b, batch, s);
    case 256: return ns_step_impl<256>(stages, nstages, b, batch, s);
    case 512: return ns_step_impl<512>(stages, nstages, b, batch, s);
    case 1024: return ns_step_impl<1024>(stages, nstages, b, batch, s);
    default: return fail(JCFD_ERR_UNSUPPORTED, "spectral grid size not built");
  }
}

int ns_launch_rfft2(int n, const NsParams& q, const float* x, float2* out, float2* pbuf, int batch,
                    hipStream_t s) {
  switch (n) {
    case 32: return NsOps<32>::rfft2(q, x, out, pbuf, batch, s);
    case 64: return NsOps<64>::rfft2(q, x, out, pbuf, batch, s);
    case 128: return NsOps<128>::rfft2(q, x, out, pbuf, batch, s);
    case 256: return NsOps<256>::rfft2(q, x, out, pbuf, batch, s);
    case 512: return NsOps<512>::rfft2(q, x, out, pbuf, batch, s);
    case 1024: return NsOps<1024>::rfft2(q, x, out, pbuf, batch, s);
    default: return fail(JCFD_ERR_UNSUPPORTED, "spectral grid size not built");
  }
}

int ns_launch_irfft2(int n, const NsParams& q, const float2* in, float* x, float2* pbuf, int batch,
                     hipStream_t s) {
  switch (n) {
    case 32: return NsOps<32>::irfft2(q, in, x, pbuf, batch, s);
    case 64: return NsOps<64>::irfft2(q, in, x, pbuf, batch, s);
    case 128: return NsOps<128>::irfft2(q, in, x, pbuf, batch, s);
    case 256: return NsOps<256>::irfft2(q, in, x, pbuf, batch, s);
    case 512: return NsOps<512>::irfft2(q, in, x, pbuf, batch, s);
    case 1024: return NsOps<1024>::irfft2(q, in, x, pbuf, batch, s);
    default: return fail(JCFD_ERR_UNSUPPORTED, "spectral grid size not built");
  }
}

namespace {
template <int N>
int ns_convert_n(bool to_internal, const float2* src, float2* dst, const int* slots, int count,
                 hipStream_t s) {
  const dim3 grid((N * (N / 2 + 1) + kThreads - 1) / kThreads, count);
  if (to_internal)
    hipLaunchKernelGGL((ns_state_convert<N, true>), grid, dim3(kThreads), 0, s, src, dst, slots);
  else
    hipLaunchKernelGGL((ns_state_convert<N, false>), grid, dim3(kThreads), 0, s, src, dst, slots);
  return check_hip(hipGetLastError(), "ns_state_convert");
}
}  // namespace

int ns_launch_state_convert(int n, bool to_internal, const float2* src, float2* dst, const int* slots,
                            int count, hipStream_t s) {
  switch (n) {
    case 32: return ns_convert_n<32>(to_internal, src, dst, slots, count, s);
    case 64: return ns_convert_n<64>(to_internal, src, dst, slots, count, s);
    case 128: return ns_convert_n<128>(to_internal, src, dst, slots, count, s);
    case 256: return ns_convert_n<256>(to_internal, src, dst, slots, count, s);
    case 512: return ns_convert_n<512>(to_internal, src, dst, slots, count, s);
    case 1024: return ns_convert_n<1024>(to_internal, src, dst, slots, count, s);
    default: return fail(JCFD_ERR_UNSUPPORTED, "spectral grid size not built");
  }
}

int ns_launch_explicit_terms(int n, const NsParams& q, const float2* w, float2* out, float2* g,
                             float2* pbuf, int batch, hipStream_t s) {
  switch (n) {
    case 32: return ns_explicit_impl<32>(q, w, out, g, pbuf, batch, s);
    case 64: return ns_explicit_impl<64>(q, w, out, g, pbuf, batch, s);
    case 128: return ns_explicit_impl<128>(q, w, out, g, pbuf, batch, s);
    case 256: return ns_explicit_impl<256>(q, w, out, g, pbuf, batch, s);
    case 512: return ns_explicit_impl<512>(q, w, out, g, pbuf, batch, s);
    case 1024: return ns_explicit_impl<1024>(q, w, out, g, pbuf, batch, s);
    default: return fail(JCFD_ERR_UNSUPPORTED, "spectral grid size not built");
  }
}

}  // namespace jcfd
