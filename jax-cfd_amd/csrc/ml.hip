// Learned-interpolation FVM convection (jax_cfd/ml/interpolations.py:31-121,
// FusedLearnedInterpolation under advections.modular_self_advection) for
// gfx950.
//
// The reference runs one CNN tower (towers.py:144-262: periodic 3x3
// convolutions, relu between them) over the stacked velocity components,
// turns each interpolation's slice of the output into polynomially
// constrained stencil coefficients, bias + logits . nullspace
// (layers.py:451-544, 586-642), and interpolates u and v to the control-volume
// faces with them (4 x 4 patches, layers_util.py:324-447) before
// advect_general (base/advection.py:34-116).  Here:
//
//   li_conv3x3_first, li_conv3x3
//                 one periodic 3x3 convolution layer as an implicit GEMM on
//                 the matrix cores, D[co][px] = sum over (tap, ci) of
//                 W[tap][ci][co] * x[ci][px + tap], + bias, relu, with fp32
//                 accuracy (the first layer on v_mfma_f32_16x16x4_f32, the
//                 others on v_mfma_f32_16x16x32_bf16 with three-part
//                 operands).  A workgroup owns 4 rows x 32 columns of
//                 pixels and up to 64 output channels; the input tile with
//                 its one-cell periodic halo goes through LDS in chunks of
//                 32 channels.  The weights are stored in MFMA operand
//                 order, so each wavefront reads its A operands straight
//                 from global memory (cache-resident: every workgroup reads
//                 the same few hundred KB), the next step's loads in flight
//                 during the current step's products; one barrier per
//                 chunk.  The tower's output layer is the
//                 constraint folded in: its 128 channels are the 8
//                 interpolations' 16 stencil coefficients each (weights
//                 W . nullspace, bias b . nullspace + constraint bias, formed
//                 in fp64 on the host), so no logits are materialised.
//   li_explicit   per row block: the 8 interpolations (16-term dot products
//                 of coefficients and 4 x 4 patches of u or v from LDS), the
//                 face fluxes aligned_c * aligned_v, their divergence, then
//                 diffusion and forcing -- the explicit terms k_u, k_v that
//                 the forward-Euler combination kernel (rows-forward mode 5)
//                 turns into u*, projected as every FVM step is.
//   li_interpolate one interpolation of one field (the interpolators of
//                 FusedLearnedInterpolation as a testing seam).
//
// Activations are planar per instance: (batch, channels, n, n) fp32.
#include <hip/hip_runtime.h>

#include <cstring>
#include <type_traits>
#include <utility>

#include "fvm_terms.h"
#include "jcfd_fft.h"
#include "jcfd_internal.h"

#pragma clang fp contract(off)

namespace jcfd {
namespace {

constexpr int kThreads = 256;
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Output tile of a convolution workgroup and its LDS halo tile.
constexpr int kConvRows = 4;                         // one row per wavefront
constexpr int kConvCols = 32;                        // two 16-pixel MFMA blocks
constexpr int kHaloW = kConvCols + 2;
constexpr int kHaloPlane = (kConvRows + 2) * kHaloW;  // 204 words

// Calls f(integral_constant<int, S>) for S = B .. E-1 (a loop the compiler
// sees fully unrolled, with compile-time step numbers).
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  if constexpr (B < E) {
    f(std::integral_constant<int, B>{});
    static_for<B + 1, E>(f);
  }
}

// The first layer (u, v; padded to 4 channels): fp32 products, one k-step of
// v_mfma_f32_16x16x4_f32 per tap.  Operand layout (checked on gfx950):
// A[i][k] in lane i + 16 k, B[k][j] in lane j + 16 k, D[i][j] in lane
// j + 16 (i / 4), register i % 4; i = output channel, j = pixel, k = input
// channel.  Its 36 products per output leave it bound by the stores of its
// activations, so the products stay as they are.  Weight fragment (tap,
// channel block cb) holds W[tap][ci = k][co = 16 cb + i] of lane i + 16 k at
// float offset (tap NCB + cb) 64 + lane.
constexpr int kFirstPitch = 208;  // plane pitch: the 4 channels of a k-step land 16 banks apart
template <int COUT, bool RELU>
__global__ __launch_bounds__(kThreads) void li_conv3x3_first(LiConvArgs a) {
  constexpr int NCB = COUT / 16;
  __shared__ float shalo[4 * kFirstPitch];
  const int n = a.n;
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const int tiles_x = n / kConvCols;
  const int t = xcd_tile(blockIdx.x, gridDim.x);
  const int i0 = (t / tiles_x) * kConvRows, j0 = (t % tiles_x) * kConvCols;
  const size_t plane = static_cast<size_t>(n) * n;
  const float* in = a.in + blockIdx.y * plane;
  const float* in_v = a.in_v + blockIdx.y * plane;
  const float* wf = static_cast<const float*>(a.w) + lane;
  float w[9][NCB];
#pragma unroll
  for (int tap = 0; tap < 9; ++tap)
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) w[tap][cb] = wf[(tap * NCB + cb) * 64];
  if (tid < kHaloPlane) {
    const int r = tid / kHaloW, cc = tid % kHaloW;
    const size_t gi = static_cast<size_t>((i0 - 1 + r) & (n - 1)) * n + ((j0 - 1 + cc) & (n - 1));
    const float x = in[gi], y = in_v[gi];
    shalo[tid] = x;
    shalo[kFirstPitch + tid] = y;
    shalo[2 * kFirstPitch + tid] = 0.f;
    shalo[3 * kFirstPitch + tid] = 0.f;
  }
  __syncthreads();
  floatx4 acc[NCB][2];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) acc[cb][0] = acc[cb][1] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int kq = lane / 16, lp = lane % 16;
#pragma unroll
  for (int tap = 0; tap < 9; ++tap) {
    const float* bin = shalo + kq * kFirstPitch + (wave + tap / 3) * kHaloW + tap % 3 + lp;
    const float b0 = bin[0], b1 = bin[16];
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      acc[cb][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[tap][cb], b0, acc[cb][0], 0, 0, 0);
      acc[cb][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[tap][cb], b1, acc[cb][1], 0, 0, 0);
    }
  }
  // out[co][i0 + wave][j0 + px] = act(acc + b[co])
  float* out = a.out + blockIdx.y * COUT * plane + static_cast<size_t>(i0 + wave) * n + j0;
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int co = cb * 16 + 4 * kq + r;
      const float bias = a.b[co];
#pragma unroll
      for (int pb = 0; pb < 2; ++pb) {
        float x = acc[cb][pb][r] + bias;
        if constexpr (RELU) x = fmaxf(x, 0.f);
        out[co * plane + pb * 16 + lp] = x;
      }
    }
}

// Shape of a hidden or output layer: k-steps of 32 (one bf16 MFMA deep), the
// input channels in chunks of CH.  A k-step is one tap of 32 channels, or,
// for 16 input channels, two taps (the ninth tap's partner has zero weights).
template <int CIN, int COUT>
struct ConvSplit {
  static constexpr int CH = CIN < 32 ? CIN : 32;      // channels per chunk
  static constexpr int CHUNKS = CIN / CH;
  static constexpr int TPS = 32 / CH;                 // taps per k-step
  static constexpr int SPC = (9 + TPS - 1) / TPS;     // k-steps per chunk
  static constexpr int STEPS = SPC * CHUNKS;
  static constexpr int CO = COUT < 64 ? COUT : 64;    // output channels per workgroup
  static constexpr int CW = CO == 64 ? 2 : 1;         // wavefronts across them
  static constexpr int PW = 4 / CW;                   // wavefronts across the 128 pixels
  static constexpr int NCB = CO / 16 / CW;            // 16-channel blocks per wavefront
  static constexpr int NPB = 8 / PW;                  // 16-pixel blocks per wavefront
};

// Hidden and output layers.  fp32 products on the bf16 matrix cores: each
// operand is the exact sum of three bf16 parts, x = x0 + x1 + x2 (each part
// the rounding of what the ones before it leave; 3 x 8 bits hold fp32's 24),
// and x w is summed from the six largest part products
// (x0 w0, x0 w1, x1 w0, x1 w1, x0 w2, x2 w0; a bf16 product is exact in
// fp32), accumulated in fp32.  What is left out, x1 w2 + x2 w1 + x2 w2, is at
// most 2^-24 of x w (x = w = 1.0038986), one rounding of the product, and far
// less on average.  Against 64 bits
// whole towers (n 32 to 256, 16 to 64 channels, 3 and 7 layers, inputs of scale
// 1 and 1e-3) err 0.29 to 0.60 as much, rms, as with v_mfma_f32_16x16x4_f32
// products, 0.40 in the mean, because each sum is rounded once per 32 products.
//
// What bounds it is the matrix cores: six v_mfma_f32_16x16x32_bf16 (16 cycles
// each) do the work of eight v_mfma_f32_16x16x4_f32 (32 cycles each).  256^2,
// 64 -> 64 channels: 50 us (99 of the 154 TFLOP/s a large fp32 product reaches)
// with fp32 products, 27 us so (1050 TFLOP/s of part products; a large bf16
// product reaches 1130); 64 -> 128: 94 and 49 us.
//
// A workgroup owns 4 rows x 32 columns of pixels and 64 output channels, a
// wavefront 64 pixels x 32 channels of them: 12 B fragments from LDS and 6 A
// fragments from global memory (L1/L2-resident, stored in operand order, the
// next step's in flight) feed 48 MFMA, half the rate either path can give.
// The pixels' parts sit in LDS as [part][8 channels][pixel][channel], so a
// fragment read is 16 consecutive 16-byte words per 16 lanes; the split is
// made once per workgroup, when a chunk of 32 channels is staged, and the
// second chunk is loaded while the first is used.
//
// Values without such a split show in what the first two parts leave: NaN for
// infinities, NaN and values whose first part is infinite (beyond 2^128 -
// 2^119), a subnormal number where the third part may end below bf16's 2^-133
// (values under 2^-110; the matrix cores keep subnormal parts).  A workgroup
// that meets one among its inputs forms its outputs from the fp32 values,
// v_mfma_f32_16x16x4_f32, the weights added up from their parts: the tower's
// layers at 256^2, 64 channels, all of them so, take 440 us against 184 with
// splits.  (Parts of a weight under 2^-133 are dropped: an output moves by
// 2^-134 of its inputs' sum at most.)
constexpr int kNoSplit = 0x297;  // v_cmp_class_f32: NaN, infinite or subnormal
template <int CIN, int COUT, bool RELU>
__global__ __launch_bounds__(kThreads, 2) void li_conv3x3(LiConvArgs a) {
  using F = ConvSplit<CIN, COUT>;
  constexpr int CH = F::CH, NCB = F::NCB, NPB = F::NPB, STEPS = F::STEPS;
  constexpr int KG = CH / 8;                            // groups of 8 channels per chunk
  constexpr int ITEMS = KG * kHaloPlane;                // (pixel, group) pairs staged per chunk
  constexpr int HPT = (ITEMS + kThreads - 1) / kThreads;
  constexpr int NBUF = F::CHUNKS > 1 ? 2 : 1;
  constexpr int ZC = COUT / F::CO;
  __shared__ bf16x8 shalo[NBUF][3][ITEMS];
  __shared__ int s_wild[F::CHUNKS][4];  // whether a wavefront staged a value without a split, per chunk
  const int n = a.n;
  const int tid = threadIdx.x, lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int tiles_x = n / kConvCols;
  const int t = xcd_tile(blockIdx.x, gridDim.x) / ZC, z = xcd_tile(blockIdx.x, gridDim.x) % ZC;
  const int i0 = (t / tiles_x) * kConvRows, j0 = (t % tiles_x) * kConvCols;
  const size_t plane = static_cast<size_t>(n) * n;
  const float* in = a.in + blockIdx.y * CIN * plane;
  const int cw = wave % F::CW, pw = wave / F::CW;
  const int cb0 = z * (F::CO / 16) + cw * NCB;          // first channel block of this wavefront
  // fragment (step, channel block, part) at wf[((step COUT/16 + block) 3 + part) 64]
  const bf16x8* wf = static_cast<const bf16x8*>(a.w) + cb0 * 3 * 64;
  const unsigned ulane = lane;
  auto load = [&](int s, bf16x8 (&w)[NCB][3]) {
    const int sc = s < STEPS ? s : STEPS - 1;  // unconditional: the last prefetch repeats
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
      for (int q = 0; q < 3; ++q) w[cb][q] = (wf + ((sc * (COUT / 16) + cb) * 3 + q) * 64)[ulane];
  };
  // halo tile of chunk g (rows i0-1 .. i0+4, columns j0-1 .. j0+32, periodic)
  float hreg[HPT][8];
  auto halo_load = [&](int g) {
#pragma unroll
    for (int k = 0; k < HPT; ++k) {
      const int e0 = tid + k * kThreads;
      const int e = e0 < ITEMS ? e0 : ITEMS - 1;
      const int kg = e / kHaloPlane, px = e % kHaloPlane, r = px / kHaloW, cc = px % kHaloW;
      const unsigned off = static_cast<unsigned>(kg * 8 * plane) + ((i0 - 1 + r) & (n - 1)) * n + ((j0 - 1 + cc) & (n - 1));
#pragma unroll
      for (int c = 0; c < 8; ++c) hreg[k][c] = (in + (g * CH + c) * plane)[off];
    }
  };
  auto halo_store = [&](int g) {
    const int buf = g % NBUF;
    bool wild = false;
#pragma unroll
    for (int k = 0; k < HPT; ++k) {
      const int e = tid + k * kThreads;
      bf16x8 p0, p1, p2;
#pragma unroll
      for (int c = 0; c < 8; ++c) {
        const float x = hreg[k][c];
        const __bf16 x0 = static_cast<__bf16>(x);
        const float r1 = x - static_cast<float>(x0);
        const __bf16 x1 = static_cast<__bf16>(r1);
        const float r2 = r1 - static_cast<float>(x1);
        wild = wild || __builtin_amdgcn_classf(r2, kNoSplit);
        p0[c] = x0;
        p1[c] = x1;
        p2[c] = static_cast<__bf16>(r2);
      }
      if (ITEMS % kThreads == 0 || e < ITEMS) {
        shalo[buf][0][e] = p0;
        shalo[buf][1][e] = p1;
        shalo[buf][2][e] = p2;
      }
    }
    const int any = __any(wild);
    if (lane == 0) s_wild[g][wave] = any;
  };
  // after the barrier that follows the chunk's halo_store
  auto chunk_is_wild = [&](int g) {
    return __builtin_amdgcn_readfirstlane(s_wild[g][0] | s_wild[g][1] | s_wild[g][2] | s_wild[g][3]) != 0;
  };
  bf16x8 wa[NCB][3], wb[NCB][3];
  load(0, wa);
  halo_load(0);
  halo_store(0);
  __syncthreads();

  floatx4 acc[NCB][NPB];
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
    for (int pb = 0; pb < NPB; ++pb) acc[cb][pb] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int kq = lane / 16, lp = lane % 16;
  // pixel block pb of this wavefront: tile pixel 16 (pw NPB + pb), two to a row
  auto block_row = [&](int pb) { return (pw * NPB + pb) / 2; };
  const int kg = kq % KG;
  const int lbase = kg * kHaloPlane + lp + block_row(0) * kHaloW;
  auto step = [&](int s, const bf16x8 (&w)[NCB][3]) {
    const int g = s / F::SPC, t0 = (s % F::SPC) * F::TPS;
    const int o0 = (t0 / 3) * kHaloW + t0 % 3;
    int off = lbase + o0;
    if constexpr (F::TPS == 2) {
      const int t1 = t0 + 1 < 9 ? t0 + 1 : 8;
      off = lbase + (kq < 2 ? o0 : (t1 / 3) * kHaloW + t1 % 3);
    }
    bf16x8 x[NPB][3];
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll
      for (int pb = 0; pb < NPB; ++pb)
        x[pb][q] = shalo[g % NBUF][q][off + (pb / 2) * kHaloW + (pb % 2) * 16];
    // The step's six part products, small ones first, in accumulators of
    // their own, which are then added to the sums: one rounding of each sum
    // per step (summing all six into it measured 10 % more error).
    constexpr int PX[6] = {2, 0, 1, 1, 0, 0}, PWT[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) {
      floatx4 part[NPB];
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int pb = 0; pb < NPB; ++pb)
          part[pb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              w[cb][PWT[q]], x[pb][PX[q]], q == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : part[pb], 0, 0, 0);
#pragma unroll
      for (int pb = 0; pb < NPB; ++pb) {
        acc[cb][pb] += part[pb];
        // an empty use: the additions are not moved behind the last step,
        // which would keep every step's part products until there
        asm volatile("" : "+v"(acc[cb][pb]));
      }
    }
  };
  // step s computes with one register set while the other receives step
  // s + 1's weights (the sets alternate, so no copy waits for a load)
  auto run = [&](auto sc, bf16x8 (&cur)[NCB][3], bf16x8 (&nxt)[NCB][3]) {
    constexpr int s = decltype(sc)::value;
    constexpr int g = s / F::SPC;
    load(s + 1, nxt);
    if constexpr (s % F::SPC == 0 && g + 1 < F::CHUNKS) halo_load(g + 1);
    step(s, cur);
    if constexpr (s % F::SPC == F::SPC - 1 && g + 1 < F::CHUNKS) {
      halo_store(g + 1);  // its buffer's last reader was chunk g - 1
      __syncthreads();
    }
  };
  bool wild = chunk_is_wild(0);
  if (!wild) {
    static_for<0, STEPS>([&](auto sc) {
      if constexpr (decltype(sc)::value % 2 == 0) run(sc, wa, wb);
      else run(sc, wb, wa);
    });
#pragma unroll
    for (int g = 1; g < F::CHUNKS; ++g) wild = wild || chunk_is_wild(g);
  }
  if (wild) {
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
      for (int pb = 0; pb < NPB; ++pb) acc[cb][pb] = floatx4{0.f, 0.f, 0.f, 0.f};
    // a step's 32 products in eight MFMA of four: k = 8 kq + e in the e-th
#pragma unroll 1
    for (int s = 0; s < STEPS; ++s) {
      const int tap = (s % F::SPC) * F::TPS + (F::TPS == 2 ? kq / 2 : 0);
      const float* xc = in + ((s / F::SPC) * CH + 8 * kg) * plane;
      load(s, wa);
#pragma unroll
      for (int pb = 0; pb < NPB; ++pb) {
        const int i = (i0 + block_row(pb) + tap / 3 - 1) & (n - 1);
        const int j = (j0 + (pb % 2) * 16 + lp + tap % 3 - 1) & (n - 1);
        float x[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = xc[e * plane + static_cast<size_t>(i) * n + j];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if (F::TPS == 2 && tap > 8) x[e] = 0.f;  // the ninth tap's partner: not 0 times an infinity
#pragma unroll
          for (int cb = 0; cb < NCB; ++cb)
            acc[cb][pb] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                static_cast<float>(wa[cb][0][e]) + (static_cast<float>(wa[cb][1][e]) + static_cast<float>(wa[cb][2][e])),
                x[e], acc[cb][pb], 0, 0, 0);
        }
      }
    }
  }

  // out[co][i0 + row][j0 + px] = act(acc + b[co])
  float* out = a.out + blockIdx.y * COUT * plane + static_cast<size_t>(i0) * n + j0;
#pragma unroll
  for (int cb = 0; cb < NCB; ++cb) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int co = (cb0 + cb) * 16 + 4 * kq + r;
      const float bias = a.b[co];
#pragma unroll
      for (int pb = 0; pb < NPB; ++pb) {
        float x = acc[cb][pb][r] + bias;
        if constexpr (RELU) x = fmaxf(x, 0.f);
        out[co * plane + block_row(pb) * n + (pb % 2) * 16 + lp] = x;
      }
    }
  }
}

// The 16-term dot product of one interpolation at cell (gi, j): coefficient
// s = 4 (a + 1) + (b + 1) multiplies x[gi + a, j + b], a, b in {-1 .. 2}
// (extract_patches' channel order).  Summed as NumPy's pairwise reduction
// of 16 terms: r_k = t_k + t_{k+8}, then ((r0+r1)+(r2+r3))+((r4+r5)+(r6+r7)).
// `s` holds LDS rows, local row lr = gi - row0; `c` points at the
// interpolation's first coefficient plane at (gi, j).
template <int N>
__device__ __forceinline__ float li_dot(const float* __restrict__ c, size_t plane,
                                        const float* s, int lr, int j) {
  float t[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int da = q / 4 - 1, db = q % 4 - 1;
    t[q] = c[q * plane] * s[(lr + da) * N + ((j + db) & (N - 1))];
  }
  float r[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) r[k] = t[k] + t[k + 8];
  return ((r[0] + r[1]) + (r[2] + r[3])) + ((r[4] + r[5]) + (r[6] + r[7]));
}

// Explicit terms of the learned self-advection step for rows [i0, i0+RB):
// k = (-div(aligned_c * aligned_v) + nu lap) + f, per component, with the
// fluxes of advect_general (advection.py:81-116, _advect_aligned 34-78), for
// the components blockIdx.z, blockIdx.z + gridDim.z, ..  The coefficients are
// what it reads, 512 B per cell; see explicit_launch for the row blocks.
template <int N, int RB>
__global__ __launch_bounds__(kThreads) void li_explicit(FvmParams p, LiExplicitArgs a) {
  constexpr int ROWS = RB + 4;  // u, v rows i0-2 .. i0+RB+1
  __shared__ float su[ROWS * N], sv[ROWS * N];
  __shared__ float fxs[(RB + 1) * N], fys[RB * N];
  const int tid = threadIdx.x;
  const int i0 = xcd_tile(blockIdx.x, gridDim.x) * RB;
  const size_t plane = static_cast<size_t>(N) * N;
  const size_t inst = a.slots ? static_cast<size_t>(a.slots[blockIdx.y]) : blockIdx.y;
  const float* u = a.u + inst * plane;
  const float* v = a.v + inst * plane;
  const float* coef = a.coef + blockIdx.y * static_cast<size_t>(kLiCoefChannels) * plane;
  staged<ROWS * N, 8, kThreads>(
      tid,
      [&](int e) {
        const size_t g = static_cast<size_t>((i0 - 2 + e / N) & (N - 1)) * N + e % N;
        return make_float2(u[g], v[g]);
      },
      [&](int e, float2 x) {
        su[e] = x.x;
        sv[e] = x.y;
      });
  const Window<N> w{su, sv};
  __syncthreads();
  // face flux of one interpolation pair at local row lr (global gi):
  // aligned_c (coefficients at base kc, field sc) * aligned_v (kv, sv_)
  auto flux = [&](int kc, const float* fc, int kv, const float* fv, int lr, int j) {
    const size_t at = static_cast<size_t>((i0 - 2 + lr) & (N - 1)) * N + j;
    const float cval = li_dot<N>(coef + kc * plane + at, plane, fc, lr, j);
    const float vval = li_dot<N>(coef + kv * plane + at, plane, fv, lr, j);
    return cval * vval;
  };
#pragma unroll 1
  for (int comp = blockIdx.z; comp < 2; comp += gridDim.z) {
    const float* sc = comp == 0 ? su : sv;  // the advected component
    const int* key = a.key + 4 * comp;      // x face: (c, velocity), y face: (c, velocity)
    const float* vx = su;                   // velocity of the x faces: u
    const float* vy = sv;                   // of the y faces: v
    // x faces of rows i0-1 .. i0+RB-1 (local rows 1 .. RB+1), y faces of rows i0 ..
    for (int e = tid; e < (RB + 1) * N; e += kThreads)
      fxs[e] = flux(key[0], sc, key[1], vx, 1 + e / N, e % N);
    for (int e = tid; e < RB * N; e += kThreads)
      fys[e] = flux(key[2], sc, key[3], vy, 2 + e / N, e % N);
    __syncthreads();
    float* kout = (comp == 0 ? a.ku : a.kv) + inst * plane;
    for (int e = tid; e < RB * N; e += kThreads) {
      const int r = e / N, j = e % N;
      const float adv = -(over_step(fxs[(r + 1) * N + j] - fxs[r * N + j], p.dx, p.rcp_dx) +
                          over_step(fys[r * N + j] - fys[r * N + ((j - 1) & (N - 1))], p.dy, p.rcp_dy));
      const float k = comp == 0 ? add_diffusion_forcing<false>(w, r + 2, j, p, p.has_forcing ? a.fx[j] : 0.f, adv)
                                : add_diffusion_forcing<true>(w, r + 2, j, p, 0.f, adv);
      kout[static_cast<size_t>(i0 + r) * N + j] = k;
    }
    __syncthreads();
  }
}

// out = interpolation `key` (coefficient planes key .. key+15) applied to x.
template <int N>
__global__ __launch_bounds__(kThreads) void li_interpolate(const float* __restrict__ coef,
                                                           const float* __restrict__ x, int key,
                                                           float* __restrict__ out) {
  constexpr int RB = kThreads / N > 0 ? kThreads / N : 1;
  constexpr int ROWS = RB + 3;
  __shared__ float sx[ROWS * N];
  const int tid = threadIdx.x;
  const int i0 = blockIdx.x * RB;
  const size_t plane = static_cast<size_t>(N) * N;
  x += blockIdx.y * plane;
  coef += blockIdx.y * static_cast<size_t>(kLiCoefChannels) * plane + key * plane;
  out += blockIdx.y * plane;
  for (int e = tid; e < ROWS * N; e += kThreads)
    sx[e] = x[static_cast<size_t>((i0 - 1 + e / N) & (N - 1)) * N + e % N];
  __syncthreads();
  for (int e = tid; e < RB * N; e += kThreads) {
    const int r = e / N, j = e % N;
    const size_t at = static_cast<size_t>(i0 + r) * N + j;
    out[at] = li_dot<N>(coef + at, plane, sx, r + 1, j);
  }
}

// ---- launchers ------------------------------------------------------------
template <int COUT, bool RELU>
int first_launch(const LiConvArgs& a, int batch, hipStream_t s) {
  const dim3 grid((a.n / kConvCols) * (a.n / kConvRows), batch);
  hipLaunchKernelGGL((li_conv3x3_first<COUT, RELU>), grid, dim3(kThreads), 0, s, a);
  return check_hip(hipGetLastError(), "li_conv3x3_first");
}

template <int COUT>
int conv_first(const LiConvArgs& a, bool relu, int batch, hipStream_t s) {
  return relu ? first_launch<COUT, true>(a, batch, s) : first_launch<COUT, false>(a, batch, s);
}

template <int CIN, int COUT, bool RELU>
int conv_launch(const LiConvArgs& a, int batch, hipStream_t s) {
  const dim3 grid((a.n / kConvCols) * (a.n / kConvRows) * (COUT / ConvSplit<CIN, COUT>::CO), batch);
  hipLaunchKernelGGL((li_conv3x3<CIN, COUT, RELU>), grid, dim3(kThreads), 0, s, a);
  return check_hip(hipGetLastError(), "li_conv3x3");
}

template <int CIN>
int conv_hidden(const LiConvArgs& a, int cout, bool relu, int batch, hipStream_t s) {
  if (relu && cout == CIN) return conv_launch<CIN, CIN, true>(a, batch, s);
  if (!relu && cout == kLiCoefChannels) return conv_launch<CIN, kLiCoefChannels, false>(a, batch, s);
  return fail(JCFD_ERR_UNSUPPORTED, "convolution " + std::to_string(CIN) + " -> " + std::to_string(cout) +
                                        (relu ? " (relu)" : "") + " not built");
}

// Launches of up to 2^17 cells leave CUs idle in the row blocks that suit
// larger ones: they take one row (whose x faces a neighbour forms again, from
// the cached coefficients) and one component per workgroup.  us, several rows
// and both components / one of each: 256^2 18.0 / 6.1, 64^2 7.0 / 3.8,
// 8 x 128^2 14.0 / 12.9; 4 x 256^2 24.0 / 26.9, 512^2 28.7 / 30.8.
template <int N>
int explicit_launch(const FvmParams& p, const LiExplicitArgs& a, int batch, hipStream_t s) {
  constexpr int RB = N <= 256 ? 4 : 2;
  if (static_cast<long long>(N) * N * batch <= 1 << 17)
    hipLaunchKernelGGL((li_explicit<N, 1>), dim3(N, batch, 2), dim3(kThreads), 0, s, p, a);
  else
    hipLaunchKernelGGL((li_explicit<N, RB>), dim3(N / RB, batch), dim3(kThreads), 0, s, p, a);
  return check_hip(hipGetLastError(), "li_explicit");
}

template <int N>
int interpolate_launch(const float* coef, const float* x, int key, float* out, int batch, hipStream_t s) {
  constexpr int RB = kThreads / N > 0 ? kThreads / N : 1;
  hipLaunchKernelGGL((li_interpolate<N>), dim3(N / RB, batch), dim3(kThreads), 0, s, coef, x, key, out);
  return check_hip(hipGetLastError(), "li_interpolate");
}

}  // namespace

namespace {
float from_bf16(uint16_t b) {
  const uint32_t u = static_cast<uint32_t>(b) << 16;
  float x;
  std::memcpy(&x, &u, sizeof(x));
  return x;
}
// Nearest bf16 (ties to even) of a finite x; the largest ones, whose nearest
// is infinite, are cut off instead.
uint16_t to_bf16(float x) {
  uint32_t u;
  std::memcpy(&u, &x, sizeof(u));
  const uint32_t r = (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;
  return static_cast<uint16_t>((r & 0x7f80u) == 0x7f80u ? u >> 16 : r);
}
}  // namespace

size_t li_conv_weight_bytes(int cinp, int cout) {
  if (cinp == 4) return static_cast<size_t>(9) * cinp * cout * sizeof(float);
  const int ch = cinp < 32 ? cinp : 32, tps = 32 / ch;
  return static_cast<size_t>((9 + tps - 1) / tps) * (cinp / ch) * 32 * cout * 3 * sizeof(uint16_t);
}

void li_conv_weight_layout(const float* w, int cinp, int cout, void* out) {
  auto weight = [&](int tap, int ci, int co) { return w[(static_cast<size_t>(tap) * cinp + ci) * cout + co]; };
  const int ncb = cout / 16;
  if (cinp == 4) {  // li_conv3x3_first
    float* frag = static_cast<float*>(out);
    for (int tap = 0; tap < 9; ++tap)
      for (int cb = 0; cb < ncb; ++cb)
        for (int l = 0; l < 64; ++l) frag[(tap * ncb + cb) * 64 + l] = weight(tap, l / 16, cb * 16 + l % 16);
    return;
  }
  // li_conv3x3: fragment (step, channel block, part), lane l, element e is
  // k = 8 (l / 16) + e of the step, output channel l % 16 of the block.  The
  // 8 k x 16 channels of 16 lanes are one contiguous run, split together.
  uint16_t* frag = static_cast<uint16_t*>(out);
  const int ch = cinp < 32 ? cinp : 32, tps = 32 / ch, spc = (9 + tps - 1) / tps;
  for (int s = 0; s < spc * (cinp / ch); ++s)
    for (int k8 = 0; k8 < 4; ++k8) {
      const int tap = (s % spc) * tps + 8 * k8 / ch, ci = (s / spc) * ch + 8 * k8 % ch;
      for (int cb = 0; cb < ncb; ++cb) {
        float x[128] = {};
        if (tap < 9) {
          const float* src = w + (static_cast<size_t>(tap) * cinp + ci) * cout + cb * 16;
          for (int i = 0; i < 16; ++i)
            for (int e = 0; e < 8; ++e) x[8 * i + e] = src[static_cast<size_t>(e) * cout + i];
        }
        for (int q = 0; q < 3; ++q) {
          uint16_t part[128];
          for (int i = 0; i < 128; ++i) {
            part[i] = to_bf16(x[i]);
            x[i] -= from_bf16(part[i]);
          }
          std::memcpy(frag + ((static_cast<size_t>(s) * ncb + cb) * 3 + q) * 512 + 128 * k8, part, sizeof(part));
        }
      }
    }
}

bool li_conv_supported(int cin, int cout, bool relu) {
  const bool hidden_out = relu && (cout == 16 || cout == 32 || cout == 64);
  const bool coef_out = !relu && cout == kLiCoefChannels;
  if (cin == 2) return hidden_out || coef_out;
  if (cin == 16 || cin == 32 || cin == 64) return (relu && cout == cin) || coef_out;
  return false;
}

int li_launch_conv(const LiConvArgs& a, int cin, int cout, bool relu, int batch, hipStream_t s) {
  if (a.n < kConvCols || (a.n & (a.n - 1)) != 0)
    return fail(JCFD_ERR_UNSUPPORTED, "learned interpolation needs n a power of two >= 32");
  if (!li_conv_supported(cin, cout, relu))
    return fail(JCFD_ERR_UNSUPPORTED, "convolution " + std::to_string(cin) + " -> " +
                                          std::to_string(cout) + " not built");
  if (cin == 2) {
    switch (cout) {
      case 16: return conv_first<16>(a, relu, batch, s);
      case 32: return conv_first<32>(a, relu, batch, s);
      case 64: return conv_first<64>(a, relu, batch, s);
      default: return conv_first<kLiCoefChannels>(a, relu, batch, s);
    }
  }
  switch (cin) {
    case 16: return conv_hidden<16>(a, cout, relu, batch, s);
    case 32: return conv_hidden<32>(a, cout, relu, batch, s);
    default: return conv_hidden<64>(a, cout, relu, batch, s);
  }
}

int li_launch_explicit(const FvmParams& p, const LiExplicitArgs& a, int batch, hipStream_t s) {
  switch (p.n) {
    case 32: return explicit_launch<32>(p, a, batch, s);
    case 64: return explicit_launch<64>(p, a, batch, s);
    case 128: return explicit_launch<128>(p, a, batch, s);
    case 256: return explicit_launch<256>(p, a, batch, s);
    case 512: return explicit_launch<512>(p, a, batch, s);
    case 1024: return explicit_launch<1024>(p, a, batch, s);
    default: return fail(JCFD_ERR_UNSUPPORTED, "learned interpolation grid size not built");
  }
}

int li_launch_interpolate(int n, const float* coef, const float* x, int key, float* out, int batch,
                          hipStream_t s) {
  switch (n) {
    case 32: return interpolate_launch<32>(coef, x, key, out, batch, s);
    case 64: return interpolate_launch<64>(coef, x, key, out, batch, s);
    case 128: return interpolate_launch<128>(coef, x, key, out, batch, s);
    case 256: return interpolate_launch<256>(coef, x, key, out, batch, s);
    case 512: return interpolate_launch<512>(coef, x, key, out, batch, s);
    case 1024: return interpolate_launch<1024>(coef, x, key, out, batch, s);
    default: return fail(JCFD_ERR_UNSUPPORTED, "learned interpolation grid size not built");
  }
}

}  // namespace jcfd
