// Conjugate-gradient pressure solve for the FVM step (gfx950).
//
// solve_cg (jax_cfd/base/pressure.py:67-112) calls
// jax.scipy.sparse.linalg.cg(laplacian, div v, x0 = 0, tol, atol): the
// unpreconditioned CG recurrence
//   alpha = gamma / <p, Ap>;  x += alpha p;  r -= alpha Ap;
//   gamma' = <r, r>;  beta = gamma' / gamma;  p = r + beta p,
// run while gamma > max(tol^2 <b, b>, atol^2) and k < maxiter, with A the
// periodic 5-point Laplacian of finite_differences.laplacian
// (finite_differences.py:127-133).
//
// The whole solve is one cooperative launch where the device can hold all the
// row blocks at once (cg_persistent); otherwise, or where a caller asks for it,
// each iteration is two kernels over row blocks:
//   cg_direction  p_k = r_k + beta_k p_{k-1} (rows +-1 halo recomputed in
//                 LDS), Ap = L p_k, per-block partial <p, Ap>; convergence is
//                 tested here against the reduced <r_k, r_k>.
//   cg_update     x += alpha p_k, r -= alpha Ap, per-block partial <r, r>.
// The same two kernels solve the implicit diffusion system of
// diffusion.solve_cg (jax_cfd/base/diffusion.py:137-167), one velocity
// component at a time: A x = x - coef L x with coef = fp32(dt viscosity),
// x0 = b = the component, so r0 = b - A b (cg_init_helmholtz).
// Dot products are reduced in a fixed order (block tree, then every block
// reduces the partials array itself), so runs are deterministic.  Once the
// test fails, block 0 raises a flag and every later kernel returns at once,
// so the host can enqueue iterations in chunks and read the flag between
// chunks.
#include <hip/hip_runtime.h>

#include "jcfd_internal.h"

#pragma clang fp contract(off)

namespace jcfd {
namespace {

constexpr int kThreads = 256;

constexpr int kMaxBlocks = 256;  // row blocks of the largest grids
constexpr int kMsgCopies = 8;
constexpr int kWaves = kThreads / 64;
static_assert(kWaves == 4, "block sums combine four wavefronts");

// Sum over a wavefront's 64 lanes by the butterfly l ^ 32, 16, 8, 4, 2, 1 (every
// lane ends with the same bits: each step adds the same two numbers in both
// lanes of a pair).  The exchanges are register moves, not LDS permutes, which
// take some 100 cycles each in the serial chain of an iteration: lane swaps for
// 32 and 16, then rotations within rows of 16 lanes and quad permutes (after
// the step of 8 the values repeat every 8 lanes, so a rotation by 4 is l ^ 4).
template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  const int b = __float_as_int(x);
  return __int_as_float(__builtin_amdgcn_update_dpp(b, b, CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float wave_sum(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(b[0]) + __uint_as_float(b[1]);
  x = x + dpp<0x128>(x);  // rotate by 8
  x = x + dpp<0x124>(x);  // rotate by 4
  x = x + dpp<0x4E>(x);   // quad 2 3 0 1
  return x + dpp<0xB1>(x);  // quad 1 0 3 2
}

// Workgroup sums of K values at once: each wavefront's sum, then the four
// wavefront sums combined as (w0 + w1) + (w2 + w3).  One barrier for all K
// sums; the order is fixed, so every workgroup gets the same result from the
// same inputs.  red holds K * kWaves floats, which another barrier must
// separate from their next use.
template <int K>
__device__ __forceinline__ void block_sums(float (&v)[K], float* red) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < K; ++q) v[q] = wave_sum(v[q]);
  if (lane == 0) {
#pragma unroll
    for (int q = 0; q < K; ++q) red[q * kWaves + wave] = v[q];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < K; ++q)
    v[q] = (red[q * kWaves] + red[q * kWaves + 1]) + (red[q * kWaves + 2] + red[q * kWaves + 3]);
}

__device__ __forceinline__ float block_sum(float v, float* red) {
  float a[1] = {v};
  block_sums<1>(a, red);
  return a[0];
}

__device__ __forceinline__ float tol2(const FvmParams& p, float bs, float rtol, float atol) {
  const float a = (rtol * rtol) * bs;
  const float b = atol * atol;
  return a > b ? a : b;
}

// Word of workgroup b's sum in copy `copy` of the sums (one copy per XCD).
__device__ __forceinline__ int sum_slot(int copy, int b) { return copy * kMaxBlocks + b; }

// This block's messages of the one-launch solve: none sent yet.
template <int N>
__device__ __forceinline__ void clear_messages(const CgBuffers& c) {
  for (int e = threadIdx.x; e < 2 * N; e += kThreads) c.msg_edge[2 * blockIdx.x * N + e] = 0;
  if (threadIdx.x < kMsgCopies) c.msg_rr[sum_slot(threadIdx.x, blockIdx.x)] = c.msg_pap[sum_slot(threadIdx.x, blockIdx.x)] = 0;
}

template <int N, int RB>
__global__ __launch_bounds__(kThreads) void cg_init(const float* __restrict__ rhs, CgBuffers c) {
  __shared__ float red[kWaves];
  const int i0 = blockIdx.x * RB;
  float rr = 0.f;
  for (int e = threadIdx.x; e < RB * N; e += kThreads) {
    const int idx = i0 * N + e;
    const float b = rhs[idx];
    c.x[idx] = 0.f;
    c.r[idx] = b - 0.f;  // r0 = b - A x0 with x0 = 0
    c.p[0][idx] = 0.f;
    rr = rr + b * b;
  }
  const float s = block_sum(rr, red);
  clear_messages<N>(c);
  if (threadIdx.x == 0) {
    c.part_rr[0][blockIdx.x] = s;
    c.part_bb[blockIdx.x] = s;
    if (blockIdx.x == 0) {
      c.status[0] = 0;
      c.status[1] = 0;
      c.status[3] = 0;  // a message of the one-launch solve did not arrive
    }
  }
}

// periodic 5-point Laplacian at (i, j) of an N x N field, summed as
// finite_differences.laplacian does (finite_differences.py:127-133)
__device__ __forceinline__ float lap5(const FvmParams& p, float centre, float up, float down, float left,
                                      float right) {
  return ((-2.f * centre) * p.lap_sum + (up + down) * p.inv_dx_sq) + (left + right) * p.inv_dy_sq;
}

// x0 = b, r0 = b - (b - coef L b), p_{-1} = 0, partial <r0, r0> and <b, b>
template <int N, int RB>
__global__ __launch_bounds__(kThreads) void cg_init_helmholtz(FvmParams p, const float* __restrict__ b,
                                                              CgBuffers c, float coef) {
  __shared__ float red[2 * kWaves];
  const int i0 = blockIdx.x * RB;
  float sums[2] = {0.f, 0.f};  // <r, r>, <b, b>
  for (int e = threadIdx.x; e < RB * N; e += kThreads) {
    const int i = i0 + e / N, j = e % N;
    const int idx = i * N + j;
    const float bc = b[idx];
    const float lap = lap5(p, bc, b[((i - 1) & (N - 1)) * N + j], b[((i + 1) & (N - 1)) * N + j],
                           b[i * N + ((j - 1) & (N - 1))], b[i * N + ((j + 1) & (N - 1))]);
    const float r = bc - (bc - coef * lap);
    c.x[idx] = bc;
    c.r[idx] = r;
    c.p[0][idx] = 0.f;
    sums[0] = sums[0] + r * r;
    sums[1] = sums[1] + bc * bc;
  }
  block_sums<2>(sums, red);
  clear_messages<N>(c);
  if (threadIdx.x == 0) {
    c.part_rr[0][blockIdx.x] = sums[0];
    c.part_bb[blockIdx.x] = sums[1];
    if (blockIdx.x == 0) {
      c.status[0] = 0;
      c.status[1] = 0;
      c.status[3] = 0;
    }
  }
}

// One direction step; HELM selects A = I - coef L over A = L.
template <int N, int RB, bool HELM>
__device__ __forceinline__ bool direction_body(const FvmParams& p, const CgBuffers& c, int k, float rtol,
                                               float atol, int maxiter, float coef, float* red,
                                               float* pt) {
  if (c.status[0]) return true;
  constexpr int NB = N / RB;
  constexpr int TOT = (RB + 2) * N, PT = (TOT + kThreads - 1) / kThreads;
  const int i0 = blockIdx.x * RB;
  const float* pold = c.p[k & 1];
  float* pnew = c.p[(k + 1) & 1];
  // r and p_{k-1} over rows i0-1 .. i0+RB, loaded before the reductions so
  // the two memory latencies overlap (indices clamped: loads unconditional)
  float rv[PT], pv[PT];
#pragma unroll
  for (int q = 0; q < PT; ++q) {
    const int e = min(static_cast<int>(threadIdx.x) + q * kThreads, TOT - 1);
    const int gi = (i0 - 1 + e / N) & (N - 1);
    rv[q] = c.r[gi * N + e % N];
    pv[q] = pold[gi * N + e % N];
  }
  // gamma_k = <r_k, r_k>, <b, b> and gamma_{k-1}, reduced together (the
  // last is unused, and part_rr of the other parity unset, at k = 0)
  float sums[3] = {0.f, 0.f, 0.f};
  for (int e = threadIdx.x; e < NB; e += kThreads) {
    sums[0] = sums[0] + c.part_rr[k & 1][e];
    sums[1] = sums[1] + c.part_bb[e];
    if (k > 0) sums[2] = sums[2] + c.part_rr[(k + 1) & 1][e];
  }
  block_sums<3>(sums, red);
  const float gamma = sums[0], bs = sums[1];
  if (!(gamma > tol2(p, bs, rtol, atol) && k < maxiter)) {
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      c.status[0] = 1;
      c.status[1] = k;
    }
    return true;
  }
  const float beta = (k == 0) ? 0.f : gamma / sums[2];
#pragma unroll
  for (int q = 0; q < PT; ++q) {
    const int e = static_cast<int>(threadIdx.x) + q * kThreads;
    if (TOT % kThreads != 0 && e >= TOT) break;
    const int lr = e / N, j = e % N;
    const int gi = (i0 - 1 + lr) & (N - 1);
    const float v = rv[q] + beta * pv[q];
    pt[e] = v;
    if (lr >= 1 && lr <= RB) pnew[gi * N + j] = v;
  }
  __syncthreads();
  float pap = 0.f;
  for (int e = threadIdx.x; e < RB * N; e += kThreads) {
    const int r = e / N, j = e % N;
    const float* row = pt + (r + 1) * N;
    const float pc = row[j];
    const float lap = lap5(p, pc, row[j - N], row[j + N], row[(j - 1) & (N - 1)], row[(j + 1) & (N - 1)]);
    const float ap = HELM ? pc - coef * lap : lap;
    c.ap[(i0 + r) * N + j] = ap;
    pap = pap + pc * ap;
  }
  const float s = block_sum(pap, red + 3 * kWaves);
  if (threadIdx.x == 0) c.part_pap[blockIdx.x] = s;
  return false;
}

template <int N, int RB>
__global__ __launch_bounds__(kThreads) void cg_direction(FvmParams p, CgBuffers c, int k, float rtol,
                                                         float atol, int maxiter) {
  __shared__ float red[4 * kWaves];
  __shared__ float pt[(RB + 2) * N];  // p_k rows i0-1 .. i0+RB
  direction_body<N, RB, false>(p, c, k, rtol, atol, maxiter, 0.f, red, pt);
}

template <int N, int RB>
__global__ __launch_bounds__(kThreads) void cg_direction_helmholtz(FvmParams p, CgBuffers c, int k,
                                                                   float rtol, float atol, int maxiter,
                                                                   float coef) {
  __shared__ float red[4 * kWaves];
  __shared__ float pt[(RB + 2) * N];
  direction_body<N, RB, true>(p, c, k, rtol, atol, maxiter, coef, red, pt);
}

template <int N, int RB>
__device__ __forceinline__ void update_body(const CgBuffers& c, int k, float* red) {
  constexpr int NB = N / RB;
  constexpr int TOT = RB * N, PU = (TOT + kThreads - 1) / kThreads;
  const int i0 = blockIdx.x * RB;
  const float* pk = c.p[(k + 1) & 1];
  // this block's x, p_k, r, Ap, loaded before the reductions (clamped)
  float xv[PU], pv[PU], rv[PU], av[PU];
#pragma unroll
  for (int q = 0; q < PU; ++q) {
    const int idx = i0 * N + min(static_cast<int>(threadIdx.x) + q * kThreads, TOT - 1);
    xv[q] = c.x[idx];
    pv[q] = pk[idx];
    rv[q] = c.r[idx];
    av[q] = c.ap[idx];
  }
  float sums[2] = {0.f, 0.f};  // gamma_k, <p, Ap>
  for (int e = threadIdx.x; e < NB; e += kThreads) {
    sums[0] = sums[0] + c.part_rr[k & 1][e];
    sums[1] = sums[1] + c.part_pap[e];
  }
  block_sums<2>(sums, red);
  const float alpha = sums[0] / sums[1];
  float rr = 0.f;
#pragma unroll
  for (int q = 0; q < PU; ++q) {
    const int e = static_cast<int>(threadIdx.x) + q * kThreads;
    if (TOT % kThreads != 0 && e >= TOT) break;
    const int idx = i0 * N + e;
    c.x[idx] = xv[q] + alpha * pv[q];
    const float rn = rv[q] - alpha * av[q];
    c.r[idx] = rn;
    rr = rr + rn * rn;
  }
  const float s = block_sum(rr, red + 2 * kWaves);
  if (threadIdx.x == 0) c.part_rr[(k + 1) & 1][blockIdx.x] = s;
}

template <int N, int RB>
__global__ __launch_bounds__(kThreads) void cg_update(CgBuffers c, int k) {
  __shared__ float red[3 * kWaves];
  if (c.status[0]) return;
  update_body<N, RB>(c, k, red);
}

// Messages of the one-launch solve: a float and the iteration it belongs to
// in one 64-bit word, written and read as relaxed agent-scope atomics.  Value
// and tag arrive together, so a reader that sees the tag has the value and
// nothing needs a fence: no cache is written back or invalidated.  The tags of
// a solve are 1, 2, ..; cg_init clears the words.
__device__ __forceinline__ void send(unsigned long long* m, int tag, float x) {
  __hip_atomic_store(m, (static_cast<unsigned long long>(static_cast<unsigned>(tag)) << 32) | __float_as_uint(x),
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until all K messages carry `tag`; their values into x.  Bounded: false
// after `polls` polls, so a launch whose workgroups do not all run ends (0: one
// poll that no message satisfies).
template <int K>
__device__ __forceinline__ bool receive(unsigned long long* const (&m)[K], int tag, float (&x)[K], int polls) {
  const unsigned want = polls > 0 ? static_cast<unsigned>(tag) : ~0u;
  bool all;
  unsigned left = polls;
  do {
    unsigned long long w[K];
    all = true;
#pragma unroll
    for (int q = 0; q < K; ++q) w[q] = __hip_atomic_load(m[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int q = 0; q < K; ++q) {
      all = all && static_cast<unsigned>(w[q] >> 32) == want;
      x[q] = __uint_as_float(static_cast<unsigned>(w[q]));
    }
  } while (!all && left-- != 0);
  return all;
}

// The whole solve in one cooperative launch (every workgroup resident at
// once).  A workgroup keeps its rows of x, r, p and the rows of r and p beside
// them in registers; per iteration it exchanges two sums with every other
// workgroup (<p, Ap>, then <r, r>) and the edge rows of r with its neighbours.
// Every workgroup adds the same sums in the same order, so all of them stop at
// the same iteration, and each sum and update has the order of the
// two-kernel form: results are bitwise the same.
//
// One buffer per message suffices: a workgroup sends message k + 1 of a kind
// only after it has every workgroup's message of the other kind that was
// sent after they read message k.
//
// What bounds it is the way of two messages through memory per iteration,
// about 1.5 us each.  The words of the sums are read by every workgroup: each
// is sent in 8 copies, one for the workgroups of each XCD (workgroups go to the
// XCDs in turn), as the readers of one word wait for each other (us per solve
// of 468 iterations at 256^2 with 1 / 4 / 8 / 16 / 64 copies: 2255 / 1855 / 1780
// / 1968 / 2327).  us per solve, two kernels per iteration / one launch: 64^2
// 946 / 395 (117 iterations), 256^2 3600 / 1780 (468), 512^2 7720 / 4700 (943),
// 1024^2 22470 / 11370 (1904).  With a counter and fences as grid barrier in
// place of the messages an iteration took 21.7 us at 256^2.
template <int N, int RB, bool HELM>
__global__ __launch_bounds__(kThreads) void cg_persistent(FvmParams p, CgBuffers c, float rtol, float atol,
                                                          int maxiter, float coef, int polls) {
  constexpr int NB = N / RB, TOT = RB * N;
  constexpr int PU = (TOT + kThreads - 1) / kThreads;    // cells per thread
  constexpr int PH = (2 * N + kThreads - 1) / kThreads;  // neighbour cells per thread: rows i0 - 1 and i0 + RB
  static_assert(NB <= kThreads && NB <= kMaxBlocks, "one message of each workgroup per thread");
  __shared__ float red[5 * kWaves];  // one area per sum of an iteration
  __shared__ float pt[(RB + 2) * N];  // p_k rows i0-1 .. i0+RB
  __shared__ int s_fail;
  const int tid = threadIdx.x, blk = blockIdx.x, i0 = blk * RB;
  // edge rows of block b: first row at 2 b, last row at 2 b + 1 (one row: the first)
  auto edge = [&](int b, int last, int j) { return c.msg_edge + ((2 * b + (RB > 1 ? last : 0)) * N + j); };
  float x[PU], rv[PU], pv[PU], av[PU], hr[PH], hp[PH];
  unsigned long long* from[1 + PH];  // this thread's messages: a workgroup's sum, neighbour cells
  unsigned long long* pap_from[1] = {c.msg_pap + sum_slot(blk % kMsgCopies, tid < NB ? tid : NB - 1)};
  from[0] = c.msg_rr + sum_slot(blk % kMsgCopies, tid < NB ? tid : NB - 1);
#pragma unroll
  for (int q = 0; q < PU; ++q) {
    const int e = min(tid + q * kThreads, TOT - 1);
    x[q] = c.x[i0 * N + e];
    rv[q] = c.r[i0 * N + e];
    pv[q] = 0.f;
    av[q] = 0.f;
  }
#pragma unroll
  for (int q = 0; q < PH; ++q) {
    const int e = min(tid + q * kThreads, 2 * N - 1), below = e / N, j = e % N;
    const int gi = (below ? i0 + RB : i0 - 1) & (N - 1);
    hr[q] = c.r[gi * N + j];
    hp[q] = 0.f;
    from[1 + q] = edge((below ? blk + 1 : blk + NB - 1) % NB, !below, j);
  }
  if (tid == 0) s_fail = 0;
  __syncthreads();
  float gamma = 0.f, gamma_prev = 0.f, limit = 0.f;
  bool done = false;
  for (int k = 0;; ++k) {
    // gamma_k = <r_k, r_k> (and <b, b>, once)
    if (k == 0) {
      float sums[2] = {0.f, 0.f};
      if (tid < NB) {
        sums[0] = sums[0] + c.part_rr[0][tid];
        sums[1] = sums[1] + c.part_bb[tid];
      }
      block_sums<2>(sums, red);
      gamma = sums[0];
      limit = tol2(p, sums[1], rtol, atol);
    } else {
      float in[1 + PH];
      if (!receive(from, k, in, polls)) s_fail = 1;
#pragma unroll
      for (int q = 0; q < PH; ++q) hr[q] = in[1 + q];
      float sums[1] = {0.f};
      if (tid < NB) sums[0] = sums[0] + in[0];
      block_sums<1>(sums, red);
      if (s_fail) break;
      gamma = sums[0];
    }
    if (!(gamma > limit && k < maxiter)) {
      done = true;
      if (blk == 0 && tid == 0) {
        c.status[0] = 1;
        c.status[1] = k;
      }
      break;
    }
    const float beta = (k == 0) ? 0.f : gamma / gamma_prev;
    gamma_prev = gamma;
#pragma unroll
    for (int q = 0; q < PU; ++q) {
      const int e = tid + q * kThreads;
      pv[q] = rv[q] + beta * pv[q];
      if (TOT % kThreads == 0 || e < TOT) pt[N + e] = pv[q];
    }
#pragma unroll
    for (int q = 0; q < PH; ++q) {
      const int e = tid + q * kThreads;
      hp[q] = hr[q] + beta * hp[q];
      if (2 * N % kThreads == 0 || e < 2 * N) pt[(e / N ? (RB + 1) * N : 0) + e % N] = hp[q];
    }
    __syncthreads();
    float pap = 0.f;
#pragma unroll
    for (int q = 0; q < PU; ++q) {
      const int e = tid + q * kThreads;
      if (TOT % kThreads != 0 && e >= TOT) break;
      const int j = e % N;
      const float* row = pt + (e / N + 1) * N;
      const float pc = row[j];
      const float lap = lap5(p, pc, row[j - N], row[j + N], row[(j - 1) & (N - 1)], row[(j + 1) & (N - 1)]);
      av[q] = HELM ? pc - coef * lap : lap;
      pap = pap + pc * av[q];
    }
    const float mine = block_sum(pap, red + 2 * kWaves);
    if (tid < kMsgCopies) send(c.msg_pap + sum_slot(tid, blk), k + 1, mine);
    float in[1];
    if (!receive(pap_from, k + 1, in, polls)) s_fail = 1;
    float sums[1] = {0.f};
    if (tid < NB) sums[0] = sums[0] + in[0];
    block_sums<1>(sums, red + 3 * kWaves);
    if (s_fail) break;
    const float alpha = gamma / sums[0];
    float rr = 0.f;
#pragma unroll
    for (int q = 0; q < PU; ++q) {
      const int e = tid + q * kThreads;
      if (TOT % kThreads != 0 && e >= TOT) break;
      x[q] = x[q] + alpha * pv[q];
      rv[q] = rv[q] - alpha * av[q];
      rr = rr + rv[q] * rv[q];
      if (e < N) send(edge(blk, 0, e), k + 1, rv[q]);
      if (RB > 1 && e >= (RB - 1) * N) send(edge(blk, 1, e - (RB - 1) * N), k + 1, rv[q]);
    }
    const float next = block_sum(rr, red + 4 * kWaves);
    if (tid < kMsgCopies) send(c.msg_rr + sum_slot(tid, blk), k + 1, next);
  }
  if (!done) {
    if (tid == 0) __hip_atomic_store(&c.status[3], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return;
  }
#pragma unroll
  for (int q = 0; q < PU; ++q) {
    const int e = tid + q * kThreads;
    if (TOT % kThreads == 0 || e < TOT) c.x[i0 * N + e] = x[q];
  }
}

template <int N> struct CgRows { static constexpr int RB = N >= 512 ? N / 256 : 1; };

template <int N>
struct CgOps {
  static constexpr int RB = CgRows<N>::RB;
  static int init(const float* rhs, const CgBuffers& c, hipStream_t s) {
    hipLaunchKernelGGL((cg_init<N, RB>), dim3(N / RB), dim3(kThreads), 0, s, rhs, c);
    return check_hip(hipGetLastError(), "cg_init");
  }
  static int iteration(const FvmParams& p, const CgBuffers& c, int k, float rtol, float atol,
                       int maxiter, hipStream_t s) {
    hipLaunchKernelGGL((cg_direction<N, RB>), dim3(N / RB), dim3(kThreads), 0, s, p, c, k, rtol,
                       atol, maxiter);
    hipLaunchKernelGGL((cg_update<N, RB>), dim3(N / RB), dim3(kThreads), 0, s, c, k);
    return check_hip(hipGetLastError(), "cg iteration");
  }
  static int init_helmholtz(const FvmParams& p, const float* b, const CgBuffers& c, float coef,
                            hipStream_t s) {
    hipLaunchKernelGGL((cg_init_helmholtz<N, RB>), dim3(N / RB), dim3(kThreads), 0, s, p, b, c, coef);
    return check_hip(hipGetLastError(), "cg_init_helmholtz");
  }
  // The whole solve as one cooperative launch (N / RB workgroups, all
  // resident).  JCFD_ERR_UNSUPPORTED when the device cannot hold them or
  // refuses the launch.
  static int persistent(const FvmParams& p, const CgBuffers& c, float rtol, float atol, int maxiter,
                        bool helm, float coef, int polls, hipStream_t s) {
    const void* fn = helm ? reinterpret_cast<const void*>(&cg_persistent<N, RB, true>)
                          : reinterpret_cast<const void*>(&cg_persistent<N, RB, false>);
    int dev = 0, coop = 0, cus = 0, per_cu = 0, rc;
    if ((rc = check_hip(hipGetDevice(&dev), "hipGetDevice")) ||
        (rc = check_hip(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev),
                        "cooperative launch attribute")) ||
        (rc = check_hip(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev), "CU count")) ||
        (rc = check_hip(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, kThreads, 0), "occupancy")))
      return rc;
    if (!coop || per_cu * cus < N / RB) return JCFD_ERR_UNSUPPORTED;
    FvmParams pp = p;
    CgBuffers cc = c;
    void* args[] = {&pp, &cc, &rtol, &atol, &maxiter, &coef, &polls};
    if (hipLaunchCooperativeKernel(fn, dim3(N / RB), dim3(kThreads), args, 0, s) == hipSuccess) return JCFD_OK;
    (void)hipGetLastError();  // nothing was launched: the caller's other form reports what is wrong, if it persists
    return JCFD_ERR_UNSUPPORTED;
  }
  static int iteration_helmholtz(const FvmParams& p, const CgBuffers& c, int k, float rtol, float atol,
                                 int maxiter, float coef, hipStream_t s) {
    hipLaunchKernelGGL((cg_direction_helmholtz<N, RB>), dim3(N / RB), dim3(kThreads), 0, s, p, c, k,
                       rtol, atol, maxiter, coef);
    hipLaunchKernelGGL((cg_update<N, RB>), dim3(N / RB), dim3(kThreads), 0, s, c, k);
    return check_hip(hipGetLastError(), "cg helmholtz iteration");
  }
};

}  // namespace

int cg_blocks(int n) { return n >= 512 ? kMaxBlocks : n; }
int cg_sum_messages() { return kMsgCopies * kMaxBlocks; }

int cg_launch_init(const FvmParams& p, const float* rhs, const CgBuffers& c, float, float, int,
                   hipStream_t s) {
  switch (p.n) {
    case 32: return CgOps<32>::init(rhs, c, s);
    case 64: return CgOps<64>::init(rhs, c, s);
    case 128: return CgOps<128>::init(rhs, c, s);
    case 256: return CgOps<256>::init(rhs, c, s);
    case 512: return CgOps<512>::init(rhs, c, s);
    case 1024: return CgOps<1024>::init(rhs, c, s);
    default: return fail(JCFD_ERR_UNSUPPORTED, "CG grid size not built");
  }
}

int cg_launch_iteration(const FvmParams& p, const CgBuffers& c, int k, float rtol, float atol,
                        int maxiter, hipStream_t s) {
  switch (p.n) {
    case 32: return CgOps<32>::iteration(p, c, k, rtol, atol, maxiter, s);
    case 64: return CgOps<64>::iteration(p, c, k, rtol, atol, maxiter, s);
    case 128: return CgOps<128>::iteration(p, c, k, rtol, atol, maxiter, s);
    case 256: return CgOps<256>::iteration(p, c, k, rtol, atol, maxiter, s);
    case 512: return CgOps<512>::iteration(p, c, k, rtol, atol, maxiter, s);
    case 1024: return CgOps<1024>::iteration(p, c, k, rtol, atol, maxiter, s);
    default: return fail(JCFD_ERR_UNSUPPORTED, "CG grid size not built");
  }
}

int cg_launch_persistent(const FvmParams& p, const CgBuffers& c, float rtol, float atol, int maxiter,
                         bool helm, float coef, int polls, hipStream_t s) {
  switch (p.n) {
    case 32: return CgOps<32>::persistent(p, c, rtol, atol, maxiter, helm, coef, polls, s);
    case 64: return CgOps<64>::persistent(p, c, rtol, atol, maxiter, helm, coef, polls, s);
    case 128: return CgOps<128>::persistent(p, c, rtol, atol, maxiter, helm, coef, polls, s);
    case 256: return CgOps<256>::persistent(p, c, rtol, atol, maxiter, helm, coef, polls, s);
    case 512: return CgOps<512>::persistent(p, c, rtol, atol, maxiter, helm, coef, polls, s);
    case 1024: return CgOps<1024>::persistent(p, c, rtol, atol, maxiter, helm, coef, polls, s);
    default: return fail(JCFD_ERR_UNSUPPORTED, "CG grid size not built");
  }
}

int cg_launch_init_helmholtz(const FvmParams& p, const float* b, const CgBuffers& c, float coef,
                             hipStream_t s) {
  switch (p.n) {
    case 32: return CgOps<32>::init_helmholtz(p, b, c, coef, s);
    case 64: return CgOps<64>::init_helmholtz(p, b, c, coef, s);
    case 128: return CgOps<128>::init_helmholtz(p, b, c, coef, s);
    case 256: return CgOps<256>::init_helmholtz(p, b, c, coef, s);
    case 512: return CgOps<512>::init_helmholtz(p, b, c, coef, s);
    case 1024: return CgOps<1024>::init_helmholtz(p, b, c, coef, s);
    default: return fail(JCFD_ERR_UNSUPPORTED, "CG grid size not built");
  }
}

int cg_launch_iteration_helmholtz(const FvmParams& p, const CgBuffers& c, int k, float rtol, float atol,
                                  int maxiter, float coef, hipStream_t s) {
  switch (p.n) {
    case 32: return CgOps<32>::iteration_helmholtz(p, c, k, rtol, atol, maxiter, coef, s);
    case 64: return CgOps<64>::iteration_helmholtz(p, c, k, rtol, atol, maxiter, coef, s);
    case 128: return CgOps<128>::iteration_helmholtz(p, c, k, rtol, atol, maxiter, coef, s);
    case 256: return CgOps<256>::iteration_helmholtz(p, c, k, rtol, atol, maxiter, coef, s);
    case 512: return CgOps<512>::iteration_helmholtz(p, c, k, rtol, atol, maxiter, coef, s);
    case 1024: return CgOps<1024>::iteration_helmholtz(p, c, k, rtol, atol, maxiter, coef, s);
    default: return fail(JCFD_ERR_UNSUPPORTED, "CG grid size not built");
  }
}

}  // namespace jcfd
