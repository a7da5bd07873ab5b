// F32 matvec and RMSNorm kernels: the GGUF F32 tensors and the norms around
// the K-quant projections of a decoder block (si_f32_matvec, metal.rs:263-305;
// si_rms_norm / si_rms_norm_heads / si_rms_norm_gated, metal.rs:121-213).
//
// Both are bound by latency at the sizes a decoder block has (a few dozen
// rows; one vector): what counts is how many dependent trips to memory a
// launch makes.  So each thread has all its loads out before it uses the
// first: a row of the matvec goes to as many waves as keep the chip busy, and
// an RMSNorm head is held in registers, with its weight (and gate) loaded
// beside it, between the sum of squares and the scaled output.
#include "si_hip_internal.h"

namespace sihip {
namespace {

// Sum over the 64 lanes of a wave, in a fixed order, broadcast to all lanes:
// each 16-lane row by DPP shifts (lane 15 of the row ends with the row's
// sum), then the four rows' sums added in row order.
__device__ __forceinline__ float wave_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x111, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x112, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x114, 0xf, 0xf, true));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x118, 0xf, 0xf, true));
  const float r0 = __shfl(v, 15, 64), r1 = __shfl(v, 31, 64);
  const float r2 = __shfl(v, 47, 64), r3 = __shfl(v, 63, 64);
  return (r0 + r1) + (r2 + r3);
}

// A float or a float4 by index, and its dot with another added to an accumulator.
__device__ __forceinline__ void fma_unit(float p, float q, float& a) { a = fmaf(p, q, a); }
__device__ __forceinline__ void fma_unit(const float4& p, const float4& q, float& a) {
  a = fmaf(p.x, q.x, a);
  a = fmaf(p.y, q.y, a);
  a = fmaf(p.z, q.z, a);
  a = fmaf(p.w, q.w, a);
}
__device__ __forceinline__ void clear(float& p) { p = 0.0f; }
__device__ __forceinline__ void clear(float4& p) { p = make_float4(0.0f, 0.0f, 0.0f, 0.0f); }

// y[r] = sum_c w[r * cols + c] * x[c], WPR waves per row: thread t of the
// row's 64 WPR takes units t, t + 64 WPR, ... of the row's n (a unit is a
// float4 where cols % 4 == 0 and w, x are 16-byte aligned, else a float),
// FLIGHT (1, 2 or 8) at a time with all their loads in flight, in two
// accumulators; then the waves' sums are added in wave order.  One wave a row and
// two loads in flight took 48 x 5120 (the gates beside a block's norm) 5.0 us, a
// row's ten dependent trips to memory; sixteen waves a row, two loads a thread,
// 2.0 us.
template <typename U, int WPR, int FLIGHT>
__global__ __launch_bounds__(WPR > 4 ? 64 * WPR : 256) void f32_matvec_kernel(
    const float* __restrict__ w, const float* __restrict__ x, float* __restrict__ y,
    uint32_t rows, uint32_t cols) {
  constexpr uint32_t kRows = WPR > 4 ? 1u : 4u / WPR;  // rows per workgroup
  constexpr uint32_t kStep = 64u * WPR;
  __shared__ float red[WPR > 4 ? WPR : 4];
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
  const uint32_t row = blockIdx.x * kRows + wave / WPR;
  float total = 0.0f;
  if (row < rows) {  // whole waves
    const U* const wr = reinterpret_cast<const U*>(w + (size_t)row * cols);
    const U* const xr = reinterpret_cast<const U*>(x);
    const uint32_t n = cols / (uint32_t)(sizeof(U) / sizeof(float));
    float a0 = 0.0f, a1 = 0.0f;
    for (size_t i = (wave % WPR) * 64u + lane; i < n; i += FLIGHT * kStep) {
      U p[FLIGHT], q[FLIGHT];
#pragma unroll
      for (int k = 0; k < FLIGHT; ++k) {
        const size_t j = i + (uint32_t)k * kStep;
        clear(p[k]);
        clear(q[k]);
        if (j < n) {
          p[k] = wr[j];
          q[k] = xr[j];
        }
      }
#pragma unroll
      for (int k = 0; k < FLIGHT; ++k) fma_unit(p[k], q[k], (k & 1) ? a1 : a0);
    }
    total = wave_sum(a0 + a1);
  }
  if constexpr (WPR > 1) {
    if (lane == 0u) red[wave] = total;
    __syncthreads();
    if (row < rows && wave % WPR == 0u && lane == 0u) {
      for (int k = 1; k < WPR; ++k) total += red[wave + k];
      y[row] = total;
    }
  } else if (row < rows && lane == 0u) {
    y[row] = total;
  }
}

// The workgroup's sum of per-wave partials, in wave order, in every thread (at
// most 16 waves; the slots of waves it does not have hold zero, so that all the
// reads go out at once).
__device__ __forceinline__ float group_sum(float v, float4 (&red)[4]) {
  const uint32_t wave = threadIdx.x >> 6, lane = threadIdx.x & 63u, waves = blockDim.x >> 6;
  v = wave_sum(v);
  float* const slot = reinterpret_cast<float*>(red);
  if (lane == 0u) slot[wave] = v;
  if (wave == 0u && lane >= waves && lane < 16u) slot[lane] = 0.0f;
  __syncthreads();
  const float4 a = red[0];
  float t = ((a.x + a.y) + a.z) + a.w;
  if (waves > 4u) {
    const float4 b = red[1], c = red[2], d = red[3];
    t = (((t + b.x) + b.y) + b.z) + b.w;
    t = (((t + c.x) + c.y) + c.z) + c.w;
    t = (((t + d.x) + d.y) + d.z) + d.w;
  }
  return t;
}

__device__ __forceinline__ void add_square(float v, float& s) {
  s = __fadd_rn(s, __fmul_rn(v, v));  // x^2 rounded, then added (qwen35.rs:36-40)
}
__device__ __forceinline__ void add_square(const float4& v, float& s) {
  add_square(v.x, s);
  add_square(v.y, s);
  add_square(v.z, s);
  add_square(v.w, s);
}
// MODE 0: x * inv * w (si_rms_norm); 1: x * inv * (1 + w) (si_rms_norm_heads);
// 2: x * inv * w * silu(g) (si_rms_norm_gated).
template <int MODE>
__device__ __forceinline__ float norm_out(float x, float inv, float w, float g) {
  const float o = __fmul_rn(x, inv);
  if (MODE == 0) return __fmul_rn(o, w);
  if (MODE == 1) return __fmul_rn(o, __fadd_rn(1.0f, w));
  return __fmul_rn(__fmul_rn(o, w), __fdiv_rn(g, __fadd_rn(1.0f, expf(-g))));
}
template <int MODE>
__device__ __forceinline__ float4 norm_out(const float4& x, float inv, const float4& w,
                                           const float4& g) {
  return make_float4(norm_out<MODE>(x.x, inv, w.x, g.x), norm_out<MODE>(x.y, inv, w.y, g.y),
                     norm_out<MODE>(x.z, inv, w.z, g.z), norm_out<MODE>(x.w, inv, w.w, g.w));
}

// One workgroup per head of head_dim values, UPT units (float4s where the
// pointers and head_dim allow, else floats) of it per thread and pass: with
// one pass (blockDim.x * UPT units) the head, its weight and its gate are
// loaded at once and kept in registers between the two phases; longer heads
// go through memory twice, UPT loads in flight.  A head of 5120 took 11 us as
// 20 dependent loads a thread twice over; 640 threads of two float4s 2.2 us
// (18.8 and 4.9 us where x and w come from HBM).
template <int MODE, typename U, int UPT>
__global__ __launch_bounds__(1024) void rms_norm_kernel(const float* __restrict__ x,
                                                        const float* __restrict__ gate,
                                                        const float* __restrict__ w,
                                                        float* __restrict__ y, uint32_t head_dim,
                                                        float eps) {
  __shared__ float4 red[4];
  const size_t base = (size_t)blockIdx.x * head_dim;
  const U* const xu = reinterpret_cast<const U*>(x + base);
  const U* const gu = reinterpret_cast<const U*>(MODE == 2 ? gate + base : x + base);
  const U* const wu = reinterpret_cast<const U*>(w);
  U* const yu = reinterpret_cast<U*>(y + base);
  const uint32_t n = head_dim / (uint32_t)(sizeof(U) / sizeof(float));
  const uint32_t step = blockDim.x, pass = step * UPT;
  U xv[UPT], wv[UPT], gv[UPT];
  auto load = [&](size_t i0, bool all) {
#pragma unroll
    for (int k = 0; k < UPT; ++k) {
      const size_t i = i0 + (uint32_t)k * step;
      clear(xv[k]);
      clear(wv[k]);
      clear(gv[k]);
      if (i < n) {
        xv[k] = xu[i];
        if (all) {
          wv[k] = wu[i];
          if (MODE == 2) gv[k] = gu[i];
        }
      }
    }
  };
  const bool held = n <= pass;
  float ss = 0.0f;
  for (size_t i0 = threadIdx.x; i0 < n; i0 += pass) {
    load(i0, held);
#pragma unroll
    for (int k = 0; k < UPT; ++k) add_square(xv[k], ss);  // (zeros past the head)
  }
  const float total = group_sum(ss, red);
  // (sum / n + eps).sqrt().recip(), each step correctly rounded
  const float inv = __fdiv_rn(1.0f, __fsqrt_rn(__fadd_rn(__fdiv_rn(total, (float)head_dim), eps)));
  for (size_t i0 = threadIdx.x; i0 < n; i0 += pass) {
    if (!held) load(i0, true);
#pragma unroll
    for (int k = 0; k < UPT; ++k) {
      const size_t i = i0 + (uint32_t)k * step;
      if (i < n) yu[i] = norm_out<MODE>(xv[k], inv, wv[k], gv[k]);
    }
  }
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0u; }

// Rows that give each thread at most one or two units take the kernel with as
// many loads unrolled: the code of eight alone costs such a launch 0.1-1.4 us
// (64 x 24 3.06 us with eight, 2.64 with one; 20000 x 128 5.17, 3.77; 6600 x 512
// 3.70 with eight, 3.42 with two).
template <typename U, int WPR>
void launch_matvec_as(const float* w, const float* x, float* y, uint32_t rows, uint32_t cols,
                      hipStream_t s) {
  constexpr uint32_t kRows = WPR > 4 ? 1u : 4u / WPR;
  const dim3 grid((rows + kRows - 1u) / kRows), block(WPR > 4 ? 64 * WPR : 256);
  const uint32_t n = cols / (uint32_t)(sizeof(U) / sizeof(float));
  if (n <= 64u * WPR)
    hipLaunchKernelGGL((f32_matvec_kernel<U, WPR, 1>), grid, block, 0, s, w, x, y, rows, cols);
  else if (n <= 128u * WPR)
    hipLaunchKernelGGL((f32_matvec_kernel<U, WPR, 2>), grid, block, 0, s, w, x, y, rows, cols);
  else
    hipLaunchKernelGGL((f32_matvec_kernel<U, WPR, 8>), grid, block, 0, s, w, x, y, rows, cols);
}
// Waves per row: as many (up to 16) as give the row's waves a unit each while
// all rows' waves stay within eight a CU (2048), else one.
template <typename U>
void launch_matvec_units(const float* w, const float* x, float* y, uint32_t rows, uint32_t cols,
                         hipStream_t s) {
  const uint32_t n = cols / (uint32_t)(sizeof(U) / sizeof(float));
  uint32_t wpr = 1u;
  while (wpr < 16u && 64u * wpr < n && (uint64_t)rows * wpr * 2u <= 2048u) wpr *= 2u;
  switch (wpr) {
    case 1: return launch_matvec_as<U, 1>(w, x, y, rows, cols, s);
    case 2: return launch_matvec_as<U, 2>(w, x, y, rows, cols, s);
    case 4: return launch_matvec_as<U, 4>(w, x, y, rows, cols, s);
    case 8: return launch_matvec_as<U, 8>(w, x, y, rows, cols, s);
    default: return launch_matvec_as<U, 16>(w, x, y, rows, cols, s);
  }
}

constexpr uint64_t kManyThreads = 256u * 1024u;

template <int MODE, typename U>
void launch_norm_units(const float* x, const float* gate, const float* w, float* y,
                       uint32_t heads, uint32_t head_dim, float eps, hipStream_t s) {
  // the fewest units a thread that hold the head with at most 1024 threads
  const uint32_t n = head_dim / (uint32_t)(sizeof(U) / sizeof(float));
  auto threads = [&](uint32_t upt) {
    return (uint32_t)min((uint64_t)1024u, (((uint64_t)n + upt - 1u) / upt + 63u) / 64u * 64u);
  };
  auto launch = [&](auto upt, auto kernel) {
    // (a launch takes less than 2^32 threads: more heads run as several)
    const uint32_t t = threads(upt), most = 0xffffffffu / t;
    for (uint32_t h0 = 0; h0 < heads; h0 += min(most, heads - h0)) {
      const size_t at = (size_t)h0 * head_dim;
      hipLaunchKernelGGL(kernel, dim3(min(most, heads - h0)), dim3(t), 0, s, x + at,
                         gate ? gate + at : nullptr, w, y + at, head_dim, eps);
    }
  };
  uint32_t upt = n <= 1024u ? 1u : n <= 2048u ? 2u : 4u;
  // More where single floats would take more threads than 1024 a CU of 256: a
  // workgroup's waves cost more than the loads they hide (4000 x 1001 13.6 us with
  // one, 7.0 with four; 4000 x 2001 17.1 with two, 12.0 with four; 256 x 1001 2.84
  // with one, 2.72 with four).  Of float4s the first choice stays ahead to 20000 x
  // 1000.
  if (sizeof(U) == sizeof(float))
    while (upt < 4u && threads(upt) > 64u && (uint64_t)heads * threads(upt) > kManyThreads)
      upt *= 2u;
  if (upt == 1u)
    launch(1u, &rms_norm_kernel<MODE, U, 1>);
  else if (upt == 2u)
    launch(2u, &rms_norm_kernel<MODE, U, 2>);
  else
    launch(4u, &rms_norm_kernel<MODE, U, 4>);
}

template <int MODE>
void launch_norm_mode(const float* x, const float* gate, const float* w, float* y, uint32_t heads,
                      uint32_t head_dim, float eps, hipStream_t s) {
  // Short heads in a float a thread while the card holds all of them at once: a
  // thread's four outputs, above all their four gates, cost more than its wider
  // loads save (48 x 128 gated 2.54 us in float4s, 2.34 in floats, 256 x 64 2.59, 2.33,
  // 256 x 512 the same; 4000 x 256 3.87, 4.63; 48 x 128 without a gate 2.36, 2.29).
  const bool narrow = head_dim <= (MODE == 2 ? 512u : 128u) &&
                      (uint64_t)heads * head_dim <= kManyThreads;
  const bool vec = !narrow && head_dim % 4u == 0u && aligned16(x) && aligned16(w) &&
                   aligned16(y) && (MODE != 2 || aligned16(gate));
  if (vec)
    launch_norm_units<MODE, float4>(x, gate, w, y, heads, head_dim, eps, s);
  else
    launch_norm_units<MODE, float>(x, gate, w, y, heads, head_dim, eps, s);
}

}  // namespace

hipError_t launch_f32_matvec(const float* w, const float* x, float* y, uint32_t rows,
                             uint32_t cols, hipStream_t s) {
  if (rows == 0 || cols == 0) return hipErrorInvalidValue;
  if (cols % 4u == 0u && aligned16(w) && aligned16(x))
    launch_matvec_units<float4>(w, x, y, rows, cols, s);
  else
    launch_matvec_units<float>(w, x, y, rows, cols, s);
  return hipGetLastError();
}

hipError_t launch_rms_norm(uint32_t mode, const float* x, const float* gate, const float* w,
                           float* y, uint32_t heads, uint32_t head_dim, float eps, hipStream_t s) {
  if (heads == 0 || head_dim == 0 || mode > 2u) return hipErrorInvalidValue;
  switch (mode) {
    case 0: launch_norm_mode<0>(x, gate, w, y, heads, head_dim, eps, s); break;
    case 1: launch_norm_mode<1>(x, gate, w, y, heads, head_dim, eps, s); break;
    default: launch_norm_mode<2>(x, gate, w, y, heads, head_dim, eps, s); break;
  }
  return hipGetLastError();
}

}  // namespace sihip
