// Shared parts of the kernels that put several activation vectors in the
// rows of the matrix-core A operand (q45_tokens_mfma, q6k_tokens_mfma): the
// group images of four vectors at a time, built in LDS, and the reduce kernel
// that adds the K slices' partial sums of a sliced launch in slice order.
//
// Group images: four vectors of four digits in the 16 A rows of
// v_mfma_i32_16x16x64_i8 (lane 16 k + 4 t + d: digit d of vector t over the 16
// elements that meet lane group k's weights).  A block is four MFMAs j, 1 KB
// each; chunk c (elements 16 c .. 16 c + 15) is at the offset a format's map
// gives, 1024 j + 256 k.
#pragma once

#include "mfma_common.h"

namespace sihip {
namespace mfma {
namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
// A plain LDS read, its wait placed by the compiler, which also waits there for
// the buffer->LDS copies in flight: only for reads before the stage loop
// (slice_err, once a launch and group).
__device__ __forceinline__ u32x4 lds_u32x4(const uint8_t* p) {
  return *(const __attribute__((address_space(3))) u32x4*)p;
}
__device__ __forceinline__ void lds_write_b16(uint32_t addr, uint32_t v) {
  asm volatile("ds_write_b16 %0, %1" : : "v"(addr), "v"(v) : "memory");
}

// The exponent slot of a block that takes the exact path: scaling by it gives
// zero.
constexpr int kBadTok = -(1 << 20);

// What a vector's side elements (mfma_common.h) may cost its dot with a row
// over a slice: 2^-21 of the row's sum |block term| where no block has more
// than eight of them, which is what the f32 rounding of such terms was bounded
// by (they are f64 here), and kRoundedTol of it for the blocks that have
// more.  A (vector, row) past that takes the slice's exact dot.  (Up to eight
// per block used to be listed and added from the exact weights; held to
// kRoundedTol like the rest, a dot that rides on them was up to 7.6e-6 off.)
// Slices of ordinary activations reach 1e-8 of the sum.
constexpr uint32_t kFewSide = 8;
constexpr float kFewTol = 0x1p-21f;

// First block of K slice k of rows of nb blocks: slices of four, the last of what
// is left; where that is one block, it takes another from the slice before it.
// One block's |term| is often enough small against what its side elements could
// cost that most launches had a row to redo: with slices of three and two at the
// end 4096 x 2304 M = 16 takes 14.3 -> 12.6 us (Q4_K), 15.3 -> 13.2 (Q5_K).
__host__ __device__ constexpr uint32_t slice_first(uint32_t k, uint32_t nb) {
  return 4u * k - (k != 0u && 4u * k + 1u == nb ? 1u : 0u);
}
// The same in a paired launch (Q6_K, odd nb), whose rows are nb + 1 blocks wide:
// an even row's own nb blocks and the next, an odd row's after the one before it.
// Where slices of four leave two blocks the even rows' first slice is the short
// one, the odd rows' the last, so that both have two blocks of the row itself.
__host__ __device__ constexpr uint32_t paired_slice_first(uint32_t k, uint32_t nb, uint32_t odd) {
  return 4u * k - (k != 0u && odd == 0u && (nb & 3u) == 1u ? 2u : 0u);
}

// LDS map of a launch whose workgroups keep up to stride = 4 blocks of ng
// groups (group g's block b is group-block gb = stride g + b): the
// group images (4 KB per group-block); with `mins`, the unit sums (256 bytes
// per group-block: lane group k's units 2 k and 2 k + 1 as two halves at
// 64 k + 4 (4 t + p), piece p of vector t); with `dsum`, 128 times each
// vector's digit sums (64 bytes per group-block, vector t's four at 16 t); per
// vector v, 4 stride bytes each, the exponents and the bounds on the side
// elements' rounding over the tolerance they are held to (kFewTol or
// kRoundedTol; infinite for a block on the exact path).
struct TokLayout {
  uint32_t img, usum, dsum, expo, rerr, total;
  uint32_t stride;
};
__host__ __device__ constexpr TokLayout tok64_layout(uint32_t stride, uint32_t ng, bool mins,
                                                     bool dsum) {
  TokLayout l{};
  l.stride = stride;
  l.img = 0u;
  l.usum = l.img + 4096u * ng * stride;
  l.dsum = l.usum + (mins ? 256u * ng * stride : 0u);
  l.expo = l.dsum + (dsum ? 64u * ng * stride : 0u);
  l.rerr = l.expo + 16u * ng * stride;
  l.total = l.rerr + 16u * ng * stride;
  return l;
}

// The wave's share of the image blocks: group-blocks q = wave + i WAVES, i <
// SHARE, of the ng groups in order of group and of the blocks 0 .. stride - 1
// (those past nbl hold nothing); lane (t, c) takes elements 16 c .. 16 c + 15 of
// vector 4 g + t.  Vectors past ntok and blocks outside the row's nb read as
// zero.
template <int WAVES, int SHARE>
__device__ __forceinline__ void load_group_x(u32x4 (&xq)[SHARE][4], const float* x, uint32_t nb,
                                             uint32_t blk0, uint32_t nbl, uint32_t ng,
                                             uint32_t ntok, uint32_t wave, uint32_t lane) {
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(x), 0, (int)(ntok * nb * 1024u), kBufferWord3);
#pragma unroll
  for (int i = 0; i < SHARE; ++i) {
    const uint32_t q = wave + (uint32_t)i * WAVES, g = q >> 2, b = q & 3u;
    if (g < ng && b < nbl) {
      const uint32_t at = ((4u * g + (lane >> 4)) * nb + blk0 + b) * 1024u + 64u * (lane & 15u);
      const uint32_t off = blk0 + b < nb ? at : 0x80000000u;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        xq[i][j] = __builtin_bit_cast(
            u32x4, __builtin_amdgcn_raw_buffer_load_b128(xr, off + 16u * j, 0, 0));
    }
  }
}

// The lane's offsets, from a stage's first row, of the copies that fill PITCH
// 16-byte slots a row in order (PIECES of them distinct).
template <int COPIES, uint32_t PITCH, uint32_t PIECES>
__device__ __forceinline__ void copy_offsets(uint32_t row_bytes, uint32_t lane,
                                             uint32_t (&vo)[COPIES]) {
#pragma unroll
  for (int i = 0; i < COPIES; ++i) {
    const uint32_t c = min(64u * (uint32_t)i + lane, 16u * PITCH - 1u), row = c / PITCH;
    vo[i] = row * row_bytes + 16u * min(c - PITCH * row, PIECES - 1u);
  }
}

// Sum over a DPP row's 16 lanes (valid in lane 15).
__device__ __forceinline__ uint32_t row_sum_u(uint32_t v) {
  v += dpp_u<kRowShr1>(v);
  v += dpp_u<kRowShr2>(v);
  v += dpp_u<kRowShr4>(v);
  return v + dpp_u<kRowShr8>(v);
}

// Whether a (vector, row) keeps its sum over the slice: `most` the largest |w|
// the row's blocks can hold, `side` the vector's slice_err, `sum_abs` the sum of
// |block term|, which is at most sum|w x| plus the bound itself (under 1 % of
// it); the factor also covers the f32 rounding here.
__device__ __forceinline__ bool side_ok(float most, float side, float sum_abs) {
  return most * side * 1.02f <= sum_abs;
}

// Turns the wave's share of activations (load_group_x) into images, with what
// else the layout keeps of them (chunk_digits: about 270 instructions a
// group-block; a build that summed the side elements' rounding errors and the
// units apart took 540, a quarter of a sixteen-vector launch).
template <int WAVES, int SHARE, bool MINS, bool DSUM, typename ChunkSlot>
__device__ __forceinline__ void build_group_images64(uint32_t sbase, const TokLayout& L,
                                                     const u32x4 (&xr)[SHARE][4], uint32_t nbl,
                                                     uint32_t ng, uint32_t wave, uint32_t lane,
                                                     ChunkSlot chunk_slot) {
  const uint32_t t = lane >> 4, c = lane & 15u;
  const uint32_t woff = chunk_slot(c) + 64u * t;
#pragma unroll
  for (int i = 0; i < SHARE; ++i) {
    const uint32_t q = wave + (uint32_t)i * WAVES, g = q >> 2, b = q & 3u;
    if (g >= ng || b >= nbl) continue;
    const uint32_t gb = L.stride * g + b;
    const uint32_t blk = sbase + L.img + 4096u * gb;
    const uint32_t vec = 4u * L.stride * (4u * g + t) + 4u * b;
    const ChunkDigits cd = chunk_digits([&](int k) { return xr[i][k >> 2][k & 3]; });
    const auto& dg = cd.dg;
    const auto& sum = cd.sum;
#pragma unroll
    for (int d = 0; d < 4; ++d)
      lds_write_b128(blk + woff + 16u * d, u32x4{dg[0][d], dg[1][d], dg[2][d], dg[3][d]});
    if constexpr (MINS) {
      // unit c / 2 (its two chunks meet in the odd lane): X_u = hi 2^16 + lo
      // in 12-bit signed pieces, the last what is left (|X_u| <= 2^35, so at
      // most 2^11, exact as a half)
      int lo = sum[0] + 256 * sum[1], hi = sum[2] + 256 * sum[3];
      lo += (int)dpp_u<kRowShr1>((uint32_t)lo);
      hi += (int)dpp_u<kRowShr1>((uint32_t)hi);
      const int p0 = (lo << 20) >> 20;
      const int rest = 16 * hi + ((lo - p0) >> 12);
      const int p1 = (rest << 20) >> 20;
      const int p2 = (rest - p1) >> 12;
      auto half = [](int p) {
        return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(float)p);
      };
      if (c & 1u) {
        const uint32_t at = sbase + L.usum + 256u * gb + 64u * (c >> 2) + 16u * t + (c & 2u);
        lds_write_b16(at, half(p0));
        lds_write_b16(at + 4u, half(p1));
        lds_write_b16(at + 8u, half(p2));
        lds_write_b16(at + 12u, 0u);
      }
    }
    if constexpr (DSUM) {
      uint32_t s[4];
#pragma unroll
      for (int d = 0; d < 4; ++d) s[d] = 128u * row_sum_u((uint32_t)sum[d]);
      if (c == 15u)
        lds_write_b128(sbase + L.dsum + 64u * gb + 16u * t, u32x4{s[0], s[1], s[2], s[3]});
    }
    const uint32_t nside = row_sum_u(cd.nside);
    if (c == 15u) {
      const float n = (float)nside * (nside <= kFewSide ? 1.0f / kFewTol : 1.0f / kRoundedTol);
      lds_write_b32(sbase + L.expo + vec, (uint32_t)(cd.bad ? kBadTok : cd.e - kFixBits));
      lds_write_b32(sbase + L.rerr + vec,
                    cd.bad ? 0x7f800000u
                        : __float_as_uint(__builtin_amdgcn_ldexpf(n, cd.e - kFixBits - 1)));
    }
  }
}

// A vector's bound on the rounding of its side elements, over its tolerance,
// summed over the nbl blocks of the slice (infinite when a block takes the
// exact path).
__device__ __forceinline__ float slice_err(const uint8_t* rerr, uint32_t nbl) {
  const u32x4 v = lds_u32x4(rerr);
  float e = __uint_as_float(v[0]);
#pragma unroll
  for (uint32_t b = 1; b < 4u; ++b)
    if (b < nbl) e += __uint_as_float(v[b]);
  return e;
}

// y[t * yrows + row] = sum over the stages s of part[(s * nv + t) * rows + row],
// in stage order (the sliced launch's second kernel; a "stage" here is the
// first kernel's unit of partial sums, a K slice).  A partial that holds
// kPartRedo (its lane failed a check in the first kernel) is the stage's
// exact dot instead: quant.rs's per-weight values of the stage's blocks of the
// row times vector t of the batch-major x, summed in f64 and rounded once.  The
// workgroup's waves take such stages together from a queue in LDS, four at a
// time; a stage past the queue's room is taken by its own thread.  (With 32
// threads a stage, a 32-weight unit each, its bytes loaded one by one, one such
// stage cost a launch 1-2 us.)  A thread with such a stage sums its rows'
// partials again in stage order, the first eight stages kept in registers.
// R rows per thread: 1, or 4 with 16-byte loads and stores (launch_tok_reduce
// takes 4 when the rows, y and the grid allow it); each row's sum is the same.
// PAIRED: rows 2 r and 2 r + 1 share place r of the partials, of ceil(rows / 2);
// the first nstages stages are the even rows' and the next nstages the odd
// rows' (paired_slice_first; the block before the row is no part of it).
constexpr uint32_t kStageBlocks = 4u;  // at most, in a stage
constexpr uint32_t kRedoQueue = 64;
template <uint32_t T>
__device__ __noinline__ float stage_exact(const uint8_t* __restrict__ w, uint32_t row,
                                          uint32_t nb, uint32_t b0, uint32_t b1,
                                          const float* __restrict__ x) {
  constexpr uint32_t kBytes = BlockBytes<T>::value;
  const uint8_t* const r = w + (size_t)row * nb * kBytes;
  double acc = 0.0;
  for (uint32_t b = b0; b < b1; ++b) {
    for (uint32_t u = 0; u < 8u; ++u) {
      float wv[32];
      decode_unit_exact<T>(r + (size_t)b * kBytes, u, wv);
      const float* const xu = x + (size_t)b * kBlockElems + 32u * u;
#pragma unroll
      for (int i = 0; i < 32; ++i) acc = fma((double)wv[i], (double)xu[i], acc);
    }
  }
  return (float)acc;
}

template <uint32_t T, int R, bool PAIRED>
__global__ __launch_bounds__(256) void tok_reduce(const float* __restrict__ part,
                                                  float* __restrict__ y, uint32_t rows,
                                                  uint32_t yrows, uint32_t nstages, uint32_t nv,
                                                  const uint8_t* __restrict__ w,
                                                  const float* __restrict__ x, uint32_t nb) {
  static_assert(R == 1 || (R == 4 && !PAIRED), "one or four rows per thread");
  constexpr uint32_t kBytes = BlockBytes<T>::value;
  __shared__ uint32_t queue[kRedoQueue];  // (row in the workgroup) << 16 | stage
  __shared__ float value[kRedoQueue];
  __shared__ uint32_t queued;
  const uint32_t tid = threadIdx.x, t = blockIdx.y;
  const uint32_t rw = (uint32_t)R * tid;                    // the thread's first row in the workgroup
  const uint32_t row = blockIdx.x * (256u * R) + rw;        // its rows row .. row + R - 1
  const uint32_t places = PAIRED ? (rows + 1u) / 2u : rows;
  const size_t step = (size_t)nv * places;
  const float* const p = part + (size_t)t * places +
                         (PAIRED ? (row >> 1) + (row & 1u) * nstages * step : (size_t)row);
  const float* const xt = x + (size_t)t * nb * kBlockElems;
  if (tid == 0u) queued = 0u;
  __syncthreads();
  // the first block of stage st of row r, and the block past its last
  auto first_block = [&](uint32_t st, uint32_t r) {
    return PAIRED ? paired_slice_first(st, nb, r & 1u) - (r & 1u) : slice_first(st, nb);
  };
  auto end_block = [&](uint32_t st, uint32_t r) { return min(first_block(st + 1u, r), nb); };
  // stages base .. base + 7 of the thread's rows, eight loads in flight
  auto load8 = [&](uint32_t base, float (&v)[8][R]) {
#pragma unroll
    for (uint32_t i = 0; i < 8u; ++i) {
      if (base + i < nstages) {
        if constexpr (R == 4) {
          const f32x4 q = *reinterpret_cast<const f32x4*>(p + (base + i) * step);
#pragma unroll
          for (int c = 0; c < R; ++c) v[i][c] = q[c];
        } else {
          v[i][0] = p[(base + i) * step];
        }
      } else {
#pragma unroll
        for (int c = 0; c < R; ++c) v[i][c] = 0.0f;
      }
    }
  };
  // the stages' sums in stage order; the stages the thread's rows leave to
  // the workgroup go to the queue
  float sum[R];
  float first[8][R];
#pragma unroll
  for (int c = 0; c < R; ++c) sum[c] = 0.0f;
  bool mine = false;
  if (row < rows) {  // (rows a multiple of R)
    for (uint32_t base = 0; base < nstages; base += 8u) {
      float v[8][R];
      load8(base, v);
#pragma unroll
      for (uint32_t i = 0; i < 8u; ++i) {
        if (base == 0u) {
#pragma unroll
          for (int c = 0; c < R; ++c) first[i][c] = v[i][c];
        }
        if (base + i >= nstages) continue;
#pragma unroll
        for (int c = 0; c < R; ++c) {
          if (__float_as_uint(v[i][c]) == kPartRedo) {
            const uint32_t k = atomicAdd(&queued, 1u);
            if (k < kRedoQueue) queue[k] = ((rw + (uint32_t)c) << 16) | (base + i);
            mine = true;
          }
          sum[c] += v[i][c];
        }
      }
    }
  }
  if (__syncthreads_or(mine)) {
    // queued stages four at a time, one a wave: lane l takes elements 4 l .. 4 l + 3
    // of each block, all their loads in flight, and the lanes' f64 dots are summed
    const uint32_t nq = min(queued, kRedoQueue);
    const uint32_t e = tid >> 6, l = tid & 63u;
    for (uint32_t k0 = 0; k0 < nq; k0 += 4u) {
      const uint32_t k = k0 + e;
      double acc = 0.0;
      if (k < nq) {
        const uint32_t r = blockIdx.x * (256u * R) + (queue[k] >> 16), st = queue[k] & 0xffffu;
        const uint32_t b0 = first_block(st, r), b1 = end_block(st, r);
#pragma unroll
        for (uint32_t i = 0; i < kStageBlocks; ++i) {
          const uint32_t b = b0 + i;
          if (b < b1) {  // (the block before an odd row's first is no part of it)
            const float4 wv = decode_four_exact<T>(w + ((size_t)r * nb + b) * kBytes, 4u * l);
            const float4 xv =
                *reinterpret_cast<const float4*>(xt + (size_t)b * kBlockElems + 4u * l);
            acc = fma((double)wv.x, (double)xv.x, acc);
            acc = fma((double)wv.y, (double)xv.y, acc);
            acc = fma((double)wv.z, (double)xv.z, acc);
            acc = fma((double)wv.w, (double)xv.w, acc);
          }
        }
      }
#pragma unroll
      for (int h = 32; h > 0; h >>= 1) acc += __shfl_xor(acc, h, 64);
      if (l == 0u && k < nq) value[k] = (float)acc;
    }
    __syncthreads();
  }
  if (row >= rows) return;
  if (mine) {  // the sums again, with the recomputed stages (unchanged for rows without one)
    const uint32_t nq = min(queued, kRedoQueue);
#pragma unroll
    for (int c = 0; c < R; ++c) sum[c] = 0.0f;
    for (uint32_t base = 0; base < nstages; base += 8u) {
      float v[8][R];
      if (base == 0u) {
#pragma unroll
        for (uint32_t i = 0; i < 8u; ++i)
#pragma unroll
          for (int c = 0; c < R; ++c) v[i][c] = first[i][c];
      } else {
        load8(base, v);
      }
#pragma unroll
      for (uint32_t i = 0; i < 8u; ++i) {
        if (base + i >= nstages) continue;
        const uint32_t st = base + i;
#pragma unroll
        for (int c = 0; c < R; ++c) {
          float vc = v[i][c];
          if (__float_as_uint(vc) == kPartRedo) {
            const uint32_t key = ((rw + (uint32_t)c) << 16) | st;
            uint32_t k = 0;
            while (k < nq && queue[k] != key) ++k;
            const uint32_t r = row + (uint32_t)c, b0 = first_block(st, r);
            vc = k < nq ? value[k]
                        : stage_exact<T>(w, r, nb, b0 < nb ? b0 : 0u, end_block(st, r), xt);
          }
          sum[c] += vc;
        }
      }
    }
  }
  float* const yo = y + (size_t)t * yrows + row;
  if constexpr (R == 4) {
    *reinterpret_cast<f32x4*>(yo) = f32x4{sum[0], sum[1], sum[2], sum[3]};
  } else {
    yo[0] = sum[0];
  }
}

// The reduce of a sliced launch of ntok vectors: four rows a thread when the
// row counts (of the launch, and yrows of a vector's outputs) are multiples of
// 4, y is 16-byte aligned (the scratch always is) and the grid still gives
// every CU two workgroups, else one.  (With one row a thread the Q6_K head,
// 151,936 rows, takes 1 us more at M = 4 and 4 us at M = 16; Q4_K 17408 rows
// at M = 16, one workgroup a CU, loses 0.4 us with four.)
template <uint32_t T, bool PAIRED = false>
void launch_tok_reduce(const float* part, float* y, uint32_t rows, uint32_t yrows,
                       uint32_t nstages, uint32_t nv, uint32_t ntok, const uint8_t* w,
                       const float* x, uint32_t nb, hipStream_t s) {
  const uint32_t g4 = (rows + 1023u) / 1024u;
  if (!PAIRED && rows % 4u == 0u && yrows % 4u == 0u && ((uintptr_t)y & 15u) == 0u &&
      (uint64_t)g4 * ntok >= 2u * (uint64_t)cu_count())
    hipLaunchKernelGGL((tok_reduce<T, 4, false>), dim3(g4, ntok), dim3(256), 0, s, part, y, rows, yrows,
                       nstages, nv, w, x, nb);
  else
    hipLaunchKernelGGL((tok_reduce<T, 1, PAIRED>), dim3((rows + 255u) / 256u, ntok), dim3(256), 0, s, part,
                       y, rows, yrows, nstages, nv, w, x, nb);
}

}  // namespace
}  // namespace mfma
}  // namespace sihip
