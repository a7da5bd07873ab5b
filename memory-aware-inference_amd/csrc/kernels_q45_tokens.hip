// Multi-token verify of Q4_K and Q5_K on the gfx950 int8 matrix cores: three
// to sixteen activation vectors in one pass over the weights (matmul-many,
// replacing si_q4_k_matmul_many, metal.rs:1052-1262).
//
// Arithmetic.  The vectors sit in the A operand of v_mfma_i32_16x16x64_i8
// (group images, tokens_common.h: four vectors of four digits in its 16
// rows) and the B operand holds weights with their 6-bit scale folded in,
// sc q = 8 (sc >> 3) q + (sc & 7) q: both products fit a byte (at most 105
// for Q4_K), so one v_pk_mul_lo_u16 makes four of them, and a block's 256
// weights meet a group in eight MFMAs whose sums need no scale any more.
// (With the scale applied to the MFMA results, as 32 multiply-adds per group
// and block, those products alone took 17408 x 5120 with sixteen vectors
// past 30 us.)  Q5_K's products reach 217: their bytes are stored less 128,
// and the MFMAs start from 128 times the block's digit sums.
//
// Lane (k, n) holds units 2 k and 2 k + 1 of a block for tile row n (qs bytes
// 32 k .. 32 k + 31), so it decodes two scales and two mins a block; MFMA j
// takes the low (j < 2) or high nibbles of its qs piece j & 1.  Result lane
// (g, n) of group G has the four digit sums of vector 4 G + g and row n:
// T_d = sum sc q D_d, |T_d| < 2^26.
//
// The min term sum_u m_u X_u is one f16 MFMA per group and block: the unit
// sums X_u (35 bits) as three 12-bit signed pieces in the A rows 4 t + p, the
// lane's two mins in B; every f32 sum is an integer below 2^24, so exact.
// Both sums are then exact f64 values and the block's term
// d (sum_d 256^d T_d) - dmin (sum_p 4096^p M_p) is formed in f64 (v_fma_f64
// issues at the f32 rate here).  In f32 the two terms' rounding was of the
// order of the whole allowance: weights quantised from zero-mean data have
// d sc q and dmin m of the same size everywhere, a few rows of most stages
// failed the check below, and their wave did the stage a second time.
//
// What a lane leaves to tok_reduce's exact recompute (kPartRedo): a stage
// with a block whose activations are not finite or reach 2^100; one whose
// sum is not finite; one with a block whose two terms cancel to below 2^-30
// of the first, so that f64 rounding could show (weights that all decode to
// zero); and one whose rounded blocks (side elements, mfma_common.h) could be
// off by more than kStageTol of its sum |block term|.
//
// Work split.  A launch cuts K into slices of four blocks: workgroup g works
// on slice g / GS for tiles g % GS, g % GS + GS, ..., keeping that slice's
// images in LDS; each wave takes (tile, slice) pairs, one stage buffer of 16
// rows x four blocks in flight, and stores the vectors' sums in the scratch;
// tok_reduce adds the slices in order.  A launch whose sums exceed the
// scratch runs as several over row ranges.
#include "mfma_common.h"
#include "si_hip_tuned.h"
#include "tokens_common.h"

namespace sihip {
namespace {

using namespace mfma;

constexpr uint32_t kSliceBlocks = 4u;

template <int QB>
struct Format {
  static constexpr uint32_t kBytes = QB == 5 ? kQ5Bytes : kQ4Bytes;
  static constexpr uint32_t kPieces = kBytes / 16u;             // 16-byte pieces per block
  static constexpr uint32_t kStage = 1024u * kPieces;           // 16 rows x four blocks
  static constexpr uint32_t kBlock = kStage / kSliceBlocks;     // a block's bytes of a stage
  static constexpr uint32_t kType = QB == 5 ? kTypeQ5K : kTypeQ4K;
};

// Launch constants: GS workgroups per slice and its division constant.
struct Tok45Args {
  uint32_t groups_per_slice, m_gps;
  void* wsp;  // the workspace, for failure reports
};

// One block of the lane's row, decoded: the scaled weights' two digits for
// the four MFMAs, the two mins as halves, d and dmin.
struct Block45 {
  i32x4 hi[4], lo[4];
  f16x4 mins;
  double d, dmin;
};

// Four byte products q s of the bytes of q (q s < 256, s in both halves).
__device__ __forceinline__ uint32_t byte_products(uint32_t q, u16x2 s) {
  return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, q) * s));
}

template <int QB>
__device__ __forceinline__ Block45 decode_block(const uint8_t* stage, uint32_t grp, uint32_t n) {
  const uint8_t* const row = stage + 16u * n;
  const u32x4 h = lds_u32x4(row);
  const uint8_t* const qs = row + (QB == 5 ? 768u : 256u) + 512u * grp;
  const u32x4 q[2] = {lds_u32x4(qs), lds_u32x4(qs + 256u)};
  Block45 b;
  const bool hi_units = grp >= 2u;
  const uint32_t sh = 16u * (grp & 1u);
  const uint32_t scw = hi_units ? (h[3] & 0x0f0f0f0fu) | ((h[1] >> 2) & 0x30303030u)
                                : h[1] & 0x3f3f3f3fu;
  const uint32_t mnw = hi_units ? ((h[3] >> 4) & 0x0f0f0f0fu) | ((h[2] >> 2) & 0x30303030u)
                                : h[2] & 0x3f3f3f3fu;
  const uint32_t sc = scw >> sh, mn = mnw >> sh;  // bytes 0, 1: units 2 grp, 2 grp + 1
  const uint32_t s_hi = (sc >> 3) & 0x0707u, s_lo = sc & 0x0707u;
  auto both = [](uint32_t v, uint32_t sel) {
    return __builtin_bit_cast(u16x2, __builtin_amdgcn_perm(0u, v, sel));
  };
  const u16x2 s[2][2] = {{both(s_hi, 0x0c000c00u), both(s_lo, 0x0c000c00u)},
                         {both(s_hi, 0x0c010c01u), both(s_lo, 0x0c010c01u)}};
  u32x4 qh[2];
  if constexpr (QB == 5) {
    qh[0] = lds_u32x4(row + 256u);
    qh[1] = lds_u32x4(row + 512u);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {  // units 2 grp (j < 2) and 2 grp + 1, qs piece j & 1
    const int u = j >> 1, pc = j & 1;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      uint32_t w = (u ? q[pc][k] >> 4 : q[pc][k]) & 0x0f0f0f0fu;
      if constexpr (QB == 5)  // bit 2 grp + u of each qh byte, rotated to bit 4
        w |= __builtin_amdgcn_alignbit(qh[pc][k], qh[pc][k], (28u + 2u * grp + u) & 31u) &
             0x10101010u;
      uint32_t ph = byte_products(w, s[u][0]), pl = byte_products(w, s[u][1]);
      if constexpr (QB == 5) {
        ph ^= 0x80808080u;  // less 128
        pl ^= 0x80808080u;
      }
      b.hi[j][k] = (int)ph;
      b.lo[j][k] = (int)pl;
    }
  }
  // 1024 + m as halves (0x6400 | m), less 1024; the MFMA's other two K slots
  // of the lane stay zero
  const f16x2 m = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, mn, 0x04010400u)) -
                  f16x2{(_Float16)1024.0f, (_Float16)1024.0f};
  b.mins = f16x4{m[0], m[1], (_Float16)0.0f, (_Float16)0.0f};
  b.d = (double)half_bits_to_float(h[0] & 0xffffu);
  b.dmin = (double)half_bits_to_float(h[0] >> 16);
  return b;
}

// Largest |w| of a block of a row (all eight units) from its header.
template <int QB>
__device__ __forceinline__ float block_bound(const u32x4& h) {
  const uint32_t sc03 = h[1] & 0x3f3f3f3fu;
  const uint32_t mn03 = h[2] & 0x3f3f3f3fu;
  const uint32_t sc47 = (h[3] & 0x0f0f0f0fu) | ((h[1] >> 2) & 0x30303030u);
  const uint32_t mn47 = ((h[3] >> 4) & 0x0f0f0f0fu) | ((h[2] >> 2) & 0x30303030u);
  const float ad = fabsf(half_bits_to_float(h[0] & 0xffffu));
  const float am = fabsf(half_bits_to_float(h[0] >> 16));
  float mx = 0.0f;
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const uint32_t sc = ((u < 4 ? sc03 : sc47) >> (8 * (u & 3))) & 0xffu;
    const uint32_t mn = ((u < 4 ? mn03 : mn47) >> (8 * (u & 3))) & 0xffu;
    mx = fmaxf(mx, fmaf(ad, (float)((QB == 5 ? 31u : 15u) * sc), am * (float)mn));
  }
  return mx;
}

template <int WAVES, int NG, int QB>
__global__ __launch_bounds__(WAVES * 64) void q45_tokens_mfma(const uint8_t* __restrict__ w,
                                                              const float* __restrict__ x,
                                                              uint32_t rows, uint32_t nb,
                                                              uint32_t ntok,
                                                              float* __restrict__ part_out,
                                                              Tok45Args ta) {
  using F = Format<QB>;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const uint32_t wave = uniform(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t grp = lane >> 4, n = lane & 15u;
  const uint32_t row_bytes = nb * F::kBytes;
  const uint32_t ntiles = (rows + 15u) / 16u;
  const uint32_t sbase = (uint32_t)(uintptr_t)smem;
  uint8_t* const wstage = smem + wave * F::kStage;

  // this workgroup's slice k (blocks blk0 .. blk0 + nbl - 1) and its tiles
  // tg, tg + GS, ...; the wave's are tiles wave, wave + WAVES, ... of those
  const FastDiv by_gps{ta.groups_per_slice, ta.m_gps};
  const uint32_t k = quo(blockIdx.x, by_gps);
  const uint32_t tg = blockIdx.x - k * ta.groups_per_slice;
  const uint32_t blk0 = kSliceBlocks * k, nbl = min(kSliceBlocks, nb - blk0);
  const TokLayout L = tok64_layout(WAVES * F::kStage, kSliceBlocks, NG, true, QB == 5);
  const uint32_t ntw = tg < ntiles ? quo(ntiles - 1u - tg, by_gps) + 1u : 0u;
  const uint32_t my_tiles = wave < ntw ? (ntw - 1u - wave) / WAVES + 1u : 0u;

  // 1. the vectors' blocks of the slice into the image area
  copy_x_group<WAVES>(smem, L.img, x, nb, blk0, nbl, NG, ntok, wave, lane);

  // 2. the copy of a tile's stage: copy i, lane l moves piece 4 i + l / 16 of
  //    row l % 16's blocks; rows past the matrix read zero
  const uint32_t voff = n * row_bytes + 16u * grp;
  auto issue = [&](uint32_t lt) {
    const uint32_t row0 = (tg + lt * ta.groups_per_slice) * 16u;
    const uint32_t nrows = min(16u, rows - row0);
    const uint8_t* const sb = w + (size_t)row0 * row_bytes + F::kBytes * blk0;
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(sb), 0, (int)(nrows * row_bytes - F::kBytes * blk0), kBufferWord3);
#pragma unroll
    for (int i = 0; i < (int)F::kPieces; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void*)(wstage + 1024 * i), 16,
                                                voff + 64u * i, 0, 0, 0);
  };

  // 3. the builders' count and the special flag cleared, the first copies and
  //    the group images: the first round of waves issues before the barrier
  //    (the empty memory queue takes its copies at once), the rest after; a
  //    builder converts exactly the blocks it copied and a wave waits for
  //    the builders' count before its first arithmetic
  const bool first_round = wave < 4u;
  if (first_round && my_tiles > 0u) issue(wave);
  if (threadIdx.x == 0u) {
    lds_write_b32(sbase + L.ready, 0u);
    lds_write_b32(sbase + L.special, 0u);
  }
  lds_wait();
  __builtin_amdgcn_s_barrier();
  if (!first_round && my_tiles > 0u) issue(wave);
  const uint32_t builders = min((uint32_t)WAVES, (uint32_t)NG * nbl);
  if (wave < builders) {
    // (the stage copies went out after the x copies and complete in order)
    if (my_tiles > 0u)
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(F::kPieces));
    else
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    // chunk 4 p + j: MFMA j, lane group p
    build_group_images64<WAVES, true, QB == 5>(sbase, L, nbl, NG, wave, lane, [](uint32_t c) {
      return 1024u * (c & 3u) + 256u * (c >> 2);
    });
    lds_wait();
    if (lane == 0u) (void)lds_add_rtn(sbase + L.ready, 1u);
  }

  // 4. the wave's tiles: lane (grp, n) accumulates, for each group G, vector
  //    4 G + grp, row n
  uint32_t fail = 0u;  // a bounded wait that gave up (kDevErr*)
  uint32_t special = 0u;
  for (uint32_t lt = wave; lt < ntw; lt += WAVES) {
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    if (lt == wave) {
      wait_count(sbase + L.ready, builders, fail);
      special = uniform(lds_read_b32(sbase + L.special));
    }
    asm volatile("" ::: "memory");  // (the stage and the images are in LDS from here on)
    double acc[NG];
    float sum_abs[NG];
    bool redo[NG];  // the lane leaves group G's stage to tok_reduce
#pragma unroll
    for (int G = 0; G < NG; ++G) {
      acc[G] = 0.0;
      sum_abs[G] = 0.0f;
      redo[G] = false;
    }
#pragma unroll 1
    for (uint32_t b = 0; b < nbl; ++b) {
      const Block45 bw = decode_block<QB>(wstage + F::kBlock * b, grp, n);
#pragma unroll
      for (int G = 0; G < NG; ++G) {
        const uint32_t gb = (uint32_t)G * nbl + b;
        const uint8_t* const img = smem + L.img + 4096u * gb + 16u * lane;
        i32x4 c0 = {0, 0, 0, 0};
        if constexpr (QB == 5)
          c0 = __builtin_bit_cast(i32x4, lds_u32x4(smem + L.dsum + 64u * gb + 16u * grp));
        i32x4 ch = c0, cl = c0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const i32x4 a = __builtin_bit_cast(i32x4, lds_u32x4(img + 1024u * j));
          ch = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, bw.hi[j], ch, 0, 0, 0);
          cl = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, bw.lo[j], cl, 0, 0, 0);
        }
        const f16x2 xs =
            __builtin_bit_cast(f16x2, lds_u32(smem + L.usum + 256u * gb + 4u * lane));
        const f32x4 cm = __builtin_amdgcn_mfma_f32_16x16x16f16(
            f16x4{xs[0], xs[1], (_Float16)0.0f, (_Float16)0.0f}, bw.mins,
            f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
        const int e = (int)lds_u32(smem + L.expo + 16u * (4u * G + grp) + 4u * b);
        double t = (double)(8 * ch[3] + cl[3]);
#pragma unroll
        for (int d = 2; d >= 0; --d) t = fma(t, 256.0, (double)(8 * ch[d] + cl[d]));
        const double m = fma(fma((double)cm[2], 4096.0, (double)cm[1]), 4096.0, (double)cm[0]);
        t *= bw.d;
        const double p = fma(-bw.dmin, m, t);
        // (not below 2^-30 of the first term, and no NaN)
        redo[G] |= !(fma(fabs(p), 0x1p30, -fabs(t)) >= 0.0);
        const double v = __builtin_amdgcn_ldexp(p, e);  // 0 for a block on the exact path (kBadTok)
        acc[G] += v;
        sum_abs[G] += fabsf((float)v);
      }
    }
    float part[NG];
#pragma unroll
    for (int G = 0; G < NG; ++G) {
      part[G] = (float)acc[G];
      redo[G] |= !(fabsf(part[G]) < __builtin_huge_valf());
    }
    if (special != 0u) {
      // blocks on the exact path, and the rounded blocks' bound
      float err[NG];
#pragma unroll
      for (int G = 0; G < NG; ++G) err[G] = 0.0f;
#pragma unroll 1
      for (uint32_t b = 0; b < nbl; ++b) {
        const float bound = block_bound<QB>(lds_u32x4(wstage + F::kBlock * b + 16u * n));
#pragma unroll
        for (int G = 0; G < NG; ++G) {
          const uint32_t at = 16u * (4u * G + grp) + 4u * b;
          const float es = __uint_as_float(lds_u32(smem + L.rerr + at));
          if (es != 0.0f) err[G] = fmaf(bound, es, err[G]);
          redo[G] |= (int)lds_u32(smem + L.expo + at) == kBadTok;
        }
      }
#pragma unroll
      for (int G = 0; G < NG; ++G)
        redo[G] |= !(err[G] * 1.01f <= kStageTol * (sum_abs[G] - err[G]));
    }
    lds_wait();  // (every read of the stage is done: the next copy may land)
    if (lt + WAVES < ntw) issue(lt + WAVES);
    const uint32_t row = (tg + lt * ta.groups_per_slice) * 16u + n;
    if (row < rows) {
#pragma unroll
      for (int G = 0; G < NG; ++G) {
        const uint32_t v = 4u * G + grp;
        if (v < ntok)
          part_out[((size_t)k * 4u * NG + v) * rows + row] =
              redo[G] ? __uint_as_float(kPartRedo) : part[G];
      }
    }
  }
  if (fail != 0u) report_device_error(ta.wsp, fail);
}

// ntok <= 4 NG vectors in one pass; false when the shape does not fit.
template <int W, int NG, int QB>
bool launch_tok45(const uint8_t* w, const float* x, float* y, uint32_t rows, uint32_t nb,
                  uint32_t ntok, const Workspace& ws, hipStream_t s, hipError_t* err) {
  using F = Format<QB>;
  const uint32_t cus = (uint32_t)cu_count();
  const uint32_t slices = (nb + kSliceBlocks - 1u) / kSliceBlocks;
  constexpr TokLayout L = tok64_layout(W * F::kStage, kSliceBlocks, NG, true, QB == 5);
  static_assert(L.total <= kLdsBytes, "the stage buffers and the images fit the LDS");
  if (slices > cus) return false;
  // the rows of one launch: all, or as many whole tiles as the scratch holds
  const size_t row_part = (size_t)slices * 4u * NG * sizeof(float);
  const uint64_t fit = ws.scratch_bytes / row_part / 16u * 16u;
  const uint32_t chunk = (uint32_t)min((uint64_t)rows, fit);
  if (chunk == 0u) return false;
  // block and tile indices divided by GS <= cus
  if ((uint64_t)(cus + (chunk + 15u) / 16u) * cus >= (1ull << 32)) return false;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&q45_tokens_mfma<W, NG, QB>),
      hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes);
  *err = attr;
  for (uint32_t r0 = 0; r0 < rows && *err == hipSuccess; r0 += chunk) {
    const uint32_t nr = min(chunk, rows - r0);
    const uint8_t* const wr = w + (size_t)r0 * nb * F::kBytes;
    Tok45Args ta{};
    ta.groups_per_slice = min(cus / slices, (nr + 15u) / 16u);
    ta.m_gps = div_magic(ta.groups_per_slice);
    ta.wsp = ws.ptr;
    hipLaunchKernelGGL((q45_tokens_mfma<W, NG, QB>), dim3(ta.groups_per_slice * slices),
                       dim3(W * 64), L.total, s, wr, x, nr, nb, ntok, ws.scratch, ta);
    *err = hipGetLastError();
    if (*err != hipSuccess) break;
    launch_tok_reduce<F::kType>(ws.scratch, y + r0, nr, rows, slices, 4u * NG, ntok, wr, x, nb,
                                kSliceBlocks, s);
    *err = hipGetLastError();
  }
  return true;
}

template <int QB>
bool launch_tok45_any(const uint8_t* w, const float* x, float* y, uint32_t rows, uint32_t nb,
                      uint32_t ntok, const Workspace& ws, hipStream_t s, hipError_t* err) {
  if (ntok <= 4u) return launch_tok45<12, 1, QB>(w, x, y, rows, nb, ntok, ws, s, err);
  if (ntok <= 8u)
    return launch_tok45<QB == 5 ? 10 : 12, 2, QB>(w, x, y, rows, nb, ntok, ws, s, err);
  if (ntok <= 12u)
    return launch_tok45<QB == 5 ? 8 : 10, 3, QB>(w, x, y, rows, nb, ntok, ws, s, err);
  return launch_tok45<8, 4, QB>(w, x, y, rows, nb, ntok, ws, s, err);
}

}  // namespace

bool mfma::launch_q45_tokens(int qb, const uint8_t* w, const float* x, float* y, uint32_t rows,
                             uint32_t nb, uint32_t ntok, const Workspace& ws, hipStream_t s,
                             hipError_t* err) {
  return qb == 5 ? launch_tok45_any<5>(w, x, y, rows, nb, ntok, ws, s, err)
                 : launch_tok45_any<4>(w, x, y, rows, nb, ntok, ws, s, err);
}

}  // namespace sihip
