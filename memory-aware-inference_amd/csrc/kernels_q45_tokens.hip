// Multi-token verify of Q4_K and Q5_K on the gfx950 int8 matrix cores: two
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
// zero); and one whose side elements (bounded by half a unit each times the
// largest weight that d and dmin allow) could be off by more than they may be
// (kFewTol, tokens_common.h).
//
// Work split.  A launch cuts K into slices of four blocks (slice_first): workgroup g works
// on slice g / GS for tiles g % GS, g % GS + GS, ..., keeping that slice's
// images in LDS; each wave takes (tile, slice) pairs, their two-block stages
// one after another through one stage buffer (buffer->LDS copies, row by row;
// the next stage's go out once the stage is in registers), and stores the
// vectors' sums in the scratch; tok_reduce adds the slices in order.  A launch
// whose sums exceed the scratch runs as several over row ranges.
//
// Measured, 17408 x 5120 Q4_K M = 4 / 8 / 16 with the reduce (4.1-4.7 us of
// it): 27.9 / 44.4 / 72.9 us with the scales applied to the MFMA results and
// f32 terms; 16.3 / 20.3 / 26.9 here.  On the way: four-block stages whose copy
// went out after the arithmetic 19.2 / 23.3 / 33.4; weights loaded straight to
// registers, a tile ahead, 17.8 / 21.2 / 28.2 (each lane's 16 bytes a cache
// access of its own).  At M = 4 the launch is bound by the weight stream behind
// its start (5 us until the first stage is in and the images are built); at
// M = 16 VALU (about 180 instructions a tile and block) and MFMA (36 of 16
// cycles) add up to 13 of the kernel's 22 us.
#include "mfma_common.h"
#include "si_hip_tuned.h"
#include "tokens_common.h"

namespace sihip {
namespace {

using namespace mfma;

constexpr uint32_t kSliceBlocks = kStageBlocks;  // (slice_first)

template <int QB>
struct Format {
  static constexpr uint32_t kBytes = QB == 5 ? kQ5Bytes : kQ4Bytes;
  static constexpr uint32_t kType = QB == 5 ? kTypeQ5K : kTypeQ4K;
  // A stage is two blocks of 16 rows.  In LDS a row keeps its 16-byte pieces in
  // order, an odd number of slots (kPitch) from the next row, so that 16 lanes
  // reading one piece of the 16 rows meet all bank groups alike.
  static constexpr uint32_t kPieces = 2u * kBytes / 16u;
  static constexpr uint32_t kPitch = kPieces | 1u;
  static constexpr int kCopies = (int)((16u * kPitch + 63u) / 64u);
  static constexpr uint32_t kStage = 1024u * kCopies;
};

// Launch constants: GS workgroups per slice and its division constant.
struct Tok45Args {
  uint32_t groups_per_slice, m_gps;
};

// The lane's pieces of a stage's two blocks: the header, its two qs pieces and
// (Q5_K) the two qh pieces.
template <int QB>
struct Raw45 {
  u32x4 h, q[2], qh[QB == 5 ? 2 : 1];
};
template <int QB>
__device__ __forceinline__ void read_stage(Raw45<QB> (&r)[2], uint32_t hb, uint32_t qb) {
  if constexpr (QB == 4)
    asm volatile(
        "ds_read_b128 %0, %6\n"
        "ds_read_b128 %1, %7\n"
        "ds_read_b128 %2, %7 offset:16\n"
        "ds_read_b128 %3, %6 offset:144\n"
        "ds_read_b128 %4, %7 offset:144\n"
        "ds_read_b128 %5, %7 offset:160\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(r[0].h), "=&v"(r[0].q[0]), "=&v"(r[0].q[1]), "=&v"(r[1].h), "=&v"(r[1].q[0]),
          "=&v"(r[1].q[1])
        : "v"(hb), "v"(qb)
        : "memory");
  else
    asm volatile(
        "ds_read_b128 %0, %10\n"
        "ds_read_b128 %1, %10 offset:16\n"
        "ds_read_b128 %2, %10 offset:32\n"
        "ds_read_b128 %3, %11\n"
        "ds_read_b128 %4, %11 offset:16\n"
        "ds_read_b128 %5, %10 offset:176\n"
        "ds_read_b128 %6, %10 offset:192\n"
        "ds_read_b128 %7, %10 offset:208\n"
        "ds_read_b128 %8, %11 offset:176\n"
        "ds_read_b128 %9, %11 offset:192\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(r[0].h), "=&v"(r[0].qh[0]), "=&v"(r[0].qh[QB - 4]), "=&v"(r[0].q[0]),
          "=&v"(r[0].q[1]), "=&v"(r[1].h), "=&v"(r[1].qh[0]), "=&v"(r[1].qh[QB - 4]),
          "=&v"(r[1].q[0]), "=&v"(r[1].q[1])
        : "v"(hb), "v"(qb)
        : "memory");
}

// Group G's operands for block B of a stage (from the stage's first block): its
// images (ia), unit sums (ua), the exponent of the lane's vector (ea) and
// (Q5_K) 128 times that vector's digit sums (da).
template <int QB, int G, int B>
__device__ __forceinline__ void read_group(uint32_t ia, uint32_t ua, uint32_t ea, uint32_t da,
                                           i32x4 (&a)[4], uint32_t& xs, int& e, i32x4& ds) {
  constexpr int kGb = (int)kSliceBlocks * G + B;
  if constexpr (QB == 5)
    asm volatile(
        "ds_read_b128 %0, %7 offset:%11\n"
        "ds_read_b128 %1, %7 offset:%12\n"
        "ds_read_b128 %2, %7 offset:%13\n"
        "ds_read_b128 %3, %7 offset:%14\n"
        "ds_read_b32 %4, %8 offset:%15\n"
        "ds_read_b32 %5, %9 offset:%16\n"
        "ds_read_b128 %6, %10 offset:%17\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3]), "=&v"(xs), "=&v"(e), "=&v"(ds)
        : "v"(ia), "v"(ua), "v"(ea), "v"(da), "i"(4096 * kGb), "i"(4096 * kGb + 1024),
          "i"(4096 * kGb + 2048), "i"(4096 * kGb + 3072), "i"(256 * kGb),
          "i"(16 * (int)kSliceBlocks * G + 4 * B), "i"(64 * kGb)
        : "memory");
  else
    asm volatile(
        "ds_read_b128 %0, %6 offset:%9\n"
        "ds_read_b128 %1, %6 offset:%10\n"
        "ds_read_b128 %2, %6 offset:%11\n"
        "ds_read_b128 %3, %6 offset:%12\n"
        "ds_read_b32 %4, %7 offset:%13\n"
        "ds_read_b32 %5, %8 offset:%14\n"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3]), "=&v"(xs), "=&v"(e)
        : "v"(ia), "v"(ua), "v"(ea), "i"(4096 * kGb), "i"(4096 * kGb + 1024),
          "i"(4096 * kGb + 2048), "i"(4096 * kGb + 3072), "i"(256 * kGb),
          "i"(16 * (int)kSliceBlocks * G + 4 * B)
        : "memory");
}

// One block of the lane's row, decoded: the scaled weights' two digits for
// the four MFMAs, the two mins as halves, d and dmin.
struct Block45 {
  i32x4 hi[4], lo[4];
  f16x4 mins;
  float df, dminf;
};

// Four byte products q s of the bytes of q (q s < 256, s in both halves).
__device__ __forceinline__ uint32_t byte_products(uint32_t q, u16x2 s) {
  return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, q) * s));
}

template <int QB>
__device__ __forceinline__ Block45 decode_block(const Raw45<QB>& r, uint32_t grp) {
  const u32x4& h = r.h;
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
#pragma unroll
  for (int j = 0; j < 4; ++j) {  // units 2 grp (j < 2) and 2 grp + 1, qs piece j & 1
    const int u = j >> 1, pc = j & 1;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      uint32_t w = (u ? r.q[pc][k] >> 4 : r.q[pc][k]) & 0x0f0f0f0fu;
      if constexpr (QB == 5)  // bit 2 grp + u of each qh byte, rotated to bit 4
        w |= __builtin_amdgcn_alignbit(r.qh[pc][k], r.qh[pc][k], (28u + 2u * grp + u) & 31u) &
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
  b.df = half_bits_to_float(h[0] & 0xffffu);
  b.dminf = half_bits_to_float(h[0] >> 16);
  return b;
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
  constexpr uint32_t kImages = (uint32_t)WAVES * F::kStage;  // after the stage buffers
  constexpr TokLayout L = tok64_layout(kSliceBlocks, NG, true, QB == 5);
  const uint32_t wave = uniform(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t grp = lane >> 4, n = lane & 15u;
  const uint32_t row_bytes = nb * F::kBytes;
  const uint32_t ntiles = (rows + 15u) / 16u;
  const uint32_t sbase = (uint32_t)(uintptr_t)smem;
  uint8_t* const wstage = smem + wave * F::kStage;

  // this workgroup's slice k (blocks blk0 .. blk0 + nbl - 1, nst stages) and
  // its tiles tg, tg + GS, ...; the wave's are tiles wave, wave + WAVES, ...
  const FastDiv by_gps{ta.groups_per_slice, ta.m_gps};
  const uint32_t k = quo(blockIdx.x, by_gps);
  const uint32_t tg = blockIdx.x - k * ta.groups_per_slice;
  const uint32_t blk0 = slice_first(k, nb), nbl = min(slice_first(k + 1u, nb), nb) - blk0;
  const uint32_t nst = (nbl + 1u) / 2u;
  const uint32_t ntw = tg < ntiles ? quo(ntiles - 1u - tg, by_gps) + 1u : 0u;

  // 1. the activations of the wave's image blocks into registers, then the
  //    copy of its first stage: copy i's slot c = 64 i + lane is piece
  //    c % kPitch of row c / kPitch, so consecutive lanes read consecutive
  //    pieces of a row (a row's spare slot re-reads its last piece; rows past
  //    the matrix read zero)
  constexpr int kShare = (NG * (int)kSliceBlocks + WAVES - 1) / WAVES;
  u32x4 xq[kShare][4];
  load_group_x<WAVES, kShare>(xq, x, nb, blk0, nbl, NG, ntok, wave, lane);
  uint32_t vo[F::kCopies];
  copy_offsets<F::kCopies, F::kPitch, F::kPieces>(row_bytes, lane, vo);
  auto issue = [&](uint32_t lt, uint32_t sl) {
    const uint32_t row0 = (tg + lt * ta.groups_per_slice) * 16u;
    const uint32_t nrows = min(16u, rows - row0);
    const uint32_t at = F::kBytes * (blk0 + 2u * sl);
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(w + (size_t)row0 * row_bytes + at), 0, (int)(nrows * row_bytes - at),
        kBufferWord3);
#pragma unroll
    for (int i = 0; i < F::kCopies; ++i) {
      const uint32_t off = vo[i];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void*)(wstage + 1024 * i), 16, off, 0, 0,
                                                0);
    }
  };
  if (wave < ntw) issue(wave, 0u);

  // 2. the group images (chunk 4 p + j: MFMA j, lane group p)
  build_group_images64<WAVES, kShare, true, QB == 5>(
      sbase + kImages, L, xq, nbl, NG, wave, lane,
      [](uint32_t c) { return 1024u * (c & 3u) + 256u * (c >> 2); });
  lds_wait();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  float side[NG];
#pragma unroll
  for (int G = 0; G < NG; ++G)
    side[G] = slice_err(smem + kImages + L.rerr + 64 * G + 16u * grp, nbl);

  // 3. the wave's tiles, stage by stage: lane (grp, n) accumulates, for each
  //    group G, vector 4 G + grp, row n
  const uint32_t hb = sbase + wave * F::kStage + 16u * F::kPitch * n;
  const uint32_t qb = hb + F::kBytes - 128u + 32u * grp;
  const uint32_t ia0 = sbase + kImages + L.img + 16u * lane;
  const uint32_t ua0 = sbase + kImages + L.usum + 4u * lane;
  const uint32_t ea0 = sbase + kImages + L.expo + 16u * grp;
  const uint32_t da0 = sbase + kImages + L.dsum + 16u * grp;
  double acc[NG], sum_abs[NG];
  bool redo[NG];  // the lane leaves group G's slice to tok_reduce
  float most = 0.0f;  // bound on the row's |w| over the slice
#pragma unroll
  for (int G = 0; G < NG; ++G) {
    acc[G] = sum_abs[G] = 0.0;
    redo[G] = false;
  }
  uint32_t sl = 0u;
  for (uint32_t lt = wave; lt < ntw;) {
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    Raw45<QB> raw[2];
    read_stage<QB>(raw, hb, qb);
    // the stage is in registers: the buffer takes the next one
    const bool last = sl + 1u == nst;
    const uint32_t lt_next = last ? lt + WAVES : lt, sl_next = last ? 0u : sl + 1u;
    if (lt_next < ntw) issue(lt_next, sl_next);
    const uint32_t ia = ia0 + 8192u * sl, ua = ua0 + 512u * sl, ea = ea0 + 8u * sl,
                   da = da0 + 128u * sl;
    static_for<2>([&](auto bc) {
      constexpr int b = decltype(bc)::value;
      if (2u * sl + b >= nbl) return;  // (an odd block count's last stage)
      const Block45 bw = decode_block<QB>(raw[b], grp);
      most = fmaxf(most, fmaf(fabsf(bw.df), QB == 5 ? 31.0f * 63.0f : 15.0f * 63.0f,
                              63.0f * fabsf(bw.dminf)));
      const double bd = (double)bw.df, bdmin = (double)bw.dminf;
      static_for<NG>([&](auto gc) {
        constexpr int G = decltype(gc)::value;
        i32x4 a[4], c0 = {0, 0, 0, 0};
        uint32_t xw;
        int e;
        read_group<QB, G, b>(ia, ua, ea, da, a, xw, e, c0);
        i32x4 ch = c0, cl = c0;
        const f16x2 xs = __builtin_bit_cast(f16x2, xw);
        const f32x4 cm = __builtin_amdgcn_mfma_f32_16x16x16f16(
            f16x4{xs[0], xs[1], (_Float16)0.0f, (_Float16)0.0f}, bw.mins,
            f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          ch = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[j], bw.hi[j], ch, 0, 0, 0);
          cl = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[j], bw.lo[j], cl, 0, 0, 0);
        }
        const double m = fma(fma((double)cm[2], 4096.0, (double)cm[1]), 4096.0, (double)cm[0]);
        double t = (double)(8 * ch[3] + cl[3]);
#pragma unroll
        for (int d = 2; d >= 0; --d) t = fma(t, 256.0, (double)(8 * ch[d] + cl[d]));
        t *= bd;
        const double p = fma(-bdmin, m, t);
        redo[G] |= cancels(p, t);
        const double v = __builtin_amdgcn_ldexp(p, e);  // 0 for kBadTok
        acc[G] += v;
        sum_abs[G] += fabs(v);
      });
    });
    if (last) {
      const uint32_t row = (tg + lt * ta.groups_per_slice) * 16u + n;
#pragma unroll
      for (int G = 0; G < NG; ++G) {
        const float part = (float)acc[G];
        const bool bad = redo[G] || !(fabsf(part) < __builtin_huge_valf()) ||
                         !side_ok(most, side[G], (float)sum_abs[G]);
        const uint32_t v = 4u * G + grp;
        if (row < rows && v < ntok)
          part_out[((size_t)k * 4u * NG + v) * rows + row] =
              bad ? __uint_as_float(kPartRedo) : part;
        acc[G] = sum_abs[G] = 0.0;
        redo[G] = false;
      }
      most = 0.0f;
    }
    lt = lt_next;
    sl = sl_next;
  }
}

// ntok <= 4 NG vectors in one pass; false when the shape does not fit.
template <int W, int NG, int QB>
bool launch_tok45(const uint8_t* w, const float* x, float* y, uint32_t rows, uint32_t nb,
                  uint32_t ntok, const Workspace& ws, hipStream_t s, hipError_t* err) {
  using F = Format<QB>;
  const uint32_t cus = (uint32_t)cu_count();
  const uint32_t slices = (nb + kSliceBlocks - 1u) / kSliceBlocks;
  constexpr uint32_t kLds =
      (uint32_t)W * F::kStage + tok64_layout(kSliceBlocks, NG, true, QB == 5).total;
  static_assert(kLds <= kLdsBytes, "the stage buffers and the images fit the LDS");
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
    hipLaunchKernelGGL((q45_tokens_mfma<W, NG, QB>), dim3(ta.groups_per_slice * slices),
                       dim3(W * 64), kLds, s, wr, x, nr, nb, ntok, ws.scratch, ta);
    *err = hipGetLastError();
    if (*err != hipSuccess) break;
    launch_tok_reduce<F::kType>(ws.scratch, y + r0, nr, rows, slices, 4u * NG, ntok, wr, x, nb, s);
    *err = hipGetLastError();
  }
  return true;
}

template <int QB>
bool launch_tok45_any(const uint8_t* w, const float* x, float* y, uint32_t rows, uint32_t nb,
                      uint32_t ntok, const Workspace& ws, hipStream_t s, hipError_t* err) {
  // Twelve waves; 8 measured 17.2 / 28.7 us at M = 4 / 16 against 16.3 / 26.9
  // (Q4_K 17408 x 5120), 16 the same.
  if (ntok <= 4u) return launch_tok45<12, 1, QB>(w, x, y, rows, nb, ntok, ws, s, err);
  if (ntok <= 8u) return launch_tok45<12, 2, QB>(w, x, y, rows, nb, ntok, ws, s, err);
  if (ntok <= 12u) return launch_tok45<12, 3, QB>(w, x, y, rows, nb, ntok, ws, s, err);
  return launch_tok45<12, 4, QB>(w, x, y, rows, nb, ntok, ws, s, err);
}

}  // namespace

bool mfma::launch_q45_tokens(int qb, const uint8_t* w, const float* x, float* y, uint32_t rows,
                             uint32_t nb, uint32_t ntok, const Workspace& ws, hipStream_t s,
                             hipError_t* err) {
  return qb == 5 ? launch_tok45_any<5>(w, x, y, rows, nb, ntok, ws, s, err)
                 : launch_tok45_any<4>(w, x, y, rows, nb, ntok, ws, s, err);
}

}  // namespace sihip
