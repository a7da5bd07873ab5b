// Q6_K matvec on the gfx950 matrix cores (replaces si_q6_k_matvec* for one
// input vector, src/metal.rs:895-1081; the output head of the greedy decode
// and the MLP down projection).
//
// Weights.  quant.rs:145-171 decodes half h (128 elements) of a block from
// ql[64h .. 64h + 64), qh[32h .. 32h + 32) and scales[8h .. 8h + 8): element
// 128h + 32t + l (t = 0..3, l = 0..31) is (6-bit q) - 32 with scale
// 8h + 2t + l / 16.  Lane group g = 2h + s of the B operand owns l in
// [16s, 16s + 16) of half h for all four t: its 16-byte pieces are ql at
// 64h + 16s (low nibbles: t = 0, high: t = 2), ql at 64h + 32 + 16s (t = 1, 3)
// and qh at 128 + 32h + 16s (two bits per t), and MFMA t of a block gets one
// scale per lane.  The MFMA takes the unsigned q (0..63); a second MFMA of the
// same image with every weight byte -32 adds the offset, so each lane's digit
// sums C_t[d] = sum (q - 32) D_d are exact integers.
//
// Per block and lane: T_d = sum_t sc_t * C_t[d] in integers, y += d * (sum_d
// T_d * 256^d) * 2^(e_b - 30) (the digit images of the activations are built
// as for Q4_K, mfma_common.h).  A block with side elements is a rounded
// block, whose rows recompute it exactly when its error bound fails the
// rounded-block check (mfma_common.h); blocks whose activations are not
// finite or reach 2^100 take the exact per-weight f32 path whole
// (w = (d * sc) * (q - 32), quant.rs rounding).
//
// Data path.  Blocks are 210 bytes, so they are not 16-byte aligned; with an
// even block count nb every row and every stage of two blocks (420 bytes)
// starts on a 4-byte boundary, which the 16-byte buffer->LDS copies need (odd
// nb runs as row pairs, PAIRED below; a matrix that starts off a word, on the
// generic kernels).  A stage is copied row by row (copy_offsets): piece q of row
// r at LDS byte 432 r + 16 q, 27 pieces a row, an odd pitch.  Pieces 0..25 are
// bytes 16 q .. 16 q + 15; piece 26 is bytes 404..419, so no copy runs past the
// stage.  A copy's words past the end of its buffer descriptor read as zero, each
// word by itself.  The second block of a stage starts 2 bytes into piece 13: its
// chunks are read as two pieces and realigned with v_alignbyte.  Scheduling, the
// LDS slot ring and the finishing wave are the Q4_K kernel's (mfma_common.h).
#include "argmax_device.h"
#include "mfma_common.h"
#include "si_hip_tuned.h"
#include "tokens_common.h"

namespace sihip {
namespace {

using namespace mfma;

constexpr uint32_t kStageRowBytes = 2u * kQ6Bytes;     // 420: two blocks of one row
constexpr uint32_t kRowPieces = 27u;                   // pieces per row and stage
constexpr uint32_t kLastPiece = kStageRowBytes - 16u;  // 404: start of piece 26
constexpr uint32_t kCopies = 7u;                       // 7 x 64 lanes >= 16 rows x 27 pieces
constexpr uint32_t kStageBytes = kCopies * 1024u;      // 7168
static_assert(16u * (kRowPieces - 1u) <= kStageRowBytes && kLastPiece % 4u == 0u,
              "pieces 0..25 and 26 lie inside the stage, 4-byte aligned");
static_assert(16u * kRowPieces <= kCopies * 64u, "copies cover every piece");

__host__ __device__ constexpr Layout layout(uint32_t waves, uint32_t depth, uint32_t nb,
                                            uint32_t slots,
                                            uint32_t sums = 1u) {
  return make_layout(kStageBytes, 2u, 0u, waves, depth, nb, slots, sums);
}

// The lane's 13 pieces of a stage buffer (piece q of row n at 432 n + 16 q;
// qa = piece 4h + s, qh = piece 8 + 2h + s, sc = piece 12 of the lane's row):
//   v0 ql chunk A, v1 ql chunk B (piece +2), v2 qh chunk, v3 scales,
//   v4 piece 13 (d of block 0) -- block 0;
//   v5,v6 / v7,v8 / v9,v10 the same chunks of block 1 (13 pieces later, two
//   pieces each), v11 piece 25 (stage bytes 400..415), v12 piece 26 (bytes
//   404..419) -- its scales and d, block 1.
// (A row's 27 pieces, an odd count, so 16 lanes reading one piece of 16 rows
// meet all bank groups alike.)
__device__ __forceinline__ void lds_read_stage(uint32_t qa, uint32_t qh, uint32_t sc,
                                               u32x4 (&v)[13]) {
  asm volatile(
      "ds_read_b128 %0, %13\n"
      "ds_read_b128 %1, %13 offset:32\n"
      "ds_read_b128 %2, %14\n"
      "ds_read_b128 %3, %15\n"
      "ds_read_b128 %4, %15 offset:16\n"
      "ds_read_b128 %5, %13 offset:208\n"
      "ds_read_b128 %6, %13 offset:224\n"
      "ds_read_b128 %7, %13 offset:240\n"
      "ds_read_b128 %8, %13 offset:256\n"
      "ds_read_b128 %9, %14 offset:208\n"
      "ds_read_b128 %10, %14 offset:224\n"
      "ds_read_b128 %11, %15 offset:208\n"
      "ds_read_b128 %12, %15 offset:224\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]),
        "=&v"(v[6]), "=&v"(v[7]), "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11]),
        "=&v"(v[12])
      : "v"(qa), "v"(qh), "v"(sc)
      : "memory");
}

// The copies of a stage: copy i, lane l moves piece c % 27 of row c / 27, c =
// 64 i + l, so that a row's 420 bytes are read by consecutive lanes; the lanes
// of the last copy past the last piece re-read it.  vo[i]: the lane's offset
// from the stage's first row.  (With sixteen rows' pieces side by side, lane l
// taking row l % 16, each lane was a cache access of its own, 448 a stage
// instead of about 130: the 151936 x 5120 head 125.8 -> 120.2 us, 5120 x 5120
// 10.1 -> 9.0, 5120 x 17408 21.8 -> 21.2.)
__device__ __forceinline__ void copy_offsets(uint32_t row_bytes, uint32_t lane,
                                             uint32_t (&vo)[kCopies]) {
#pragma unroll
  for (uint32_t i = 0; i < kCopies; ++i) {
    const uint32_t c = min(64u * i + lane, 16u * kRowPieces - 1u);
    const uint32_t row = (c * 2428u) >> 16;  // c / 27 for c < 432
    vo[i] = row * row_bytes + min(16u * (c - kRowPieces * row), kLastPiece);
  }
}

// The 8 A images of a stage (block b, MFMA t at addr + 1024 b + 256 t), read
// only by the lanes in `mask`; the other lanes keep their (zero) registers.
__device__ __forceinline__ void lds_read_images(uint32_t addr, uint64_t mask, i32x4 (&a)[8]) {
  uint64_t saved;
  asm volatile(
      "s_mov_b64 %[sv], exec\n"
      "s_mov_b64 exec, %[m]\n"
      "ds_read_b128 %0, %[ad]\n"
      "ds_read_b128 %1, %[ad] offset:256\n"
      "ds_read_b128 %2, %[ad] offset:512\n"
      "ds_read_b128 %3, %[ad] offset:768\n"
      "ds_read_b128 %4, %[ad] offset:1024\n"
      "ds_read_b128 %5, %[ad] offset:1280\n"
      "ds_read_b128 %6, %[ad] offset:1536\n"
      "ds_read_b128 %7, %[ad] offset:1792\n"
      "s_waitcnt lgkmcnt(0)\n"
      "s_mov_b64 exec, %[sv]"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]),
        "+v"(a[7]), [sv] "=&s"(saved)
      : [ad] "v"(addr), [m] "s"(mask)
      : "memory");
}

// The stage's two block exponents (ea) and their side counts (one byte
// each, at ea + kCountOff).
__device__ __forceinline__ void lds_read_expo(uint32_t ea, u32x2& ex, uint32_t& cnt) {
  static_assert(kCountOff == 512, "the offset below");
  asm volatile(
      "ds_read_b64 %0, %2\n"
      "ds_read_u16 %1, %2 offset:512\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(ex), "=&v"(cnt)
      : "v"(ea)
      : "memory");
}

// Signed byte of w at bit offset `bit` (an int8 scale).
__device__ __forceinline__ int scale_at(uint32_t w, uint32_t bit) {
  return (int)__builtin_amdgcn_sbfe((int)w, bit, 8u);
}

// The 16 bytes that start 2 bytes into piece lo (and end in piece hi).
__device__ __forceinline__ u32x4 skip2(const u32x4& lo, const u32x4& hi) {
  return u32x4{__builtin_amdgcn_alignbyte(lo[1], lo[0], 2), __builtin_amdgcn_alignbyte(lo[2], lo[1], 2),
               __builtin_amdgcn_alignbyte(lo[3], lo[2], 2), __builtin_amdgcn_alignbyte(hi[0], lo[3], 2)};
}

// Unsigned 6-bit weights (0..63) of the lane's four sets t from its ql chunks
// a (l), b (l + 32) and qh chunk h (quant.rs:155-159).
__device__ __forceinline__ void q6_sets(const u32x4& a, const u32x4& b, const u32x4& h,
                                        i32x4 (&q)[4]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    q[0][k] = (int)((a[k] & 0x0f0f0f0fu) | ((h[k] << 4) & 0x30303030u));
    q[1][k] = (int)((b[k] & 0x0f0f0f0fu) | ((h[k] << 2) & 0x30303030u));
    q[2][k] = (int)(((a[k] >> 4) & 0x0f0f0f0fu) | (h[k] & 0x30303030u));
    q[3][k] = (int)(((b[k] >> 4) & 0x0f0f0f0fu) | ((h[k] >> 2) & 0x30303030u));
  }
}

// Fast-path dot of one block for one lane, its digit sums combined in f32 or (two
// vectors, as in the kernel of more) f64.
template <typename Real = float>
__device__ __forceinline__ Real block_terms(const i32x4 (&q)[4], const int (&sc)[4], float d,
                                             const i32x4& a0, const i32x4& a1, const i32x4& a2,
                                             const i32x4& a3, int eb) {
  const i32x4 zero = {0, 0, 0, 0};
  const int m32 = (int)0xe0e0e0e0u;  // -32 in every byte
  const i32x4 neg32 = {m32, m32, m32, m32};
  i32x4 c0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, q[0], zero, 0, 0, 0);
  i32x4 c1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, q[1], zero, 0, 0, 0);
  i32x4 c2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a2, q[2], zero, 0, 0, 0);
  i32x4 c3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a3, q[3], zero, 0, 0, 0);
  c0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, neg32, c0, 0, 0, 0);
  c1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, neg32, c1, 0, 0, 0);
  c2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a2, neg32, c2, 0, 0, 0);
  c3 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a3, neg32, c3, 0, 0, 0);
  int t[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    t[k] = mad_i24(sc[3], c3[k],
                   mad_i24(sc[2], c2[k], mad_i24(sc[1], c1[k], __mul24(sc[0], c0[k]))));
  if constexpr (std::is_same_v<Real, double>) {
    double tc = (double)t[3];
#pragma unroll
    for (int k = 2; k >= 0; --k) tc = fma(tc, 256.0, (double)t[k]);
    return __builtin_amdgcn_ldexp((double)d * tc, eb);
  } else {
    const float tc =
        fmaf(fmaf(fmaf((float)t[3], 256.0f, (float)t[2]), 256.0f, (float)t[1]), 256.0f, (float)t[0]);
    return __builtin_amdgcn_ldexpf(d * tc, eb);
  }
}

// Exact per-weight path of one block: xs = x of the block + 128 h + 16 s.
__device__ __forceinline__ float block_exact(const i32x4 (&q)[4], const int (&sc)[4], float d,
                                             const float* __restrict__ xs) {
  float acc = 0.0f;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int qv = (int)(((uint32_t)q[t][i >> 2] >> (8 * (i & 3))) & 0xffu) - 32;
      acc = fmaf(k6_value_exact(d, sc[t], qv), xs[32 * t + i], acc);
    }
  }
  return acc;
}

// Largest |w| of the lane's share of a block: |d| * 32 * max |scale|.
__device__ __forceinline__ float q6_bound(const int (&sc)[4], float d) {
  const int m = max(max(abs(sc[0]), abs(sc[1])), max(abs(sc[2]), abs(sc[3])));
  return fabsf(d) * (float)(32 * m);
}

// GROUPED: the rows are those
// of the group's matrices of one K, one after the other (every matrix but the
// last a whole number of tiles); tile t reads the matrix whose tiles reach
// past t.
//
// ARGMAX (one matrix): the greedy argmax of y under tie rule
// aa.rule, fused: each workgroup keeps the best candidate of the rows it
// stores, and the workgroups reduce theirs through the workspace's argmax
// area into *aa.result (argmax_device.h).
//
// SLICED (one matrix): a K-sliced launch (SliceArgs,
// mfma_common.h); the LDS holds the images and metadata of the workgroup's
// slice only, stage r of the matrix at local stage r - r_lo.
//
// VECS = 2 (one matrix, whole rows): two vectors, one after the other in x, in
// one pass over the weights: the LDS holds both vectors' images (hand_off_two).
//
// PAIRED (one matrix of an odd block count nr): the launch sees
// rows / 2 rows of nb = 2 nr blocks, row r being rows 2 r and 2 r + 1 of the
// matrix one after the other.  Such a pair of rows starts on a 4-byte
// boundary (the rows themselves alternate by 2 bytes), so the two-block
// stages and their copies are the even case's.  Block b of a launch row
// meets x block b mod nr (x sits twice in the image area); the sums of its
// blocks b < nr go to y[2 r] and the rest to y[2 r + 1], the stage that
// holds blocks nr - 1 and nr handing one sum to each.  A workgroup past those
// of the schedule takes the last row of an odd row count, alone, on the exact
// per-weight path (the launch then leaves it a CU): as a launch of its own that
// row took 4097 x 11008 to 20.5 us, here it takes 16.0.

// y[0] = the dot of one row (w: its nr blocks) with x, by a whole workgroup:
// thread t decodes units t, t + 64 WAVES, ... as quant.rs does.
template <int WAVES>
__device__ __forceinline__ void last_row_dot(const uint8_t* __restrict__ w,
                                             const float* __restrict__ x, float* __restrict__ y,
                                             uint32_t nr, uint8_t* smem) {
  float acc = 0.0f;
  for (uint32_t u = threadIdx.x; u < 8u * nr; u += 64u * WAVES) {
    float v[32];
    decode_unit_exact<kTypeQ6K>(w + (size_t)(u >> 3) * kQ6Bytes, u & 7u, v);
    const float* const xu = x + 32u * (size_t)u;
#pragma unroll
    for (int i = 0; i < 32; ++i) acc = fmaf(v[i], xu[i], acc);
  }
#pragma unroll
  for (int h = 32; h > 0; h >>= 1) acc += __shfl_xor(acc, h, 64);
  float* const part = reinterpret_cast<float*>(smem);
  if ((threadIdx.x & 63u) == 0u) part[threadIdx.x >> 6] = acc;
  __syncthreads();
  if (threadIdx.x == 0u) {
    for (int k = 1; k < WAVES; ++k) acc += part[k];
    y[0] = acc;
  }
}

struct ArgmaxArgs {
  uint64_t* result;
  uint32_t rule;
};
template <int WAVES, int DEPTH, bool GROUPED, bool ARGMAX = false, bool SLICED = false,
          bool PAIRED = false, int VECS = 1>
__global__ __launch_bounds__(WAVES * 64) void q6k_matvec_mfma(const uint8_t* __restrict__ w,
                                                              const float* __restrict__ x,
                                                              float* __restrict__ y, uint32_t rows,
                                                              uint32_t nb, void* __restrict__ wsp,
                                                              SchedArgs sa, uint32_t prefetch,
                                                              GroupArgs ga, ArgmaxArgs aa,
                                                              SliceArgs sla) {
  static_assert(!ARGMAX || !GROUPED, "argmax over one matrix");
  static_assert(!SLICED || (!GROUPED && !ARGMAX), "slices of one matrix");
  static_assert(!PAIRED || !GROUPED, "row pairs of one matrix");
  static_assert(!(PAIRED && SLICED && ARGMAX), "sliced row pairs: no argmax");
  static_assert(VECS == 1 || (VECS == 2 && !GROUPED && !ARGMAX && !SLICED && !PAIRED),
                "two vectors with whole rows of one matrix");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  if constexpr (GROUPED) load_group_args_early(ga);
  if constexpr (PAIRED && !ARGMAX) {
    if (blockIdx.x >= (SLICED ? sla.slices * sla.tgroups : sa.packed >> 16)) {
      last_row_dot<WAVES>(w + (size_t)rows * nb * kQ6Bytes, x, y + 2u * (size_t)rows, nb / 2u,
                          smem);
      return;
    }
  }
  const uint32_t slots = sa.packed & 0xffu;
  const uint32_t ntiles = (rows + 15u) / 16u;
  const uint32_t nstages = (nb + 1u) / 2u;
  // the schedule: whole and split tiles (sc), or K slices (ss)
  Sched sc{};
  SliceSched ss{};
  if constexpr (SLICED)
    ss = make_slice_sched(ntiles, sla, sa);
  else
    sc = make_sched(ntiles, nstages, WAVES, sa);
  // the stages whose images the LDS holds: [st0, st0 + nst), local index st - st0
  const uint32_t st0 = SLICED ? ss.r_lo : 0u;
  const uint32_t nbl = SLICED ? 2u * ss.ns : VECS * nb;
  const Layout L = layout(WAVES, DEPTH, SLICED ? 2u * ss.pstride : VECS * nb, slots,
                          PAIRED || VECS == 2 ? 2u : 1u);
  const uint32_t nr = nb / 2u;  // PAIRED: blocks of one matrix row
  const SplitWs ws = split_ws(wsp);
  const uint32_t wave = uniform(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t grp = lane >> 4, n = lane & 15u;
  const uint32_t half = grp >> 1, sub = grp & 1u;
  const uint32_t row_bytes = nb * kQ6Bytes;
  const uint32_t sbase = (uint32_t)(uintptr_t)smem;
  uint8_t* const wstage = smem + wave * DEPTH * kStageBytes;

  // 1. x into the image area, natural order (block b at img + 1024 b)
  if constexpr (PAIRED) {
    // x twice over; a slice, the stretch of it that its stages meet
    copy_x<WAVES>(smem, L.img, x, nbl, wave, lane, nr, 2u * st0);
  } else {
    copy_x<WAVES>(smem, L.img, x + (size_t)2u * st0 * kBlockElems, nbl, wave, lane);
  }

  // 2. this wave's pairs k = wave, wave + WAVES, ... of the workgroup's pairs
  //    (pair_at: a tile and its stage) and the copies of its first DEPTH, pair
  //    j into buffer j % DEPTH (copy_offsets).  All copies lie inside the stage's
  //    420 bytes of their row.
  auto pair_of = [&](uint32_t k) -> Pair {
    if constexpr (SLICED)
      return pair_at(ss, k);
    else
      return pair_at(sc, k, nstages);
  };
  const uint32_t npairs = SLICED ? ss.npairs : sc.npairs;
  uint32_t vo[kCopies];
  copy_offsets(row_bytes, lane, vo);
  const uint32_t my_pairs = wave < npairs ? (npairs - 1u - wave) / WAVES + 1u : 0u;
  // the stage bytes of a pair's tile and the tile's row count
  auto tile_at = [&](const Pair& pr, uint32_t& nrows) -> const uint8_t* {
    uint32_t row0 = pr.tile * 16u, mrows = rows;
    const uint8_t* wm = w;
    if constexpr (GROUPED) {
      wm = ga.w[0];
      mrows = ga.rows[0];
#pragma unroll
      for (uint32_t k = 1; k < kMaxGroup; ++k)
        if (pr.tile >= ga.tile_end[k - 1]) {
          wm = ga.w[k];
          mrows = ga.rows[k];
          row0 = (pr.tile - ga.tile_end[k - 1]) * 16u;
        }
    }
    nrows = min(16u, mrows - row0);
    return wm + (size_t)row0 * row_bytes + kStageRowBytes * pr.r;
  };
  auto issue = [&](uint32_t j) {
    const Pair pr = pair_of(wave + j * WAVES);
    const uint32_t st = pr.r;
    uint32_t nrows;
    const uint8_t* sb = tile_at(pr, nrows);
    // the descriptor ends at the tile's last row: pieces past it read zero
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(sb), 0, (int)(nrows * row_bytes - kStageRowBytes * st),
        kBufferWord3);
    uint8_t* dst = wstage + (j % DEPTH) * kStageBytes;
#pragma unroll
    for (int i = 0; i < (int)kCopies; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void*)(dst + 1024 * i), 16, vo[i], 0, 0,
                                                0);
  };
  // A long image build (48 blocks or more in the workgroup's range, every
  // wave a builder): the ring slots are set and a barrier passed first, so
  // that every wave's x copies go out ahead of all weight copies, and a
  // builder past the first round of waves (one per SIMD) builds before it
  // issues its own copies -- the memory queue, full of the first round's
  // copies, would hold it at them, and its images, for microseconds (the
  // 68-block down projection's images were done 3 us later that way).
  const bool long_build = nbl >= 48u;
  if (long_build) {
    init_slots<WAVES>(sbase, L, slots);
    lds_wait();
    __builtin_amdgcn_s_barrier();
  }
  const bool build_first = long_build && wave >= 4u && 4u * wave < nbl;
  // With one stage in flight, up to `prefetch` (<= 2) later pairs of the wave
  // are touched into L2 while the images are built: every 128-byte line of
  // their rows' 420 bytes is read 4 bytes wide (offsets 0, 128, 256, 384 and
  // 416 of each row) into a 256-byte LDS sink past the layout that nothing
  // reads.  Their copies then find the lines in L2.
  const uint32_t npf = DEPTH == 1 && my_pairs > 1u ? min(min(prefetch, 2u), my_pairs - 1u) : 0u;
  auto issue_first = [&]() {
#pragma unroll
    for (int j = 0; j < DEPTH; ++j)
      if ((uint32_t)j < my_pairs) issue(j);
    for (uint32_t j = 1; j <= npf; ++j) {
      const Pair pr = pair_of(wave + j * WAVES);
      uint32_t nrows;
      const uint8_t* sb = tile_at(pr, nrows);
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint8_t*>(sb), 0, (int)(nrows * row_bytes - kStageRowBytes * pr.r),
          kBufferWord3);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void*)(smem + L.total), 4,
                                                n * row_bytes + 128u * grp, 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void*)(smem + L.total), 4,
                                                n * row_bytes + kStageRowBytes - 4u, 0, 0, 0);
    }
  };
  if (!build_first) issue_first();

  // 3. ring slots (unless set above), then (once the x copies have landed)
  //    digit images and exponents
  if (!long_build) init_slots<WAVES>(sbase, L, slots);
  // the stage copies (then the touches) were issued after x's and complete in
  // order
  const uint32_t early = build_first ? 0u : min((uint32_t)DEPTH, my_pairs);
  if (early >= 3u)
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(3 * kCopies));
  else if (early == 2u)
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 * kCopies));
  else if (early == 1u && npf == 2u)
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(kCopies + 4));
  else if (early == 1u && npf == 1u)
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(kCopies + 2));
  else if (early == 1u)
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(kCopies));
  else
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
  // chunk c = 8 h + 2 t + s: MFMA t of lane group 2 h + s
  build_images<WAVES>(sbase, L, nbl, wave, grp, n, [](uint32_t c) {
    return 256u * ((c >> 1) & 3u) + 64u * (2u * (c >> 3) + (c & 1u));
  });
  if (build_first) issue_first();
  lds_wait();
  __builtin_amdgcn_s_barrier();

  // 4. the wave's pairs
  const bool upper = half != 0u;  // lane groups 2, 3: scales 8..15
  const uint32_t base = sbase + wave * DEPTH * kStageBytes + 16u * kRowPieces * n;
  const uint32_t qa0 = base + 16u * (4u * half + sub);
  const uint32_t qh0 = base + 16u * (8u + 2u * half + sub);
  const uint32_t sc0 = base + 16u * 12u;
  const uint32_t sb_lo = 8u * sub, sb_hi = 8u * sub + 16u;  // bit offsets of the lane's scales
  i32x4 A[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) A[t] = i32x4{0, 0, 0, 0};
  uint64_t best = 0u;  // ARGMAX: the best candidate of the rows this lane stored
  uint32_t fail = 0u;  // a bounded wait that gave up (kDevErr*)
  for (uint32_t j = 0; j < my_pairs; ++j) {
    const Pair pr = pair_of(wave + j * WAVES);
    const uint32_t st = pr.r, ls = st - st0;  // matrix stage, LDS stage
    const uint32_t later = min((uint32_t)DEPTH - 1u, my_pairs - 1u - j);
    if (DEPTH >= 3 && later >= 2u)
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 * kCopies));
    else if (DEPTH >= 2 && later >= 1u)
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(kCopies));
    else
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    const uint32_t buf = (j % DEPTH) * kStageBytes;
    u32x4 v[13];
    lds_read_stage(qa0 + buf, qh0 + buf, sc0 + buf, v);
    if (j + DEPTH < my_pairs) issue(j + DEPTH);  // the buffer just read is free again
    u32x2 ex;
    uint32_t cnt;
    if constexpr (VECS == 1) {
      lds_read_images(sbase + L.img + 2048u * ls + 16u * n, kActiveLanes, A);
      lds_read_expo(sbase + L.expo + 8u * ls, ex, cnt);
    }
    // block 0: scales[8h + s + 2t] = bytes s, s + 2 of words 2h, 2h + 1 of v3
    i32x4 q0[4];
    q6_sets(v[0], v[1], v[2], q0);
    const uint32_t w0 = upper ? v[3][2] : v[3][0], w1 = upper ? v[3][3] : v[3][1];
    const int sc_0[4] = {scale_at(w0, sb_lo), scale_at(w0, sb_hi), scale_at(w1, sb_lo),
                         scale_at(w1, sb_hi)};
    const float d0 = half_bits_to_float(v[4][0] & 0xffffu);
    // block 1: its scale j < 14 is byte 2 + j of piece 25; scales 14, 15 and
    // d are the last word of piece 26
    i32x4 q1[4];
    q6_sets(skip2(v[5], v[6]), skip2(v[7], v[8]), skip2(v[9], v[10]), q1);
    const uint32_t u0 = upper ? v[11][2] : v[11][0], u1 = upper ? v[11][3] : v[11][1];
    const uint32_t u2 = upper ? v[12][3] : v[11][2];
    const int sc_1[4] = {scale_at(u0, sb_hi), scale_at(u1, sb_lo), scale_at(u1, sb_hi),
                         scale_at(u2, sb_lo)};
    const float d1 = half_bits_to_float(v[12][3] >> 16);

    if constexpr (VECS == 2) {
      // one vector after the other, the second one's images a row's stages on (a
      // loop kept as one, with the exact path's decode kept inside it: both
      // vectors' unrolled, or 128 decoded weights held for them, spill)
      auto exact = [&](const i32x4 (&q)[4], const int (&sc)[4], float d, const float* xs) {
        i32x4 own[4] = {q[0], q[1], q[2], q[3]};
        asm volatile("" : "+v"(own[0]), "+v"(own[1]), "+v"(own[2]), "+v"(own[3]));
        return block_exact(own, sc, d, xs);
      };
      double sum1 = 0.0, sum2 = 0.0;
#pragma unroll 1
      for (uint32_t vec = 0; vec < 2u; ++vec) {
        const uint32_t at = ls + vec * nstages;
        lds_read_images(sbase + L.img + 2048u * at + 16u * n, kActiveLanes, A);
        lds_read_expo(sbase + L.expo + 8u * at, ex, cnt);
        const int e0 = __builtin_amdgcn_readfirstlane(ex[0]);
        const int e1 = __builtin_amdgcn_readfirstlane(ex[1]);
        const double c0 = block_terms<double>(q0, sc_0, d0, A[0], A[1], A[2], A[3], e0);
        const double c1 = block_terms<double>(q1, sc_1, d1, A[4], A[5], A[6], A[7], e1);
        double s0 = e0 != kBadBlock ? c0 : 0.0, s1 = e1 != kBadBlock ? c1 : 0.0;
        const uint32_t counts = __builtin_amdgcn_readfirstlane(cnt);
        uint32_t redo = 0u;
        if (counts != 0u) {
          const float pp[2] = {(float)s0, (float)s1};
          redo = rounded_redo<2>(sbase + L.expo + L.side_off + 2u * kSideBytes * at, counts, grp,
                                 pp, [&](auto b) {
                                   return decltype(b)::value == 0 ? q6_bound(sc_0, d0)
                                                                  : q6_bound(sc_1, d1);
                                 });
        }
        const float* const xs = x + 256u * (size_t)(vec * nb) + 512u * st + 128u * half + 16u * sub;
        if (e0 == kBadBlock || (redo & 1u)) s0 = exact(q0, sc_0, d0, xs);
        if (e1 == kBadBlock || (redo & 2u)) s1 = exact(q1, sc_1, d1, xs + 256);
        sum1 = sum2;
        sum2 = sum_lane_groups(s0 + s1);
      }
      hand_off_two(sbase, L, slots, sc, pr, nstages, sum1, sum2, lane, rows, y, fail);
      continue;
    }
    const int e0 = __builtin_amdgcn_readfirstlane(ex[0]);
    const int e1 = __builtin_amdgcn_readfirstlane(ex[1]);
    const float c0 = block_terms(q0, sc_0, d0, A[0], A[1], A[2], A[3], e0);
    const float c1 = block_terms(q1, sc_1, d1, A[4], A[5], A[6], A[7], e1);
    float pp[2] = {e0 != kBadBlock ? c0 : 0.0f, e1 != kBadBlock ? c1 : 0.0f};
    const float* const xs = x + 512u * st + 128u * half + 16u * sub;
    const uint32_t counts = __builtin_amdgcn_readfirstlane(cnt);
    uint32_t redo = 0u;
    if (counts != 0u) {
      const uint32_t list = sbase + L.expo + L.side_off + 2u * kSideBytes * ls;
      redo = rounded_redo<2>(list, counts, grp, pp, [&](auto b) {
        return decltype(b)::value == 0 ? q6_bound(sc_0, d0) : q6_bound(sc_1, d1);
      });
    }
    if constexpr (PAIRED) {
      // the blocks' own x blocks (b mod nr) on the exact path, and each
      // block's sum to its row of the pair
      const uint32_t vb0 = 2u * st, vb1 = vb0 + 1u;
      const float* const x0 = x + 256u * (vb0 < nr ? vb0 : vb0 - nr) + 128u * half + 16u * sub;
      const float* const x1 = x + 256u * (vb1 < nr ? vb1 : vb1 - nr) + 128u * half + 16u * sub;
      if (e0 == kBadBlock || (redo & 1u)) pp[0] = block_exact(q0, sc_0, d0, x0);
      if (e1 == kBadBlock || (redo & 2u)) pp[1] = block_exact(q1, sc_1, d1, x1);
      float ra = 0.0f, rb = 0.0f;
      if (vb1 < nr) {
        ra = sum_lane_groups(pp[0] + pp[1]);
      } else if (vb0 >= nr) {
        rb = sum_lane_groups(pp[0] + pp[1]);
      } else {
        ra = sum_lane_groups(pp[0]);
        rb = sum_lane_groups(pp[1]);
      }
      if constexpr (SLICED)
        hand_off_slice<true>(sbase, L, ss, pr, ra, lane, rows, y, ws, fail, rb);
      else
        hand_off<1, ARGMAX, true>(sbase, L, slots, sc, pr, nstages, ra, lane, rows, y, ws,
                                  fail, &best, aa.rule, rb);
      continue;
    }
    if (e0 == kBadBlock || (redo & 1u)) pp[0] = block_exact(q0, sc_0, d0, xs);
    if (e1 == kBadBlock || (redo & 2u)) pp[1] = block_exact(q1, sc_1, d1, xs + 256);
    const float rowsum = sum_lane_groups(pp[0] + pp[1]);

    // hand the 16 row partials to the tile's slot; the last stage finishes it
    if constexpr (SLICED)
      hand_off_slice(sbase, L, ss, pr, rowsum, lane, rows, y, ws, fail);
    else
      hand_off<1, ARGMAX>(sbase, L, slots, sc, pr, nstages, rowsum, lane, rows, y, ws, fail,
                          &best, aa.rule);
  }
  if (fail != 0u) report_device_error(wsp, fail);
  if constexpr (ARGMAX) {
    // the workgroup's best, once every wave is done with the LDS, then the
    // grid's through the workspace
    best = wave_max_u64(best);
    __syncthreads();
    uint64_t* const wave_best = reinterpret_cast<uint64_t*>(smem);
    if (lane == 0u) wave_best[wave] = best;
    __syncthreads();
    if (wave == 0u) {
      const uint64_t m = lane < (uint32_t)WAVES ? wave_best[lane] : 0u;
      argmax_publish_wave(wave_max_u64(m), wsp, aa.result, lane);
    }
  }
}

// ---- Several activation vectors in the MFMA rows ---------------------------
//
// A pass over the weights with up to sixteen activation vectors (matmul-many,
// replacing si_q6_k_matmul_many, metal.rs:1052-1262; the batched head of
// qwen35_runtime.rs:2194-2197 takes up to eight candidates) puts the vectors
// in the rows of the A operand of v_mfma_i32_16x16x64_i8 (group images of
// four vectors, tokens_common.h) and folds each weight's int8 scale into the
// B operand: sc (q - 32), 13 bits signed, as two int8 digits of base 256.
// 16-bit lanes form P = sc q + (128 - 32 sc), two weights per v_pk_mad_u16; its
// high byte is the high digit and its low byte less 128 the low one.  A block
// meets four vectors in eight MFMAs whose sums need no scale, and result lane
// (g, n) of group G has the four digit sums of vector 4 G + g and row n, T_d =
// 256 hi + lo (|T_d| < 2^28), summed over d in f64.  (With the scales applied to
// the MFMA results, 64 multiply-adds per four vectors and block, and K = 32
// MFMAs half of whose A rows were zero, sixteen vectors took the 151936 x 5120
// head 318 us.)
//
// K slices and stages.  A launch cuts K into slices of four blocks: workgroup
// g works on slice g / GS for tiles g % GS, g % GS + GS, ..., keeping that
// slice's images in LDS; each wave takes (tile, slice) pairs, their two-block
// stages one after another through one stage buffer (the next stage's copy
// goes out once the stage is in registers), and stores the vectors' sums over
// the slice in the scratch; tok_reduce adds the slices in order.  A launch
// whose sums exceed the scratch runs as several over row ranges.  A (vector,
// row) that meets a block on the exact path, whose sum is not finite, or
// whose side elements (half a unit each times 4096 |d|, the largest |w| a
// block can hold) could be off by more than they may be (kFewTol,
// tokens_common.h) stores kPartRedo for the slice, and tok_reduce recomputes it
// exactly.
//
// PAIRED (odd block counts, where a row starts 2 bytes off 4 every second
// time): the even rows and the odd rows as two matrices of row stride 2 nb
// blocks, nb + 1 blocks wide so that both start aligned and the stages are
// whole: an even row with the block after it, an odd row with the block before
// it, whose activations read as zero.  Slices 0 .. `slices` - 1 are the even
// rows', the next `slices` the odd rows', and a "row" here is a pair.
// 4096 x 11008, M = 2 / 4 / 8 / 16: 28.3 / 55.3 / 108.5 / 215.6 us one vector
// at a time, 15.3 / 15.5 / 17.4 / 20.5 so.
constexpr uint32_t kTokBlocks = kStageBlocks;

struct Q6TokArgs {
  uint32_t groups_per_slice, m_gps;
  uint32_t slices;  // PAIRED
};

// The two digits of the lane's 64 scaled weights of a block: set t's four
// words of 6-bit q and its scale.
__device__ __forceinline__ void q6_digits(const i32x4 (&q)[4], const int (&sc)[4],
                                          i32x4 (&hi)[4], i32x4 (&lo)[4]) {
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const uint16_t s = (uint16_t)sc[t], o = (uint16_t)(128 - 32 * sc[t]);
    const u16x2 s2 = {s, s}, o2 = {o, o};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t w = (uint32_t)q[t][k];
      const u16x2 even = __builtin_bit_cast(u16x2, w & 0x00ff00ffu);
      const u16x2 odd = __builtin_bit_cast(u16x2, __builtin_amdgcn_perm(0u, w, 0x0c030c01u));
      const uint32_t pe = __builtin_bit_cast(uint32_t, (u16x2)(even * s2 + o2));
      const uint32_t po = __builtin_bit_cast(uint32_t, (u16x2)(odd * s2 + o2));
      hi[t][k] = (int)__builtin_amdgcn_perm(po, pe, 0x07030501u);
      lo[t][k] = (int)(__builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u);
    }
  }
}

// Group G's four A operands of block B of a stage (ia: the lane's place in the
// stage's first image of group 0) and the exponent of the lane's vector (ea).
template <int G, int B>
__device__ __forceinline__ void lds_read_group(uint32_t ia, uint32_t ea, i32x4 (&a)[4], int& e) {
  constexpr int kAt = 4096 * ((int)kTokBlocks * G + B);
  asm volatile(
      "ds_read_b128 %0, %5 offset:%7\n"
      "ds_read_b128 %1, %5 offset:%8\n"
      "ds_read_b128 %2, %5 offset:%9\n"
      "ds_read_b128 %3, %5 offset:%10\n"
      "ds_read_b32 %4, %6 offset:%11\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(a[0]), "=&v"(a[1]), "=&v"(a[2]), "=&v"(a[3]), "=&v"(e)
      : "v"(ia), "v"(ea), "i"(kAt), "i"(kAt + 1024), "i"(kAt + 2048), "i"(kAt + 3072),
        "i"(16 * (int)kTokBlocks * G + 4 * B)
      : "memory");
}

template <int WAVES, int NG, bool PAIRED>
__global__ __launch_bounds__(WAVES * 64) void q6k_tokens_mfma(const uint8_t* __restrict__ w,
                                                              const float* __restrict__ x,
                                                              uint32_t rows, uint32_t nb,
                                                              uint32_t ntok,
                                                              float* __restrict__ part_out,
                                                              Q6TokArgs ta) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr uint32_t kImages = (uint32_t)WAVES * kStageBytes;  // after the stage buffers
  constexpr TokLayout L = tok64_layout(kTokBlocks, NG, false, false);
  const uint32_t wave = uniform(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t grp = lane >> 4, n = lane & 15u;
  const uint32_t half = grp >> 1, sub = grp & 1u;
  const uint32_t row_bytes = (PAIRED ? 2u : 1u) * nb * kQ6Bytes;
  const uint32_t sbase = (uint32_t)(uintptr_t)smem;
  uint8_t* const wstage = smem + wave * kStageBytes;

  // this workgroup's slice k (blocks blk0 .. blk0 + nbl - 1, nst stages) and
  // its tiles tg, tg + GS, ...; the wave's are tiles wave, wave + WAVES, ...
  const FastDiv by_gps{ta.groups_per_slice, ta.m_gps};
  const uint32_t k = quo(blockIdx.x, by_gps);
  const uint32_t tg = blockIdx.x - k * ta.groups_per_slice;
  const uint32_t odd = PAIRED && k >= ta.slices ? 1u : 0u;
  const uint32_t ks = PAIRED ? k - odd * ta.slices : k;
  auto first = [&](uint32_t i) {
    return PAIRED ? paired_slice_first(i, nb, odd) : kTokBlocks * i;
  };
  const uint32_t blk0 = first(ks);
  const uint32_t nbl = min(first(ks + 1u), nb + (PAIRED ? 1u : 0u)) - blk0, nst = nbl / 2u;
  const uint32_t places = PAIRED ? (rows + 1u) / 2u : rows;  // of the partials
  const uint32_t trows = odd ? rows / 2u : places;           // the slice's rows
  const uint32_t ntiles = (trows + 15u) / 16u;
  const uint32_t ntw = tg < ntiles ? quo(ntiles - 1u - tg, by_gps) + 1u : 0u;

  // 1. the activations of the wave's image blocks into registers, then the
  //    copy of its first stage (copy_offsets; rows past the matrix read zero)
  constexpr int kShare = (NG * (int)kTokBlocks + WAVES - 1) / WAVES;
  u32x4 xq[kShare][4];
  load_group_x<WAVES, kShare>(xq, x, nb, blk0 - odd, nbl, NG, ntok, wave, lane);
  uint32_t vo[kCopies];
  copy_offsets(row_bytes, lane, vo);
  auto issue = [&](uint32_t lt, uint32_t sl) {
    const uint32_t row0 = (tg + lt * ta.groups_per_slice) * 16u;
    const uint32_t nrows = min(16u, trows - row0);
    uint32_t at = kQ6Bytes * blk0 + kStageRowBytes * sl;
    if constexpr (PAIRED) at += odd * (nb - 1u) * kQ6Bytes;
    uint32_t size = nrows * row_bytes;
    if constexpr (PAIRED) {
      // the last pair of an odd row count is one row, its last 2 bytes the
      // lower half of a word: the size is rounded up to that word, which the last
      // block's d lies in (the words of its piece past it read as zero)
      if (2u * (row0 + nrows) > rows) size = (size - nb * kQ6Bytes + 3u) & ~3u;
    }
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(w + (size_t)row0 * row_bytes + at), 0, (int)(size - at),
        kBufferWord3);
#pragma unroll
    for (int i = 0; i < (int)kCopies; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void*)(wstage + 1024 * i), 16, vo[i], 0,
                                                0, 0);
  };
  if (wave < ntw) issue(wave, 0u);

  // 2. the group images: chunk c = 8 h + 2 t + s meets lane group 2 h + s in MFMA t
  build_group_images64<WAVES, kShare, false, false>(
      sbase + kImages, L, xq, nbl, NG, wave, lane,
      [](uint32_t c) { return 1024u * ((c >> 1) & 3u) + 256u * (2u * (c >> 3) + (c & 1u)); });
  lds_wait();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  float side[NG];
#pragma unroll
  for (int G = 0; G < NG; ++G)
    side[G] = slice_err(smem + kImages + L.rerr + 64 * G + 16u * grp, nbl);

  // 3. the wave's tiles, stage by stage: lane (grp, n) accumulates, for each
  //    group G, vector 4 G + grp, row n
  const uint32_t base = sbase + wave * kStageBytes + 16u * kRowPieces * n;
  const uint32_t qa0 = base + 16u * (4u * half + sub);
  const uint32_t qh0 = base + 16u * (8u + 2u * half + sub);
  const uint32_t sc0 = base + 16u * 12u;
  const uint32_t sb_lo = 8u * sub, sb_hi = 8u * sub + 16u;  // bit offsets of the lane's scales
  const bool upper = half != 0u;                            // scales 8..15
  const uint32_t ia0 = sbase + kImages + L.img + 16u * lane;
  const uint32_t ea0 = sbase + kImages + L.expo + 16u * grp;
  double acc[NG], sum_abs[NG];
  float most = 0.0f;  // bound on the row's |w| over the slice
#pragma unroll
  for (int G = 0; G < NG; ++G) acc[G] = sum_abs[G] = 0.0;
  uint32_t sl = 0u;
  for (uint32_t lt = wave; lt < ntw;) {
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    u32x4 v[13];
    lds_read_stage(qa0, qh0, sc0, v);
    // the stage is in registers: the buffer takes the next one
    const bool last = sl + 1u == nst;
    const uint32_t lt_next = last ? lt + WAVES : lt, sl_next = last ? 0u : sl + 1u;
    if (lt_next < ntw) issue(lt_next, sl_next);
    const uint32_t ia = ia0 + 8192u * sl, ea = ea0 + 8u * sl;
    static_for<2>([&](auto bc) {
      constexpr int b = decltype(bc)::value;
      // block 0: scales[8h + s + 2t] = bytes s, s + 2 of words 2h, 2h + 1 of v3;
      // block 1: its scale j < 14 is byte 2 + j of piece 25, scales 14, 15 and
      // d are the last word of piece 26
      i32x4 q[4];
      int sc[4];
      float d;
      if constexpr (b == 0) {
        q6_sets(v[0], v[1], v[2], q);
        const uint32_t w0 = upper ? v[3][2] : v[3][0], w1 = upper ? v[3][3] : v[3][1];
        sc[0] = scale_at(w0, sb_lo);
        sc[1] = scale_at(w0, sb_hi);
        sc[2] = scale_at(w1, sb_lo);
        sc[3] = scale_at(w1, sb_hi);
        d = half_bits_to_float(v[4][0] & 0xffffu);
      } else {
        q6_sets(skip2(v[5], v[6]), skip2(v[7], v[8]), skip2(v[9], v[10]), q);
        const uint32_t u0 = upper ? v[11][2] : v[11][0], u1 = upper ? v[11][3] : v[11][1];
        const uint32_t u2 = upper ? v[12][3] : v[11][2];
        sc[0] = scale_at(u0, sb_hi);
        sc[1] = scale_at(u1, sb_lo);
        sc[2] = scale_at(u1, sb_hi);
        sc[3] = scale_at(u2, sb_lo);
        d = half_bits_to_float(v[12][3] >> 16);
      }
      i32x4 hi[4], lo[4];
      q6_digits(q, sc, hi, lo);
      most = fmaxf(most, 4096.0f * fabsf(d));
      const double dd = (double)d;
      static_for<NG>([&](auto gc) {
        constexpr int G = decltype(gc)::value;
        i32x4 a[4];
        int e;
        lds_read_group<G, b>(ia, ea, a, e);
        i32x4 ch = {0, 0, 0, 0}, cl = {0, 0, 0, 0};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          ch = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[t], hi[t], ch, 0, 0, 0);
          cl = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[t], lo[t], cl, 0, 0, 0);
        }
        double t = (double)(256 * ch[3] + cl[3]);
#pragma unroll
        for (int c = 2; c >= 0; --c) t = fma(t, 256.0, (double)(256 * ch[c] + cl[c]));
        const double term = __builtin_amdgcn_ldexp(t * dd, e);  // 0 for kBadTok
        acc[G] += term;
        sum_abs[G] += fabs(term);
      });
    });
    if (last) {
      const uint32_t row = (tg + lt * ta.groups_per_slice) * 16u + n;
#pragma unroll
      for (int G = 0; G < NG; ++G) {
        const float part = (float)acc[G];
        const bool redo = !(fabsf(part) < __builtin_huge_valf()) ||
                          !side_ok(most, side[G], (float)sum_abs[G]);
        const uint32_t vec = 4u * G + grp;
        if (row < trows && vec < ntok)
          part_out[((size_t)k * 4u * NG + vec) * places + row] =
              redo ? __uint_as_float(kPartRedo) : part;
        acc[G] = sum_abs[G] = 0.0;
      }
      most = 0.0f;
    }
    lt = lt_next;
    sl = sl_next;
  }
}

template <int W, int D, bool G = false, bool AM = false, bool P = false, int V = 1>
bool launch_wd(const uint8_t* w, const float* x, float* y, uint32_t rows, uint32_t nb,
               const Workspace& ws, hipStream_t s, hipError_t* err,
               const GroupArgs& ga = GroupArgs{}, const ArgmaxArgs& aa = ArgmaxArgs{},
               bool last_row = false) {
  const uint32_t ntiles = (rows + 15u) / 16u;
  const uint32_t nstages = (nb + 1u) / 2u;
  // (two vectors: whole tiles, as without a workspace)
  const LaunchShape ls = launch_shape(ntiles, nstages, W, V == 2 ? 0u : ws.bytes, P ? 2u : 1u,
                                      (uint32_t)cu_count() - (last_row ? 1u : 0u));
  const uint32_t grid = ls.groups;
  const uint32_t slots = ring_slots(W, D, ls.tiles_per_group, (V == 2 ? 4u : P ? 2u : 1u) * nstages);
  // One pair touched ahead pays where the image build is long (the 68-block
  // down projection: 1 us of 22); with 20 blocks (the output head) it costs.
  static const int pf_env = env_int("SI_HIP_Q6K_PREFETCH", -1);
  const uint32_t prefetch = pf_env >= 0 ? (uint32_t)pf_env : (nb >= 48u ? 1u : 0u);
  const uint32_t lds =
      layout(W, D, V * nb, slots, P || V == 2 ? 2u : 1u).total + (D == 1 && prefetch ? 256u : 0u);
  SchedArgs sa;
  if (lds > kLdsBytes || !make_sched_args(ntiles, nstages, slots, ls, &sa)) return false;
  // the argmax: an entry per workgroup, the waves' candidates at the LDS start
  if (AM && (grid > kArgmaxMaxGroups || (P ? 2u : 1u) * (uint64_t)rows >= kArgmaxMaxRows ||
             ws.bytes < kWorkspaceBytes))
    return false;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&q6k_matvec_mfma<W, D, G, AM, false, P, V>),
      hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes);
  if (attr != hipSuccess) {
    *err = attr;
    return true;
  }
  hipLaunchKernelGGL((q6k_matvec_mfma<W, D, G, AM, false, P, V>),
                     dim3(grid + (last_row ? 1u : 0u)), dim3(W * 64), lds, s, w, x, y, rows, nb,
                     ws.ptr, sa, D == 1 ? prefetch : 0u, ga, aa, SliceArgs{});
  *err = hipGetLastError();
  return true;
}

// A K-sliced launch in S slices (false when the shape or the LDS does not fit).
// P: row pairs, rows and nb being the pairs' (rows / 2 rows of 2 nr blocks).
template <int W, int D, bool P = false>
bool launch_sliced(const uint8_t* w, const float* x, float* y, uint32_t rows, uint32_t nb,
                   uint32_t S, const Workspace& ws, hipStream_t s, hipError_t* err,
                   bool last_row = false) {
  const uint32_t ntiles = (rows + 15u) / 16u;
  const uint32_t nstages = nb / 2u;
  // even nb (4-byte aligned rows and stages); in-tile offsets (16 rows) and
  // descriptor sizes are 32-bit; the slice's blocks bound the LDS metadata
  if (rows == 0u || nb == 0u || (nb & 1u) != 0u || (uint64_t)nb * kQ6Bytes * 16u > 0x7fffffffu)
    return false;
  SliceShape sh;
  if (!slice_shape(ntiles, nstages, S, (uint32_t)cu_count() - (last_row ? 1u : 0u), ws.bytes, &sh,
                   P ? 128u : 64u))
    return false;
  if (2u * sh.ns_max > kMaxMetaBlocks) return false;
  const uint32_t slots = ring_slots(W, D, sh.tiles_per_group, sh.ns_max);
  static const int pf_env = env_int("SI_HIP_Q6K_PREFETCH", -1);
  const uint32_t prefetch = D == 1 && pf_env > 0 ? (uint32_t)pf_env : 0u;
  const uint32_t lds =
      layout(W, D, 2u * sh.ns_max, slots, P ? 2u : 1u).total + (prefetch ? 256u : 0u);
  if (lds > kLdsBytes || slots > 0xffu || sh.groups > 0xffffu) return false;
  SchedArgs sa{};
  sa.packed = (sh.groups << 16) | slots;
  sa.m_slots = div_magic(slots);
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&q6k_matvec_mfma<W, D, false, false, true, P>),
      hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes);
  if (attr != hipSuccess) {
    *err = attr;
    return true;
  }
  hipLaunchKernelGGL((q6k_matvec_mfma<W, D, false, false, true, P>),
                     dim3(sh.groups + (last_row ? 1u : 0u)), dim3(W * 64), lds, s, w, x, y, rows,
                     nb, ws.ptr, sa, prefetch, GroupArgs{}, ArgmaxArgs{}, sh.args);
  *err = hipGetLastError();
  return true;
}

// Slices for a one-vector launch, or 0.  A workgroup builds the images of
// the blocks it reads before its first stage, about 0.07-0.1 us per block,
// and only its first stages (one per wave, plus a pair touched into L2) are
// in flight meanwhile; slicing shrinks the build S-fold but rounds each
// slice's stages and each workgroup's tiles up.  Measured (MI355X, us):
//   rows x cols      unsliced  S = 2   S = 3   S = 4
//   640 x 17408        10.4     10.2     8.6     8.4
//   2560 x 17408       15.6     17.6    14.7    15.3
//   2048 x 16384       12.3     10.6    13.7    11.1
//   512 x 12288        10.1      8.1     7.3     7.2
//   4096 x 14336       15.3     16.7    19.4    16.1
//   5120 x 17408       21.9     24.2    24.7    24.3
//   8192 x 28672       49.9     48.2    55.8    54.6
//   2048 x 32768       51.2     17.7    20.3    18.1
//   2560 x 9728         9.7     10.3     9.6     9.9
// and, rows of odd block counts taken as pairs (four waves unsliced): 4096 x
// 11008 - / 14.5 / 16.1 / 14.8, 2047 x 11008 - / 12.3 / 9.9 / 12.4, 8192 x 11008
// 21.9 / 23.1 / 26.3 / 22.2, 1360 x 17408 11.2 / 10.8 / 9.6 / 10.2.
// and, with more pairs in rows whose images leave room for four waves at most
// (unsliced / S = 2 / 3 / 4; - : not even those):
//   3000 x 23552   24.9 / 22.1 / 23.1 / 21.7    5120 x 23552   35.9 / 32.4 / 31.2 / 33.5
//   7000 x 24064   43.3 / 40.0 / 43.8 / 44.3   15062 x 25088   79.5 / 78.5 / 81.3 / 85.7
//  24000 x 24064  110.8 / 115 / 120 / 131      30000 x 25088  140.1 / 144 / 149 / 164
//   8192 x 32768      - / 51.5 / 59.1 / 57.2   10000 x 14080      - / 38.0 / 36.2 / 37.0
//  24000 x 11520   66.9 / 60.2 / 62.1 / 67.0 (row pairs)
//  10000 x 11008      - /    - / 31.0 / 29.5   10000 x 11520   38.4 / 33.3 / 31.4 / 33.1
// A pair costs 3 % more in three slices than in two and 22 % more in four (12 %
// with row pairs).
// So: four slices, or three where that leaves the busiest workgroup fewer
// pairs, when the unsliced launch's busiest workgroup has at most two rounds
// of pairs (24; its build is then exposed) and slicing adds it none or the
// rows are long (48 blocks or more); with more pairs, only when the unsliced
// images leave room for fewer than eight waves (very long rows), in the
// number of two to four whose busiest workgroup takes the least time, except
// that whole rows stay where four waves fit and more than 250 pairs hide their
// build.
uint32_t q6_slices(uint32_t ntiles, uint32_t nb, size_t ws_bytes, bool pairs = false,
                   uint64_t cus = (uint64_t)cu_count()) {
  static const int env = env_int("SI_HIP_Q6K_SLICES", -1);
  if (env >= 0) return (uint32_t)env;
  const uint32_t nst = nb / 2u;
  if (nst < 16u) return 0u;
  auto most = [&](uint32_t S) {  // the busiest sliced workgroup's pairs
    const uint64_t gs = std::min<uint64_t>(ntiles, cus / S);
    return (ntiles + gs - 1u) / gs * ((nst + S - 1u) / S);
  };
  if (nb > kMaxMetaBlocks) {
    // rows longer than the unsliced kernel takes must slice: the fewest
    // slices (from four) whose images (64 blocks at most) leave the stage
    // buffers of 12 waves room in the LDS
    uint32_t S = 4u;
    while (S < 64u && S < cus && (nst + S - 1u) / S > 32u) S *= 2u;
    return S == 4u && cus >= 4u && (nst + 2u) / 3u <= 32u && most(3u) < most(4u) ? 3u : S;
  }
  // the unsliced launch's busiest workgroup (launch_shape's choice at 12 waves)
  const uint64_t most0 = launch_shape(ntiles, nst, 12u, ws_bytes, 1u, (uint32_t)cus).busiest;
  if (cus < 4u) return 0u;
  if (most0 <= 24u) {
    const uint32_t S = most(3u) < most(4u) ? 3u : 4u;
    return most(S) <= most0 || nb >= 48u ? S : 0u;
  }
  const uint32_t slots =
      ring_slots(8u, 1u, launch_shape(ntiles, nst, 8u, ws_bytes, 1u, (uint32_t)cus).tiles_per_group,
                 pairs ? 2u * nst : nst);
  if (layout(8u, 1u, nb, slots, pairs ? 2u : 1u).total <= kLdsBytes) return 0u;
  if (!pairs && most0 > 250u && layout(4u, 1u, nb, 4u).total <= kLdsBytes) return 0u;
  const uint32_t four = pairs ? 112u : 122u;
  auto cost = [&](uint32_t S) { return most(S) * (S == 2u ? 100u : S == 3u ? 103u : four); };
  uint32_t best = 2u;
  for (uint32_t S : {3u, 4u})
    if (cost(S) < cost(best)) best = S;
  return best;
}

// An odd block count over an even row count runs as row pairs (PAIRED) of
// 2 nb blocks.
bool q6_shape_ok(uint32_t rows, uint32_t nb);
bool paired_ok(uint32_t rows, uint32_t nb) {
  return (nb & 1u) == 1u && rows >= 2u && (rows & 1u) == 0u && q6_shape_ok(rows / 2u, 2u * nb);
}

// even nb (4-byte aligned rows and stages); in-tile offsets (16 rows) and the
// descriptor sizes are 32-bit
bool q6_shape_ok(uint32_t rows, uint32_t nb) {
  return nb != 0 && (nb & 1u) == 0 && nb <= kMaxMetaBlocks && rows != 0 &&
         (uint64_t)nb * kQ6Bytes * 16u <= 0x7fffffffu &&
         (uint64_t)nb * 1024u <= 0x7fffffffu &&
         (uint64_t)((rows + 15u) / 16u) * (nb / 2u) <= 0xffffffffu &&
         quotients_fit((rows + 15u) / 16u, nb / 2u);
}

}  // namespace

namespace {
// An odd block count nb: row pairs, K-sliced by the rule of the even case (and
// always past 64 blocks, where the pairs' rows exceed what the unsliced
// kernel takes), else unsliced; the last row of an odd row count beside them.
bool launch_pairs(const uint8_t* w, const float* x, float* y, uint32_t rows, uint32_t nb,
                  bool may_slice, const Workspace& ws, hipStream_t s, hipError_t* err) {
  if ((nb & 1u) == 0u || rows < 2u) return false;
  const uint32_t prows = rows / 2u, pnb = 2u * nb;
  const bool last = (rows & 1u) != 0u;
  if (may_slice) {
    const uint32_t S = q6_slices((prows + 15u) / 16u, pnb, ws.bytes, true,
                                 (uint64_t)cu_count() - (last ? 1u : 0u));
    if (S >= 2u && (launch_sliced<12, 1, true>(w, x, y, prows, pnb, S, ws, s, err, last) ||
                    launch_sliced<8, 1, true>(w, x, y, prows, pnb, S, ws, s, err, last)))
      return true;
  }
  const GroupArgs ga{};
  const ArgmaxArgs aa{};
  return q6_shape_ok(prows, pnb) &&
         (launch_wd<12, 1, false, false, true>(w, x, y, prows, pnb, ws, s, err, ga, aa, last) ||
          launch_wd<10, 1, false, false, true>(w, x, y, prows, pnb, ws, s, err, ga, aa, last) ||
          launch_wd<8, 1, false, false, true>(w, x, y, prows, pnb, ws, s, err, ga, aa, last) ||
          launch_wd<4, 1, false, false, true>(w, x, y, prows, pnb, ws, s, err, ga, aa, last));
}

// ntok <= 4 NG vectors in one pass; false when the shape does not fit.
template <int W, int NG, bool P>
bool launch_tok6(const uint8_t* w, const float* x, float* y, uint32_t rows, uint32_t nb,
                 uint32_t ntok, const Workspace& ws, hipStream_t s, hipError_t* err) {
  constexpr uint32_t kLds =
      (uint32_t)W * kStageBytes + tok64_layout(kTokBlocks, NG, false, false).total;
  static_assert(kLds <= kLdsBytes, "the stage buffers and the images fit the LDS");
  constexpr uint32_t kPer = P ? 2u : 1u;  // rows a place of the partials
  const uint32_t cus = (uint32_t)cu_count();
  const uint32_t slices = (nb + (P ? 1u : 0u) + kTokBlocks - 1u) / kTokBlocks;
  // 32-bit offsets of the weights in a tile and of the activations
  if (kPer * slices > cus || (uint64_t)nb * kPer * kQ6Bytes * 16u > 0x7fffffffu ||
      (uint64_t)ntok * nb * 1024u > 0x7fffffffu)
    return false;
  if (!P && !q6_shape_ok(rows, nb)) return false;
  // the rows of one launch: all, or as many whole tiles as the scratch holds
  const size_t place_part = (size_t)kPer * slices * 4u * NG * sizeof(float);
  const uint64_t fit = ws.scratch_bytes / place_part / 16u * 16u * kPer;
  const uint32_t chunk = (uint32_t)min((uint64_t)rows, fit);
  if (chunk == 0u) return false;
  // block and tile indices divided by GS <= cus
  if ((uint64_t)(cus + (chunk + 15u) / 16u) * cus >= (1ull << 32)) return false;
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&q6k_tokens_mfma<W, NG, P>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes);
  *err = attr;
  for (uint32_t r0 = 0; r0 < rows && *err == hipSuccess; r0 += chunk) {
    const uint32_t nr = min(chunk, rows - r0);
    const uint8_t* const wr = w + (size_t)r0 * nb * kQ6Bytes;
    Q6TokArgs ta{};
    ta.slices = slices;
    ta.groups_per_slice = min(cus / (kPer * slices), ((nr + kPer - 1u) / kPer + 15u) / 16u);
    ta.m_gps = div_magic(ta.groups_per_slice);
    hipLaunchKernelGGL((q6k_tokens_mfma<W, NG, P>), dim3(ta.groups_per_slice * kPer * slices),
                       dim3(W * 64), kLds, s, wr, x, nr, nb, ntok, ws.scratch, ta);
    *err = hipGetLastError();
    if (*err != hipSuccess) break;
    launch_tok_reduce<kTypeQ6K, P>(ws.scratch, y + r0, nr, rows, slices, 4u * NG, ntok, wr, x, nb, s);
    *err = hipGetLastError();
  }
  return true;
}

// Twelve waves; 8 and 16 measured the same within 1 % up to eight vectors, 8
// took 198 against 193 us at sixteen (151936 x 5120).
template <bool P>
bool launch_tok6_any(const uint8_t* w, const float* x, float* y, uint32_t rows, uint32_t nb,
                     uint32_t ntok, const Workspace& ws, hipStream_t s, hipError_t* err) {
  if (ntok <= 4u) return launch_tok6<12, 1, P>(w, x, y, rows, nb, ntok, ws, s, err);
  if (ntok <= 8u) return launch_tok6<12, 2, P>(w, x, y, rows, nb, ntok, ws, s, err);
  if (ntok <= 12u) return launch_tok6<12, 3, P>(w, x, y, rows, nb, ntok, ws, s, err);
  return launch_tok6<12, 4, P>(w, x, y, rows, nb, ntok, ws, s, err);
}
}  // namespace

bool launch_q6k_matvec_mfma(const uint8_t* w, const float* x, float* y, uint32_t rows,
                            uint32_t cols, const Workspace& ws, hipStream_t s, hipError_t* err) {
  const uint32_t nb = cols / kBlockElems;
  static const int cfg = env_int("SI_HIP_Q6K_MFMA_CFG", 0);
  // An odd row count as well: pairs where the generic kernel (one wave per
  // row) is slower.  Its time grows with the row, 257 x 5376 6.9 us to 6.5 of
  // the pairs, 65 x 6912 6.9 / 6.7, 65 x 8448 9.2 / 7.5, 17 x 65280 59 / 15.6,
  // and with the rows from about four a SIMD, 4097 x 256 4.7 / 4.8,
  // 8193 x 1280 10.0 / 6.3, 3073 x 2816 8.7 / 7.6; below, 2049 x 2816 7.1 / 7.4,
  // 2049 x 1280 4.4 / 5.7, 129 x 2816 4.4 / 6.8.
  const bool pairs = (rows & 1u) == 0u ||
                     (rows >= 3u && (rows >= 4096u || nb >= 27u || (uint64_t)rows * nb >= 32768u));
  if ((nb & 1u) == 1u && pairs)
    return launch_pairs(w, x, y, rows, nb, cfg == 0, ws, s, err);
  if (cfg == 0 && nb > kMaxMetaBlocks) {  // (q6_shape_ok takes none of these)
    const uint32_t S = q6_slices((rows + 15u) / 16u, nb, ws.bytes);
    return S >= 2u && (launch_sliced<12, 1>(w, x, y, rows, nb, S, ws, s, err) ||
                       launch_sliced<8, 1>(w, x, y, rows, nb, S, ws, s, err));
  }
  if (!q6_shape_ok(rows, nb)) return false;
  switch (cfg) {
    case 1: return launch_wd<12, 1>(w, x, y, rows, nb, ws, s, err);
    case 2: return launch_wd<8, 2>(w, x, y, rows, nb, ws, s, err);
    case 3: return launch_wd<8, 1>(w, x, y, rows, nb, ws, s, err);
    case 4: return launch_wd<6, 2>(w, x, y, rows, nb, ws, s, err);
    default: break;
  }
  const uint32_t S = q6_slices((rows + 15u) / 16u, nb, ws.bytes);
  if (S >= 2u && (launch_sliced<12, 1>(w, x, y, rows, nb, S, ws, s, err) ||
                  launch_sliced<8, 1>(w, x, y, rows, nb, S, ws, s, err)))
    return true;
  return launch_wd<12, 1>(w, x, y, rows, nb, ws, s, err) || launch_wd<10, 1>(w, x, y, rows, nb, ws, s, err) ||
         launch_wd<8, 1>(w, x, y, rows, nb, ws, s, err) || launch_wd<4, 1>(w, x, y, rows, nb, ws, s, err);
}

bool launch_q6k_matvec_argmax_mfma(const uint8_t* w, const float* x, float* y, uint32_t rows,
                                   uint32_t cols, uint32_t rule, uint64_t* result,
                                   const Workspace& ws, hipStream_t s, hipError_t* err) {
  if (!word_aligned(w)) return false;
  const uint32_t nb = cols / kBlockElems;
  const ArgmaxArgs aa{result, rule};
  if (paired_ok(rows, nb))
    return launch_wd<12, 1, false, true, true>(w, x, y, rows / 2u, 2u * nb, ws, s, err,
                                                  GroupArgs{}, aa) ||
           launch_wd<8, 1, false, true, true>(w, x, y, rows / 2u, 2u * nb, ws, s, err,
                                                 GroupArgs{}, aa);
  if (!q6_shape_ok(rows, nb)) return false;
  return launch_wd<12, 1, false, true>(w, x, y, rows, nb, ws, s, err, GroupArgs{}, aa) ||
         launch_wd<8, 1, false, true>(w, x, y, rows, nb, ws, s, err, GroupArgs{}, aa);
}

// (even block counts past kMaxMetaBlocks run one vector at a time)
bool launch_q6k_matmul_mfma(const uint8_t* w, const float* x, float* y, uint32_t rows,
                            uint32_t cols, uint32_t batch, const Workspace& ws, hipStream_t s,
                            hipError_t* err) {
  if (batch < 2u || batch > 16u) return false;
  const uint32_t nb = cols / kBlockElems;
  // Odd row and block counts: the generic kernel, a wave a row, where it is faster.
  // Its latency is that of one row, some 0.7 us a vector for each eight blocks,
  // against the 7 to 8 us of the pass and the reduce here: five or six vectors in
  // rows of up to eight blocks and two of up to sixteen, or eleven and five over a
  // single row, whose loads meet nobody else's; and it does every weight's products one by
  // one, which many rows, or many of their sums, make the larger part.  Us, generic
  // / here: 257 x 768 M = 6 / 8 6.8 / 8.1, 8.1 / 8.0; 513 x 2304 M = 2 / 3 7.7 /
  // 8.0, 9.3 / 8.1; one row of 1792 M = 8 / 16 6.9 / 8.0, 12.0 / 10.0; 2049 x 1280
  // M = 3 / 4 7.8 / 8.1, 9.4 / 8.1; 4097 x 256 M = 2 / 3 6.2 / 6.7, 7.5 / 6.9;
  // 4097 x 1280 M = 2 9.2 / 8.5.
  const uint32_t most = rows == 1u ? (nb < 8u ? 11u : 5u) : nb < 6u ? 6u : nb < 8u ? 5u : 2u;
  if ((nb & 1u) != 0u && (rows & 1u) != 0u && nb < 16u && batch <= most &&
      (uint64_t)rows * batch <= 10300u && (uint64_t)rows * batch * nb <= 32768u)
    return false;
  // Two vectors over short rows: whole rows in one launch, no reduce behind it
  // (two_vectors, mfma_common.h).
  if (batch == 2u && two_vectors(kTypeQ6K, rows, nb) && q6_shape_ok(rows, nb) &&
      launch_wd<12, 1, false, false, false, 2>(w, x, y, rows, nb, ws, s, err))
    return true;
  return (nb & 1u) != 0u ? launch_tok6_any<true>(w, x, y, rows, nb, batch, ws, s, err)
                         : launch_tok6_any<false>(w, x, y, rows, nb, batch, ws, s, err);
}

bool mfma::launch_q6k_matvec_group(const GroupArgs& ga, uint32_t total_rows, uint32_t cols,
                             const float* x, float* y, const Workspace& ws, hipStream_t s,
                             hipError_t* err) {
  const uint32_t nb = cols / kBlockElems;
  if (!q6_shape_ok(total_rows, nb)) return false;
  return launch_wd<12, 1, true>(ga.w[0], x, y, total_rows, nb, ws, s, err, ga) ||
         launch_wd<8, 1, true>(ga.w[0], x, y, total_rows, nb, ws, s, err, ga);
}

}  // namespace sihip
