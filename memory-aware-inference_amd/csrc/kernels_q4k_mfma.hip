// Q4_K matvec on the gfx950 matrix cores (replaces si_q4_k_matvec* for one
// input vector, src/metal.rs:310-494).
//
// The dot of a 32-weight unit, sum_i q_i * x_i with q_i in 0..15, is done as
// an exact integer product on v_mfma_i32_16x16x64_i8:
//
//  * Activations.  Each 256-element block b of x is written in fixed point,
//    x_i = X_i * 2^(e_b - 30) with |X_i| <= 2^30 (e_b from the block's largest
//    |x|), and X_i = sum_d D_d * 256^d in four signed byte digits (|D| <= 128,
//    the top one <= 64).  Rounding x to X costs at most 2^-31 of the block's
//    largest activation.
//  * Weights.  A 16-byte piece of qs masked with 0x0f (or shifted by 4 first)
//    is 16 int8 weights.
//  * Units stay apart.  Lane l of the B operand is row l % 16 of a 16-row
//    tile; lane group g = l / 16 supplies the qs bytes [32g, 32g + 32) of the
//    block, i.e. units 2g (low nibbles) and 2g + 1 (high nibbles).  Rows
//    4g..4g+3 of the A operand hold the four digits of the activations that
//    meet group g's weights and are zero elsewhere, so output rows 4g + d are
//    digit d of group g's unit sums, and they land in lane group g -- the
//    lanes that hold that unit's scale and min.
//
// Per block and lane: C_e, C_o (4 digits each) from four MFMAs; T_d = sc_e *
// C_e[d] + sc_o * C_o[d] in integers; y += (d * (sum_d T_d * 256^d) - dmin *
// (m_e * X_e + m_o * X_o)) * 2^(e_b-30), X_u the exact sum of unit u's
// fixed-point activations, so both terms see the same rounded activations
// and the pair is sum_i w_i X_i 2^(e_b-30) with w_i the weight of quant.rs.
// Both sums are exact integers below 2^53 and the terms are formed in f64
// (block_dot), so their rounding shows only where every w_i of a lane's share
// cancels inside its own decode (d sc q = dmin m); a lane that sees that
// (cancels) recomputes its share of the stage on the exact per-weight path, so
// the dot stays within 2e-5 * sum|w*x| on every input.  Blocks whose
// activations are not finite or reach 2^100 take the exact per-weight f32
// path instead, so NaN/Inf propagate as in the reference.
//
// Data path.  One persistent workgroup of WAVES waves per CU.  At start it
// turns all of x into digit images in LDS (1 KB per block, plus unit sums and
// exponents) while each wave's first stage of weights is already in flight.
// Workgroup g of G owns the 16-row tiles g, g + G, ...; their (tile,
// stage) pairs, a stage being four blocks (16 rows x 576 bytes), go to the
// waves round-robin, so every wave streams its own sequence of stages.
// Weights arrive by 16-byte buffer->LDS copies in piece-major order (LDS
// byte 16 (16 q + r) is piece q of row r), so every read is a conflict-free
// 16-lane sweep; a wave's next stage is in flight while it computes.  Only
// the 16 lanes whose A rows carry digits read images, two blocks at a time
// (exec-masked; the other lanes hold zeros for the whole kernel).  A wave leaves its stage's 16 row
// partials in an LDS slot of the tile and counts them with an LDS atomic; the
// wave that completes the tile sums the partials in stage order and stores
// the rows, so results do not depend on timing.  With MATS = 2 (fused SwiGLU
// gate/up, replacing si_q4_k_fused_gate_up, metal.rs:498-587) a tile's pairs
// cover the stages of both matrices, which share the activation images, and
// the finishing wave stores silu(gate) * up.  LDS is only touched through
// inline asm and the one barrier is a bare s_barrier: the compiler neither
// counts nor orders buffer->LDS copies, and a fence would drain them.
#include "mfma_common.h"
#include "si_hip_tuned.h"

namespace sihip {
namespace {

using namespace mfma;

// Block bytes of the two formats this kernel reads (QB = quant bits): 144
// (Q4_K) and 176 (Q5_K), both multiples of 16.  A stage is 16 rows x SB
// blocks (SB = 4, or 2 for the one-vector kernel's finer form): SB * 9 (or
// 11) 16-byte pieces per row, moved by stage_copies 64-lane copies, the last
// one's lanes past the row's pieces re-reading its last piece.
__host__ __device__ constexpr uint32_t block_bytes(int qb) { return qb == 5 ? kQ5Bytes : kQ4Bytes; }
__host__ __device__ constexpr uint32_t block_pieces(int qb) { return block_bytes(qb) / 16u; }
__host__ __device__ constexpr uint32_t stage_copies(int qb, int sb = 4) {
  return (16u * (uint32_t)sb * block_pieces(qb) + 63u) / 64u;
}
__host__ __device__ constexpr uint32_t stage_bytes(int qb, int sb = 4) {
  return 1024u * stage_copies(qb, sb);
}
static_assert(stage_bytes(4) == 64u * kQ4Bytes && stage_bytes(5) == 64u * kQ5Bytes,
              "four-block stages fill their copies exactly");

// Full-line copies (LINES: Q4_K in four-block stages, nb = 4 mod 8 blocks per
// row, the matrix 128-byte aligned).  A row's four blocks of a stage are 576
// bytes, four and a half 128-byte lines, and rows of 144 nb bytes start 64
// bytes apart modulo a line, so even rows start their even stages on a line
// and odd rows 64 bytes into one, the other way round in odd stages.  A stage
// moves as the five whole lines that hold it (the half line it shares with
// the next or the previous stage included): ten copies, copy (j, c) taking
// line j of the eight rows 2 i + c, lane 8 i + ((k + (i >> 1)) & 7) of it
// piece k of its row's line, into LDS region 2 j + (c ^ parity of the
// stage).  Every copy reads whole lines, which the nontemporal policy streams
// without fetching a line twice.  In odd stages lane n of the matrix-core
// layout takes row n ^ 1, so that every lane meets a row of one alignment in
// one LDS region at every stage and keeps one table of read addresses; a
// 16-lane read of one piece of the 16 rows meets 16 different LDS bank groups
// (the rotation by i >> 1 spreads the rows that share a line slot, and the
// two alignments sit half a line apart).
constexpr uint32_t kLineCopies = 10u;
constexpr uint32_t kLineStage = 1024u * kLineCopies;  // 16 rows x 5 lines
constexpr int kNontemporal = 2;                       // buffer cache policy: NT

// LDS map (make_layout): SB-block stages, 64 bytes of unit sums per block.
__host__ __device__ constexpr Layout layout(uint32_t waves, uint32_t depth, uint32_t nb,
                                            uint32_t slots, uint32_t mats, int qb = 4, int sb = 4,
                                            bool lines = false) {
  return make_layout(lines ? kLineStage : stage_bytes(qb, sb), (uint32_t)sb, 64u, waves, depth,
                     nb, slots, mats);
}

// The lane's header and two qs pieces of the four blocks of a full-line stage
// buffer, each at its own address (a[3 b], a[3 b + 1], a[3 b + 2]) plus IMM.
template <int IMM>
__device__ __forceinline__ void lds_read_weights_at(const uint32_t (&a)[12], u32x4 (&v)[12]) {
  asm volatile(
      "ds_read_b128 %0, %12 offset:%24\n"
      "ds_read_b128 %1, %13 offset:%24\n"
      "ds_read_b128 %2, %14 offset:%24\n"
      "ds_read_b128 %3, %15 offset:%24\n"
      "ds_read_b128 %4, %16 offset:%24\n"
      "ds_read_b128 %5, %17 offset:%24\n"
      "ds_read_b128 %6, %18 offset:%24\n"
      "ds_read_b128 %7, %19 offset:%24\n"
      "ds_read_b128 %8, %20 offset:%24\n"
      "ds_read_b128 %9, %21 offset:%24\n"
      "ds_read_b128 %10, %22 offset:%24\n"
      "ds_read_b128 %11, %23 offset:%24\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]),
        "=&v"(v[6]), "=&v"(v[7]), "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11])
      : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]), "v"(a[7]),
        "v"(a[8]), "v"(a[9]), "v"(a[10]), "v"(a[11]), "i"(IMM)
      : "memory");
}

// The lane's header and two qs pieces of the four blocks of a stage buffer:
// header of block b at hb + 2304 b, qs pieces at qb + 2304 b (+256).
__device__ __forceinline__ void lds_read_weights(uint32_t hb, uint32_t qb, u32x4 (&v)[12]) {
  asm volatile(
      "ds_read_b128 %0, %12\n"
      "ds_read_b128 %1, %13\n"
      "ds_read_b128 %2, %13 offset:256\n"
      "ds_read_b128 %3, %12 offset:2304\n"
      "ds_read_b128 %4, %13 offset:2304\n"
      "ds_read_b128 %5, %13 offset:2560\n"
      "ds_read_b128 %6, %12 offset:4608\n"
      "ds_read_b128 %7, %13 offset:4608\n"
      "ds_read_b128 %8, %13 offset:4864\n"
      "ds_read_b128 %9, %12 offset:6912\n"
      "ds_read_b128 %10, %13 offset:6912\n"
      "ds_read_b128 %11, %13 offset:7168\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]),
        "=&v"(v[6]), "=&v"(v[7]), "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11])
      : "v"(hb), "v"(qb)
      : "memory");
}

// The same for the two blocks of a two-block stage.
__device__ __forceinline__ void lds_read_weights2(uint32_t hb, uint32_t qb, u32x4 (&v)[6]) {
  asm volatile(
      "ds_read_b128 %0, %6\n"
      "ds_read_b128 %1, %7\n"
      "ds_read_b128 %2, %7 offset:256\n"
      "ds_read_b128 %3, %6 offset:2304\n"
      "ds_read_b128 %4, %7 offset:2304\n"
      "ds_read_b128 %5, %7 offset:2560\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5])
      : "v"(hb), "v"(qb)
      : "memory");
}

typedef double f64x2 __attribute__((ext_vector_type(2)));
// Unit sums of the lane's two units in the four blocks (xb + 64 b), the
// four block exponents (eb) and their four side counts (one byte each, at
// eb + kCountOff).
__device__ __forceinline__ void lds_read_sums(uint32_t xb, uint32_t eb, f64x2 (&xs)[4], i32x4& ex,
                                              uint32_t& cnt) {
  static_assert(kCountOff == 512, "the offset below");
  asm volatile(
      "ds_read_b128 %0, %6\n"
      "ds_read_b128 %1, %6 offset:64\n"
      "ds_read_b128 %2, %6 offset:128\n"
      "ds_read_b128 %3, %6 offset:192\n"
      "ds_read_b128 %4, %7\n"
      "ds_read_b32 %5, %7 offset:512\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(xs[0]), "=&v"(xs[1]), "=&v"(xs[2]), "=&v"(xs[3]), "=&v"(ex), "=&v"(cnt)
      : "v"(xb), "v"(eb)
      : "memory");
}
// The same for the two blocks of a two-block stage (exponents in ex[0..1],
// the two side counts in the low 16 bits of cnt).
__device__ __forceinline__ void lds_read_sums2(uint32_t xb, uint32_t eb, f64x2 (&xs)[2], i32x4& ex,
                                               uint32_t& cnt) {
  static_assert(kCountOff == 512, "the offset below");
  u32x2 e2;
  asm volatile(
      "ds_read_b128 %0, %4\n"
      "ds_read_b128 %1, %4 offset:64\n"
      "ds_read_b64 %2, %5\n"
      "ds_read_u16 %3, %5 offset:512\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(xs[0]), "=&v"(xs[1]), "=&v"(e2), "=&v"(cnt)
      : "v"(xb), "v"(eb)
      : "memory");
  ex = i32x4{(int)e2[0], (int)e2[1], 0, 0};
}
// The 8 A images of two blocks (block b, MFMA t at addr + 1024 b + 256 t),
// read only by the lanes in `mask`; the other lanes keep their registers.
__device__ __forceinline__ void lds_read_images8(uint32_t addr, uint64_t mask, i32x4 (&a)[8]) {
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

__device__ __forceinline__ i32x4 low_nibbles(const u32x4& q) {
  return i32x4{(int)(q[0] & 0x0f0f0f0fu), (int)(q[1] & 0x0f0f0f0fu), (int)(q[2] & 0x0f0f0f0fu),
               (int)(q[3] & 0x0f0f0f0fu)};
}
__device__ __forceinline__ i32x4 high_nibbles(const u32x4& q) {
  return i32x4{(int)((q[0] >> 4) & 0x0f0f0f0fu), (int)((q[1] >> 4) & 0x0f0f0f0fu),
               (int)((q[2] >> 4) & 0x0f0f0f0fu), (int)((q[3] >> 4) & 0x0f0f0f0fu)};
}

// Exact per-weight f32 dot of 16 nibbles (low or high half of each byte of q)
// with 16 activations.
__device__ __forceinline__ float exact_dot16(const u32x4& q, int shift, float d1, float m1,
                                             const float* __restrict__ xs, float acc) {
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const uint32_t nib = (q[j >> 2] >> (8 * (j & 3) + shift)) & 0x0fu;
    acc = fmaf(k4_value_exact(d1, m1, nib), xs[j], acc);
  }
  return acc;
}

// One block of one lane's row, decoded once for every activation vector:
// B operands (low/high nibbles of its two qs pieces), the 6-bit scales and
// mins of units 2 grp, 2 grp + 1, d and dmin.
struct BlockQ4 {
  i32x4 la, ha, lb, hb;
  int sce, sco;
  float mne, mno, d, dmin;
};
__device__ __forceinline__ BlockQ4 decode_q4(const u32x4& h, const u32x4& qa, const u32x4& qb,
                                             bool hi_units, int bsh) {
  BlockQ4 w;
  const uint32_t sc03 = h[1] & 0x3f3f3f3fu;
  const uint32_t mn03 = h[2] & 0x3f3f3f3fu;
  const uint32_t sc47 = (h[3] & 0x0f0f0f0fu) | ((h[1] >> 2) & 0x30303030u);
  const uint32_t mn47 = ((h[3] >> 4) & 0x0f0f0f0fu) | ((h[2] >> 2) & 0x30303030u);
  const uint32_t scw = hi_units ? sc47 : sc03;
  const uint32_t mnw = hi_units ? mn47 : mn03;
  w.sce = (int)((scw >> bsh) & 0xffu);
  w.sco = (int)((scw >> (bsh + 8)) & 0xffu);
  w.mne = (float)((mnw >> bsh) & 0xffu);
  w.mno = (float)((mnw >> (bsh + 8)) & 0xffu);
  w.la = low_nibbles(qa);
  w.ha = high_nibbles(qa);
  w.lb = low_nibbles(qb);
  w.hb = high_nibbles(qb);
  w.d = half_bits_to_float(h[0] & 0xffffu);
  w.dmin = half_bits_to_float(h[0] >> 16);
  return w;
}

// Fast-path dot of one decoded block with the activations' images (xs: the
// exact fixed-point sums of the lane's two units), in f64 from exact integers:
// the digit sums T_d = sc_e C_e[d] + sc_o C_o[d] (|T_d| < 2^24), their total
// sum_d 256^d T_d (< 2^50) and the mins' sum; only the two products with d and
// dmin round, at 2^-53.  `redo` when the terms cancel so far that this could
// show.  (In f32 the rounding was bounded by 2^-21 of the terms; weights
// quantised from zero-mean data have d sc q and dmin m of one size, and one
// row-stage in some thousand failed its check, a wave's whole stage then
// waiting for the per-weight path.  On such weights, us: 17408 x 5120 12.2 ->
// 11.5, 1024 x 5120 7.8 -> 6.3, the 6144 + 1024 + 1024 group 11.6 -> 8.7.)
template <int QB>
__device__ __forceinline__ double block_dot(const BlockQ4& w, const i32x4& a0, const i32x4& a1,
                                            const i32x4& a2, const i32x4& a3, const f64x2& xs,
                                            int eb, bool& redo) {
  const i32x4 zero = {0, 0, 0, 0};
  i32x4 ce = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, w.la, zero, 0, 0, 0);
  i32x4 co = __builtin_amdgcn_mfma_i32_16x16x64_i8(a2, w.ha, zero, 0, 0, 0);
  ce = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, w.lb, ce, 0, 0, 0);
  co = __builtin_amdgcn_mfma_i32_16x16x64_i8(a3, w.hb, co, 0, 0, 0);
  const int t0 = __mul24(w.sce, ce[0]) + __mul24(w.sco, co[0]);
  const int t1 = __mul24(w.sce, ce[1]) + __mul24(w.sco, co[1]);
  const int t2 = __mul24(w.sce, ce[2]) + __mul24(w.sco, co[2]);
  const int t3 = __mul24(w.sce, ce[3]) + __mul24(w.sco, co[3]);
  // |X| <= 2^30, so |D_3| <= 64: 256 T_3 + T_2 fits 32 bits for both formats
  // (Q5_K: 31 63 64 64 256 + 2^24 < 2^31), 256 T_1 + T_0 for Q4_K
  // (15 63 64 128 257 < 2^31)
  const double hi = (double)(256 * t3 + t2);
  double tc;
  if constexpr (QB == 4)
    tc = fma(hi, 65536.0, (double)(256 * t1 + t0));
  else
    tc = fma(hi, 65536.0, fma((double)t1, 256.0, (double)t0));
  const double um = fma((double)w.mne, xs[0], (double)w.mno * xs[1]);
  const double dt = (double)w.d * tc;
  const double p = fma(-(double)w.dmin, um, dt);
  redo |= cancels(p, dt);
  return __builtin_amdgcn_ldexp(p, eb);
}

// Exact per-weight path of one block (activations not finite or >= 2^100).
__device__ __forceinline__ float block_exact(const u32x4& h, const u32x4& qa, const u32x4& qb,
                                             bool hi_units, int bsh, const float* __restrict__ xs) {
  const uint32_t sc03 = h[1] & 0x3f3f3f3fu;
  const uint32_t mn03 = h[2] & 0x3f3f3f3fu;
  const uint32_t sc47 = (h[3] & 0x0f0f0f0fu) | ((h[1] >> 2) & 0x30303030u);
  const uint32_t mn47 = ((h[3] >> 4) & 0x0f0f0f0fu) | ((h[2] >> 2) & 0x30303030u);
  const uint32_t scw = hi_units ? sc47 : sc03;
  const uint32_t mnw = hi_units ? mn47 : mn03;
  const uint32_t sce = (scw >> bsh) & 0xffu, sco = (scw >> (bsh + 8)) & 0xffu;
  const uint32_t mne = (mnw >> bsh) & 0xffu, mno = (mnw >> (bsh + 8)) & 0xffu;
  const float d = half_bits_to_float(h[0] & 0xffffu);
  const float dmin = half_bits_to_float(h[0] >> 16);
  const float d1e = __fmul_rn(d, (float)sce), m1e = __fmul_rn(dmin, (float)mne);
  const float d1o = __fmul_rn(d, (float)sco), m1o = __fmul_rn(dmin, (float)mno);
  float acc = exact_dot16(qa, 0, d1e, m1e, xs, 0.0f);
  acc = exact_dot16(qb, 0, d1e, m1e, xs + 16, acc);
  acc = exact_dot16(qa, 4, d1o, m1o, xs + 32, acc);
  return exact_dot16(qb, 4, d1o, m1o, xs + 48, acc);
}

// Q5_K (quant.rs:67-125): the lane's header, the two qh pieces and its two qs
// pieces of the four blocks of a stage buffer -- block b's pieces start at
// hb + 2816 b (header, qh at +256, +512) and qb + 2816 b (qs, +256).
__device__ __forceinline__ void lds_read_weights5(uint32_t hb, uint32_t qb, u32x4 (&v)[20]) {
  asm volatile(
      "ds_read_b128 %0, %20\n"
      "ds_read_b128 %1, %20 offset:256\n"
      "ds_read_b128 %2, %20 offset:512\n"
      "ds_read_b128 %3, %21\n"
      "ds_read_b128 %4, %21 offset:256\n"
      "ds_read_b128 %5, %20 offset:2816\n"
      "ds_read_b128 %6, %20 offset:3072\n"
      "ds_read_b128 %7, %20 offset:3328\n"
      "ds_read_b128 %8, %21 offset:2816\n"
      "ds_read_b128 %9, %21 offset:3072\n"
      "ds_read_b128 %10, %20 offset:5632\n"
      "ds_read_b128 %11, %20 offset:5888\n"
      "ds_read_b128 %12, %20 offset:6144\n"
      "ds_read_b128 %13, %21 offset:5632\n"
      "ds_read_b128 %14, %21 offset:5888\n"
      "ds_read_b128 %15, %20 offset:8448\n"
      "ds_read_b128 %16, %20 offset:8704\n"
      "ds_read_b128 %17, %20 offset:8960\n"
      "ds_read_b128 %18, %21 offset:8448\n"
      "ds_read_b128 %19, %21 offset:8704\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]),
        "=&v"(v[6]), "=&v"(v[7]), "=&v"(v[8]), "=&v"(v[9]), "=&v"(v[10]), "=&v"(v[11]),
        "=&v"(v[12]), "=&v"(v[13]), "=&v"(v[14]), "=&v"(v[15]), "=&v"(v[16]), "=&v"(v[17]),
        "=&v"(v[18]), "=&v"(v[19])
      : "v"(hb), "v"(qb)
      : "memory");
}

// The same for the two blocks of a two-block stage.
__device__ __forceinline__ void lds_read_weights5x2(uint32_t hb, uint32_t qb, u32x4 (&v)[10]) {
  asm volatile(
      "ds_read_b128 %0, %10\n"
      "ds_read_b128 %1, %10 offset:256\n"
      "ds_read_b128 %2, %10 offset:512\n"
      "ds_read_b128 %3, %11\n"
      "ds_read_b128 %4, %11 offset:256\n"
      "ds_read_b128 %5, %10 offset:2816\n"
      "ds_read_b128 %6, %10 offset:3072\n"
      "ds_read_b128 %7, %10 offset:3328\n"
      "ds_read_b128 %8, %11 offset:2816\n"
      "ds_read_b128 %9, %11 offset:3072\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]),
        "=&v"(v[6]), "=&v"(v[7]), "=&v"(v[8]), "=&v"(v[9])
      : "v"(hb), "v"(qb)
      : "memory");
}

// 5-bit weights of units 2 grp (low nibbles + qh bit 2 grp) and 2 grp + 1
// (high nibbles + bit 2 grp + 1) from 16 qs bytes and the matching 16 qh
// bytes.  rot_lo / rot_hi rotate that qh bit of every byte to bit 4
// (v_alignbit of a word with itself is a rotate right).
__device__ __forceinline__ void q5_operands(const u32x4& qs, const u32x4& qh, uint32_t rot_lo,
                                            uint32_t rot_hi, i32x4& lo, i32x4& hi) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const uint32_t tl = __builtin_amdgcn_alignbit(qh[k], qh[k], rot_lo);
    const uint32_t th = __builtin_amdgcn_alignbit(qh[k], qh[k], rot_hi);
    lo[k] = (int)((qs[k] & 0x0f0f0f0fu) | (tl & 0x10101010u));
    hi[k] = (int)(((qs[k] >> 4) & 0x0f0f0f0fu) | (th & 0x10101010u));
  }
}

__device__ __forceinline__ BlockQ4 decode_q5(const u32x4& h, const u32x4& qh0, const u32x4& qh1,
                                             const u32x4& qa, const u32x4& qb, bool hi_units,
                                             int bsh, uint32_t rot_lo, uint32_t rot_hi) {
  BlockQ4 w = decode_q4(h, qa, qb, hi_units, bsh);  // scales, mins, d, dmin
  q5_operands(qa, qh0, rot_lo, rot_hi, w.la, w.ha);
  q5_operands(qb, qh1, rot_lo, rot_hi, w.lb, w.hb);
  return w;
}

// Exact per-weight f32 dot of 16 weights given as bytes (0..31) with 16
// activations.
__device__ __forceinline__ float exact_dot16_bytes(const i32x4& q, float d1, float m1,
                                                   const float* __restrict__ xs, float acc) {
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const uint32_t v = ((uint32_t)q[j >> 2] >> (8 * (j & 3))) & 0xffu;
    acc = fmaf(k4_value_exact(d1, m1, v), xs[j], acc);
  }
  return acc;
}

// Exact per-weight path of one decoded Q5_K block (same element order as
// block_exact).
__device__ __forceinline__ float block_exact5(const BlockQ4& w, const u32x4& h, bool hi_units,
                                              int bsh, const float* __restrict__ xs) {
  const uint32_t sc03 = h[1] & 0x3f3f3f3fu;
  const uint32_t mn03 = h[2] & 0x3f3f3f3fu;
  const uint32_t sc47 = (h[3] & 0x0f0f0f0fu) | ((h[1] >> 2) & 0x30303030u);
  const uint32_t mn47 = ((h[3] >> 4) & 0x0f0f0f0fu) | ((h[2] >> 2) & 0x30303030u);
  const uint32_t scw = hi_units ? sc47 : sc03;
  const uint32_t mnw = hi_units ? mn47 : mn03;
  const uint32_t sce = (scw >> bsh) & 0xffu, sco = (scw >> (bsh + 8)) & 0xffu;
  const uint32_t mne = (mnw >> bsh) & 0xffu, mno = (mnw >> (bsh + 8)) & 0xffu;
  const float d = half_bits_to_float(h[0] & 0xffffu);
  const float dmin = half_bits_to_float(h[0] >> 16);
  const float d1e = __fmul_rn(d, (float)sce), m1e = __fmul_rn(dmin, (float)mne);
  const float d1o = __fmul_rn(d, (float)sco), m1o = __fmul_rn(dmin, (float)mno);
  float acc = exact_dot16_bytes(w.la, d1e, m1e, xs, 0.0f);
  acc = exact_dot16_bytes(w.lb, d1e, m1e, xs + 16, acc);
  acc = exact_dot16_bytes(w.ha, d1o, m1o, xs + 32, acc);
  return exact_dot16_bytes(w.hb, d1o, m1o, xs + 48, acc);
}

// The weights of a stage of SB blocks in registers, per format: Q4_K keeps
// (header, qs piece a, qs piece b) per block, Q5_K adds the two qh pieces.
template <int QB, int SB = 4>
struct StageRegs {
  static constexpr int kPer = QB == 5 ? 5 : 3;
  u32x4 v[SB * kPer];
  __device__ __forceinline__ void read(uint32_t hb, uint32_t qb) {
    if constexpr (QB == 5 && SB == 4)
      lds_read_weights5(hb, qb, v);
    else if constexpr (QB == 5)
      lds_read_weights5x2(hb, qb, v);
    else if constexpr (SB == 4)
      lds_read_weights(hb, qb, v);
    else
      lds_read_weights2(hb, qb, v);
  }
  // a full-line stage buffer (Q4_K, four blocks): each piece at its own address
  template <int IMM>
  __device__ __forceinline__ void read_at(const uint32_t (&a)[12]) {
    static_assert(QB == 4 && SB == 4, "full-line stages: Q4_K, four blocks");
    lds_read_weights_at<IMM>(a, v);
  }
  __device__ __forceinline__ BlockQ4 decode(int b, bool hi_units, int bsh, uint32_t rot_lo,
                                            uint32_t rot_hi) const {
    if constexpr (QB == 5)
      return decode_q5(v[5 * b], v[5 * b + 1], v[5 * b + 2], v[5 * b + 3], v[5 * b + 4],
                       hi_units, bsh, rot_lo, rot_hi);
    else
      return decode_q4(v[3 * b], v[3 * b + 1], v[3 * b + 2], hi_units, bsh);
  }
  __device__ __forceinline__ float exact(int b, bool hi_units, int bsh, uint32_t rot_lo,
                                         uint32_t rot_hi, const float* __restrict__ xs) const {
    if constexpr (QB == 5)
      return block_exact5(decode(b, hi_units, bsh, rot_lo, rot_hi), v[5 * b], hi_units, bsh, xs);
    else
      return block_exact(v[3 * b], v[3 * b + 1], v[3 * b + 2], hi_units, bsh, xs);
  }
};

// Largest |w| of the lane's two units of a decoded Q4_K (QMAX 15) or Q5_K
// (QMAX 31) block: |d| sc QMAX + |dmin| m, the larger of the two units.
template <int QMAX>
__device__ __forceinline__ float k4_bound(const BlockQ4& w) {
  const float ad = fabsf(w.d), am = fabsf(w.dmin);
  return fmaxf(fmaf(ad, (float)(w.sce * QMAX), am * w.mne),
               fmaf(ad, (float)(w.sco * QMAX), am * w.mno));
}

// One vector's partial dot of the lane's row over stage s (blocks SB s ..
// SB s + nlive - 1), whose images and metadata sit at LDS stage ls: the MFMA
// digit sums, the rounded blocks' check (an exact recompute of them for a row
// that fails it), and the exact path for blocks that need it, summed over the
// lane groups
// (every lane of a row gets the row's sum).
template <int QB, int SB, typename Sum = float>
__device__ __forceinline__ Sum stage_rowsum(const StageRegs<QB, SB>& v, uint32_t sbase,
                                              const Layout& L, uint32_t ls, uint32_t s,
                                              uint32_t nlive, uint32_t grp, uint32_t n,
                                              i32x4 (&A)[8], bool hi_units, int bsh,
                                              uint32_t rot_lo, uint32_t rot_hi,
                                              const float* __restrict__ x) {
  static_assert(SB == 4 || SB == 2, "four- or two-block stages");
  f64x2 xs[SB];
  i32x4 ex;
  uint32_t cnt;
  if constexpr (SB == 4)
    lds_read_sums(sbase + L.xsum + 256u * ls + 16u * grp, sbase + L.expo + 16u * ls, xs, ex, cnt);
  else
    lds_read_sums2(sbase + L.xsum + 128u * ls + 16u * grp, sbase + L.expo + 8u * ls, xs, ex, cnt);
  float part[SB];
  double acc = 0.0;
  bool redo = false;  // the lane's share takes the per-weight path
  bool bad_any = false;
#pragma unroll
  for (int h = 0; h < SB / 2; ++h) {
    lds_read_images8(sbase + L.img + 1024u * SB * ls + 2048u * h + 16u * n, kActiveLanes, A);
#pragma unroll
    for (int b2 = 0; b2 < 2; ++b2) {
      const int b = 2 * h + b2;
      const int eb = __builtin_amdgcn_readfirstlane(ex[b]);
      const bool use = (uint32_t)b < nlive, fast = use && eb != kBadBlock;
      bad_any |= use && eb == kBadBlock;
      bool r = false;
      const double c =
          block_dot<QB>(v.decode(b, hi_units, bsh, rot_lo, rot_hi), A[4 * b2], A[4 * b2 + 1],
                        A[4 * b2 + 2], A[4 * b2 + 3], xs[b], eb, r);
      redo |= fast && r;
      acc += fast ? c : 0.0;
      part[b] = fast ? (float)c : 0.0f;
    }
  }
  redo |= !(fabs(acc) < __builtin_huge_val());
  // the rounded blocks' check; blocks on the exact path, and every live block
  // of a lane that fails a check, take the per-weight path
  const uint32_t counts = live_counts(__builtin_amdgcn_readfirstlane(cnt), nlive);
  const uint32_t rmask = rounded_mask(counts);
  if (rmask != 0u) {
    const uint32_t list = sbase + L.expo + L.side_off + (uint32_t)SB * kSideCountBytes * ls;
    const float err = rounded_bound<SB>(list, rmask, grp, ex, [&](auto b) {
      return k4_bound<QB == 5 ? 31 : 15>(
          v.decode(decltype(b)::value, hi_units, bsh, rot_lo, rot_hi));
    });
    float apart = 0.0f;
#pragma unroll
    for (int b = 0; b < SB; ++b) apart += fabsf(part[b]);
    redo |= !rounded_ok(err, apart);
  }
  Sum sum = (Sum)acc;
  if (bad_any || __builtin_amdgcn_ballot_w64(redo) != 0u) {
    if (bad_any || redo) {
      sum = Sum(0);
#pragma unroll
      for (int b = 0; b < SB; ++b) {
        if ((uint32_t)b < nlive &&
            (redo || __builtin_amdgcn_readfirstlane(ex[b]) == kBadBlock))
          part[b] = v.exact(b, hi_units, bsh, rot_lo, rot_hi,
                            x + 256u * ((uint32_t)SB * s + b) + 64u * grp);
        sum += part[b];
      }
    }
  }
  return sum_lane_groups(sum);
}

// GROUPED: the rows are those of the group's matrices with one K, one after the
// other (every matrix but the last a whole number of 16-row tiles), and tile
// t's weights are those of the matrix whose tiles reach past t.
//
// SLICED (one matrix, one vector): a K-sliced launch (SliceArgs,
// mfma_common.h); the LDS holds the images and metadata of the workgroup's
// slice only, stage s of the matrix at local stage s - r_lo.
// SB (one matrix, one vector): blocks per stage, 4, or 2 for shapes whose
// workgroups have few pairs per wave (finer pairs, a shorter last one).
// LINES (Q4_K, one vector, four-block stages of whole rows, nb a multiple of
// 4, every matrix 128-byte aligned): full-line copies (kLineCopies above).
// VECS = 2 (one matrix, whole rows): two vectors, one after the other in x, in
// one pass over the weights: the LDS holds both vectors' images, the second
// vector's from a whole stage on (hand_off_two).
template <int WAVES, int DEPTH, int MATS, int QB, bool GROUPED, bool SLICED = false,
          int SB = 4, bool LINES = false, int VECS = 1>
__global__ __launch_bounds__(WAVES * 64) void q4k_matvec_mfma(const uint8_t* __restrict__ w,
                                                              const uint8_t* __restrict__ w2,
                                                              const float* __restrict__ x,
                                                              float* __restrict__ y, uint32_t rows,
                                                              uint32_t nb, void* __restrict__ wsp,
                                                              SchedArgs sa, GroupArgs ga,
                                                              SliceArgs sla) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  static_assert(QB == 4 || QB == 5, "Q4_K or Q5_K");
  static_assert(!SLICED || (MATS == 1 && !GROUPED), "slices of one matrix");
  static_assert(SB == 4 || (SB == 2 && MATS == 1), "two-block stages: one matrix");
  static_assert(!LINES || (QB == 4 && SB == 4 && !SLICED && DEPTH <= 2),
                "full-line stages: Q4_K, four blocks, whole rows");
  static_assert(VECS == 1 || (VECS == 2 && MATS == 1 && !GROUPED && !SLICED && !LINES),
                "two vectors with whole rows of one matrix");
  if constexpr (GROUPED) load_group_args_early(ga);
  const uint32_t slots = sa.packed & 0xffu;
  // copy instructions per stage
  constexpr uint32_t kPieces = LINES ? kLineCopies : stage_copies(QB, SB);
  constexpr uint32_t kRowPieces = SB * block_pieces(QB);  // 16-byte pieces per row and stage
  constexpr uint32_t kStage = LINES ? kLineStage : stage_bytes(QB, SB);
  const uint32_t ntiles = (rows + 15u) / 16u;
  const uint32_t nstages = (nb + SB - 1u) / SB;
  const uint32_t tstages = MATS * nstages;  // pairs (and partials) per tile
  // the schedule: whole and split tiles (sc), or K slices (ss)
  Sched sc{};
  SliceSched ss{};
  if constexpr (SLICED)
    ss = make_slice_sched(ntiles, sla, sa);
  else
    sc = make_sched(ntiles, tstages, WAVES, sa);
  // the stages whose images the LDS holds: from st0, nbl blocks
  const uint32_t st0 = SLICED ? ss.r_lo : 0u;
  const uint32_t nbl = SLICED ? min(SB * ss.ns, nb - SB * st0) : VECS == 2 ? SB * nstages + nb : nb;
  const Layout L = layout(WAVES, DEPTH,
                          SLICED ? SB * ss.pstride : VECS == 2 ? 2u * SB * nstages : nb, slots,
                          VECS == 2 ? 2u : MATS, QB, SB, LINES);
  const SplitWs ws = split_ws(wsp);
  const uint32_t wave = uniform(threadIdx.x >> 6);
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t grp = lane >> 4, n = lane & 15u;
  const uint32_t row_bytes = nb * block_bytes(QB);
  const uint32_t sbase = (uint32_t)(uintptr_t)smem;
  uint8_t* const wstage = smem + wave * DEPTH * kStage;

  // 1. x into the image area, natural order (block b at img + 1024 b)
  if constexpr (VECS == 2)
    copy_two_x<WAVES>(smem, L.img, x, nb, SB * nstages, wave, lane);
  else
    copy_x<WAVES>(smem, L.img, x + (size_t)SB * st0 * kBlockElems, nbl, wave, lane);

  // 2. this wave's pairs k = wave, wave + WAVES, ... of the workgroup's pairs
  //    (pair_at: a tile and its partial r, r being stage r % nstages of
  //    matrix r / nstages), and the copies of its first DEPTH, pair j of the
  //    wave into buffer j % DEPTH.  Piece
  //    c = 64 i + lane of a stage is piece c / 16 of row c % 16's 576 bytes.
  auto pair_of = [&](uint32_t k) -> Pair {
    if constexpr (SLICED)
      return pair_at(ss, k);
    else
      return pair_at(sc, k, tstages);
  };
  const uint32_t npairs = SLICED ? ss.npairs : sc.npairs;
  const uint32_t voff = n * row_bytes + 16u * grp;
  // LINES: lcopy0 / lcopy1, the copy lane's byte offset in its tile for rows
  // 2 i and 2 i + 1 before 576 s - 64 m (the row's stage starts 64 m bytes
  // into its first line, m = c ^ parity of the stage).
  uint32_t lcopy0 = 0u, lcopy1 = 0u;
  if constexpr (LINES) {
    const uint32_t li = lane >> 3, k = ((lane & 7u) - (li >> 1)) & 7u;
    lcopy0 = 2u * li * row_bytes + 16u * k;
    lcopy1 = lcopy0 + row_bytes;
  }
  const uint32_t my_pairs = wave < npairs ? (npairs - 1u - wave) / WAVES + 1u : 0u;
  auto issue = [&](uint32_t j, const Pair& pr) {
    const uint32_t mat = MATS > 1 && pr.r >= nstages ? 1u : 0u, st = pr.r - mat * nstages;
    uint32_t row0 = pr.tile * 16u, mrows = rows;
    const uint8_t* wm = mat ? w2 : w;
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
    const uint32_t nrows = min(16u, mrows - row0);
    if constexpr (LINES) {
      // the tile's rows from its first byte (128-byte aligned); rows past
      // the tile's last read zero
      const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint8_t*>(wm + (size_t)row0 * row_bytes), 0, (int)(nrows * row_bytes),
          kBufferWord3);
      uint8_t* dst = wstage + (j % DEPTH) * kStage;
      const uint32_t odd = st & 1u;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        // (the stage's terms are uniform: one add per copy class)
        const uint32_t vo =
            (c ? lcopy1 : lcopy0) + (4u * kQ4Bytes * st - 64u * ((uint32_t)c ^ odd));
        uint8_t* const region = dst + 1024u * ((uint32_t)c ^ odd);
        // (the line's offset goes into the lane offset: an instruction offset
        // would move the LDS destination by the same amount)
#pragma unroll
        for (int jl = 0; jl < 5; ++jl)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void*)(region + 2048 * jl), 16,
                                                    vo + 128u * jl, 0, 0, kNontemporal);
      }
      return;
    }
    const uint8_t* sb = wm + (size_t)row0 * row_bytes + SB * block_bytes(QB) * st;
    // the descriptor ends at the tile's last row: pieces past it read zero
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(sb), 0, (int)(nrows * row_bytes - SB * block_bytes(QB) * st),
        kBufferWord3);
    uint8_t* dst = wstage + (j % DEPTH) * kStage;
#pragma unroll
    for (int i = 0; i < (int)kPieces; ++i) {
      // (a stage of SB = 2 ends inside its last copy: those lanes re-read the
      // row's last piece, which adds no traffic)
      const uint32_t off = 4u * (uint32_t)i + 3u < kRowPieces
                               ? voff + 64u * i
                               : n * row_bytes + 16u * min(4u * i + grp, kRowPieces - 1u);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_void*)(dst + 1024 * i), 16, off, 0, 0, 0);
    }
  };
  // (with one stage in flight, the pair of the next stage, worked out when
  // its copy is issued, is kept for its turn)
  Pair pr_next = pair_of(wave);
  auto issue_first = [&]() {
#pragma unroll
    for (int j = 0; j < DEPTH; ++j)
      if ((uint32_t)j < my_pairs) issue(j, j == 0 ? pr_next : pair_of(wave + j * WAVES));
  };

  // 3. ring slots and the builders' count, set before any wave goes on (the
  //    waves start together, so this barrier costs little).  The first round
  //    of waves (one per SIMD, and every builder), whose copies the empty
  //    memory queue takes at once, issue their first copies before it; the
  //    later waves, whose copies the queue holds back, after it, so that none
  //    of them keeps the others at the barrier.  A builder that issued late
  //    would hold every wave's first arithmetic back with its images.  The
  //    waves that copied x (the builders) turn it
  //    into digit images, unit sums and exponents once it has landed (the
  //    copies complete in issue order).  A wave reads images only once every
  //    builder has counted itself done (wait_images): no barrier makes a
  //    wave whose stage has landed wait for the waves whose copies the
  //    memory queue still holds back.
  const bool first_round = wave < max(4u, min((uint32_t)WAVES, (nbl + 3u) / 4u));
  if (first_round) issue_first();
  init_slots<WAVES>(sbase, L, slots);
  lds_wait();
  __builtin_amdgcn_s_barrier();
  const uint32_t builders = min((uint32_t)WAVES, (nbl + 3u) / 4u);
  if (!first_round) issue_first();
  if (wave < builders) {
    const uint32_t early = min((uint32_t)DEPTH, my_pairs);
    if (early >= 3u)
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(3 * kPieces));
    else if (early == 2u)
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 * kPieces));
    else if (early == 1u)
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(kPieces));
    else
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    // chunk c = 4 p + t: units 2p, 2p + 1 of lane group p, MFMA t
    build_images<WAVES>(sbase, L, nbl, wave, grp, n,
                        [](uint32_t c) { return 256u * (c & 3u) + 64u * (c >> 2); });
    lds_wait();
    if (lane == 0u) (void)lds_add_rtn(sbase + L.ready, 1u);
  }

  // 4. the wave's pairs
  const bool hi_units = grp >= 2u;       // units 4..7 use the packed upper scales
  const int bsh = 16 * (int)(grp & 1u);  // byte of unit 2 grp within its scale word
  const uint32_t hb0 = sbase + wave * DEPTH * kStage + 16u * n;
  // qs pieces of lane group grp: Q4_K pieces 1 + 2 grp, Q5_K 3 + 2 grp
  const uint32_t qb0 = hb0 + (QB == 5 ? 768u : 256u) + 512u * grp;
  // Q5_K: rotations that bring qh bits 2 grp / 2 grp + 1 of each byte to bit 4
  const uint32_t rot_lo = (28u + 2u * grp) & 31u, rot_hi = (29u + 2u * grp) & 31u;
  // the images of two blocks at a time: the lanes that do not read them keep
  // zeros, so the registers stay live through the loop (32 rather than 64)
  i32x4 A[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) A[t] = i32x4{0, 0, 0, 0};
  // LINES: the lane's 12 pieces of a stage in buffer 0 (the header, qs
  // pieces 1 + 2 grp and 2 + 2 grp of each block), the same at every stage:
  // the lane's row (n, or n ^ 1 in odd stages) starts its stage 64 m bytes
  // into its first line, m = n & 1, so piece q sits at position q + 4 m of
  // the row's five lines, line j = pos / 8 in LDS region 2 j + (n & 1), slot
  // 8 (n >> 1) + ((pos + (n >> 2)) & 7).
  uint32_t lread[12];
  if constexpr (LINES) {
    const uint32_t ri = n >> 1, rc = n & 1u, phi = n >> 2;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
#pragma unroll
      for (int pc = 0; pc < 3; ++pc) {
        const uint32_t q = 9u * b + (pc == 0 ? 0u : (uint32_t)pc + 2u * grp);
        const uint32_t pos = q + 4u * rc;
        lread[3 * b + pc] = sbase + wave * DEPTH * kStage + 1024u * (2u * (pos >> 3) + rc) +
                            128u * ri + 16u * (((pos & 7u) + phi) & 7u);
      }
    }
  }
  uint32_t fail = 0u;  // a bounded wait that gave up (kDevErr*)
  bool images = false;  // every builder's images seen done
  // The fused gate/up (two matrices) with one stage in flight and three or
  // more pairs per wave: a wave claims the workgroup's pairs after its first
  // (pair `wave`) from a counter (L.ready + 4) as it issues their copies, so
  // the waves whose first copies went out late take fewer pairs instead of
  // finishing after the rest (17408 x 5120, 42 pairs per workgroup: 20.9 ->
  // 19.3 us).  With fewer pairs per wave an early wave would take a third
  // pair and end a whole pair later (the 17408 x 5120 matvec, 21 pairs per
  // workgroup: 11.2 -> 12.7 us), and in one-matrix kernels the claim's code
  // alone cost the headline 0.13 us, so there wave w takes pairs w,
  // w + WAVES, ...  Which wave computes a pair changes no sum: a tile's
  // finishing wave adds its partials in order.
  constexpr bool kClaimable = DEPTH == 1 && MATS == 2;
  const bool claims = kClaimable && npairs >= 3u * (uint32_t)WAVES;
  uint32_t knext = wave;  // claims: the index of pr_next
  for (uint32_t j = 0; claims ? knext < npairs : j < my_pairs; ++j) {
    const Pair pr = DEPTH == 1 ? pr_next : pair_of(wave + j * WAVES);
    const uint32_t s = MATS > 1 && pr.r >= nstages ? pr.r - nstages : pr.r;  // stage
    const uint32_t later = min((uint32_t)DEPTH - 1u, my_pairs - 1u - j);
    if (DEPTH >= 3 && later >= 2u)
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 * kPieces));
    else if (DEPTH >= 2 && later >= 1u)
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(kPieces));
    else
      __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    const uint32_t buf = (j % DEPTH) * kStage;
    StageRegs<QB, SB> v;
    if constexpr (LINES) {
      if (DEPTH > 1 && (j & 1u) != 0u)
        v.template read_at<(int)kLineStage>(lread);
      else
        v.template read_at<0>(lread);
    } else {
      v.read(hb0 + buf, qb0 + buf);
    }
    // The buffer just read is free again.  Its next copy goes out after the
    // stage's arithmetic: while the memory queue is full, issuing a copy holds
    // the wave, and the stage in registers would wait for it.
    auto issue_next = [&]() {
      if (kClaimable && claims) {
        knext = lds_claim(sbase + L.ready + 4u);
        if (knext < npairs) {
          const Pair pn = pair_of(knext);
          issue(0u, pn);
          pr_next = pn;
        }
      } else if (j + DEPTH < my_pairs) {
        const Pair pn = pair_of(wave + (j + DEPTH) * WAVES);
        issue(j + DEPTH, pn);
        if (DEPTH == 1) pr_next = pn;
      }
    };
    const uint32_t nlive = min((uint32_t)SB, nb - SB * s);
    if (!images) {
      wait_images(sbase, L, builders, fail);
      images = true;
    }
    if constexpr (VECS == 2) {
      const double s0 = stage_rowsum<QB, SB, double>(v, sbase, L, s, s, nlive, grp, n, A, hi_units,
                                                     bsh, rot_lo, rot_hi, x);
      const double s1 = stage_rowsum<QB, SB, double>(v, sbase, L, s + nstages, s, nlive, grp, n, A,
                                                     hi_units, bsh, rot_lo, rot_hi,
                                                     x + (size_t)nb * kBlockElems);
      issue_next();
      hand_off_two(sbase, L, slots, sc, pr, nstages, s0, s1, lane, rows, y, fail);
      continue;
    }
    float rowsum = stage_rowsum(v, sbase, L, s - st0, s, nlive, grp, n, A, hi_units, bsh,
                                rot_lo, rot_hi, x);
    // LINES: in odd stages lane n summed row n ^ 1; swap adjacent lanes back
    if (LINES && (s & 1u) != 0u) rowsum = dpp<kQuadSwap>(rowsum);
    issue_next();

    // hand the 16 row partials to the tile's slot; the last stage finishes it
    if constexpr (SLICED)
      hand_off_slice(sbase, L, ss, pr, rowsum, lane, rows, y, ws, fail);
    else
      hand_off<MATS>(sbase, L, slots, sc, pr, nstages, rowsum, lane, rows, y, ws, fail);
  }
  if (fail != 0u) report_device_error(wsp, fail);
}

template <int W, int D, int M, int QB = 4, bool G = false, int SB = 4, bool LN = false, int V = 1>
bool launch_wd(const uint8_t* w, const uint8_t* w2, const float* x, float* y, uint32_t rows,
               uint32_t nb, const Workspace& ws, hipStream_t s, hipError_t* err,
               const GroupArgs& ga = GroupArgs{}) {
  const uint32_t ntiles = (rows + 15u) / 16u;
  const uint32_t tstages = (nb + SB - 1u) / SB * M;
  // (two vectors: whole tiles, as without a workspace)
  const LaunchShape ls = launch_shape(ntiles, tstages, W, V == 2 ? 0u : ws.bytes, M);
  const uint32_t grid = ls.groups;
  const uint32_t slots = ring_slots(W, D, ls.tiles_per_group, V == 2 ? 4u * tstages : tstages);
  const uint32_t lds =
      layout(W, D, V == 2 ? 2u * SB * tstages : nb, slots, V == 2 ? 2 : M, QB, SB, LN).total;
  SchedArgs sa;
  if (lds > kLdsBytes || !make_sched_args(ntiles, tstages, slots, ls, &sa)) return false;
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&q4k_matvec_mfma<W, D, M, QB, G, false, SB, LN, V>),
      hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes);
  if (attr != hipSuccess) {
    *err = attr;
    return true;
  }
  hipLaunchKernelGGL((q4k_matvec_mfma<W, D, M, QB, G, false, SB, LN, V>), dim3(grid),
                     dim3(W * 64), lds, s, w, w2, x, y, rows, nb, ws.ptr, sa, ga, SliceArgs{});
  *err = hipGetLastError();
  return true;
}

// Whether a Q4_K launch of whole rows can take full-line copies: four-block
// stages that fill every row, rows of 144 nb bytes with nb = 4 mod 8 (64
// bytes past a whole number of lines) and 128-byte aligned matrices, so that
// every tile starts on a line.
bool lines_fit(uint32_t nb, const uint8_t* w, const uint8_t* w2 = nullptr) {
  static const int env = env_int("SI_HIP_Q4K_LINES", 1);
  auto aligned = [](const uint8_t* p) { return ((uintptr_t)p & 127u) == 0u; };
  return env != 0 && nb % 8u == 4u && aligned(w) && (w2 == nullptr || aligned(w2));
}

// A K-sliced launch of one vector in S slices (false when the shape or the
// LDS does not fit).  The slice's blocks, not the row's, bound the LDS
// metadata, so rows longer than the unsliced kernels take run here.
template <int W, int D, int QB, int SB = 4>
bool launch_sliced(const uint8_t* w, const float* x, float* y, uint32_t rows, uint32_t nb,
                   uint32_t S, const Workspace& ws, hipStream_t s, hipError_t* err) {
  const uint32_t ntiles = (rows + 15u) / 16u;
  const uint32_t nstages = (nb + SB - 1u) / SB;
  if (rows == 0u || nb == 0u || (uint64_t)nb * block_bytes(QB) * 16u > 0x7fffffffu) return false;
  SliceShape sh;
  if (!slice_shape(ntiles, nstages, S, (uint32_t)cu_count(), ws.bytes, &sh)) return false;
  if (SB * sh.ns_max > kMaxMetaBlocks) return false;
  const uint32_t slots = ring_slots(W, D, sh.tiles_per_group, sh.ns_max);
  const uint32_t lds = layout(W, D, SB * sh.ns_max, slots, 1u, QB, SB).total;
  if (lds > kLdsBytes || slots > 0xffu || sh.groups > 0xffffu) return false;
  SchedArgs sa{};
  sa.packed = (sh.groups << 16) | slots;
  sa.m_slots = div_magic(slots);
  static const hipError_t attr = hipFuncSetAttribute(
      reinterpret_cast<const void*>(&q4k_matvec_mfma<W, D, 1, QB, false, true, SB>),
      hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLdsBytes);
  if (attr != hipSuccess) {
    *err = attr;
    return true;
  }
  hipLaunchKernelGGL((q4k_matvec_mfma<W, D, 1, QB, false, true, SB>), dim3(sh.groups),
                     dim3(W * 64), lds, s, w, nullptr, x, y, rows, nb, ws.ptr, sa, GroupArgs{},
                     sh.args);
  *err = hipGetLastError();
  return true;
}

// Slices for a one-vector Q4_K / Q5_K launch, or 0.  The same rule as the
// Q6_K kernel's (q6_slices), measured on this kernel (MI355X, us, weights
// quantised from zero-mean ones, 600 MB of them in turn):
//   type  rows x cols    unsliced  S = 2   S = 4   S = 8
//   Q4_K  5120 x 17408     20.0     18.3    16.7    22.0   (unsliced: 8 waves)
//   Q4_K  2048 x 16384     13.4     10.5     9.5    12.4
//   Q4_K  640 x 17408      11.2     10.5     7.7     8.4
//   Q4_K  8192 x 28672              38.6    35.5    41.3
//   Q4_K  2560 x 34816     66.0     24.7    18.8    18.4   (unsliced: generic kernel)
//   Q4_K  2560 x 9728      10.1              9.0           (two-block stages 8.9)
//   Q4_K  17408 x 5120     12.3             23.6
//   Q4_K  5120 x 5120       7.8             10.4
//   Q4_K  8192 x 8192      11.9     13.0    14.0
//   Q4_K  12288 x 8192     15.9             19.1
//   Q4_K  4096 x 8192       9.1             10.7
//   Q4_K  4096 x 12288     12.5     11.0    10.9           (unsliced: 8 waves)
//   Q5_K  5120 x 17408     21.5     24.0    22.0    27.8   (unsliced: two-block)
//   Q5_K  5120 x 5120       9.7             11.0
// So: rows of fewer than 8 stages (K < 8192) stay whole; four slices when
// the unsliced launch's busiest workgroup has at most two rounds of pairs
// (24) and slicing takes some of them (a tie keeps the whole rows) or the
// rows are long (64 blocks or more); with more pairs, only rows whose
// images leave room for fewer than eight waves (or exceed the LDS
// metadata), in four slices, else two, when that adds no pairs.  Rows
// longer than the unsliced kernels take must slice.
// The (tile, stage) pairs of an unsliced launch's busiest workgroup.
uint64_t busiest_pairs(uint32_t ntiles, uint32_t tparts, uint32_t waves, size_t ws_bytes) {
  return launch_shape(ntiles, tparts, waves, ws_bytes, 1u).busiest;
}

// Whether an unsliced one-vector launch of W waves and SB-block stages fits
// the LDS.
bool unsliced_fits(uint32_t ntiles, uint32_t nb, uint32_t waves, int qb, int sb,
                   size_t ws_bytes) {
  const uint32_t tparts = (nb + sb - 1u) / sb;
  const LaunchShape ls = launch_shape(ntiles, tparts, waves, ws_bytes, 1u);
  const uint32_t slots = ring_slots(waves, 1u, ls.tiles_per_group, tparts);
  return layout(waves, 1u, nb, slots, 1u, qb, sb).total <= kLdsBytes;
}

struct SliceChoice {
  uint32_t slices = 0;   // 0: unsliced
  uint64_t most0 = 0;    // busiest unsliced workgroup's pairs (0: not weighed)
  uint64_t most_s = 0;   // busiest sliced workgroup's pairs at `slices`
  bool forced = false;   // SI_HIP_Q4K_SLICES fixed `slices`
};

SliceChoice q4_slices(uint32_t ntiles, uint32_t nb, size_t ws_bytes, int qb) {
  SliceChoice c;
  static const int env = env_int("SI_HIP_Q4K_SLICES", -1);
  if (env >= 0) {
    c.slices = (uint32_t)env;
    c.forced = true;
    return c;
  }
  const uint32_t nst = (nb + 3u) / 4u;
  if (nst < 8u) return c;
  const uint64_t cus = (uint64_t)cu_count();
  auto most = [&](uint32_t S) {  // the busiest sliced workgroup's pairs
    const uint64_t gs = std::min<uint64_t>(ntiles, cus / S);
    return (ntiles + gs - 1u) / gs * ((nst + S - 1u) / S);
  };
  if (nb > kMaxMetaBlocks) {
    // rows longer than the unsliced kernels take must slice: the fewest
    // slices (from four) whose images leave the stage buffers of 12 waves
    // (Q4_K, 32 blocks) or 8 (Q5_K, 64 blocks) room in the LDS
    const uint32_t cap = qb == 5 ? 16u : 8u;  // stages per slice
    uint32_t S = 4u;
    while (S < 64u && S < cus && (nst + S - 1u) / S > cap) S *= 2u;
    c.slices = S;
    return c;
  }
  c.most0 = busiest_pairs(ntiles, nst, qb == 5 ? 8u : 12u, ws_bytes);
  auto pick = [&](uint32_t S) {
    c.slices = S;
    c.most_s = most(S);
    return c;
  };
  if (c.most0 <= 24u) return most(4u) < c.most0 || nb >= 64u ? pick(4u) : c;
  if (layout(8u, 1u, nb, 2u, 1u, qb).total <= kLdsBytes) return c;
  for (uint32_t S : {4u, 2u})
    if (most(S) <= c.most0) return pick(S);
  return c;
}

// Whether one Q4_K / Q5_K vector runs as two-block stages (12 waves,
// unsliced) rather than the slices of `sc` or four-block stages.  A stage of
// two blocks halves each pair, so more waves share a short launch; it costs
// more per block (twice the pairs, hand-offs and waits).  Measured as above
// (us; the four-block kernel unsliced at 12 waves, or at 8 where 12 do not
// fit):
//   type  rows x cols    4-block  sliced  2-block
//   Q4_K  4096 x 4096       6.1      -       5.8
//   Q4_K  8192 x 5120       8.3      -       8.3
//   Q4_K  5120 x 5120       7.9      -       7.8
//   Q4_K  1024 x 5120       6.5      -       6.0
//   Q4_K  4096 x 8192       9.1    10.7      9.0
//   Q4_K  8192 x 6144       9.2      -       9.7   (12 pairs per workgroup)
//   Q4_K  8192 x 8192      11.9    14.0     12.3   (16)
//   Q4_K  17408 x 5120     12.3      -      14.8   (22)
//   Q4_K  4096 x 14336     14.1    13.0     13.7   (12 waves do not fit)
//   Q4_K  2048 x 11008       -      8.1     10.0
//   Q4_K  1024 x 17408     11.9     8.1     11.6
//   Q5_K  5120 x 5120       9.7      -       8.4
//   Q5_K  8192 x 8192      15.1    15.9     14.2
//   Q5_K  17408 x 5120     17.2      -      16.7
//   Q5_K  5120 x 17408       -     22.0     21.5
//   Q5_K  2560 x 17408       -     14.5     15.3
//   Q5_K  640 x 17408        -      8.1     11.2
//   Q5_K  1024 x 8192        -      7.4      8.7
// So Q4_K takes two-block stages when the four-block launch leaves waves idle
// (fewer pairs per workgroup than waves) and the two-block one needs at most two
// rounds, or (three rounds) in rows of more than 40 blocks, which leave 12 waves
// of four-block stages room for a few ring slots only, or none (a group of 3200 +
// 512 + 512 x 10496 13.7 us, 12.1 in two-block stages); Q5_K, whose four-block
// stages leave registers for only 8 waves, whenever 12 waves fit.  Slices stay
// where every unsliced workgroup would build the whole row's activation images for
// a small share of the work: at most a quarter as many tiles as CUs, rows of 64
// blocks or more over fewer tiles than CUs, and rows past 32 blocks whose busiest
// workgroup the slices shorten.
bool two_block_stages(uint32_t ntiles, uint32_t nb, size_t ws_bytes, int qb,
                      const SliceChoice& sc) {
  constexpr uint32_t kWaves = 12u;
  if (sc.forced || !unsliced_fits(ntiles, nb, kWaves, qb, 2, ws_bytes)) return false;
  const uint32_t cus = (uint32_t)cu_count();
  if (sc.slices >= 2u && (ntiles <= cus / 4u || (nb >= 64u && ntiles < cus) ||
                          (nb > 32u && sc.most_s < sc.most0)))
    return false;
  if (qb == 5) return true;
  if (nb > 56u) return false;
  const uint64_t rounds2 = (busiest_pairs(ntiles, (nb + 1u) / 2u, kWaves, ws_bytes) + kWaves - 1u) /
                           kWaves;
  if (nb > 40u) return rounds2 <= 3u;
  return rounds2 <= 2u && busiest_pairs(ntiles, (nb + 3u) / 4u, kWaves, ws_bytes) < kWaves;
}

// Whether the unsliced kernel of SB-block stages takes the shape (the
// offsets, pair counts and quotients its schedule forms).
bool shape_ok(uint32_t rows, uint32_t cols, uint32_t mats, int qb, uint32_t sb = 4u) {
  const uint32_t nb = cols / kBlockElems;
  const uint64_t pairs = (uint64_t)((rows + 15u) / 16u) * ((nb + sb - 1u) / sb) * mats;
  return rows != 0 && nb != 0 && nb <= kMaxMetaBlocks &&
         (uint64_t)nb * block_bytes(qb) * 16u <= 0x7fffffffu &&
         (uint64_t)nb * 1024u <= 0x7fffffffu && pairs <= 0xffffffffu &&
         quotients_fit((rows + 15u) / 16u, (nb + sb - 1u) / sb * mats);
}

// Whether a sliced launch takes two-block stages: when the busiest sliced
// workgroup of four-block stages has fewer pairs than 12 waves, so that
// waves would idle.  Measured as above (us, S = 4, four- / two-block): Q4_K
// 1024 x 17408 9.0 / 8.0, 640 x 17408 8.6 / 7.7, 2048 x 16384 9.4 / 9.5,
// 1000 x 12800 7.9 / 7.7, 2048 x 11008 8.6 / 8.1; Q5_K 1024 x 17408 9.9 / 8.5,
// 2048 x 16384 10.4 / 10.0; with more pairs four-block stages win: Q4_K
// 2560 x 17408 10.9 / 12.0, 5120 x 17408 16.9 / 20.7.
// SI_HIP_Q4K_SLICE_SB (2 or 4) fixes the choice.
bool sliced_two_block(uint32_t ntiles, uint32_t nb, uint32_t S, size_t ws_bytes) {
  static const int env = env_int("SI_HIP_Q4K_SLICE_SB", 0);
  if (env == 2 || env == 4) return env == 2;
  SliceShape sh;
  if (!slice_shape(ntiles, (nb + 3u) / 4u, S, (uint32_t)cu_count(), ws_bytes, &sh)) return false;
  return (uint64_t)sh.tiles_per_group * sh.ns_max < 12u;
}

// Two-block stages or the sliced launch, when two_block_stages or q4_slices
// asks for one.
template <int QB>
bool try_sliced(const uint8_t* w, const float* x, float* y, uint32_t rows, uint32_t cols,
                const Workspace& ws, hipStream_t s, hipError_t* err) {
  const uint32_t nb = cols / kBlockElems;
  if (rows == 0u || nb == 0u) return false;
  const uint32_t ntiles = (rows + 15u) / 16u;
  const SliceChoice sc = q4_slices(ntiles, nb, ws.bytes, QB);
  if (shape_ok(rows, cols, 1u, QB, 2u) && two_block_stages(ntiles, nb, ws.bytes, QB, sc) &&
      launch_wd<12, 1, 1, QB, false, 2>(w, nullptr, x, y, rows, nb, ws, s, err))
    return true;
  const uint32_t S = sc.slices;
  if (S < 2u) return false;
  if (sliced_two_block(ntiles, nb, S, ws.bytes) &&
      launch_sliced<12, 1, QB, 2>(w, x, y, rows, nb, S, ws, s, err))
    return true;
  if constexpr (QB == 4) {  // (Q5_K's weight registers leave room for 8 waves)
    if (launch_sliced<12, 1, QB>(w, x, y, rows, nb, S, ws, s, err)) return true;
  }
  return launch_sliced<8, 1, QB>(w, x, y, rows, nb, S, ws, s, err) ||
         launch_sliced<4, 1, QB>(w, x, y, rows, nb, S, ws, s, err);
}

// One vector, Q5_K in four-block stages (8 waves: their 20 weight pieces per
// wave leave too few registers for 12).
bool launch_q5k_one(const uint8_t* w, const float* x, float* y, uint32_t rows, uint32_t nb,
                    const Workspace& ws, hipStream_t s, hipError_t* err) {
  static const int cfg = env_int("SI_HIP_Q5K_MFMA_CFG", 0);
  switch (cfg) {
    case 1: return launch_wd<8, 1, 1, 5>(w, nullptr, x, y, rows, nb, ws, s, err);
    case 2:
      return shape_ok(rows, nb * kBlockElems, 1u, 5, 2u) &&
             launch_wd<12, 1, 1, 5, false, 2>(w, nullptr, x, y, rows, nb, ws, s, err);
    default: break;
  }
  return launch_wd<8, 1, 1, 5>(w, nullptr, x, y, rows, nb, ws, s, err) ||
         launch_wd<4, 1, 1, 5>(w, nullptr, x, y, rows, nb, ws, s, err);
}

}  // namespace

bool launch_q4k_matvec_mfma(const uint8_t* w, const float* x, float* y, uint32_t rows,
                            uint32_t cols, const Workspace& ws, hipStream_t s, hipError_t* err) {
  static const int cfg = env_int("SI_HIP_Q4K_MFMA_CFG", 0);
  if (cfg == 0 && try_sliced<4>(w, x, y, rows, cols, ws, s, err)) return true;
  if (!shape_ok(rows, cols, 1u, 4)) return false;
  const uint32_t nb = cols / kBlockElems;
  switch (cfg) {
    case 5:
      return shape_ok(rows, cols, 1u, 4, 2u) &&
             launch_wd<12, 1, 1, 4, false, 2>(w, nullptr, x, y, rows, nb, ws, s, err);
    case 1: return launch_wd<12, 1, 1>(w, nullptr, x, y, rows, nb, ws, s, err);
    case 2: return launch_wd<8, 1, 1>(w, nullptr, x, y, rows, nb, ws, s, err);
    case 3: return launch_wd<4, 3, 1>(w, nullptr, x, y, rows, nb, ws, s, err);
    case 4: return launch_wd<5, 3, 1>(w, nullptr, x, y, rows, nb, ws, s, err);
    case 6:
      return lines_fit(nb, w) &&
             launch_wd<6, 2, 1, 4, false, 4, true>(w, nullptr, x, y, rows, nb, ws, s, err);
    case 7:
      return lines_fit(nb, w) &&
             launch_wd<12, 1, 1, 4, false, 4, true>(w, nullptr, x, y, rows, nb, ws, s, err);
    case 8:
      return lines_fit(nb, w) &&
             launch_wd<8, 1, 1, 4, false, 4, true>(w, nullptr, x, y, rows, nb, ws, s, err);
    default: break;
  }
  // full-line copies where the shape allows them (17408 x 5120, us, 600 MB of
  // copies in turn): 12 waves 12.3, 8 waves 14.1, 6 waves with two stages in
  // flight 16.4 (the stage arithmetic needs three waves per SIMD to hide its
  // latency); the half-line copies at 12 waves 13.0.  (Out of the 256 MB Infinity
  // Cache, which the nontemporal lines pass by, the half-line copies are up to 3 %
  // ahead; a model's weights come from HBM.)
  if (lines_fit(nb, w) &&
      launch_wd<12, 1, 1, 4, false, 4, true>(w, nullptr, x, y, rows, nb, ws, s, err))
    return true;
  return launch_wd<12, 1, 1>(w, nullptr, x, y, rows, nb, ws, s, err) ||
         launch_wd<8, 1, 1>(w, nullptr, x, y, rows, nb, ws, s, err) ||
         launch_wd<4, 1, 1>(w, nullptr, x, y, rows, nb, ws, s, err);
}

static_assert(kMaxGroupWeights == kMaxGroup, "the C ABI's group limit is the kernels'");

bool launch_matvec_group(uint32_t type, const uint8_t* const* w, const uint32_t* rows,
                         uint32_t count, uint32_t cols, const float* x, float* y,
                         const Workspace& ws, hipStream_t s, hipError_t* err) {
  if (count < 2u || count > kMaxGroup) return false;
  GroupArgs ga{};
  for (uint32_t k = 0; k < kMaxGroup; ++k) ga.tile_end[k] = 0xffffffffu;
  uint64_t tiles = 0, total = 0;
  for (uint32_t k = 0; k < count; ++k) {
    if (rows[k] == 0u || (k + 1u < count && rows[k] % 16u != 0u) || !word_aligned(w[k]))
      return false;
    ga.w[k] = w[k];
    ga.rows[k] = rows[k];
    total += rows[k];
    tiles += (rows[k] + 15u) / 16u;
    if (total > 0xffffffffu) return false;
    ga.tile_end[k] = (uint32_t)tiles;
  }
  const uint32_t nb = cols / kBlockElems, trows = (uint32_t)total;
  // two-block stages where one matrix of the group's rows would take them
  static const int group_two_block = env_int("SI_HIP_GROUP_TWO_BLOCK", 1);
  if (group_two_block != 0 && (type == kTypeQ4K || type == kTypeQ5K) &&
      shape_ok(trows, cols, 1u, type == kTypeQ4K ? 4 : 5, 2u) &&
      two_block_stages((uint32_t)tiles, nb, ws.bytes, type == kTypeQ4K ? 4 : 5, SliceChoice{})) {
    if (type == kTypeQ4K &&
        launch_wd<12, 1, 1, 4, true, 2>(w[0], nullptr, x, y, trows, nb, ws, s, err, ga))
      return true;
    if (type == kTypeQ5K &&
        launch_wd<12, 1, 1, 5, true, 2>(w[0], nullptr, x, y, trows, nb, ws, s, err, ga))
      return true;
  }
  switch (type) {
    case kTypeQ4K:
      return shape_ok(trows, cols, 1u, 4) &&
             (launch_wd<12, 1, 1, 4, true>(w[0], nullptr, x, y, trows, nb, ws, s, err, ga) ||
              launch_wd<8, 1, 1, 4, true>(w[0], nullptr, x, y, trows, nb, ws, s, err, ga));
    case kTypeQ5K:
      return shape_ok(trows, cols, 1u, 5) &&
             (launch_wd<8, 1, 1, 5, true>(w[0], nullptr, x, y, trows, nb, ws, s, err, ga) ||
              launch_wd<4, 1, 1, 5, true>(w[0], nullptr, x, y, trows, nb, ws, s, err, ga));
    case kTypeQ6K:
      return launch_q6k_matvec_group(ga, trows, cols, x, y, ws, s, err);
    default:
      return false;
  }
}

bool launch_q5k_matvec_mfma(const uint8_t* w, const float* x, float* y, uint32_t rows,
                            uint32_t cols, const Workspace& ws, hipStream_t s, hipError_t* err) {
  static const int cfg = env_int("SI_HIP_Q5K_MFMA_CFG", 0);
  if (cfg == 0 && try_sliced<5>(w, x, y, rows, cols, ws, s, err)) return true;
  if (!shape_ok(rows, cols, 1u, 5)) return false;
  return launch_q5k_one(w, x, y, rows, cols / kBlockElems, ws, s, err);
}

bool launch_q4k_matmul_mfma(const uint8_t* w, const float* x, float* y, uint32_t rows,
                            uint32_t cols, uint32_t batch, const Workspace& ws, hipStream_t s,
                            hipError_t* err) {
  if (batch < 2 || batch > 16 || !shape_ok(rows, cols, 1u, 4)) return false;
  const uint32_t nb = cols / kBlockElems;
  if (batch == 2u && two_vectors(kTypeQ4K, rows, nb) && shape_ok(rows, cols, 1u, 4, 2u) &&
      launch_wd<12, 1, 1, 4, false, 2, false, 2>(w, nullptr, x, y, rows, nb, ws, s, err))
    return true;
  return launch_q45_tokens(4, w, x, y, rows, nb, batch, ws, s, err);
}

bool launch_q5k_matmul_mfma(const uint8_t* w, const float* x, float* y, uint32_t rows,
                            uint32_t cols, uint32_t batch, const Workspace& ws, hipStream_t s,
                            hipError_t* err) {
  if (batch < 2 || batch > 16 || !shape_ok(rows, cols, 1u, 5)) return false;
  const uint32_t nb = cols / kBlockElems;
  if (batch == 2u && two_vectors(kTypeQ5K, rows, nb) && shape_ok(rows, cols, 1u, 5, 2u) &&
      launch_wd<12, 1, 1, 5, false, 2, false, 2>(w, nullptr, x, y, rows, nb, ws, s, err))
    return true;
  return launch_q45_tokens(5, w, x, y, rows, nb, batch, ws, s, err);
}

bool launch_q4k_gate_up_mfma(const uint8_t* gate, const uint8_t* up, const float* x, float* h,
                             uint32_t rows, uint32_t cols, const Workspace& ws, hipStream_t s,
                             hipError_t* err) {
  if (!shape_ok(rows, cols, 2u, 4)) return false;
  const uint32_t nb = cols / kBlockElems;
  static const int cfg = env_int("SI_HIP_GATE_UP_MFMA_CFG", 0);
  switch (cfg) {
    case 1: return launch_wd<12, 1, 2>(gate, up, x, h, rows, nb, ws, s, err);
    case 2: return launch_wd<8, 1, 2>(gate, up, x, h, rows, nb, ws, s, err);
    case 3: return launch_wd<10, 1, 2>(gate, up, x, h, rows, nb, ws, s, err);
    case 4:
      return lines_fit(nb, gate, up) &&
             launch_wd<6, 2, 2, 4, false, 4, true>(gate, up, x, h, rows, nb, ws, s, err);
    case 5:
      return lines_fit(nb, gate, up) &&
             launch_wd<12, 1, 2, 4, false, 4, true>(gate, up, x, h, rows, nb, ws, s, err);
    default: break;
  }
  // full-line copies at 12 waves: 17408 x 5120 21.3 us against 22.1
  if (lines_fit(nb, gate, up) &&
      launch_wd<12, 1, 2, 4, false, 4, true>(gate, up, x, h, rows, nb, ws, s, err))
    return true;
  // 12 waves (163 VGPRs, no spills) against 8, half-line copies, us: 17408 x 5120
  // 22.1 / 23.9, 14336 x 4096 16.8 / 17.4, 11008 x 4096 14.1 / 14.6, 8192 x 2048
  // and 4096 x 4096 level at 7.8
  return launch_wd<12, 1, 2>(gate, up, x, h, rows, nb, ws, s, err) ||
         launch_wd<8, 1, 2>(gate, up, x, h, rows, nb, ws, s, err) ||
         launch_wd<4, 1, 2>(gate, up, x, h, rows, nb, ws, s, err);
}

}  // namespace sihip
