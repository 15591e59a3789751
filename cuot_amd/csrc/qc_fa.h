// qc_fa.h -- the field, the Cantor basis and the chunk maps of the Frobenius-orbit
// transform (qc_fa.hip).
//
// Field: GF(16) = GF(2)[y]/(y^4 + y + 1), GF(2^16) = GF(16)[w]/(w^4 + y w^2 +
// y^2 w + y^3) (nibble g of a word: coefficient of w^g), GF(2^32) = GF(2^16)[theta]
// with theta^2 = theta + nu (high half: coefficient of theta).  Nibbles, because a
// product by a constant is then a choice between 16 patterns of XORs per
// constant nibble, every output plane taking one three-input XOR.
// Basis: beta_0 = 1, beta_i^2 + beta_i = beta_{i-1}, beta_15 = nu and therefore
// beta_16 = theta; above 16 each beta is a root of x^2 + x = beta_{i-1}
// (coordinate 0 clear).  The lowest, which tell lanes of a wavefront apart, are
// 1 + y + y^2, y^2, y^3 and w^2 + y^2 w: the reduction polynomial was chosen for
// that (and for its one-XOR coefficients), the roots upwards for clear nibbles.
#pragma once

#include "gf32.h"

constexpr uint32_t FA_NU = 0x2c1e;

constexpr uint32_t fa_mul4(uint32_t a, uint32_t b) {
  uint32_t r = 0;
  for (int i = 0; i < 4; i++)
    if ((b >> i) & 1) r ^= a << i;
  for (int i = 6; i >= 4; i--)
    if ((r >> i) & 1) r ^= 0x13u << (i - 4);
  return r;
}

constexpr uint32_t fa_mul16(uint32_t a, uint32_t b) {
  uint32_t p[7] = {};
  for (int i = 0; i < 4; i++)
    for (int j = 0; j < 4; j++) p[i + j] ^= fa_mul4((a >> (4 * i)) & 15, (b >> (4 * j)) & 15);
  for (int i = 6; i >= 4; i--) {
    p[i - 2] ^= fa_mul4(2, p[i]);
    p[i - 3] ^= fa_mul4(4, p[i]);
    p[i - 4] ^= fa_mul4(8, p[i]);
  }
  return p[0] | p[1] << 4 | p[2] << 8 | p[3] << 12;
}

constexpr uint32_t fa_mul32(uint32_t a, uint32_t b) {
  const uint32_t a0 = a & 0xFFFFu, a1 = a >> 16, b0 = b & 0xFFFFu, b1 = b >> 16;
  const uint32_t p0 = fa_mul16(a0, b0), p1 = fa_mul16(a1, b1), p2 = fa_mul16(a0 ^ a1, b0 ^ b1);
  return (p0 ^ fa_mul16(FA_NU, p1)) | ((p2 ^ p0) << 16);
}

struct FaBeta16 {
  uint32_t v[16];
};

constexpr FaBeta16 fa_beta16() {
  FaBeta16 b{};
  b.v[15] = FA_NU;
  for (int i = 14; i >= 0; i--) b.v[i] = fa_mul16(b.v[i + 1], b.v[i + 1]) ^ b.v[i + 1];
  return b;
}

inline constexpr FaBeta16 kFaBeta = fa_beta16();
static_assert(kFaBeta.v[0] == 1, "nu has trace 1");
static_assert(kFaBeta.v[1] == 7 && kFaBeta.v[2] == 4 && kFaBeta.v[3] == 8 && kFaBeta.v[4] == 0x140,
              "what the products by lane-dependent constants assume");

// all 32
struct FaBasis {
  uint32_t v[32];
};

constexpr FaBasis fa_basis() {
  FaBasis b{};
  uint32_t* beta = b.v;
  for (int i = 0; i < 16; i++) beta[i] = kFaBeta.v[i];
  beta[16] = 0x10000u;
  uint32_t img[32] = {0};
  for (int j = 1; j < 32; j++) img[j] = fa_mul32(1u << j, 1u << j) ^ (1u << j);
  for (int i = 17; i < 32; i++) {
    // x^2 + x = beta[i-1]: elimination on the images of the 31 unit vectors
    uint32_t bv[32] = {0}, bm[32] = {0};
    for (int j = 1; j < 32; j++) {
      uint32_t v = img[j], m = 1u << j;
      while (v) {
        const int h = 31 - __builtin_clz(v);
        if (!bm[h]) {
          bv[h] = v;
          bm[h] = m;
          break;
        }
        v ^= bv[h];
        m ^= bm[h];
      }
    }
    uint32_t v = beta[i - 1], m = 0;
    while (v) {
      const int h = 31 - __builtin_clz(v);
      v ^= bv[h];
      m ^= bm[h];
    }
    beta[i] = m;
  }
  return b;
}

// Transform of products of 2^K coefficients: the points are beta_a + the span
// of beta_i, i < c or c < i <= K - 5, with c = min(K - 5, 15) and a = 16 + c.
// At coefficient index bits K-4 .. K-1 every point has the same s_k value,
// beta_{a-k}: four bits (three in a half-length input) are one GF(2^16) value.
// kc = 0 for K <= 20, K - 20 above.
struct FaChunk {
  uint32_t pack[16];    // pack[q] = product over the bits b of q of beta_{a-(K-4+b)}
  uint32_t unpack[16];  // bit j of unpack[q]: coordinate j contributes to coefficient q
};

constexpr FaChunk fa_chunk(int kc) {
  FaChunk m{};
  for (int q = 0; q < 16; q++) {
    m.pack[q] = 1;
    for (int b = 0; b < 4; b++)
      if ((q >> b) & 1) m.pack[q] = fa_mul16(m.pack[q], kFaBeta.v[15 - kc - b]);
  }
  uint32_t a[16] = {}, inv[16] = {};
  for (int r = 0; r < 16; r++) {
    for (int q = 0; q < 16; q++) a[r] |= ((m.pack[q] >> r) & 1u) << q;
    inv[r] = 1u << r;
  }
  for (int c = 0; c < 16; c++) {
    int piv = c;
    while (!((a[piv] >> c) & 1u)) piv++;  // the products are a basis
    const uint32_t ta = a[piv], ti = inv[piv];
    a[piv] = a[c];
    inv[piv] = inv[c];
    a[c] = ta;
    inv[c] = ti;
    for (int r = 0; r < 16; r++)
      if (r != c && ((a[r] >> c) & 1u)) {
        a[r] ^= a[c];
        inv[r] ^= inv[c];
      }
  }
  for (int q = 0; q < 16; q++) m.unpack[q] = inv[q];
  return m;
}

constexpr int FA_KC_MAX = 5;  // K <= 25
template <int KC>
inline constexpr FaChunk kFaChunk = fa_chunk(KC);

// out[0..15] = the GF(2^16) value of 8 chunk-bit planes (bits K-4 .. K-2)
template <int KC>
GF32_HD void fa_pack_planes(const uint32_t* in, uint32_t* out) {
#pragma unroll
  for (int j = 0; j < 16; j++) {
    uint32_t s = 0;
#pragma unroll
    for (int q = 0; q < 8; q++)
      if ((kFaChunk<KC>.pack[q] >> j) & 1u) s ^= in[q];
    out[j] = s;
  }
}

// out[0..15] = the 16 coefficient planes (bits K-4 .. K-1) of a value
template <int KC>
GF32_HD void fa_unpack_planes(const uint32_t* in, uint32_t* out) {
#pragma unroll
  for (int q = 0; q < 16; q++) {
    uint32_t s = 0;
#pragma unroll
    for (int j = 0; j < 16; j++)
      if ((kFaChunk<KC>.unpack[q] >> j) & 1u) s ^= in[j];
    out[q] = s;
  }
}

#if defined(__HIPCC__)
// ---- bitsliced products by a constant ------------------------------------------------
// Bit planes: planes 4g .. 4g+3 are the coefficient of w^g, plane i of a group that
// of y^i.

// v and the sums of its even plane pairs
struct FaOp {
  uint32_t p[16], lo[4], hi[4];
  __device__ __forceinline__ explicit FaOp(const uint32_t* v) {
#pragma unroll
    for (int i = 0; i < 16; i++) p[i] = v[i];
#pragma unroll
    for (int g = 0; g < 4; g++) {
      lo[g] = v[4 * g] ^ v[4 * g + 1];
      hi[g] = v[4 * g + 2] ^ v[4 * g + 3];
    }
  }
};

// Nibble cases: plane i of d v as the sum of p0 .. p3, l = p0 + p1, h = p2 + p3 of the
// group; X2 takes one of them, X3 two.
#define FA_D1(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X2(a0, p0) X2(a1, p1) X2(a2, p2) X2(a3, p3)
#define FA_D2(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X2(a0, p3) X3(a1, p0, p3) X2(a2, p1) X2(a3, p2)
#define FA_D3(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X3(a0, p0, p3) X3(a1, l, p3) X3(a2, p1, p2) X2(a3, h)
#define FA_D4(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X2(a0, p2) X2(a1, h) X3(a2, p0, p3) X2(a3, p1)
#define FA_D5(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X3(a0, p0, p2) X3(a1, p1, h) X3(a2, p0, h) X3(a3, p1, p3)
#define FA_D6(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X2(a0, h) X3(a1, p0, p2) X3(a2, l, p3) X3(a3, p1, p2)
#define FA_D7(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X3(a0, p0, h) X3(a1, l, p2) X3(a2, l, h) X3(a3, p1, h)
#define FA_D8(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X2(a0, p1) X3(a1, p1, p2) X2(a2, h) X3(a3, p0, p3)
#define FA_D9(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X2(a0, l) X2(a1, p2) X2(a2, p3) X2(a3, p0)
#define FA_D10(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X3(a0, p1, p3) X3(a1, l, h) X3(a2, p1, h) X3(a3, p0, h)
#define FA_D11(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X3(a0, l, p3) X3(a1, p0, h) X3(a2, p1, p3) X3(a3, p0, p2)
#define FA_D12(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X3(a0, p1, p2) X3(a1, p1, p3) X3(a2, p0, p2) X3(a3, l, p3)
#define FA_D13(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X3(a0, l, p2) X2(a1, p3) X2(a2, p0) X2(a3, l)
#define FA_D14(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X3(a0, p1, h) X2(a1, l) X3(a2, l, p2) X3(a3, l, h)
#define FA_D15(X2, X3, a0, a1, a2, a3, p0, p1, p2, p3, l, h) \
  X3(a0, l, h) X2(a1, p0) X2(a2, l) X3(a3, l, p2)
#define FA_ADD2(a, x) "v_xor_b32 " a ", " x ", " a "\n"
#define FA_ADD3(a, x, y) "v_bitop3_b32 " a ", " a ", " x ", " y " bitop3:0x96\n"
#define FA_SET2(a, x) "v_mov_b32 " a ", " x "\n"
#define FA_SET3(a, x, y) "v_xor_b32 " a ", " x ", " y "\n"
#define FA_CASE(D, X2, X3) \
  "FA" #D "_%=:\n" \
  FA_D##D(X2, X3, "%[a0]", "%[a1]", "%[a2]", "%[a3]", "%[p0]", "%[p1]", "%[p2]", "%[p3]", \
          "%[l0]", "%[h0]") \
  FA_D##D(X2, X3, "%[a4]", "%[a5]", "%[a6]", "%[a7]", "%[p4]", "%[p5]", "%[p6]", "%[p7]", \
          "%[l1]", "%[h1]") \
  FA_D##D(X2, X3, "%[a8]", "%[a9]", "%[a10]", "%[a11]", "%[p8]", "%[p9]", "%[p10]", "%[p11]", \
          "%[l2]", "%[h2]") \
  FA_D##D(X2, X3, "%[a12]", "%[a13]", "%[a14]", "%[a15]", "%[p12]", "%[p13]", "%[p14]", "%[p15]", \
          "%[l3]", "%[h3]") \
  "s_branch FAend_%=\n"
#define FA_BIT(B, ONE) "s_bitcmp1_b32 %[d], " #B "\ns_cbranch_scc1 FA" #ONE "_%=\n"
#define FA_CASES(X2, X3)                                                                                            \
  FA_BIT(3, t8) FA_BIT(2, t4) FA_BIT(1, t2) FA_BIT(0, 1) "FA0_%=:\n" X2##_ZERO "s_branch FAend_%=\n"             \
  FA_CASE(1, X2, X3)                                                                                                \
  "FAt2_%=:\n" FA_BIT(0, 3) FA_CASE(2, X2, X3) FA_CASE(3, X2, X3)                                                  \
  "FAt4_%=:\n" FA_BIT(1, t6) FA_BIT(0, 5) FA_CASE(4, X2, X3) FA_CASE(5, X2, X3)                                  \
  "FAt6_%=:\n" FA_BIT(0, 7) FA_CASE(6, X2, X3) FA_CASE(7, X2, X3)                                                  \
  "FAt8_%=:\n" FA_BIT(2, t12) FA_BIT(1, t10) FA_BIT(0, 9) FA_CASE(8, X2, X3) FA_CASE(9, X2, X3)                \
  "FAt10_%=:\n" FA_BIT(0, 11) FA_CASE(10, X2, X3) FA_CASE(11, X2, X3)                                              \
  "FAt12_%=:\n" FA_BIT(1, t14) FA_BIT(0, 13) FA_CASE(12, X2, X3) FA_CASE(13, X2, X3)                             \
  "FAt14_%=:\n" FA_BIT(0, 15) FA_CASE(14, X2, X3) FA_CASE(15, X2, X3) "FAend_%=:\n"
#define FA_ADD2_ZERO
#define FA_SET2_ZERO \
  "v_mov_b32 %[a0], 0\n" "v_mov_b32 %[a1], 0\n" "v_mov_b32 %[a2], 0\n" "v_mov_b32 %[a3], 0\n" \
  "v_mov_b32 %[a4], 0\n" "v_mov_b32 %[a5], 0\n" "v_mov_b32 %[a6], 0\n" "v_mov_b32 %[a7], 0\n" \
  "v_mov_b32 %[a8], 0\n" "v_mov_b32 %[a9], 0\n" "v_mov_b32 %[a10], 0\n" "v_mov_b32 %[a11], 0\n" \
  "v_mov_b32 %[a12], 0\n" "v_mov_b32 %[a13], 0\n" "v_mov_b32 %[a14], 0\n" "v_mov_b32 %[a15], 0\n"
#define FA_OPERANDS(C) \
  [a0] C(a[0]), [a1] C(a[1]), [a2] C(a[2]), [a3] C(a[3]), \
  [a4] C(a[4]), [a5] C(a[5]), [a6] C(a[6]), [a7] C(a[7]), \
  [a8] C(a[8]), [a9] C(a[9]), [a10] C(a[10]), [a11] C(a[11]), \
  [a12] C(a[12]), [a13] C(a[13]), [a14] C(a[14]), [a15] C(a[15]) \
      : [p0] "v"(v.p[0]), [p1] "v"(v.p[1]), [p2] "v"(v.p[2]), [p3] "v"(v.p[3]), \
        [p4] "v"(v.p[4]), [p5] "v"(v.p[5]), [p6] "v"(v.p[6]), [p7] "v"(v.p[7]), \
        [p8] "v"(v.p[8]), [p9] "v"(v.p[9]), [p10] "v"(v.p[10]), [p11] "v"(v.p[11]), \
        [p12] "v"(v.p[12]), [p13] "v"(v.p[13]), [p14] "v"(v.p[14]), [p15] "v"(v.p[15]), \
        [l0] "v"(v.lo[0]), [h0] "v"(v.hi[0]), [l1] "v"(v.lo[1]), [h1] "v"(v.hi[1]), \
        [l2] "v"(v.lo[2]), [h2] "v"(v.hi[2]), [l3] "v"(v.lo[3]), [h3] "v"(v.hi[3]), \
        [d] "s"(d) \
      : "scc"
#define FA_OUT(x) "=&v"(x)
#define FA_INOUT(x) "+&v"(x)

// a (^)= d v for the low nibble d of a wavefront-uniform word: a scalar branch to
// one operation per plane.  One block of assembly: with the cases in C++ the
// compiler put moves of whole accumulators between them.
template <bool SET>
__device__ __forceinline__ void fa_digit(uint32_t* a, const FaOp& v, uint32_t d) {
  if constexpr (SET)
    asm(FA_CASES(FA_SET2, FA_SET3) : FA_OPERANDS(FA_OUT));
  else
    asm(FA_CASES(FA_ADD2, FA_ADD3) : FA_OPERANDS(FA_INOUT));
}

// a = w a
__device__ __forceinline__ void fa_times_w(uint32_t* a) {
  const uint32_t h0 = a[12], h1 = a[13], h2 = a[14], h3 = a[15], h03 = h0 ^ h3, h12 = h1 ^ h2, h23 = h2 ^ h3;
#pragma unroll
  for (int i = 0; i < 4; i++) a[12 + i] = a[8 + i];
  const uint32_t y1[4] = {h3, h03, h1, h2}, y2[4] = {h2, h23, h03, h1}, y3[4] = {h1, h12, h23, h03};
#pragma unroll
  for (int i = 0; i < 4; i++) {
    a[8 + i] = a[4 + i] ^ y1[i];
    a[4 + i] = a[i] ^ y2[i];
    a[i] = y3[i];
  }
}

// a = c v, c in GF(2^16) the same in the whole wavefront
__device__ __forceinline__ void fa_mulc16(const uint32_t* v, uint32_t c, uint32_t* a) {
  const FaOp op(v);
  fa_digit<true>(a, op, c >> 12);
  fa_times_w(a);
  fa_digit<false>(a, op, c >> 8);
  fa_times_w(a);
  fa_digit<false>(a, op, c >> 4);
  fa_times_w(a);
  fa_digit<false>(a, op, c);
}

// x ^= y & m (in assembly: the compiler regroups long sums of these into half as
// many operations again, and spills)
__device__ __forceinline__ void fa_add_masked(uint32_t& x, uint32_t y, uint32_t m) {
  asm("v_bitop3_b32 %0, %0, %1, %2 bitop3:0x78" : "+v"(x) : "v"(y), "v"(m));
}

// the same for any c (per lane): every bit of c is a mask
__device__ __forceinline__ void fa_mulv16(const uint32_t* v, uint32_t c, uint32_t* a) {
#pragma unroll
  for (int i = 0; i < 16; i++) a[i] = 0;
#pragma unroll
  for (int q = 3; q >= 0; q--) {
    if (q < 3) fa_times_w(a);
    uint32_t m[4];
#pragma unroll
    for (int j = 0; j < 4; j++) m[j] = (uint32_t)((int32_t)(c << (31 - 4 * q - j)) >> 31);
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const uint32_t p0 = v[4 * g], p1 = v[4 * g + 1], p2 = v[4 * g + 2], p3 = v[4 * g + 3];
      const uint32_t p03 = p0 ^ p3, p12 = p1 ^ p2, p23 = p2 ^ p3;
      const uint32_t y[4][4] = {{p0, p1, p2, p3}, {p3, p03, p1, p2}, {p2, p23, p03, p1}, {p1, p12, p23, p03}};
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < 4; i++) fa_add_masked(a[4 * g + i], y[j][i], m[j]);
    }
  }
}

// a ^= (sum over the bits b of d of beta_{b+1}) v for d < 16 (per lane)
__device__ __forceinline__ void fa_add_low(const uint32_t* v, uint32_t d, uint32_t* a) {
  uint32_t m[4];
#pragma unroll
  for (int j = 0; j < 4; j++) m[j] = (uint32_t)((int32_t)(d << (31 - j)) >> 31);
#pragma unroll
  for (int g = 0; g < 4; g++) {  // 1 + y + y^2
    const uint32_t p0 = v[4 * g], p1 = v[4 * g + 1], p2 = v[4 * g + 2], p3 = v[4 * g + 3], p01 = p0 ^ p1;
    fa_add_masked(a[4 * g], p0 ^ p2 ^ p3, m[0]);
    fa_add_masked(a[4 * g + 1], p01 ^ p2, m[0]);
    fa_add_masked(a[4 * g + 2], p01 ^ p2 ^ p3, m[0]);
    fa_add_masked(a[4 * g + 3], p1 ^ p2 ^ p3, m[0]);
  }
  if (!__any(d > 1)) return;
#pragma unroll
  for (int g = 0; g < 4; g++) {  // y^2
    const uint32_t p0 = v[4 * g], p1 = v[4 * g + 1], p2 = v[4 * g + 2], p3 = v[4 * g + 3];
    fa_add_masked(a[4 * g], p2, m[1]);
    fa_add_masked(a[4 * g + 1], p2 ^ p3, m[1]);
    fa_add_masked(a[4 * g + 2], p0 ^ p3, m[1]);
    fa_add_masked(a[4 * g + 3], p1, m[1]);
  }
  if (!__any(d > 3)) return;
#pragma unroll
  for (int g = 0; g < 4; g++) {  // y^3
    const uint32_t p0 = v[4 * g], p1 = v[4 * g + 1], p2 = v[4 * g + 2], p3 = v[4 * g + 3];
    fa_add_masked(a[4 * g], p1, m[2]);
    fa_add_masked(a[4 * g + 1], p1 ^ p2, m[2]);
    fa_add_masked(a[4 * g + 2], p2 ^ p3, m[2]);
    fa_add_masked(a[4 * g + 3], p0 ^ p3, m[2]);
  }
  if (!__any(d > 7)) return;
  uint32_t x[16];  // w^2 + y^2 w
#pragma unroll
  for (int i = 0; i < 16; i++) x[i] = v[i] & m[3];
  fa_times_w(x);
#pragma unroll
  for (int g = 0; g < 4; g++) {
    a[4 * g] ^= x[4 * g + 2];
    a[4 * g + 1] ^= x[4 * g + 2] ^ x[4 * g + 3];
    a[4 * g + 2] ^= x[4 * g] ^ x[4 * g + 3];
    a[4 * g + 3] ^= x[4 * g + 1];
  }
  fa_times_w(x);
#pragma unroll
  for (int i = 0; i < 16; i++) a[i] ^= x[i];
}

// u += c v in GF(2^32) for c = c0 + c1 theta the same in the whole wavefront, nc =
// nu c1:  u0 += c0 v0 + nc v1,  u1 += c1 v0 + (c0 + c1) v1.  Four products that
// share two accumulators beat three that do not: 360 operations on average
// against 390 (a zero nibble costs a branch only).
__device__ __forceinline__ void fa_add_mul16x2(uint32_t* u, const FaOp& v0, const FaOp& v1, uint32_t c, uint32_t d) {
  uint32_t a[16];
  fa_digit<true>(a, v0, c >> 12);
  fa_digit<false>(a, v1, d >> 12);
  fa_times_w(a);
  fa_digit<false>(a, v0, c >> 8);
  fa_digit<false>(a, v1, d >> 8);
  fa_times_w(a);
  fa_digit<false>(a, v0, c >> 4);
  fa_digit<false>(a, v1, d >> 4);
  fa_times_w(a);
  fa_digit<false>(a, v0, c);
  fa_digit<false>(a, v1, d);
#pragma unroll
  for (int i = 0; i < 16; i++) u[i] ^= a[i];
}

__device__ __forceinline__ void fa_add_mul32(uint32_t* u, const uint32_t* v, uint32_t c, uint32_t nc) {
  const FaOp v0(v), v1(v + 16);
  fa_add_mul16x2(u, v0, v1, c, nc);
  __builtin_amdgcn_sched_barrier(0);  // one accumulator at a time
  fa_add_mul16x2(u + 16, v0, v1, c >> 16, c ^ (c >> 16));
}

// v = c v for any c (per lane), three products:
//   c0 v0 + (nu c1) v1,   c0 v0 + (c0 + c1) (v0 + v1)
// (one after the other, for registers)
__device__ __forceinline__ void fa_mulv32(uint32_t* v, uint32_t c, uint32_t nc) {
  uint32_t t[16], a[16], b[16];
#pragma unroll
  for (int i = 0; i < 16; i++) t[i] = v[i] ^ v[16 + i];
  fa_mulv16(v, c, a);
  __builtin_amdgcn_sched_barrier(0);
  fa_mulv16(v + 16, nc, b);
#pragma unroll
  for (int i = 0; i < 16; i++) v[i] = a[i] ^ b[i];
  __builtin_amdgcn_sched_barrier(0);
  fa_mulv16(t, c ^ (c >> 16), b);
#pragma unroll
  for (int i = 0; i < 16; i++) v[16 + i] = a[i] ^ b[i];
}

// scalar products (preparation)
__device__ __forceinline__ uint32_t fa_times_y(uint32_t x) {  // every nibble
  const uint32_t t = (x >> 3) & 0x11111111u;
  return ((x << 1) & 0xEEEEEEEEu) ^ t ^ (t << 1);
}

__device__ __forceinline__ uint32_t fa_mul16_dev(uint32_t a, uint32_t b) {
  uint32_t y[4] = {a, 0, 0, 0}, r = 0;
#pragma unroll
  for (int j = 1; j < 4; j++) y[j] = fa_times_y(y[j - 1]);
#pragma unroll
  for (int g = 0; g < 4; g++) {
    uint32_t t = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) t ^= y[j] & (uint32_t)((int32_t)(b << (31 - 4 * g - j)) >> 31);
    r ^= t << (4 * g);
  }
  uint32_t h = r >> 16;  // w^4 .. w^6
  h ^= fa_times_y(h >> 8);
  const uint32_t y1 = fa_times_y(h), y2 = fa_times_y(y1), y3 = fa_times_y(y2);
  return (r ^ (y1 << 8) ^ (y2 << 4) ^ y3) & 0xFFFFu;
}

__device__ __forceinline__ uint32_t fa_mul32_dev(uint32_t a, uint32_t b, uint32_t nb) {  // nb = nu b1
  const uint32_t a0 = a & 0xFFFFu, a1 = a >> 16, b0 = b & 0xFFFFu, b1 = b >> 16;
  const uint32_t p0 = fa_mul16_dev(a0, b0);
  return p0 ^ fa_mul16_dev(a1, nb) | (fa_mul16_dev(a0 ^ a1, b0 ^ b1) ^ p0) << 16;
}
#endif
