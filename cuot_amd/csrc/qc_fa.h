// qc_fa.h -- constants of the Frobenius-orbit transform (qc_fa.hip): the Cantor
// basis it runs on and the chunk maps between coefficient bits and GF(2^16).
//
// Basis: beta_0 = 1, beta_i^2 + beta_i = beta_{i-1}, chosen so that beta_15 is
// the tower's nu and therefore beta_16 its theta (theta^2 + theta = nu).  The
// lower half follows from beta_15 downwards; above 16 each beta is a root of
// x^2 + x = beta_{i-1} (coordinate 0 clear).
#pragma once

#include "gf32.h"

struct FaBeta16 {
  uint32_t v[16];
};

constexpr FaBeta16 fa_beta16() {
  FaBeta16 b{};
  b.v[15] = CUOT_GF16_NU;
  for (int i = 14; i >= 0; i--) b.v[i] = gf16_mul(b.v[i + 1], b.v[i + 1]) ^ b.v[i + 1];
  return b;
}

inline constexpr FaBeta16 kFaBeta = fa_beta16();
static_assert(kFaBeta.v[0] == 1, "nu has trace 1");

// all 32 (host)
static inline void fa_basis(uint32_t beta[32]) {
  for (int i = 0; i < 16; i++) beta[i] = kFaBeta.v[i];
  beta[16] = 0x10000u;
  for (int i = 17; i < 32; i++) {
    // x^2 + x = beta[i-1]: elimination on the images of the 31 unit vectors
    uint32_t bv[32] = {0}, bm[32] = {0};
    for (int j = 1; j < 32; j++) {
      uint32_t v = gf32_mul(1u << j, 1u << j) ^ (1u << j), m = 1u << j;
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
}

// Transform of products of 2^K coefficients: the points are beta_a + the span
// of beta_i, i < c or c < i <= K - 5, with c = min(K - 5, 15) and a = 16 + c.
// At coefficient index bits K-4 .. K-1 every point has the same s_k value,
// beta_{a-k}: four bits (three in a half-length input) are one GF(2^16) value.
// kc = 0 for K <= 20, K - 20 above.
struct FaChunk {
  uint32_t pack[16];    // value of chunk bit pattern 1 << q ... pack[q] = product over the bits b of q of beta_{a-(K-4+b)}
  uint32_t unpack[16];  // bit j of unpack[q]: coordinate j contributes to coefficient q
};

constexpr FaChunk fa_chunk(int kc) {
  FaChunk m{};
  for (int q = 0; q < 16; q++) {
    m.pack[q] = 1;
    for (int b = 0; b < 4; b++)
      if ((q >> b) & 1) m.pack[q] = gf16_mul(m.pack[q], kFaBeta.v[15 - kc - b]);
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
