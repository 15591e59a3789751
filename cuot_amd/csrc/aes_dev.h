// aes_dev.h -- AES-128 encryption on gfx950 with LDS-resident T-tables.
//
// CDNA4 has no AES instructions.  Each round is done with the 256-entry 32-bit
// table T0 (SubBytes + MixColumns of a row-0 byte) and T1 = T0 rotated by a
// byte; the tables of rows 2 and 3 are T0 and T1 rotated by 16, applied to the
// XOR of both lookups with one rotate.
//
// Layout: entry x is 256 bytes of LDS, 32 copies of T0[x] then 32 copies of
// T1[x]; lane l reads copy l % 32.  What bounds AES here is VALU issue, then
// the LDS: 160 dword reads per block at two cycles per wavefront allow 1.2e11
// AES/s.  The 256-byte entry makes a lookup address one v_perm_b32 (byte k of
// the state word over the lane's byte offset, for any k, with T1 behind the
// instruction's immediate offset), where 128-byte entries take a bit-field
// extract and a multiply-add; T1 saves two of three rotates per column; and
// the 32 copies keep each half wavefront on 32 distinct banks.  A round's
// column is 8 VALU operations (4 v_perm, XOR, rotate, three-input XOR, key)
// instead of 14, a block ~340 instead of 577.  Measured for pairs of AES on
// one input: 32 copies of T0 alone 5.0e10 AES/s, this form 8.3e10 with two
// 512-lane workgroups per CU (64 KB each) and 9.3e10 with two of 1024; 64
// copies of T0 7.6e10; four tables of 32 copies (128 KB, one 1024-lane
// workgroup per CU) 9.4e10, which leaves no room for tree nodes.
//
// The tables are computed on the host from the FIPS-197 definition of the
// S-box (multiplicative inverse + affine map) and uploaded at init.
//
// State words are little-endian columns: word c = bytes 4c..4c+3 of the block,
// i.e. the block's memory layout.  Output = FIPS-197 AES-128 of the 16 bytes.
#pragma once

#include "common.h"

#define CUOT_AES_LDS_WORDS (256 * 64)
// lanes of a workgroup that shares one table (two such workgroups per CU)
#define CUOT_AES_WG 512

// Grid of a kernel that streams n blocks through such workgroups: four rounds
// of the chip's 512 resident ones balance the tail and still spread each table
// fill over many blocks.
inline unsigned cuot_aes_grid(int64_t n) {
  int64_t g = (n + CUOT_AES_WG - 1) / CUOT_AES_WG;
  if (g > 2048) g = 2048;
  return g < 1 ? 1u : (unsigned)g;
}

typedef __attribute__((address_space(3))) const char* lds_cptr;

struct AesLds {
  lds_cptr base;      // the table (first in the kernel's LDS, so that it folds into the offset)
  uint32_t lane_off;  // (lane % 32) * 4 bytes, below 256
};

// Fill the table.  Call from all threads of the block, then sync.
// T0g: the 256-word table in global memory (uploaded by cuot_init).
// 16-byte chunk i of the table belongs to entry i / 16, its chunks 8..15 to T1.
CUOT_DEV void aes_stage_table(uint32_t* lds, const uint32_t* __restrict__ T0g, int tid, int nthreads) {
#pragma unroll 8
  for (int i = tid; i < CUOT_AES_LDS_WORDS / 4; i += nthreads) {
    const uint32_t t = T0g[i >> 4];
    const uint32_t v = (i & 8) ? (t << 8) | (t >> 24) : t;
    ((uint4*)lds)[i] = make_uint4(v, v, v, v);
  }
}

CUOT_DEV AesLds aes_lds(const uint32_t* lds) {
  AesLds a;
  a.base = (lds_cptr)lds;
  a.lane_off = (threadIdx.x & 31u) * 4u;
  return a;
}

// T0 (T = 0) or T1 (T = 1) at byte K of w
template <int K, int T>
CUOT_DEV uint32_t tlook(const AesLds& a, uint32_t w) {
  const uint32_t off = __builtin_amdgcn_perm(w, a.lane_off, 0x0c0c0000u | ((4u + K) << 8));
  return *(const __attribute__((address_space(3))) uint32_t*)(a.base + off + 128 * T);
}

// a ^ b ^ c as one three-input bit operation (table 0x96)
CUOT_DEV uint32_t aes_x3(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_bitop3_b32 %0, %1, %2, %3 bitop3:0x96" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

CUOT_DEV uint32_t aes_col(const AesLds& a, uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3, uint32_t k) {
  const uint32_t t0 = tlook<0, 0>(a, w0), t1 = tlook<1, 1>(a, w1);
  const uint32_t u = tlook<2, 0>(a, w2) ^ tlook<3, 1>(a, w3);
  return aes_x3(t0, t1, __builtin_amdgcn_alignbit(u, u, 16)) ^ k;
}

// Last round: S-box bytes recovered from the tables (bytes of T0[x]: 2s, s, s,
// 3s; of T1[x]: 3s, 2s, s, s)
CUOT_DEV uint32_t aes_col_last(const AesLds& a, uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3,
                               uint32_t k) {
  const uint32_t t0 = tlook<0, 0>(a, w0), t1 = tlook<1, 1>(a, w1);
  const uint32_t t2 = tlook<2, 0>(a, w2), t3 = tlook<3, 1>(a, w3);
  const uint32_t lo = __builtin_amdgcn_perm(t0, t1, 0x0c0c0205u);  // byte 1 of t0, byte 2 of t1
  const uint32_t hi = __builtin_amdgcn_perm(t2, t3, 0x02060c0cu);  // byte 2 of t2, byte 2 of t3
  return (lo | hi) ^ k;
}

// rk: 44 little-endian round-key words (FIPS w[0..43] in memory order).
CUOT_DEV blk aes_enc(const AesLds& a, const uint32_t* __restrict__ rk, blk in) {
  uint32_t s0 = in.x ^ rk[0], s1 = in.y ^ rk[1], s2 = in.z ^ rk[2], s3 = in.w ^ rk[3];
#pragma unroll
  for (int r = 1; r < 10; r++) {
    uint32_t n0 = aes_col(a, s0, s1, s2, s3, rk[4 * r + 0]);
    uint32_t n1 = aes_col(a, s1, s2, s3, s0, rk[4 * r + 1]);
    uint32_t n2 = aes_col(a, s2, s3, s0, s1, rk[4 * r + 2]);
    uint32_t n3 = aes_col(a, s3, s0, s1, s2, rk[4 * r + 3]);
    s0 = n0;
    s1 = n1;
    s2 = n2;
    s3 = n3;
  }
  blk o;
  o.x = aes_col_last(a, s0, s1, s2, s3, rk[40]);
  o.y = aes_col_last(a, s1, s2, s3, s0, rk[41]);
  o.z = aes_col_last(a, s2, s3, s0, s1, rk[42]);
  o.w = aes_col_last(a, s3, s0, s1, s2, rk[43]);
  return o;
}

// GGM two-key PRG: left = AES_k0(p) ^ p, right = AES_k1(p) ^ p.
// rk2: 88 words, key 0 schedule then key 1 schedule.
CUOT_DEV void ggm_expand(const AesLds& a, const uint32_t* __restrict__ rk2, blk p, blk& l, blk& r) {
  l = bxor(aes_enc(a, rk2, p), p);
  r = bxor(aes_enc(a, rk2 + 44, p), p);
}
