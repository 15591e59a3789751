// qc_fa.hip -- the quasi-cyclic encoder's product for 2^12 < n <= 2^24: an
// additive FFT over GF(2^32) on one point per Frobenius orbit.
//
//     y_i = x_i ^ XOR_{k < n} a_{(i-k) mod n} x_{n+k},   i < n
//
// (the same map as qc.hip; the reference's float cuFFT version is
// silent/quasi_cyclic.cu:118-128), for all 128 bit-rows at once.
//
// The operands have coefficients in GF(2), so their values at the 32 conjugates
// of a point of GF(2^32) are conjugates of each other: a product of 2^K
// coefficients is fixed by its values at 2^(K-5) points, one per orbit, 32 bits
// each.  Packing 16 coefficients per GF(2^32) element instead (qc.hip) spends
// twice the elements, half of every element being room for the chunk products.
// The idea is the Frobenius additive FFT of Li, Chen, Kuo, Cheng and Yang
// (ISSAC 2018); the points and the bitsliced form are chosen here:
//
//   points  beta_a + span{beta_i : i < c or c < i <= K-5},  c = min(K-5, 15),
//           a = 16 + c, on the Cantor basis of qc_fa.h.  Their images under
//           s_c are beta_16 + span{beta_1, ...}, of degree 32 and pairwise not
//           conjugate for K <= 27, so the orbits are full and distinct.
//   layers  index bit k of a polynomial in the novel basis is evaluated with
//           s_k(point) = beta_{a-k} + C(bits above k), C(g) = sum g_b beta_{b+1}:
//     k = K-2 .. K-4   the same constant at every point: eight coefficients
//                      become one GF(2^16) value (a fixed 16 x 8 map; 16 x 16
//                      for the full product's four bits)
//     k = K-5 .. c+1   butterflies over GF(2^16) (K > 20)
//     k = c            the constant has a theta part of 1 and no free bit: two
//                      GF(2^16) values u, v become u + delta v + theta v
//     k = c-1 .. 0     butterflies over GF(2^32)
//
// Encode (per party), blocks x_{n+i} being coefficient i of all 128 rows:
//   128-row bit transpose, novel-basis conversion of every row string in LDS
//   (conv_fast.h), transpose back (for K > 21 the strings are the 2^16
//   coefficients of an expansion in powers of s_16, made on the blocks before
//   that, and the first pass converts across the strings); for K > 20 a pass of
//   the GF(2^16) layers, halves of the elements apart; a pass of up to seven
//   GF(2^32) layers; one of the lowest eight, the product by A^ and the inverse
//   of the eight; the mirror image back; y.
// Between passes the data is element major: element e is 32 planes x 16 bytes
// in one run, so that every tile reads and writes whole lines.
#include <string.h>

#include "conv_fast.h"
#include "kernels.h"
#include "qc_fa.h"
#include "transpose32.h"

namespace {

__constant__ uint2 c_fa_beta[32];  // beta_i and nu times its theta part
__constant__ uint32_t c_fa_pack[FA_KC_MAX + 1][8];

constexpr int FA_KMIN = 14, FA_KMAX = 25;
constexpr int FA_STR = 20;  // longest row string converted in LDS (128 KB, 144 KB padded)

CUOT_DEV uint4 x4(uint4 a, uint4 b) { return make_uint4(a.x ^ b.x, a.y ^ b.y, a.z ^ b.z, a.w ^ b.w); }
CUOT_DEV uint4 z4() { return make_uint4(0, 0, 0, 0); }

// ---- twiddles -----------------------------------------------------------------
// C(g) and nu times its theta part from three 256-entry tables of the low 24 bits of g
constexpr int FA_CTAB = 3 * 256;

CUOT_DEV uint2 x2(uint2 a, uint2 b) { return make_uint2(a.x ^ b.x, a.y ^ b.y); }

CUOT_DEV void fa_ctab_fill(uint2* tab, int tid, int nth) {
  for (int i = tid; i < FA_CTAB; i += nth) {
    const int q = i >> 8, v = i & 255;
    uint2 c = make_uint2(0, 0);
    for (int b = 0; b < 8; b++)
      if ((v >> b) & 1) c = x2(c, c_fa_beta[8 * q + b + 1]);
    tab[i] = c;
  }
}

CUOT_DEV uint2 fa_ctab(const uint2* tab, uint32_t g) {
  return x2(x2(tab[g & 255], tab[256 + ((g >> 8) & 255)]), tab[512 + ((g >> 16) & 255)]);
}

// ---- GF(2^16) layers (K > 20) -------------------------------------------------------
enum { FA_FWD = 0, FA_INV = 1, FA_FUSED = 2 };

struct FaArgs {
  const uint4* nat_in;  // natural order coefficients (first pass)
  uint4* nat_out;       // natural order coefficients (last inverse pass)
  uint4* E;             // element-major data
  const uint32_t* ahat;
  const uint32_t* const* ahats;  // per-instance A^ (batch) or NULL
  int64_t XS;                    // instance stride of all three buffers in blocks
  int K, c, a;
  int lo, R;     // layers of element bits lo .. lo + R - 1
  int contract;  // the layer k = c before the forward or after the inverse layers
};

constexpr int FA_TL = 8;    // log2 elements of a tile
constexpr int FA_NT = 512;  // lanes

// First and last pass: the layers above c, KC of them, where the halves of the
// elements transform apart under GF(2^16) constants (blockIdx.z: the half).  LDS
// tile: 2^KC elements 2^c apart times 2^(8-KC) consecutive ones, 16 planes x 4
// words each and 4 words of padding; one (butterfly, word) per lane and layer.
constexpr int FA_ST16 = 68;

// LDS slot of tile element e: the butterflies of the lowest tile layers touch
// elements whose slots share their residue mod 8 (the element stride is 4 mod
// 64 banks); reflecting every odd group of eight spreads them
CUOT_DEV int fa_slot(int e) { return e ^ (((e >> 3) & 1) * 7); }

template <int KC, bool INV>
__device__ __forceinline__ void fa_layer16(const FaArgs& a, uint32_t* lds, const uint2* ctab, int s) {
  constexpr int LGC = FA_TL - KC, C = 1 << LGC;
  const int w = threadIdx.x & 3, cc = (threadIdx.x >> 2) & (C - 1), bp = (threadIdx.x >> 2) >> LGC;
  const int tu = ((bp >> s) << (s + 1)) | (bp & ((1 << s) - 1)), tv = tu | (1 << s);
  uint32_t* pu = lds + fa_slot(tu * C + cc) * FA_ST16 + w;
  uint32_t* pv = lds + fa_slot(tv * C + cc) * FA_ST16 + w;
  uint32_t xv[16], acc[16];
#pragma unroll
  for (int p = 0; p < 16; p++) {
    xv[p] = pv[4 * p];
    if (INV) pv[4 * p] = xv[p] ^= pu[4 * p];
  }
  // the first lane's constant for all, and what the others' g add to it: a
  // wavefront covers 16 neighbouring (butterfly, column) pairs, so at most the
  // low four bits of g differ
  const uint32_t g = (uint32_t)(tu >> (s + 1)), g0 = __builtin_amdgcn_readfirstlane(g), d = g ^ g0;
  fa_mulc16(xv, __builtin_amdgcn_readfirstlane(c_fa_beta[a.a - a.c - 1 - s].x ^ fa_ctab(ctab, g0).x), acc);
  if (__any(d != 0)) fa_add_low(xv, d, acc);
#pragma unroll
  for (int p = 0; p < 16; p++) {
    const uint32_t un = pu[4 * p] ^ acc[p];
    pu[4 * p] = un;
    if (!INV) pv[4 * p] = xv[p] ^ un;
  }
  __syncthreads();
}

// chunk maps on the staged tile: 8 coefficient planes -> 16 coordinates, and
// 16 coordinates -> 16 coefficient planes
template <int KC, bool UN>
__device__ __forceinline__ void fa_chunks(uint32_t* lds) {
  for (int tau = threadIdx.x; tau < 4 << FA_TL; tau += FA_NT) {
    uint32_t* pe = lds + fa_slot(tau >> 2) * FA_ST16 + (tau & 3);
    uint32_t in[16], out[16];
#pragma unroll
    for (int p = 0; p < (UN ? 16 : 8); p++) in[p] = pe[4 * p];
    if constexpr (UN)
      fa_unpack_planes<KC>(in, out);
    else
      fa_pack_planes<KC>(in, out);
#pragma unroll
    for (int p = 0; p < 16; p++) pe[4 * p] = out[p];
  }
  __syncthreads();
}

// Conversion of the coefficient rows of a half-mode tile between the s_16-adic
// and the novel basis: row rho (index bits 16 up) is a coefficient of X = s_16,
// whose subspace polynomials are s_k(X) = X^(2^k) + sum of X^e, e = 2^j for the
// proper submasks j of k (levels as in conv_bits.h, one row instead of one
// bit).  Row rho lies in plane rho >> r of element (rho mod 2^r) * C + column,
// r = KC.  The terms are compile-time constants: with runtime term lists the two
// passes took 1000 us more at n = 2^24, where this adds 170 and 250 us to theirs.
constexpr bool fa_is_term(int k, int j) { return j < k && (j & ~k) == 0; }
constexpr int fa_jmax(int k) {
  int m = 0;
  for (int j = 0; j < k; j++)
    if (fa_is_term(k, j)) m = j;
  return m;
}

template <int KC>
__device__ __forceinline__ uint4& fa_row(uint32_t* lds, int rho, int c) {
  return *(uint4*)&lds[fa_slot(((rho & ((1 << KC) - 1)) << (8 - KC)) + c) * FA_ST16 + 4 * (rho >> KC)];
}

// v ^= rows hb + s + half - e for the terms e = 2^J > s (FIX) or lb-side rows
// hb + s - e for e <= s
template <int KC, int K, bool FIX, int J = 0>
__device__ __forceinline__ void fa_row_terms(uint32_t* lds, uint4& v, int hb, int s, int c) {
  if constexpr (J < K) {
    if constexpr (fa_is_term(K, J)) {
      constexpr int e = 1 << J;
      if (FIX ? e > s : e <= s) v = x4(v, fa_row<KC>(lds, FIX ? hb + s + (1 << K) - e : hb + s - e, c));
    }
    fa_row_terms<KC, K, FIX, J + 1>(lds, v, hb, s, c);
  }
}

template <int KC, bool INV, int STEP = 1>
__device__ __forceinline__ void fa_outer(uint32_t* lds) {
  constexpr int NB = KC + (INV ? 4 : 3);  // row bits; level 0 has no lower terms
  if constexpr (STEP < NB) {
    constexpr int K = INV ? STEP : NB - STEP, half = 1 << K, LGC = 8 - KC, C = 1 << LGC, LGE = fa_jmax(K);
#pragma unroll
    for (int phase = 0; phase < 2; phase++) {
      if ((phase == 0) != INV) {
        constexpr int cnt = (1 << (NB - 1 - K)) << (LGE + LGC);  // hi rows i < e_max
        for (int x = threadIdx.x; x < cnt; x += FA_NT) {
          const int c = x & (C - 1), i = (x >> LGC) & ((1 << LGE) - 1), hb = ((x >> (LGC + LGE)) * 2 + 1) * half;
          uint4 v = fa_row<KC>(lds, hb + i, c);
          fa_row_terms<KC, K, true>(lds, v, hb, i, c);
          fa_row<KC>(lds, hb + i, c) = v;
        }
      } else {
        constexpr int cnt = 1 << (NB - 1 + LGC);
#pragma unroll 1
        for (int x = threadIdx.x; x < cnt; x += FA_NT) {
          const int c = x & (C - 1), lo = x >> LGC, j = lo & (half - 1), lb = (lo >> K) * 2 * half;
          uint4 v = fa_row<KC>(lds, lb + j, c);
          fa_row_terms<KC, K, false>(lds, v, lb + half, j, c);
          fa_row<KC>(lds, lb + j, c) = v;
        }
      }
      __syncthreads();
    }
    fa_outer<KC, INV, STEP + 1>(lds);
  }
}

// address of element e's coefficient q of half h in natural order
CUOT_DEV int64_t fa_nat(const FaArgs& a, int64_t e, int h, int q) {
  return ((int64_t)q << (a.K - 4)) | ((e >> a.c) << (a.c + 1)) | ((int64_t)h << a.c) | (e & (((int64_t)1 << a.c) - 1));
}

// staging addresses come from an opaque copy of the lane index, so that the
// compiler recomputes them per phase instead of holding them through the layers
__device__ __forceinline__ int opaque_tid() {
  int t = (int)threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

template <int KC, bool INV>
__global__ __launch_bounds__(FA_NT) __attribute__((amdgpu_waves_per_eu(4))) void fa_pass16(FaArgs a) {
  extern __shared__ uint32_t lds[];
  constexpr int LGC = FA_TL - KC, C = 1 << LGC, TC = 1 << FA_TL;
  const int64_t ioff = (int64_t)blockIdx.y * a.XS;
  uint4* E = a.E + ioff;
  const uint4* nin = a.nat_in + ioff;
  uint4* nout = a.nat_out + ioff;
  const int h = (int)blockIdx.z;
  const int64_t ntiles = ((int64_t)1 << (a.K - 5)) >> FA_TL;
  uint2* ctab = (uint2*)(lds + TC * FA_ST16);
  fa_ctab_fill(ctab, threadIdx.x, FA_NT);  // read after the first barrier
  // a tile's base is its first column: the 2^KC elements are all those 2^c apart
  auto elem = [&](int64_t tile, int el) { return (tile << LGC) + ((int64_t)(el >> LGC) << a.c) + (el & (C - 1)); };
  // staged word f: plane fastest in element-major data, element fastest in natural order
  uint4 v[8];
  auto load_tile = [&](int64_t tile) {
    const int tid = opaque_tid();
#pragma unroll
    for (int u = 0; u < (INV ? 8 : 4); u++) {
      const int f = tid + u * FA_NT;
      v[u] = z4();
      if constexpr (INV)
        v[u] = E[elem(tile, f >> 4) * 32 + 16 * h + (f & 15)];
      else
        v[u] = nin[fa_nat(a, elem(tile, f & (TC - 1)), h, f >> FA_TL)];
    }
  };
  // workgroups are dealt to the 8 XCDs in turn: one XCD's take neighbouring tiles
  const int64_t G = gridDim.x, bx = blockIdx.x;
  const int64_t slot = (G & 7) ? bx : (bx & 7) * (G >> 3) + (bx >> 3);
  if (slot < ntiles) load_tile(slot);
  for (int64_t tile = slot; tile < ntiles; tile += G) {
    int tid = opaque_tid();
#pragma unroll
    for (int u = 0; u < (INV ? 8 : 4); u++) {
      const int f = tid + u * FA_NT;
      *(uint4*)&lds[fa_slot(INV ? f >> 4 : f & (TC - 1)) * FA_ST16 + (INV ? f & 15 : f >> FA_TL) * 4] = v[u];
    }
    __syncthreads();
    if constexpr (!INV) {
      if constexpr (KC > 1) fa_outer<KC, false>(lds);
      fa_chunks<KC, false>(lds);
    }
    // one loop, so that the layer's code is there once
#pragma unroll 1
    for (int step = 0; step < KC; step++) fa_layer16<KC, INV>(a, lds, ctab, INV ? step : KC - 1 - step);
    if constexpr (INV) {
      fa_chunks<KC, true>(lds);
      if constexpr (KC > 1) fa_outer<KC, true>(lds);
    }
    uint4 w[8];
    tid = opaque_tid();
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int f = tid + u * FA_NT;
      w[u] = z4();
      w[u] = *(const uint4*)&lds[fa_slot(INV ? f & (TC - 1) : f >> 4) * FA_ST16 + (INV ? f >> FA_TL : f & 15) * 4];
    }
    // the next tile's loads are issued before this tile's stores
    if (tile + G < ntiles) load_tile(tile + G);
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const int f = tid + u * FA_NT;
      if constexpr (INV)
        nout[fa_nat(a, elem(tile, f & (TC - 1)), h, f >> FA_TL)] = w[u];
      else
        E[elem(tile, f >> 4) * 32 + 16 * h + (f & 15)] = w[u];
    }
    __syncthreads();
  }
}

// ---- GF(2^32) passes: layers k < c ------------------------------------------------
// A workgroup of 512 lanes holds a tile of 256 elements (2^R of them 2^lo apart
// times 2^lgC consecutive ones) in registers: lane P * 4 + w has word w of the
// two elements of butterfly P, all 32 planes of both.  Between layers a lane
// gives one of the two to the lane whose P differs in the next layer's bit and
// takes one: through LDS where that is another wavefront, by lane swaps inside
// one.  Held in LDS (128 elements a tile, 256 lanes at 250 registers, every layer
// reading and writing all of it), two wavefronts per SIMD waited half of the
// time; registers hold twice the tile at four wavefronts, and three passes do
// where five did.  At n = 2^24 the passes took 355 + 312 + 924 + 314 + 342 us, now
// 298 + 645 + 305; the middle one issues vector operations all the time, the
// others run at 3.6 TB/s.  Tiles of 128 elements (twice the workgroups where
// there are few) gain 3 to 4 % of an encode at n = 2^16 .. 2^17, 1 % at 2^18 and
// lose from there on: not worth the second set of kernels.
constexpr int FA_ST = 132;  // LDS words of a staged element: 32 planes x 4, 4 of padding

// give u (where this lane's P has bit b set) or v to the lane whose P differs in
// that bit and take the same from it
// (N lanes further; the quads of a row whose bit is set are the BANKS)
template <int N, int BANKS>
__device__ __forceinline__ void fa_swap_dpp(uint32_t* u, uint32_t* v) {
#pragma unroll
  for (int p = 0; p < 32; p++) {
    const int a = (int)u[p], b = (int)v[p];
    u[p] = (uint32_t)__builtin_amdgcn_update_dpp(a, b, 0x110 | N, 0xF, BANKS, false);       // row_shr
    v[p] = (uint32_t)__builtin_amdgcn_update_dpp(b, a, 0x100 | N, 0xF, 0xF ^ BANKS, false);  // row_shl
  }
}

__device__ __forceinline__ void fa_swap_lds(uint32_t* lds, uint32_t* g, int other) {
#pragma unroll
  for (int p = 0; p < 32; p++) lds[p * FA_NT + threadIdx.x] = g[p];
  __syncthreads();
#pragma unroll
  for (int p = 0; p < 32; p++) g[p] = lds[p * FA_NT + other];
  __syncthreads();
}

__device__ __forceinline__ void fa_swap(uint32_t* lds, uint32_t* u, uint32_t* v, int P, int b) {
  // (b opaque in between: as one chain of choices the compiler merges all ways
  // behind 64 moves)
#define FA_OPAQUE(x) \
  x = __builtin_amdgcn_readfirstlane(x); \
  asm volatile("" : "+s"(x))
  if (b >= 4) {  // another wavefront; the bit is this one's
    const int other = (int)threadIdx.x ^ (4 << b);
    int bit = __builtin_amdgcn_readfirstlane(P >> b) & 1;
    if (bit) fa_swap_lds(lds, u, other);
    FA_OPAQUE(bit);
    if (!bit) fa_swap_lds(lds, v, other);
  }
  FA_OPAQUE(b);
  if (b == 3) {
#pragma unroll
    for (int p = 0; p < 32; p++) {
      const auto r = __builtin_amdgcn_permlane32_swap(u[p], v[p], false, false);
      u[p] = r[0];
      v[p] = r[1];
    }
  }
  FA_OPAQUE(b);
  if (b == 2) {
#pragma unroll
    for (int p = 0; p < 32; p++) {
      const auto r = __builtin_amdgcn_permlane16_swap(u[p], v[p], false, false);
      u[p] = r[0];
      v[p] = r[1];
    }
  }
  FA_OPAQUE(b);
  if (b == 1) fa_swap_dpp<8, 0xC>(u, v);
  FA_OPAQUE(b);
  if (b == 0) fa_swap_dpp<4, 0xA>(u, v);
}

CUOT_DEV int fa_insert(int P, int b, int r) { return ((P >> b) << (b + 1)) | (r << b) | (P & ((1 << b) - 1)); }

template <int MODE, bool NAT>
__global__ __launch_bounds__(FA_NT) __attribute__((amdgpu_waves_per_eu(4))) void fa_pass32(FaArgs a) {
  extern __shared__ uint32_t lds[];
  constexpr int TL = FA_TL, NT = FA_NT, NH = 1 << (TL - 1);  // NH: elements of half a tile
  const int64_t ioff = (int64_t)blockIdx.y * a.XS;
  uint4* E = a.E + ioff;
  const uint4* nin = a.nat_in + ioff;
  uint4* nout = a.nat_out + ioff;
  const uint32_t* ahat = a.ahats ? a.ahats[blockIdx.y] : a.ahat;
  const int tid = threadIdx.x, w = tid & 3, P = tid >> 2;
  const int lgC = TL - a.R, C = 1 << lgC;
  const int64_t cblocks = ((int64_t)1 << a.lo) >> lgC;
  const int64_t ntiles = ((int64_t)1 << (a.K - 5)) >> TL;
  uint2* ctab = (uint2*)(lds + NH * FA_ST);
  fa_ctab_fill(ctab, tid, NT);  // read after the first barrier
  // the register bit of the tile index when the tile is read and written
  const int rin = MODE == FA_INV ? lgC : TL - 1, rout = MODE == FA_FWD ? lgC : TL - 1;
  const int64_t G = gridDim.x, bx = blockIdx.x;
  // workgroups are dealt to the 8 XCDs in turn: one XCD's take neighbouring tiles
  const int64_t slot = (G & 7) ? bx : (bx & 7) * (G >> 3) + (bx >> 3);
  for (int64_t tile = slot; tile < ntiles; tile += G) {
    const int64_t eb = ((tile >> (a.lo - lgC)) << (a.lo + a.R)) | ((tile & (cblocks - 1)) << lgC);
    // Addresses are sums over the bits of the index: a part of the lane's bits (32
    // bits of it) and a scalar one, both per half of the tile (register bit r).
    auto off = [&](int i) { return ((uint32_t)(i >> lgC) << a.lo) | (uint32_t)(i & (C - 1)); };
    uint32_t u[32], v[32];
    // the tile's two halves, NH elements each, through LDS
    uint4 st[8];
    constexpr bool NIN = NAT && MODE == FA_FWD, NOUT = NAT && MODE == FA_INV;
    // natural order, word f = tid + NT k: element fastest, then coefficient (QB
    // bits) and half; else plane fastest, then element
    auto addr = [&](uint4* p, bool nat, int QB, int reg, int r, int tid, int k) {
      const int fh = nat ? 4 * k : (NT >> 5) * k, fl = nat ? tid >> (TL - 1) : tid >> 5;  // the index above the fastest part
      int64_t sc;
      uint32_t ln;
      if (nat) {
        auto hq = [&](int x) { return (uint32_t)(x & ((1 << QB) - 1)) << (a.K - 4) | (uint32_t)(x >> QB) << a.c; };
        sc = eb + off(r << reg) + hq(fh);
        ln = off(fa_insert(tid & (NH - 1), reg, 0)) + hq(fl);
      } else {
        sc = (eb + off(fa_insert(fh, reg, r))) * 32;
        ln = off(fa_insert(fl, reg, 0)) * 32 + (tid & 31);
      }
      return (uint4*)((char*)(p + sc) + (size_t)(ln * 16));
    };
    auto fetch = [&](int r) {
      const int tid = opaque_tid();
#pragma unroll
      for (int k = 0; k < (NIN ? 4 : 8); k++) {
        st[k] = z4();
        st[k] = *addr(NIN ? (uint4*)nin : E, NIN, 3, rin, r, tid, k);
      }
    };
    auto take = [&]() {
      const int tid = opaque_tid();
#pragma unroll
      for (int k = 0; k < (NIN ? 4 : 8); k++) {
        const int f = tid + k * NT;
        if constexpr (NIN)
          *(uint4*)&lds[(f & (NH - 1)) * FA_ST + (f >> (TL + 2)) * 64 + ((f >> (TL - 1)) & 7) * 4] = st[k];
        else
          *(uint4*)&lds[(f >> 5) * FA_ST + (f & 31) * 4] = st[k];
      }
    };
    auto read = [&](uint32_t* x) {
      if constexpr (NIN) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
          uint32_t t[8];
#pragma unroll
          for (int q = 0; q < 8; q++) t[q] = lds[P * FA_ST + h * 64 + q * 4 + w];
          fa_pack_planes<0>(t, x + 16 * h);
        }
      } else {
#pragma unroll
        for (int p = 0; p < 32; p++) x[p] = lds[P * FA_ST + p * 4 + w];
      }
    };
    fetch(0);
    take();
    __syncthreads();
    fetch(1);
    read(u);
    __syncthreads();
    take();
    __syncthreads();
    read(v);
    __syncthreads();
    uint2 ac = make_uint2(0, 0), an = make_uint2(0, 0);
    if constexpr (MODE == FA_FUSED) {
      ac = *(const uint2*)&ahat[eb + 2 * P];
      an = *(const uint2*)&ahat[((int64_t)1 << (a.K - 5)) + eb + 2 * P];
    }
    // layer k = c: half 0 ^= delta * half 1, delta = C(bits above c), one constant
    // for the tile (its own inverse)
    auto contract = [&]() {
      const uint32_t delta = __builtin_amdgcn_readfirstlane(fa_ctab(ctab, (uint32_t)(eb >> a.c)).x);
      uint32_t t[16];
      fa_mulc16(u + 16, delta, t);
#pragma unroll
      for (int p = 0; p < 16; p++) u[p] ^= t[p];
      fa_mulc16(v + 16, delta, t);
#pragma unroll
      for (int p = 0; p < 16; p++) v[p] ^= t[p];
    };
    if (MODE == FA_FWD && a.contract) contract();
    const int layers = TL - lgC;
    // forward from tile bit 7 down to lgC, then back up; one loop, so that the
    // layer's code is there once
    for (int step = 0; step < (MODE == FA_FUSED ? 2 * layers : layers); step++) {
      const bool inv = MODE == FA_INV || (MODE == FA_FUSED && step >= layers);
      const int up = MODE == FA_FUSED ? step - layers : step;
      const int b = inv ? lgC + up : TL - 1 - step;
      int sw = step == 0 ? -1 : inv ? b - 1 : b;  // the bit of P to swap with
      if constexpr (MODE == FA_FUSED) {
        if (step == layers) {
          sw = -1;
          asm volatile("" : "+v"(ac.x), "+v"(ac.y), "+v"(an.x), "+v"(an.y));  // their 96 masks stay in here
          fa_mulv32(u, ac.x, an.x);
          __builtin_amdgcn_sched_barrier(0);
          fa_mulv32(v, ac.y, an.y);
        }
      }
      FA_OPAQUE(sw);
      fa_swap(lds, u, v, P, sw);
      const int k = a.lo + b - lgC;
      const uint32_t e = (uint32_t)eb + off(fa_insert(P, b, 0));
      const uint32_t g = ((e >> a.c) << (a.c - k)) | ((e & ((1u << a.c) - 1)) >> (k + 1));
      // the first lane's constant for all, and what the others' g add to it: a
      // wavefront covers 16 neighbouring P, so at most the low four bits differ
      const uint32_t g0 = __builtin_amdgcn_readfirstlane(g), d = g ^ g0;
      const uint2 c = x2(c_fa_beta[a.a - k], fa_ctab(ctab, g0));
      // (fused: by a mask, as a branch costs moves of both)
      auto add_u = [&](bool now) {
        if constexpr (MODE == FA_FUSED) {
#pragma unroll
          for (int p = 0; p < 32; p++) asm("v_bitop3_b32 %0, %0, %1, %2 bitop3:0x78" : "+v"(v[p]) : "v"(u[p]), "s"(0 - (int)now));
        } else if (now) {
#pragma unroll
          for (int p = 0; p < 32; p++) v[p] ^= u[p];
        }
      };
      add_u(inv);
      fa_add_mul32(u, v, __builtin_amdgcn_readfirstlane(c.x), __builtin_amdgcn_readfirstlane(c.y));
      if (__any(d != 0)) {
        fa_add_low(v, d, u);
        fa_add_low(v + 16, d, u + 16);
      }
      add_u(!inv);
    }
    if (MODE == FA_INV && a.contract) contract();
    auto put = [&](const uint32_t* x) {
      if constexpr (NOUT) {
#pragma unroll
        for (int h = 0; h < 2; h++) {
          uint32_t t[16];
          fa_unpack_planes<0>(x + 16 * h, t);
#pragma unroll
          for (int q = 0; q < 16; q++) lds[P * FA_ST + h * 64 + q * 4 + w] = t[q];
        }
      } else {
#pragma unroll
        for (int p = 0; p < 32; p++) lds[P * FA_ST + p * 4 + w] = x[p];
      }
    };
    auto store = [&](int r) {
      const int tid = opaque_tid();
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const int f = tid + k * NT;
        *addr(NOUT ? nout : E, NOUT, 4, rout, r, tid, k) =
            *(const uint4*)&lds[NOUT ? (f & (NH - 1)) * FA_ST + (f >> (TL + 3)) * 64 + ((f >> (TL - 1)) & 15) * 4
                                     : (f >> 5) * FA_ST + (f & 31) * 4];
      }
    };
    __syncthreads();
    put(u);
    __syncthreads();
    store(0);
    __syncthreads();
    put(v);
    __syncthreads();
    store(1);
    __syncthreads();
  }
}

// ---- s_16-adic levels on blocks (K > 21) ------------------------------------------
// Expansion of a polynomial in powers of s_16 = x^65536 + x: s_16^(2^i) has one
// lower term, so the level of index bit b = 16 + i takes, with half = 2^b and
// e = 2^i, q = hi with its first e coefficients corrected by its last ones, and
// lo_j ^= q_{j-e} (backwards the same with the two steps exchanged).  Away from
// the first coefficients of a half all levels are their own inverses, commute
// and move coefficient j of a row 2^b further to j + e of this one, so R of them
// are one pass over skewed columns (below), bound by memory: 2^24 coefficients
// 16 bytes wide in 102 us (5.26 TB/s).  At n = 2^24 the forward levels take 207
// us and the backward ones with the output 490.  The novel basis' own levels
// (s_23 has 15 lower terms) one pass each took 934 and 1510 with the same
// output, the s_16-adic ones as a gather of (3/2)^R reads per output 310 and 1000.
// At K = 21 a single level of three terms is left, done in the output: 388 us an
// encode of n = 2^20 against 413 this way.
// The source: an instance's natural-order buffer, or x_{n+i}, zero from n on.
struct FaSrc {
  const uint4* p;
  int64_t n;
  __device__ __forceinline__ uint4 operator[](int64_t i) const { return i < n ? p[i] : make_uint4(0, 0, 0, 0); }
};

// exact value of index I after the levels of bits b0 .. b (backwards) or
// b .. b0 + R - 1 (forwards); only near the start of a half
template <bool INV, int L>
__device__ __attribute__((noinline)) uint4 fa_s16_slow(const FaSrc& in, int64_t I, int b0, int R) {
  if constexpr (L == 0) {
    return in[I];
  } else {
    const int b = INV ? b0 + L - 1 : b0 + R - L;
    const int64_t half = (int64_t)1 << b, e = half >> 16;
    const int64_t pos = I & (2 * half - 1), hi = I - pos + half;
    uint4 v = fa_s16_slow<INV, L - 1>(in, I, b0, R);
    if (pos < half) {
      if (pos >= e) {
        const int64_t s = pos - e;
        v = x4(v, fa_s16_slow<INV, L - 1>(in, hi + s, b0, R));
        if (!INV && s < e) v = x4(v, fa_s16_slow<INV, L - 1>(in, hi + s + half - e, b0, R));
      }
    } else if (pos - half < e) {
      v = x4(v, fa_s16_slow<INV, L - 1>(in, I + half - e, b0, R));
    }
    return v;
  }
}

// the first 2 * (sum of the shifts) coefficients above bit b0 take the exact form
constexpr int64_t fa_s16_edge(int R, int b0) { return (int64_t)2 << (R + b0 - 16); }

// Skewed column c of the 2^R rows of 2^b0 coefficients at base: coefficient
// c - T 2^(b0-16) of row T.  The levels stay inside a column, where they are a
// butterfly of R stages, so every coefficient is read and written once.  Rows
// whose coefficient lies below the exact ones or past the row are not valid
// (and no valid one takes them in).  Rows below FROM are left out.
template <int R, int FROM = 0>
__device__ __forceinline__ void fa_s16_column(const FaSrc& in, int64_t base, int64_t c, int b0, uint4 (&v)[1 << R]) {
#pragma unroll
  for (int T = FROM; T < (1 << R); T++) {
    const int64_t j = c - ((int64_t)T << (b0 - 16));
    v[T] = j >= 0 && j < ((int64_t)1 << b0) ? in[base + ((int64_t)T << b0) + j] : make_uint4(0, 0, 0, 0);
  }
#pragma unroll
  for (int b = 0; b < R; b++)
#pragma unroll
    for (int T = FROM; T < (1 << R); T++)
      if (!(T >> b & 1)) v[T] = x4(v[T], v[T | 1 << b]);
}

// columns from the first valid coefficient of row 0 to the last one of row 2^R - 1
constexpr int64_t fa_s16_columns(int R, int b0) {
  return ((int64_t)1 << b0) - fa_s16_edge(R, b0) + ((((int64_t)1 << R) - 1) << (b0 - 16));
}

// Bits B0 .. B0 + R - 1 of N coefficients, a column per lane.  The rows' first
// coefficients, whose exact form is a long chain of dependent reads, go to
// workgroups of their own, one per lane.
template <bool INV, bool SRC, int R, int B0>
__global__ __launch_bounds__(256) void fa_s16_level(const QcIo* __restrict__ io, QcIo io1, const uint4* __restrict__ in,
                                                    uint4* __restrict__ out, int64_t XS, int64_t N) {
  FaSrc src;
  if (SRC) {
    const QcIo q = io ? io[blockIdx.y] : io1;
    src.p = q.x + q.n;
    src.n = q.n;
  } else {
    src.p = in + (int64_t)blockIdx.y * XS;
    src.n = N;
  }
  uint4* dst = out + (int64_t)blockIdx.y * XS;
  const int tid = threadIdx.x;
  constexpr int64_t EDGE = fa_s16_edge(R, B0);
  const int64_t edges = (N >> B0) * EDGE, nedge = (edges + 255) / 256;
  if ((int64_t)blockIdx.x < nedge) {
    const int64_t x = (int64_t)blockIdx.x * 256 + tid;
    if (x >= edges) return;
    const int64_t i = ((x / EDGE) << B0) | (x & (EDGE - 1));
    dst[i] = fa_s16_slow<INV, R>(src, i, B0, R);
    return;
  }
  constexpr int64_t per = (fa_s16_columns(R, B0) + 255) / 256;  // workgroups per 2^R rows
  const int64_t tile = (int64_t)blockIdx.x - nedge;
  const int64_t c = EDGE + (tile % per) * 256 + tid, base = (tile / per) << (B0 + R);
  uint4 v[1 << R];
  fa_s16_column<R>(src, base, c, B0, v);
#pragma unroll
  for (int T = 0; T < (1 << R); T++) {
    const int64_t j = c - ((int64_t)T << (B0 - 16));
    if (j >= EDGE && j < ((int64_t)1 << B0)) dst[base + ((int64_t)T << B0) + j] = v[T];
  }
}

// ---- input: blocks to 128 bit-row strings of S = 2^mp bits ---------------------------
// SRC: from x_{n+i}
template <bool SRC>
__global__ __launch_bounds__(256) void fa_rows_in(const QcIo* __restrict__ io, QcIo io1, const uint4* __restrict__ in,
                                                  int64_t XS, int64_t N, int mp, uint32_t* __restrict__ rows) {
  __shared__ uint32_t sm[128][33];
  FaSrc src;
  if (SRC) {
    const QcIo q = io ? io[blockIdx.y] : io1;
    src.p = q.x + q.n;
    src.n = q.n;
  } else {
    src.p = in + (int64_t)blockIdx.y * XS;
    src.n = N;
  }
  rows += (int64_t)blockIdx.y * XS * 4;
  const int lane = threadIdx.x & 31;
  const int grp = threadIdx.x >> 5;
  const int64_t rw = (int64_t)1 << (mp - 5);  // words per row string
  // tiles of 1024 blocks (32 words of every row)
  for (int64_t tile = blockIdx.x; tile < (N >> 10); tile += gridDim.x) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int tl = grp * 4 + r;
      const int64_t i = (tile << 10) + tl * 32 + lane;
      const uint4 v = src[i];
      sm[0 * 32 + lane][tl] = cuot_transpose32(v.x, lane);
      sm[1 * 32 + lane][tl] = cuot_transpose32(v.y, lane);
      sm[2 * 32 + lane][tl] = cuot_transpose32(v.z, lane);
      sm[3 * 32 + lane][tl] = cuot_transpose32(v.w, lane);
    }
    __syncthreads();
    const int64_t str = (tile << 10) >> mp, w0 = ((tile << 10) & (((int64_t)1 << mp) - 1)) >> 5;
    uint32_t* dst = rows + str * 128 * rw + w0;
    for (int f = threadIdx.x; f < 128 * 8; f += 256) {
      const int k = f >> 3, tl = (f & 7) * 4;
      *(uint4*)&dst[(int64_t)k * rw + tl] = make_uint4(sm[k][tl], sm[k][tl + 1], sm[k][tl + 2], sm[k][tl + 3]);
    }
    __syncthreads();
  }
}

// ---- output -------------------------------------------------------------------------
// y_i = x_i ^ H_i ^ H_{i+n}, H the product's coefficients.  TOP (K = 21): its two
// halves go through the last level on the way, s_20 = x^(2^20) + x^65536 + x^16 + x.
template <bool TOP>
__global__ __launch_bounds__(256) void fa_output(const uint4* __restrict__ H, int64_t XS, const QcIo* __restrict__ io,
                                                 QcIo io1) {
  const QcIo q = io ? io[blockIdx.y] : io1;
  H += (int64_t)blockIdx.y * XS;
  auto h_at = [&](int64_t i) {
    uint4 v = H[i];
    if constexpr (TOP) {
      constexpr int64_t half = (int64_t)1 << 20;
#pragma unroll
      for (int e = 1; e <= 65536; e = e == 1 ? 16 : e * 4096) {
        if (i < half ? i >= e : i - half < e) v = x4(v, H[i < half ? half + i - e : i + half - e]);
      }
    }
    return v;
  };
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < q.n; i += (int64_t)gridDim.x * 256)
    q.y[i] = x4(q.x[i], x4(h_at(i), h_at(i + q.n)));
}

// The same through the last levels, bits 20 .. K-1 (R of them).  With n = m 2^20
// + r, the coefficients i + n of one skewed column's i are again one column, r +
// 16 m further, m rows up, or one row more and 2^20 back where j + r passes the
// row's end.  That column goes through LDS, as m is no constant.  i or i + n at
// a row's start: lanes of their own, 2 EDGE per row of y.
constexpr int FA_OT = 128;

template <int R>
__global__ __launch_bounds__(FA_OT) void fa_output_s16(const uint4* __restrict__ H, int64_t XS,
                                                       const QcIo* __restrict__ io, QcIo io1) {
  constexpr int B0 = 20, LOW = 1 << (R - 2);  // n > 2^(K-2)
  constexpr int64_t EDGE = fa_s16_edge(R, B0), ROW = (int64_t)1 << B0;
  __shared__ uint4 second[((1 << R) - LOW) * FA_OT];
  const QcIo q = io ? io[blockIdx.y] : io1;
  FaSrc src;
  src.p = H + (int64_t)blockIdx.y * XS;
  src.n = XS;
  const int64_t m = q.n >> B0, r = q.n & (ROW - 1), rows = (q.n + ROW - 1) >> B0;
  const int64_t nedge = rows * 2 * EDGE / FA_OT;
  if ((int64_t)blockIdx.x < nedge) {
    const int64_t x = (int64_t)blockIdx.x * FA_OT + threadIdx.x, k = x & (EDGE - 1);
    const int64_t j = x & EDGE ? (k - r) & (ROW - 1) : k, i = (x / (2 * EDGE)) << B0 | j;
    if (i >= q.n || ((x & EDGE) && j < EDGE)) return;
    uint4 v = q.x[i];
#pragma unroll 1
    for (int s = 0; s < 2; s++) v = x4(v, fa_s16_slow<true, R>(src, s ? i + q.n : i, B0, R));
    q.y[i] = v;
    return;
  }
  const int64_t c = EDGE + ((int64_t)blockIdx.x - nedge) * FA_OT + threadIdx.x;
  if (c - 16 * (rows - 1) >= ROW) return;
  const bool carry = c - 16 * (rows - 1) + r >= ROW;
  const int up = (int)m + (carry ? 1 : 0);
  {
    uint4 v[1 << R];
    fa_s16_column<R, LOW>(src, 0, c + r + 16 * m + (carry ? 16 - ROW : 0), B0, v);
#pragma unroll
    for (int T = LOW; T < (1 << R); T++) second[(T - LOW) * FA_OT + threadIdx.x] = v[T];
  }
  uint4 v[1 << R];
  fa_s16_column<R>(src, 0, c, B0, v);
#pragma unroll
  for (int T = 0; T <= (1 << (R - 1)); T++) {
    const int64_t j = c - 16 * T, i = (int64_t)T << B0 | j;
    if (T < rows && j >= EDGE && j < ROW && ((j + r) & (ROW - 1)) >= EDGE && i < q.n)
      q.y[i] = x4(q.x[i], x4(v[T], second[(T + up - LOW) * FA_OT + threadIdx.x]));
  }
}

CUOT_DEV int fa_terms(int k, uint32_t* e) {
  int c = 0;
  for (int j = 0; j < k; j++)
    if ((j & ~k) == 0) e[c++] = 1u << j;
  return c;
}

// ---- A^: the scalar transform of the single polynomial a ------------------------------
// One 32-bit word per point.  The words behind A^ (a word per point again) hold
// a's bits while they are converted and nu times the values' theta parts in the end.
__global__ __launch_bounds__(256) void fa_prep_bits(const QcPrep* __restrict__ pr, QcPrep pr1, int K) {
  const QcPrep q = pr ? pr[blockIdx.y] : pr1;
  uint32_t* T = q.ahat + ((int64_t)1 << (K - 5));
  const int64_t nb = (q.n + 7) / 8;
  for (int64_t w = (int64_t)blockIdx.x * 256 + threadIdx.x; w < ((int64_t)1 << (K - 6)); w += (int64_t)gridDim.x * 256) {
    uint32_t v = 0;
#pragma unroll
    for (int b = 0; b < 4; b++)
      if (4 * w + b < nb) v |= (uint32_t)q.a_bits[4 * w + b] << (8 * b);
    const int64_t left = q.n - 32 * w;
    if (left <= 0)
      v = 0;
    else if (left < 32)
      v &= (1u << left) - 1u;
    T[w] = v;
  }
}

// forward conversion level k >= 20 on a's bit string, out of place (from the
// first or second half of the words behind A^ to the other)
__global__ __launch_bounds__(256) void fa_prep_level(const QcPrep* __restrict__ pr, QcPrep pr1, int K, int k, int src) {
  const QcPrep q = pr ? pr[blockIdx.y] : pr1;
  const int64_t NW = (int64_t)1 << (K - 6);
  const uint32_t* in = q.ahat + ((int64_t)1 << (K - 5)) + (src ? NW : 0);
  uint32_t* out = q.ahat + ((int64_t)1 << (K - 5)) + (src ? 0 : NW);
  uint32_t e[16];
  const int ne = fa_terms(k, e);
  const int64_t hw = (int64_t)1 << (k - 5);  // words per half
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < NW; i += (int64_t)gridDim.x * 256) {
    const int64_t pos = i & (2 * hw - 1);
    const uint32_t* hi = in + (i - pos) + hw;
    // word s of the quotient's half: hi with its first e_max bits corrected
    auto quot = [&](int64_t s) {
      uint32_t v = hi[s];
      for (int r = 0; r < ne; r++) {
        const int64_t ew = e[r] >> 5;
        if (e[r] >= 32) {
          if (s < ew) v ^= hi[s + hw - ew];
        } else if (s == 0) {
          v ^= hi[hw - 1] >> (32 - e[r]);
        }
      }
      return v;
    };
    uint32_t v;
    if (pos >= hw) {
      v = quot(pos - hw);
    } else {
      v = in[i];
      for (int t = 0; t < ne; t++) {
        const int64_t ew = e[t] >> 5;
        const int sh = (int)(e[t] & 31);
        if (pos < ew) continue;
        const uint32_t x = quot(pos - ew);
        if (sh == 0)
          v ^= x;
        else
          v ^= (x << sh) | (pos - ew >= 1 ? quot(pos - ew - 1) >> (32 - sh) : 0u);
      }
    }
    out[i] = v;
  }
}

struct FaSync {
  __device__ void operator()() const { __syncthreads(); }
};

// levels below 2^mp on each string of 2^mp bits, in place (one workgroup each)
__global__ __launch_bounds__(1024) void fa_prep_rows(const QcPrep* __restrict__ pr, QcPrep pr1, int K, int mp, int src) {
  extern __shared__ uint32_t sw[];
  const QcPrep q = pr ? pr[blockIdx.y] : pr1;
  const int64_t nw = (int64_t)1 << (mp - 5);
  uint32_t* g = q.ahat + ((int64_t)1 << (K - 5)) + (src ? (int64_t)1 << (K - 6) : 0) + (int64_t)blockIdx.x * nw;
  for (int64_t i = threadIdx.x; i < nw; i += 1024) sw[cbp_at<true>(i)] = g[i];
  __syncthreads();
  cbp_convert<true, false>(sw, 0, mp, threadIdx.x, 1024, FaSync());
  for (int64_t i = threadIdx.x; i < nw; i += 1024) g[i] = sw[cbp_at<true>(i)];
}

constexpr int FA_PT = 10;  // log2 words of a preparation tile

// Element bits lo .. lo + R - 1 on tiles of 2^R words 2^lo apart times 2^lgC
// consecutive ones; the first tile pass takes the words from a's converted bits.
__global__ __launch_bounds__(512) void fa_prep_fft(const QcPrep* __restrict__ pr, QcPrep pr1, int K, int c, int aidx,
                                                   int lo, int R, int lgC, int first, int src) {
  __shared__ uint32_t L[1 << FA_PT];
  __shared__ uint2 ctab[FA_CTAB];
  const QcPrep q = pr ? pr[blockIdx.y] : pr1;
  uint32_t* A = q.ahat;
  const int nt = blockDim.x;
  fa_ctab_fill(ctab, threadIdx.x, nt);
  const int C = 1 << lgC, TW = 1 << (R + lgC);
  const int64_t tile = blockIdx.x;
  const int64_t cb = tile & ((((int64_t)1 << lo) >> lgC) - 1), hib = tile >> (lo - lgC);
  auto eidx = [&](int i) { return (hib << (lo + R)) | ((int64_t)(i >> lgC) << lo) | (cb * C + (i & (C - 1))); };
  if (first) {
    const uint32_t* T = A + ((int64_t)1 << (K - 5)) + (src ? (int64_t)1 << (K - 6) : 0);
    const uint32_t* pk = c_fa_pack[K <= 20 ? 0 : K - 20];
    for (int i = threadIdx.x; i < TW; i += nt) {
      const int64_t e = eidx(i);
      uint32_t v = 0;
      for (int h = 0; h < 2; h++) {
        const int64_t idx = ((e >> c) << (c + 1)) | ((int64_t)h << c) | (e & (((int64_t)1 << c) - 1));
        uint32_t x = 0;
        for (int b = 0; b < 8; b++) {
          const int64_t ci = ((int64_t)b << (K - 4)) | idx;
          if ((T[ci >> 5] >> (ci & 31)) & 1u) x ^= pk[b];
        }
        v |= x << (16 * h);
      }
      L[i] = v;
    }
  } else {
    for (int i = threadIdx.x; i < TW; i += nt) L[i] = A[eidx(i)];
  }
  __syncthreads();
  for (int s = R - 1; s >= 0; s--) {
    const int b = lo + s;  // element bit
    if (b == c - 1 && K - 5 > c) {
      // layer k = c between the two kinds: half 0 ^= C(bits above) * half 1
      for (int i = threadIdx.x; i < TW; i += nt) {
        const uint32_t x = L[i];
        L[i] = x ^ fa_mul16_dev(x >> 16, fa_ctab(ctab, (uint32_t)(eidx(i) >> c)).x);
      }
      __syncthreads();
    }
    const int k = b >= c ? b + 1 : b;
    const uint2 off = c_fa_beta[aidx - k];
    for (int t = threadIdx.x; t < (TW >> 1); t += nt) {
      const int cc = t & (C - 1), bp = t >> lgC;
      const int tu = ((bp >> s) << (s + 1)) | (bp & ((1 << s) - 1));
      const int u = tu * C + cc, v = u + (C << s);
      const uint32_t e = (uint32_t)eidx(u);
      const uint32_t xv = L[v];
      uint32_t xu = L[u];
      if (b >= c) {
        const uint32_t cst = off.x ^ fa_ctab(ctab, e >> (b + 1)).x;
        xu ^= fa_mul16_dev(xv & 0xffffu, cst) | (fa_mul16_dev(xv >> 16, cst) << 16);
      } else {
        const uint32_t g = ((e >> c) << (c - k)) | ((e & ((1u << c) - 1)) >> (k + 1));
        const uint2 cst = x2(off, fa_ctab(ctab, g));
        xu ^= fa_mul32_dev(xv, cst.x, cst.y);
      }
      L[u] = xu;
      L[v] = xv ^ xu;
    }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < TW; i += nt) {
    const int64_t e = eidx(i);
    A[e] = L[i];
    if (lo == 0) A[((int64_t)1 << (K - 5)) + e] = fa_mul16_dev(L[i] >> 16, FA_NU);
  }
}

// ---- host -------------------------------------------------------------------------------
int g_fa_ready = 0;

constexpr size_t FA_LDS16 = 256 * FA_ST16 * 4 + FA_CTAB * sizeof(uint2);

template <int KC>
hipError_t fa_allow_lds16() {
  hipError_t e = hipFuncSetAttribute((const void*)fa_pass16<KC, false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                     (int)FA_LDS16);
  if (!e)
    e = hipFuncSetAttribute((const void*)fa_pass16<KC, true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)FA_LDS16);
  return e;
}

constexpr size_t FA_LDS32 = (FA_ST * 4 << (FA_TL - 1)) + FA_CTAB * sizeof(uint2);

template <int MODE, bool NAT>
hipError_t fa_allow_lds32() {
  return hipFuncSetAttribute((const void*)fa_pass32<MODE, NAT>, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)FA_LDS32);
}

hipError_t fa_configure() {
  if (g_fa_ready) return hipSuccess;
  uint32_t basis[32], pack[FA_KC_MAX + 1][8];
  fa_basis(basis);
  uint2 beta[32];
  for (int i = 0; i < 32; i++) beta[i] = make_uint2(basis[i], fa_mul16(FA_NU, basis[i] >> 16));
  const FaChunk ch[FA_KC_MAX + 1] = {kFaChunk<0>, kFaChunk<1>, kFaChunk<2>, kFaChunk<3>, kFaChunk<4>, kFaChunk<5>};
  // pack[b]: bits 0..2 of b are index bits K-4 .. K-2
  for (int i = 0; i <= FA_KC_MAX; i++)
    for (int q = 0; q < 8; q++) pack[i][q] = ch[i].pack[q];
  hipError_t e = hipMemcpyToSymbol(HIP_SYMBOL(c_fa_beta), beta, sizeof(beta));
  if (!e) e = hipMemcpyToSymbol(HIP_SYMBOL(c_fa_pack), pack, sizeof(pack));
  if (!e) e = fa_allow_lds32<FA_FWD, false>();
  if (!e) e = fa_allow_lds32<FA_FWD, true>();
  if (!e) e = fa_allow_lds32<FA_FUSED, false>();
  if (!e) e = fa_allow_lds32<FA_INV, false>();
  if (!e) e = fa_allow_lds32<FA_INV, true>();
  if (!e) e = fa_allow_lds16<1>();
  if (!e) e = fa_allow_lds16<2>();
  if (!e) e = fa_allow_lds16<3>();
  if (!e) e = fa_allow_lds16<4>();
  if (!e) e = fa_allow_lds16<5>();
  if (!e)
    e = hipFuncSetAttribute((const void*)fa_prep_rows, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)cbp_words(32 * 1024, true) * 4);
  if (!e) g_fa_ready = 1;
  return e;
}

int fa_log(int64_t n) {  // K: 2^(K-1) >= n
  int K = 1;
  while (((int64_t)1 << (K - 1)) < n) K++;
  return K;
}

unsigned capg(int64_t v, int64_t cap) { return (unsigned)(v < 1 ? 1 : (v > cap ? cap : v)); }

template <bool INV, bool SRC, int R, int B0>
void fa_launch_level(const QcIo* io, QcIo io1, const uint4* in, uint4* out, int64_t XS, int64_t N, int B,
                     hipStream_t st) {
  const int64_t wgs =
      ((N >> B0) * fa_s16_edge(R, B0) + 255) / 256 + (N >> (B0 + R)) * ((fa_s16_columns(R, B0) + 255) / 256);
  cuot_rec_begin(st, "fa_s16_level", 32.0 * (double)N * B);
  hipLaunchKernelGGL((fa_s16_level<INV, SRC, R, B0>), dim3((unsigned)wgs, (unsigned)B), dim3(256), 0, st, io, io1, in,
                     out, XS, N);
  cuot_rec_end(st);
}

template <bool INV>
void fa_launch16(const FaArgs& a, int B, hipStream_t st) {
  const int64_t ntiles = ((int64_t)1 << (a.K - 5)) >> FA_TL;
  // two resident workgroups on each of the 256 CUs; every one walks many tiles
  const dim3 grid(capg(ntiles, 256 / B < 1 ? 1 : 256 / B), (unsigned)B, 2);
  const double per = 512.0 * (double)((int64_t)1 << (a.K - 5)) * B;
  cuot_rec_begin(st, "fa_pass16", INV ? per * 2.0 : per * 1.5);
  switch (a.K - 20) {
#define FA_CASE(KC) \
  case KC: hipLaunchKernelGGL((fa_pass16<KC, INV>), grid, dim3(FA_NT), FA_LDS16, st, a); break;
    FA_CASE(1)
    FA_CASE(2)
    FA_CASE(3)
    FA_CASE(4)
    FA_CASE(5)
#undef FA_CASE
  }
  cuot_rec_end(st);
}

template <int MODE, bool NAT>
void fa_launch32(const FaArgs& a, int B, hipStream_t st) {
  const int64_t ntiles = ((int64_t)1 << (a.K - 5)) >> FA_TL;
  // two resident workgroups on each of the 256 CUs; every one walks many tiles
  const int64_t cap = 512 / B < 1 ? 1 : 512 / B;
  const double per = 512.0 * (double)((int64_t)1 << (a.K - 5)) * B;
  cuot_rec_begin(st, MODE == FA_FUSED ? "fa_pass32 fused" : "fa_pass32", NAT && MODE == FA_FWD ? per * 1.5 : per * 2.0);
  hipLaunchKernelGGL((fa_pass32<MODE, NAT>), dim3(capg(ntiles, cap), (unsigned)B), dim3(FA_NT), FA_LDS32, st, a);
  cuot_rec_end(st);
}

hipError_t fa_transform(const FaArgs& base, int B, hipStream_t st, hipEvent_t ready) {
  const int K = base.K, c = base.c, r = K - 5 - c;
  // upper passes, [lo, lo + R) from the top down to the fused pass's eight layers:
  // one, of at most seven (fewer layers each with the knob)
  const int knob = cuot_knobs().qc_radix;
  int los[16], Rs[16], np = 0;
  for (int top = c; top > FA_TL;) {
    Rs[np] = top - FA_TL < 7 ? top - FA_TL : 7;
    if (knob > 0 && knob < Rs[np]) Rs[np] = knob;
    los[np] = top - Rs[np];
    top = los[np++];
  }
  if (r > 0) fa_launch16<false>(base, B, st);
  FaArgs a;
  for (int i = 0; i < np; i++) {
    a = base;
    a.lo = los[i];
    a.R = Rs[i];
    a.contract = r > 0 && i == 0;
    if (r == 0 && i == 0)
      fa_launch32<FA_FWD, true>(a, B, st);
    else
      fa_launch32<FA_FWD, false>(a, B, st);
  }
  // the first launch that reads A^
  if (ready) {
    hipError_t e = hipStreamWaitEvent(st, ready, 0);
    if (e != hipSuccess) return e;
  }
  a = base;
  a.R = FA_TL;
  fa_launch32<FA_FUSED, false>(a, B, st);
  for (int i = np - 1; i >= 0; i--) {
    a = base;
    a.lo = los[i];
    a.R = Rs[i];
    a.contract = r > 0 && i == 0;
    if (r == 0 && i == 0)
      fa_launch32<FA_INV, true>(a, B, st);
    else
      fa_launch32<FA_INV, false>(a, B, st);
  }
  if (r > 0) fa_launch16<true>(base, B, st);
  return hipGetLastError();
}

}  // namespace

bool cuot_qc_fa_selected(int64_t n) {
  const int K = fa_log(n);
  return K >= FA_KMIN && K <= FA_KMAX;
}

hipError_t cuot_qc_fa_configure() { return fa_configure(); }

// two buffers of 2^K blocks per instance (the matrix-core encoder of small
// codes asks for four)
size_t cuot_qc_fa_scratch_bytes(int64_t n, int B) {
  return (size_t)B * (cuot_qc_mfma_eligible(n) ? 4 : 2) * ((size_t)16 << fa_log(n));
}

hipError_t cuot_launch_qc_fa_prepare(const QcPrep* pr, QcPrep pr1, int B, int K, hipStream_t st) {
  hipError_t e = fa_configure();
  if (e != hipSuccess) return e;
  const int c = K - 5 < 15 ? K - 5 : 15, aidx = 16 + c;
  const int64_t nw = (int64_t)1 << (K - 6);
  hipLaunchKernelGGL(fa_prep_bits, dim3(capg(nw / 256, 1024), (unsigned)B), dim3(256), 0, st, pr, pr1, K);
  int src = 0;
  for (int k = K - 2; k >= FA_STR; k--, src ^= 1)
    hipLaunchKernelGGL(fa_prep_level, dim3(capg(nw / 256, 1024), (unsigned)B), dim3(256), 0, st, pr, pr1, K, k, src);
  const int mp = K - 1 < FA_STR ? K - 1 : FA_STR;
  hipLaunchKernelGGL(fa_prep_rows, dim3(1u << (K - 1 - mp), (unsigned)B), dim3(1024),
                     (size_t)cbp_words((int64_t)1 << (mp - 5), true) * 4, st, pr, pr1, K, mp, src);
  const int bits = K - 5;
  const int Rl = bits < FA_PT ? bits : FA_PT, Ru = bits - Rl;
  if (Ru > 0)
    hipLaunchKernelGGL(fa_prep_fft, dim3(1u << (bits - FA_PT), (unsigned)B), dim3(512), 0, st, pr, pr1, K, c, aidx, Rl,
                       Ru, FA_PT - Ru, 1, src);
  hipLaunchKernelGGL(fa_prep_fft, dim3(1u << (bits - Rl), (unsigned)B), dim3(512), 0, st, pr, pr1, K, c, aidx, 0, Rl, 0,
                     Ru > 0 ? 0 : 1, src);
  return hipGetLastError();
}

hipError_t cuot_launch_qc_fa_encode(const QcIo* io, QcIo io1, const uint32_t* ahat1, const uint32_t* const* ahats, int B,
                                    int K, int64_t nmax, void* scratch, hipStream_t st, hipEvent_t ready) {
  hipError_t e = fa_configure();
  if (e != hipSuccess) return e;
  const int64_t XS = (int64_t)1 << K;  // blocks per instance and buffer
  uint4* X = (uint4*)scratch;
  uint4* Y = X + (int64_t)B * XS;
  const int64_t Nin = XS >> 1;
  // forward conversion; the natural-order coefficients end up in X: row strings
  // of the whole length, or for K > 21 of 2^16 coefficients under s_16-adic
  // levels (the first pass converts the rows of those)
  const bool adic = K > 21;
  {
    const int mp = adic ? 16 : K - 1;
    if (adic) {
      switch (K - 21) {
        case 1: fa_launch_level<false, true, 1, 20>(io, io1, X, Y, XS, Nin, B, st); break;
        case 2: fa_launch_level<false, true, 2, 20>(io, io1, X, Y, XS, Nin, B, st); break;
        case 3: fa_launch_level<false, true, 3, 20>(io, io1, X, Y, XS, Nin, B, st); break;
        default: fa_launch_level<false, true, 4, 20>(io, io1, X, Y, XS, Nin, B, st); break;
      }
      fa_launch_level<false, false, 4, 16>(io, io1, Y, X, XS, Nin, B, st);
    }
    cuot_rec_begin(st, "fa_rows_in", 32.0 * (double)Nin * B);
    const dim3 rgrid(capg(Nin >> 10, 8192), (unsigned)B);
    if (!adic)
      hipLaunchKernelGGL(fa_rows_in<true>, rgrid, dim3(256), 0, st, io, io1, X, XS, Nin, mp, (uint32_t*)Y);
    else
      hipLaunchKernelGGL(fa_rows_in<false>, rgrid, dim3(256), 0, st, io, io1, X, XS, Nin, mp, (uint32_t*)Y);
    cuot_rec_end(st);
    const int64_t S = (int64_t)1 << mp, words = S / 32;
    const int P = (int)(Nin >> mp);
    if ((e = cuot_launch_conv_rows(4096, st, (uint32_t*)Y, words, 128ll * P * B, 128ll * P, XS * 4, mp, 0))) return e;
    if ((e = cuot_launch_transpose_planes2(Y, S, X, true, B * P, P, XS * 4, 128 * words, XS, S, st))) return e;
  }
  FaArgs a;
  memset(&a, 0, sizeof(a));
  a.nat_in = X;
  a.nat_out = X;
  a.E = Y;
  a.ahat = ahat1;
  a.ahats = ahats;
  a.XS = XS;
  a.K = K;
  a.c = K - 5 < 15 ? K - 5 : 15;
  a.a = 16 + a.c;
  if ((e = fa_transform(a, B, st, ready))) return e;
  // inverse conversion of the 2^K coefficients in X
  const int mp = adic ? 16 : (K < 20 ? K : 20);
  const int64_t S = (int64_t)1 << mp, words = S / 32;
  const int P = 1 << (K - mp);
  if ((e = cuot_launch_transpose_planes2(X, S, Y, false, B * P, P, XS, S, XS * 4, 128 * words, st))) return e;
  if ((e = cuot_launch_conv_rows(8192, st, (uint32_t*)Y, words, 128ll * P * B, 128ll * P, XS * 4, mp, 1))) return e;
  if ((e = cuot_launch_transpose_planes2(Y, S, X, true, B * P, P, XS * 4, 128 * words, XS, S, st))) return e;
  if (adic) fa_launch_level<true, false, 4, 16>(io, io1, X, Y, XS, XS, B, st);
  cuot_rec_begin(st, "fa_output", 48.0 * (double)nmax * B);
  switch (K <= 20 ? 0 : K - 20) {
    case 0:
      hipLaunchKernelGGL(fa_output<false>, dim3(capg((nmax + 255) / 256, 16384), (unsigned)B), dim3(256), 0, st, X, XS,
                         io, io1);
      break;
    case 1:
      hipLaunchKernelGGL(fa_output<true>, dim3(capg((nmax + 255) / 256, 16384), (unsigned)B), dim3(256), 0, st, X, XS,
                         io, io1);
      break;
#define FA_CASE(R)                                                                                               \
  case R:                                                                                                        \
    hipLaunchKernelGGL(fa_output_s16<R>,                                                                         \
                       dim3((unsigned)(((nmax + ((int64_t)1 << 20) - 1) >> 20) * 2 * fa_s16_edge(R, 20) / FA_OT + \
                                       (fa_s16_columns(R, 20) + FA_OT - 1) / FA_OT),                             \
                            (unsigned)B),                                                                        \
                       dim3(FA_OT), 0, st, Y, XS, io, io1);                                                      \
    break;
    FA_CASE(2)
    FA_CASE(3)
    FA_CASE(4)
    FA_CASE(5)
#undef FA_CASE
  }
  cuot_rec_end(st);
  return hipGetLastError();
}
