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
//   conversion to the novel basis on the blocks: passes over columns for the
//   powers of s_16 and s_8, two over tiles for the 16 bits below (bits 16 up: in
//   the first pass of the transform); for K > 20 a pass of the GF(2^16) layers,
//   halves of the elements apart; a pass of up to seven GF(2^32) layers; one of
//   the lowest eight, the product by A^ and the inverse of the eight; the mirror
//   image back; y.  For K <= 16 the conversion runs on 128 strings of bits, one a
//   row, transposed there and back (conv_fast.h).
// Between passes the data is element major: element e is 32 planes x 16 bytes
// in one run, so that every tile reads and writes whole lines.
#include <string.h>

#include <type_traits>

#include "conv_fast.h"
#include "kernels.h"
#include "qc_fa.h"
#include "transpose32.h"

namespace {

struct alignas(8) FaConsts {
  uint32_t beta[32][2];              // beta_i and nu times its theta part
  uint32_t pack[FA_KC_MAX + 1][8];  // [kc][q]: bits 0..2 of q are index bits K-4 .. K-2
};

constexpr FaConsts fa_consts() {
  FaConsts c{};
  const FaBasis b = fa_basis();
  for (int i = 0; i < 32; i++) {
    c.beta[i][0] = b.v[i];
    c.beta[i][1] = fa_mul16(FA_NU, b.v[i] >> 16);
  }
  const FaChunk ch[FA_KC_MAX + 1] = {kFaChunk<0>, kFaChunk<1>, kFaChunk<2>, kFaChunk<3>, kFaChunk<4>, kFaChunk<5>};
  for (int i = 0; i <= FA_KC_MAX; i++)
    for (int q = 0; q < 8; q++) c.pack[i][q] = ch[i].pack[q];
  return c;
}

// part of the code object, so that every device has them
__constant__ FaConsts c_fa = fa_consts();

CUOT_DEV uint2 fa_beta(int i) { return make_uint2(c_fa.beta[i][0], c_fa.beta[i][1]); }

constexpr int FA_KMIN = 14, FA_KMAX = 25;
// Log2 of the strings of a's bits that are converted in LDS.  A run prepares A^
// beside the receiver's trees, which from n = 2^19 on have a workgroup on every
// CU; 1024 lanes need the registers of a whole CU and wait for its trees to end:
// at n = 2^20 strings of 2^18 bits took 83 us there, 23 alone.  K > 20: strings of
// 2^16 bits on 512 lanes, which fit beside a tree (31 us there; the added level
// launches cost 3 of 73 us where A^ is prepared alone): run of n = 2^20 607 ->
// 580 us, 2^21 1091 -> 1015, 2^24 8660 -> 8480.  K <= 20: the trees mostly leave CUs
// free, and the launches or half the lanes cost what they save (n = 300000 367 -> 375).
constexpr int fa_str(int K) { return K > 20 ? 16 : K > 19 ? 18 : K - 1; }

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
      if ((v >> b) & 1) c = x2(c, fa_beta(8 * q + b + 1));
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

// A pass holds a tile of 256 elements (rows 2^lo apart times consecutive columns)
// in registers: lane P * 4 + w has word w of the two elements of butterfly P.
// Between layers a lane gives one of the two to the lane whose P differs in the
// next layer's bit and takes one: through LDS where that is another wavefront, by
// lane swaps inside one.
// give u (where this lane's P has bit b set) or v to the lane whose P differs in
// that bit and take the same from it
// (N lanes further; the quads of a row whose bit is set are the BANKS)
template <int NP, int N, int BANKS>
__device__ __forceinline__ void fa_swap_dpp(uint32_t* u, uint32_t* v) {
#pragma unroll
  for (int p = 0; p < NP; p++) {
    const int a = (int)u[p], b = (int)v[p];
    u[p] = (uint32_t)__builtin_amdgcn_update_dpp(a, b, 0x110 | N, 0xF, BANKS, false);       // row_shr
    v[p] = (uint32_t)__builtin_amdgcn_update_dpp(b, a, 0x100 | N, 0xF, 0xF ^ BANKS, false);  // row_shl
  }
}

template <int NP>
__device__ __forceinline__ void fa_swap(uint32_t* lds, uint32_t* u, uint32_t* v, int P, int b) {
  // (b opaque in between: as one chain of choices the compiler merges all ways
  // behind 64 moves)
#define FA_OPAQUE(x) \
  x = __builtin_amdgcn_readfirstlane(x); \
  asm volatile("" : "+s"(x))
  if (b >= 4) {  // another wavefront; the bit is this one's, b the workgroup's
    auto put = [&](const uint32_t* g) {
#pragma unroll
      for (int p = 0; p < NP; p++) lds[p * FA_NT + threadIdx.x] = g[p];
    };
    auto get = [&](uint32_t* g) {
      const int other = (int)threadIdx.x ^ (4 << b);
#pragma unroll
      for (int p = 0; p < NP; p++) g[p] = lds[p * FA_NT + other];
    };
    // only the copies depend on the bit: all wavefronts meet at the same barriers
    int bit = __builtin_amdgcn_readfirstlane(P >> b) & 1;
    if (bit) put(u);
    FA_OPAQUE(bit);
    if (!bit) put(v);
    __syncthreads();
    FA_OPAQUE(bit);
    if (bit) get(u);
    FA_OPAQUE(bit);
    if (!bit) get(v);
    __syncthreads();
  }
  FA_OPAQUE(b);
  if (b == 3) {
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const auto r = __builtin_amdgcn_permlane32_swap(u[p], v[p], false, false);
      u[p] = r[0];
      v[p] = r[1];
    }
  }
  FA_OPAQUE(b);
  if (b == 2) {
#pragma unroll
    for (int p = 0; p < NP; p++) {
      const auto r = __builtin_amdgcn_permlane16_swap(u[p], v[p], false, false);
      u[p] = r[0];
      v[p] = r[1];
    }
  }
  FA_OPAQUE(b);
  if (b == 1) fa_swap_dpp<NP, 8, 0xC>(u, v);
  FA_OPAQUE(b);
  if (b == 0) fa_swap_dpp<NP, 4, 0xA>(u, v);
}

CUOT_DEV int fa_insert(int P, int b, int r) { return ((P >> b) << (b + 1)) | (r << b) | (P & ((1 << b) - 1)); }

// ---- basis conversion in registers ----------------------------------------------------
// Between the monomial basis and the novel one, every split of the index bits at
// r = 16, 8, 4, 2, 1 is an expansion in powers of s_r = x^(2^r) + x, followed by
// the same for the bits above the split (X = s_r) and below it (the conversion of
// Lin, Al-Naffouri, Han and Yang, 2016, after Gao and Mateer's Taylor expansions,
// 2010; the columns in registers below are this file's).  s_r^(2^i) has
// one lower term, so the level of bit b = r + i takes, with half = 2^b and e =
// 2^i, q = hi with its first e coefficients corrected by its last ones, and
// lo_j ^= q_{j-e} (backwards the same with the two steps exchanged): 32 such
// levels for 16 bits, where the novel basis' own levels, bit by bit, have 65
// lower terms (s_15 alone 15).
CUOT_DEV void fa_add(uint32_t& a, uint32_t b, uint32_t k) { a ^= b & k; }
CUOT_DEV void fa_add(uint4& a, uint4 b, uint32_t k) {
  a.x ^= b.x & k;
  a.y ^= b.y & k;
  a.z ^= b.z & k;
  a.w ^= b.w & k;
}
CUOT_DEV void fa_add(uint2& a, uint2 b, uint32_t k) {
  a.x ^= b.x & k;
  a.y ^= b.y & k;
}
CUOT_DEV void fa_add(uint32_t& a, uint32_t b) { a ^= b; }
CUOT_DEV void fa_add(uint2& a, uint2 b) { a = x2(a, b); }
CUOT_DEV void fa_add(uint4& a, uint4 b) { a = x4(a, b); }

// The levels of R bits from b0 on stay inside the columns
//     c + T (2^b0 - u),   T = 0 .. 2^R,   u = 2^(b0-r),   c < 2^b0 - u
// of a group of 2^(b0+R) coefficients (the last one exists for c < 2^R u): at bit
// b0 + i element T meets element T + 2^i, whether as q_{j-e} of its lower
// coefficient, as correction or not at all.  Element T lies in row T of 2^b0
// coefficients for T <= m = c / u, at the end of row T - 1 above; where m >= 2^R
// (no EDGE) all levels are plain butterflies and commute.  Where a group has 2^b0
// rows (b0 = R = 4, u = 1) column 0 has one element more, the group's last.
template <bool INV, int R, bool EDGE, int FROM = 0, int N, typename V>
__device__ __forceinline__ void fa_column_levels(V (&v)[N], int m) {
  if constexpr (!EDGE) {
#pragma unroll
    for (int i = 0; i < R; i++)
#pragma unroll
      for (int T = FROM; T < (1 << R); T++)
        if (!(T >> i & 1)) fa_add(v[T], v[T | 1 << i]);
  } else {
#pragma unroll
    for (int s = 0; s < R; s++) {
      const int i = INV ? s : R - 1 - s, d = 1 << i;
#pragma unroll
      for (int ph = 0; ph < 2; ph++) {
#pragma unroll
        for (int T = FROM; T + d <= (1 << R); T++) {
          if ((ph == 0) != INV) {  // a half's first e coefficients
            if ((T & (2 * d - 1)) == d) fa_add(v[T], v[T + d], T <= m && T + d > m ? ~0u : 0u);
          } else {
            const bool lo = !(T & d), lo1 = T > 0 && !((T - 1) & d);  // row T's bit, row T - 1's
            if (lo || lo1) fa_add(v[T], v[T + d], (T > m ? lo1 : lo && ((T & (d - 1)) || T + d <= m)) ? ~0u : 0u);
          }
        }
        if (N == (1 << R) + 2 && (ph == 0) != INV) fa_add(v[(1 << R) + 1 - d], v[(1 << R) + 1], m == 0 ? ~0u : 0u);
      }
    }
  }
}

// one level on 2^N coefficients in registers
template <int N, int B, int E, bool INV, typename V>
__device__ __forceinline__ void fa_reg_level(V (&v)[1 << N]) {
#pragma unroll
  for (int ph = 0; ph < 2; ph++)
#pragma unroll
    for (int g = 0; g < (1 << N); g += 2 << B)
#pragma unroll
      for (int j = 0; j < (1 << B); j++) {
        const int hi = g + (1 << B);
        if ((ph == 0) != INV) {
          if (j < E) fa_add(v[hi + j], v[hi + j + (1 << B) - E]);
        } else {
          if (j >= E) fa_add(v[g + j], v[hi + j - E]);
        }
      }
}

// whole conversion of N <= 4 bits in registers
template <int N, bool INV, typename V>
__device__ __forceinline__ void fa_reg_conv(V (&v)[1 << N]) {
  if constexpr (!INV) {
    if constexpr (N == 4) fa_reg_level<N, 3, 2, INV>(v);  // powers of s_2
    if constexpr (N >= 3) fa_reg_level<N, 2, 1, INV>(v);
    if constexpr (N == 4) fa_reg_level<N, 3, 4, INV>(v);  // bits 2, 3
    if constexpr (N >= 2) fa_reg_level<N, 1, 1, INV>(v);  // bits 0, 1
  } else {
    if constexpr (N >= 2) fa_reg_level<N, 1, 1, INV>(v);
    if constexpr (N == 4) fa_reg_level<N, 3, 4, INV>(v);
    if constexpr (N >= 3) fa_reg_level<N, 2, 1, INV>(v);
    if constexpr (N == 4) fa_reg_level<N, 3, 2, INV>(v);
  }
}

// Conversion of 2^(4+H) rows, H <= 4, as three steps on registers between which
// the rows go through LDS: the powers of s_4 in columns (c < 15), the bits below
// (16 neighbouring rows) and the bits above (2^H rows 16 apart).
template <int H, bool INV, typename V, typename L, typename S>
__device__ __forceinline__ void fa_step_s4(int c, const L& ld, const S& st) {
  V v[(1 << H) + (H == 4 ? 2 : 1)];
#pragma unroll
  for (int T = 0; T < (1 << H); T++) v[T] = ld(c + 15 * T);
  v[1 << H] = V();
  if (c < (1 << H)) v[1 << H] = ld(c + (15 << H));
  if constexpr (H == 4) {
    v[17] = V();
    if (c == 0) v[17] = ld(255);
  }
  fa_column_levels<INV, H, true>(v, c);
#pragma unroll
  for (int T = 0; T < (1 << H); T++) st(c + 15 * T, v[T]);
  if (c < (1 << H)) st(c + (15 << H), v[1 << H]);
  if constexpr (H == 4) {
    if (c == 0) st(255, v[17]);
  }
}

template <int N, int STRIDE, bool INV, typename V, typename L, typename S>
__device__ __forceinline__ void fa_step_conv(int row, const L& ld, const S& st) {
  V v[1 << N];
#pragma unroll
  for (int k = 0; k < (1 << N); k++) v[k] = ld(row + k * STRIDE);
  fa_reg_conv<N, INV>(v);
#pragma unroll
  for (int k = 0; k < (1 << N); k++) st(row + k * STRIDE, v[k]);
}

constexpr int FA_ST16 = 68;

// LDS slot of tile element e where a step's lanes touch elements eight apart (the
// element stride is 4 mod 64 banks): reflecting every odd group of eight spreads them
CUOT_DEV int fa_slot(int e) { return e ^ (((e >> 3) & 1) * 7); }

// The coefficient rows of a half-mode tile, from powers of s_16 to the novel basis
// (INV: back): row rho (index bits 16 up, X = s_16) lies in plane rho >> KC of
// element (rho mod 2^KC) * C + column.  A lane takes one word of a row.  Level by
// level over the whole tile in LDS, with the novel basis' own terms, the two
// passes took 65 and 70 us more at n = 2^24.
template <int KC>
__device__ __forceinline__ uint32_t& fa_row(uint32_t* lds, int rho, int col, int w) {
  return lds[fa_slot(((rho & ((1 << KC) - 1)) << (FA_TL - KC)) + col) * FA_ST16 + 4 * (rho >> KC) + w];
}

// staging (and the rows' conversion) addresses come from an opaque copy of the lane index, so that the
// compiler recomputes them per phase instead of holding them through the layers
__device__ __forceinline__ int opaque_tid() {
  int t = (int)threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

template <int KC, bool INV>
__device__ __forceinline__ void fa_outer(uint32_t* lds) {
  constexpr int NB = KC + (INV ? 4 : 3), H = NB > 8 ? 4 : NB - 4, LGW = FA_TL - KC + 2;  // words of a row: columns x 4
  // (the longest conversions' addresses would spill the next tile's loads)
  const int tid = INV && KC > 3 ? opaque_tid() : (int)threadIdx.x;
  const int w = tid & 3, col = (tid >> 2) & ((1 << (LGW - 2)) - 1);
  auto halves = [&](auto step, int tasks) {  // tasks per 2^(4+H) rows
    for (int x = tid >> LGW; x < tasks << (NB - 4 - H); x += FA_NT >> LGW) {
      const int base = NB > 8 ? (x / tasks) << 8 : 0;
      step(
          NB > 8 ? x % tasks : x, [&](int r) { return fa_row<KC>(lds, base + r, col, w); },
          [&](int r, uint32_t v) { fa_row<KC>(lds, base + r, col, w) = v; });
    }
    __syncthreads();
  };
  [[maybe_unused]] auto s4 = [&] {
    halves([](int c, const auto& ld, const auto& st) { if (c < 15) fa_step_s4<H, INV, uint32_t>(c, ld, st); }, 16);
  };
  auto s8 = [&] {  // bit 8 of nine: lo_j ^= q_{j-1}
    if constexpr (NB > 8) {
      if (!INV) {
        if (tid >> LGW == 0) fa_row<KC>(lds, 256, col, w) ^= fa_row<KC>(lds, 511, col, w);
        __syncthreads();
      }
      for (int x = (tid >> LGW) + 1; x < 256; x += FA_NT >> LGW)
        fa_row<KC>(lds, x, col, w) ^= fa_row<KC>(lds, 255 + x, col, w);
      __syncthreads();
      if (INV) {
        if (tid >> LGW == 0) fa_row<KC>(lds, 256, col, w) ^= fa_row<KC>(lds, 511, col, w);
        __syncthreads();
      }
    }
  };
  if constexpr (!INV) {
    s8();
    if constexpr (H > 0) s4();
  }
  halves([](int r, const auto& ld, const auto& st) { fa_step_conv<4, 1, INV, uint32_t>(16 * r, ld, st); }, 1 << H);
  if constexpr (H > 1)
    halves([](int r, const auto& ld, const auto& st) { fa_step_conv<H, 16, INV, uint32_t>(r, ld, st); }, 16);
  if constexpr (INV) {
    if constexpr (H > 0) s4();
    s8();
  }
}

// address of element e's coefficient q of half h in natural order
CUOT_DEV int64_t fa_nat(const FaArgs& a, int64_t e, int h, int q) {
  return ((int64_t)q << (a.K - 4)) | ((e >> a.c) << (a.c + 1)) | ((int64_t)h << a.c) | (e & (((int64_t)1 << a.c) - 1));
}

// First and last pass (K > 20): the layers above c, KC of them, where the halves of
// the elements transform apart under GF(2^16) constants (blockIdx.z: the half).
// Tiles of 2^KC elements 2^c apart times 2^(8-KC) consecutive ones.  On the natural
// side the tile's coefficients lie in LDS for the rows' conversion, 16 planes x 4
// words an element and 4 words of padding.  At n = 2^24 the two passes take 240 and
// 440 us (3.4 and 2.4 TB/s); with the whole tile in LDS through the layers 300 and
// 445, of which 190 and 310 were vector operations.
template <int KC, bool INV>
__global__ __launch_bounds__(FA_NT) __attribute__((amdgpu_waves_per_eu(4))) void fa_pass16(FaArgs a) {
  extern __shared__ uint32_t lds[];
  constexpr int LGC = FA_TL - KC, C = 1 << LGC, TC = 1 << FA_TL, NH = TC / 2;
  const int64_t ioff = (int64_t)blockIdx.y * a.XS;
  uint4* E = a.E + ioff;
  const uint4* nin = a.nat_in + ioff;
  uint4* nout = a.nat_out + ioff;
  const int h = (int)blockIdx.z, w = threadIdx.x & 3, P = threadIdx.x >> 2;
  const int64_t ntiles = ((int64_t)1 << (a.K - 5)) >> FA_TL;
  uint2* ctab = (uint2*)(lds + TC * FA_ST16);
  fa_ctab_fill(ctab, threadIdx.x, FA_NT);  // read after the first barrier
  // Staged word f = tid + 512 k: plane fastest in element-major data, element fastest
  // in natural order.  A tile's base is its first column (the 2^KC elements are all
  // those 2^c apart); an address is a scalar part of the base and k's bits plus one
  // of the lane's.
  auto off = [&](int el) { return ((int64_t)(el >> LGC) << a.c) + (el & (C - 1)); };
  auto eptr = [&](int64_t tile, int tid, int k) {
    const uint32_t ln = (uint32_t)off(tid >> 4) * 32 + (tid & 15);
    return (uint4*)((char*)(E + ((tile << LGC) + off(32 * k)) * 32 + 16 * h) + (size_t)(ln * 16));
  };
  auto nptr = [&](uint4* p, int64_t tile, int tid, int k) {
    const uint32_t ln = (uint32_t)fa_nat(a, off(tid & (TC - 1)), 0, tid >> FA_TL);
    return (uint4*)((char*)(p + fa_nat(a, tile << LGC, h, 2 * k)) + (size_t)(ln * 16));
  };
  // LDS slot of an element on the element-major side: by register bit (tile bit
  // LGC), then P
  auto eslot = [&](int el) { return ((el >> LGC) & 1) * NH + ((el >> (LGC + 1)) << LGC | (el & (C - 1))); };
  uint4 st[8];
  auto load_tile = [&](int64_t tile) {
    const int tid = opaque_tid();
#pragma unroll
    for (int k = 0; k < (INV ? 8 : 4); k++) {
      st[k] = z4();
      if constexpr (INV)
        st[k] = *eptr(tile, tid, k);
      else
        st[k] = *nptr((uint4*)nin, tile, tid, k);
    }
  };
  // workgroups are dealt to the 8 XCDs in turn: one XCD's take neighbouring tiles
  const int64_t G = gridDim.x, bx = blockIdx.x;
  const int64_t slot = (G & 7) ? bx : (bx & 7) * (G >> 3) + (bx >> 3);
  if (slot < ntiles) load_tile(slot);
  for (int64_t tile = slot; tile < ntiles; tile += G) {
    int tid = opaque_tid();
#pragma unroll
    for (int k = 0; k < (INV ? 8 : 4); k++) {
      const int f = tid + k * FA_NT;
      *(uint4*)&lds[(INV ? eslot(f >> 4) : fa_slot(f & (TC - 1))) * FA_ST16 + (INV ? f & 15 : f >> FA_TL) * 4] = st[k];
    }
    __syncthreads();
    uint32_t u[16], v[16];
    if constexpr (!INV) {
      fa_outer<KC, false>(lds);
      uint32_t t[8];
#pragma unroll
      for (int p = 0; p < 8; p++) t[p] = lds[fa_slot(P) * FA_ST16 + 4 * p + w];
      fa_pack_planes<KC>(t, u);
#pragma unroll
      for (int p = 0; p < 8; p++) t[p] = lds[fa_slot(NH + P) * FA_ST16 + 4 * p + w];
      fa_pack_planes<KC>(t, v);
    } else {
#pragma unroll
      for (int p = 0; p < 16; p++) u[p] = lds[P * FA_ST16 + 4 * p + w];
#pragma unroll
      for (int p = 0; p < 16; p++) v[p] = lds[(NH + P) * FA_ST16 + 4 * p + w];
    }
    __syncthreads();
    // tile bits 7 .. LGC, or back up; one loop, so that the layer's code is there once
#pragma unroll 1
    for (int step = 0; step < KC; step++) {
      const int b = INV ? LGC + step : FA_TL - 1 - step;
      int sw = step == 0 ? -1 : INV ? b - 1 : b;  // the bit of P to swap with
      FA_OPAQUE(sw);
      fa_swap<16>(lds, u, v, P, sw);
      // the first lane's constant for all, and what the others' g add to it
      const uint32_t g = (uint32_t)(P >> b), g0 = __builtin_amdgcn_readfirstlane(g), d = g ^ g0;
      const uint2 c = x2(fa_beta(a.a - a.c - 1 - (b - LGC)), fa_ctab(ctab, g0));
      uint32_t acc[16];
      if constexpr (INV) {
#pragma unroll
        for (int p = 0; p < 16; p++) v[p] ^= u[p];
      }
      fa_mulc16(v, __builtin_amdgcn_readfirstlane(c.x), acc);
#pragma unroll
      for (int p = 0; p < 16; p++) u[p] ^= acc[p];
      if (__any(d != 0)) fa_add_low(v, d, u);
      if constexpr (!INV) {
#pragma unroll
        for (int p = 0; p < 16; p++) v[p] ^= u[p];
      }
    }
    __syncthreads();
    if constexpr (!INV) {
#pragma unroll
      for (int p = 0; p < 16; p++) lds[P * FA_ST16 + 4 * p + w] = u[p];
#pragma unroll
      for (int p = 0; p < 16; p++) lds[(NH + P) * FA_ST16 + 4 * p + w] = v[p];
      __syncthreads();
    } else {
      uint32_t t[16];
      fa_unpack_planes<KC>(u, t);
#pragma unroll
      for (int p = 0; p < 16; p++) lds[fa_slot(P) * FA_ST16 + 4 * p + w] = t[p];
      fa_unpack_planes<KC>(v, t);
#pragma unroll
      for (int p = 0; p < 16; p++) lds[fa_slot(NH + P) * FA_ST16 + 4 * p + w] = t[p];
      __syncthreads();
      fa_outer<KC, true>(lds);
    }
    // the next tile's loads are issued before this tile's stores
    if (tile + G < ntiles) load_tile(tile + G);
    tid = opaque_tid();
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const int f = tid + k * FA_NT;
      const uint4 o = *(const uint4*)&lds[(INV ? fa_slot(f & (TC - 1)) : eslot(f >> 4)) * FA_ST16 +
                                          (INV ? f >> FA_TL : f & 15) * 4];
      if constexpr (INV)
        *nptr(nout, tile, tid, k) = o;
      else
        *eptr(tile, tid, k) = o;
    }
    __syncthreads();
  }
}

// ---- GF(2^32) passes: layers k < c ------------------------------------------------
// Tiles of 2^R elements 2^lo apart times 2^(8-R) consecutive ones, all 32 planes.
// Held in LDS (128 elements a tile, 256 lanes at 250 registers, every layer
// reading and writing all of it), two wavefronts per SIMD waited half of the
// time; registers hold twice the tile at four wavefronts, and three passes do
// where five did.  At n = 2^24 the passes took 355 + 312 + 924 + 314 + 342 us, now
// 298 + 645 + 305; the middle one issues vector operations all the time, the
// others run at 3.6 TB/s.  Tiles of 128 elements (twice the workgroups where
// there are few) gain 3 to 4 % of an encode at n = 2^16 .. 2^17, 1 % at 2^18 and
// lose from there on: not worth the second set of kernels.
constexpr int FA_ST = 132;  // LDS words of a staged element: 32 planes x 4, 4 of padding

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
      // the index above the fastest part
      const int fh = nat ? 4 * k : (NT >> 5) * k, fl = nat ? tid >> (TL - 1) : tid >> 5;
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
          // planes of index bits 16 up: from powers of s_16 to the novel basis
          if (a.K == 20) fa_reg_conv<3, false>(t);
          if (a.K == 19) fa_reg_level<3, 2, 2, false>(t);
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
      fa_swap<32>(lds, u, v, P, sw);
      const int k = a.lo + b - lgC;
      const uint32_t e = (uint32_t)eb + off(fa_insert(P, b, 0));
      const uint32_t g = ((e >> a.c) << (a.c - k)) | ((e & ((1u << a.c) - 1)) >> (k + 1));
      // the first lane's constant for all, and what the others' g add to it: a
      // wavefront covers 16 neighbouring P, so at most the low four bits differ
      const uint32_t g0 = __builtin_amdgcn_readfirstlane(g), d = g ^ g0;
      const uint2 c = x2(fa_beta(a.a - k), fa_ctab(ctab, g0));
      // (fused: by a mask, as a branch costs moves of both)
      auto add_u = [&](bool now) {
        if constexpr (MODE == FA_FUSED) {
#pragma unroll
          for (int p = 0; p < 32; p++)
            asm("v_bitop3_b32 %0, %0, %1, %2 bitop3:0x78" : "+v"(v[p]) : "v"(u[p]), "s"(0 - (int)now));
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
          if (a.K == 20) fa_reg_conv<4, true>(t);
          if (a.K == 19) {
            fa_reg_level<4, 2, 2, true>(t);
            fa_reg_level<4, 3, 2, true>(t);
          }
          if (a.K == 18) fa_reg_level<4, 3, 4, true>(t);
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

// ---- s_16- and s_8-adic levels on blocks (K > 16) ------------------------------------
// All R levels of a call are one pass, each coefficient read and written once and
// memory the bound: 2^24 blocks in 100 us (5.4 TB/s).  The novel basis' own levels
// from bit 20 up, one pass each, took 934 us forward and 1510 back with the output
// at n = 2^24; the powers of s_16 take 200 and 490, and in bit strings, as the
// bits below then were, the conversion cost 50 us each way at n = 2^20 beside the
// transposes (76 us of an encode before the transform, now 44, and 107 behind it,
// now 64).
// The source: an instance's natural-order buffer, or x_{n+i}, zero from n on.
struct FaSrc {
  const uint4* p;
  int64_t n;
  __device__ __forceinline__ uint4 operator[](int64_t i) const { return i < n ? p[i] : make_uint4(0, 0, 0, 0); }
};

// The product's 2n coefficients (in p, digits of powers of s_16 of 2^16 coefficients
// each, before the levels of bits 16 up) folded to n = 2^(K-1): with e = n / 2^16,
// s_16^e = x^n + x^e, so modulo x^n + 1 the upper half h counts 1 + x^e times.  In
// the digits, x^e h is h rotated by e and, for a digit's last e coefficients,
// which x^(2^16) = s_16 + x carries into the next digit, once more one further in
// their own; the last digit's carry is 1 + x^e again.  EDGE: with what falls on a
// digit's first coefficients; the others' is the rotation alone.
template <typename V, int PARTS, bool EDGE>
struct FaFold {
  const V* p;
  int64_t n, e;
  __device__ __forceinline__ V operator[](int64_t i) const {
    V v = p[i * PARTS];
    fa_add(v, p[(n + i) * PARTS]);
    fa_add(v, p[(n + ((i - e) & (n - 1))) * PARTS]);
    if (EDGE) {
      const int64_t j = i & 65535;
      if (j >= 1 && j <= e) fa_add(v, p[(n + i + 65535 - e) * PARTS]);
      if (i >= e && i < 2 * e) fa_add(v, p[(2 * n - 2 * e + i) * PARTS]);
    }
    return v;
  }
};

// columns of 2^16 - 1 from here on hold no coefficient below 2e of a digit (element
// T of column c is coefficient c - T or, for c < T, one of the digit before)
__device__ __forceinline__ int64_t fa_fold_edge(int64_t n) { return (n >> 15) + 32; }

// elements FROM .. 2^R of column c of the group at base (the last one, beyond
// the group for most columns, only with EDGE)
template <int R, bool EDGE, int FROM = 0, typename SRC, typename V>
__device__ __forceinline__ void fa_column_load(const SRC& in, int64_t base, int64_t c, int64_t ncol, int64_t group,
                                               V (&v)[(1 << R) + 1]) {
#pragma unroll
  for (int T = FROM; T < (1 << R); T++) v[T] = in[base + c + T * ncol];
  v[1 << R] = V();
  if (EDGE && c + (ncol << R) < group) v[1 << R] = in[base + c + (ncol << R)];
}

// Bits B0 .. B0 + R - 1 of N coefficients, a column per lane; from a buffer, x or a
// buffer of 2N folded.
enum { FA_BUF, FA_X, FA_FOLD };
template <bool INV, int SRC, int S, int R, int B0>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void fa_adic_level(
    const QcIo* __restrict__ io, QcIo io1, const uint4* __restrict__ in, uint4* __restrict__ out, int64_t XS, int64_t N) {
  constexpr int64_t U = (int64_t)1 << (B0 - S), NCOL = ((int64_t)1 << B0) - U, GROUP = (int64_t)1 << (B0 + R);
  constexpr int64_t per = (NCOL + 255) / 256;  // workgroups per group
  FaSrc src;
  if (SRC == FA_X) {
    const QcIo q = io ? io[blockIdx.y] : io1;
    src.p = q.x + q.n;
    src.n = q.n;
  } else {
    src.p = in + (int64_t)blockIdx.y * XS;
    src.n = N;
  }
  uint4* dst = out + (int64_t)blockIdx.y * XS;
  const int64_t c0 = (int64_t)(blockIdx.x % per) * 256, c = c0 + threadIdx.x;
  const int64_t base = (int64_t)(blockIdx.x / per) << (B0 + R);
  if (c >= NCOL) return;
  uint4 v[(1 << R) + 1];
  if (c0 < U << R || (SRC == FA_FOLD && c0 < fa_fold_edge(N))) {
    if constexpr (SRC == FA_FOLD)
      fa_column_load<R, true>(FaFold<uint4, 1, true>{src.p, N, N >> 16}, base, c, NCOL, GROUP, v);
    else
      fa_column_load<R, true>(src, base, c, NCOL, GROUP, v);
    fa_column_levels<INV, R, true>(v, (int)(c / U));
    if (c < U << R) dst[base + c + (NCOL << R)] = v[1 << R];
  } else {
    if constexpr (SRC == FA_FOLD)
      fa_column_load<R, false>(FaFold<uint4, 1, false>{src.p, N, N >> 16}, base, c, NCOL, GROUP, v);
    else
      fa_column_load<R, false>(src, base, c, NCOL, GROUP, v);
    fa_column_levels<INV, R, false>(v, 0);
  }
#pragma unroll
  for (int T = 0; T < (1 << R); T++) dst[base + c + T * NCOL] = v[T];
}

// ---- input: blocks x_{n+i} to 128 bit-row strings of N = 2^mp bits ---------------------
__global__ __launch_bounds__(256) void fa_rows_in(const QcIo* __restrict__ io, QcIo io1, int64_t XS, int mp,
                                                  uint32_t* __restrict__ rows) {
  __shared__ uint32_t sm[128][33];
  const QcIo q = io ? io[blockIdx.y] : io1;
  FaSrc src;
  src.p = q.x + q.n;
  src.n = q.n;
  const int64_t N = (int64_t)1 << mp;
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
    uint32_t* dst = rows + (tile << 5);
    for (int f = threadIdx.x; f < 128 * 8; f += 256) {
      const int k = f >> 3, tl = (f & 7) * 4;
      *(uint4*)&dst[(int64_t)k * rw + tl] = make_uint4(sm[k][tl], sm[k][tl + 1], sm[k][tl + 2], sm[k][tl + 3]);
    }
    __syncthreads();
  }
}

// ---- output -------------------------------------------------------------------------
// y_i = x_i ^ H_i ^ H_{i+n}, H the product's coefficients
__global__ __launch_bounds__(256) void fa_output(const uint4* __restrict__ H, int64_t XS, const QcIo* __restrict__ io,
                                                 QcIo io1) {
  const QcIo q = io ? io[blockIdx.y] : io1;
  H += (int64_t)blockIdx.y * XS;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < q.n; i += (int64_t)gridDim.x * 256)
    q.y[i] = x4(q.x[i], x4(H[i], H[i + q.n]));
}

// The same through the last levels, bits B0 .. K-1 (R of them, B0 = 16 or 20).  The
// coefficients i + n of a column's i are a column again: with n = Q (2^B0 - u) + r,
// the one r further, Q elements up (or past the last column around to the first, one more
// up).  It goes through LDS, as Q is no constant.
// A lane takes a block or, with 33 of them to a column, half of one (at n =
// 2^20 19 us, with whole ones, at 190 registers, 40).
constexpr int FA_OT = 128;

template <int R>
struct FaOut {
  static constexpr int PARTS = R > 4 ? 2 : 1;
  using V = std::conditional_t<PARTS == 2, uint2, uint4>;
  const V* p;
  __device__ __forceinline__ V operator[](int64_t i) const { return p[i * PARTS]; }
};

template <int R, int B0, bool EDGE, typename V = typename FaOut<R>::V>
__device__ __forceinline__ void fa_output_column(const FaOut<R>& H, const FaOut<R>& x, V* y, int64_t n, int64_t c,
                                                 int64_t c2, int up, V* second) {
  constexpr int LOW = R > 1 ? 1 << (R - 2) : 0, LU = B0 - 16;  // Q >= LOW: n > 2^(K-2)
  constexpr int64_t NCOL = ((int64_t)1 << B0) - (1 << LU), GROUP = (int64_t)1 << (B0 + R);
  V v[(1 << R) + 1];
  fa_column_load<R, EDGE, LOW>(H, 0, c2, NCOL, GROUP, v);
  fa_column_levels<true, R, EDGE, LOW>(v, (int)(c2 >> LU));
#pragma unroll
  for (int T = LOW; T <= (1 << R); T++)
    if (T >= up && T - up <= (1 << (R - 1))) second[(T - up) * FA_OT + threadIdx.x] = v[T];
  fa_column_load<R, EDGE>(H, 0, c, NCOL, GROUP, v);
  fa_column_levels<true, R, EDGE>(v, (int)(c >> LU));
#pragma unroll
  for (int T = 0; T <= (1 << (R - 1)); T++) {
    const int64_t i = c + T * NCOL;
    if (i < n) {
      V o = x[i];
      fa_add(o, v[T]);
      fa_add(o, second[T * FA_OT + threadIdx.x]);
      y[i * FaOut<R>::PARTS] = o;
    }
  }
}

template <int R, int B0>
__global__ __launch_bounds__(FA_OT) __attribute__((amdgpu_waves_per_eu(2))) void fa_output_adic(
    const uint4* __restrict__ H, int64_t XS, const QcIo* __restrict__ io, QcIo io1) {
  using V = typename FaOut<R>::V;
  constexpr int64_t U = (int64_t)1 << (B0 - 16), NCOL = ((int64_t)1 << B0) - U, ECOL = U << R;
  constexpr int PARTS = FaOut<R>::PARTS, COLS = FA_OT / PARTS;
  __shared__ V second[((1 << (R - 1)) + 1) * FA_OT];
  const QcIo q = io ? io[blockIdx.y] : io1;
  const int part = threadIdx.x % PARTS;
  FaOut<R> h, x;
  h.p = (const V*)(H + (int64_t)blockIdx.y * XS) + part;
  x.p = (const V*)q.x + part;
  V* y = (V*)q.y + part;
  const int64_t c0 = (int64_t)blockIdx.x * COLS, c = c0 + threadIdx.x / PARTS, r = q.n % NCOL;
  if (c >= NCOL) return;
  const bool wrap = c + r >= NCOL;
  const int up = (int)(q.n / NCOL) + (wrap ? 1 : 0);
  const int64_t d0 = c0 + r >= NCOL ? c0 + r - NCOL : c0 + r;  // first lane's second column
  const int64_t c2 = c + r - (wrap ? NCOL : 0);
  if (c0 < ECOL || d0 < ECOL || d0 + COLS > NCOL)
    fa_output_column<R, B0, true>(h, x, y, q.n, c, c2, up, second);
  else
    fa_output_column<R, B0, false>(h, x, y, q.n, c, c2, up, second);
}

// The same for n = 2^(K-1), H folded to n coefficients (or FOLD: still to be): one
// column a lane gives its outputs, no column is worked out twice.  At n = 2^24 the
// folding level and this take 175 + 172 us, the level and the output above 204 + 291
// (of which x and y are 107 at the copy rate).
template <int R, int B0, bool FOLD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void fa_output_cyclic(
    const uint4* __restrict__ H, QcIo q) {
  using V = typename FaOut<R>::V;
  constexpr int PARTS = FaOut<R>::PARTS;
  constexpr int64_t U = (int64_t)1 << (B0 - 16), NCOL = ((int64_t)1 << B0) - U, GROUP = (int64_t)1 << (B0 + R);
  const int part = threadIdx.x % PARTS;
  const int64_t c0 = (int64_t)blockIdx.x * (256 / PARTS), c = c0 + threadIdx.x / PARTS;
  if (c >= NCOL) return;
  FaOut<R> h, x;
  h.p = (const V*)H + part;
  x.p = (const V*)q.x + part;
  V* y = (V*)q.y + part;
  V v[(1 << R) + 1];
  if (c0 < U << R || (FOLD && c0 < fa_fold_edge(GROUP))) {
    if constexpr (FOLD)
      fa_column_load<R, true>(FaFold<V, PARTS, true>{h.p, GROUP, GROUP >> 16}, 0, c, NCOL, GROUP, v);
    else
      fa_column_load<R, true>(h, 0, c, NCOL, GROUP, v);
    fa_column_levels<true, R, true>(v, (int)(c / U));
  } else {
    if constexpr (FOLD)
      fa_column_load<R, false>(FaFold<V, PARTS, false>{h.p, GROUP, GROUP >> 16}, 0, c, NCOL, GROUP, v);
    else
      fa_column_load<R, false>(h, 0, c, NCOL, GROUP, v);
    fa_column_levels<true, R, false>(v, 0);
  }
#pragma unroll
  for (int T = 0; T <= (1 << R); T++) {
    const int64_t i = c + T * NCOL;
    if (i < GROUP) {
      V o = x[i];
      fa_add(o, v[T]);
      y[i * PARTS] = o;
    }
  }
}

// ---- conversion of 2^16 coefficients on blocks (K > 16) --------------------------------
// A workgroup of 256 lanes converts 2^12 blocks, 16 or 17 per lane and step, the
// steps exchanging through LDS.  ROWS: the outer bits 8 .. 15, 256 rows 256 apart
// times 16 consecutive columns; else 4096 consecutive blocks, the s_8-adic levels
// of bits 8 .. 11 (those of 12 .. 15: fa_adic_level) and the bits below 8.
// Memory is the bound: 2^24 blocks in 108 us and, ROWS, 88; back 2^25 in 226 and
// 171 (with the next tile's blocks fetched ahead 225, and ROWS spills).  As strings
// of bits, transposed there and back, the 16 bits took 531 us for 2^24 coefficients
// and 971 back for 2^25, level by level on blocks in LDS (tiles of 512 lanes, two
// barriers a level) 387 and 677 with bits 12 .. 15.
constexpr int FA_CT = 256;

template <bool INV, bool ROWS>
__global__ __launch_bounds__(FA_CT) __attribute__((amdgpu_waves_per_eu(2))) void fa_conv_tile(
    const uint4* in, uint4* out, int64_t XS) {
  extern __shared__ uint4 sm[];
  const int tid = threadIdx.x, x = tid & 15, y = tid >> 4;
  const int64_t tile = blockIdx.x;
  const int64_t g0 = (int64_t)blockIdx.y * XS + (ROWS ? ((tile >> 4) << 16) + ((tile & 15) << 4) : tile << 12);
  // row r of column (or block of 256) cl, in memory and in LDS (padded: 16 lanes
  // 256 bytes apart otherwise meet in the same banks)
  auto mem = [&](int cl, int r) { return g0 + (ROWS ? (r << 8) + cl : (cl << 8) + r); };
  auto slot = [&](int cl, int r) -> uint4& {
    const int i = ROWS ? (r << 4) + cl : (cl << 8) + r;
    return sm[i + (i >> 4)];
  };
  // lanes of a step: the faster index where neighbours are contiguous
  const int xc = ROWS ? x : y, xr = ROWS ? y : x;
  auto lds_ld = [&](int r) { return slot(xc, r); };
  auto lds_st = [&](int r, uint4 v) { slot(xc, r) = v; };
  auto mem_ld = [&](int r) { return in[mem(xc, r)]; };
  auto mem_st = [&](int r, uint4 v) { out[mem(xc, r)] = v; };
  // 16 neighbouring rows per lane
  auto low = [&] {
    fa_step_conv<4, 1, INV, uint4>(16 * xr, lds_ld, lds_st);
    __syncthreads();
  };
  // the s_8-adic levels of 16 blocks of 256
  auto s8 = [&](const auto& ld, const auto& st) {
    if (tid < 255) {
      uint4 v[17];
#pragma unroll
      for (int T = 0; T < 16; T++) v[T] = ld(tid + 255 * T);
      v[16] = z4();
      if (tid < 16) v[16] = ld(tid + 255 * 16);
      if (tid < 64)
        fa_column_levels<INV, 4, true>(v, tid);
      else
        fa_column_levels<INV, 4, false>(v, 0);
#pragma unroll
      for (int T = 0; T < 16; T++) st(tid + 255 * T, v[T]);
      if (tid < 16) st(tid + 255 * 16, v[16]);
    }
  };
  auto lin_ld = [&](int i) { return sm[i + (i >> 4)]; };
  auto lin_st = [&](int i, uint4 v) { sm[i + (i >> 4)] = v; };
  if constexpr (!INV) {
    if constexpr (ROWS) {
      if (xr < 15) fa_step_s4<4, INV, uint4>(xr, mem_ld, lds_st);
    } else {
      s8([&](int i) { return in[g0 + i]; }, lin_st);
      __syncthreads();
      if (xr < 15) fa_step_s4<4, INV, uint4>(xr, lds_ld, lds_st);
    }
    __syncthreads();
    low();
    fa_step_conv<4, 16, INV, uint4>(xr, lds_ld, mem_st);
  } else {
    fa_step_conv<4, 16, INV, uint4>(xr, mem_ld, lds_st);
    __syncthreads();
    low();
    if constexpr (ROWS) {
      if (xr < 15) fa_step_s4<4, INV, uint4>(xr, lds_ld, mem_st);
    } else {
      if (xr < 15) fa_step_s4<4, INV, uint4>(xr, lds_ld, lds_st);
      __syncthreads();
      s8(lin_ld, [&](int i, uint4 v) { out[g0 + i] = v; });
    }
  }
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

// one step of the forward conversion level KL on a's bit string, in place: the
// correction of the upper halves or (LO) the lower halves' update.  Two launches
// of a few us a level; as one, out of place, the update worked every correction
// out again, and with its runs of terms in memory it took 180 us at n = 2^24 for
// levels 20 .. 23, 690 beside the receiver's trees.
template <int KL, bool LO>
__global__ __launch_bounds__(256) void fa_prep_level(const QcPrep* __restrict__ pr, QcPrep pr1, int K) {
  const QcPrep q = pr ? pr[blockIdx.y] : pr1;
  uint32_t* T = q.ahat + ((int64_t)1 << (K - 5));
  const int64_t tid = (int64_t)blockIdx.x * 256 + threadIdx.x, nth = (int64_t)gridDim.x * 256;
  if (LO)
    cbt_lo_update<KL>(T, (int64_t)1 << (K - 6), tid, nth);
  else
    cbt_hi_fix<KL>(T, (int64_t)1 << (K - 6), tid, nth);
}

struct FaSync {
  __device__ void operator()() const { __syncthreads(); }
};

// levels below 2^mp on each string of 2^mp bits, in place (one workgroup each)
__global__ __launch_bounds__(1024) void fa_prep_rows(const QcPrep* __restrict__ pr, QcPrep pr1, int K, int mp) {
  const int nl = (int)blockDim.x;
  extern __shared__ uint32_t sw[];
  const QcPrep q = pr ? pr[blockIdx.y] : pr1;
  const int64_t nw = (int64_t)1 << (mp - 5);
  uint32_t* g = q.ahat + ((int64_t)1 << (K - 5)) + (int64_t)blockIdx.x * nw;
  for (int64_t i = threadIdx.x; i < nw; i += nl) sw[cbp_at<true>(i)] = g[i];
  __syncthreads();
  cbp_convert<true, false>(sw, 0, mp, threadIdx.x, nl, FaSync());
  for (int64_t i = threadIdx.x; i < nw; i += nl) g[i] = sw[cbp_at<true>(i)];
}

constexpr int FA_PT = 10;  // log2 words of a preparation tile

// Element bits lo .. lo + R - 1 on tiles of 2^R words 2^lo apart times 2^lgC
// consecutive ones; the first tile pass takes the words from a's converted bits.
__global__ __launch_bounds__(512) void fa_prep_fft(const QcPrep* __restrict__ pr, QcPrep pr1, int K, int c, int aidx,
                                                   int lo, int R, int lgC, int first) {
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
    const uint32_t* T = A + ((int64_t)1 << (K - 5));
    const uint32_t* pk = c_fa.pack[K <= 20 ? 0 : K - 20];
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
    const uint2 off = fa_beta(aidx - k);
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
constexpr size_t FA_LDS16 = 256 * FA_ST16 * 4 + FA_CTAB * sizeof(uint2);

constexpr size_t FA_LDSC = (4096 + 256) * 16;

template <bool INV, bool ROWS>
hipError_t fa_allow_ldsc() {
  return hipFuncSetAttribute((const void*)fa_conv_tile<INV, ROWS>, hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)FA_LDSC);
}

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

hipError_t fa_allow_lds() {
  hipError_t e = fa_allow_lds32<FA_FWD, false>();
  if (!e) e = fa_allow_lds32<FA_FWD, true>();
  if (!e) e = fa_allow_lds32<FA_FUSED, false>();
  if (!e) e = fa_allow_lds32<FA_INV, false>();
  if (!e) e = fa_allow_lds32<FA_INV, true>();
  if (!e) e = fa_allow_ldsc<false, false>();
  if (!e) e = fa_allow_ldsc<false, true>();
  if (!e) e = fa_allow_ldsc<true, false>();
  if (!e) e = fa_allow_ldsc<true, true>();
  if (!e) e = fa_allow_lds16<1>();
  if (!e) e = fa_allow_lds16<2>();
  if (!e) e = fa_allow_lds16<3>();
  if (!e) e = fa_allow_lds16<4>();
  if (!e) e = fa_allow_lds16<5>();
  return e;
}

hipError_t fa_configure() {
  static CuotDeviceOnce once;
  return once.run(fa_allow_lds);
}

int fa_log(int64_t n) {  // K: 2^(K-1) >= n
  int K = 1;
  while (((int64_t)1 << (K - 1)) < n) K++;
  return K;
}

unsigned capg(int64_t v, int64_t cap) { return (unsigned)(v < 1 ? 1 : (v > cap ? cap : v)); }

template <bool INV, int SRC, int S, int R, int B0>
void fa_launch_level(const QcIo* io, QcIo io1, const uint4* in, uint4* out, int64_t XS, int64_t N, int B,
                     hipStream_t st) {
  const int64_t wgs = (N >> (B0 + R)) * ((((int64_t)1 << B0) - ((int64_t)1 << (B0 - S)) + 255) / 256);
  cuot_rec_begin(st, "fa_adic_level", 32.0 * (double)N * B);
  hipLaunchKernelGGL((fa_adic_level<INV, SRC, S, R, B0>), dim3((unsigned)wgs, (unsigned)B), dim3(256), 0, st, io, io1, in,
                     out, XS, N);
  cuot_rec_end(st);
}

template <bool INV, bool ROWS>
void fa_launch_conv(const uint4* in, uint4* out, int64_t XS, int64_t N, int B, hipStream_t st) {
  cuot_rec_begin(st, "fa_conv_tile", 32.0 * (double)N * B);
  hipLaunchKernelGGL((fa_conv_tile<INV, ROWS>), dim3((unsigned)(N >> 12), (unsigned)B), dim3(FA_CT), FA_LDSC, st, in, out,
                     XS);
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
  cuot_rec_begin(st, "fa_pass32", NAT && MODE == FA_FWD ? per * 1.5 : per * 2.0);
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
  const int mp = fa_str(K);
  for (int k = K - 2; k >= mp; k--) {
    const dim3 grid(capg(nw / 512, 1024), (unsigned)B);
    switch (k) {
#define FA_CASE(KL)                                                                     \
  case KL:                                                                              \
    hipLaunchKernelGGL((fa_prep_level<KL, false>), grid, dim3(256), 0, st, pr, pr1, K); \
    hipLaunchKernelGGL((fa_prep_level<KL, true>), grid, dim3(256), 0, st, pr, pr1, K);  \
    break;
      FA_CASE(16)
      FA_CASE(17)
      FA_CASE(18)
      FA_CASE(19)
      FA_CASE(20)
      FA_CASE(21)
      FA_CASE(22)
      FA_CASE(23)
#undef FA_CASE
    }
  }
  const dim3 strings(1u << (K - 1 - mp), (unsigned)B);
  const size_t lds = (size_t)cbp_words((int64_t)1 << (mp - 5), true) * 4;
  hipLaunchKernelGGL(fa_prep_rows, strings, dim3(K > 20 ? 512 : 1024), lds, st, pr, pr1, K, mp);
  const int bits = K - 5;
  const int Rl = bits < FA_PT ? bits : FA_PT, Ru = bits - Rl;
  if (Ru > 0)
    hipLaunchKernelGGL(fa_prep_fft, dim3(1u << (bits - FA_PT), (unsigned)B), dim3(512), 0, st, pr, pr1, K, c, aidx, Rl,
                       Ru, FA_PT - Ru, 1);
  hipLaunchKernelGGL(fa_prep_fft, dim3(1u << (bits - Rl), (unsigned)B), dim3(512), 0, st, pr, pr1, K, c, aidx, 0, Rl, 0,
                     Ru > 0 ? 0 : 1);
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
  // forward conversion; the natural-order coefficients end up in X: for K <= 16
  // row strings, above levels of powers of s_16 and, for the 2^16 coefficients
  // of those, the rest on blocks (the first pass converts index bits 16 up)
  const bool adic = K > 16;
  if (adic) {
    switch (K - 17) {
#define FA_CASE(R)                                                                        \
  case R:                                                                                 \
    fa_launch_level<false, FA_X, 16, R, 16>(io, io1, nullptr, X, XS, Nin, B, st);        \
    break;
#define FA_CASE2(R)                                                                       \
  case 4 + R:                                                                             \
    fa_launch_level<false, FA_X, 16, R, 20>(io, io1, nullptr, Y, XS, Nin, B, st);        \
    fa_launch_level<false, FA_BUF, 16, 4, 16>(io, io1, Y, X, XS, Nin, B, st);             \
    break;
      FA_CASE(1)
      FA_CASE(2)
      FA_CASE(3)
      FA_CASE(4)
      FA_CASE(5)
      FA_CASE2(2)
      FA_CASE2(3)
      FA_CASE2(4)
#undef FA_CASE
#undef FA_CASE2
    }
    if (K == 17)
      fa_launch_level<false, FA_X, 8, 4, 12>(io, io1, nullptr, Y, XS, Nin, B, st);
    else
      fa_launch_level<false, FA_BUF, 8, 4, 12>(io, io1, X, Y, XS, Nin, B, st);
    fa_launch_conv<false, false>(Y, X, XS, Nin, B, st);
    fa_launch_conv<false, true>(X, X, XS, Nin, B, st);
  } else {
    const int64_t S = Nin, words = S / 32;
    cuot_rec_begin(st, "fa_rows_in", 32.0 * (double)Nin * B);
    hipLaunchKernelGGL(fa_rows_in, dim3(capg(Nin >> 10, 8192), (unsigned)B), dim3(256), 0, st, io, io1, XS, K - 1,
                       (uint32_t*)Y);
    cuot_rec_end(st);
    if ((e = cuot_launch_conv_rows(4096, st, (uint32_t*)Y, words, 128ll * B, 128, XS * 4, K - 1, 0))) return e;
    if ((e = cuot_launch_transpose_planes2(Y, S, X, true, B, 1, XS * 4, 128 * words, XS, S, st))) return e;
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
  // inverse conversion of the 2^K coefficients in X, for one n = 2^(K-1) folded
  // to n of them before the levels of bits 16 up.  Encode, general form -> folded:
  // n = 2^24 3505 -> 3357 us, 2^23 1647 -> 1581, 2^22 806 -> 783, 2^21 406 -> 403; 2^20 266
  // -> 269 and 2^19, 2^18 the same, where the output is short either way.  A batch's
  // members differ in n and take the general form.
  const bool cyclic = K > 21 && !io && io1.n == Nin;
  if (adic) {
    fa_launch_conv<true, true>(X, X, XS, XS, B, st);
    fa_launch_conv<true, false>(X, Y, XS, XS, B, st);
    fa_launch_level<true, FA_BUF, 8, 4, 12>(io, io1, Y, X, XS, XS, B, st);
    if (cyclic) {
      if (K > 22) fa_launch_level<true, FA_FOLD, 16, 4, 16>(io, io1, X, Y, XS, XS / 2, B, st);
    } else if (K > 21) {
      fa_launch_level<true, FA_BUF, 16, 4, 16>(io, io1, X, Y, XS, XS, B, st);
    }
  } else {
    const int64_t words = XS / 32;
    if ((e = cuot_launch_transpose_planes2(X, XS, Y, false, B, 1, XS, XS, XS * 4, 128 * words, st))) return e;
    if ((e = cuot_launch_conv_rows(8192, st, (uint32_t*)Y, words, 128ll * B, 128, XS * 4, K, 1))) return e;
    if ((e = cuot_launch_transpose_planes2(Y, XS, X, true, B, 1, XS * 4, 128 * words, XS, XS, st))) return e;
  }
  cuot_rec_begin(st, cyclic ? "fa_output_cyclic" : adic ? "fa_output_adic" : "fa_output", 48.0 * (double)nmax * B);
  switch (cyclic ? K : K - 16) {
    default:
      hipLaunchKernelGGL(fa_output, dim3(capg((nmax + 255) / 256, 16384), (unsigned)B), dim3(256), 0, st, X, XS, io, io1);
      break;
#define FA_CASE(N, R, B0, SRC)                                                                                      \
  case N:                                                                                                           \
    hipLaunchKernelGGL((fa_output_adic<R, B0>), dim3((FaOut<R>::PARTS << B0) / FA_OT, (unsigned)B), dim3(FA_OT), 0, st, SRC, XS, \
                       io, io1);                                                                                    \
    break;
    FA_CASE(1, 1, 16, X)
    FA_CASE(2, 2, 16, X)
    FA_CASE(3, 3, 16, X)
    FA_CASE(4, 4, 16, X)
    FA_CASE(5, 5, 16, X)
    FA_CASE(6, 2, 20, Y)
    FA_CASE(7, 3, 20, Y)
    FA_CASE(8, 4, 20, Y)
    FA_CASE(9, 5, 20, Y)
#undef FA_CASE
#define FA_CASE(N, R, B0, FOLD, SRC)                                                                                 \
  case N:                                                                                                            \
    hipLaunchKernelGGL((fa_output_cyclic<R, B0, FOLD>), dim3((FaOut<R>::PARTS << B0) / 256), dim3(256), 0, st, SRC, io1); \
    break;
    FA_CASE(22, 5, 16, true, X)
    FA_CASE(23, 2, 20, false, Y)
    FA_CASE(24, 3, 20, false, Y)
    FA_CASE(25, 4, 20, false, Y)
#undef FA_CASE
  }
  cuot_rec_end(st);
  return hipGetLastError();
}
