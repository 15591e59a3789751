// bits.hip -- bit-level kernels around the QC code:
//   * sparse encode of the receiver's regular noise (choice bits):
//       b_i = e_i ^ XOR_{p in pos, p >= n} a_{(i - (p - n)) mod n},  i < n,
//     i.e. the same code applied to the weight-t vector e (the reference's
//     cyclic_mat_vec_prod + Mat::modp, silent/quasi_cyclic.cu:130-161, on the
//     workload's 2n -> n code);
//   * the 128-row bit transpose with the reference's bit order
//     (gpu/gpu_ops.cu:31-70): row k bit m = bit k of block m, bit k = byte k/8
//     bit k%8, LSB-first within bytes -- done as 32x32 in-register transposes
//     across 32 lanes, staged through LDS so both sides are coalesced.
#include "kernels.h"
#include "transpose32.h"

namespace {

// 32 bits of the cyclic n-bit vector a starting at bit `start` (bit b of the
// result = a[(start + b) mod n]).  a is padded with at least one zero word.
CUOT_DEV uint32_t cyc_window(const uint32_t* __restrict__ a, int64_t n, int64_t start) {
  uint32_t out = 0;
  int got = 0;
  while (got < 32) {
    const int64_t s = start >= n ? start - n : start;  // start < 2n on every call
    int64_t avail = n - s;  // bits before wrap
    int take = (int)((32 - got) < avail ? (32 - got) : avail);
    const int64_t wi = s >> 5;
    const int sh = (int)(s & 31);
    uint64_t two = (uint64_t)a[wi] | ((uint64_t)a[wi + 1] << 32);
    uint32_t bits = (uint32_t)(two >> sh);
    if (take < 32) bits &= (1u << take) - 1u;
    out |= bits << got;
    got += take;
    start = s + take;
  }
  return out;
}

// out = e_0 ^ a * e_1 for the w set positions of e.  A wavefront takes 128 output
// words (two a lane, which share their middle word) and every fourth position,
// four of them in flight; the four wavefronts' sums meet in LDS.  Bound by L2
// reads at large n (2^24 bits, 1024 positions: 249 us) and by the chain of
// positions at small ones: with all positions in turn in one lane 2^20 bits and
// 128 positions took 27 us, now 9, 190731 and 94 20, now 8, 4000037 and 512 105,
// now 40.
constexpr int SP_WORDS = 128, SP_CHUNK = 512;

__global__ __launch_bounds__(256) void sparse_encode(const uint32_t* __restrict__ a, int64_t n,
                                                     const int64_t* __restrict__ pos, int w,
                                                     uint32_t* __restrict__ out) {
  __shared__ int64_t shift[SP_CHUNK];
  __shared__ uint32_t res[SP_WORDS];
  const int64_t nw = (n + 31) >> 5, last = (n - 1) >> 5;
  const int tid = threadIdx.x, wave = tid >> 6;
  const int64_t B0 = (int64_t)blockIdx.x * SP_WORDS, W0 = B0 + 2 * (tid & 63), lo = W0 * 32;
  if (tid < SP_WORDS) res[tid] = 0u;
  uint32_t acc[2] = {0u, 0u};
  for (int q0 = 0; q0 < w; q0 += SP_CHUNK) {
    const int cnt = w - q0 < SP_CHUNK ? w - q0 : SP_CHUNK;
    __syncthreads();
    for (int q = tid; q < SP_CHUNK && q < cnt + 16; q += 256) {  // four rounds of four
      const int64_t p = q < cnt ? pos[q0 + q] : -1;
      shift[q] = p >= n && p < 2 * n ? p - n : -1;
      const int64_t rel = (p >> 5) - B0;
      if (p >= 0 && p < n && rel >= 0 && rel < SP_WORDS) atomicXor(&res[rel], 1u << (p & 31));
    }
    __syncthreads();
    if (W0 >= nw) continue;
    for (int q = wave; q < cnt; q += 16) {
      uint32_t x[4][3];
      int sh[4];
      bool whole[4];
      int64_t start[4];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        const int64_t s = q + 4 * k < SP_CHUNK ? shift[q + 4 * k] : -1;  // out_i ^= a_{(i - s) mod n}
        start[k] = lo - s;                                               // in (-n, n)
        if (start[k] < 0) start[k] += n;
        whole[k] = s >= 0 && start[k] + 64 <= n;
        if (s < 0) start[k] = -1;
        const int64_t wi = whole[k] ? start[k] >> 5 : 0;
        sh[k] = (int)(start[k] & 31);
        x[k][0] = a[wi];
        x[k][1] = a[wi + 1 < last ? wi + 1 : last];
        x[k][2] = a[wi + 2 < last ? wi + 2 : last];
      }
#pragma unroll
      for (int k = 0; k < 4; k++) {
        if (whole[k]) {
          acc[0] ^= (uint32_t)(((uint64_t)x[k][1] << 32 | x[k][0]) >> sh[k]);
          acc[1] ^= (uint32_t)(((uint64_t)x[k][2] << 32 | x[k][1]) >> sh[k]);
        } else if (start[k] >= 0) {  // past the row's end
#pragma unroll
          for (int r = 0; r < 2; r++)
            if (lo + 32 * r < n) acc[r] ^= cyc_window(a, n, (start[k] + 32 * r) % n);
        }
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 2; r++)
    if (acc[r]) atomicXor(&res[2 * (tid & 63) + r], acc[r]);
  __syncthreads();
  if (tid < SP_WORDS && B0 + tid < nw) {
    uint32_t v = res[tid];
    const int64_t left = n - (B0 + tid) * 32;
    if (left < 32) v &= (1u << left) - 1u;
    out[B0 + tid] = v;
  }
}

// n >= 2^25 and a multiple of 32: there are words enough for a lane to take all
// positions, and the window of position s starts at the same bit offset sb = s mod 32
// in every word, so output word W takes (a[W - so] << sb) | (a[W - so - 1] >> (32 - sb))
// with so = s / 32 (indices mod n / 32); two consecutive words share their loads.
// sparse_encode / this, us: 2^24 bits, 1024 positions 235 / 257; 2^25, 16 13 / 11, 1024
// 453 / 419; 2^26, 16 24 / 17, 1024 879 / 811; 2^27, 1024 1732 / 1566.
constexpr int SPR = 2;
constexpr int64_t SP_WIDE_MIN = (int64_t)1 << 25;

__global__ void sparse_encode_wide(const uint32_t* __restrict__ a, int64_t n, const int64_t* __restrict__ pos, int w,
                                   uint32_t* __restrict__ out) {
  const int64_t nw = n >> 5;
  for (int64_t W0 = ((int64_t)blockIdx.x * 256 + threadIdx.x) * SPR; W0 < nw; W0 += (int64_t)gridDim.x * 256 * SPR) {
    uint32_t acc[SPR] = {};
    for (int q = 0; q < w; q++) {
      const int64_t p = pos[q];
      if (p < 0 || p >= 2 * n) continue;
      if (p < n) {
        const int64_t pw = (p >> 5) - W0;
#pragma unroll
        for (int r = 0; r < SPR; r++)
          if (pw == r) acc[r] ^= 1u << (p & 31);
        continue;
      }
      const int64_t s = p - n;  // out_i ^= a_{(i - s) mod n}
      const int sb = (int)(s & 31);
      int64_t i = W0 - (s >> 5) - 1;  // in [-nw, nw)
      if (i < 0) i += nw;
      uint32_t prev = a[i];
#pragma unroll
      for (int r = 0; r < SPR; r++) {
        if (++i == nw) i = 0;
        const uint32_t cur = a[i];
        acc[r] ^= sb ? (cur << sb) | (prev >> (32 - sb)) : cur;
        prev = cur;
      }
    }
#pragma unroll
    for (int r = 0; r < SPR; r++)
      if (W0 + r < nw) out[W0 + r] = acc[r];
  }
}

// ---- transpose ---------------------------------------------------------------
CUOT_DEV uint32_t transpose32(uint32_t x, int lane) { return cuot_transpose32(x, lane); }

// blocks -> rows.  WG: 256 lanes, 1024 blocks (32 tiles of 32 blocks).
// rows: 128 rows of N bits, row stride N/32 words.  blockIdx.y selects a plane
// (input plane stride in_ps blocks, output plane stride out_ps words).
__global__ __launch_bounds__(256) void transpose_fwd(const uint4* __restrict__ in, int64_t N,
                                                     uint32_t* __restrict__ rows, int P, int64_t in_is, int64_t in_ps,
                                                     int64_t out_is, int64_t out_ps) {
  __shared__ uint32_t sm[128][33];
  const int inst = (int)blockIdx.y / P, pl = (int)blockIdx.y % P;
  in += inst * in_is + pl * in_ps;
  rows += inst * out_is + pl * out_ps;
  const int lane = threadIdx.x & 31;
  const int grp = threadIdx.x >> 5;  // 8 groups of 32 lanes
  const int64_t ntile = N / 32;
  for (int64_t t0 = (int64_t)blockIdx.x * 32; t0 < ntile; t0 += (int64_t)gridDim.x * 32) {
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int tl = grp * 4 + r;  // tile within the group of 32 tiles
      const int64_t tile = t0 + tl;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (tile < ntile) v = in[tile * 32 + lane];
      sm[0 * 32 + lane][tl] = transpose32(v.x, lane);
      sm[1 * 32 + lane][tl] = transpose32(v.y, lane);
      sm[2 * 32 + lane][tl] = transpose32(v.z, lane);
      sm[3 * 32 + lane][tl] = transpose32(v.w, lane);
    }
    __syncthreads();
    const int64_t rw = N / 32;  // words per row
    if ((N & 127) == 0) {
      // rows of a multiple of 4 words: 16-byte stores (4 words of one row per lane)
      for (int f = threadIdx.x; f < 128 * 8; f += 256) {
        const int k = f >> 3, tl = (f & 7) * 4;
        if (t0 + tl < ntile)
          *(uint4*)&rows[(int64_t)k * rw + t0 + tl] = make_uint4(sm[k][tl], sm[k][tl + 1], sm[k][tl + 2], sm[k][tl + 3]);
      }
    } else {
      for (int f = threadIdx.x; f < 128 * 32; f += 256) {
        const int k = f >> 5, tl = f & 31;
        if (t0 + tl < ntile) rows[(int64_t)k * rw + t0 + tl] = sm[k][tl];
      }
    }
    __syncthreads();
  }
}

// rows -> blocks
__global__ __launch_bounds__(256) void transpose_inv(const uint32_t* __restrict__ rows, int64_t N,
                                                     uint4* __restrict__ out, int P, int64_t in_is, int64_t in_ps,
                                                     int64_t out_is, int64_t out_ps) {
  __shared__ uint32_t sm[128][33];
  const int inst = (int)blockIdx.y / P, pl = (int)blockIdx.y % P;
  rows += inst * in_is + pl * in_ps;
  out += inst * out_is + pl * out_ps;
  const int lane = threadIdx.x & 31;
  const int grp = threadIdx.x >> 5;
  const int64_t ntile = N / 32;
  const int64_t rw = N / 32;
  for (int64_t t0 = (int64_t)blockIdx.x * 32; t0 < ntile; t0 += (int64_t)gridDim.x * 32) {
    if ((N & 127) == 0) {
      // rows of a multiple of 4 words: 16-byte loads (4 words of one row per lane)
      for (int f = threadIdx.x; f < 128 * 8; f += 256) {
        const int k = f >> 3, tl = (f & 7) * 4;
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (t0 + tl < ntile) v = *(const uint4*)&rows[(int64_t)k * rw + t0 + tl];
        sm[k][tl] = v.x;
        sm[k][tl + 1] = v.y;
        sm[k][tl + 2] = v.z;
        sm[k][tl + 3] = v.w;
      }
    } else {
      for (int f = threadIdx.x; f < 128 * 32; f += 256) {
        const int k = f >> 5, tl = f & 31;
        sm[k][tl] = (t0 + tl < ntile) ? rows[(int64_t)k * rw + t0 + tl] : 0u;
      }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int tl = grp * 4 + r;
      const int64_t tile = t0 + tl;
      uint4 v;
      v.x = transpose32(sm[0 * 32 + lane][tl], lane);
      v.y = transpose32(sm[1 * 32 + lane][tl], lane);
      v.z = transpose32(sm[2 * 32 + lane][tl], lane);
      v.w = transpose32(sm[3 * 32 + lane][tl], lane);
      if (tile < ntile) out[tile * 32 + lane] = v;
    }
    __syncthreads();
  }
}

unsigned grid_for(int64_t total, int64_t cap = 1 << 16) {
  int64_t g = (total + 255) / 256;
  if (g > cap) g = cap;
  if (g < 1) g = 1;
  return (unsigned)g;
}

}  // namespace

hipError_t cuot_launch_sparse(const uint32_t* a_words, int64_t n, const int64_t* pos, int w, uint32_t* out,
                              hipStream_t st) {
  const int64_t nw = (n + 31) >> 5;
  if (n >= SP_WIDE_MIN && (n & 31) == 0) {
    hipLaunchKernelGGL(sparse_encode_wide, dim3(grid_for((nw + SPR - 1) / SPR)), dim3(256), 0, st, a_words, n, pos, w,
                       out);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(sparse_encode, dim3((unsigned)((nw + SP_WORDS - 1) / SP_WORDS)), dim3(256), 0, st, a_words, n, pos,
                     w, out);
  return hipGetLastError();
}

hipError_t cuot_launch_transpose_planes2(const void* in, int64_t N, void* out, bool inverse, int planes, int P,
                                        int64_t in_is, int64_t in_ps, int64_t out_is, int64_t out_ps,
                                        hipStream_t st) {
  if (planes < 1 || P < 1 || planes > 65535) return hipErrorInvalidValue;
  int64_t ntile = N / 32;
  int64_t g = (ntile + 31) / 32;
  int64_t cap = planes > 1 ? 16384 / planes : 8192;
  if (cap < 1) cap = 1;
  if (g > cap) g = cap;
  if (g < 1) g = 1;
  dim3 grid((unsigned)g, (unsigned)planes);
  cuot_rec_begin(st, inverse ? "transpose_inv" : "transpose_fwd", 2.0 * 16.0 * (double)N * planes);
  if (!inverse)
    hipLaunchKernelGGL(transpose_fwd, grid, dim3(256), 0, st, (const uint4*)in, N, (uint32_t*)out, P, in_is, in_ps,
                       out_is, out_ps);
  else
    hipLaunchKernelGGL(transpose_inv, grid, dim3(256), 0, st, (const uint32_t*)in, N, (uint4*)out, P, in_is, in_ps,
                       out_is, out_ps);
  cuot_rec_end(st);
  return hipGetLastError();
}

hipError_t cuot_launch_transpose_planes(const void* in, int64_t N, void* out, bool inverse, int planes,
                                       int64_t in_ps, int64_t out_ps, hipStream_t st) {
  return cuot_launch_transpose_planes2(in, N, out, inverse, planes, planes, 0, in_ps, 0, out_ps, st);
}

hipError_t cuot_launch_transpose(const void* in, int64_t N, void* out, bool inverse, hipStream_t st) {
  return cuot_launch_transpose_planes(in, N, out, inverse, 1, 0, 0, st);
}
