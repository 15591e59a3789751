// proto.hip -- small protocol-glue kernels of the SOT / Ferret instances:
// seed-derived setup fix-ups, the SOT sender's masked base-OT rows, the
// receiver's view of them, and Ferret's secret sum and bootstrap COTs.
#include <string.h>

#include "aes_dev.h"
#include "kernels.h"

namespace {

unsigned grid_for(int64_t total) {
  int64_t g = (total + 255) / 256;
  if (g > 65535) g = 65535;
  if (g < 1) g = 1;
  return (unsigned)g;
}

// Everything an instance derives from its seed, in one launch (it was up to six
// PRG streams, a fix-up, the bootstrap, its interleaved copy and a copy of
// Delta: nine launches in front of every instance, 20-30 us of a small one).
// AES_seed({index, stream}): 0 Delta, 1 roots, 2 punctured indices, 3 circulant
// a, 4/5 base-OT messages, 7/8 Ferret bootstrap K and choice bits.  Workgroups
// take 512 items of one section each: trees, then a's blocks, the base-OT
// messages, the bootstrap COTs.
struct SetupKArgs {
  const uint32_t* T0;
  uint32_t rk[44];
  SetupArgs p;
  int64_t ablk;              // blocks of a, with one of zero padding
  unsigned wa, wm, wk;       // first workgroup of the sections after the trees
};

CUOT_DEV blk seed_block(const AesLds& aes, const uint32_t* rk, uint32_t stream, int64_t i) {
  return aes_enc(aes, rk, make_uint4((uint32_t)i, (uint32_t)((uint64_t)i >> 32), stream, 0u));
}

__global__ __launch_bounds__(CUOT_AES_WG) void setup_kernel(SetupKArgs a) {
  __shared__ __align__(16) uint32_t tab[CUOT_AES_LDS_WORDS];
  __shared__ uint4 sh[5];  // Ferret: the workgroup's 512 choice bits, Delta
  aes_stage_table(tab, a.T0, threadIdx.x, CUOT_AES_WG);
  __syncthreads();
  const AesLds aes = aes_lds(tab);
  const SetupArgs& p = a.p;
  const int tid = threadIdx.x;
  const unsigned b = blockIdx.x;
  if (b == 0 && tid == 0) {
    blk d = seed_block(aes, a.rk, 0, 0);
    d.x |= 1u;
    *p.delta = d;
    if (p.delta_out) *p.delta_out = d;
  }
  if (b < a.wa) {
    // roots; choices c[t][h] = 1 - bit (h-1-d) of alpha_t; pos_t = t*2^h + alpha
    const int64_t i = (int64_t)b * CUOT_AES_WG + tid;
    if (i >= p.t) return;
    p.roots[i] = seed_block(aes, a.rk, 1, i);
    const uint32_t alpha = seed_block(aes, a.rk, 2, i).x & (uint32_t)((1ull << p.h) - 1);
    for (int d = 0; d < p.h; d++) p.choice[i * p.h + d] = (uint8_t)(1u - ((alpha >> (p.h - 1 - d)) & 1u));
    if (p.pos) p.pos[i] = (i << p.h) + alpha;
  } else if (b < a.wm) {
    // a's bits, zero from n on
    const int64_t i = (int64_t)(b - a.wa) * CUOT_AES_WG + tid;
    if (i >= a.ablk) return;
    blk v = seed_block(aes, a.rk, 3, i);
    uint32_t* w = (uint32_t*)&v;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int64_t lo = i * 128 + 32 * q;
      if (lo >= p.n)
        w[q] = 0;
      else if (lo + 32 > p.n)
        w[q] &= (1u << (p.n - lo)) - 1u;
    }
    ((blk*)p.a_words)[i] = v;
  } else if (b < a.wk) {
    const int64_t i = (int64_t)(b - a.wm) * CUOT_AES_WG + tid;
    if (i >= p.t * p.h) return;
    p.m0b[i] = seed_block(aes, a.rk, 4, i);
    p.m1b[i] = seed_block(aes, a.rk, 5, i);
  } else {
    // bootstrap COTs: K_j (LSB 0), M_j = K_j ^ c_j * Delta, both interleaved
    const int64_t j0 = (int64_t)(b - a.wk) * CUOT_AES_WG;
    if (tid < 5) {
      blk v = seed_block(aes, a.rk, tid < 4 ? 8 : 0, tid < 4 ? j0 / 128 + tid : 0);
      if (tid == 4) v.x |= 1u;
      sh[tid] = v;
    }
    __syncthreads();
    const int64_t j = j0 + tid;
    if (j >= p.k) return;
    blk K = seed_block(aes, a.rk, 7, j);
    K.x &= ~1u;
    const uint32_t c = (((const uint32_t*)sh)[tid >> 5] >> (tid & 31)) & 1u;
    const blk M = c ? bxor(K, sh[4]) : K;
    p.K[j] = K;
    p.Mr[j] = M;
    if (p.kkp) {
      p.kkp[2 * j] = K;
      p.kkp[2 * j + 1] = M;
    }
  }
}

// silent/sender.cu:80-103: M0[d] = m0b[d] ^ L_d, M1[d] = m1b[d] ^ R_d (d < h);
// M0[h] = m0b[h-1] ^ R_{h-1} ^ Delta, M1[h] = m1b[h-1] ^ L_{h-1} ^ Delta.
// With csum the same lane also forms the receiver's view of its rows (below).
__global__ void sot_msgs_kernel(const blk* sums, const blk* m0b, const blk* m1b, const blk* delta, int64_t t,
                                int h, blk* M0, blk* M1, const uint8_t* choice, blk* csum, blk* fin) {
  const blk D = *delta;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < t * h; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t tr = i / h;
    const int d = (int)(i % h);
    const blk L = sums[(tr * h + d) * 2], R = sums[(tr * h + d) * 2 + 1];
    const blk b0 = m0b[d * t + tr], b1 = m1b[d * t + tr];
    const blk x0 = bxor(b0, L), x1 = bxor(b1, R);
    M0[d * t + tr] = x0;
    M1[d * t + tr] = x1;
    const int c = csum ? choice[tr * h + d] : 0;
    const blk mc = c ? b1 : b0;
    if (csum) csum[tr * h + d] = bxor(c ? x1 : x0, mc);
    if (d == h - 1) {
      const blk f0 = bxor(bxor(b0, R), D), f1 = bxor(bxor(b1, L), D);
      M0[h * t + tr] = f0;
      M1[h * t + tr] = f1;
      if (csum) fin[tr] = bxor(c ? f1 : f0, mc);
    }
  }
}

// The receiver's view (silent/recver.cu:143-157): mc = m_c base-OT message;
// chosen sum at level d = M_c[d] ^ mc[d]; final = M_c[h] ^ mc[h-1].
__global__ void sot_recv_prep_kernel(const uint8_t* choice, const blk* M0, const blk* M1, const blk* m0b,
                                     const blk* m1b, int64_t t, int h, blk* csum, blk* fin) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < t * h; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t tr = i / h;
    const int d = (int)(i % h);
    const int c = choice[tr * h + d];
    const blk mc = c ? m1b[d * t + tr] : m0b[d * t + tr];
    csum[tr * h + d] = bxor(c ? M1[d * t + tr] : M0[d * t + tr], mc);
    if (d == h - 1) fin[tr] = bxor(c ? M1[h * t + tr] : M0[h * t + tr], mc);
  }
}

// Ferret: secret_sum = (L_h ^ R_h) & ~1 ^ Delta (spcot_sender.h:49-58) and
// the receiver's chosen sums (OT of the level sums, mpcot_reg.h:146-157).
__global__ void ferret_sums_kernel(const blk* sums, const blk* delta, const uint8_t* choice, int64_t t, int h,
                                   blk* ssum, blk* csum, blk* lsum, blk* rsum) {
  const blk D = *delta;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < t * h; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t tr = i / h;
    const int d = (int)(i % h);
    const blk L = sums[i * 2], R = sums[i * 2 + 1];
    if (csum) csum[i] = choice[i] ? R : L;
    if (lsum) lsum[i] = L;
    if (rsum) rsum[i] = R;
    if (d == h - 1) {
      blk s = bxor(L, R);
      s.x &= ~1u;
      ssum[tr] = bxor(s, D);
    }
  }
}

__global__ void interleave_kernel(const blk* __restrict__ a, const blk* __restrict__ b, int64_t k,
                                  blk* __restrict__ out) {
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < k; j += (int64_t)gridDim.x * blockDim.x) {
    out[2 * j] = a[j];
    out[2 * j + 1] = b[j];
  }
}

}  // namespace

hipError_t cuot_launch_interleave(const blk* a, const blk* b, int64_t k, blk* out, hipStream_t st) {
  hipLaunchKernelGGL(interleave_kernel, dim3(grid_for(k)), dim3(256), 0, st, a, b, k, out);
  return hipGetLastError();
}

hipError_t cuot_launch_setup(const uint32_t rk[44], const SetupArgs& p, hipStream_t st) {
  SetupKArgs a;
  a.T0 = cuot_device_T0();
  memcpy(a.rk, rk, sizeof(a.rk));
  a.p = p;
  a.ablk = p.a_words ? (p.n + 127) / 128 + 1 : 0;
  auto wgs = [](int64_t items) { return (unsigned)((items + CUOT_AES_WG - 1) / CUOT_AES_WG); };
  a.wa = p.t > 0 ? wgs(p.t) : 1;  // workgroup 0 writes Delta whatever there is
  a.wm = a.wa + wgs(a.ablk);
  a.wk = a.wm + (p.m0b ? wgs(p.t * p.h) : 0);
  const unsigned total = a.wk + (p.K ? wgs(p.k) : 0);
  cuot_rec_begin(st, "setup_kernel", 16.0 * (double)(p.t + a.ablk + (p.m0b ? 2 * p.t * p.h : 0) + (p.K ? 4 * p.k : 0)));
  hipLaunchKernelGGL(setup_kernel, dim3(total), dim3(CUOT_AES_WG), 0, st, a);
  cuot_rec_end(st);
  return hipGetLastError();
}

hipError_t cuot_launch_sot_msgs(const blk* sums, const blk* m0b, const blk* m1b, const blk* delta, int64_t t,
                                int h, blk* M0, blk* M1, const uint8_t* choice, blk* csum, blk* fin, hipStream_t st) {
  hipLaunchKernelGGL(sot_msgs_kernel, dim3(grid_for(t * h)), dim3(256), 0, st, sums, m0b, m1b, delta, t, h, M0, M1,
                     choice, csum, fin);
  return hipGetLastError();
}

hipError_t cuot_launch_sot_recv_prep(const uint8_t* choice, const blk* M0, const blk* M1, const blk* m0b,
                                     const blk* m1b, int64_t t, int h, blk* csum, blk* fin, hipStream_t st) {
  hipLaunchKernelGGL(sot_recv_prep_kernel, dim3(grid_for(t * h)), dim3(256), 0, st, choice, M0, M1, m0b, m1b, t, h,
                     csum, fin);
  return hipGetLastError();
}

hipError_t cuot_launch_ferret_sums(const blk* sums, const blk* delta, const uint8_t* choice, int64_t t, int h,
                                   blk* ssum, blk* csum, blk* lsum, blk* rsum, hipStream_t st) {
  hipLaunchKernelGGL(ferret_sums_kernel, dim3(grid_for(t * h)), dim3(256), 0, st, sums, delta, choice, t, h, ssum,
                     csum, lsum, rsum);
  return hipGetLastError();
}
