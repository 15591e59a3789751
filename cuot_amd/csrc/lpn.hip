// lpn.hip -- Ferret's 10-local primal LPN as one fused kernel:
//   out[i] = noise[i] ^ XOR_{j<10} kk[idx(i, j)]
// with the indices generated on the fly by AES under the LPN seed exactly as
// emp-ot's LpnF2 does (ferret/emp-ot/emp-ot/ferret/lpn_f2.h:46-79):
//   rows i..i+3 (a "__compute4" group): AES(makeBlock(i, m)) for m < 10 gives
//     40 words; row i+q uses words 10q..10q+9, idx = w & mask, minus k if >= k;
//   the last 1..4 rows of every task ("__compute1"): AES(makeBlock(i, m)) for
//     m < 3, idx = w[j] % k.
// Tasks split [0, n) in equal widths n/ntasks with the last task taking the
// remainder (LpnF2::bench, lpn_f2.h:100-115, commented out in the reference
// tree; each task is LpnF2::task, lpn_f2.h:72-79).  The reference GPU path materialises the index
// array and uses other counters (gpu/gpu_ops.cu:102-109, dev_layer.cu:146-186);
// this kernel keeps the emp-ot definition and never writes indices to HBM.
//
// Both roles share the (public) indices, so one launch can produce the
// sender's and the receiver's outputs from the same AES work.
#include <string.h>

#include "aes_dev.h"
#include "kernels.h"

namespace {

constexpr int D = 10;


// Two lanes share a __compute4 group: with both roles in one launch the lane's
// parity is its role, each lane computes five of the group's ten AES blocks and
// takes the other's index words from its neighbour; with one role the parity
// picks two of the four rows.  The gathers miss L2 and wait on the last-level
// cache, so what counts is how many are in flight and how many cache lines an
// instruction touches: a pair's two 16-byte reads of the interleaved table fall
// into one line of one instruction (a lane reading both took two instructions
// per line), and at ~110 registers four waves fit a SIMD (three at ~157).
// n = 10,168,320, both roles: 1.68 -> 1.31 ms.
struct LpnKArgs {
  const uint32_t* T0;
  uint32_t rk[44];
  int64_t n, k;
  uint32_t mask;
  int64_t width;   // n / ntasks
  int ntasks;
  int64_t units_per_task;  // units of a full-width task
  int64_t units_total;
  int64_t wg_units;  // batch: units per workgroup
  uint32_t lo, cnt;  // rows of the table this launch covers (cnt = 0: all, through pointers)
  const blk* noise[2];
  const blk* kk[2];
  const blk* kkp;  // both roles' kk interleaved (kkp[2j], kkp[2j+1]) or NULL
  blk* out[2];
  int nroles;
};

// number of __compute4 groups and __compute1 rows of a task of `rows` rows
CUOT_DEV void task_shape(int64_t rows, int64_t& g4, int64_t& t1) {
  g4 = rows > 4 ? (rows - 4 + 3) / 4 : 0;
  t1 = rows - 4 * g4;
}

// One role's view of a slice of the table.  With a uniform base (BUF) the slice
// is a buffer descriptor: a row outside it reads as zero, so a launch that
// covers part of the table takes no branch per gather.  Else block idx of the
// lane's role is p[idx].
template <bool BUF>
struct KkView {
  const blk* p;
  __amdgpu_buffer_rsrc_t rs;
  uint32_t add;  // byte offset (idx << sh) + add, modulo 2^32
  int sh;
};

template <bool BUF>
CUOT_DEV void lpn_gather(const KkView<BUF>& v, uint32_t idx, blk& acc) {
  if constexpr (BUF) {
    const blk_vec x = __builtin_amdgcn_raw_buffer_load_b128(v.rs, (int)((idx << v.sh) + v.add), 0, 0);
    acc = bxor(acc, make_uint4(x.x, x.y, x.z, x.w));
  } else {
    acc = bxor(acc, ldb(v.p + idx));
  }
}

// w & mask, minus k if >= k (mask < 2k, so one subtraction is enough and the
// wrapped difference of a smaller value is the larger number)
CUOT_DEV uint32_t lpn_idx(const LpnKArgs& a, uint32_t w) {
  const uint32_t x = w & a.mask, y = x - (uint32_t)a.k;
  return x < y ? x : y;
}

// the word of the pair's lane SRC (0 or 1), in both lanes
template <int SRC>
CUOT_DEV uint32_t pair_word(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, SRC ? 0xf5 : 0xa0, 0xf, 0xf, true);  // quad [0,0,2,2] or [1,1,3,3]
}

// unit u on the lane pair (lane & 1 = par): a __compute4 group of four rows or
// one __compute1 row.  Both lanes of a pair take the same branches.
template <int NR, bool BUF>
CUOT_DEV void lpn_unit(const AesLds& aes, const LpnKArgs& a, int64_t u, int par) {
  // locate the task and the unit inside it
  int64_t task = 0;
  if (a.ntasks > 1) {
    task = a.units_total >> 32 ? u / a.units_per_task : (int64_t)((uint32_t)u / (uint32_t)a.units_per_task);
    if (task >= a.ntasks) task = a.ntasks - 1;
  }
  const int64_t start = task * a.width;
  const int64_t end = (task == a.ntasks - 1) ? a.n : start + a.width;
  const int64_t lu = u - task * a.units_per_task;
  int64_t g4, t1;
  task_shape(end - start, g4, t1);
  const int role = NR == 2 ? par : 0;
  KkView<BUF> kk;
  if constexpr (BUF) {
    // kkp (two roles interleaved) or kk[0] (one role), rows [lo, lo + cnt)
    const int rb = NR == 2 ? 32 : 16;
    const char* base = (const char*)(NR == 2 ? a.kkp : a.kk[0]);
    kk.rs = __builtin_amdgcn_make_buffer_rsrc((void*)(base + (int64_t)a.lo * rb), 0, (int)(a.cnt * rb), 0x00020000);
    kk.sh = NR == 2 ? 5 : 4;
    kk.add = (uint32_t)(16 * role) - a.lo * (uint32_t)rb;
  } else {
    kk.p = a.kk[role];
  }
  const blk* noise = a.noise[role];
  blk* out = a.out[role];
  if (lu < g4) {
    const int64_t i = start + 4 * lu;
    // this lane's five blocks: words 20 par .. 20 par + 19 of the group, the
    // indices of rows 2 par and 2 par + 1
    uint32_t w[2 * D];
#pragma unroll
    for (int m = 0; m < 5; m++) {
      const blk c = make_uint4((uint32_t)(m + 5 * par), 0u, (uint32_t)i, (uint32_t)((uint64_t)i >> 32));
      const blk e = aes_enc(aes, a.rk, c);
      w[4 * m + 0] = lpn_idx(a, e.x);
      w[4 * m + 1] = lpn_idx(a, e.y);
      w[4 * m + 2] = lpn_idx(a, e.z);
      w[4 * m + 3] = lpn_idx(a, e.w);
    }
    constexpr int NROW = NR == 2 ? 4 : 2;
    const int64_t r0 = NR == 2 ? i : i + 2 * par;
    blk acc[NROW];
#pragma unroll
    for (int q = 0; q < NROW; q++) acc[q] = ldb(noise + r0 + q);
#pragma unroll
    for (int q = 0; q < NROW; q++) {
#pragma unroll
      for (int j = 0; j < D; j++) {
        const uint32_t v = w[(q & 1) * D + j];
        lpn_gather(kk, NR == 1 ? v : (q < 2 ? pair_word<0>(v) : pair_word<1>(v)), acc[q]);
      }
    }
#pragma unroll
    for (int q = 0; q < NROW; q++) stb(out + r0 + q, acc[q]);
  } else if (lu - g4 < t1) {
    const int64_t i = start + 4 * g4 + (lu - g4);
    uint32_t w[12];
#pragma unroll
    for (int m = 0; m < 3; m++) {
      const blk c = make_uint4((uint32_t)m, 0u, (uint32_t)i, (uint32_t)((uint64_t)i >> 32));
      const blk e = aes_enc(aes, a.rk, c);
      w[4 * m + 0] = e.x;
      w[4 * m + 1] = e.y;
      w[4 * m + 2] = e.z;
      w[4 * m + 3] = e.w;
    }
    if (NR == 1 && par) return;  // one row, one role: the even lane's
    blk acc = ldb(noise + i);
#pragma unroll
    for (int j = 0; j < D; j++) lpn_gather(kk, w[j] % (uint32_t)a.k, acc);
    stb(out + i, acc);
  }
}

constexpr int LPN_UNITS = CUOT_AES_WG / 2;  // units per workgroup pass
constexpr int LPN_BATCH_PASSES = 4;         // batch: passes per workgroup (one table fill for all)

template <int NR, bool BUF>
__global__ __launch_bounds__(CUOT_AES_WG) __attribute__((amdgpu_waves_per_eu(4))) void lpn_kernel(LpnKArgs a) {
  __shared__ __align__(16) uint32_t tab[CUOT_AES_LDS_WORDS];
  aes_stage_table(tab, a.T0, threadIdx.x, CUOT_AES_WG);
  __syncthreads();
  const AesLds aes = aes_lds(tab);
  const int64_t stride = (int64_t)gridDim.x * LPN_UNITS;
  for (int64_t u = (int64_t)blockIdx.x * LPN_UNITS + (threadIdx.x >> 1); u < a.units_total; u += stride)
    lpn_unit<NR, BUF>(aes, a, u, threadIdx.x & 1);
}

// Batch: wg_start[i] = first WG of instance i (prefix of ceil(units / wg_units));
// one WG covers wg_units units of a single instance, so the round keys stay
// uniform.
template <int NR>
__global__ __launch_bounds__(CUOT_AES_WG) __attribute__((amdgpu_waves_per_eu(4))) void lpn_batch_kernel(
    const LpnKArgs* __restrict__ tabs, const int64_t* __restrict__ wg_start, int ninst) {
  __shared__ __align__(16) uint32_t tab[CUOT_AES_LDS_WORDS];
  const int64_t g = blockIdx.x;
  int lo = 0, hi = ninst - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (wg_start[mid] <= g)
      lo = mid;
    else
      hi = mid - 1;
  }
  const LpnKArgs& a = tabs[lo];
  aes_stage_table(tab, a.T0, threadIdx.x, CUOT_AES_WG);
  __syncthreads();
  const AesLds aes = aes_lds(tab);
  const int64_t u0 = (g - wg_start[lo]) * a.wg_units;
  const int64_t u1 = u0 + a.wg_units < a.units_total ? u0 + a.wg_units : a.units_total;
  if (a.cnt) {
    for (int64_t u = u0 + (threadIdx.x >> 1); u < u1; u += LPN_UNITS) lpn_unit<NR, true>(aes, a, u, threadIdx.x & 1);
  } else {
    for (int64_t u = u0 + (threadIdx.x >> 1); u < u1; u += LPN_UNITS) lpn_unit<NR, false>(aes, a, u, threadIdx.x & 1);
  }
}

int64_t units_of(int64_t rows) {
  int64_t g4 = rows > 4 ? (rows - 4 + 3) / 4 : 0;
  return g4 + (rows - 4 * g4);
}

}  // namespace

namespace {

bool fill_args(const LpnLaunch& l, LpnKArgs& a) {
  memset(&a, 0, sizeof(a));
  if (l.n <= 0 || l.k < 1 || l.nroles < 1 || l.nroles > 2) return false;
  a.T0 = cuot_device_T0();
  memcpy(a.rk, l.rk, sizeof(a.rk));
  a.n = l.n;
  a.k = l.k;
  uint32_t mask = 1;  // lpn_f2.h:27-31
  while ((int64_t)mask < l.k) mask = (mask << 1) | 1u;
  a.mask = mask;
  a.ntasks = l.ntasks < 1 ? 1 : l.ntasks;
  a.width = l.n / a.ntasks;
  const int64_t last_rows = l.n - (int64_t)(a.ntasks - 1) * a.width;
  a.units_per_task = units_of(a.width);
  if (a.units_per_task < 1) a.units_per_task = 1;
  // full-width tasks then the last one; the kernel maps u -> task by division,
  // so the last task's units start at (ntasks-1)*units_per_task
  a.units_total = (int64_t)(a.ntasks - 1) * a.units_per_task + units_of(last_rows);
  // batch: several passes per table fill once an instance has work for many
  // workgroups; a small one spreads its units over as many as it can
  a.wg_units = a.units_total >= (int64_t)512 * LPN_UNITS * LPN_BATCH_PASSES ? LPN_UNITS * LPN_BATCH_PASSES : LPN_UNITS;
  a.nroles = l.nroles;
  // a slice is addressed by 32-bit byte offsets from a uniform base: one role's
  // table, or both interleaved; other tables go through the lanes' pointers
  a.lo = 0;
  a.cnt = 0;
  if ((l.nroles == 2 ? l.kkp != nullptr : true) && l.k * 16 * l.nroles < ((int64_t)1 << 32)) a.cnt = (uint32_t)l.k;
  for (int r = 0; r < l.nroles; r++) {
    a.noise[r] = l.noise[r];
    a.kk[r] = l.kk[r];
    a.kkp = l.nroles == 2 ? l.kkp : nullptr;
    a.out[r] = l.out[r];
  }
  return true;
}

// Launches that each gather from one slice of the table, adding to what the
// one before left in out.  The gathers are bound by their L2 misses: whatever
// the issue rate, ~57e9 lines/s arrive from the last-level cache, and a table
// of T MB hits an XCD's 4 MB L2 about 4/T of the time.  Halving the table takes
// the index AES twice (0.4 ms at n = 10,168,320, both roles) and pays from
// about 11 MB on: k = 262,144 (8 MB) 1.03 ms whole, 1.07 in two; 327,680 (10 MB)
// 1.14 / 1.13; 393,216 (12 MB) 1.24 / 1.16; 452,160 (14 MB) 1.32 / 1.22;
// three slices lose everywhere (1.58 at 452,160).  An L2 has to see its share of the
// table again and again: with few rows per k the second pass costs what it is
// (whole / two slices, us; one role: k = 730,000, n = 11,406 20 / 39, 365,000 56 / 62,
// 730,000 110 / 102, 2,190,000 264 / 240; k = 1,600,000, n = k 273 / 290, 2k 490 / 476;
// both: k = 452,160, n = 2k 141 / 145, 4k 280 / 271, 10k 607 / 574; k = 800,000
// (26 MB), n = 6k 751 / 786, 10k 1234 / 1210; k = 1,600,000 (51 MB), n = 10k 2771 / 2881).
int lpn_slices(const LpnKArgs& a) {
  const int64_t bytes = (int64_t)a.cnt * 16 * a.nroles;
  if (bytes <= (11ll << 20)) return 1;
  if (a.nroles == 1) return a.n >= 2 * a.k ? 2 : 1;
  if (bytes > (32ll << 20)) return 1;
  return a.n >= (bytes > (16ll << 20) ? 10 : 4) * a.k ? 2 : 1;
}

// Workgroups: one wave of them, two a CU, so that each fills its AES table once
// (2048 -> 512, us; one role / both: n = 1,048,576 65 / 71 -> 56 / 65, 3,145,728 160 / 214 ->
// 152 / 200, 10,168,320 both 1179 -> 1147, 20,000,000 both 3190 -> 2900), but for one role
// with many rows, where it loses (20,000,000 1853 -> 1928).
int64_t lpn_grid(const LpnKArgs& a) {
  const int64_t g = (a.units_total + LPN_UNITS - 1) / LPN_UNITS;
  const int knob = cuot_knobs().lpn_wgs;
  const int64_t cap = knob > 0 ? knob : a.nroles == 1 && a.units_total > (1 << 20) ? 2048 : 512;
  return g > cap ? cap : g < 1 ? 1 : g;
}

}  // namespace

hipError_t cuot_launch_lpn(const LpnLaunch& l, hipStream_t st) {
  if (l.n <= 0) return hipSuccess;
  LpnKArgs a;
  if (!fill_args(l, a)) return hipErrorInvalidValue;
  const int64_t g = lpn_grid(a);
  // algorithmic bytes per role and row: noise in, d gathers, row out
  cuot_rec_begin(st, "lpn_kernel", 16.0 * (D + 2) * (double)l.n * l.nroles);
  const int ns = lpn_slices(a);
  for (int q = 0; q < ns; q++) {
    if (a.cnt) {
      a.lo = (uint32_t)(l.k * q / ns);
      a.cnt = (uint32_t)(l.k * (q + 1) / ns) - a.lo;
    }
    if (q)
      for (int r = 0; r < l.nroles; r++) a.noise[r] = l.out[r];
    if (l.nroles == 2 && a.cnt)
      hipLaunchKernelGGL((lpn_kernel<2, true>), dim3((unsigned)g), dim3(CUOT_AES_WG), 0, st, a);
    else if (l.nroles == 2)
      hipLaunchKernelGGL((lpn_kernel<2, false>), dim3((unsigned)g), dim3(CUOT_AES_WG), 0, st, a);
    else if (a.cnt)
      hipLaunchKernelGGL((lpn_kernel<1, true>), dim3((unsigned)g), dim3(CUOT_AES_WG), 0, st, a);
    else
      hipLaunchKernelGGL((lpn_kernel<1, false>), dim3((unsigned)g), dim3(CUOT_AES_WG), 0, st, a);
  }
  cuot_rec_end(st);
  return hipGetLastError();
}

size_t cuot_lpn_args_bytes() { return sizeof(LpnKArgs); }

int64_t cuot_lpn_args_fill(const LpnLaunch& l, void* out) {
  LpnKArgs a;
  if (!fill_args(l, a)) return -1;
  memcpy(out, &a, sizeof(a));
  return (a.units_total + a.wg_units - 1) / a.wg_units;
}

hipError_t cuot_launch_lpn_batch(const void* tabs_d, const int64_t* wg_start_d, int ninst, int64_t total_wgs,
                                 int nroles, hipStream_t st) {
  if (ninst < 1 || total_wgs < 1 || total_wgs > 0x7fffffff) return hipErrorInvalidValue;
  if (nroles == 2)
    hipLaunchKernelGGL(lpn_batch_kernel<2>, dim3((unsigned)total_wgs), dim3(CUOT_AES_WG), 0, st, (const LpnKArgs*)tabs_d,
                       wg_start_d, ninst);
  else
    hipLaunchKernelGGL(lpn_batch_kernel<1>, dim3((unsigned)total_wgs), dim3(CUOT_AES_WG), 0, st, (const LpnKArgs*)tabs_d,
                       wg_start_d, ninst);
  return hipGetLastError();
}
