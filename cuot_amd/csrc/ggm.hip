// ggm.hip -- fused breadth-first GGM tree expansion with level sums, for the
// sender (full trees) and the receiver (punctured trees rebuilt from its own
// view: chosen level sums + choice bits), in SOT and Ferret flavours.
//
// One workgroup of 512 lanes owns one tree (the reference launches one kernel
// per level plus a multi-pass reduction per level; gpu/aes_op.cu:176-266,
// gpu/gpu_matrix.cu:155-169).  Per tree:
//   A. top levels 0..top breadth-first in LDS, one parent per lane (top = h
//      for h <= 9, else top = h - L with L = min(h - 9, 6), so 2^top is 512 or
//      1024 nodes), level sums by a workgroup XOR reduction; the receiver
//      resolves the sibling of its punctured path at every level
//      (silent/recver.cu:98-115, spcot_recver.h:66-95).
//   B. (h > 9) every lane expands 2^top/512 depth-`top` nodes depth-first for
//      L levels, with a fully unrolled path stack in registers; leaves go
//      straight to HBM, per-depth left/right sums are reduced over the
//      workgroup.  The punctured depth-`top` node contributes nothing.
//   C. (receiver, h > 9) the punctured depth-`top` subtree is rebuilt level
//      by level in LDS from the chosen sums and the workgroup sums of phase B.
// Child rule: left = AES_k0(p) ^ p, right = AES_k1(p) ^ p (twokeyprp.h:7-23).
//
// Bound by the AES (aes_dev.h): the 64 KB table is shared by 512 lanes so that
// two workgroups fit a CU, one's breadth-first levels (a serial chain of AES
// latencies) running beside the other's subtrees.  Sender / receiver: 1024
// trees of depth 15 1.35 / 1.41 -> 0.81 / 0.90 ms (8.3e10 AES/s), 1270 of depth
// 13 0.48 / 0.54 -> 0.31 / 0.33 ms (256 lanes and a 32 KB table before).
#include "aes_dev.h"
#include "kernels.h"

namespace {

constexpr int WG = CUOT_AES_WG;
constexpr int NWAVE = WG / 64;
constexpr int LMAX = 6;      // deepest per-lane DFS (register budget)
constexpr int MAXTOP = 10;   // deepest LDS breadth-first level (h <= 16)

// value of the lane XOR_MASK away (1, 2, 8: DPP; 4, 16: swizzle; 32: permute)
template <int XOR_MASK>
CUOT_DEV uint32_t lane_xor(uint32_t v) {
  if constexpr (XOR_MASK == 1)
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, true);  // quad [1,0,3,2]
  else if constexpr (XOR_MASK == 2)
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x4e, 0xf, 0xf, true);  // quad [2,3,0,1]
  else if constexpr (XOR_MASK == 8)
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xf, 0xf, true);  // row rotate by 8 of 16
  else if constexpr (XOR_MASK == 32)
    return (uint32_t)__shfl_xor((int)v, 32, 64);
  else
    return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, (XOR_MASK << 10) | 0x1f);
}

// XOR of two blocks over a wavefront, scattered: lane l returns word
// bitreverse3(l & 7) of the eight words (a, b).  Each exchange halves the words
// a lane still owns, so 10 exchanges do what 48 would for all words in every
// lane.
CUOT_DEV uint32_t wave_xor2(blk a, blk b) {
  const uint32_t lane = threadIdx.x;
  uint32_t v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
  uint32_t k4[4], k2[2];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t keep = (lane & 1) ? v[i + 4] : v[i], send = (lane & 1) ? v[i] : v[i + 4];
    k4[i] = keep ^ lane_xor<1>(send);
  }
#pragma unroll
  for (int i = 0; i < 2; i++) {
    const uint32_t keep = (lane & 2) ? k4[i + 2] : k4[i], send = (lane & 2) ? k4[i] : k4[i + 2];
    k2[i] = keep ^ lane_xor<2>(send);
  }
  uint32_t r = ((lane & 4) ? k2[1] : k2[0]) ^ lane_xor<4>((lane & 4) ? k2[0] : k2[1]);
  r ^= lane_xor<8>(r);
  r ^= lane_xor<16>(r);
  return r ^ lane_xor<32>(r);
}

// XOR of one block over a wavefront: lane l returns word bitreverse2(l & 3)
CUOT_DEV uint32_t wave_xor1(blk a) {
  const uint32_t lane = threadIdx.x;
  const uint32_t k0 = ((lane & 1) ? a.z : a.x) ^ lane_xor<1>((lane & 1) ? a.x : a.z);
  const uint32_t k1 = ((lane & 1) ? a.w : a.y) ^ lane_xor<1>((lane & 1) ? a.y : a.w);
  uint32_t r = ((lane & 2) ? k1 : k0) ^ lane_xor<2>((lane & 2) ? k0 : k1);
  r ^= lane_xor<4>(r);
  r ^= lane_xor<8>(r);
  r ^= lane_xor<16>(r);
  return r ^ lane_xor<32>(r);
}

CUOT_DEV int bitrev3(int i) { return ((i & 1) << 2) | (i & 2) | ((i >> 2) & 1); }

CUOT_DEV blk clear_lsb(blk v) {
  v.x &= ~1u;
  return v;
}

// NB: breadth-first nodes held (2^9, or 2^10 for trees of depth 16)
template <int NB>
struct Lds {
  uint32_t aes[CUOT_AES_LDS_WORDS];  // first: the table's LDS address folds into the lookups' offsets
  blk nodes[NB];
  blk sums[2 * 16];                // [depth][L,R] for depths 1..16 (index depth-1)
  uint32_t red[LMAX][NWAVE][8];    // per-wave XORs
  blk csum[16];                    // receiver: the tree's chosen sums
  uint8_t choice[16];              // receiver: the tree's choice bits
  blk ext[2 * 16];                 // receiver: level sums of the tree's other subtrees
};

// word i of the workgroup XOR parked in red[slot]
template <int NB>
CUOT_DEV uint32_t red_word(const Lds<NB>& s, int slot, int i) {
  uint32_t r = 0;
#pragma unroll
  for (int w = 0; w < NWAVE; w++) r ^= s.red[slot][w][i];
  return r;
}

CUOT_DEV uint32_t* words(blk* b) { return (uint32_t*)b; }

// word i (0..3) of one side's sum in a breadth-first level: waves 0..3 hold the
// left children's XORs in red[0][wave][0..3], waves 4..7 the right ones'
template <int NB>
CUOT_DEV uint32_t side_word(const Lds<NB>& s, int side, int i) {
  const int w0 = side * (NWAVE / 2);
  uint32_t r = 0;
#pragma unroll
  for (int w = 0; w < NWAVE / 2; w++) r ^= s.red[0][w0 + w][i];
  return r;
}

// Breadth-first expansion in LDS of `nlev` levels below nodes[0].  The lower
// half of the workgroup computes left children (k0), the upper half right ones
// (k1): a level is a serial chain of one AES and the LDS reads of a second one
// on the same lane would lengthen every round of it.
// Receiver mode resolves the sibling on the punctured path at each level
// using chosen sums csum[d0 + r] and external (outside-LDS) side sums ext.
// Returns the punctured index at the last level (receiver) in *punct_out.
// `final_rule`: apply the punctured-leaf rule at the last level.
template <bool RECV, int NB>
CUOT_DEV void bfs_levels(const AesLds& aes, const GgmKArgs& a, Lds<NB>& s, int64_t tree, int d0, int nlev,
                         const blk* ext, bool final_rule, int* punct_out) {
  constexpr int HALF = WG / 2;
  constexpr int Q = NB / WG;  // parents per lane: at most NB / 2 parents in a level
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int side = __builtin_amdgcn_readfirstlane(tid / HALF);
  const int j0 = tid % HALF;
  const uint32_t* rk = a.rk + 44 * side;
  int punct = 0;
  for (int r = 0; r < nlev; r++) {
    const int w = 1 << r;
    const int d = d0 + r;  // sum index: depth d+1
    blk ch[Q], sum = bzero();
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const int j = j0 + q * HALF;
      ch[q] = bzero();
      if (j < w && !(RECV && j == punct)) {
        const blk p = s.nodes[j];
        ch[q] = bxor(aes_enc(aes, rk, p), p);
      }
      sum = bxor(sum, ch[q]);
    }
    const uint32_t x = wave_xor1(sum);
    if (lane < 4) s.red[0][wave][((lane & 1) << 1) | (lane >> 1)] = x;
    __syncthreads();  // all reads of nodes[] are done
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const int j = j0 + q * HALF;
      if (j < w && !(RECV && j == punct)) s.nodes[2 * j + side] = ch[q];
    }
    if (!RECV) {
      if (tid < 8) words(&s.sums[2 * d])[tid] = side_word(s, tid >> 2, tid & 3);
    } else {
      const int c = s.choice[d] ? 1 : 0;
      const int sib = 2 * punct + c;
      const int np = 2 * punct + (1 - c);
      if (tid < 8) {
        // lanes 0..3: the sibling from the chosen side's sum; 4..7: the
        // punctured node, zero until the last level closes it
        const int i = tid & 3;
        const int sd = tid < 4 ? c : 1 - c;
        uint32_t v = side_word(s, sd, i);
        if (ext) v ^= ((const uint32_t*)&ext[2 * r + sd])[i];
        if (tid < 4) {
          words(&s.nodes[sib])[i] = v ^ words(&s.csum[d])[i];
        } else {
          uint32_t f = 0;
          if (final_rule && r == nlev - 1) {
            f = ((const uint32_t*)&a.fin[tree])[i];
            if (a.mode == CUOT_MODE_SOT) {
              f ^= v;  // silent/recver.cu:106-112 final layer: opposite-side sum
            } else {
              // spcot_recver.h:56-63: all other leaves, LSB cleared, xor secret;
              // the chosen side with the sibling is its chosen sum
              uint32_t o = v ^ words(&s.csum[d])[i];
              if (i == 0) o &= ~1u;
              f ^= o;
            }
          }
          words(&s.nodes[np])[i] = f;
        }
      }
      punct = np;
    }
    __syncthreads();
  }
  *punct_out = punct;
}

// Unrolled depth-first expansion of one node for L levels (phase B).
// Leaf pairs jj = 0 .. 2^(L-1)-1 are produced in order.  Going from pair jj-1
// to jj, the path changes below relative depth r0 = L-1-ctz(jj): the node at
// r0 is the pending right child saved when its parent was expanded, and every
// node below it is a left child expanded on the spot.  All branches depend on
// jj only, so they are uniform across the wave and every array index is
// static after unrolling (no scratch).
// Sums of this subtree are xored into sl/sr[1..L].
template <int L>
CUOT_DEV void dfs_subtree(const AesLds& aes, const uint32_t* rk, blk root, blk* leaves, int64_t leaf0,
                          int64_t n_out, bool ferret, blk* sl, blk* sr) {
  blk rightc[L > 1 ? L : 1];
  const uint32_t npairs = 1u << (L - 1);
  for (uint32_t jj = 0; jj < npairs; jj++) {
    const int r0 = (jj == 0) ? 0 : (L - 1 - __builtin_ctz(jj));
    blk cur = root;
#pragma unroll
    for (int r = 1; r <= L - 1; r++) {
      if (r == r0) {
        cur = rightc[r];
      } else if (r > r0) {
        blk lc, rc;
        ggm_expand(aes, rk, cur, lc, rc);
        cur = lc;
        rightc[r] = rc;
        sl[r] = bxor(sl[r], lc);
        sr[r] = bxor(sr[r], rc);
      }
    }
    blk lf, rf;
    ggm_expand(aes, rk, cur, lf, rf);
    sl[L] = bxor(sl[L], lf);
    sr[L] = bxor(sr[L], rf);
    const int64_t g = leaf0 + 2 * (int64_t)jj;
    if (ferret) {
      lf = clear_lsb(lf);
      rf = clear_lsb(rf);
    }
    if (g < n_out) stb(leaves + g, lf);
    if (g + 1 < n_out) stb(leaves + g + 1, rf);
  }
}

// What a workgroup does with its tree:
//   SEND   the sender's subtree p of 2^s (the whole tree when s = 0)
//   PUNCT  the receiver's punctured subtree at depth s (the whole tree when s = 0)
//   KNOWN  the receiver's subtree p of 2^s, unless it is the punctured one
// With s > 0 every workgroup of a tree repeats the top s levels.  SEND adds its
// level sums below depth s to the zeroed output with XOR atomics; KNOWN parks
// them in its own slot of a.part, and PUNCT, the next launch, combines the
// slots of the tree's other subtrees into the sums it rebuilds from.
enum { SEND, PUNCT, KNOWN };

template <int L, int WHAT, int NB>
CUOT_DEV void ggm_tree(const GgmKArgs& a, Lds<NB>& s, int64_t tree, int p) {
  constexpr bool RECV = WHAT != SEND;
  constexpr bool P = WHAT == PUNCT;
  const int tid = threadIdx.x;
  const int h = a.h;
  const int sp = a.s;
  aes_stage_table(s.aes, a.T0, tid, WG);
  if (tid == 0) s.nodes[0] = RECV ? bzero() : ldb(a.roots + tree);
  if (RECV && tid < h) {
    s.csum[tid] = ldb(a.csum + tree * h + tid);
    s.choice[tid] = a.choice[tree * h + tid];
  }
  __syncthreads();
  const AesLds aes = aes_lds(s.aes);
  const bool ferret = a.mode == CUOT_MODE_FERRET;
  const int top = h - sp - L;
  int punct = 0;
  if constexpr (P) {
    // the punctured prefix follows the sides not chosen
    for (int d = 0; d < sp; d++) punct = 2 * punct + (s.choice[d] ? 0 : 1);
    p = punct;
    // sums of the other subtrees, depths sp + 1 .. h (s.sums from index 2 sp)
    if (sp > 0) {
      const int nw = (h - sp) * 8;  // words
      const uint32_t* slots = (const uint32_t*)(a.part + ((tree << sp) * (h - sp)) * 2);
      for (int i = tid; i < nw; i += WG) {
        uint32_t v = 0;
        for (int q = 0; q < (1 << sp); q++)
          if (q != punct) v ^= slots[q * nw + i];
        words(&s.ext[0])[i] = v;
      }
      __syncthreads();
    }
  } else if (sp > 0) {
    bfs_levels<RECV>(aes, a, s, tree, 0, sp, nullptr, false, &punct);
    if (RECV && p == punct) return;  // uniform over the workgroup
    const blk root = s.nodes[p];
    __syncthreads();
    if (tid == 0) s.nodes[0] = root;
    __syncthreads();
  }
  punct = 0;
  bfs_levels<P>(aes, a, s, tree, sp, top, sp > 0 ? s.ext : nullptr, L == 0, &punct);
  const int64_t tree0 = (tree << h) + ((int64_t)p << (h - sp));

  if constexpr (L == 0) {
    // whole tree fits the top phase: write leaves from LDS
    for (int f = tid; f < (1 << top); f += WG) {
      blk v = s.nodes[f];
      if (ferret && !(P && f == punct)) v = clear_lsb(v);
      const int64_t g = tree0 + f;
      if (g < a.n_out) stb(a.leaves + g, v);
    }
  } else {
    // ---- phase B: per-lane depth-first subtrees --------------------------
    blk tl[L + 1], tr[L + 1];
#pragma unroll
    for (int r = 0; r <= L; r++) {
      tl[r] = bzero();
      tr[r] = bzero();
    }
    for (int f = tid; f < (1 << top); f += WG)
      if (!(P && f == punct))
        dfs_subtree<L>(aes, a.rk, s.nodes[f], a.leaves, tree0 + ((int64_t)f << L), a.n_out, ferret, tl, tr);
#pragma unroll
    for (int r = 1; r <= L; r++) {
      const uint32_t x = wave_xor2(tl[r], tr[r]);
      if ((tid & 63) < 8) s.red[r - 1][tid >> 6][bitrev3(tid & 63)] = x;
    }
    __syncthreads();
    if (tid < 8 * L) {
      const int d = top + (tid >> 3);  // below depth sp
      uint32_t v = red_word(s, tid >> 3, tid & 7);
      if (P && sp > 0) v ^= words(&s.ext[2 * d])[tid & 7];
      words(&s.sums[2 * (sp + d)])[tid & 7] = v;
    }
    __syncthreads();
    if constexpr (P) {
      // ---- phase C: rebuild the punctured depth-`top` subtree -------------
      const int pt = punct;
      if (tid == 0) s.nodes[0] = bzero();
      __syncthreads();
      int pl = 0;
      bfs_levels<true>(aes, a, s, tree, sp + top, L, &s.sums[2 * (sp + top)], true, &pl);
      const int64_t base = tree0 + ((int64_t)pt << L);
      if (tid < (1 << L)) {
        blk v = s.nodes[tid];
        if (ferret && tid != pl) v = clear_lsb(v);
        const int64_t g = base + tid;
        if (g < a.n_out) stb(a.leaves + g, v);
      }
    }
  }
  if constexpr (WHAT == SEND) {
    __syncthreads();
    blk* out = a.sums + tree * 2 * h;
    if (sp == 0) {
      if (tid < 2 * h) stb(out + tid, s.sums[tid]);
    } else {
      if (p == 0 && tid < 2 * sp) stb(out + tid, s.sums[tid]);
      const int nw = (h - sp) * 4;  // 64-bit words below depth sp
      if (tid < nw)
        atomicXor((unsigned long long*)(out + 2 * sp) + tid, ((const unsigned long long*)(s.sums + 2 * sp))[tid]);
    }
  }
  if constexpr (WHAT == KNOWN) {
    __syncthreads();
    if (tid < 2 * (h - sp)) stb(a.part + ((tree << sp) + p) * (h - sp) * 2 + tid, s.sums[2 * sp + tid]);
  }
}

// nodes to hold: 2^10 only where the breadth-first top can reach it (h = 16
// with L = 6, or a smaller L by the knob); the smaller form lets two
// workgroups share a CU
template <int L, int WHAT, int NB>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(4))) void ggm_kernel(GgmKArgs) {
  __shared__ __align__(16) Lds<NB> s;
  // the argument block read through its pointer: as a value the 88 round-key
  // words are held across the subtree loop and spill
  const GgmKArgs& a = *(const GgmKArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  if (WHAT == PUNCT)
    ggm_tree<L, WHAT>(a, s, blockIdx.x, 0);
  else
    ggm_tree<L, WHAT>(a, s, blockIdx.x >> a.s, (int)(blockIdx.x & ((1u << a.s) - 1)));
}

// zero level sums for the workgroups that add to them
__global__ __launch_bounds__(256) void ggm_zero_kernel(blk* p, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) stb(p + i, bzero());
}

// Batch: one WG per tree of every instance in the table; start[i] is the first
// global tree of instance i (start[ninst] = total).  All instances share the
// form (L and the node array's size).
template <int L, bool RECV, int NB>
__global__ __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(4))) void ggm_batch_kernel(
    const GgmKArgs* __restrict__ tab, const int64_t* __restrict__ start, int ninst) {
  __shared__ __align__(16) Lds<NB> s;
  const int64_t g = blockIdx.x;
  int lo = 0, hi = ninst - 1;  // last i with start[i] <= g
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (start[mid] <= g)
      lo = mid;
    else
      hi = mid - 1;
  }
  ggm_tree<L, RECV ? PUNCT : SEND>(tab[lo], s, g - start[lo], 0);
}

// Depth-first levels L per lane.  Every lane of the workgroup has a subtree from
// depth 9 on, so L = h - 9; depth 16 keeps L = 6 for the registers and puts two
// subtrees on a lane.
int ggm_rule(int h) {
  if (h <= 9) return 0;
  return h - 9 < LMAX ? h - 9 : LMAX;
}

// the split of whole trees that the knob asks for, 0 where it has none for this depth
int ggm_knob(int h) {
  const int k = cuot_knobs().ggm_dfs;
  const int hi = h - 8 < LMAX ? h - 8 : LMAX;
  return k >= 1 && k <= hi && h - k <= MAXTOP ? k : 0;
}

int ggm_split(int h) {
  const int k = ggm_knob(h);
  return k ? k : ggm_rule(h);
}

// L, plus 16 when the breadth-first top is deeper than 2^9 nodes
int ggm_form(int h, int L) { return L + (h - L > 9 ? 16 : 0); }

// log2 of the workgroups per tree.  With few trees one workgroup each leaves
// most CUs idle, and a tree takes as long as one CU's AES rate allows.  The
// split aims at two workgroups per CU; a subtree keeps at least 8 levels, and
// trees stay whole where the repeated top and the second launch (zeroed sums,
// or the receiver's punctured subtrees) cost what the split saves.  Whole ->
// split, us: sender depth 12: 64 trees 48 -> 36; 13: 3 trees 75 -> 33, 64
// 76 -> 43, 128 77 -> 53; 14: 100 130 -> 75; 15: 40 237 -> 78; 16: 16 449 -> 58.
// Receiver depth 12: 50 -> 50 (whole); 13: 3 81 -> 54, 64 80 -> 63, 65 80 -> 78
// (whole from there); 14: 100 137 -> 118; 15: 40 246 -> 122; 16: 16 458 -> 94.
int ggm_wg_split(int64_t t, int h, bool recv) {
  if (h < (recv ? 13 : 12) || t > (recv && h == 13 ? 64 : 128)) return 0;
  int s = 0;
  while ((t << (s + 1)) <= 512 && s + 1 <= h - 8) s++;
  return s;
}

template <int WHAT>
hipError_t launch_form(const GgmKArgs& a, int L, int64_t wgs, hipStream_t st) {
  dim3 grid((unsigned)wgs), block(WG);
  switch (ggm_form(a.h - a.s, L)) {
#define CUOT_GGM_CASE(X, NB)                                              \
  case X + (NB > 512 ? 16 : 0):                                           \
    hipLaunchKernelGGL((ggm_kernel<X, WHAT, NB>), grid, block, 0, st, a); \
    break;
#define CUOT_GGM_CASES   \
  CUOT_GGM_CASE(0, 512)  \
  CUOT_GGM_CASE(1, 512)  \
  CUOT_GGM_CASE(2, 512)  \
  CUOT_GGM_CASE(3, 512)  \
  CUOT_GGM_CASE(4, 512)  \
  CUOT_GGM_CASE(5, 512)  \
  CUOT_GGM_CASE(6, 512)  \
  CUOT_GGM_CASE(1, 1024) \
  CUOT_GGM_CASE(2, 1024) \
  CUOT_GGM_CASE(3, 1024) \
  CUOT_GGM_CASE(4, 1024) \
  CUOT_GGM_CASE(5, 1024) \
  CUOT_GGM_CASE(6, 1024)
    CUOT_GGM_CASES
#undef CUOT_GGM_CASE
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_ggm(GgmKArgs a, bool recv, hipStream_t st) {
  const int64_t nl = (a.t << a.h) < a.n_out ? (a.t << a.h) : a.n_out;
  const int k = ggm_knob(a.h);
  a.s = k || (recv && a.part == nullptr) ? 0 : ggm_wg_split(a.t, a.h, recv);
  const int L = k ? k : ggm_rule(a.h - a.s);
  hipError_t e = hipSuccess;
  cuot_rec_begin(st, recv ? "ggm_kernel<recv>" : "ggm_kernel<send>", 16.0 * (double)nl);
  if (!recv) {
    if (a.s > 0) {
      const int64_t nz = a.t * 2 * a.h;
      hipLaunchKernelGGL(ggm_zero_kernel, dim3((unsigned)((nz + 255) / 256)), dim3(256), 0, st, a.sums, nz);
    }
    e = launch_form<SEND>(a, L, a.t << a.s, st);
  } else {
    if (a.s > 0) e = launch_form<KNOWN>(a, L, a.t << a.s, st);
    if (!e) e = launch_form<PUNCT>(a, L, a.t, st);
  }
  cuot_rec_end(st);
  return e;
}

template <bool RECV>
hipError_t launch_ggm_batch(const GgmKArgs* tab, const int64_t* start, int ninst, int64_t total, int form,
                            hipStream_t st) {
  dim3 grid((unsigned)total), block(WG);
  switch (form) {
#define CUOT_GGM_CASE(X, NB)                                                                    \
  case X + (NB > 512 ? 16 : 0):                                                                 \
    hipLaunchKernelGGL((ggm_batch_kernel<X, RECV, NB>), grid, block, 0, st, tab, start, ninst); \
    break;
    CUOT_GGM_CASES
#undef CUOT_GGM_CASE
#undef CUOT_GGM_CASES
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

int cuot_ggm_form(int h) { return ggm_form(h, ggm_split(h)); }

size_t cuot_ggm_part_bytes(int64_t t, int h) {
  const int s = ggm_wg_split(t, h, true);
  return s > 0 ? (size_t)(t << s) * (h - s) * 2 * sizeof(blk) : 0;
}

hipError_t cuot_launch_ggm(const GgmKArgs& a, bool receiver, hipStream_t st) { return launch_ggm(a, receiver, st); }

hipError_t cuot_launch_ggm_batch(const GgmKArgs* tab_d, const int64_t* start_d, int ninst, int64_t total_trees,
                                 int form, bool receiver, hipStream_t st) {
  if (ninst < 1 || total_trees < 1 || total_trees > 0x7fffffff) return hipErrorInvalidValue;
  return receiver ? launch_ggm_batch<true>(tab_d, start_d, ninst, total_trees, form, st)
                  : launch_ggm_batch<false>(tab_d, start_d, ninst, total_trees, form, st);
}
