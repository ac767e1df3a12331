// Tree-sparse attention backward for gfx950 (MI355X).
//
// The reference has no backward (README.md:198 lists it as missing).  This is
// the gradient of the function its forward computes
// (block_sparse_tree_fwd_kernel, tree_sparse_flashattn.py:163-339): with
// z = sm_scale * q.k over a row's visible keys (the dense prefix [0, P) and the
// tree keys its CSR row marks), P = softmax(z), O = P V,
//   dV = P^T dO,  dP = dO V^T,  dS = P * (dP - rowsum(dO * O)),
//   dQ = sm_scale * dS K,  dK = sm_scale * dS^T Q,
// summed over the G query heads of each kv head.  P is recomputed from the
// forward's per-row log-sum-exp (tsfa_fwd_lse).
//
// Kernels (one call = two or three launches, no host synchronisation):
//   * bwd_prep_vis_kernel, two jobs in one launch:
//     prep -- per query row (16 lanes): Dv = rowsum(dO * O) in fp32, the
//     log2-domain LSE, and (when the dQ pass is split) the row of the fp32 dQ
//     accumulator cleared.  Rows with no visible key (LSE = -inf) and the
//     padding rows of the last 32-row tile get LSE = +inf and Dv = 0, so their
//     P and dS are exactly 0;
//     visibility -- per (32-row tile, tree key) a word (bit m: row 32*tile + m
//     sees the key), from the CSR metadata;
//   * kv_role of bwd_main_kernel (key-parallel, dK and dV): a workgroup owns 128 keys of
//     one (batch, kv head) -- prefix keys and tree keys in separate blocks --
//     as 4 key groups x 2 row groups of waves; each wave keeps dK^T and dV^T
//     of its 32 keys in registers while its row group walks every other
//     32-row tile of the (batch, kv head) (rows token-major, r = t*G + g, as
//     in the forward).  Per tile, on v_mfma_f32_32x32x16: S = Q K^T and dP =
//     dO V^T (a lane holds one key), then dV^T += dO^T P and dK^T += Q^T dS
//     with P and dS taken straight from the S / dP accumulators (the MFMA k
//     order is permuted to the order the accumulator holds rows in; the dO^T
//     / Q^T operands come from ds_read_b64_tr_b16 in the same order).  Q / dO
//     tiles, their row statistics and the tree block's mask words move HBM
//     -> LDS with global_load_lds, double-buffered per row group; one LDS
//     copy of each tile serves both the row reads and the transposed reads
//     (a swizzle that is conflict-free for both patterns).  The row groups
//     merge their sums through LDS at the end;
//   * dq_role of bwd_main_kernel (row-parallel, dQ): half a workgroup owns 128
//     rows and a split of the 32-key units; S^T, dP^T, dS^T recomputed per unit
//     and dQ^T += K^T dS^T accumulated in registers; an unsplit chunk writes dQ
//     directly, split chunks add once per workgroup to the fp32 accumulator;
//   * bwd_dq_kernel (split chunks only): dQ = sm_scale * accumulator in the
//     input dtype.
// The two roles are independent once the first launch has run; in one launch
// the dQ workgroups fill the CUs that the dK / dV ones leave idle (264 of one
// per CU at the Llama-3-8B shape: a second round of 8).

#include <math.h>
#include <stdlib.h>

#include <algorithm>
#include <atomic>
#include <type_traits>
#include <utility>

#include "tsfa_internal.h"

namespace tsfa {
namespace bwd {

constexpr int kWaves = 8;                 // 4 key groups x 2 row groups
// kBlockKeys, kTileRows, kMaxStateInts: tsfa_plan.h
static_assert(kWaves * 64 == kMainThreads, "launch size");
constexpr int kBufs = 2;                  // Q / dO tile buffers per row group: loads run one step ahead

// 16-byte-chunk XOR swizzle of a row-major [rows][D] LDS tile (row period
// 16), conflict-free for both read patterns of the kernel:
//   * row reads (ds_read_b128, a quarter-wave reads chunk c of 16 rows): the
//     16 rows land on 16 distinct 16-byte bank slots;
//   * transposed reads (ds_read_b64_tr_b16, a half-wave reads 4 consecutive
//     rows x 64 bytes): the 4 rows land on 4 distinct 64-byte bank windows.
template <int D> __device__ inline int swz(int row) {
  if constexpr (D == 128) {
    return ((row & 3) << 2) | ((row >> 2) & 3);
  } else {
    const int j = row >> 1;
    return ((j & 1) << 2) | ((j >> 1) & 3);
  }
}

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // m0 is reserved; the clobber documents the write
// 16 bytes per active lane HBM -> LDS: lane i's bytes land at lds_base + 16*i.
__device__ inline void dma16(const void* src, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(src), "s"(lds_base)
               : "memory", "m0");
}
// The same with a scalar base and a 32-bit lane offset (no per-lane 64-bit
// address held in registers).
__device__ inline void dma16_s(const void* sbase, uint32_t voff, uint32_t lds_base) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(voff), "s"(sbase), "s"(lds_base)
               : "memory", "m0");
}
#pragma clang diagnostic pop

template <int N> __device__ inline void vm_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}
__device__ inline void sync_lds() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ inline uint32_t lds_addr(const void* p) { return (uint32_t)(uintptr_t)(const TSFA_LDS void*)p; }
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// LDS reads at addr + off (off: the instruction's immediate offset).
template <typename V> __device__ inline V lds_ld(uint32_t addr, int off = 0) {
  return *(const TSFA_LDS V*)((const TSFA_LDS char*)(uintptr_t)addr + off);
}
__device__ inline i16x4 lds_tr(uint32_t addr, int off) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((TSFA_LDS i16x4*)((TSFA_LDS char*)(uintptr_t)addr + off));
}
__device__ inline void fence_order() { __builtin_amdgcn_sched_barrier(0); }
template <typename V, typename U> __device__ inline V bit_cast(U u) { return __builtin_bit_cast(V, u); }

struct BwdArgs {
  const void* q;
  const void* k;
  const void* v;
  const void* dout;
  void* dk;
  void* dv;
  float* dq_acc;            // [B*Hkv][D][n_tiles*32] fp32 (d-major: a wave's atomics cover whole lines)
  const float* rowstat;     // [B*Hkv][n_tiles][2][32]: log2 LSE, then Dv, of the tile's rows
  const uint32_t* vis;      // [n_trees][n_tiles][n_tkeys] visibility words of tree keys
  int64_t sqb, sqh, sqm, skb, skh, skn, svb, svh, svn, sdob, sdoh, sdom, sdkb, sdkh, sdkn, sdvb, sdvh, sdvn;
  int64_t vis_tree_stride;  // 0: one tree for the batch
  float scale_log2;         // sm_scale * log2(e) (signed), never 0
  float dk_scale;           // sm_scale
  int num_kv_heads, group, q_len, kv_len, prefix_len;
  int n_tiles, n_pb, n_tb, n_tkeys;
  int n_items, items_per_xcd;
  uint32_t group_magic;     // floor(2^32 / group) + 1 (group > 1): R / group = umulhi(R, magic) for R < 2^21
  int tile_fast;            // whole Q / dO tiles at a scalar base + fixed 32-bit lane offsets (group divides 32)
  int key_fast;             // the same for whole 32-key K / V units
  // row-parallel dQ kernel
  void* dq;                 // dq_direct: the kernel writes sm_scale * dQ here (one split per chunk)
  int64_t sdqb, sdqh, sdqm;
  float dq_scale;
  int dq_direct;
  int n_pu, n_tu;           // prefix / tree units of 32 keys
  int n_chunks, n_splits, units_per_split, q_items, q_pairs_per_xcd;
  int dq_first;     // dQ workgroups before the dK / dV ones
  int first_block;  // of this launch (0, or the second pass's first block when they run one after the other)
};

typedef __attribute__((address_space(4))) BwdArgs KArgs;  // in the kernel's argument segment

template <int D> constexpr size_t kv_lds_bytes() {
  // K block | V block | 2 groups x kBufs x (Q tile, dO tile) | 2 x kBufs x 32 row stats |
  // 2 x kBufs x 128 mask words
  return 2 * (size_t)kBlockKeys * D * 2 + 2 * 2 * kBufs * (size_t)kTileRows * D * 2 + 2 * kBufs * kTileRows * 8 +
         2 * kBufs * kBlockKeys * 4;
}

// Workgroup = 8 waves: key group kg = wave & 3 owns keys key0 + 32kg + [0, 32);
// row group rg = wave >> 2 takes every other 32-row tile.  Each SIMD runs one
// wave of each row group, so one wave's softmax-like VALU work and LDS waits
// overlap the other's MFMAs.  Both groups accumulate dK^T / dV^T of the same
// keys; group 1 hands its sums to group 0 through LDS at the end.
//
// What bounds it: latency, not a pipe (MFMA busy 36 % and 8.6 VALU per MFMA
// at the 1024-token tree behind 16k keys when the step ran S and dP, then
// all of the softmax, then dV and dK: both waves of a SIMD sat in the same
// phase).  A tile now runs four MFMA groups with the VALU work between the
// MFMAs of the next group that does not need it -- S; dP with P's
// exponentials; dV with dS; dK -- and operands read RA / VA MFMAs ahead, in a
// fixed order.  Blocks whose 128 keys are all visible compile without the
// mask, and whole tiles of a group that divides 32 are addressed by a scalar
// base plus fixed lane offsets (the general path costs ~15 VALU per 1 KB
// load): 1.53 M -> 1.27 M cycles at that shape, 243 -> 105 VALU instructions
// per 32 MFMAs.
template <typename T, int D>
__device__ __forceinline__ void kv_role(const KArgs& a, const int blk, unsigned char* smem) {
  typedef typename Mma<T>::vec8 V8;
  constexpr int ROWB = D * 2;                 // bytes of one row
  constexpr int KSTEPS = D / 16;
  constexpr int DT = D / 32;
  constexpr int CPR = D / 8;                  // 16-byte chunks per row
  constexpr int RPL = 64 / CPR;               // rows per 1 KB load
  constexpr int TILE_B = kTileRows * ROWB;
  constexpr int KBLK_B = kBlockKeys * ROWB;
  constexpr int LPT = TILE_B / 1024;          // 1 KB loads per Q (or dO) tile
  constexpr int TPW = 2 * LPT / 4;            // tile loads per wave (4 waves per row group)
  constexpr int KPW = 2 * KBLK_B / 1024 / kWaves;  // K + V block loads per wave
  static_assert(kBufs == 2, "the exchange at the end reuses the K, V and tile areas");
  static_assert(TPW >= 1 && KPW >= 1 && 2 * LPT == TPW * 4, "load split");

  unsigned char* kblk = smem;
  unsigned char* vblk = kblk + KBLK_B;
  unsigned char* tiles = vblk + KBLK_B;  // group g, buffer s: Q at tiles + 2*(g*kBufs + s)*TILE_B, dO after
  float* rs = reinterpret_cast<float*>(tiles + 2 * 2 * kBufs * TILE_B);            // [g][s][2][32]
  uint32_t* visw = reinterpret_cast<uint32_t*>(rs + 2 * kBufs * 2 * kTileRows);    // [g][s][128]

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave & 3, rg = wave >> 2;
  const int ln = lane & 31, lh = lane >> 5;

  // XCD-aware item order: consecutive block ids go to different XCDs and each
  // XCD gets a contiguous item range, so the key blocks of one (b, kv head),
  // which read the same Q / dO tiles, share an L2.
  const int item = (blk & 7) * a.items_per_xcd + (blk >> 3);
  if (item >= a.n_items) return;
  const int nkb = a.n_pb + a.n_tb;
  const int kb = item % nkb;
  const int bk = item / nkb;
  const int kvh = bk % a.num_kv_heads, b = bk / a.num_kv_heads;
  const bool tree_blk = kb >= a.n_pb;
  const int tkb = kb - a.n_pb;
  const int key0 = tree_blk ? a.prefix_len + tkb * kBlockKeys : kb * kBlockKeys;
  const int key_end = tree_blk ? a.kv_len : a.prefix_len;  // keys of this block: [key0, min(key0 + 128, key_end))
  const int G = a.group;
  const int TG = a.q_len * G;
  const float sl2 = a.scale_log2;  // signed: exp2(s * sl2 - lse2) for either sign of sm_scale

  const T* kbase = static_cast<const T*>(a.k) + b * a.skb + kvh * a.skh;
  const T* vbase = static_cast<const T*>(a.v) + b * a.svb + kvh * a.svh;
  const T* qbase = static_cast<const T*>(a.q) + b * a.sqb + (int64_t)kvh * G * a.sqh;
  const T* dobase = static_cast<const T*>(a.dout) + b * a.sdob + (int64_t)kvh * G * a.sdoh;
  const float* rsbase = a.rowstat + (int64_t)bk * a.n_tiles * (2 * kTileRows);
  const uint32_t* visbase =
      a.vis + (int64_t)b * a.vis_tree_stride + (tree_blk ? (int64_t)tkb * kBlockKeys : 0);

  // K and V blocks HBM -> LDS (keys past the end repeat the last key; masked).
#pragma unroll
  for (int i = 0; i < KPW; ++i) {
    const int u = wave * KPW + i;  // 0 .. 2*KBLK_B/1024 - 1: K loads, then V loads
    const bool is_v = u >= KBLK_B / 1024;
    const int ul = is_v ? u - KBLK_B / 1024 : u;
    const int row = ul * RPL + lane / CPR, pos = lane % CPR;
    const int key = min(key0 + row, a.kv_len - 1);
    const T* src = (is_v ? vbase + (int64_t)key * a.svn : kbase + (int64_t)key * a.skn) + ((pos ^ swz<D>(row)) << 3);
    dma16(src, lds_addr((is_v ? vblk : kblk) + ul * 1024));
  }

  // The tiles of row group rg: step n handles tile 2n + rg.
  const int n_steps = (a.n_tiles + 1) >> 1;
  const int my_tiles = (a.n_tiles + 1 - rg) >> 1;  // steps with a tile for this group

  // Q / dO tile j -> this group's buffer s, with its row statistics (key
  // group 0) and, for tree blocks, the 128 keys' mask words (key group 1).
  // Key groups 0 and 1 move the Q tile, 2 and 3 the dO tile.  Rows past the
  // end repeat the last row; their statistics make P = dS = 0.
  const bool is_do = kg >= 2;
  const T* tbase = is_do ? dobase : qbase;
  const int64_t tsh = is_do ? a.sdoh : a.sqh, tsm = is_do ? a.sdom : a.sqm;
  auto load_row = [&](int i) { return ((kg & 1) * TPW + i) * RPL + lane / CPR; };
  uint32_t toff[TPW];  // tile_fast: lane byte offsets from the tile's first token
#pragma unroll
  for (int i = 0; i < TPW; ++i) {
    const int row = load_row(i), t = G == 1 ? row : row / G;
    toff[i] = (uint32_t)(((int64_t)(row - t * G) * tsh + (int64_t)t * tsm + (((lane % CPR) ^ swz<D>(row)) << 3)) * 2);
  }
  const int tpt = a.tile_fast ? kTileRows / G : 0;  // tokens per tile
  auto issue_tile = [&](int j, int s) {
    const uint32_t tl = lds_addr(tiles + 2 * (rg * kBufs + s) * TILE_B + (is_do ? TILE_B : 0) + (kg & 1) * TPW * 1024);
    if (a.tile_fast && (j + 1) * kTileRows <= TG) {
      const T* src = tbase + (int64_t)j * tpt * tsm;
#pragma unroll
      for (int i = 0; i < TPW; ++i) dma16_s(src, toff[i], tl + i * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        const int row = load_row(i);
        const int R = min(j * kTileRows + row, TG - 1);
        const int t = G == 1 ? R : (int)__umulhi((uint32_t)R, a.group_magic);
        const int g = R - t * G;
        dma16(tbase + g * tsh + (int64_t)t * tsm + (((lane % CPR) ^ swz<D>(row)) << 3), tl + i * 1024);
      }
    }
    if (kg == 0) {
      if (lane < 2 * kTileRows * 4 / 16)
        dma16_s(rsbase + (int64_t)j * (2 * kTileRows), 16u * lane, lds_addr(rs + (rg * kBufs + s) * 2 * kTileRows));
    } else if (kg == 1 && tree_blk) {
      if (lane < kBlockKeys * 4 / 16)
        dma16_s(visbase + (int64_t)j * a.n_tkeys, 16u * lane, lds_addr(visw + (rg * kBufs + s) * kBlockKeys));
    }
  };
  if (my_tiles > 0) issue_tile(rg, 0);

  const int mykey = key0 + 32 * kg + ln;
  const bool key_ok = mykey < key_end && mykey < key0 + kBlockKeys;
  const bool all_keys = !tree_blk && key0 + kBlockKeys <= key_end;  // every key visible to every row

  // LDS offsets (bytes).  Row reads: lane (row ln, lh) reads chunk 2kk + lh,
  // at r_off0 ^ (kk << 5).  Transposed reads: lane (x = lane>>4, i = lane&15)
  // reads 8 bytes of row 8jj + 4(x>>1) + (i>>2) (+16 per k-step) at d = dt*32
  // + 16(x&1) + 4(i&3), i.e. at (t_off0 ^ (dt << 6) ^ (jj << 5)) + 8jj rows
  // (8 rows on, the swizzle flips chunk bit 1); after the transpose it holds
  // rows +[0,4) of d = dt*32 + 16(x&1) + i.
  const int vx = lane >> 4, vi = lane & 15;
  const int trow = 4 * (vx >> 1) + (vi >> 2);
  const uint32_t r_off0 = (uint32_t)(ln * ROWB + ((lh ^ swz<D>(ln)) << 4));
  const uint32_t t_off0 =
      (uint32_t)(trow * ROWB + (((2 * (vx & 1) + ((vi & 3) >> 1)) ^ swz<D>(trow)) << 4) + ((vi & 1) << 3));
  const uint32_t kmine = lds_addr(kblk + 32 * kg * ROWB);  // V: KBLK_B further

  f32x16 dk[DT], dv[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) dk[dt][i] = dv[dt][i] = 0.f;

  // The wave's V operand (head_dim 64: K's too) stays in registers for the
  // whole walk (K's as well would take head_dim 128 past 256 registers).
  constexpr int KR = D == 64 ? 0 : KSTEPS;  // first operand pair whose key side is held
  i16x8 held[2 * KSTEPS - KR];
  vm_wait<0>();
  sync_lds();
#pragma unroll
  for (int x = KR; x < 2 * KSTEPS; ++x)
    held[x - KR] = lds_ld<i16x8>((kmine + r_off0) ^ (uint32_t)((x % KSTEPS) << 5), x < KSTEPS ? 0 : KBLK_B);

  // One tile from buffer s.  masked_c: tree blocks and the prefix's partial
  // last block (P = 0 for the lane's key where its mask bit is clear).
  auto tile_step = [&](auto masked_c, int s) {
    constexpr bool MASKED = decltype(masked_c)::value;
    constexpr int RA = 3;          // row-operand pairs read ahead
    constexpr int VA = 3;          // transposed pairs read ahead
    constexpr int EP = 16 / KSTEPS;  // P (dS) elements between two MFMAs
    constexpr int NG = 2 * DT;     // dV (dK) MFMAs
    static_assert(NG == KSTEPS, "one slice of P and of dS per MFMA");
    const uint32_t qt = lds_addr(tiles + 2 * (rg * kBufs + s) * TILE_B);
    // (read offsets formed anew each tile: hoisted out of the loop they spill)
    uint32_t q0 = qt + r_off0, k0 = kmine + r_off0, t0 = qt + t_off0;
    asm volatile("" : "+v"(q0), "+v"(k0), "+v"(t0));
    const uint32_t st = lds_addr(rs + (rg * kBufs + s) * 2 * kTileRows) + 16u * lh;
    uint32_t w = 0;
    if constexpr (MASKED) {
      w = key_ok ? 0xffffffffu : 0u;
      if (tree_blk) w &= visw[(rg * kBufs + s) * kBlockKeys + 32 * kg + ln];
      w >>= 4 * lh;
    }
    // S = Q K^T, dP = dO V^T: M = rows, N = keys; lane (key ln, lh) holds
    // rows 8(i/4) + 4lh + i%4 of its key.  Operand pair x: S's k-steps, then dP's.
    i16x8 fa[2 * KSTEPS], fb[2 * KSTEPS];
    auto rd = [&](int x) {
      const uint32_t c = (uint32_t)((x % KSTEPS) << 5);
      fa[x] = lds_ld<i16x8>(q0 ^ c, x < KSTEPS ? 0 : TILE_B);
      if (x >= KR) fb[x] = held[x - KR];
      else fb[x] = lds_ld<i16x8>(k0 ^ c);
    };
    // transposed pair x: dO's NG, then Q's (one LDS copy serves both reads)
    i16x4 tl[2 * NG], th[2 * NG];
    auto rt = [&](int x) {
      const int g = x % NG, dt = g >> 1, s2 = g & 1;
      const uint32_t c = t0 ^ (uint32_t)(dt << 6);
      const int off = (x < NG ? TILE_B : 0) + 16 * s2 * ROWB;
      tl[x] = lds_tr(c, off);
      th[x] = lds_tr(c ^ 32u, off + 8 * ROWB);
    };
    auto tr = [&](int x) { return bit_cast<V8>(__builtin_shufflevector(tl[x], th[x], 0, 1, 2, 3, 4, 5, 6, 7)); };
    f32x4 lse4[4], dv4[4];  // statistics of the lane's rows 8q + 4lh + [0, 4)
    f32x16 sc, dp;
    V8 pb[2], db[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) sc[i] = dp[i] = 0.f;
    auto p_slice = [&](int y) {
#pragma unroll
      for (int i = EP * y; i < EP * (y + 1); ++i) {
        float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[i], sl2, -lse4[i >> 2][i & 3]));
        if constexpr (MASKED) p = ((w >> (8 * (i >> 2) + (i & 3))) & 1u) ? p : 0.f;
        sc[i] = p;
        pb[i >> 3][i & 7] = (T)p;
      }
    };
    auto ds_slice = [&](int y) {
#pragma unroll
      for (int i = EP * y; i < EP * (y + 1); ++i) db[i >> 3][i & 7] = (T)(sc[i] * (dp[i] - dv4[i >> 2][i & 3]));
    };
#pragma unroll
    for (int x = 0; x < RA; ++x) rd(x);
#pragma unroll
    for (int q = 0; q < 4; ++q) lse4[q] = lds_ld<f32x4>(st, 32 * q);
    fence_order();
#pragma unroll
    for (int x = 0; x < KSTEPS; ++x) {
      rd(x + RA);
      sc = Mma<T>::run(bit_cast<V8>(fa[x]), bit_cast<V8>(fb[x]), sc);
      fence_order();
    }
#pragma unroll
    for (int x = KSTEPS; x < 2 * KSTEPS; ++x) {
      if (x + RA < 2 * KSTEPS) rd(x + RA);
      else rt(x + RA - 2 * KSTEPS);
      dp = Mma<T>::run(bit_cast<V8>(fa[x]), bit_cast<V8>(fb[x]), dp);
      if (x > KSTEPS) p_slice(x - KSTEPS - 1);
      fence_order();
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) dv4[q] = lds_ld<f32x4>(st, 4 * kTileRows + 32 * q);
    // dV^T += dO^T P, dK^T += Q^T dS: M = d, N = keys, k-step s2 covers rows
    // 16s2 + 8(e/4) + 4lh + e%4 -- elements 8s2 .. 8s2+7 of the accumulator.
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      rt(g + VA);
      dv[g >> 1] = Mma<T>::run(tr(g), pb[g & 1], dv[g >> 1]);
      if (g == 0) p_slice(KSTEPS - 1);
      else ds_slice(g - 1);
      fence_order();
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      if (g + VA < NG) rt(NG + g + VA);
      dk[g >> 1] = Mma<T>::run(tr(NG + g), db[g & 1], dk[g >> 1]);
      if (g == 0) ds_slice(NG - 1);
      fence_order();
    }
  };

  // (one loop per kind of block, no branch around a step: a merge of
  // accumulators inside the loop costs copies of all of them)
  auto walk = [&](auto masked_c) {
    for (int n = 0; n < my_tiles; ++n) {
      const int s = n & (kBufs - 1);
      // This group's tile of step n landed (and on the first step the K / V
      // blocks); every wave is done with step n-1, whose buffers step n+1's
      // tiles load into.
      vm_wait<0>();
      sync_lds();
      if (n + 1 < my_tiles) issue_tile(2 * (n + 1) + rg, s ^ 1);
      tile_step(masked_c, s);
    }
  };
  if (all_keys) walk(std::false_type{});
  else walk(std::true_type{});
  if (my_tiles < n_steps) {  // group 1 has no tile on the last step of an odd count
    vm_wait<0>();            // (a single tile: its share of the K / V blocks)
    sync_lds();
  }

  // Row group 1 hands dK^T / dV^T to row group 0 through LDS (the K / V
  // blocks and tile buffers at the start of LDS are free now): register r of
  // lane l at xch[kg][r][l].
  vm_wait<0>();
  sync_lds();
  float* xch = reinterpret_cast<float*>(smem);
  static_assert(4 * 2 * DT * 16 * 64 * 4 <= 2 * KBLK_B + 2 * 2 * kBufs * TILE_B, "exchange fits in K, V and tiles");
  float* xw = xch + kg * (2 * DT * 16 * 64);
  if (rg == 1) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        xw[((2 * dt) * 16 + i) * 64 + lane] = dk[dt][i];
        xw[((2 * dt + 1) * 16 + i) * 64 + lane] = dv[dt][i];
      }
  }
  sync_lds();
  if (rg == 1) return;

  // dK = sm_scale dK^T, dV = dV^T: lane (key ln, lh) holds d = dt*32 +
  // 8(i/4) + 4lh + i%4 of its key.
  if (key_ok) {
    T* dkp = static_cast<T*>(a.dk) + b * a.sdkb + kvh * a.sdkh + (int64_t)mykey * a.sdkn + 4 * lh;
    T* dvp = static_cast<T*>(a.dv) + b * a.sdvb + kvh * a.sdvh + (int64_t)mykey * a.sdvn + 4 * lh;
    typedef T T4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        T4 x, y;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int i = 4 * q + e;
          x[e] = (T)((dk[dt][i] + xw[((2 * dt) * 16 + i) * 64 + lane]) * a.dk_scale);
          y[e] = (T)(dv[dt][i] + xw[((2 * dt + 1) * 16 + i) * 64 + lane]);
        }
        *reinterpret_cast<T4*>(dkp + dt * 32 + 8 * q) = x;
        *reinterpret_cast<T4*>(dvp + dt * 32 + 8 * q) = y;
      }
  }
}

// ------------------------------------------------------------- dQ kernel
constexpr int kQWaves = 4;   // 32 rows each: 128-row chunks
constexpr int kRing = 4;     // LDS ring stages of 32-key units

template <int D> constexpr size_t dq_lds_bytes() {
  // kRing x (K unit, V unit, mask words of the chunk's 4 row tiles x 32 keys, padded to 256 bytes)
  return (size_t)kRing * (2 * 32 * D * 2 + 4 * 32 * 4);
}

// Wait until at most k units (LPU loads each) of this wave are in flight.
template <int LPU, int K> __device__ inline void wait_units(int k) {
  if constexpr (K == 0) {
    vm_wait<0>();
  } else {
    if (k >= K) {
      vm_wait<K * LPU>();
      return;
    }
    wait_units<LPU, K - 1>(k);
  }
}

// Row-parallel dQ: half a workgroup owns a 128-row chunk of one (b, kv head) (one
// 32-row tile per wave, Q and dO fragments in registers) and one split of its
// 32-key units (prefix units, then the tree units), streamed through a
// 4-stage LDS ring.  Per unit, on v_mfma_f32_32x32x16:
//   S^T = K Q^T and dP^T = V dO^T (a lane holds one row, so its LSE and Dv
//   are scalars), P^T and dS^T on the VALU, then dQ^T += K^T dS^T with dS^T
//   taken straight from the accumulator (k order permuted to the order it
//   holds keys in; K^T from ds_read_b64_tr_b16 in the same order).
// The workgroup's dQ^T adds to the fp32 accumulator once at the end
// (atomics: several splits of one chunk add to the same rows).
//
// What bounds it: VALU issue and latency (40 % MFMA busy, 10.5 VALU per MFMA
// at the 1024-token tree behind 16k keys when every unit built and tested a
// visibility bit per score and the softmax sat between the MFMA groups).  A
// unit runs S^T; dP^T with the exponentials between its MFMAs; dQ^T's first
// half with the second half's dS between; whole prefix units compile
// without the visibility tests and load at a scalar base plus fixed lane
// offsets: 1.04 M -> 0.78 M cycles at that shape, 227 -> 88 VALU instructions
// per 24 MFMAs.
template <typename T, int D>
__device__ __forceinline__ void dq_role(const KArgs& a, const int blk, unsigned char* smem) {
  typedef typename Mma<T>::vec8 V8;
  constexpr int ROWB = D * 2;
  constexpr int KSTEPS = D / 16;
  constexpr int DT = D / 32;
  constexpr int CPR = D / 8;
  constexpr int RPL = 64 / CPR;
  constexpr int HALF = 32 * ROWB;          // K (or V) bytes of one unit
  constexpr int VISB = 4 * 32 * 4;         // mask words of the chunk's 4 row tiles for the unit's 32 keys
  constexpr int SB = 2 * HALF + VISB;      // ring stage
  constexpr int LPH = HALF / 1024;         // 1 KB loads per half
  constexpr int UPW = 2 * LPH / kQWaves;   // K + V loads per wave per unit (wave 0 of a tree unit: one more)
  static_assert(UPW >= 1 && UPW * kQWaves == 2 * LPH && SB % 256 == 0, "load split, aligned stages");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int half = __builtin_amdgcn_readfirstlane(tid >> 8);
  const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);
  unsigned char* ring = smem + half * kRing * SB;
  const int ln = lane & 31, lh = lane >> 5;

  // item order: chunk fastest (the chunks of one (b, kv head) read the same
  // K / V units), XCD-aware as in the forward
  const int pair = (blk & 7) * a.q_pairs_per_xcd + (blk >> 3);
  if (2 * pair >= a.q_items) return;
  const int item = min(2 * pair + half, a.q_items - 1);
  const bool live = 2 * pair + half < a.q_items;
  const int chunk = item % a.n_chunks;
  int rest = item / a.n_chunks;
  const int sp = rest % a.n_splits;
  const int bk = rest / a.n_splits;
  const int kvh = bk % a.num_kv_heads, b = bk / a.num_kv_heads;
  const int G = a.group;
  const int TG = a.q_len * G;
  const int TGP = a.n_tiles * kTileRows;
  const int P = a.prefix_len;
  const float sl2 = a.scale_log2;
  const int tile = chunk * kQWaves + wave;     // this wave's 32-row tile
  const bool active = live && tile < a.n_tiles;
  const int r = tile * kTileRows + ln;         // this lane's row
  const int n_units = a.n_pu + a.n_tu;
  const int u_lo = sp * a.units_per_split;
  const int mine = live ? max(0, min(a.units_per_split, n_units - u_lo)) : 0;
  // steps of the workgroup: the longer half's (the halves share its barriers)
  const int sp0 = (2 * pair) / a.n_chunks % a.n_splits, sp1 = min(2 * pair + 1, a.q_items - 1) / a.n_chunks % a.n_splits;
  const int n_wg = min(a.units_per_split, n_units - min(sp0, sp1) * a.units_per_split);

  const T* kbase = static_cast<const T*>(a.k) + b * a.skb + kvh * a.skh;
  const T* vbase = static_cast<const T*>(a.v) + b * a.svb + kvh * a.svh;
  const uint32_t* visbase = a.vis + (int64_t)b * a.vis_tree_stride;

  // Q^T and dO^T operands (B[d][row]: lane (row ln, lh) holds d = 16kk + 8lh
  // + [0, 8)) and the row's statistics, in registers for the whole walk.
  // Loaded before any ring load and consumed at once, so the compiler's wait
  // for them covers nothing else.
  i16x8 qf[KSTEPS], df[KSTEPS];
  float lse2 = INFINITY, dvr = 0.f;
  {
    const int R = min(r, TG - 1);
    const int t = R / G, g = R - t * G;
    const T* qp = static_cast<const T*>(a.q) + b * a.sqb + (int64_t)(kvh * G + g) * a.sqh + (int64_t)t * a.sqm + 8 * lh;
    const T* dp = static_cast<const T*>(a.dout) + b * a.sdob + (int64_t)(kvh * G + g) * a.sdoh +
                  (int64_t)t * a.sdom + 8 * lh;
#pragma unroll
    for (int kk = 0; kk < KSTEPS; ++kk) {
      qf[kk] = *reinterpret_cast<const i16x8*>(qp + 16 * kk);
      df[kk] = *reinterpret_cast<const i16x8*>(dp + 16 * kk);
    }
    if (active) {
      const float* st = a.rowstat + ((int64_t)bk * a.n_tiles + tile) * (2 * kTileRows) + ln;
      lse2 = st[0];  // padding rows: +inf, 0
      dvr = st[kTileRows];
    }
#pragma unroll
    for (int kk = 0; kk < KSTEPS; ++kk) asm volatile("" : : "v"(qf[kk]), "v"(df[kk]));
    asm volatile("" : : "v"(lse2), "v"(dvr));
  }

  auto key0_of = [&](int u) { return u < a.n_pu ? 32 * u : P + 32 * (u - a.n_pu); };
  // HBM -> LDS: this wave's share of unit u into stage st (waves 0, 1 move
  // K, 2, 3 V).
  const bool is_v = wave >= kQWaves / 2;
  const T* ubase = is_v ? vbase : kbase;
  const int64_t ustride = is_v ? a.svn : a.skn;
  const int urow0 = (wave % (kQWaves / 2)) * UPW * RPL;
  uint32_t uoff[UPW];  // key_fast: lane byte offsets from the unit's first key
#pragma unroll
  for (int i = 0; i < UPW; ++i) {
    const int row = urow0 + i * RPL + lane / CPR;
    uoff[i] = (uint32_t)(((int64_t)row * ustride + (((lane % CPR) ^ swz<D>(row)) << 3)) * 2);
  }
  auto issue = [&](int st, int u) {
    unsigned char* sb = ring + st * SB;
    const int key0 = key0_of(u);
    const uint32_t dst = lds_addr(sb + (is_v ? HALF : 0) + (wave % (kQWaves / 2)) * UPW * 1024);
    if (a.key_fast && key0 + 32 <= a.kv_len) {
      const T* src = ubase + (int64_t)key0 * ustride;
#pragma unroll
      for (int i = 0; i < UPW; ++i) dma16_s(src, uoff[i], dst + i * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < UPW; ++i) {
        const int row = urow0 + i * RPL + lane / CPR;
        const int key = min(key0 + row, a.kv_len - 1);
        dma16(ubase + (int64_t)key * ustride + (((lane % CPR) ^ swz<D>(row)) << 3), dst + i * 1024);
      }
    }
    if (wave == 0 && u >= a.n_pu) {
      // words [tile][tree key]: 4 tiles x 32 keys x 4 B, 8 lanes per tile
      if (lane < 32) {
        const int jt = min(chunk * kQWaves + (lane >> 3), a.n_tiles - 1);
        dma16(visbase + (int64_t)jt * a.n_tkeys + 32 * (u - a.n_pu) + 4 * (lane & 7), lds_addr(sb + 2 * HALF));
      }
    }
  };

  // LDS offsets: row reads of K / V (lane (key ln, lh), chunk 2kk + lh) at
  // r_off0 ^ (kk << 5), transposed reads of K (rows 8jj + 4(x>>1) + (i>>2), d
  // = dt*32 + 16(x&1) + 4(i&3)) at (t_off0 ^ (dt << 6) ^ (jj << 5)) + 8jj
  // rows; the tiles use the same swizzle as the dK / dV kernel.
  const int vx = lane >> 4, vi = lane & 15;
  const int trow = 4 * (vx >> 1) + (vi >> 2);
  const uint32_t r_off0 = (uint32_t)(ln * ROWB + ((lh ^ swz<D>(ln)) << 4));
  const uint32_t t_off0 =
      (uint32_t)(trow * ROWB + (((2 * (vx & 1) + ((vi & 3) >> 1)) ^ swz<D>(trow)) << 4) + ((vi & 1) << 3));

  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[dt][i] = 0.f;

  // One unit from the stage at LDS address sb.  masked_c: tree units and the
  // prefix's partial last unit (vis16: the lane's 16 keys).
  auto unit_step = [&](auto masked_c, uint32_t sb, uint32_t vis16) {
    constexpr bool MASKED = decltype(masked_c)::value;
    constexpr int RA = 4;            // row-operand reads ahead of their MFMA
    constexpr int EP = 16 / KSTEPS;  // elements of P between two MFMAs
    // (read offsets formed anew each unit, as in the dK / dV kernel)
    uint32_t r0 = sb + r_off0, t0 = sb + t_off0;
    asm volatile("" : "+v"(r0), "+v"(t0));
    // operand x: K's k-steps (S^T), then V's (dP^T)
    i16x8 f[2 * KSTEPS];
    auto rd = [&](int x) {
      f[x] = lds_ld<i16x8>(r0 ^ (uint32_t)((x % KSTEPS) << 5), x < KSTEPS ? 0 : HALF);
    };
    // transposed K pair x = s2 * DT + dt
    i16x4 tl[2 * DT], th[2 * DT];
    auto rt = [&](int x) {
      const uint32_t c = t0 ^ (uint32_t)((x % DT) << 6);
      tl[x] = lds_tr(c, 16 * (x / DT) * ROWB);
      th[x] = lds_tr(c ^ 32u, (16 * (x / DT) + 8) * ROWB);
    };
    // S^T = K Q^T, dP^T = V dO^T: M = keys, N = rows; lane (row ln, lh)
    // holds keys 8(i/4) + 4lh + i%4.
    f32x16 sc, dp;
    V8 db[2];
#pragma unroll
    for (int i = 0; i < 16; ++i) sc[i] = dp[i] = 0.f;
    auto p_slice = [&](int y) {
#pragma unroll
      for (int i = EP * y; i < EP * (y + 1); ++i) {
        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(sc[i], sl2, -lse2));
        sc[i] = MASKED && !((vis16 >> i) & 1u) ? 0.f : p;
      }
    };
    auto ds = [&](int i) { db[i >> 3][i & 7] = (T)(sc[i] * (dp[i] - dvr)); };
#pragma unroll
    for (int x = 0; x < RA; ++x) rd(x);
    fence_order();
#pragma unroll
    for (int x = 0; x < KSTEPS; ++x) {
      rd(x + RA);
      sc = Mma<T>::run(bit_cast<V8>(f[x]), bit_cast<V8>(qf[x]), sc);
      fence_order();
    }
#pragma unroll
    for (int x = KSTEPS; x < 2 * KSTEPS; ++x) {
      if (x + RA < 2 * KSTEPS) rd(x + RA);
      else if (x + RA - 2 * KSTEPS < 2 * DT) rt(x + RA - 2 * KSTEPS);
      dp = Mma<T>::run(bit_cast<V8>(f[x]), bit_cast<V8>(df[x - KSTEPS]), dp);
      if (x > KSTEPS) p_slice(x - KSTEPS - 1);
      fence_order();
    }
    p_slice(KSTEPS - 1);
#pragma unroll
    for (int i = 0; i < 8; ++i) ds(i);
    // dQ^T += K^T dS^T: M = d, N = rows, k-step s2 covers keys 16s2 + 8(e/4)
    // + 4lh + e%4 -- elements 8s2 .. 8s2+7 of the accumulator.
#pragma unroll
    for (int x = 0; x < 2 * DT; ++x) {
      if (x + RA < 2 * DT) rt(x + RA);
      const i16x8 kT = __builtin_shufflevector(tl[x], th[x], 0, 1, 2, 3, 4, 5, 6, 7);
      acc[x % DT] = Mma<T>::run(bit_cast<V8>(kT), db[x / DT], acc[x % DT]);
      if (x < DT) {
#pragma unroll
        for (int i = 8 + 8 / DT * x; i < 8 + 8 / DT * (x + 1); ++i) ds(i);
      }
      fence_order();
    }
  };

  auto step = [&](int j) {
    // The waves meet before every second unit: units j and j+1 landed for
    // every wave (at first kRing-2 later units in flight, at least UPW loads
    // each), and every wave is done with units j-2 and j-1, whose stages the
    // next two reuse.  A barrier per unit, with K and V read from LDS for
    // every tile of the dK / dV role: the 1024-token tree behind 16k keys 957
    // us, 936 without; 4 head_dim 64 sequences of 300 tokens 91.6 -> 87.4.
    if ((j & 1) == 0) {
      wait_units<UPW, kRing - 2>(j == 0 ? max(0, min(mine - 2, kRing - 2)) : 0);
      sync_lds();
      if (j > 0) {
        if (j + kRing - 2 < mine) issue((j + kRing - 2) % kRing, u_lo + j + kRing - 2);
        if (j + kRing - 1 < mine) issue((j + kRing - 1) % kRing, u_lo + j + kRing - 1);
      }
    }
    return lds_addr(ring + (j % kRing) * SB);
  };
  for (int j = 0; j < kRing && j < mine; ++j) issue(j, u_lo + j);
  // whole prefix units, then the masked ones (a loop each: a merge of
  // accumulators inside a loop costs copies of all of them)
  const int n_full = min(max(P / 32 - u_lo, 0), mine);
  if (active) {
    for (int j = 0; j < n_full; ++j) unit_step(std::false_type{}, step(j), 0u);
    for (int j = n_full; j < mine; ++j) {
      const uint32_t sb = step(j);
      const int u = u_lo + j;
      // visibility of the lane's 16 keys from its row: prefix keys below P;
      // tree keys: bit ln of each key's word for this wave's tile
      uint32_t vis16 = 0;
      if (u >= a.n_pu) {
        const uint32_t wv = sb + 2 * HALF + wave * 128 + 16 * lh;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const u32x4 w4 = lds_ld<u32x4>(wv, 32 * q);
          vis16 |= ((w4[0] >> ln) & 1u) << (4 * q + 0);
          vis16 |= ((w4[1] >> ln) & 1u) << (4 * q + 1);
          vis16 |= ((w4[2] >> ln) & 1u) << (4 * q + 2);
          vis16 |= ((w4[3] >> ln) & 1u) << (4 * q + 3);
        }
      } else {
        const int key0 = 32 * u;
#pragma unroll
        for (int i = 0; i < 16; ++i) vis16 |= (uint32_t)(key0 + 8 * (i >> 2) + 4 * lh + (i & 3) < P) << i;
      }
      unit_step(std::true_type{}, sb, vis16);
    }
  } else {
    for (int j = 0; j < mine; ++j) step(j);
  }
  for (int j = (mine + 1) / 2; j < (n_wg + 1) / 2; ++j) sync_lds();
  // lane (row ln, lh) holds d = dt*32 + 8(i/4) + 4lh + i%4.  One split per
  // chunk: the workgroup owns its rows' dQ and writes it in the input dtype.
  // Otherwise it adds to the d-major fp32 accumulator (each instruction's 64
  // lanes cover two whole 128-byte lines).
  if (active && mine > 0) {
    if (a.dq_direct) {
      if (r < TG) {
        const int t = r / G, g = r - t * G;
        T* dst = static_cast<T*>(a.dq) + b * a.sdqb + (int64_t)(kvh * G + g) * a.sdqh + (int64_t)t * a.sdqm + 4 * lh;
        typedef T T4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            T4 x;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = (T)(acc[dt][4 * q + e] * a.dq_scale);
            *reinterpret_cast<T4*>(dst + dt * 32 + 8 * q) = x;
          }
      }
    } else {
      float* dq = a.dq_acc + ((int64_t)bk * D + 4 * lh) * TGP + r;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int i = 0; i < 16; ++i)
          atomicAdd(dq + (int64_t)(dt * 32 + 8 * (i >> 2) + (i & 3)) * TGP, acc[dt][i]);
    }
  }
}

// The two passes in one launch, so the second one's workgroups fill the CUs
// that the first one's last round leaves idle (dq_split_plan: which is first).
// Two launches, the second on a side stream forked and joined by events, cost
// 46 us of host time per call against 10 us, so short training steps were
// bound by it (8B shape, one layer's step: 196 -> 145 us), and the fork and
// join on the device (its backward in a graph 59 -> 52 us; the 1024-token
// tree's 1160 -> 991 with the loops above).  A dQ workgroup is two halves of
// four waves with a row chunk and a ring each, as two workgroups per CU were.
template <typename T, int D>
__global__ __launch_bounds__(kWaves * 64) __attribute__((amdgpu_waves_per_eu(2, 2)))
void bwd_main_kernel(const BwdArgs a) {
  extern __shared__ __attribute__((aligned(256))) unsigned char smem[];  // tile bases keep bits 0-7 clear
  const int id = blockIdx.x + a.first_block;
  const int n_first = 8 * (a.dq_first ? a.q_pairs_per_xcd : a.items_per_xcd);
  const int blk = id < n_first ? id : id - n_first;
  // each role reads the arguments through a pointer of its own: loads hoisted
  // above the branch for both spill SGPRs
  const KArgs* ap = (const KArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  if ((id < n_first) != (a.dq_first != 0)) {
    asm volatile("" : "+s"(ap));
    kv_role<T, D>(*ap, blk, smem);
  } else {
    asm volatile("" : "+s"(ap));
    dq_role<T, D>(*ap, blk, smem);
  }
}

template <int D> constexpr size_t main_lds_bytes() {
  return kv_lds_bytes<D>() > 2 * dq_lds_bytes<D>() ? kv_lds_bytes<D>() : 2 * dq_lds_bytes<D>();
}

// ------------------------------------------------------------ prep / dq / vis
struct PrepArgs {
  const void* o;
  const void* dout;
  const float* lse;  // [B, Hq, q_len]
  float* rowstat;    // [B*Hkv][n_tiles][2][32]: log2 LSE, then Dv
  float* dq_acc;     // [B*Hkv][D][TGP]
  int64_t sob, soh, som, sdob, sdoh, sdom;
  int batch, num_heads, num_kv_heads, group, q_len, n_tiles;
  int zero_dq;       // clear the accumulator (the dQ kernel adds into it)
};

// 16 lanes per row of the padded row space B*Hkv*TGP (workgroup `blk` of the
// prep range).
template <typename T, int D>
__device__ inline void bwd_prep(const PrepArgs& a, int blk) {
  constexpr int EPL = D / 16;  // elements per lane
  const int64_t gid = (int64_t)blk * 256 + threadIdx.x;
  const int64_t row = gid >> 4;
  const int part = (int)(gid & 15);
  const int TG = a.q_len * a.group;
  const int TGP = a.n_tiles * kTileRows;
  const int64_t nrows = (int64_t)a.batch * a.num_kv_heads * TGP;
  const bool live = row < nrows;
  const int64_t bk = live ? row / TGP : 0;
  const int R = live ? (int)(row - bk * TGP) : 0;
  const bool real = live && R < TG;
  float acc = 0.f, lse = -INFINITY;
  if (real) {
    const int t = R / a.group, g = R - t * a.group;
    const int kvh = (int)(bk % a.num_kv_heads), b = (int)(bk / a.num_kv_heads);
    const int h = kvh * a.group + g;
    typedef T TV __attribute__((ext_vector_type(EPL)));
    const TV ov = *reinterpret_cast<const TV*>(static_cast<const T*>(a.o) + b * a.sob + (int64_t)h * a.soh +
                                               (int64_t)t * a.som + part * EPL);
    const TV dv = *reinterpret_cast<const TV*>(static_cast<const T*>(a.dout) + b * a.sdob + (int64_t)h * a.sdoh +
                                               (int64_t)t * a.sdom + part * EPL);
#pragma unroll
    for (int e = 0; e < EPL; ++e) acc += (float)ov[e] * (float)dv[e];
    lse = a.lse[((int64_t)b * a.num_heads + h) * a.q_len + t];
  }
  if (a.zero_dq) {  // the block's 16 * D floats of the accumulator, whatever rows they are
    f32x4* z = reinterpret_cast<f32x4*>(a.dq_acc + (int64_t)blk * 16 * D) + threadIdx.x;
#pragma unroll
    for (int e = 0; e < EPL / 4; ++e) z[e * 256] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int off = 8; off >= 1; off >>= 1) acc += __shfl_xor(acc, off, 16);
  if (live && part == 0) {
    const bool empty = !(lse > -INFINITY);  // no visible key (or a padding row)
    float* st = a.rowstat + (row / kTileRows) * (2 * kTileRows) + row % kTileRows;
    st[0] = empty ? INFINITY : lse * 1.4426950408889634f;
    st[kTileRows] = empty ? 0.f : acc;
  }
}

struct DqArgs {
  const float* dq_acc;  // [B*Hkv][D][tgp]
  void* dq;
  int64_t sqb, sqh, sqm;
  float scale;
  int batch, num_kv_heads, group, q_len, tgp;
};

// Thread (bk, part, R), R fastest: 8 d of one row, read d-major (coalesced
// across the threads of a part).
template <typename T, int D>
__global__ __launch_bounds__(256) void bwd_dq_kernel(const DqArgs a) {
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int TG = a.q_len * a.group;
  const int64_t per_bk = (int64_t)(D / 8) * TG;
  if (gid >= (int64_t)a.batch * a.num_kv_heads * per_bk) return;
  const int64_t bk = gid / per_bk;
  const int rem = (int)(gid - bk * per_bk);
  const int part = rem / TG, R = rem - part * TG;
  const int t = R / a.group, g = R - t * a.group;
  const int kvh = (int)(bk % a.num_kv_heads), b = (int)(bk / a.num_kv_heads);
  const float* src = a.dq_acc + ((int64_t)bk * D + part * 8) * a.tgp + R;
  typedef T T8 __attribute__((ext_vector_type(8)));
  T8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] = (T)(src[(int64_t)e * a.tgp] * a.scale);
  *reinterpret_cast<T8*>(static_cast<T*>(a.dq) + b * a.sqb + (int64_t)(kvh * a.group + g) * a.sqh +
                         (int64_t)t * a.sqm + part * 8) = o;
}

struct VisArgs {
  const int32_t* row_ptr;
  const int32_t* col_idx;
  const int8_t* blk_type;
  const int32_t* payload;
  const int32_t* offset;
  int64_t ms_row_ptr, ms_col_idx, ms_blk_type, ms_payload, ms_offset;
  uint32_t* vis;  // [n_trees][n_tiles][n_tkeys]
  int64_t tree_stride;
  int group, q_len, block_m, block_n, n_tree_blocks, tree_key_limit, n_tiles, n_tkeys;
};

// One workgroup per (tile, tree, 64 tree keys): the block states of the
// tile's q-blocks (0 ZERO, -1 FULL, 1 + offset MIXED) expand into LDS, then
// each thread decides one (key, row) bit and a ballot assembles the 32-row
// words (lanes 0-31: one key, lanes 32-63: the next).
__device__ inline void bwd_vis(const VisArgs& a, int tile, int tree, int zc, int* st, int* rps) {
  const int c0 = zc * 64;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int G = a.group, BM = a.block_m, BN = a.block_n, ntb = a.n_tree_blocks;
  const int TG = a.q_len * G;
  const int r_lo = tile * kTileRows;
  const int r_hi = min(r_lo + kTileRows, TG) - 1;
  uint32_t* out = a.vis + (int64_t)tree * a.tree_stride + (int64_t)tile * a.n_tkeys;
  const int qb_lo = (r_lo / G) / BM, qb_hi = (r_hi / G) / BM, nqbc = qb_hi - qb_lo + 1;
  const int32_t* rp = a.row_ptr + tree * a.ms_row_ptr;
  const int32_t* ci = a.col_idx + tree * a.ms_col_idx;
  const int8_t* bt = a.blk_type + tree * a.ms_blk_type;
  const int32_t* pl = a.payload + tree * a.ms_payload;
  const int32_t* of = a.offset + tree * a.ms_offset;
  for (int i = tid; i < nqbc * ntb; i += 256) st[i] = 0;
  if (tid <= nqbc) rps[tid] = rp[qb_lo + tid];
  __syncthreads();
  for (int e = rps[0] + tid; e < rps[nqbc]; e += 256) {
    int qq = 0;
    while (qq + 1 < nqbc && rps[qq + 1] <= e) ++qq;
    const int tb = ci[e];
    // a block of any kind but MIXED is FULL (tree_sparse_flashattn.py:313-318)
    if (tb >= 0 && tb < ntb) st[qq * ntb + tb] = (bt[e] != TSFA_MIXED_BLOCK) ? -1 : (of[e] + 1);
  }
  __syncthreads();
  const int R = r_lo + (lane & 31);
  const int t = R / G, qb = t / BM;
#pragma unroll
  for (int pass = 0; pass < 8; ++pass) {
    const int c = c0 + pass * 8 + wave * 2 + (lane >> 5);  // this thread's tree key
    bool bit = false;
    if (R <= r_hi && c < a.tree_key_limit) {
      const int tb = c / BN;
      const int e = st[(qb - qb_lo) * ntb + tb];
      bit = e < 0;
      if (e > 0) {
        const int flat = (t - qb * BM) * BN + (c - tb * BN);
        bit = ((uint32_t)pl[e - 1 + (flat >> 5)] >> (flat & 31)) & 1u;
      }
    }
    const uint64_t bal = __ballot(bit);
    if ((lane & 31) == 0 && c < a.n_tkeys) out[c] = (uint32_t)(bal >> (lane & 32));
  }
}

// (The state table is sized to the tree and the accumulator cleared in whole
// lines: with 32 KB of LDS per block and 4-byte stores a row stride apart this
// launch took 25 us at the 1024-token tree behind 16k keys, 18.5 now.)
// Prep and visibility words in one launch: blocks [0, prep_blocks) run the
// prep, the rest one (tile, tree, 64-key chunk) of the visibility words each.
template <typename T, int D>
__global__ __launch_bounds__(256) void bwd_prep_vis_kernel(const PrepArgs pa, const VisArgs va, int prep_blocks,
                                                           int vis_chunks) {
  extern __shared__ int st[];  // block states of a visibility tile
  __shared__ int rps[72];
  const int blk = blockIdx.x;
  if (blk < prep_blocks) {
    bwd_prep<T, D>(pa, blk);
    return;
  }
  const int v = blk - prep_blocks;
  const int zc = v % vis_chunks, rest = v / vis_chunks;
  bwd_vis(va, rest % va.n_tiles, rest / va.n_tiles, zc, st, rps);
}

// ------------------------------------------------------------------- host
template <typename T, int D>
int launch_bwd(const BwdArgs& ba, const PrepArgs& pa, const VisArgs& va, const DqArgs& da, const BwdPlan& p,
               bool has_tree, hipStream_t stream) {
  static std::atomic<uint64_t> attr_set{0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return TSFA_ERR_DEVICE;
  const uint64_t bit = 1ull << (dev & 63);
  if ((attr_set.load(std::memory_order_acquire) & bit) == 0) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&bwd_main_kernel<T, D>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)main_lds_bytes<D>()) != hipSuccess)
      return TSFA_ERR_LAUNCH;
    attr_set.fetch_or(bit, std::memory_order_acq_rel);
  }
  const int64_t prep_threads = (int64_t)pa.batch * pa.num_kv_heads * p.n_tiles * kTileRows * 16;
  const int64_t prep_blocks = (prep_threads + 255) / 256;
  const int vis_chunks = p.n_tkeys / 64;
  const int64_t vis_blocks = has_tree ? (int64_t)p.n_tiles * p.n_trees * vis_chunks : 0;
  if (prep_blocks + vis_blocks > INT32_MAX) return TSFA_ERR_UNSUPPORTED;
  const size_t state_bytes = (size_t)std::max(1, p.nqbc_max * va.n_tree_blocks) * sizeof(int);
  hipLaunchKernelGGL((bwd_prep_vis_kernel<T, D>), dim3((unsigned)(prep_blocks + vis_blocks)), dim3(256), state_bytes,
                     stream, pa, va, (int)prep_blocks, std::max(1, vis_chunks));
  if (hipGetLastError() != hipSuccess) return TSFA_ERR_LAUNCH;
  auto launch_main = [&](int first, int blocks) {
    BwdArgs a = ba;
    a.first_block = first;
    if (blocks > 0)
      hipLaunchKernelGGL((bwd_main_kernel<T, D>), dim3((unsigned)blocks), dim3(kWaves * 64), main_lds_bytes<D>(),
                         stream, a);
    return hipGetLastError() == hipSuccess;
  };
  // TSFA_BWD_CONCURRENT=0 (measurements), or more threads than a grid holds:
  // one pass after the other
  const int n1 = 8 * (ba.dq_first ? ba.q_pairs_per_xcd : ba.items_per_xcd);
  const int n2 = 8 * (ba.dq_first ? ba.items_per_xcd : ba.q_pairs_per_xcd);
  const bool joint = config().bwd_concurrent != 0 && one_launch(n1, n2);
  if (joint ? !launch_main(0, n1 + n2) : !launch_main(0, n1) || !launch_main(n1, n2))
    return TSFA_ERR_LAUNCH;
  if (ba.dq_direct) return TSFA_OK;
  const int64_t dq_threads = (int64_t)da.batch * da.num_kv_heads * da.q_len * da.group * (D / 8);
  hipLaunchKernelGGL((bwd_dq_kernel<T, D>), dim3((unsigned)((dq_threads + 255) / 256)), dim3(256), 0, stream, da);
  return hipGetLastError() == hipSuccess ? TSFA_OK : TSFA_ERR_LAUNCH;
}

}  // namespace bwd
}  // namespace tsfa

using namespace tsfa;
using namespace tsfa::bwd;

extern "C" int tsfa_bwd(const void* q, const void* k, const void* v, const void* o, const float* lse,
                        const void* dout, void* dq, void* dk, void* dv, const int32_t* row_ptr,
                        const int32_t* col_idx, const int8_t* blk_type, const int32_t* mixed_mask_payload,
                        const int32_t* mixed_mask_offset, const int64_t* meta_seq_stride, const int64_t* strides,
                        float sm_scale, int batch, int num_heads, int num_kv_heads, int q_len, int kv_len,
                        int prefix_len, int n_q_blocks, int n_tree_blocks, int gqa_group_size, int block_m,
                        int block_n, int head_dim, int dtype, void* workspace, size_t workspace_bytes,
                        tsfa_stream_t stream_) {
  int st = tsfa_fwd_check_args(batch, num_heads, num_kv_heads, q_len, kv_len, prefix_len, n_q_blocks,
                               n_tree_blocks, gqa_group_size, block_m, block_n, head_dim, dtype);
  if (st != TSFA_OK) return st;
  // the backward kernels: 16-bit inputs, head_dim 64 or 128
  if ((dtype != TSFA_DTYPE_FP16 && dtype != TSFA_DTYPE_BF16) || (head_dim != 64 && head_dim != 128))
    return TSFA_ERR_UNSUPPORTED;
  if (batch == 0 || q_len == 0) return TSFA_OK;
  if (strides == nullptr || meta_seq_stride == nullptr) return TSFA_ERR_INVALID_ARGUMENT;
  const void* ptrs[9] = {q, k, v, o, dout, dq, dk, dv, lse};
  for (const void* ptr : ptrs)
    if (ptr == nullptr) return TSFA_ERR_INVALID_ARGUMENT;
  if (row_ptr == nullptr) return TSFA_ERR_INVALID_ARGUMENT;
  // strides: q, k, v, o, dout, dq, dk, dv -- (b, h, n, d) each
  for (int i = 0; i < 8; ++i) {
    if (strides[4 * i + 3] != 1) return TSFA_ERR_UNSUPPORTED;
    for (int j = 0; j < 3; ++j)
      if (strides[4 * i + j] % 8 != 0) return TSFA_ERR_UNSUPPORTED;
  }
  for (int i = 0; i < 8; ++i)
    if (reinterpret_cast<uintptr_t>(ptrs[i]) % 16 != 0) return TSFA_ERR_UNSUPPORTED;
  bool per_seq = false;
  for (int i = 0; i < 5; ++i) {
    if (meta_seq_stride[i] < 0) return TSFA_ERR_INVALID_ARGUMENT;
    per_seq = per_seq || meta_seq_stride[i] != 0;
  }
  const int n_trees = per_seq ? batch : 1;
  BwdPlan p;
  st = make_bwd_plan(batch, num_kv_heads, q_len, kv_len, prefix_len, gqa_group_size, head_dim, block_m,
                     n_tree_blocks, n_trees, &p);
  if (st != TSFA_OK) return st;
  if (workspace == nullptr || workspace_bytes < p.rowstat_bytes + p.dq_bytes + p.vis_bytes)
    return TSFA_ERR_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(workspace) % 256 != 0) return TSFA_ERR_WORKSPACE;
  char* ws = static_cast<char*>(workspace);
  float* rowstat = reinterpret_cast<float*>(ws);
  float* dq_acc = reinterpret_cast<float*>(ws + p.rowstat_bytes);
  uint32_t* vis = reinterpret_cast<uint32_t*>(ws + p.rowstat_bytes + p.dq_bytes);
  const int tree_key_limit =
      (int)std::min<int64_t>((int64_t)n_tree_blocks * block_n, (int64_t)kv_len - prefix_len);

  // signed: P = exp2(q.k * sl2 - lse2); a zero scale becomes a vanishing one
  float sl2 = sm_scale * 1.4426950408889634f;
  if (sl2 == 0.f) sl2 = 1e-30f;

  PrepArgs pa;
  pa.o = o;
  pa.dout = dout;
  pa.lse = lse;
  pa.rowstat = rowstat;
  pa.dq_acc = dq_acc;
  pa.sob = strides[12];
  pa.soh = strides[13];
  pa.som = strides[14];
  pa.sdob = strides[16];
  pa.sdoh = strides[17];
  pa.sdom = strides[18];
  pa.batch = batch;
  pa.num_heads = num_heads;
  pa.num_kv_heads = num_kv_heads;
  pa.group = gqa_group_size;
  pa.q_len = q_len;
  pa.n_tiles = p.n_tiles;

  VisArgs va;
  va.row_ptr = row_ptr;
  va.col_idx = col_idx;
  va.blk_type = blk_type;
  va.payload = mixed_mask_payload;
  va.offset = mixed_mask_offset;
  va.ms_row_ptr = meta_seq_stride[0];
  va.ms_col_idx = meta_seq_stride[1];
  va.ms_blk_type = meta_seq_stride[2];
  va.ms_payload = meta_seq_stride[3];
  va.ms_offset = meta_seq_stride[4];
  va.vis = vis;
  va.tree_stride = (int64_t)p.n_tiles * p.n_tkeys;
  va.group = gqa_group_size;
  va.q_len = q_len;
  va.block_m = block_m;
  va.block_n = block_n;
  va.n_tree_blocks = n_tree_blocks;
  va.tree_key_limit = tree_key_limit;
  va.n_tiles = p.n_tiles;
  va.n_tkeys = p.n_tkeys;

  BwdArgs ba;
  ba.q = q;
  ba.k = k;
  ba.v = v;
  ba.dout = dout;
  ba.dk = dk;
  ba.dv = dv;
  ba.dq_acc = dq_acc;
  ba.rowstat = rowstat;
  ba.vis = vis;
  ba.sqb = strides[0];
  ba.sqh = strides[1];
  ba.sqm = strides[2];
  ba.skb = strides[4];
  ba.skh = strides[5];
  ba.skn = strides[6];
  ba.svb = strides[8];
  ba.svh = strides[9];
  ba.svn = strides[10];
  ba.sdob = strides[16];
  ba.sdoh = strides[17];
  ba.sdom = strides[18];
  ba.sdkb = strides[24];
  ba.sdkh = strides[25];
  ba.sdkn = strides[26];
  ba.sdvb = strides[28];
  ba.sdvh = strides[29];
  ba.sdvn = strides[30];
  ba.vis_tree_stride = n_trees > 1 ? va.tree_stride : 0;
  ba.scale_log2 = sl2;
  ba.dk_scale = sm_scale;
  ba.num_kv_heads = num_kv_heads;
  ba.group = gqa_group_size;
  ba.q_len = q_len;
  ba.kv_len = kv_len;
  ba.prefix_len = prefix_len;
  ba.n_tiles = p.n_tiles;
  ba.n_pb = p.n_pb;
  ba.n_tb = p.n_tb;
  ba.n_tkeys = p.n_tkeys;
  ba.n_items = batch * num_kv_heads * (p.n_pb + p.n_tb);
  // row-parallel dQ: 128-row chunks; the 32-key units (prefix, then the tree
  // keys up to tree_key_limit) split by dq_split_plan (each split adds its chunk's
  // dQ once with atomics: splits x rows x D x 4 bytes of atomic traffic; an
  // unsplit chunk writes dQ directly)
  ba.n_pu = ceil_div(prefix_len, 32);
  ba.n_tu = ceil_div(tree_key_limit, 32);
  ba.n_chunks = ceil_div(p.n_tiles, kQWaves);
  {
    int cus = 256;
    if (device_cu_count(&cus) != TSFA_OK) return TSFA_ERR_DEVICE;
    const int n_units = ba.n_pu + ba.n_tu;
    const int64_t base = (int64_t)batch * num_kv_heads * ba.n_chunks;
    int splits = 1;
    bool dq_first = false;
    if (n_units > 0)
      dq_split_plan(ba.n_items, (p.n_tiles + 1) / 2, base, n_units, head_dim, (int64_t)p.dq_bytes, cus, &splits,
                    &dq_first);
    ba.dq_first = dq_first ? 1 : 0;
    ba.units_per_split = std::max(1, ceil_div(n_units, splits));
    ba.n_splits = std::max(1, ceil_div(n_units, ba.units_per_split));
    const int64_t q_items = n_units > 0 ? base * ba.n_splits : 0;
    if (q_items > INT32_MAX / 2) return TSFA_ERR_UNSUPPORTED;
    ba.q_items = (int)q_items;
    ba.q_pairs_per_xcd = ((ba.q_items + 1) / 2 + 7) / 8;
  }
  ba.dq = dq;
  ba.sdqb = strides[20];
  ba.sdqh = strides[21];
  ba.sdqm = strides[22];
  ba.dq_scale = sm_scale;
  ba.dq_direct = (ba.n_splits == 1 && ba.q_items > 0) ? 1 : 0;
  pa.zero_dq = ba.dq_direct ? 0 : 1;
  ba.group_magic = gqa_group_size > 1 ? (uint32_t)((((uint64_t)1) << 32) / (uint64_t)gqa_group_size + 1) : 0u;
  ba.items_per_xcd = (ba.n_items + 7) / 8;
  ba.tile_fast = tile_offsets_fit(gqa_group_size, ba.sqh, ba.sqm, head_dim) &&
                 tile_offsets_fit(gqa_group_size, ba.sdoh, ba.sdom, head_dim);
  ba.key_fast = unit_offsets_fit(ba.skn, head_dim) && unit_offsets_fit(ba.svn, head_dim);

  DqArgs da;
  da.dq_acc = dq_acc;
  da.dq = dq;
  da.sqb = strides[20];
  da.sqh = strides[21];
  da.sqm = strides[22];
  da.scale = sm_scale;
  da.batch = batch;
  da.num_kv_heads = num_kv_heads;
  da.group = gqa_group_size;
  da.q_len = q_len;
  da.tgp = p.n_tiles * kTileRows;

  const bool has_tree = p.n_tb > 0;
  hipStream_t stream = reinterpret_cast<hipStream_t>(stream_);
  if (dtype == TSFA_DTYPE_BF16)
    return head_dim == 128 ? launch_bwd<__bf16, 128>(ba, pa, va, da, p, has_tree, stream)
                           : launch_bwd<__bf16, 64>(ba, pa, va, da, p, has_tree, stream);
  return head_dim == 128 ? launch_bwd<_Float16, 128>(ba, pa, va, da, p, has_tree, stream)
                         : launch_bwd<_Float16, 64>(ba, pa, va, da, p, has_tree, stream);
}
