// Prefill kernels around the GEMM, behind the reference's C-ABI: the RoPE + KV-cache write that
// follows a QKV GEMM (hi_rope_cache; src/api.cu:579-586, kernels.cuh:1120-1158, ctypes
// scripts/hipinfer.py:164-168) and causal prefill attention over a cache slot (hi_flash_prefill,
// hi_flash_prefill_lse; api.cu:594-623, kernels.cuh:1160-1329, ctypes hipinfer.py:171-202).
//
// Flash prefill for gfx950 (D = 64 or 128):
//  * block = 32 RG query rows (RG 4, or 2 for small grids) of one query head and 2 RG waves: the waves of row group g (g and
//    g + RG) share its 32 rows and split every 128-key tile, keys 0..63 and 64..127, each with its
//    own online-softmax state; the pair merges (m, l, O) through LDS at the end. Two waves per
//    SIMD let one wave's softmax run beside the other's matrix work. The wave's Q rows stay in
//    registers as v_mfma_f32_32x32x16_f16 operands for the whole kernel;
//  * 128-key K/V tiles of the head's cache rows go straight from global memory into LDS by buffer
//    DMA (no register staging), two LDS stages each: K tile j + 2 and V tile j + 1 stream in while
//    tile j is computed, one barrier per tile. Both tiles keep the cache's row-major order with their
//    16-byte chunks XOR-swizzled by the key; the swizzle is applied to the DMA's per-lane source
//    address, since a DMA instruction writes 64 consecutive 16-byte LDS slots;
//  * the tiles are pipelined inside each wave: while the softmax of tile j runs on the vector units,
//    the matrix cores work on the logits of tile j + 1 and on tile j's P.V, interleaved instruction by
//    instruction. What bounds it: at T = 2048 after 4096 positions (Hq 32, Hkv 8, D 128) the MFMAs
//    alone take about half of the GPU's cycles and the clock drops to 1.8 GHz under the load; 204 ->
//    173 us (850 -> 1000 TFLOP/s) against back-to-back products, T = 1024 from 0 26.6 -> 22.1 us, 333
//    rows after 1500 36.8 -> 27.2, D = 64 T = 2048 after 2048 76.7 -> 68;
//  * S^T = K Q^T over the wave's 64 keys, in 32-key MFMA blocks: with the K fragment as first
//    operand each lane ends with 16 keys per block of ONE query row (split between lanes l and
//    l + 32), so the row max and sum of the online softmax are the lane's own values; lanes l and
//    l ^ 32 exchange them only where the reference max moves and at the end;
//  * logits are scaled by log2(e) / sqrt(D) and the softmax runs in base 2 (the reference's
//    log2-domain form, kernels.cuh:1236-1262); P is rounded to fp16 for P.V, the row sum l keeps
//    fp32 p, as the reference does. exp2 is the hardware's v_exp_f32, whose results below 2^-126
//    flush to zero: such p round to fp16 zero anyway and vanish against l >= 1 in fp32. A row's
//    reference max moves only when the row's max passes it by more than 2^8 (p <= 256), and O is
//    rescaled only then;
//  * O^T += V^T P^T: the P registers of a lane are already a B fragment of the next product once
//    the key order inside each 16-key step is permuted identically for P and V^T (lane half fk
//    takes keys 4 fk + 0..3 and 8 + 4 fk + 0..3), so P never goes through LDS. The V^T fragments
//    come from the row-major V tile through ds_read_tr16_b64, which transposes 4 keys x 16 d
//    blocks within each 16-lane group; O^T keeps the lane -> query row map, so the per-row
//    rescale by exp2(m_old - m_new) is per lane;
//  * causal mask on absolute positions (row t at p0 + t sees keys 0..p0+t): only the block's last
//    one or two tiles (and an odd one before them) carry the mask arithmetic, and a wave leaves out
//    the key halves wholly above its rows' diagonal; cache rows past the block's last key read as
//    zeros (the DMA's buffer range ends there);
//  * blocks run the longest query tiles (the most keys) first, across all heads.
#include <type_traits>

#include "hi_common.h"

namespace {

constexpr int kFpRG = 4;              // 32-row groups per block (2 waves each); 2 for small grids
constexpr int kFpKPW = 64;            // keys per wave per tile (32-key MFMA blocks of the wave's half)
constexpr int kFpBKV = 2 * kFpKPW;    // keys per tile
constexpr int kFpStages = 2;          // LDS stages of K/V tiles
constexpr float kFpMaxLag = 8.f;      // log2 of how far a row's reference max may trail its max

// XOR term of key r's 16-byte chunks in the K tile: the 16 keys (D = 128) or 8 key pairs (D = 64)
// that one 128-bit fragment read serves per cycle land on distinct banks.
template <int D>
__device__ __forceinline__ int k_swz(int r) {
  if constexpr (D == 128) return r & 15;
  else return (r >> 1) & 7;
}
// XOR term of key r's chunks in the V tile. A transpose read covers keys r..r+3 (r % 4 == 0) at
// 4 consecutive chunks per 32 lanes and 2 per 16 lanes; the terms 0, 6, 12, 10 (D = 128) or 0, 6,
// 4, 2 (D = 64) for r % 4 = 0..3 move those chunks to distinct banks at either width.
template <int D>
__device__ __forceinline__ int v_swz(int r) {
  const int a = r & 3;
  return ((2 * a) ^ (4 * a)) & (D / 8 - 1);
}

// LDS of one block: two stages of K tiles and two of V tiles while the keys stream, then in the same
// bytes the O^T accumulators the second wave of each row group hands to the first; last, the second
// waves' m and l. It is dynamic LDS: reads of a __shared__ array that a DMA instruction also writes
// made the compiler wait for every DMA in flight (s_waitcnt vmcnt(0)) before the first of them, right
// after the next tile's DMA had been issued, so that no tile streamed in while another was computed.
template <int D, int RG>
struct FpSmem {
  static constexpr int kTile = kFpBKV * D / 8;                // 16-byte chunks of one K or V tile
  static constexpr int kMl = 2 * kFpStages * kTile;           // chunk index of m and l
  static constexpr size_t kBytes = kMl * 16 + 2 * RG * 64 * 4;
  static_assert(RG * (D / 32) * 64 * 64 <= kMl * 16, "merge fits the stages");
};

typedef short i16x4 __attribute__((ext_vector_type(4)));

// The two builtins below sit in the device pass only: in this kernel's host pass they made the
// compiler drop the kernel's launch stub without a diagnostic (an undefined symbol at load).
// 16-byte buffer DMA of each lane's chunk at byte offset voff into LDS slot lane of `lds`.
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t rs, void* lds, int voff) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_void_t*)lds, 16, voff, 0, 0, 0);
#endif
}
// ds_read_tr16_b64 at LDS address p: within each 16-lane group, lane i receives element i % 4 of
// the 4 halves lane 4 e + i / 4 addresses, as its element e.
__device__ __forceinline__ f16x4 lds_read_tr16(const f16* __restrict__ p) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_bit_cast(f16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)p));
#else
  return f16x4{};
#endif
}

template <int D, int RG>
__global__ void __launch_bounds__(128 * RG)
    flash_prefill_kernel(const f16* __restrict__ q, int64_t ldq, const f16* __restrict__ kc,
                         const f16* __restrict__ vc, int max_seq, f16* __restrict__ out, int64_t ldo, int T, int p0,
                         int Hq, int Hkv, float scale_log2, float* __restrict__ lse) {
  constexpr int NW = 2 * RG, BQ = 32 * RG;
  constexpr int CPR = D / 8;                   // 16-byte chunks per key row
  constexpr int IPW = kFpBKV * CPR / 64 / NW;  // DMA instructions per wave per tile and operand
  constexpr int DT = D / 32;                   // 32-row output tiles of O^T
  constexpr int NQ = D / 16;                   // MFMAs of one 32-key block's logits
  static_assert(IPW * 64 * NW == kFpBKV * CPR, "tile DMA split");
  static_assert(kFpStages == 2 && kFpKPW == 64, "the tile body is written for two stages and two key blocks");
  using Sm = FpSmem<D, RG>;
  extern __shared__ u32x4 fp_smem[];
  u32x4* const ks_ = fp_smem;                                // [2][kTile]: K stages
  u32x4* const vs_ = fp_smem + kFpStages * Sm::kTile;        // [2][kTile]: V stages
  f32x16* const mo = reinterpret_cast<f32x16*>(fp_smem);     // [RG][DT][64]: the merge
  float* const ml = reinterpret_cast<float*>(fp_smem + Sm::kMl);  // [2][RG][64]: the second waves' m and l

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = wave % RG, kh = wave / RG;     // row group, key half
  const int fr = lane & 31, fk = lane >> 5;
  // grid (Hq, query tiles), dispatched x first: all heads' longest query tile first; block x runs
  // on XCD x % 8, which takes a contiguous range of query heads (those sharing a KV head)
  const int q0 = (gridDim.y - 1 - blockIdx.y) * BQ;
  const int h = Hq % 8 ? blockIdx.x : (blockIdx.x % 8) * (Hq / 8) + blockIdx.x / 8, hk = h / (Hq / Hkv);
  const int qw = q0 + rg * 32;                  // this wave's first query row
  const int qi = qw + fr;                       // this lane's query row
  const int qpos = p0 + qi;
  const int kv_end = p0 + min(q0 + BQ, T);      // keys any row of the block can see
  const int nt = (kv_end + kFpBKV - 1) / kFpBKV;  // key tiles; the first n_full hold no masked key
  const int n_full = (p0 + q0 + 1) / kFpBKV;

  // this lane's Q fragments: row qi, d = 16 ks + 8 fk + 0..7 (zero past T)
  f16x8 qf[NQ];
#pragma unroll
  for (int ks = 0; ks < NQ; ks++) {
    u32x4 v = {0u, 0u, 0u, 0u};
    if (qi < T) v = *reinterpret_cast<const u32x4*>(q + (int64_t)qi * ldq + h * D + 16 * ks + 8 * fk);
    qf[ks] = __builtin_bit_cast(f16x8, v);
  }

  // the head's cache rows 0..kv_end-1: loads past them return zeros
  const __amdgpu_buffer_rsrc_t k_rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<f16*>(kc + (int64_t)hk * max_seq * D), (short)0, kv_end * D * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t v_rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<f16*>(vc + (int64_t)hk * max_seq * D), (short)0, kv_end * D * 2, 0x00020000);
  // DMA instruction i of this wave fills slots (wave IPW + i) * 64 + lane of a tile: slot s holds
  // key s / CPR, physical chunk s % CPR, i.e. logical chunk (s % CPR) ^ swz(key)
  int koff[IPW], voff[IPW];
#pragma unroll
  for (int i = 0; i < IPW; i++) {
    const int s = (wave * IPW + i) * 64 + lane, r = s / CPR, p = s % CPR;
    koff[i] = (r * D + 8 * (p ^ k_swz<D>(r))) * 2;
    voff[i] = (r * D + 8 * (p ^ v_swz<D>(r))) * 2;
  }
  // issue instruction i of the next K (V) tile into stage st; koff / voff then point at the one after
  auto issue_k = [&](int i, int st) {
    lds_dma16(k_rs, ks_ + st * Sm::kTile + (wave * IPW + i) * 64, koff[i]);
    koff[i] += kFpBKV * D * 2;
    asm volatile("" : "+v"(koff[i]));  // one running offset, not a base and an induction variable
  };
  auto issue_v = [&](int i, int st) {
    lds_dma16(v_rs, vs_ + st * Sm::kTile + (wave * IPW + i) * 64, voff[i]);
    voff[i] += kFpBKV * D * 2;
    asm volatile("" : "+v"(voff[i]));
  };

  // transpose reads of V: lane j of each 16-lane group g reads 4 d of key 4 (g / 2) + j / 4 (+ the
  // step's key base), d = 16 (g % 2) + 4 (j % 4) (+ the output tile's d base); the group's lane i
  // then holds d = 16 (g % 2) + i of those 4 keys. Keys of one read are 4-aligned, so the swizzle
  // term is the lane's own.
  const int vr = 4 * fk + ((lane & 15) >> 2);                  // key within a 16-key step
  const int vc0 = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);   // logical chunk within a 32-d tile
  const f16* vb[DT];                                           // the lane's first read of each output tile
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
    vb[dt] = reinterpret_cast<const f16*>(vs_) + (kFpKPW * kh + vr) * D + 8 * ((4 * dt + vc0) ^ v_swz<D>(vr)) + 4 * (lane & 1);
  const int kr = kFpKPW * kh + fr;                             // K row of this lane's first fragments
  const int ksw = k_swz<D>(kr);                                // the same for every block (kr % 16)
  const int xaddr = (lane ^ 32) << 2;                          // lane l ^ 32, for ds_bpermute
  auto xor32 = [&](float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(xaddr, __builtin_bit_cast(int, v)));
  };

  // m_i: the row's reference max (the same in lanes l and l ^ 32); l_i: this lane's share of the
  // row's sum (its own keys; the two lanes' shares are added at the end)
  float m_i = -__builtin_huge_valf(), l_i = 0.f;
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int e = 0; e < 16; e++) o[dt][e] = 0.f;

  // S^T = K Q^T over 32-key block kt of the wave's keys in K stage st; lane (row fr, half fk) gets
  // keys 32 kt + 8 g + 4 fk + e
  auto logits = [&](int st, int kt, f32x16& s) {
    f32x16 a;
#pragma unroll
    for (int e = 0; e < 16; e++) a[e] = 0.f;
#pragma unroll
    for (int ks = 0; ks < NQ; ks++) {
      const f16x8 kf = __builtin_bit_cast(f16x8, ks_[st * Sm::kTile + (kr + 32 * kt) * CPR + ((2 * ks + fk) ^ ksw)]);
      a = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[ks], a, 0, 0, 0);
    }
    s = a;
  };
  // the V^T fragments of block kt (V stage st): of step ss, lane half fk holds keys 32 kt + 16 ss +
  // 4 fk + 0..3 and 32 kt + 16 ss + 8 + 4 fk + 0..3 of the wave's keys, as P's registers do
  auto load_v = [&](int st, int kt, f16x8 (&vf)[2][DT]) {
#pragma unroll
    for (int ss = 0; ss < 2; ss++)
#pragma unroll
      for (int dt = 0; dt < DT; dt++) {
        const f16* pa = vb[dt] + st * (Sm::kTile * 8) + (32 * kt + 16 * ss) * D;
        const f16x4 fa = lds_read_tr16(pa), fb = lds_read_tr16(pa + 8 * D);  // key + 8: same swizzle term
        vf[ss][dt] = f16x8{fa[0], fa[1], fa[2], fa[3], fb[0], fb[1], fb[2], fb[3]};
      }
  };
  // O^T += V^T P^T of one 32-key block
  auto pv = [&](const f16x8 (&vf)[2][DT], const f16x8 (&pf)[2]) {
#pragma unroll
    for (int ss = 0; ss < 2; ss++)
#pragma unroll
      for (int dt = 0; dt < DT; dt++) o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[ss][dt], pf[ss], o[dt], 0, 0, 0);
  };
  // p = exp2(c s - m) of one block, its sum into l_i, fp16 p in P.V operand order
  auto softmax = [&](const f32x16& s, float m_use, f16x8 (&pf)[2]) {
    float sum0 = 0.f, sum1 = 0.f;
#pragma unroll
    for (int e = 0; e < 16; e += 2) {
      const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e], scale_log2, -m_use));
      const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[e + 1], scale_log2, -m_use));
      sum0 += p;
      sum1 += p1;
      pf[e >> 3][e & 7] = (f16)p;
      pf[e >> 3][(e & 7) + 1] = (f16)p1;
    }
    l_i += sum0 + sum1;
  };

  // One key tile t (stage t & 1, given as a constant in the main loop): the softmax and P.V of its
  // logits sc, with the logits of tile t + 1 into sn in between. A wave issues in order, so the
  // MFMAs of one product are interleaved with the vector work of the other tile's softmax by
  // scheduling groups; otherwise each product's MFMAs run back to back, then the softmax with the
  // matrix cores idle (both waves of a SIMD leave the tile's barrier together). The P.V of the
  // tile's second block (pl, its V fragments vl read before the next barrier) runs after that
  // barrier: matrix work that needs no LDS while the first K fragments are on their way.
  f16x8 pl[2], vl[2][DT];
#pragma unroll
  for (int ss = 0; ss < 2; ss++) {
    pl[ss] = f16x8{};
#pragma unroll
    for (int dt = 0; dt < DT; dt++) vl[ss][dt] = f16x8{};
  }
  auto tile = [&](auto stc, auto maskc, auto nextc, int t, f32x16 (&sc)[2], f32x16 (&sn)[2]) {
    constexpr bool MASK = decltype(maskc)::value;  // the tile holds keys past some row's diagonal
    constexpr bool NEXT = decltype(nextc)::value;  // there is a tile t + 1
    const int st = stc;
    wait_lgkm0();
    wait_vmcnt<0>();     // this wave's shares of K tile t + 1 and V tile t are in LDS
    barrier_no_fence();  // every share is, and every wave is done with K tile t and V tile t - 1
    const int k0 = t * kFpBKV + kFpKPW * kh;  // this wave's first key
    if constexpr (MASK) {
#pragma unroll
      for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int e = 0; e < 16; e++) {
          const int kp = k0 + 32 * kt + 8 * (e >> 2) + 4 * fk + (e & 3);
          if (kp > qpos) sc[kt][e] = -__builtin_huge_valf();
        }
    }
    // the row's reference max m_i moves only when the tile's scaled max exceeds it by more than 2^8,
    // so p = exp2(c s - m_i) stays at most 256 (exact range for fp16 P and fp32 sums) and O is
    // rescaled only then; lanes l and l ^ 32 then agree on the new one. The max of the raw logits is
    // scaled once (c > 0 keeps the order) and c s - m_i is one fma
    // The MFMAs of this tile up to its first P.V, in slots: the last block's P.V, then (NEXT) the
    // logits of tile t + 1. The 2 IPW DMA instructions of K tile t + 2 and V tile t + 1 go out over the
    // slots of the first logits block; with 4 waves, each issuing twice as many and without a second
    // wave on its SIMD to fill its stalls, over all of them (64 rows after 2000 positions 26.1 ->
    // 22.6 us, 512 after 2048 36.0 -> 32.7; 8 waves: no gain, 2 % slower at T = 2048 after 4096).
    constexpr int ND = 2 * IPW, LA = 3;  // DMA instructions, LDS reads ahead of their MFMA
    constexpr int S0 = RG == 2 ? 0 : 2 * DT, NS = RG == 2 ? 2 * DT + 2 * NQ : NQ;
    auto dma_here = [](int m) constexpr {  // DMA instructions that go before slot m
      int n = 0;
      for (int j = 0; j < ND; j++) n += S0 + j * NS / ND == m;
      return n;
    };
    constexpr int kDma = (ND + NS - 1) / NS;  // at most this many before one slot
    auto dma = [&](int m) {
#pragma unroll
      for (int j = 0; j < ND; j++)
        if (S0 + j * NS / ND == m) j < IPW ? issue_k(j, st) : issue_v(j - IPW, st ^ 1);
    };
    auto load_k = [&](int kt, int ks) {
      return __builtin_bit_cast(f16x8, ks_[(st ^ 1) * Sm::kTile + (kr + 32 * kt) * CPR + ((2 * ks + fk) ^ ksw)]);
    };
    float mx = -__builtin_huge_valf();
    f16x8 kf[NQ];
    f32x16 a0;
#pragma unroll
    for (int e = 0; e < 16; e++) a0[e] = 0.f;
#pragma unroll
    for (int m = 0; m < 2 * DT; m++) {
      if constexpr (NEXT) {
        dma(m);
        if (m >= 2 * DT - LA) kf[m - (2 * DT - LA)] = load_k(0, m - (2 * DT - LA));
      }
      o[m % DT] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vl[m / DT][m % DT], pl[m / DT], o[m % DT], 0, 0, 0);
    }
    if constexpr (NEXT) {
#pragma unroll
      for (int ks = 0; ks < NQ; ks++) {
        dma(2 * DT + ks);
        if (ks + LA < NQ) kf[ks + LA] = load_k(0, ks + LA);
        a0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[ks], qf[ks], a0, 0, 0, 0);
      }
      sn[0] = a0;
    }
#pragma unroll
    for (int kt = 0; kt < 2; kt++)
#pragma unroll
      for (int e = 0; e < 16; e++) mx = fmaxf(mx, sc[kt][e]);
    constexpr int kMaskOps = MASK ? 8 : 0;  // more vector work per MFMA
#pragma unroll
    for (int m = 0; m < 2 * DT; m++) {
      if (NEXT && dma_here(m)) __builtin_amdgcn_sched_group_barrier(0x020, kDma, 0);  // DMA
      if (NEXT && m >= 2 * DT - LA) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);             // MFMA (the last block's P.V)
      __builtin_amdgcn_sched_group_barrier(0x002, 2 + kMaskOps, 0);  // VALU (the max)
    }
    if constexpr (NEXT) {
#pragma unroll
      for (int ks = 0; ks < NQ; ks++) {
        if (dma_here(2 * DT + ks)) __builtin_amdgcn_sched_group_barrier(0x020, kDma, 0);
        if (ks + LA < NQ) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);           // MFMA (logits)
        __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
      }
    }
    if (__any(mx * scale_log2 > m_i + kFpMaxLag)) {  // m_i = -inf: moves to the first finite max
      mx = fmaxf(mx, xor32(mx)) * scale_log2;
      const bool move = mx > m_i + kFpMaxLag;
      const float alpha = move ? __builtin_amdgcn_exp2f(m_i - mx) : 1.f;
      if (move) m_i = mx;
      l_i *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; dt++)
#pragma unroll
        for (int e = 0; e < 16; e++) o[dt][e] *= alpha;
    }
    // m_i is -inf only for a row that has seen no key yet (one whose first key lies in the other
    // half): every logit is then -inf and every p 0
    const float m_use = m_i == -__builtin_huge_valf() ? 0.f : m_i;
    f16x8 pf[2], vf[2][DT];
    if constexpr (NEXT) {
      f32x16 a1;
#pragma unroll
      for (int e = 0; e < 16; e++) a1[e] = 0.f;
#pragma unroll
      for (int ks = 0; ks < LA; ks++) kf[ks] = load_k(1, ks);
#pragma unroll
      for (int ks = 0; ks < NQ; ks++) {
        dma(2 * DT + NQ + ks);
        if (ks + LA < NQ) kf[ks + LA] = load_k(1, ks + LA);
        a1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[ks], qf[ks], a1, 0, 0, 0);
      }
      sn[1] = a1;
    }
    softmax(sc[0], m_use, pf);
    load_v(st, 0, vf);
    pv(vf, pf);
    softmax(sc[1], m_use, pl);
    load_v(st, 1, vl);
    if constexpr (NEXT) {
      __builtin_amdgcn_sched_group_barrier(0x100, LA, 0);
#pragma unroll
      for (int ks = 0; ks < NQ; ks++) {
        if (dma_here(2 * DT + NQ + ks)) __builtin_amdgcn_sched_group_barrier(0x020, kDma, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        if (ks + LA >= NQ) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);             // MFMA (logits)
        __builtin_amdgcn_sched_group_barrier(0x002, 56 / NQ, 0);       // VALU (softmax of block 0)
      }
#pragma unroll
      for (int i = 0; i < 2 * DT; i++) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);             // MFMA (P.V of block 0)
        __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 56 / (2 * DT), 0); // VALU (softmax of block 1)
      }
    }
  };

  // ---- prologue: K tiles 0 and 1 and V tile 0 in flight, the logits of tile 0
#pragma unroll
  for (int i = 0; i < IPW; i++) issue_k(i, 0);
#pragma unroll
  for (int i = 0; i < IPW; i++) {
    issue_v(i, 0);
    issue_k(i, 1);
  }
  wait_vmcnt<2 * IPW>();
  barrier_no_fence();
  f32x16 sa[2], sb[2];
  logits(0, 0, sa[0]);
  logits(0, 1, sa[1]);
  constexpr std::integral_constant<int, 0> kEven{};
  constexpr std::integral_constant<int, 1> kOdd{};
  int t = 0;
  const std::true_type yes{};
  const std::false_type no{};
  for (; t + 2 <= n_full && t + 2 < nt; t += 2) {
    tile(kEven, no, yes, t, sa, sb);
    tile(kOdd, no, yes, t + 1, sb, sa);
  }
  // The other tiles may hold masked keys. A wave leaves out a tile whose keys (its half) lie wholly past
  // its rows' diagonal or the block's last key, as it does every later one, but for its share of the
  // DMA and the barrier: their weights are 0, but 0 times an infinity or NaN in a later row's V is not.
  auto live = [&](int t) {
    const int k0 = t * kFpBKV + kFpKPW * kh;
    return k0 <= p0 + qw + 31 && k0 < kv_end;
  };
  for (; t + 1 < nt; t++) {  // an odd full tile, the first of two tiles on the diagonal
    if (live(t)) {
      tile(t & 1, yes, yes, t, sa, sb);
      sa[0] = sb[0];
      sa[1] = sb[1];
    } else {
      wait_lgkm0();
      wait_vmcnt<0>();
      barrier_no_fence();
#pragma unroll
      for (int i = 0; i < IPW; i++) {
        issue_k(i, t & 1);
        issue_v(i, (t & 1) ^ 1);
      }
    }
  }
  if (live(t)) {
    tile(t & 1, yes, no, t, sa, sb);
  } else {
    wait_lgkm0();
    wait_vmcnt<0>();
    barrier_no_fence();
  }

  pv(vl, pl);

  // ---- merge the two key halves of each row group: the second wave hands (m, l, O) over
  wait_vmcnt<0>();
  __syncthreads();  // every wave is done with the stages, and no DMA is in flight
  l_i += xor32(l_i);
  if (kh == 1) {
#pragma unroll
    for (int dt = 0; dt < DT; dt++) mo[(rg * DT + dt) * 64 + lane] = o[dt];
    ml[rg * 64 + lane] = m_i;
    ml[(RG + rg) * 64 + lane] = l_i;
  }
  __syncthreads();
  if (kh == 1 || qi >= T) return;
  const float m1 = ml[rg * 64 + lane], l1 = ml[(RG + rg) * 64 + lane];
  const float m = fmaxf(m_i, m1);  // finite: key 0 is visible to every row
  const float a0 = __builtin_amdgcn_exp2f(m_i - m), a1 = __builtin_amdgcn_exp2f(m1 - m);
  const float l = l_i * a0 + l1 * a1;
  if (lse && fk == 0) lse[(int64_t)h * T + qi] = m + log2f(l);
  const float inv = 1.f / l;
  f16* orow = out + (int64_t)qi * ldo + h * D;
#pragma unroll
  for (int dt = 0; dt < DT; dt++) {
    const f32x16 o1 = mo[(rg * DT + dt) * 64 + lane];
#pragma unroll
    for (int g = 0; g < 4; g++) {
      f16x4 v;
#pragma unroll
      for (int e = 0; e < 4; e++) v[e] = (f16)((o[dt][4 * g + e] * a0 + o1[4 * g + e] * a1) * inv);
      *reinterpret_cast<f16x4*>(orow + dt * 32 + 8 * g + 4 * fk) = v;
    }
  }
}

// Any alignment (2-byte accesses only): block (row, head group), one wave per head of the row's
// Hq + 2 Hkv heads. A q head is rotated in place, a k head rotated into the cache, a v head copied
// into the cache; lane j takes the pairs (j, j + D/2), (j + 64, j + 64 + D/2), ... of its head.
// Each pair goes through rope_pair, as in the 16-byte kernel below, so both give the same bits.
constexpr int kRopeHeadsPerBlock = 4;

__global__ void __launch_bounds__(64 * kRopeHeadsPerBlock)
    rope_cache_heads_kernel(f16* qkv, int64_t ldq, int Hq, int Hkv, int D, const f16x2* __restrict__ cs,
                            const int* __restrict__ pos, int pos_base, int slot_base, f16* kc, f16* vc, int max_seq) {
  const int r = blockIdx.x, lane = threadIdx.x & 63;
  const int head = blockIdx.y * kRopeHeadsPerBlock + (threadIdx.x >> 6);
  if (head >= Hq + 2 * Hkv) return;
  const int at = pos ? pos[r] : pos_base + r;                  // position in the cache
  const int64_t cslot = pos ? (int64_t)slot_base + r : slot_base;
  f16* src = qkv + (int64_t)r * ldq + (int64_t)head * D;
  if (head >= Hq + Hkv) {
    f16* dst = vc + ((cslot * Hkv + (head - Hq - Hkv)) * max_seq + at) * D;
    for (int e = lane; e < D; e += 64) dst[e] = src[e];
    return;
  }
  f16* dst = head < Hq ? src : kc + ((cslot * Hkv + (head - Hq)) * max_seq + at) * D;
  const int half = D >> 1;
  const f16x2* tab = cs + (int64_t)at * half;
  for (int j = lane; j < half; j += 64) {
    f16 lo = src[j], hi = src[j + half];
    rope_pair(lo, hi, tab[j]);
    dst[j] = lo;
    dst[j + half] = hi;
  }
}

// The same with 16-byte accesses: a thread step rotates 8 pairs of one head (the 8 elements at d
// and the 8 at d + D/2, and their 8 table entries) or copies 8 elements of v. Used when D/2 is a
// multiple of 8 and every row, cache and the table are 16-byte aligned; each pair is rotated by
// rope_pair, as above, so the two kernels give the same bits.
__global__ void __launch_bounds__(256)
    rope_cache_v8_kernel(f16* qkv, int64_t ldq, int Hq, int Hkv, int D, const f16x2* __restrict__ cs,
                         const int* __restrict__ pos, int pos_base, int slot_base, f16* kc, f16* vc, int max_seq) {
  const int HD = D / 2, C = HD / 8, row = blockIdx.x;
  const int p = pos ? pos[row] : pos_base + row;
  const int slot = pos ? slot_base + row : slot_base;
  f16* base = qkv + (int64_t)row * ldq;
  const int nrot = (Hq + Hkv) * C, nv = Hkv * D / 8;
  for (int i = threadIdx.x; i < nrot + nv; i += blockDim.x) {
    if (i < nrot) {
      const int hh = i / C, d = (i - hh * C) * 8;
      f16* x = base + hh * D;
      f16x8 a = *reinterpret_cast<const f16x8*>(x + d), b = *reinterpret_cast<const f16x8*>(x + d + HD);
      const u32x4* tp = reinterpret_cast<const u32x4*>(cs + (int64_t)p * HD + d);
      const u32x4 c0 = tp[0], c1 = tp[1];
#pragma unroll
      for (int j = 0; j < 8; j++) {
        f16 y1 = a[j], y2 = b[j];
        rope_pair(y1, y2, as_h2(j < 4 ? c0[j] : c1[j - 4]));
        a[j] = y1;
        b[j] = y2;
      }
      f16* dst = hh < Hq ? x : kc + (((int64_t)slot * Hkv + hh - Hq) * max_seq + p) * D;
      *reinterpret_cast<f16x8*>(dst + d) = a;
      *reinterpret_cast<f16x8*>(dst + d + HD) = b;
    } else {
      const int c = i - nrot, h = c / (D / 8), e = (c - h * (D / 8)) * 8;
      *reinterpret_cast<u32x4*>(vc + (((int64_t)slot * Hkv + h) * max_seq + p) * D + e) =
          *reinterpret_cast<const u32x4*>(base + (Hq + Hkv + h) * D + e);
    }
  }
}

bool aligned(const void* p, uintptr_t a) { return ((uintptr_t)p & (a - 1)) == 0; }

int flash_prefill(const void* q, int ldq, const void* kc, const void* vc, int max_seq, void* out, int ldo, int T,
                  int p0, int Hq, int Hkv, int D, float* lse, void* stream, const char* who) {
  if (!hi_device()) return -2;
  if (D != 64 && D != 128) HI_FAIL("%s: head_dim %d not supported (64 or 128)", who, D);
  if (T < 0 || p0 < 0 || Hkv < 1 || Hq < Hkv || Hq % Hkv || max_seq < 1 || (int64_t)p0 + T > max_seq)
    HI_FAIL("%s: bad shape T=%d p0=%d Hq=%d Hkv=%d max_seq=%d", who, T, p0, Hq, Hkv, max_seq);
  if (T == 0) return 0;
  if ((int64_t)max_seq * D * 2 > INT32_MAX)  // a head's cache rows are addressed by 32-bit byte offsets
    HI_FAIL("%s: max_seq %d too long for 32-bit cache offsets (at most %d at D=%d)", who, max_seq,
            (int)(INT32_MAX / (2 * D)), D);
  if (!q || !kc || !vc || !out) HI_FAIL("%s: null tensor pointer", who);
  if (!aligned(q, 16) || ldq % 8 || ldq < Hq * D) HI_FAIL("%s: q must be 16-byte aligned, ldq %% 8 == 0, ldq >= Hq*D", who);
  if (!aligned(kc, 16) || !aligned(vc, 16)) HI_FAIL("%s: kc / vc must be 16-byte aligned", who);
  if (!aligned(out, 8) || ldo % 4 || ldo < Hq * D) HI_FAIL("%s: out must be 8-byte aligned, ldo %% 4 == 0, ldo >= Hq*D", who);
  const float scale_log2 = 1.4426950408889634f / sqrtf((float)D);
  const HiDevice* d = hi_device();
  if (!d) return -2;
  // Query rows per block: 128, or 64 while that grid is still resident at once. A CU takes a key tile
  // for 64 rows only 10-25 % faster than for 128, but the longest query tile is half as tall and a
  // small grid reaches twice the CUs: T = 512 from 0 (Hq 32, D 128) 14.4 -> 11.1 us, 64 rows after
  // 2000 28.4 -> 22.6, 777 rows of 12 heads 16.6 -> 12.7; past one round it loses (640 rows after 2048
  // 39.8 -> 48.9). At D = 64 two such blocks share a CU: that pays while most tiles are short of
  // the diagonal (777 rows from 0 12.3 -> 10.2 us), not after a long prefix (960 after 2048 34.5 -> 35.3).
  const int slots = D == 64 && p0 < T ? 2 * d->cus : d->cus;
  const bool small = (int64_t)Hq * ((T + 63) / 64) <= slots;
  const int rg = small ? 2 : kFpRG, bq = 32 * rg;
  if ((T + bq - 1) / bq > 65535) HI_FAIL("%s: T=%d exceeds %d query rows", who, T, 65535 * bq);
  const dim3 grid(Hq, (T + bq - 1) / bq);
  const hipStream_t s = (hipStream_t)stream;
  const auto kern = D == 128 ? (small ? flash_prefill_kernel<128, 2> : flash_prefill_kernel<128, kFpRG>)
                             : (small ? flash_prefill_kernel<64, 2> : flash_prefill_kernel<64, kFpRG>);
  const size_t lds = D == 128 ? (small ? FpSmem<128, 2>::kBytes : FpSmem<128, kFpRG>::kBytes)
                              : (small ? FpSmem<64, 2>::kBytes : FpSmem<64, kFpRG>::kBytes);
  const int bpc = hi_blocks_per_cu(reinterpret_cast<const void*>(kern), 64 * 2 * rg, lds);  // lifts the LDS limit
  if (bpc < 0) return -2;
  if (bpc == 0) HI_FAIL("%s: the kernel does not fit on a CU", who);
  hipLaunchKernelGGL(kern, grid, dim3(64 * 2 * rg), lds, s, (const f16*)q, (int64_t)ldq, (const f16*)kc,
                     (const f16*)vc, max_seq, (f16*)out, (int64_t)ldo, T, p0, Hq, Hkv, scale_log2, lse);
  HI_TRY(hipGetLastError());
  return 0;
}

}  // namespace

// RoPE + KV-cache write for M qkv rows [M, ldq] = [q (Hq*D) | k (Hkv*D) | v (Hkv*D)]: q rotated in
// place, rotated k and raw v to kc / vc [slots][Hkv][max_seq][D]. Row m sits at position pos[m] in
// slot slot_base + m (pos non-null: decode) or at pos_base + m in slot slot_base (prefill).
// cs: [max_seq][D/2] (cos, sin) fp16 pairs. Positions must lie in [0, max_seq).
HI_EXPORT int hi_rope_cache(void* qkv, int ldq, int M, int Hq, int Hkv, int D, const void* cs, const int* pos,
                            int pos_base, int slot_base, void* kc, void* vc, int max_seq, void* stream) {
  if (!hi_device()) return -2;
  if (M < 0 || Hq < 1 || Hkv < 1 || D < 2 || D % 2 || max_seq < 1 || slot_base < 0)
    HI_FAIL("hi_rope_cache: bad shape M=%d Hq=%d Hkv=%d D=%d max_seq=%d", M, Hq, Hkv, D, max_seq);
  if (M == 0) return 0;
  if (!qkv || !cs || !kc || !vc) HI_FAIL("hi_rope_cache: null tensor pointer");
  if (ldq < (Hq + 2 * Hkv) * D) HI_FAIL("hi_rope_cache: ldq %d < (Hq + 2 Hkv) D", ldq);
  if ((Hq + 2 * Hkv + kRopeHeadsPerBlock - 1) / kRopeHeadsPerBlock > 65535)
    HI_FAIL("hi_rope_cache: %d heads per row exceed the launch grid", Hq + 2 * Hkv);
  if (!pos && (pos_base < 0 || (int64_t)pos_base + M > max_seq))
    HI_FAIL("hi_rope_cache: positions %d..%d outside the cache (max_seq %d)", pos_base, pos_base + M - 1, max_seq);
  if (!aligned(cs, 4)) HI_FAIL("hi_rope_cache: cs must be 4-byte aligned");
  const bool v8 = D % 16 == 0 && ldq % 8 == 0 && aligned(qkv, 16) && aligned(cs, 16) && aligned(kc, 16) && aligned(vc, 16);
  if (v8)
    hipLaunchKernelGGL(rope_cache_v8_kernel, dim3(M), dim3(256), 0, (hipStream_t)stream, (f16*)qkv, (int64_t)ldq, Hq, Hkv,
                       D, (const f16x2*)cs, pos, pos_base, slot_base, (f16*)kc, (f16*)vc, max_seq);
  else
    hipLaunchKernelGGL(rope_cache_heads_kernel, dim3(M, (Hq + 2 * Hkv + kRopeHeadsPerBlock - 1) / kRopeHeadsPerBlock),
                       dim3(64 * kRopeHeadsPerBlock), 0, (hipStream_t)stream, (f16*)qkv, (int64_t)ldq, Hq, Hkv, D,
                       (const f16x2*)cs, pos, pos_base, slot_base, (f16*)kc, (f16*)vc, max_seq);
  HI_TRY(hipGetLastError());
  return 0;
}

// Causal prefill attention of T query rows (row t at position p0 + t; head h at columns h*D of
// q [T, ldq]) over one cache slot kc / vc [Hkv][max_seq][D], keys 0..p0+t; out [T, ldo].
HI_EXPORT int hi_flash_prefill(const void* q, int ldq, const void* kc, const void* vc, int max_seq, void* out, int ldo,
                               int T, int p0, int Hq, int Hkv, int D, void* stream) {
  return flash_prefill(q, ldq, kc, vc, max_seq, out, ldo, T, p0, Hq, Hkv, D, nullptr, stream, "hi_flash_prefill");
}

// The same, and each row's log2-domain log-sum-exp of the scaled logits into lse [Hq][T] fp32.
HI_EXPORT int hi_flash_prefill_lse(const void* q, int ldq, const void* kc, const void* vc, int max_seq, void* out,
                                   int ldo, int T, int p0, int Hq, int Hkv, int D, float* lse, void* stream) {
  if (!lse) HI_FAIL("hi_flash_prefill_lse: lse must not be null");
  return flash_prefill(q, ldq, kc, vc, max_seq, out, ldo, T, p0, Hq, Hkv, D, lse, stream, "hi_flash_prefill_lse");
}
