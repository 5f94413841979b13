// Decode-step kernels around the GEMVs, behind the reference's C-ABI: split-KV decode attention
// (hi_decode_attn, hi_decode_work_bytes; src/api.cu:643-720, ctypes scripts/hipinfer.py:21-22,30)
// and the greedy argmax (hi_argmax; api.cu:838-840, kernels.cuh:1883-1931). hi_embed (the
// reference's internal embed_kernel, kernels.cuh:1876-1881, called from decode_step api.cu:1900)
// is exported as well so that a caller can assemble a whole decode step from C-ABI calls.
//
// Decode attention, one new token per sequence, for gfx950. The cache is read once, so the floor is
// its bytes; what lies above it is the chain of one launch (position, tiles, partials, counter,
// merge) and, over ragged batches, the wait for the longest blocks:
//  * block = (split, kv head, sequence); every block serves all G query heads of its kv head, so the
//    cache is read once per GQA group. A split covers a contiguous run of keys; the number of splits
//    in use is derived on the device from pos[b], so a captured graph stays valid while the context
//    grows;
//  * a wave takes 32-key tiles. Logits are S^T = K Q^T and the output O^T = V^T P^T, both on 16x16x32
//    MFMAs with the group's heads as columns (1 to 8 of 16; the products are free beside the loads).
//    K and V go straight from memory into operand registers: which key is which row of a K operand,
//    and which dim which row of a V operand, is chosen so that the logits of a lane are its P operand
//    and the V rows are read whole, the transpose being v_perms inside a lane. No LDS, no shuffle but
//    the maximum's. A tile's registers are refilled for the next tile as soon as they are used (K
//    behind the logits, V behind P.V), so a wave keeps 8 to 16 KB in flight;
//  * logits are exact fp16 products in fp32 sums, scaled by log2(e) / sqrt(D) in fp32 (the
//    reference's log2-domain softmax, kernels.cuh:1522); the weights are fp16 for P.V (as the
//    reference's tensor-core path packs them, kernels.cuh:1455-1460) and fp32 in their sum;
//  * online softmax per wave, the block's waves merged through LDS;
//  * measured, cold caches, against one key per lane with v_dot2 and K through LDS (56-64 KB of it, so
//    two blocks per CU and no overlap of loads with arithmetic inside a wave), us: 48 sequences of 100
//    to 2000 keys, 32/8 heads of 128: 49.6 -> 43.5; 64 of 1000: 51.4 -> 47.2 (5.6 TB/s); 40 of 200 to
//    1600, 32/4 heads of 64: 24.6 -> 15.4; one of 4001, 32/8 of 128: 11.7 -> 10.5; four of 700 to 800,
//    32/4 of 64: 11.1 -> 7.4;
//  * splits hand their partials (o, m, l) to the last-arriving block of their (sequence, kv head)
//    with agent-coherent (sc1) stores and loads and a relaxed agent-scope counter, which the last
//    block resets: no L2 writeback/invalidate fence (gfx950's agent-scope fence costs several
//    microseconds), and the caller's zeroed work buffer stays zeroed, as the reference requires
//    (api.cu:648-650).
#include <type_traits>

#include "hi_common.h"
#include "hi_internal.h"

namespace {

constexpr int kDecodeCounters = 4096;  // as api.cu:651: counters at a fixed offset, then partials
constexpr int kDecodeMaxSplits = 64;
constexpr int kDaTile = 32;  // keys per wave tile (one k step of P.V)

__device__ __forceinline__ float ld_coherent(const float* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_coherent(float* p, float v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Maximum (or sum) over the four 16-lane rows of a wave, each lane with the lanes of its own column.
template <bool MAX>
__device__ __forceinline__ float rows_reduce(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = MAX ? fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1])) : __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = MAX ? fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1])) : __uint_as_float(b[0]) + __uint_as_float(b[1]);
#endif
  return v;
}

// Splits in use for `len` keys when a launch has S per pair, S1 of them to give every CU its two blocks (one of
// 8 waves): of those, one per 256 keys, but down to 128 keys a split while there are at most
// 16 (what the merge requests in one round): shorter waves finish sooner, and more splits cost more
// in the merge (one sequence of 4001 keys, 32/8 heads: 16 splits 10.8 us, 32 splits 12.5; of 2500: 16
// 9.5, 10 9.9). Up to 256 keys one split, which has no partials and no merge (200 keys, two splits / one, us:
// one sequence 7.3 / 5.8, 8 of them 8.6 / 6.2, 24 10.5 / 6.9). Beyond S1, where the launch has them
// (decode_splits_max), only for runs over 1024 keys, which would end a ragged batch late.
__device__ __forceinline__ int splits_used(int len, int S, int S1) {
  if (len <= 256) return 1;
  return max(min(S1, max((len + 255) / 256, min(16, (len + 127) / 128))), min(S, (len + 1023) / 1024));
}

// LDS of one block: the waves' partial results and the split merge's tables.
template <int G, int D, int NWV>
struct DaSmem {
  float wo[NWV][G][D];
  float wm[NWV][G], wl[NWV][G];
  float sm[G][kDecodeMaxSplits], sw[G][kDecodeMaxSplits];
  int is_last;
};

template <int G, int D, int NWV>
__global__ void __launch_bounds__(NWV * 64, 3) decode_attn_kernel(
    const f16* __restrict__ q, int ldq, const f16* __restrict__ kc, const f16* __restrict__ vc, int max_seq, int Hkv,
    const int* __restrict__ pos, float* part, int* counters, int S, int S1, f16* __restrict__ out,
    int ldo, float scale_log2, int kv_slot) {
  constexpr int KS = D / 32;               // k steps of a logits product
  constexpr int DL = D / 16;               // V dims (and P.V products) per lane
  constexpr int BK = NWV * kDaTile;        // keys per block pass
  constexpr int NT = NWV * 64;
  typedef typename std::conditional<DL == 8, u32x4, u32x2>::type VT;
  __shared__ DaSmem<G, D, NWV> sh;
  // blocks in split-major order: the splits a sequence uses (split < S_eff) come first in dispatch
  // order, so they spread over the CUs instead of sharing them with blocks that exit at once
  const int nhb = gridDim.x / S;  // (sequence, kv head) pairs
  const int split = blockIdx.x / nhb, hk = blockIdx.x % Hkv, b = (blockIdx.x % nhb) / Hkv;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int Hq = Hkv * G;
  const int len = min(pos[b] + 1, max_seq);
  const int S_eff = splits_used(len, S, S1);
  if (split >= S_eff) return;
  const int chunk = (len + S_eff - 1) / S_eff;
  const int start = split * chunk, end = min(len, start + chunk);
  const int64_t cb = kv_slot >= 0 ? kv_slot : b;
  const f16* Kh = kc + (cb * Hkv + hk) * (int64_t)max_seq * D;
  const f16* Vh = vc + (cb * Hkv + hk) * (int64_t)max_seq * D;
  const __amdgpu_buffer_rsrc_t k_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<f16*>(Kh), (short)0, end * D * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t v_rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<f16*>(Vh), (short)0, end * D * 2, 0x00020000);

  const int r = lane & 15, fk = lane >> 4;
  // Logits as S^T = K Q^T (16x16x32): A row r of block a is the tile's key 8 (r / 4) + 4 a + r % 4,
  // so lane group fk of the C layout ends up with keys 8 fk .. 8 fk + 7 of head r, in order: the B
  // operand of the 32-key P.V product, without a shuffle. Rows at or past the split's end read as
  // zeros through the buffer bounds.
  const unsigned k_off = (8 * (r >> 2) + (r & 3)) * D * 2 + 16 * fk;
  // V: lane (r, fk) loads dims DL r .. of keys 8 fk + i, whole rows per instruction; P.V product n
  // takes dim n of every lane's DL as its A row, over the lane's 8 keys (D = 64: 8-byte loads of 4 dims).
  const unsigned v_off = 8 * fk * D * 2 + DL * 2 * r;
  u32x4 kf[2][KS];
  VT vf[8];
  auto load_k = [&](int t0) {
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int s = 0; s < KS; s++)
        kf[a][s] = __builtin_amdgcn_raw_buffer_load_b128(k_rs, k_off + (unsigned)t0 * (D * 2) + 4 * a * D * 2 + 64 * s,
                                                         0, 0);
  };
  auto load_v = [&](int t0) {
#pragma unroll
    for (int i = 0; i < 8; i++) {
      const unsigned off = v_off + (unsigned)t0 * (D * 2) + i * D * 2;
      if constexpr (DL == 8) vf[i] = __builtin_amdgcn_raw_buffer_load_b128(v_rs, off, 0, 0);
      else vf[i] = __builtin_amdgcn_raw_buffer_load_b64(v_rs, off, 0, 0);
    }
  };
  const int t_first = start + wave * kDaTile;
  const f16* qg = q + (int64_t)b * ldq + (hk * G + (r < G ? r : 0)) * D + 8 * fk;
  float m = -__builtin_huge_valf(), l = 0.f;  // of head r; l over this lane's keys only
  f32x4 o[DL];                                // O^T: dim DL (4 fk + i) + n of head r in o[n][i]
#pragma unroll
  for (int n = 0; n < DL; n++) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (t_first < end) {
    load_k(t_first);
    __builtin_amdgcn_sched_barrier(0);
    u32x4 qf[KS];
#pragma unroll
    for (int s = 0; s < KS; s++) qf[s] = *reinterpret_cast<const u32x4*>(qg + 32 * s);
    load_v(t_first);
    // One tile; the next tile's K is requested as soon as this one's is used, and so is its V.
    auto tile = [&](int t0, auto last) {
      constexpr bool LAST = decltype(last)::value;
      f32x4 sc[2];
#pragma unroll
      for (int a = 0; a < 2; a++) {
        sc[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; s++)
          sc[a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, kf[a][s]),
                                                         __builtin_bit_cast(f16x8, qf[s]), sc[a], 0, 0, 0);
      }
      if constexpr (!LAST) {
        __builtin_amdgcn_sched_barrier(0);
        load_k(t0 + BK);
        __builtin_amdgcn_sched_barrier(0);
      }
      float p[8];
      float mx = -__builtin_huge_valf();
#pragma unroll
      for (int k = 0; k < 8; k++) {
        p[k] = sc[k >> 2][k & 3] * scale_log2;
        if (LAST && t0 + 8 * fk + k >= end) p[k] = -__builtin_huge_valf();
        mx = fmaxf(mx, p[k]);
      }
      const float m_old = m;
      m = fmaxf(m, rows_reduce<true>(mx));
      // -inf while every logit so far is (an infinity in K or q): their weights are 0
      const float mn = m == -__builtin_huge_valf() ? 0.f : m;
      const float alpha = exp2f(m_old - mn);  // 0 on the first tile (m = -inf)
      float ps = 0.f;
      f16x8 pf;
#pragma unroll
      for (int k = 0; k < 8; k++) {
        p[k] = exp2f(p[k] - mn);
        ps += p[k];
        pf[k] = (f16)p[k];
      }
      l = __builtin_fmaf(l, alpha, ps);
#pragma unroll
      for (int n = 0; n < DL; n++)
#pragma unroll
        for (int i = 0; i < 4; i++) o[n][i] *= alpha;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < DL; n++) {
        u32x4 w;
#pragma unroll
        for (int k = 0; k < 4; k++)
          w[k] = __builtin_amdgcn_perm(vf[2 * k + 1][n >> 1], vf[2 * k][n >> 1], n & 1 ? 0x07060302u : 0x05040100u);
        o[n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), pf, o[n], 0, 0, 0);
      }
      if constexpr (!LAST) {
        __builtin_amdgcn_sched_barrier(0);
        load_v(t0 + BK);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    int t0 = t_first;
    for (; t0 + BK < end; t0 += BK) tile(t0, std::false_type{});
    tile(t0, std::true_type{});
  }
  l = rows_reduce<false>(l);

  // ---- merge the block's waves (a wave without keys has m = -inf and weight 0)
  if (r < G) {
    if (fk == 0) {
      sh.wm[wave][r] = m;
      sh.wl[wave][r] = l;
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int n = 0; n < DL; n += 4)
        *reinterpret_cast<f32x4*>(&sh.wo[wave][r][DL * (4 * fk + i) + n]) =
            f32x4{o[n][i], o[n + 1][i], o[n + 2][i], o[n + 3][i]};
  }
  __syncthreads();
  const bool single = S_eff == 1;
  float* po = part + (int64_t)kDecodeCounters;  // partials follow the counters (floats)
  for (int i = tid; i < G * D; i += NT) {
    const int g = i / D, d = i % D;
    float M = -__builtin_huge_valf();
#pragma unroll
    for (int w = 0; w < NWV; w++) M = fmaxf(M, sh.wm[w][g]);
    float L = 0.f, O = 0.f;
#pragma unroll
    for (int w = 0; w < NWV; w++) {
      const float f = sh.wm[w][g] == -__builtin_huge_valf() ? 0.f : exp2f(sh.wm[w][g] - M);
      L = __builtin_fmaf(sh.wl[w][g], f, L);
      O = __builtin_fmaf(sh.wo[w][g][d], f, O);
    }
    if (single) {
      out[(int64_t)b * ldo + (hk * G + g) * D + d] = (f16)(O / L);
    } else {
      const int64_t pi = ((int64_t)b * Hq + hk * G + g) * kDecodeMaxSplits + split;
      st_coherent(po + pi * (D + 2) + d, O);
      if (d == 0) {
        st_coherent(po + pi * (D + 2) + D, M);
        st_coherent(po + pi * (D + 2) + D + 1, L);
      }
    }
  }
  if (single) return;
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): this thread's partial stores are complete
  __syncthreads();
  if (tid == 0) {
    int* ctr = counters + b * Hkv + hk;
    const int done = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    sh.is_last = done == S_eff - 1;
    if (sh.is_last) __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next launch
  }
  __syncthreads();
  if (!sh.is_last) return;
  // ---- the last block merges the S_eff splits of every head of its group, in split order. The
  //      (m, l) pairs and the first 16 splits' partial outputs are requested in one round; the
  //      split weights exp2(m_s - M) / L are formed once per head while those loads are in flight.
  constexpr int EPT = (G * D + NT - 1) / NT;  // output elements per thread
  float v0[EPT][16];
#pragma unroll
  for (int e = 0; e < EPT; e++) {
    const int i = tid + e * NT;
    const int g = min(i / D, G - 1), d = i % D;
    const float* pp = po + ((int64_t)b * Hq + hk * G + g) * kDecodeMaxSplits * (D + 2) + d;
#pragma unroll
    for (int k = 0; k < 16; k++) v0[e][k] = ld_coherent(pp + (int64_t)min(k, S_eff - 1) * (D + 2));
  }
  for (int i = tid; i < G * S_eff; i += NT) {
    const int g = i / S_eff, s2 = i - g * S_eff;
    const float* pp = po + (((int64_t)b * Hq + hk * G + g) * kDecodeMaxSplits + s2) * (D + 2);
    sh.sm[g][s2] = ld_coherent(pp + D);
    sh.sw[g][s2] = ld_coherent(pp + D + 1);
  }
  __syncthreads();
  for (int g = wave; g < G; g += NWV) {
    float M = -__builtin_huge_valf();
    for (int s2 = lane; s2 < S_eff; s2 += 64) M = fmaxf(M, sh.sm[g][s2]);
    M = wave_max(M);
    float Lp = 0.f;
    for (int s2 = lane; s2 < S_eff; s2 += 64)
      Lp = __builtin_fmaf(sh.sw[g][s2], exp2f(sh.sm[g][s2] - M), Lp);
    const float Lt = wave_sum(Lp);
    for (int s2 = lane; s2 < S_eff; s2 += 64) sh.sw[g][s2] = exp2f(sh.sm[g][s2] - M) / Lt;
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < EPT; e++) {
    const int i = tid + e * NT;
    if (i < G * D) {
      const int g = i / D, d = i % D;
      const float* pp = po + ((int64_t)b * Hq + hk * G + g) * kDecodeMaxSplits * (D + 2) + d;
      float O = 0.f;
#pragma unroll
      for (int k = 0; k < 16; k++) O = __builtin_fmaf(v0[e][k], k < S_eff ? sh.sw[g][k] : 0.f, O);
      for (int s0 = 16; s0 < S_eff; s0 += 16) {
        float v[16];
#pragma unroll
        for (int k = 0; k < 16; k++) v[k] = ld_coherent(pp + (int64_t)min(s0 + k, S_eff - 1) * (D + 2));
#pragma unroll
        for (int k = 0; k < 16; k++) O = __builtin_fmaf(v[k], s0 + k < S_eff ? sh.sw[g][s0 + k] : 0.f, O);
      }
      out[(int64_t)b * ldo + (hk * G + g) * D + d] = (f16)O;
    }
  }
}

// Splits of a (sequence, kv head) pair that give every CU two blocks (as api.cu:643-646), at most the
// work buffer's 64.
int decode_splits(int B, int Hkv, int cus) { return min((2 * cus + B * Hkv - 1) / (B * Hkv), kDecodeMaxSplits); }

// Blocks of 8 waves where that is 16 or more (at most about an eighth as many pairs as CUs): a launch this
// small is a chain of latencies, and a block of 256 keys is then one tile per wave (one sequence of
// 2500 keys 9.45 -> 9.0 us, of 8000 14.8 -> 13.8, four of 700 to 800 at D = 64 8.1 -> 7.4); with more
// pairs 4 waves balance better (40 sequences of 300 to 2400, 12/2 heads: 19.5 against 25.5). A CU holds one
// such block at D = 128 (12 waves of 137 registers), so the launch has at most one for each: with two, the
// lengths that use more than half of them run a part-filled second round (32/8 heads of 128, two / one, us: one
// sequence of 12000 21.4 / 17.0, two of 6000 20.8 / 16.7, four of 2000 15.3 / 11.9, one of 32000 34.4 / 29.6; two
// of 6000, 32/4 heads of 64, 10.5 / 10.4, of 20000 18.5 / 15.3).
constexpr int kDaWideSplits = 16;
int decode_splits_wide(int B, int Hkv, int cus) { return min(max(cus / (B * Hkv), 1), kDecodeMaxSplits); }

// Splits per pair that a launch has for its long runs (splits_used): 2 S1, or S1 where more would be spread
// worse over the CUs. A batch may be uniform, all of its pairs then take S1 + 1 splits at once: S1 blocks
// a pair that are a whole number for every CU stay that, and so do those whose last layer over the CUs
// would be left emptier by more than a sixteenth of all layers. At S1 = 1 a second split also brings the
// partials and their merge, and a part-filled second round of blocks (a CU holds 3 at D = 128). Measured
// with 32/8 heads of 128, S1 alone / up to 2 S1, us: 64 x 1025 keys 49.6 / 55.1, 64 x 2000 94.1 / 100.5,
// 120 x 1025 91.6 / 101.8, 16 x 4097 52.8 / 57.1, 44 x 2049 70.9 / 76.7; 24 x 3073 66.0 / 60.6, 52 x 2049
// 89.5 / 85.8, 30 of 500 to 4000 70.0 / 66.0, 24 of 576 to 4608 68.8 / 54.5. It reads no lengths: a
// sequence's sums do not depend on its neighbours'.
int decode_splits_max(int B, int Hkv, int S1, int cus) {
  const int n0 = B * Hkv * S1, n1 = n0 + B * Hkv;  // blocks
  const int l0 = (n0 + cus - 1) / cus, l1 = (n1 + cus - 1) / cus;  // layers of one block a CU
  // n0 / (l0 cus) and n1 / (l1 cus) are the shares of the layers that are filled
  const bool worse = S1 == 1 || n0 % cus == 0 || 16 * ((int64_t)n0 * l1 - (int64_t)n1 * l0) > (int64_t)l0 * l1 * cus;
  return worse ? S1 : min(2 * S1, kDecodeMaxSplits);
}

template <int D>
int decode_attn_d(int G, dim3 grid, hipStream_t s, const f16* q, int ldq, const f16* kc, const f16* vc, int max_seq,
                  int Hkv, const int* pos, float* part, int* counters, int S, int S1, bool wide, f16* out, int ldo,
                  float sl2, int kv_slot) {
#define HI_DA(g)                                                                                              \
  case g:                                                                                                     \
    if (wide)                                                                                                 \
      hipLaunchKernelGGL((decode_attn_kernel<g, D, 8>), grid, dim3(512), 0, s, q, ldq, kc, vc, max_seq, Hkv,  \
                         pos, part, counters, S, S1, out, ldo, sl2, kv_slot);                                     \
    else                                                                                                      \
      hipLaunchKernelGGL((decode_attn_kernel<g, D, 4>), grid, dim3(256), 0, s, q, ldq, kc, vc, max_seq, Hkv,  \
                         pos, part, counters, S, S1, out, ldo, sl2, kv_slot);                                     \
    break;
  switch (G) {
    HI_DA(1) HI_DA(2) HI_DA(3) HI_DA(4) HI_DA(5) HI_DA(6) HI_DA(7) HI_DA(8)
    default: HI_FAIL("hi_decode_attn: unsupported GQA group %d (1..8)", G);
  }
#undef HI_DA
  HI_TRY(hipGetLastError());
  return 0;
}

// ---- greedy argmax: largest logit, NaN above every number, lowest index on ties; a row of -inf
//      gives 0 (kernels.cuh:1883-1931)
__device__ __forceinline__ bool argmax_better(float v, int i, float best, int bi) {
  const bool vn = v != v, bn = best != best;
  if (vn != bn) return vn;
  return (vn || v == best) ? i < bi : v > best;
}

constexpr int kArgmaxThreads = 1024;
constexpr int kArgmaxLoads = 16;
__global__ void __launch_bounds__(kArgmaxThreads) argmax_kernel(const f16* __restrict__ logits, int V,
                                                                int* __restrict__ tok_out) {
  __shared__ float bv[kArgmaxThreads / 64];
  __shared__ int bi[kArgmaxThreads / 64];
  const f16* row = logits + (int64_t)blockIdx.x * V;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  float best = -__builtin_huge_valf();
  int idx = 0;
  auto scan = [&](int i) {  // one logit by the exact rule
    const float v = (float)row[i];
    if (argmax_better(v, i, best, idx)) { best = v; idx = i; }
  };
  if (((uintptr_t)row & 15) == 0) {  // 8 logits per 16-byte chunk, then the tail
    // Thread t takes chunks t, t + kArgmaxThreads, ..., issuing up to kArgmaxLoads loads before
    // looking at any (a 128K vocabulary row in one round trip). Per chunk, packed fp16 max and
    // add only: the chunk's max against the thread's best (strictly greater replaces it, so the
    // thread keeps its lowest chunk holding its max), and a running sum that turns NaN if any
    // logit is NaN (or, harmlessly, if +inf and -inf overflow meet). Afterwards the thread finds
    // its index inside that chunk (reloaded from L2; keeping its words in registers measured no
    // faster); a thread whose sum is NaN rescans its chunks by the exact rule.
    const int V8 = V / 8;
    f16 cbest = (f16)(-__builtin_huge_valf());
    int cidx = tid < V8 ? tid : -1;
    f16x2 nsum = {(f16)0.f, (f16)0.f};
    for (int c0 = tid; c0 < V8; c0 += kArgmaxThreads * kArgmaxLoads) {
      u32x4 v[kArgmaxLoads];
#pragma unroll
      for (int u = 0; u < kArgmaxLoads; u++) {
        const int c = c0 + u * kArgmaxThreads;
        v[u] = c < V8 ? *reinterpret_cast<const u32x4*>(row + 8 * c) : u32x4{0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int u = 0; u < kArgmaxLoads; u++) {
        const int c = c0 + u * kArgmaxThreads;
        if (c < V8) {
          const f16x2 x0 = as_h2(v[u][0]), x1 = as_h2(v[u][1]), x2 = as_h2(v[u][2]), x3 = as_h2(v[u][3]);
          const f16x2 m = __builtin_elementwise_max(__builtin_elementwise_max(x0, x1), __builtin_elementwise_max(x2, x3));
          const f16 cm = m.x > m.y ? m.x : m.y;
          nsum += (x0 + x1) + (x2 + x3);
          if (cm > cbest) {
            cbest = cm;
            cidx = c;
          }
        }
      }
    }
    if (nsum.x != nsum.x || nsum.y != nsum.y) {
      for (int c = tid; c < V8; c += kArgmaxThreads)
        for (int i = 8 * c; i < 8 * c + 8; i++) scan(i);
    } else if (cidx >= 0) {
      const u32x4 w = *reinterpret_cast<const u32x4*>(row + 8 * cidx);
      best = (float)cbest;
      idx = 8 * cidx + 7;
#pragma unroll
      for (int e = 7; e >= 0; e--)  // the first logit equal to the chunk's max (-0 equals +0)
        if ((float)as_h2(w[e >> 1])[e & 1] == best) idx = 8 * cidx + e;
    }
    for (int i = 8 * V8 + tid; i < V; i += kArgmaxThreads) scan(i);
  } else {
    for (int i = tid; i < V; i += kArgmaxThreads) scan(i);
  }
  for (int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, 64);
    const int oi = __shfl_xor(idx, o, 64);
    if (argmax_better(ov, oi, best, idx)) { best = ov; idx = oi; }
  }
  if (lane == 0) {
    bv[wave] = best;
    bi[wave] = idx;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < kArgmaxThreads / 64; w++)
      if (argmax_better(bv[w], bi[w], best, idx)) { best = bv[w]; idx = bi[w]; }
    tok_out[blockIdx.x] = idx;
  }
}

// ---- embedding rows: x[b] = table[tok[b]] (H halves), 16 bytes per thread
__global__ void __launch_bounds__(256) embed_kernel(const int* __restrict__ tok, const f16* __restrict__ table, int V,
                                                    int H, f16* __restrict__ x, int64_t ldx) {
  const int b = blockIdx.x;
  const int t = tok[b];
  if (t < 0 || t >= V) return;  // an id outside the vocabulary leaves the row untouched
  const u32x4* src = reinterpret_cast<const u32x4*>(table + (int64_t)t * H);
  u32x4* dst = reinterpret_cast<u32x4*>(x + (int64_t)b * ldx);
  for (int i = threadIdx.x; i < H / 8; i += blockDim.x) dst[i] = src[i];
}

}  // namespace

// Work bytes for hi_decode_attn (as api.cu:651-655): 4096 int counters the caller zeroes once (the
// kernel leaves them zeroed), then B * Hq * 64 * (D + 2) fp32 partials.
HI_EXPORT size_t hi_decode_work_bytes(int B, int Hq, int Hkv, int D) {
  (void)Hkv;
  return (size_t)kDecodeCounters * 4 + (size_t)(B > 0 ? B : 0) * (Hq > 0 ? Hq : 0) * kDecodeMaxSplits * (D + 2) * 4;
}

static int decode_attn_run(const void* q, int ldq, const void* kc, const void* vc, int max_seq, const int* pos,
                           void* out, int ldo, int B, int Hq, int Hkv, int D, void* work, int kv_slot, void* s,
                           const char* who) {
  const HiDevice* d = hi_device();
  if (!d) return -2;
  if (D != 64 && D != 128) HI_FAIL("%s: head dim %d (64 or 128)", who, D);
  if (B < 0 || Hkv < 1 || Hq < Hkv || Hq % Hkv || Hq / Hkv > 8 || max_seq < 1)
    HI_FAIL("%s: B %d, Hq %d, Hkv %d (Hq / Hkv in 1..8), max_seq %d", who, B, Hq, Hkv, max_seq);
  if (B == 0) return 0;
  if ((int64_t)max_seq * D * 2 > INT32_MAX)  // a head's cache rows are addressed by 32-bit byte offsets
    HI_FAIL("%s: max_seq %d too long for 32-bit cache offsets (at most %d at D=%d)", who, max_seq,
            (int)(INT32_MAX / (2 * D)), D);
  if (B * Hkv > kDecodeCounters) HI_FAIL("%s: B*Hkv %d > %d", who, B * Hkv, kDecodeCounters);
  if (!q || !kc || !vc || !pos || !out || !work) HI_FAIL("%s: null pointer", who);
  if (((uintptr_t)q & 15) || ldq % 8 || ((uintptr_t)kc & 15) || ((uintptr_t)vc & 15) || ((uintptr_t)work & 3) ||
      (((uintptr_t)out) & 1))
    HI_FAIL("%s: q, kc and vc must be 16-byte aligned and ldq a multiple of 8", who);
  if (ldq < Hq * D || ldo < Hq * D) HI_FAIL("%s: ldq %d / ldo %d < Hq * D = %d", who, ldq, ldo, Hq * D);
  // one sequence (kv_slot >= 0): a batch of one's split count, so every row matches that decode
  const int Bs = kv_slot >= 0 ? 1 : B;
  int S1 = decode_splits(Bs, Hkv, d->cus), S;
  const bool wide = S1 >= kDaWideSplits;
  if (wide) S = S1 = decode_splits_wide(Bs, Hkv, d->cus);
  else S = decode_splits_max(Bs, Hkv, S1, d->cus);
  const float sl2 = 1.4426950408889634f / sqrtf((float)D);
  const dim3 grid(S * Hkv * B);  // split-major: (split, sequence, kv head)
  int* counters = (int*)work;
  float* part = (float*)work;
  const hipStream_t st = (hipStream_t)s;
  if (D == 64)
    return decode_attn_d<64>(Hq / Hkv, grid, st, (const f16*)q, ldq, (const f16*)kc, (const f16*)vc, max_seq, Hkv, pos,
                             part, counters, S, S1, wide, (f16*)out, ldo, sl2, kv_slot);
  return decode_attn_d<128>(Hq / Hkv, grid, st, (const f16*)q, ldq, (const f16*)kc, (const f16*)vc, max_seq, Hkv, pos,
                            part, counters, S, S1, wide, (f16*)out, ldo, sl2, kv_slot);
}

// out[b, h*D : (h+1)*D] = softmax(q_h . K[0..pos[b]] / sqrt(D)) V for every query head h of
// sequence b, K/V read from cache slot b ([slots][Hkv][max_seq][D] fp16), the kv head of h being
// h / (Hq / Hkv). work: hi_decode_work_bytes(B, Hq, Hkv, D) bytes, zeroed once by the caller.
HI_EXPORT int hi_decode_attn(const void* q, int ldq, const void* kc, const void* vc, int max_seq, const int* pos,
                             void* out, int ldo, int B, int Hq, int Hkv, int D, void* work, void* s) {
  return decode_attn_run(q, ldq, kc, vc, max_seq, pos, out, ldo, B, Hq, Hkv, D, work, -1, s, "hi_decode_attn");
}

int decode_attn_slot(const void* q, int ldq, const void* kc, const void* vc, int max_seq, const int* pos, void* out,
                     int ldo, int R, int Hq, int Hkv, int D, void* work, int kv_slot, hipStream_t s) {
  if (kv_slot < 0) HI_FAIL("decode_attn_slot: kv_slot %d < 0", kv_slot);
  return decode_attn_run(q, ldq, kc, vc, max_seq, pos, out, ldo, R, Hq, Hkv, D, work, kv_slot, s, "decode_attn_slot");
}

// tok_out[b] = argmax of logits[b, 0:V] (fp16): NaN ranks above every number, ties go to the
// lowest index, an all -inf row gives 0 (api.cu:838-840).
HI_EXPORT int hi_argmax(const void* logits, int B, int V, int* tok_out, void* s) {
  if (!hi_device()) return -2;
  if (B < 0 || V < 1) HI_FAIL("hi_argmax: B %d, V %d", B, V);
  if (B == 0) return 0;
  if (!logits || !tok_out || ((uintptr_t)logits & 1)) HI_FAIL("hi_argmax: null or misaligned pointer");
  hipLaunchKernelGGL(argmax_kernel, dim3(B), dim3(kArgmaxThreads), 0, (hipStream_t)s, (const f16*)logits, V, tok_out);
  HI_TRY(hipGetLastError());
  return 0;
}

// x[b, 0:H] = table[tok[b], 0:H] for b < B (no reference export: the reference's engine runs its
// embed_kernel internally). Token ids outside [0, V) leave the row untouched.
HI_EXPORT int hi_embed(const int* tok, const void* table, int V, int H, void* x, int ldx, int B, void* s) {
  if (!hi_device()) return -2;
  if (B < 0 || V < 1 || H < 8 || H % 8 || ldx % 8 || ldx < H) HI_FAIL("hi_embed: B %d V %d H %d ldx %d", B, V, H, ldx);
  if (B == 0) return 0;
  if (!tok || !table || !x || ((uintptr_t)table & 15) || ((uintptr_t)x & 15))
    HI_FAIL("hi_embed: null pointer or table / x not 16-byte aligned");
  hipLaunchKernelGGL(embed_kernel, dim3(B), dim3(256), 0, (hipStream_t)s, tok, (const f16*)table, V, H, (f16*)x,
                     (int64_t)ldx);
  HI_TRY(hipGetLastError());
  return 0;
}
