// Prefill GEMM for gfx950: C[M, N'] (epi) A[M, K] @ W[N, K]^T with fp16 MFMA and fp32 accumulation.
//
// Replaces the reference's portable WMMA gemm_kernel<BM, BN, BK, WGM, WGN, EPI, Q8>
// (src/kernels.cuh:305-506) behind the same C-ABI (hi_gemm, hi_gemm_w8; api.cu:566-577).
//
// Design:
//  * a block of WM x WN waves (4 or 8) owns a BM x BN output tile; each wave a (BM/WM) x (BN/WN)
//    sub-tile built from v_mfma_f32_32x32x16_f16 tiles (A and W are both K-contiguous, so each
//    lane's 8-half fragment is one 16-byte LDS read). The big tiles give each wave a 128 x 128 (or
//    128 x 64) sub-tile, so every 16-byte fragment read feeds four (or two) MFMAs; with 8 waves two
//    share each SIMD, so one wave's MFMAs cover the other's LDS waits, barrier and DMA issue;
//  * K advances in 64-deep tiles through an S-stage ring in LDS fed by gfx950's direct
//    global->LDS loads (global_load_lds_dwordx4): no register staging, the next S-1 tiles in flight
//    while the MFMAs consume the current one;
//  * within a tile the fragments of step s+1 are read from LDS while the MFMAs of step s run (the
//    order is pinned with scheduling-group barriers: MFMA, LDS read, MFMA, ...); the one barrier
//    per tile sits before the last step, after its fragments are in registers, and frees the tile's
//    stage. The DMA that refills it goes out in parts behind the MFMAs of the following steps: issued
//    in one burst after the barrier, a wave's 8-16 DMA instructions held up its own MFMAs while the
//    CU's L1 path (64 B per clock) worked through 64 KB. Measured on one card each, cold weights,
//    burst -> parts: M = 2048, N = 28672, K = 4096 (256 x 256) 440 -> 416 us; M = 2048, N = 4096,
//    K = 14336 (256 x 128) 236 -> 217; M = 1000, N = 5120, K = 3072 (128 x 160) 41.4 -> 39.0; int8
//    M = 333, N = 17920, K = 1536 32.4 -> 30.8; M = 512, N = 11264, K = 2048 34.3 -> 31.4.
//    The refill is unconditional (past the split's last tile it re-reads the first), so the loop
//    body has no branch and its DMA waits are compile-time counts;
//  * LDS rows hold 16-byte chunks at positions XOR-swizzled by the row (c ^ ((r >> 1) & 7) for
//    128-byte rows, c ^ ((r >> 2) & 3) for 64-byte int8 rows): the 16 lanes one 128-bit read serves
//    per cycle then cover all 64 banks. The swizzle is applied on the global side (each DMA lane
//    fetches the chunk that belongs at its fixed LDS slot);
//  * the k order inside each 32-deep half tile is permuted identically for A and W: step 2j + h
//    gives lane (row, half fk) the k values 32j + 16 fk + 8 h + 0..7. An int8 lane then reads its
//    two steps' 16 weights as one 16-byte chunk (a conflict-free 128-bit read) and dequantises
//    them per fragment: exact int8 -> fp16 unpack, one packed fp16 multiply by the row scale =
//    fp16(q * s), the weight the reference's int8 GEMM computes with (kernels.cuh:86-94, 336-341);
//  * the DMA goes through buffer resources based at the block's first rows, so each lane keeps
//    32-bit offsets only and rows past M or N read zeros (never stored); a K tail of 32
//    (K % 64 == 32) is the last tile's first half only, handled outside the main loop;
//  * the tile index is remapped so each of the 8 XCDs (blocks are dealt round-robin across them)
//    gets a contiguous run of tiles, rasterised in groups of 8 tile rows, so the A and W panels a
//    run needs stay in that XCD's L2;
//  * the W fragment is the MFMA's first operand, so each lane ends with 16 results of ONE output
//    row, four consecutive columns per register quad: the epilogue stores 8 bytes at a time, and
//    a gate column and its up column (16 apart) sit in the same lane -- no cross-lane traffic;
//  * epilogues (reference kernels.cuh:454-505): 0 store (+ bias, fp32 before the rounding),
//    1 residual (fp16 add), 2 SwiGLU over 16-column gate/up groups;
//  * split-K: gridDim.y blocks share a tile and write fp32 partials [split][M][N]; a second kernel
//    sums them in split order (deterministic) and runs the epilogue. The kernel boundary makes the
//    partials visible across XCDs; an in-kernel "last block reduces" handoff would need an
//    agent-scope fence, which writes back and invalidates the XCD's L2 on this part.
#pragma once
#include <type_traits>

#include "hi_common.h"

struct GemmArgs {
  const f16* A;
  int64_t lda;
  const void* W;       // [N, K] fp16 or int8
  const f16* scales;   // int8 row scales [N] or nullptr
  const f16* bias;     // [N] (epilogue 0) or nullptr
  f16* C;
  int64_t ldc;
  int M, N, K;
  int kt_per_split;    // K tiles per split (gridDim.y splits)
  float* ws;           // split-K partials: [splits][M][N] fp32
  bool vec_c;          // C (and the residual read) allow 8-byte accesses: C 8-byte aligned, ldc % 4 == 0
  bool vec16_c;        // ... and 16-byte ones (C 16-byte aligned, ldc % 8 == 0): the LDS-staged epilogue
  // grouped mode (MoE experts): group e owns sorted rows [grp_off[e], grp_off[e+1]) and the
  // weights at W + e * grp_wstride bytes; its row tiles are [grp_tiles[e], grp_tiles[e+1]) of the
  // global row-tile count (block id / column tiles). Sorted row q is A row q and C row q, unless
  // grp_perm is given: then with grp_gather A row q is A row grp_perm[q] / grp_k (A has
  // grp_a_rows rows; rows are gathered by the tile DMA itself), and with grp_scatter C row q is
  // C row grp_perm[q]
  const int* grp_off;
  const int* grp_tiles;
  int grp_n;
  int64_t grp_wstride;
  const int* grp_perm;
  int grp_k, grp_a_rows;
  bool grp_gather, grp_scatter;
  // epilogue 1 with split-K only: the second pass also writes norm_y = RMSNorm(C) * norm_w (rows
  // of N <= 8192 halves, C and norm_y contiguous: ldc == N); nullptr: the plain second pass
  const f16* norm_w;
  f16* norm_y;
  float norm_eps;
};

constexpr int kGemmBK = 64;
constexpr int kGemmMaxGroups = 256;  // grouped mode: at most this many groups (MoE experts)
// Four consecutive fp16 values at p: one 8-byte access when `vec` (p 8-byte aligned), else four.
__device__ __forceinline__ f16x4 load4(const f16* p, bool vec) {
  if (vec) return *reinterpret_cast<const f16x4*>(p);
  return f16x4{p[0], p[1], p[2], p[3]};
}
__device__ __forceinline__ void store4(f16* p, f16x4 v, bool vec) {
  if (vec) {
    *reinterpret_cast<f16x4*>(p) = v;
  } else {
    p[0] = v[0];
    p[1] = v[1];
    p[2] = v[2];
    p[3] = v[3];
  }
}

// Half offset of logical 16-byte chunk `c` of row `r` in an LDS tile of BK-half rows (256, 128 or
// 64 bytes): the XOR term spreads the 16 rows one 128-bit read serves per cycle over all 64 banks.
template <int BK>
__device__ __forceinline__ int lds_off(int r, int c) {
  if constexpr (BK == 128) return r * 128 + ((c ^ (r & 15)) << 3);
  else if constexpr (BK == 64) return r * 64 + ((c ^ ((r >> 1) & 7)) << 3);
  else return r * 32 + ((c ^ ((r >> 2) & 3)) << 3);
}
// Byte offset of logical 16-byte chunk `c` of row `r` in an LDS tile of BK-byte int8 rows.
template <int BK>
__device__ __forceinline__ int lds_off8(int r, int c) {
  if constexpr (BK == 64) return r * 64 + ((c ^ ((r >> 2) & 3)) << 4);
  else return r * 32 + ((c ^ ((r >> 3) & 1)) << 4);
}

// Scheduling pattern of one step: behind each of the step's NM MFMAs one of the ND LDS reads of the
// next step's fragments, then the NV DMA instructions of the refill under way, spread over the MFMAs
// left (then whichever is left over). The reads are issued early and their latency hides under the
// matrix work instead of being sunk next to their first use, and no DMA instruction queues up
// behind another one in front of the MFMAs.
template <int NM, int ND, int NV = 0>
__device__ __forceinline__ void sched_step() {
  constexpr int P = ND < NM ? ND : NM, R = NM - P;  // MFMAs before and after the last read
#pragma unroll
  for (int i = 0; i < P; i++) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
  }
  if constexpr (ND > P) __builtin_amdgcn_sched_group_barrier(0x100, ND - P, 0);
  int v = 0;
#pragma unroll
  for (int i = 0; i < R; i++) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
#pragma unroll
    for (; v * R < (i + 1) * NV; v++) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // DMA
  }
#pragma unroll
  for (; v < NV; v++) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
}

// Grouped mode: what a thread loads of the groups before anything else (thread e < grp_n its group's tile
// start and first row, thread 0 also the totals).
struct GrpLoad {
  int tile, off, tiles_all, off_all;
};
__device__ __forceinline__ GrpLoad grp_load(const GemmArgs& g) {
  GrpLoad l{};
  const int tid = threadIdx.x;
  if (tid < g.grp_n) {
    l.tile = g.grp_tiles[tid];
    l.off = g.grp_off[tid];
  }
  if (tid == 0) {
    l.tiles_all = g.grp_tiles[g.grp_n];
    l.off_all = g.grp_off[g.grp_n];
  }
  return l;
}

template <int BM, int BN, int WM, int WN, int S, int EPI, bool Q8, bool GRP = false, int BK = 64, int KG = 1, int SB = S>
__global__ void __launch_bounds__(64 * WM * WN * KG) gemm_kernel(GemmArgs g) {
  constexpr bool PRELOADED = false;
  constexpr GrpLoad loaded{};
#include "gemm_body.h"
}

// Grouped mode with the tile's shape chosen on the device, which knows the groups' sizes: BM x BN or, where
// grp_tiles[grp_n + 1] is not 0, BN x BM (and WN x WM waves; the wave tile, the ring and the order of the sums
// are the same). That word is loaded with the groups, so the choice costs no round trip of its own.
template <int BM, int BN, int WM, int WN, int S, int EPI, int BK>
__device__ __forceinline__ void gemm_grp_shape(GemmArgs g, GrpLoad loaded) {
  constexpr bool Q8 = false, GRP = true, PRELOADED = true;
  constexpr int KG = 1, SB = S;
#include "gemm_body.h"
}
template <int BM, int BN, int WM, int WN, int S, int EPI, int BK>
__global__ void __launch_bounds__(64 * WM * WN) gemm_grp_kernel(GemmArgs g) {
  const int turned = g.grp_tiles[g.grp_n + 1];
  const GrpLoad loaded = grp_load(g);
  if (turned == 0)
    gemm_grp_shape<BM, BN, WM, WN, S, EPI, BK>(g, loaded);
  else
    gemm_grp_shape<BN, BM, WN, WM, S, EPI, BK>(g, loaded);
}

// Split-K second pass: sum the fp32 partials [splits][M][N] in split order (deterministic) and run
// the epilogue with the main kernel's rounding; each thread owns 4 consecutive output columns.
template <int EPI>
__global__ void __launch_bounds__(256) gemm_splitk_reduce(const float* __restrict__ ws, int splits, int M, int N,
                                                          const f16* __restrict__ bias, f16* C, int64_t ldc,
                                                          bool vec_c) {
  const int n_out = EPI == 2 ? N / 2 : N;
  const int64_t idx = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (idx >= (int64_t)M * n_out) return;
  const int row = (int)(idx / n_out), oc = (int)(idx - (int64_t)row * n_out);
  const int64_t plane = (int64_t)M * N;
  f16* dst = C + (int64_t)row * ldc + oc;
  f16x4 o;
  if constexpr (EPI == 2) {
    const int gc = (oc >> 4) * 32 + (oc & 15);  // gate column; its up column is gc + 16
    f32x4 gs = {0.f, 0.f, 0.f, 0.f}, us = gs;
    for (int z = 0; z < splits; z++) {
      gs += *reinterpret_cast<const f32x4*>(ws + z * plane + (int64_t)row * N + gc);
      us += *reinterpret_cast<const f32x4*>(ws + z * plane + (int64_t)row * N + gc + 16);
    }
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = silu_mul_fast(gs[e], us[e]);
  } else {
    f32x4 t = {0.f, 0.f, 0.f, 0.f};
    for (int z = 0; z < splits; z++) t += *reinterpret_cast<const f32x4*>(ws + z * plane + (int64_t)row * N + oc);
    if constexpr (EPI == 1) {
      const f16x4 r = load4(dst, vec_c);
#pragma unroll
      for (int e = 0; e < 4; e++) o[e] = r[e] + (f16)t[e];
    } else {
      f16x4 b = {(f16)0.f, (f16)0.f, (f16)0.f, (f16)0.f};
      if (bias) b = load4(bias + oc, ((uintptr_t)bias & 7) == 0);
#pragma unroll
      for (int e = 0; e < 4; e++) o[e] = (f16)(t[e] + (float)b[e]);
    }
  }
  store4(dst, o, vec_c);
}

// Tile configurations: {BM, BN, WM, WN, stages, BK[, K groups]}; WM x WN waves per K group, BK-deep
// K tiles. The
// 32-deep ones give the big 8-wave tiles four (or six) stages in the same LDS as two 64-deep
// ones: more K tiles in flight to cover the global->LDS latency. 128 x 160 and 128 x 96 (four
// waves stacked along M, each 32 rows by the whole width) cut N = 5120 and N = 3072 at M = 1024
// into exactly 256 tiles, one per CU, with no split-K. 32 x 256 (four waves side by side, 32 x 64
// each) serves batched decode (M <= 32) on the widest projections: 32 KB of weights per stage.
// 256 x 192 (eight waves of 64 x 96) cuts N = 3072 at M = 1024 into 64 big tiles, 256 blocks with
// a 4-way split-K: half the staged bytes of 128 x 96 for the same K range. The two 128-deep small
// tiles (fp16 weights, K % 128 == 0) fetch each W row in 256-byte runs per K tile instead of
// 128-byte ones, for the weight-streaming small-M shapes. The last, 128 x 160 in two K groups
// (eight waves: two 4-wave pipelines on the two halves of the K tiles, each with its own 2-stage
// ring, group 1's sums handed to group 0 through LDS at the end), puts two waves on each SIMD
// for the same one-tile-per-CU cut of N = 5120: QKV of Llama-3.2-3B at M = 1024 in 42.3 against
// 45.6 us. The same split of 128 x 96 (o, down) measured no faster, and neither did four-wave
// tiles whose waves hold 64 rows (37 % fewer LDS fragment reads per MFMA): neither latency nor the
// LDS reads bound the narrow tiles.
struct GemmCfg {
  int bm, bn, wm, wn, st, bk, kg = 1;  // kg: K groups of wm x wn waves (two waves on each SIMD at kg 2)
};
constexpr GemmCfg kGemmCfgs[] = {{256, 256, 2, 2, 2, 64}, {256, 128, 2, 2, 3, 64}, {128, 256, 2, 2, 3, 64},
                                 {64, 128, 2, 2, 4, 64},  {128, 128, 2, 2, 2, 64}, {64, 64, 2, 2, 4, 64},
                                 {32, 128, 1, 4, 4, 64},  {128, 64, 2, 2, 4, 64},  {256, 256, 2, 4, 2, 64},
                                 {256, 128, 2, 4, 3, 64}, {256, 256, 2, 4, 4, 32}, {256, 128, 2, 2, 6, 32},
                                 {128, 256, 2, 4, 6, 32}, {128, 160, 4, 1, 4, 64}, {128, 96, 4, 1, 4, 64},
                                 {32, 256, 1, 4, 4, 64},  {256, 192, 4, 2, 2, 64}, {64, 128, 2, 2, 3, 128},
                                 {128, 64, 2, 2, 3, 128}, {128, 160, 4, 1, 2, 64, 2}};
constexpr int kGemmNumCfgs = sizeof(kGemmCfgs) / sizeof(kGemmCfgs[0]);
// A config exists for a weight format when its A and W tiles split into whole 1 KB DMA
// instructions per wave (int8 W rows are half as wide: 128 x 160 and 128 x 96 are fp16 only).
constexpr bool gemm_cfg_ok(int c, bool q8) {
  const int nw = kGemmCfgs[c].wm * kGemmCfgs[c].wn, bk = kGemmCfgs[c].bk;
  const int a = kGemmCfgs[c].bm * 2 * bk, b = kGemmCfgs[c].bn * (q8 ? bk : 2 * bk);
  return a % (1024 * nw) == 0 && b % (1024 * nw) == 0 && a >= 1024 * nw && b >= 1024 * nw && !(q8 && bk == 128);
}
// ... and for a shape: 128-deep tiles have no K tail, so they need K % 128 == 0.
constexpr bool gemm_cfg_fits(int c, bool q8, int K) {
  return gemm_cfg_ok(c, q8) && (kGemmCfgs[c].bk < 128 || K % 128 == 0) &&
         (kGemmCfgs[c].kg == 1 || (K % kGemmCfgs[c].bk == 0 && (K / kGemmCfgs[c].bk) % kGemmCfgs[c].kg == 0));
}
// The grouped (MoE expert) GEMM's tile: 128 x 128, four 64-deep stages (128 KB of LDS, one block
// per CU). 128 rows hold a whole expert's share of a 256-token prefill (top-8 of 32 experts: about
// 64 rows each), so each expert's weights are streamed once; a 64-row tile split most experts into
// two row tiles, each streaming the same weights.
constexpr int kGrpBM = 128, kGrpBN = 128, kGrpWM = 2, kGrpWN = 2, kGrpStages = 4, kGrpBK = 64;
// The big tiles for experts of more than 128 rows: 256 x 128 or 128 x 256 (8 waves, three stages of 48 KB).
constexpr int kGrpTallBM = 256, kGrpTallWM = 4, kGrpTallStages = 3;
// Ring stages of a config's A and W tiles. The 64-deep 256 x 256 and 256 x 192 tiles hold one more
// stage for W than for A (in fp16, 256 x 256 fills the CU's 160 KB with it): with two stages of
// both, each tile's DMA has less than one tile of MFMA work to land and must go out in one burst;
// with a third W stage it is spread over the tile, A first, and W (weights, from HBM) is requested
// two tiles ahead. int8 W rows are half as wide and leave room for one stage more of each.
constexpr bool gemm_odd_ring(int c) { return kGemmCfgs[c].bm == 256 && kGemmCfgs[c].bn >= 192 && kGemmCfgs[c].bk == 64; }
constexpr int gemm_sa(int c, bool q8) { return gemm_odd_ring(c) && q8 ? 3 : kGemmCfgs[c].st; }
constexpr int gemm_sb(int c, bool q8) { return gemm_odd_ring(c) ? gemm_sa(c, q8) + 1 : kGemmCfgs[c].st; }
// LDS of the staged epilogue: the fp16 tile with 16-byte row padding, then one C row index per row
constexpr size_t gemm_stage_bytes(int bm, int bn) { return (size_t)bm * (bn + 8) * 2 + (size_t)bm * 4; }
inline size_t gemm_lds_bytes(int cfg, bool q8) {
  const GemmCfg& c = kGemmCfgs[cfg];
  const size_t ring = (size_t)c.kg * (gemm_sa(cfg, q8) * c.bm * c.bk * 2 + gemm_sb(cfg, q8) * c.bn * (q8 ? c.bk : 2 * c.bk));
  const bool staged = c.kg == 1 && c.wn == 1;  // the kernel's kStaged (grouped tiles size their own)
  return staged && gemm_stage_bytes(c.bm, c.bn) > ring ? gemm_stage_bytes(c.bm, c.bn) : ring;
}

// Split-K second pass of a residual GEMM fused with the RMSNorm that reads its result: one block
// of kNormThreads per row sums the row's partials in split order and adds the residual exactly as
// gemm_splitk_reduce<1> does, writes the row back, and normalises it as rmsnorm_kernel does (the
// same chunk ownership, summation order and norm_finish), so both outputs are bit-identical to
// the two kernels run in turn. With the split count ZS fixed at compile time (2..8) a thread issues
// all its loads of a chunk's partials before it adds them: with one row per block the pass is
// otherwise one memory round trip per split (ZS = 0: any count, one split at a time). RC chunks
// per thread: 1 for rows of up to 4096 halves (rmsnorm_kernel's second chunk then only adds exact
// zeros), else kNormChunks. Rows of N <= 8192 halves (N % 8 == 0), C and y contiguous.
template <int RC, int ZS>
__global__ void __launch_bounds__(kNormThreads) gemm_splitk_reduce_rmsnorm(const float* __restrict__ ws, int splits,
                                                                           int M, int N, f16* C,
                                                                           const f16* __restrict__ w,
                                                                           f16* __restrict__ y, float eps) {
  static_assert(RC >= 1 && RC <= kNormChunks, "chunks per thread");
  __shared__ float red[kNormThreads / 64];
  const int tid = threadIdx.x, n8 = N / 8, row = blockIdx.x;
  const int64_t plane = (int64_t)M * N;
  f16* xr = C + (int64_t)row * N;
  const float* pr = ws + (int64_t)row * N;
  u32x4 hv[RC], wv[RC];
#pragma unroll
  for (int j = 0; j < RC; j++) {
    const int c = tid + j * kNormThreads;
    hv[j] = wv[j] = u32x4{0u, 0u, 0u, 0u};
    if (c < n8) {
      wv[j] = *reinterpret_cast<const u32x4*>(w + 8 * c);
      const f16x8 r = *reinterpret_cast<const f16x8*>(xr + 8 * c);
      f32x4 t0 = {0.f, 0.f, 0.f, 0.f}, t1 = t0;
      if constexpr (ZS > 0) {
        f32x4 a[ZS], b[ZS];
#pragma unroll
        for (int z = 0; z < ZS; z++) {
          a[z] = *reinterpret_cast<const f32x4*>(pr + z * plane + 8 * c);
          b[z] = *reinterpret_cast<const f32x4*>(pr + z * plane + 8 * c + 4);
        }
#pragma unroll
        for (int z = 0; z < ZS; z++) {
          t0 += a[z];
          t1 += b[z];
        }
      } else {
        for (int z = 0; z < splits; z++) {
          t0 += *reinterpret_cast<const f32x4*>(pr + z * plane + 8 * c);
          t1 += *reinterpret_cast<const f32x4*>(pr + z * plane + 8 * c + 4);
        }
      }
      f16x8 h;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        h[e] = r[e] + (f16)t0[e];
        h[4 + e] = r[4 + e] + (f16)t1[e];
      }
      hv[j] = __builtin_bit_cast(u32x4, h);
      *reinterpret_cast<u32x4*>(xr + 8 * c) = hv[j];
    }
  }
  float ss = 0.f;
#pragma unroll
  for (int j = 0; j < RC; j++)
#pragma unroll
    for (int p = 0; p < 4; p++) {
      const f16x2 h = as_h2(hv[j][p]);
      ss = dot2(h, h, ss);
    }
  const float rs = norm_finish(ss, red, N, eps);
  f16* yr = y + (int64_t)row * N;
#pragma unroll
  for (int j = 0; j < RC; j++) {
    const int c = tid + j * kNormThreads;
    if (c >= n8) continue;
    u32x4 o;
#pragma unroll
    for (int p = 0; p < 4; p++) {
      const f16x2 xh = as_h2(hv[j][p]), wh = as_h2(wv[j][p]);
      f16x2 t;
      t.x = wh.x * (f16)((float)xh.x * rs);
      t.y = wh.y * (f16)((float)xh.y * rs);
      o[p] = as_u32(t);
    }
    *reinterpret_cast<u32x4*>(yr + 8 * c) = o;
  }
}

typedef void (*SplitkRmsnormFn)(const float*, int, int, int, f16*, const f16*, f16*, float);
template <int RC>
inline SplitkRmsnormFn splitk_rmsnorm_for(int splits) {
  switch (splits) {
    case 2: return gemm_splitk_reduce_rmsnorm<RC, 2>;
    case 3: return gemm_splitk_reduce_rmsnorm<RC, 3>;
    case 4: return gemm_splitk_reduce_rmsnorm<RC, 4>;
    case 5: return gemm_splitk_reduce_rmsnorm<RC, 5>;
    case 6: return gemm_splitk_reduce_rmsnorm<RC, 6>;
    case 8: return gemm_splitk_reduce_rmsnorm<RC, 8>;
    default: return gemm_splitk_reduce_rmsnorm<RC, 0>;
  }
}
inline SplitkRmsnormFn splitk_rmsnorm_kernel(bool one_chunk, int splits) {
  return one_chunk ? splitk_rmsnorm_for<1>(splits) : splitk_rmsnorm_for<kNormChunks>(splits);
}

template <int BM, int BN, int WM, int WN, int S, int EPI, bool Q8, int BK, int KG, int SB>
int gemm_launch(const GemmArgs& g, int cfg, int splits, hipStream_t s) {
  const size_t lds = gemm_lds_bytes(cfg, Q8);
  const void* fn = reinterpret_cast<const void*>(&gemm_kernel<BM, BN, WM, WN, S, EPI, Q8, false, BK, KG, SB>);
  const int bpc = hi_blocks_per_cu(fn, 64 * WM * WN * KG, lds);  // also lifts the dynamic-LDS limit
  if (bpc < 0) return -2;
  if (bpc == 0) HI_FAIL("gemm: tile %dx%d does not fit on a CU", BM, BN);
  const int tiles = ((g.M + BM - 1) / BM) * ((g.N + BN - 1) / BN);
  hipLaunchKernelGGL((gemm_kernel<BM, BN, WM, WN, S, EPI, Q8, false, BK, KG, SB>), dim3(tiles, splits),
                     dim3(64 * WM * WN * KG), lds, s, g);
  HI_TRY(hipGetLastError());
  if (splits > 1 && EPI == 1 && g.norm_y) {
    hipLaunchKernelGGL(splitk_rmsnorm_kernel(g.N <= 8 * kNormThreads, splits), dim3(g.M), dim3(kNormThreads), 0, s, g.ws,
                       splits, g.M, g.N, g.C, g.norm_w, g.norm_y, g.norm_eps);
    HI_TRY(hipGetLastError());
  } else if (splits > 1) {
    const int64_t quads = (int64_t)g.M * (EPI == 2 ? g.N / 2 : g.N) / 4;
    hipLaunchKernelGGL(gemm_splitk_reduce<EPI>, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, s, g.ws, splits,
                       g.M, g.N, g.bias, g.C, g.ldc, g.vec_c);
    HI_TRY(hipGetLastError());
  }
  return 0;
}

template <int EPI>
int gemm_run(const GemmArgs& g, int cfg, int splits, bool q8, hipStream_t s);
// Resident blocks per CU of a config's kernel (occupancy API). Kernels are only ever named in
// their own instance file: naming one elsewhere would instantiate (and register) a second copy.
template <int EPI>
int gemm_blocks_per_cu(int cfg, bool q8);

#define HI_GEMM_K(i, q)                                                                                        \
  gemm_kernel<kGemmCfgs[i].bm, kGemmCfgs[i].bn, kGemmCfgs[i].wm, kGemmCfgs[i].wn, gemm_sa(i, q), EPI, q, false,  \
              kGemmCfgs[i].bk, kGemmCfgs[i].kg, gemm_sb(i, q)>
#define HI_GEMM_CFG(i, q)                                                                                      \
  if constexpr (gemm_cfg_ok(i, q)) {                                                                           \
    if (cfg == i && q8 == q)                                                                                   \
      return gemm_launch<kGemmCfgs[i].bm, kGemmCfgs[i].bn, kGemmCfgs[i].wm, kGemmCfgs[i].wn, gemm_sa(i, q), EPI, \
                         q, kGemmCfgs[i].bk, kGemmCfgs[i].kg, gemm_sb(i, q)>(g, cfg, splits, s);                              \
  }
#define HI_GEMM_OCC(i)                                                                                         \
  if constexpr (gemm_cfg_ok(i, true))                                                                          \
    if (cfg == i && q8)                                                                                        \
      return hi_blocks_per_cu(reinterpret_cast<const void*>(&HI_GEMM_K(i, true)),                              \
                              64 * kGemmCfgs[i].wm * kGemmCfgs[i].wn * kGemmCfgs[i].kg, gemm_lds_bytes(i, true)); \
  if constexpr (gemm_cfg_ok(i, false))                                                                         \
    if (cfg == i && !q8)                                                                                       \
      return hi_blocks_per_cu(reinterpret_cast<const void*>(&HI_GEMM_K(i, false)),                             \
                              64 * kGemmCfgs[i].wm * kGemmCfgs[i].wn * kGemmCfgs[i].kg, gemm_lds_bytes(i, false));
#define HI_GEMM_DEFINE_RUN(EPIV)                                                                               \
  template <>                                                                                                  \
  int gemm_run<EPIV>(const GemmArgs& g, int cfg, int splits, bool q8, hipStream_t s) {                        \
    constexpr int EPI = EPIV;                                                                                  \
    HI_GEMM_CFG(0, false) HI_GEMM_CFG(1, false) HI_GEMM_CFG(2, false) HI_GEMM_CFG(3, false)                    \
    HI_GEMM_CFG(4, false) HI_GEMM_CFG(5, false) HI_GEMM_CFG(6, false) HI_GEMM_CFG(7, false)                    \
    HI_GEMM_CFG(8, false) HI_GEMM_CFG(9, false) HI_GEMM_CFG(10, false) HI_GEMM_CFG(11, false)                  \
    HI_GEMM_CFG(12, false) HI_GEMM_CFG(13, false) HI_GEMM_CFG(14, false) HI_GEMM_CFG(15, false)                \
    HI_GEMM_CFG(16, false) HI_GEMM_CFG(17, false) HI_GEMM_CFG(18, false) HI_GEMM_CFG(19, false)                \
    HI_GEMM_CFG(0, true) HI_GEMM_CFG(1, true) HI_GEMM_CFG(2, true) HI_GEMM_CFG(3, true)                        \
    HI_GEMM_CFG(4, true) HI_GEMM_CFG(5, true) HI_GEMM_CFG(6, true) HI_GEMM_CFG(7, true)                        \
    HI_GEMM_CFG(8, true) HI_GEMM_CFG(9, true) HI_GEMM_CFG(10, true) HI_GEMM_CFG(11, true) HI_GEMM_CFG(12, true) \
    HI_GEMM_CFG(13, true) HI_GEMM_CFG(14, true) HI_GEMM_CFG(15, true) HI_GEMM_CFG(16, true)                   \
    HI_GEMM_CFG(19, true)                                                                                      \
    HI_FAIL("gemm: no kernel for config %d", cfg);                                                             \
  }                                                                                                            \
  template <>                                                                                                  \
  int gemm_blocks_per_cu<EPIV>(int cfg, bool q8) {                                                             \
    constexpr int EPI = EPIV;                                                                                  \
    HI_GEMM_OCC(0) HI_GEMM_OCC(1) HI_GEMM_OCC(2) HI_GEMM_OCC(3) HI_GEMM_OCC(4) HI_GEMM_OCC(5) HI_GEMM_OCC(6)    \
    HI_GEMM_OCC(7) HI_GEMM_OCC(8) HI_GEMM_OCC(9) HI_GEMM_OCC(10) HI_GEMM_OCC(11) HI_GEMM_OCC(12)              \
    HI_GEMM_OCC(13) HI_GEMM_OCC(14) HI_GEMM_OCC(15) HI_GEMM_OCC(16) HI_GEMM_OCC(17) HI_GEMM_OCC(18)            \
    HI_GEMM_OCC(19)                                                                                            \
    return -1;                                                                                                 \
  }
