// The body of the GEMM kernels; gemm.h includes it in each of their functions. It uses their template parameters
// BM, BN, WM, WN, S, EPI, Q8, GRP, BK, KG, SB, the argument g and, where PRELOADED, the thread's GrpLoad `loaded`.
// One text and not one inlined function: as a function, the compiler ordered the same code differently in every
// instance, up to 10 % slower (256 x 192, M = 2048, N = 4096, K = 14336: 239 -> 264 us; 128 x 96, M = 777, N =
// 2560, K = 2048: 15.9 -> 17.2).
  constexpr int TM = BM / WM, TN = BN / WN;          // wave tile
  constexpr int FM = TM / 32, FN = TN / 32;          // MFMA tiles per wave
  constexpr int A_ST = BM * BK;                      // halves per stage
  constexpr int B_ROWB = Q8 ? BK : 2 * BK;           // bytes of one W row per K tile
  constexpr int RPI = 512 / BK;                      // fp16 rows per 1 KB DMA instruction
  constexpr int RPI8 = 1024 / BK;                    // int8 rows per 1 KB DMA instruction
  constexpr int B_ST = BN * B_ROWB / 2;              // halves per stage
  constexpr int NW = WM * WN;                        // waves per block (4 or 8)
  constexpr int A_LD = BM * 2 * BK / 1024 / NW;      // 1 KB DMA instructions per wave per K tile (A)
  constexpr int B_LD = BN * B_ROWB / 1024 / NW;      // ... (W)
  constexpr int L = A_LD + B_LD;                     // vector-memory ops per lane per K tile
  // A refill (one K tile of A and of W into the stages just freed) is issued in NP parts, one per
  // step of MFMAs after the barrier that freed them, so that no wave's DMA instructions queue up
  // behind one another in front of its MFMAs. A two-stage ring has no tile of slack and issues it in
  // the first step; one with a third W stage takes A first, in two steps, W then has a tile more to
  // land. Other rings take W first (cold weights come from HBM, the activations mostly from L2).
  constexpr int NP = SB == 2 ? 1 : BK == 32 || S == 2 || GRP ? 2 : 4;
  constexpr auto part_n = [](int p) constexpr {
    int n = 0;
    for (int i = 0; i < L; i++) n += i * NP / L == p;
    return n;
  };
  // the v-th instruction of part p, as an index for issue_one (A first)
  constexpr auto part_at = [](int p, int v) constexpr {
    int i = 0;
    while (i * NP / L != p) i++;
    i += v;
    return SB == S ? (i + A_LD) % L : i;
  };
  static_assert((NW == 4 || NW == 8) && FM >= 1 && FN >= 1 && TM % 32 == 0 && TN % 32 == 0, "wave tiling");
  static_assert(A_LD >= 1 && B_LD >= 1 && A_LD * 1024 * NW == BM * 2 * BK && B_LD * 1024 * NW == BN * B_ROWB &&
                    S >= 2 && S <= 8 && (SB == S || SB == S + 1) && (S - 1) * L + B_LD < 64 && 3 * L < 64,
                "pipeline shape: every wave issues the same whole number of 1 KB DMA instructions");
  static_assert(!(GRP && Q8), "grouped (expert) GEMMs take fp16 weights");
  static_assert(BK == 128 || BK == 64 || BK == 32, "K tile depth");
  static_assert(BK != 128 || (!Q8 && !GRP), "128-deep K tiles take fp16 weights (and K % 128 == 0)");
  static_assert(KG == 1 || (KG == 2 && !GRP), "one or two K groups (not in grouped mode)");
  // The dynamic LDS follows the static (the split-K flag below); a 16-byte element type makes the
  // compiler start it on a 16-byte boundary, which every 128-bit LDS access and DMA here needs.
  extern __shared__ u32x4 smem_raw[];
  // KG K groups of WM x WN waves each run the whole pipeline below on their share of the K tiles,
  // each with its own S-stage ring; group 0 adds the other groups' sums at the end
  const int tid = threadIdx.x, lane = tid & 63;
  const int kg = KG > 1 ? (tid >> 6) / NW : 0;  // this wave's K group
  const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) - kg * NW);  // its index within the group
  f16* smem = reinterpret_cast<f16*>(smem_raw) + kg * (S * A_ST + SB * B_ST);
  f16* As = smem;               // [S][BM][64]
  f16* Bs = smem + S * A_ST;    // [SB][BN][64] fp16, or [SB][BN][64 bytes] int8

  const int wm = wave / WN, wn = wave % WN;
  const int N = g.N, K = g.K;
  int M = g.M;
  const f16* Ap = g.A;
  f16* Cp = g.C;
  const char* Wb = reinterpret_cast<const char*>(g.W);
  const int tiles_n = (N + BN - 1) / BN;
  int tm, tn, ntiles;
  [[maybe_unused]] int grp_r0 = 0;  // grouped mode: the group's first sorted row
  if constexpr (GRP) {
    // find this block's group: grp_tiles[e] <= row tile < grp_tiles[e + 1] (the prefix is
    // non-decreasing, so e is the number of groups whose tiles start at or before the row tile,
    // minus one); blocks past the last row tile (the grid is sized for the worst case) exit. The threads
    // load the groups at once (grp_load): one memory round trip, then one counting barrier.
    static_assert(64 * NW * KG >= kGemmMaxGroups, "one thread per group");
    __shared__ int s_tiles[kGemmMaxGroups + 1], s_off[kGemmMaxGroups + 1];
    const int E = g.grp_n, mt = blockIdx.x / tiles_n;
    tn = blockIdx.x - mt * tiles_n;
    const GrpLoad gl = PRELOADED ? loaded : grp_load(g);
    if (tid < E) {
      s_tiles[tid] = gl.tile;
      s_off[tid] = gl.off;
    }
    if (tid == 0) {
      s_tiles[E] = gl.tiles_all;
      s_off[E] = gl.off_all;
    }
    const int lo = __syncthreads_count(tid < E && gl.tile <= mt) - 1;
    if (mt >= s_tiles[E]) return;
    grp_r0 = s_off[lo];
    M = s_off[lo + 1] - grp_r0;
    if (!g.grp_gather) Ap += grp_r0 * g.lda;
    if (!g.grp_scatter) Cp += grp_r0 * g.ldc;
    Wb += lo * g.grp_wstride;
    tm = mt - s_tiles[lo];
    ntiles = 0;
  } else {
    const int tiles_m = (M + BM - 1) / BM;
    ntiles = tiles_m * tiles_n;
    // tile index: blocks are dealt round-robin over the 8 XCDs; give each XCD a contiguous run of
    // tile ids (the part of the grid that divides by 8; the remainder keeps its id)
    int pid = blockIdx.x;
    const int per = ntiles / 8;
    if (pid < per * 8) pid = (pid % 8) * per + pid / 8;
    constexpr int GM = 8;
    const int per_group = GM * tiles_n, first = (pid / per_group) * GM;
    const int gsize = min(tiles_m - first, GM), r = pid % per_group;
    tm = first + r % gsize;
    tn = r / gsize;
  }
  const int bm = tm * BM, bn = tn * BN;

  const int nkt = (K + BK - 1) / BK;
  // K tiles of this split (>= 1), cut into KG equal runs, one per K group (the host offers KG > 1
  // only when K % BK == 0 and the runs come out equal, so every group loops alike)
  const int nloc = (min(nkt, (int)blockIdx.y * g.kt_per_split + g.kt_per_split) - (int)blockIdx.y * g.kt_per_split) / KG;
  const int kt0 = blockIdx.y * g.kt_per_split + kg * nloc;
  // the last tile holds only 32 k (K % 64 == 32 with 64-deep tiles; K % 32 == 0 always)
  const bool half_tail = BK == 64 && (K & 63) != 0 && kt0 + nloc == nkt;

  // ---- DMA of one K tile into stage st, through buffer resources based at the block's first A
  //      and W rows. Lane l of an instruction covering 8 (A, W fp16) or 16 (W int8) rows fills LDS
  //      slot l: it fetches the chunk the swizzle puts there. Offsets are bounds-checked against
  //      the rows that exist: rows past M or N read zeros (never stored). Chunks past K (the second
  //      half of a half tile) read bytes of the next row or zeros, and are never used.
  const int valid_m = min(M - bm, BM), valid_n = min(N - bn, BN);
  const bool gather = GRP && g.grp_gather;  // A rows through grp_perm: the resource spans all of A
  const int a_bytes = gather ? (int)(((int64_t)(g.grp_a_rows - 1) * g.lda + K) * 2)
                             : (int)(((int64_t)(valid_m - 1) * g.lda + K) * 2);
  const __amdgpu_buffer_rsrc_t a_rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<f16*>(gather ? Ap : Ap + (int64_t)bm * g.lda), (short)0, a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t b_rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char*>(Wb + (int64_t)bn * K * (Q8 ? 1 : 2)), (short)0, (int)((int64_t)valid_n * K * (Q8 ? 1 : 2)),
      0x00020000);
  // this lane's byte offset within an instruction's rows; the swizzle term of a 256-byte row r is
  // (r & 15), which over an instruction's 4 rows depends on the instruction's index mod 4 and
  // lane / 16; of a 128-byte row ((r >> 1) & 7), which over an instruction's 8 rows depends on the
  // instruction's parity and lane / 16; of a 64-byte row ((r >> 2) & 3) and of a 32-byte int8 row
  // ((r >> 3) & 1), which depend on the lane only
  const int a_r = lane / (BK / 8), a_p = lane % (BK / 8);
  int a_lo[4], b_lo[4];  // per instruction index mod 4 (mod 2 for 128-byte rows; unused entries)
#pragma unroll
  for (int par = 0; par < 4; par++) {
    const int sw = BK == 128 ? (par * 4 + a_r) & 15 : BK == 64 ? (par * 4 + (a_r >> 1)) & 7 : (a_r >> 2) & 3;
    a_lo[par] = (int)((int64_t)a_r * g.lda * 2) + ((a_p ^ sw) << 4);
    if constexpr (Q8) {
      b_lo[par] = BK == 64 ? (lane >> 2) * K + (((lane & 3) ^ ((lane >> 4) & 3)) << 4)
                           : (lane >> 1) * K + (((lane & 1) ^ ((lane >> 4) & 1)) << 4);
    } else {
      b_lo[par] = a_r * K * 2 + ((a_p ^ sw) << 4);
    }
  }
  // grouped gather: this lane's row of each A instruction is sorted row grp_r0 + bm + ri + a_r,
  // fetched from A row grp_perm[that] / grp_k; rows past the group's count get an offset past the
  // resource, so they read zeros
  int a_go[A_LD];  // set and read in grouped mode only
  if constexpr (GRP) {
#pragma unroll
    for (int i = 0; i < A_LD; i++) {
      const int ri = (wave * A_LD + i) * RPI, r = bm + ri + a_r;
      const int lo_i = a_lo[(ri / RPI) % (BK == 128 ? 4 : 2)] - (int)((int64_t)a_r * g.lda * 2);  // the chunk term
      if (gather)
        a_go[i] = r < M ? (int)((int64_t)(g.grp_perm[grp_r0 + r] / g.grp_k) * g.lda * 2) + lo_i : a_bytes;
      else
        a_go[i] = a_lo[(ri / RPI) % (BK == 128 ? 4 : 2)] + (int)((int64_t)ri * g.lda * 2);
    }
  }
  // one DMA instruction of K tile kt_a / kt_b: A instruction i < A_LD into A stage sa, W
  // instruction i - A_LD into W stage sb
  auto issue_one = [&](int i, int kt_a, int sa, int kt_b, int sb) {
    if (i < A_LD) {
      const int k0 = kt_a * BK;
      f16* as = As + sa * A_ST;
      const int ri = (wave * A_LD + i) * RPI;
      // (a plain conditional: an `if constexpr` here kept clang from emitting the grouped kernels)
      const int off = GRP ? a_go[i < A_LD ? i : 0] : a_lo[(ri / RPI) % (BK == 128 ? 4 : 2)] + (int)((int64_t)ri * g.lda * 2);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_rs, (lds_void_t*)(as + ri * BK), 16, off + k0 * 2, 0, 0, 0);
    } else {
      const int k0 = kt_b * BK, j = i - A_LD;
      char* bs = reinterpret_cast<char*>(Bs + sb * B_ST);
      if constexpr (Q8) {
        const int ri = (wave * B_LD + j) * RPI8;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rs, (lds_void_t*)(bs + ri * BK), 16, b_lo[0] + ri * K + k0, 0, 0, 0);
      } else {
        const int ri = (wave * B_LD + j) * RPI;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rs, (lds_void_t*)(bs + ri * 2 * BK), 16,
                                                 b_lo[(ri / RPI) % (BK == 128 ? 4 : 2)] + ri * K * 2 + k0 * 2, 0, 0, 0);
      }
    }
  };
  const int fr = lane & 31, fk = lane >> 5;  // fragment row (or column) and k half
  // grouped scatter: the C row of each of this lane's fragment rows, requested now so that the
  // epilogue waits for nothing
  int c_row[FM];
#pragma unroll
  for (int i = 0; i < FM; i++) {
    const int row = bm + wm * TM + i * 32 + fr;
    c_row[i] = (GRP && g.grp_scatter && row < M) ? g.grp_perm[grp_r0 + row] : row;
  }
  f16x2 bsc[FN];                             // int8: the scale of the W row each B fragment reads
#pragma unroll
  for (int j = 0; j < FN; j++) {
    bsc[j] = f16x2{(f16)0.f, (f16)0.f};
    if constexpr (Q8) {
      const f16 sv = g.scales[min(bn + wn * TN + j * 32 + fr, N - 1)];
      bsc[j] = f16x2{sv, sv};
    }
  }
  // LDS offsets of this lane's fragment rows (halves for A / fp16 W, bytes for int8 W), per chunk
  // parity: the swizzle term of row r is ((r >> 1) & 7) (or (r >> 2) & 3), fixed per lane
  int a_row[FM], b_row[FN];
#pragma unroll
  for (int i = 0; i < FM; i++) a_row[i] = (wm * TM + i * 32 + fr);
#pragma unroll
  for (int j = 0; j < FN; j++) b_row[j] = (wn * TN + j * 32 + fr);

  // The memory instructions of one step, in the order sched_step expects: the fragments of step
  // s = 2 jh + h of the tile in stages sa (A) and sb (W), W's first (the first MFMAs need one A
  // fragment and all of W's), then NV DMA instructions, dma(v) the v-th. fp16 W: one fragment per
  // step; int8 W: both steps of half jh come as one raw 16-byte chunk, read where WQ is set.
  auto step_mem = [&](auto wq, auto nv, int sa, int sb, int s, f16x8 (&af)[FM], f16x8 (&bf)[FN], u32x4 (&bq)[FN],
                      auto dma) {
    const int c = 4 * (s >> 1) + 2 * fk + (s & 1), cq = 2 * (s >> 1) + fk;
    const f16* as = As + sa * A_ST;
    const f16* bs = Bs + sb * B_ST;
    if constexpr (!Q8 || decltype(wq)::value) {
#pragma unroll
      for (int j = 0; j < FN; j++) {
        if constexpr (Q8)
          bq[j] = *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(bs) + lds_off8<BK>(b_row[j], cq));
        else
          bf[j] = *reinterpret_cast<const f16x8*>(bs + lds_off<BK>(b_row[j], c));
      }
    }
#pragma unroll
    for (int i = 0; i < FM; i++) af[i] = *reinterpret_cast<const f16x8*>(as + lds_off<BK>(a_row[i], c));
#pragma unroll
    for (int v = 0; v < decltype(nv)::value; v++) dma(v);
  };

  f32x16 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[i][j][e] = 0.f;

  // the MFMAs of one step; int8 fragments are dequantised from half h of the raw chunk
  auto mfmas = [&](int h, const f16x8 (&af)[FM], const f16x8 (&bf)[FN], const u32x4 (&bq)[FN]) {
    f16x8 b[FN];
#pragma unroll
    for (int j = 0; j < FN; j++) {
      if constexpr (Q8) {
        f16x2 p0, p1, p2, p3;
        i8x4_to_f16(bq[j][2 * h], p0, p1);
        i8x4_to_f16(bq[j][2 * h + 1], p2, p3);
        p0 = p0 * bsc[j];  // fp16(q * s), one rounding each
        p1 = p1 * bsc[j];
        p2 = p2 * bsc[j];
        p3 = p3 * bsc[j];
        b[j] = f16x8{p0.x, p0.y, p1.x, p1.y, p2.x, p2.y, p3.x, p3.y};
      } else {
        b[j] = bf[j];
      }
    }
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
      for (int j = 0; j < FN; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(b[j], af[i], acc[i][j], 0, 0, 0);
  };

  // ---- prologue: the whole ring in flight (past the split's last tile, its first tile again: a
  //      stage is filled every time, so the outstanding-DMA count is the same in every iteration);
  //      the first fragments of tile 0 in registers
  auto tile_or_first = [&](int kt) { return kt < kt0 + nloc ? kt : kt0; };
#pragma unroll
  for (int s = 0; s < SB; s++) {
#pragma unroll
    for (int i = 0; i < L; i++)
      if (i >= A_LD || s < S) issue_one(i, tile_or_first(kt0 + s), s, tile_or_first(kt0 + s), s);
  }
  int ra = kt0, rb = kt0, rsa = 0, rsb = 0;  // the refill under way: K tiles ra / rb into stages rsa / rsb
  wait_vmcnt<(S - 1) * A_LD + (SB - 1) * B_LD>();
  barrier_no_fence();
  int sa = 0, sb = 0;  // the current tile's stages
  f16x8 af0[FM], af1[FM], bf0[FN], bf1[FN];
  u32x4 bq0[FN], bq1[FN];  // int8: raw chunks of the tile's first and second 32-deep half
  constexpr std::true_type kWQ{};   // int8: the step that reads a half's raw chunks ...
  constexpr std::false_type kNoQ{};  // ... and the one that does not
  constexpr std::integral_constant<int, 0> kNoDma{};
  auto no_dma = [](int) {};
  step_mem(kWQ, kNoDma, 0, 0, 0, af0, bf0, bq0, no_dma);

  constexpr int NM = FM * FN;               // MFMAs per step
  constexpr int ND = FM + (Q8 ? 0 : FN);    // LDS reads per step (int8 W: + FN every other step)
  // part p of the refill under way
  auto dma_part = [&](int p) {
    return [&, p](int v) { issue_one(part_at(p, v), ra, rsa, rb, rsb); };
  };
  // the tile's last fragments are in registers: the next tile has landed for every wave, and the
  // current tile's stages are free for the next refill (its part 0 goes out in the step that
  // follows, the other parts in the next tile's first steps)
  auto next_tile = [&](int t) {
    wait_lgkm0();
    wait_vmcnt<(S - 2) * L + (SB > S ? B_LD : 0)>();
    barrier_no_fence();
    ra = tile_or_first(kt0 + t + S);
    rb = tile_or_first(kt0 + t + SB);
    rsa = sa;
    rsb = sb;
    sa = sa + 1 == S ? 0 : sa + 1;
    sb = sb + 1 == SB ? 0 : sb + 1;
  };
  // Each depth's `tile` is one tile but the last: its steps with the parts of the refill under way
  // (none in tile 0, whose ring the prologue has filled), and the handover to the next tile.
  constexpr std::integral_constant<int, part_n(0)> kP0{};
  if constexpr (BK == 128) {
    // ---- 128-deep fp16 tiles (K % 128 == 0): 8 steps each, fragments one step ahead, the same
    //      k order as two consecutive 64-deep tiles (so the same sums, bit for bit)
    auto tile = [&](int t, auto refill) {
      constexpr bool R = decltype(refill)::value && NP > 1;
      auto pair = [&](auto part, int s) {
        constexpr int P = decltype(part)::value;
        constexpr std::integral_constant<int, (R ? part_n(P) : 0)> nv{};
        step_mem(kWQ, nv, sa, sb, s, af1, bf1, bq0, dma_part(P));
        mfmas(0, af0, bf0, bq0);
        sched_step<NM, ND, (R ? part_n(P) : 0)>();
        step_mem(kWQ, kNoDma, sa, sb, s + 1, af0, bf0, bq0, no_dma);
        mfmas(0, af1, bf1, bq0);
        sched_step<NM, ND>();
      };
      pair(std::integral_constant<int, 1>{}, 1);
      pair(std::integral_constant<int, 2>{}, 3);
      pair(std::integral_constant<int, 3>{}, 5);
      step_mem(kWQ, kNoDma, sa, sb, 7, af1, bf1, bq0, no_dma);
      mfmas(0, af0, bf0, bq0);
      sched_step<NM, ND>();
      next_tile(t);
      step_mem(kWQ, kP0, sa, sb, 0, af0, bf0, bq0, dma_part(0));
      mfmas(0, af1, bf1, bq0);
      sched_step<NM, ND, part_n(0)>();
    };
    if (nloc > 1) tile(0, std::false_type{});
    for (int t = 1; t < nloc - 1; t++) tile(t, std::true_type{});
#pragma unroll
    for (int p = 0; p < 4; p++) {
      step_mem(kWQ, kNoDma, sa, sb, 2 * p + 1, af1, bf1, bq0, no_dma);
      mfmas(0, af0, bf0, bq0);
      if (p < 3) step_mem(kWQ, kNoDma, sa, sb, 2 * p + 2, af0, bf0, bq0, no_dma);
      mfmas(0, af1, bf1, bq0);
    }
  } else if constexpr (BK == 64) {
    // ---- 64-deep tiles: 4 steps each, fragments one step ahead
    auto tile = [&](int t, auto refill) {
      constexpr bool R = decltype(refill)::value && NP > 1;
      constexpr std::integral_constant<int, (R ? part_n(1) : 0)> p1{};
      constexpr std::integral_constant<int, (R ? part_n(2) : 0)> p2{};
      constexpr std::integral_constant<int, (R ? part_n(3) : 0)> p3{};
      step_mem(kNoQ, p1, sa, sb, 1, af1, bf1, bq0, dma_part(1));
      mfmas(0, af0, bf0, bq0);
      sched_step<NM, ND, (R ? part_n(1) : 0)>();
      step_mem(kWQ, p2, sa, sb, 2, af0, bf0, bq1, dma_part(2));
      mfmas(1, af1, bf1, bq0);
      sched_step<NM, ND + (Q8 ? FN : 0), (R ? part_n(2) : 0)>();
      step_mem(kNoQ, p3, sa, sb, 3, af1, bf1, bq1, dma_part(3));
      mfmas(0, af0, bf0, bq1);
      sched_step<NM, ND, (R ? part_n(3) : 0)>();
      next_tile(t);
      step_mem(kWQ, kP0, sa, sb, 0, af0, bf0, bq0, dma_part(0));
      mfmas(1, af1, bf1, bq1);
      sched_step<NM, ND + (Q8 ? FN : 0), part_n(0)>();
    };
    if (nloc > 1) tile(0, std::false_type{});
    for (int t = 1; t < nloc - 1; t++) tile(t, std::true_type{});
    // ---- the last tile (its first half only when K % 64 == 32)
    {
      step_mem(kNoQ, kNoDma, sa, sb, 1, af1, bf1, bq0, no_dma);
      mfmas(0, af0, bf0, bq0);
      mfmas(1, af1, bf1, bq0);
      if (!half_tail) {
        step_mem(kWQ, kNoDma, sa, sb, 2, af0, bf0, bq1, no_dma);
        step_mem(kNoQ, kNoDma, sa, sb, 3, af1, bf1, bq1, no_dma);
        mfmas(0, af0, bf0, bq1);
        mfmas(1, af1, bf1, bq1);
      }
    }
  } else {
    // ---- 32-deep tiles: 2 steps each, fragments one step ahead; int8 W holds both steps of a
    //      tile in one raw 16-byte chunk per fragment (bq0), the next tile's read into bqn first
    auto tile = [&](int t, auto refill) {
      constexpr bool R = decltype(refill)::value && NP > 1;
      constexpr std::integral_constant<int, (R ? part_n(1) : 0)> p1{};
      step_mem(kNoQ, p1, sa, sb, 1, af1, bf1, bq0, dma_part(1));
      mfmas(0, af0, bf0, bq0);
      sched_step<NM, ND, (R ? part_n(1) : 0)>();
      next_tile(t);
      [[maybe_unused]] u32x4 bqn[FN];
      step_mem(kWQ, kP0, sa, sb, 0, af0, bf0, bqn, dma_part(0));
      mfmas(1, af1, bf1, bq0);
      sched_step<NM, ND + (Q8 ? FN : 0), part_n(0)>();
      if constexpr (Q8) {
#pragma unroll
        for (int j = 0; j < FN; j++) bq0[j] = bqn[j];
      }
    };
    if (nloc > 1) tile(0, std::false_type{});
    for (int t = 1; t < nloc - 1; t++) tile(t, std::true_type{});
    step_mem(kNoQ, kNoDma, sa, sb, 1, af1, bf1, bq0, no_dma);
    mfmas(0, af0, bf0, bq0);
    mfmas(1, af1, bf1, bq0);
  }
  wait_vmcnt<0>();  // the refills issued past the last tile have landed before the block ends
  if constexpr (KG > 1) {
    // the other group's sums to group 0 through the idle rings (element e of a wave's fragment
    // set as one 256-byte row over its lanes), added in group order: deterministic
    constexpr int NE = FM * FN * 16;
    float* xf = reinterpret_cast<float*>(smem_raw);
    barrier_no_fence();  // every wave's last fragment reads are done with the rings
    if (kg == 1) {
#pragma unroll
      for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++)
#pragma unroll
          for (int e = 0; e < 16; e++) xf[((wave * NE) + (i * FN + j) * 16 + e) * 64 + lane] = acc[i][j][e];
    }
    __syncthreads();
    if (kg == 1) return;
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
      for (int j = 0; j < FN; j++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[i][j][e] += xf[((wave * NE) + (i * FN + j) * 16 + e) * 64 + lane];
  }

  // ---- result layout (W fragment as the MFMA's first operand): lane (fk, fr) of tile (i, j) holds
  //      row fr of the tile's 32 rows, columns 8 g + 4 fk + 0..3 in acc[i][j][4 g .. 4 g + 3]:
  //      four consecutive output columns per register quad

  // ---- staged epilogue (grouped tiles and the one-wave-wide 128 x 96 / 128 x 160 tiles; one K
  //      group, no split, C 16-byte addressable): the finished fp16 tile goes through LDS and leaves
  //      in 16-byte chunks, whole row segments per store instruction. Stored straight from the
  //      fragments, each store instruction writes 16 bytes into each of 32 rows (about 150 ns per
  //      instruction measured on the grouped down GEMM, 16 per lane there, 12-20 on the wide-wave
  //      tiles); staged, four to six rows of contiguous chunks. Other tiles keep the direct path:
  //      there the staged code cost registers (4-12 VGPRs, more spills on 256 x 256) for no gain.
  //      The roundings are the direct path's: the bias is added in fp32 before the fp16 rounding,
  //      SwiGLU is formed from the fp32 sums, and the residual is added (fp16 add) to the rounded
  //      product in the copy.
  constexpr bool kStaged = KG == 1 && (GRP || WN == 1);
  if (kStaged && gridDim.y == 1 && g.vec16_c) {
    constexpr int BNO = EPI == 2 ? BN / 2 : BN;  // output columns of the tile
    // LDS row stride in halves: 16 bytes of padding put the 32 rows one fragment write covers on
    // every bank once per 16 rows (BNO % 16 == 0)
    constexpr int CS = BNO + 8;
    static_assert(BNO % 16 == 0, "staged tile row padding");
    f16* cs = reinterpret_cast<f16*>(smem_raw);
    int* s_row = reinterpret_cast<int*>(cs + BM * CS);  // C row of each tile row
    barrier_no_fence();  // every wave is done with the rings (their DMA landed above)
#pragma unroll
    for (int i = 0; i < FM; i++) {
      const int lr = wm * TM + i * 32 + fr;
      if (wn == 0 && fk == 0) s_row[lr] = c_row[i];
#pragma unroll
      for (int j = 0; j < FN; j++) {
        const int lc0 = wn * TN + j * 32;  // the 32-column MFMA tile's first column in the tile
        if constexpr (EPI == 2) {
#pragma unroll
          for (int q = 0; q < 2; q++) {
            f16x4 o;
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = silu_mul_fast(acc[i][j][4 * q + e], acc[i][j][4 * q + 8 + e]);
            *reinterpret_cast<f16x4*>(cs + lr * CS + (lc0 >> 1) + 8 * q + 4 * fk) = o;
          }
        } else {
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const int lc = lc0 + 8 * q + 4 * fk;
            f16x4 o;
            if constexpr (EPI == 1) {
#pragma unroll
              for (int e = 0; e < 4; e++) o[e] = (f16)acc[i][j][4 * q + e];
            } else {
              f16x4 b = {(f16)0.f, (f16)0.f, (f16)0.f, (f16)0.f};
              if (g.bias && bn + lc < N) b = load4(g.bias + bn + lc, ((uintptr_t)g.bias & 7) == 0);
#pragma unroll
              for (int e = 0; e < 4; e++) o[e] = (f16)(acc[i][j][4 * q + e] + (float)b[e]);
            }
            *reinterpret_cast<f16x4*>(cs + lr * CS + lc) = o;
          }
        }
      }
    }
    __syncthreads();
    constexpr int CPR = BNO / 8;  // 16-byte chunks per tile row
    const int bno = EPI == 2 ? bn / 2 : bn, ncol = min((EPI == 2 ? N / 2 : N) - bno, BNO);
    for (int c = tid; c < BM * CPR; c += 64 * NW) {
      const int r = c / CPR, cc = c - r * CPR;
      if (r >= valid_m || cc * 8 >= ncol) continue;  // N % 16 == 0: a chunk is all in or all out
      f16x8 v = *reinterpret_cast<const f16x8*>(cs + r * CS + cc * 8);
      f16* dst = Cp + (int64_t)s_row[r] * g.ldc + bno + cc * 8;
      if constexpr (EPI == 1) {
        const f16x8 rv = *reinterpret_cast<const f16x8*>(dst);
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = rv[e] + v[e];  // fp16 add, correctly rounded
      }
      *reinterpret_cast<f16x8*>(dst) = v;
    }
    return;
  }
  if (gridDim.y > 1) {
    // split-K: this split's fp32 partial [split][M][N]; a second kernel (gemm_splitk_reduce) sums
    // the splits in order and runs the epilogue, after the kernel boundary made them visible
    float* part = g.ws + (int64_t)blockIdx.y * M * N;
#pragma unroll
    for (int i = 0; i < FM; i++) {
      const int row = bm + wm * TM + i * 32 + fr;
      if (row >= M) continue;
#pragma unroll
      for (int j = 0; j < FN; j++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int col = bn + wn * TN + j * 32 + 8 * q + 4 * fk;
          if (col < N)
            *reinterpret_cast<f32x4*>(part + (int64_t)row * N + col) =
                f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < FM; i++) {
    const int row = bm + wm * TM + i * 32 + fr;
    if (row >= M) continue;
    f16* crow = Cp + (int64_t)c_row[i] * g.ldc;
#pragma unroll
    for (int j = 0; j < FN; j++) {
      const int c0 = bn + wn * TN + j * 32;  // first column of the 32-column MFMA tile
      if (c0 >= N) continue;
      if constexpr (EPI == 2) {
        // gate columns c0 + 0..15 and their up columns c0 + 16..31 sit in the same lane
#pragma unroll
        for (int q = 0; q < 2; q++) {
          f16x4 o;
#pragma unroll
          for (int e = 0; e < 4; e++) o[e] = silu_mul_fast(acc[i][j][4 * q + e], acc[i][j][4 * q + 8 + e]);
          store4(crow + (c0 >> 1) + 8 * q + 4 * fk, o, g.vec_c);
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int col = c0 + 8 * q + 4 * fk;
          if (col >= N) continue;  // N % 16 == 0: the last 32-column tile can end 16 columns past N
          f16x4 o;
          if constexpr (EPI == 1) {
            const f16x4 r = load4(crow + col, g.vec_c);
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = r[e] + (f16)acc[i][j][4 * q + e];  // fp16 add, rounded
          } else {
            f16x4 b = {(f16)0.f, (f16)0.f, (f16)0.f, (f16)0.f};
            if (g.bias) b = load4(g.bias + col, ((uintptr_t)g.bias & 7) == 0);
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = (f16)(acc[i][j][4 * q + e] + (float)b[e]);
          }
          store4(crow + col, o, g.vec_c);
        }
      }
    }
  }
