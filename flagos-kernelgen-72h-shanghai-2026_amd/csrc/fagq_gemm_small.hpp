// fagq_gemm_small.hpp - the fp8 block-scaled GEMM's kernels for products whose
// 256-row tiles would leave most of the chip idle: decode steps and chunks.
// Included by fagq_gemm.hip inside its namespace, after the operand helpers.
//
// Two kernels, chosen with their tile by pick_small (fagq_gemm.hip):
//   fagq_gemm_waves_kernel - the waves of a workgroup split K.  Each wave holds
//     the whole tile's accumulators and stages its own k-blocks through its own
//     LDS, so the loop has no barrier; the partial tiles are added at the end.
//     What it moves per k-block is the tile's rows and columns once, the least
//     any split of the tile can, and 8 waves keep 8 k-blocks in flight.
//   fagq_gemm_ring_kernel - the waves split the tile, and share a ring of
//     k-blocks in LDS.  For the larger tiles, whose accumulators one wave cannot
//     hold.
// No tile is wider than 128 columns.  The columns of those whose width divides
// 128 lie in one 128-column weight block; a 96-column tile may straddle two, and
// each of its 16-column tiles takes its own block's scale.

// ------------------------------------------------------------------ K split over waves

// W waves; tile 16 TM x 16 TN; wave w takes k-blocks w, w + W, ...  Its loads
// of U k-blocks are in flight in VGPRs: eight consecutive lanes read one row's
// 128 bytes (the MFMA's operand layout read straight from memory puts four
// rows in every four lanes, and took 13.6 instead of 9.1 us at 32 x 4096 x
// 7168).  A k-block then passes through the wave's own 2 (TM + TN) KB of LDS,
// which turns it into operand order; the registers it leaves are refilled
// before its products run.  K-blocks past the last have an offset that no
// buffer reaches, nor their scales': they read zeros, and add nothing.
//
// Bound by the rows and columns each CU has to read, (16 TM + 16 TN) K bytes at
// about 60 KB/us and CU; below that by latency.  us per call in a replayed
// graph (weights rotated, UE8M0 scales), 256 x 192 / 256 tiles before and this
// kernel: 1 x 4096 x 7168 50.3 -> 6.9 (16 x 16), 32 x 4096 x 7168 51.2 -> 8.1
// (32 x 32), 128 x 4096 x 7168 52.9 -> 11.9 (32 x 64), 32 x 1024 x 512 8.3 ->
// 3.2 (16 x 16).
template <int ASF, int BSF, int TM, int TN, int W, int U>
__global__ void __launch_bounds__(64 * W) fagq_gemm_waves_kernel(const GArgs g) {
  constexpr int BM = 16 * TM, BN = 16 * TN;
  constexpr int kStage = (TM + TN) * 16 * kBK;           // one k-block of one wave
  constexpr int kPartial = TM * TN * 1024;               // one wave's fp32 tile
  __shared__ __attribute__((aligned(1024))) uint8_t lds[W * (kStage > kPartial ? kStage : kPartial)];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int mt, nt;
  tile_coords((int)blockIdx.x, g.m_tiles, g.n_tiles, g.m_tiles, mt, nt);
  const int m0 = mt * BM, n0 = nt * BN;
  const int mrows = g.M - m0 < BM ? g.M - m0 : BM;
  const int nrows = g.N - n0 < BN ? g.N - n0 : BN;
  const rsrc_t ra = make_rsrc(g.a + (int64_t)m0 * g.K, (uint32_t)mrows * (uint32_t)g.K);
  const rsrc_t rb = make_rsrc(g.b + (int64_t)n0 * g.K, (uint32_t)nrows * (uint32_t)g.K);
  const rsrc_t ras = make_rsrc(g.as, g.as_bytes);
  const rsrc_t rbs = make_rsrc(g.bs, g.bs_bytes);

  // Load u of an operand covers rows 8 u .. 8 u + 7, the lane's row lane / 8
  // at 16-byte chunk lane % 8; it is written where lds_frag reads that chunk.
  const int crow = lane >> 3;
  const uint32_t voff = (uint32_t)crow * (uint32_t)g.K + (uint32_t)(lane & 7) * 16u;
  uint8_t* const stage = lds + wave * kStage;
  uint8_t* const put = stage + crow * kBK + swz(lane & 7, crow) * 16;
  const int r = lane & 15;
  constexpr uint32_t asb = ASF == SF_F32 ? 4u : 1u, bsb = BSF == SF_F32 ? 4u : 1u;
  const uint32_t as_voff = (uint32_t)(m0 + r) * (uint32_t)g.as_mstride * asb;
  const uint32_t bs_row = (uint32_t)(n0 >> 7) * (uint32_t)g.kblocks;

  struct Block {
    u32x4 b[2 * TN], a[2 * TM];
    uint32_t sb, sa[TM];
  };
  auto load = [&](Block& x, int i) {
    const int kb = wave + W * i;
    const bool ok = kb < g.kblocks;
    // 2^31 and up: past every operand (4 MiB at most: 64 rows, K <= 2^16) and scale
    // array (128 MiB at most: 2^16 rows, 512 k-blocks of 4 bytes).
    const uint32_t far = 0x80000000u;
    const uint32_t ko = (uint32_t)__builtin_amdgcn_readfirstlane(
        (int)(ok ? (uint32_t)kb * (uint32_t)kBK : far));
    const uint32_t so = (uint32_t)__builtin_amdgcn_readfirstlane((int)(ok ? 0u : far));
    const uint32_t kc = ok ? (uint32_t)kb : 0u;
#pragma unroll
    for (int j = 0; j < 2 * TN; ++j)
      x.b[j] = __builtin_amdgcn_raw_buffer_load_b128(rb, voff + 8u * j * (uint32_t)g.K + ko, 0, 0);
#pragma unroll
    for (int t = 0; t < 2 * TM; ++t)
      x.a[t] = __builtin_amdgcn_raw_buffer_load_b128(ra, voff + 8u * t * (uint32_t)g.K + ko, 0, 0);
    x.sb = load_scale<BSF>(rbs, so + (bs_row + kc) * bsb);
#pragma unroll
    for (int t = 0; t < TM; ++t)
      x.sa[t] = load_scale<ASF>(ras, so + as_voff + (kc * (uint32_t)g.as_kstride +
                                                     16u * t * (uint32_t)g.as_mstride) * asb);
  };

  f32x4 acc[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int t = 0; t < TM; ++t) acc[j][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // Products of the k-block in x, after k-block `next` (if any) is on its way
  // into x.  A wave's LDS accesses run in order, so its stage needs no barrier.
  auto step = [&](Block& x, bool refill, int next) {
    uint32_t sa[TM];
#pragma unroll
    for (int t = 0; t < TM; ++t) sa[t] = x.sa[t];
    const uint32_t sb = x.sb;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < 2 * TN; ++j) *reinterpret_cast<u32x4*>(put + j * 1024) = x.b[j];
#pragma unroll
    for (int t = 0; t < 2 * TM; ++t) *reinterpret_cast<u32x4*>(put + (2 * TN + t) * 1024) = x.a[t];
    issue_order_fence();
    __builtin_amdgcn_sched_barrier(0);
    if (refill) load(x, next);
    __builtin_amdgcn_sched_barrier(0);
    i32x8 af[TM], bf[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) bf[j] = lds_frag(stage, 16 * j + r, lane);
#pragma unroll
    for (int t = 0; t < TM; ++t) af[t] = lds_frag(stage, 16 * (TN + t) + r, lane);
    issue_order_fence();
    const uint32_t sbs[1] = {sb};
    products<ASF, BSF>(acc, bf, af, sbs, sa);
  };

  Block x[U];
#pragma unroll
  for (int u = 0; u < U; ++u) load(x[u], u);
  const int steps = (g.kblocks + W - 1) / W;             // the first wave's k-blocks
  int i = 0;
  for (; i + U < steps; i += U) {
#pragma unroll
    for (int u = 0; u < U; ++u) step(x[u], true, i + u + U);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) step(x[u], false, 0);

  // The partial tiles, added in wave order.
  __syncthreads();                                       // the stages have been read
  f32x4* const part = reinterpret_cast<f32x4*>(lds);
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int t = 0; t < TM; ++t) part[((wave * TN + j) * TM + t) * 64 + lane] = acc[j][t];
  __syncthreads();
  const rsrc_t rc = make_rsrc(g.c + (int64_t)m0 * g.N, (uint32_t)mrows * (uint32_t)g.N * 2u);
  for (int q = wave; q < TM * TN; q += W) {
    const int j = q / TM, t = q % TM, ncol = n0 + 16 * j;
    if (ncol >= g.N) continue;                           // uniform over the wave
    f32x4 v = part[q * 64 + lane];
#pragma unroll
    for (int w = 1; w < W; ++w) {
      const f32x4 p = part[(w * TN * TM + q) * 64 + lane];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += p[e];
    }
    store_tile(rc, g.N, v, 16 * t + r, ncol, lane);
  }
}

// ------------------------------------------------------------------ ring of k-blocks

// WM x WN waves of 16 TM x 16 TN outputs share S stages of LDS, each one
// k-block of the tile's rows and columns.  In step k (one barrier) a wave
// issues k-block k + S's scale loads and copies into the stage that the
// barrier freed, reads the fragments of k + 1 and multiplies k from registers.
// Both the scales and the copies run S k-blocks ahead: vector-memory results
// return in order, so scales loaded one k-block ahead would also wait for
// every older copy and leave one k-block in flight whatever S is (31.9 against
// 28.3 us at 1000 x 2112 x 7168).  The sums run in k-block order, as in the
// ping-pong kernel.
//
// Bound by the copies (a copy-only build takes 22-24 of 28-30 us at 1000 x 2112
// x 7168: about 80 KB/us and CU, each k-block's first reader in an XCD waiting
// for memory) and by LDS, which serves 128 bytes a cycle: (WN + 1) 16 TM WM +
// (WM + 1) 16 TN WN cycles a k-block against MFMA's 8 TM TN WM WN.  us per call,
// UE8M0, 256-row tiles before and this kernel: 256 x 4096 x 7168 55.4 -> 16.0
// (64 x 64), 512 x 4096 x 7168 55.7 -> 23.0 (128 x 64), 1000 x 2112 x 7168 56.4
// -> 25.5 (96 x 96; 128 x 128: 30.2), 1500 x 4096 x 7168 57.3 -> 46.4 (192 x 128).
// The 96 x 96 tile with 6 waves: 24.8 .. 27.7 there, but 46 against 41 us at 2048 x 2112 x
// 7168, where two workgroups share a CU.  4 waves with 4 or 6 stages took 29.5 and 32.0,
// which says nothing of the depth: with LDS for one workgroup per CU only, the launch
// bounds allow 512 registers, the compiler keeps the 36 accumulators in AGPRs, and each
// k-block then moves them to VGPRs and back (51 v_accvgpr moves a k-block, none with 3 stages).
template <int TM_, int TN_, int WM_, int WN_, int S_>
struct Ring {
  static constexpr int TM = TM_, TN = TN_, WM = WM_, WN = WN_, S = S_;
  static constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN, WAVES = WM * WN;
  static constexpr int STAGE = (BM + BN) * kBK;
  static constexpr int PER_CU = 160 * 1024 / (S * STAGE);          // workgroups by LDS
  static constexpr int COPIES = (BM + BN) / 8 / WAVES;             // 1 KB copies per wave and stage
  static constexpr int NB = 128 % BN ? 2 : 1;                      // weight blocks of a wave's columns
  static_assert(COPIES * WAVES * 8 == BM + BN, "the waves share a stage's copies evenly");
  static_assert(S >= 3 && PER_CU >= 1 && BN <= 128 && (S - 1) * (COPIES + TM + NB) < 64,
                "ring geometry");
};

template <int ASF, int BSF, class R>
__global__ void __launch_bounds__(64 * R::WAVES, R::PER_CU * R::WAVES / 4)
fagq_gemm_ring_kernel(const GArgs g) {
  constexpr int TM = R::TM, TN = R::TN, S = R::S, C = R::COPIES;
  constexpr int kScaleLoads = TM + R::NB;                    // memory instructions of load_scales
  __shared__ __attribute__((aligned(1024))) uint8_t lds[S * R::STAGE];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave % R::WM, wn = wave / R::WM;
  int mt, nt;
  tile_coords((int)blockIdx.x, g.m_tiles, g.n_tiles, kGroupM, mt, nt);
  const int m0 = mt * R::BM, n0 = nt * R::BN;
  const int mrows = g.M - m0 < R::BM ? g.M - m0 : R::BM;
  const int nrows = g.N - n0 < R::BN ? g.N - n0 : R::BN;
  const rsrc_t ra = make_rsrc(g.a + (int64_t)m0 * g.K, (uint32_t)mrows * (uint32_t)g.K);
  const rsrc_t rb = make_rsrc(g.b + (int64_t)n0 * g.K, (uint32_t)nrows * (uint32_t)g.K);
  const rsrc_t ras = make_rsrc(g.as, g.as_bytes);
  const rsrc_t rbs = make_rsrc(g.bs, g.bs_bytes);
  const int last = g.kblocks - 1;

  // As in the ping-pong kernel: copy `inst` fills stage rows 8 inst .. + 7 (the
  // activation rows, then the weight rows), the lane fetching the chunk that
  // the swizzle puts at its place.  K-blocks past the last fetch the last one
  // again, into stages nobody reads, so that every step issues the same.
  const int crow = lane >> 3;
  const uint32_t cvoff = (uint32_t)crow * (uint32_t)g.K + (uint32_t)swz(lane & 7, crow) * 16u;
  auto copy_stage = [&](int kb, int slot) {
    const int kc = kb < last ? kb : last;
#pragma unroll
    for (int u = 0; u < C; ++u) {
      const int inst = wave * C + u;
      const bool act = inst < R::BM / 8;
      const int rows8 = act ? inst : inst - R::BM / 8;
      const uint32_t off = cvoff + (uint32_t)__builtin_amdgcn_readfirstlane(
          (int)((uint32_t)rows8 * 8u * (uint32_t)g.K + (uint32_t)kc * (uint32_t)kBK));
      lds_void_t* const dst = (lds_void_t*)(lds + slot * R::STAGE + inst * 1024);
      if (act) __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, dst, 16, off, 0, 0, 0);
      else __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, dst, 16, off, 0, 0, 0);
    }
  };
  constexpr uint32_t asb = ASF == SF_F32 ? 4u : 1u, bsb = BSF == SF_F32 ? 4u : 1u;
  const int r = lane & 15;
  const uint32_t as_voff = (uint32_t)(m0 + wm * 16 * TM + r) * (uint32_t)g.as_mstride * asb;
  const int wcol = n0 + wn * 16 * TN;
  // The wave's column tiles from jsplit on lie in the next weight block (NB 2).
  // Past the last column that may be no block of B at all: out of range, zero.
  const uint32_t bs_row = (uint32_t)(wcol >> 7) * (uint32_t)g.kblocks;
  const int jsplit = ((wcol & -128) + 128 - wcol) / 16;
  struct Scales {
    uint32_t b[R::NB], a[TM];
  };
  auto load_scales = [&](int kb) {
    const int kc = kb < last ? kb : last;
    Scales s;
#pragma unroll
    for (int i = 0; i < R::NB; ++i)
      s.b[i] = load_scale<BSF>(rbs, (bs_row + (uint32_t)(i * g.kblocks + kc)) * bsb);
#pragma unroll
    for (int t = 0; t < TM; ++t)
      s.a[t] = load_scale<ASF>(ras, as_voff + ((uint32_t)kc * (uint32_t)g.as_kstride +
                                               16u * t * (uint32_t)g.as_mstride) * asb);
    return s;
  };
  auto read_frags = [&](int slot, i32x8 (&bf)[TN], i32x8 (&af)[TM]) {
    const uint8_t* ta = lds + slot * R::STAGE;
    const uint8_t* tb = ta + R::BM * kBK;
#pragma unroll
    for (int t = 0; t < TM; ++t) af[t] = lds_frag(ta, wm * 16 * TM + 16 * t + r, lane);
#pragma unroll
    for (int j = 0; j < TN; ++j) bf[j] = lds_frag(tb, wn * 16 * TN + 16 * j + r, lane);
  };

  f32x4 acc[TN][TM];
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int t = 0; t < TM; ++t) acc[j][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  // K-block k: stage and scales k % S, fragment set k % 2; the loop is unrolled
  // so that all three are constants.
  constexpr int kUnroll = S % 2 ? 2 * S : S;
  i32x8 bf[2][TN], af[2][TM];
  Scales sc[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    sc[s] = load_scales(s);
    issue_order_fence();
    copy_stage(s, s);
    issue_order_fence();
  }
  __builtin_amdgcn_s_waitcnt(vmcnt_imm((S - 1) * (C + kScaleLoads)));
  pp_barrier();
  read_frags(0, bf[0], af[0]);
  auto step = [&](auto phase, int k) {
    constexpr int p = decltype(phase)::value;
    // This wave's copies of k + 1 have landed (k + 2 .. k + S - 1 follow them),
    // and its fragments of k; after the barrier everybody's have.
    __builtin_amdgcn_s_waitcnt(vmcnt_imm((S - 2) * (C + kScaleLoads)));
    pp_barrier();
    const Scales s = sc[p % S];
    sc[p % S] = load_scales(k + S);
    issue_order_fence();
    copy_stage(k + S, p % S);
    issue_order_fence();
    read_frags((p + 1) % S, bf[(p + 1) % 2], af[(p + 1) % 2]);
    __builtin_amdgcn_sched_barrier(0);
    constexpr int kB = R::NB == 1 ? 1 : TN;
    uint32_t sb[kB];
#pragma unroll
    for (int j = 0; j < kB; ++j) sb[j] = R::NB == 1 || j < jsplit ? s.b[0] : s.b[R::NB - 1];
    products<ASF, BSF>(acc, bf[p % 2], af[p % 2], sb, s.a);
    __builtin_amdgcn_sched_barrier(0);
  };
  bool more = true;                                      // uniform over the workgroup
  for (int k = 0; more;) {
    unrolled<kUnroll>([&](auto phase) {
      if (more) {
        step(phase, k);
        more = ++k < g.kblocks;
      }
    });
  }
  __builtin_amdgcn_s_waitcnt(kVmcnt0);                   // the copies past the last k-block

  const rsrc_t rc = make_rsrc(g.c + (int64_t)m0 * g.N, (uint32_t)mrows * (uint32_t)g.N * 2u);
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int ncol = wcol + 16 * j;
    if (ncol >= g.N) continue;                           // uniform over the wave
#pragma unroll
    for (int t = 0; t < TM; ++t) store_tile(rc, g.N, acc[j][t], wm * 16 * TM + 16 * t + r, ncol, lane);
  }
}
