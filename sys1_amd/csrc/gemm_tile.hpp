// Projection GEMM for gfx950: y[M,N] = epi(x[M,K] . w[N,K]^T) on
// v_mfma_f32_32x32x16_bf16.  One kernel template covers both regimes:
//   - large M: MFMA-bound output tiles, one k-stream per tile;
//   - small M (the weight-streaming regime): BM = the padded token count,
//     BN = 256, with K split over workgroups so that every CU streams weight.
//
// Tile:    BM x BN output tile, BK = 64 or 32, WM x WN waves, each wave owns a
//          (BM/WM) x (BN/WN) sub-tile of 32x32 MFMA blocks.  The MFMA takes the
//          weight block as A and the activation block as B, so a lane's
//          accumulator holds runs of 4 consecutive output features of one
//          token.
// Loads:   global -> LDS directly (buffer_load ... lds, no VGPR staging).  One
//          wave instruction fills 1 KB of LDS = 8 rows x 128 B (BK = 64) or
//          16 rows x 64 B (BK = 32); the lanes of a row read its line
//          (coalesced) in a permuted chunk order that realises the LDS swizzle
//          below.  The x and w instructions of a
//          k-tile form one list dealt round-robin to the waves, so every wave
//          issues the same count and vmcnt bookkeeping stays exact.
// LDS:     per operand, row-major rows of BK bf16; the 16-byte chunk c of
//          row r sits at position c ^ f(r), f(r) = (r ^ r/8) & 7 for 128 B
//          rows ((r ^ r/4) & 3 for 64 B rows).
//          With this f the MFMA operand reads (lanes 0-31: 32 rows of one
//          chunk, lanes 32-63: the next chunk) run without LDS bank conflicts
//          on gfx950 (SQ_LDS_BANK_CONFLICT = 0 measured; the plain r & 7 and
//          (r + r/8) & 7 swizzles measure 2-way).
// Pipeline: STAGES LDS stages fed as one stream of k-tiles that runs across
//          the work items a persistent workgroup serves, so the next item's
//          loads overlap the current item's last k-tiles and its epilogue.
//          Fragments are double-buffered in registers across k-steps, and the
//          last k-step's MFMAs run after the barrier, overlapping the next
//          k-tile's first LDS reads; the freed stage's refill is issued
//          behind them (spread between them with one workgroup per CU).
// Epilogue: straight from registers: lane pairs (l, l+32) exchange halves
//          with v_permlane32_swap so that every lane stores (and reads the
//          residual as) 16 contiguous bytes; no LDS, so all of it goes to
//          pipeline stages.
// Stream-K: the weight-streaming shapes split the flattened (tile, k-tile)
//          iteration space into one equal contiguous range per workgroup, so
//          every CU streams the same share of the weight (optionally after a
//          phase of whole tiles: the hybrid schedule of TileWalk).  A range covers at
//          most a partial head segment, whole tiles, and a partial tail
//          segment; a partial segment writes its f32 accumulators to the
//          workspace (head or tail slot of its workgroup), and, per wave
//          slice of the tile, the last owner to arrive (an arrival counter
//          per tile and wave) sums the slice's partials in workgroup order --
//          deterministic whatever the arrival order -- applies the epilogue
//          to it and re-arms the counter.
#pragma once
#define SYS1_GEMM_TILE_HPP

#include <type_traits>

#include "common.hpp"

namespace sys1 {

__device__ __forceinline__ f32x16 mfma32(const i32x4& a, const i32x4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                  __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// LDS row swizzle: chunk c of row r is stored at position c ^ swz(r).
// Measured conflict-free for the 32-lane fragment reads on gfx950: 128-byte
// rows (BK = 64, 8 chunks) use (r ^ r/8) & 7, 64-byte rows (BK = 32, 4
// chunks) use (r ^ r/4) & 3.
template <int BK>
__device__ __forceinline__ int lds_swz(int row) {
  if constexpr (BK == 64) return (row ^ (row >> 3)) & 7;
  else return (row ^ (row >> 2)) & 3;
}

template <int BM, int BN, int WM, int WN, int STAGES, int BK_>
struct TileShape {
  // (a blocked weight's k-tile is one 4 KB block per 32 tile rows)
  static_assert(BN % kBlkRows == 0 && BK_ == kBlkK, "tiles start on weight blocks of the blocked layout");
  static constexpr int kWaves = WM * WN;
  static constexpr int kThreads = kWaves * 64;
  static constexpr int BK = BK_;
  static_assert(BK == 32 || BK == 64, "k-tile of 32 or 64");
  static constexpr int TM = BM / WM;
  static constexpr int TN = BN / WN;
  static constexpr int FM = TM / 32;
  static constexpr int FN = TN / 32;
  static constexpr int KS = BK / 16;                 // MFMA k-steps per k-tile
  static constexpr int kRowBytes = BK * 2;           // 128 or 64
  static constexpr int CPR = BK / 8;                 // 16-byte chunks per row
  static constexpr int RPI = 1024 / kRowBytes;       // rows per DMA instruction (1 KB)
  static constexpr int kXBytes = BM * kRowBytes;     // one stage of x
  static constexpr int kWBytes = BN * kRowBytes;
  static constexpr int kStageBytes = kXBytes + kWBytes;
  static constexpr int kStagesBytes = STAGES * kStageBytes;
  static constexpr int kLdsBytes = kStagesBytes;
  static constexpr int XT = BM / RPI;                // DMA instructions per k-tile: x
  static constexpr int DT = (BM + BN) / RPI;         // x and w together
  static constexpr int kDma = DT / kWaves;           // per wave per k-tile
  static_assert(TM % 32 == 0 && TN % 32 == 0, "wave tile must be whole 32x32 blocks");
  static_assert(BM % RPI == 0 && BN % RPI == 0, "whole DMA instructions per tile");
  static_assert(STAGES >= 2, "at least double buffering");
  static_assert(kLdsBytes <= 160 * 1024, "LDS budget of one gfx950 CU");
  static_assert(kDma * (STAGES - 1) < 64, "vmcnt field");
};

// A segment of a workgroup's k-tile stream: k-tiles [kt0, kt1) of one tile.
struct Segment {
  int tm, tn;     // tile coordinates
  int kt0, kt1;   // k-tile range
  int pos;        // position in this workgroup's step sequence
  int st;         // stream-phase tile index (tile - dp_tiles), -1 in the tile phase
  int spos;       // stream-phase position of its first k-tile (st * kt_count + kt0)
};

// Persistent schedule over tiles rasterised in groups of group_m tile rows
// (tiles in flight together share x row panels and w column panels in L2).
// The grid holds at most (CUs x resident workgroups per CU) workgroups G.
//   Tile phase: tiles [0, dp_tiles), each a whole segment.  Workgroup b
//     serves XCD b % 8 and walks that XCD's contiguous share of these tiles
//     with stride (workgroups on the XCD).
//   Stream phase: the k-iterations of tiles [dp_tiles, tiles) flattened,
//     T = (tiles - dp_tiles) * kt_count; workgroup g < G' = min(G, T) owns
//     [start(g), start(g+1)), start(g) = g * T / G'.  A tile split over several
//     workgroups is summed by its last arriving owner.
// dp_tiles = tiles is the plain persistent tile schedule; dp_tiles = 0 is
// pure stream-K (the weight-streaming small-M shapes); in between is the
// hybrid that runs whole rounds of tiles and spreads the last, partial round
// over every CU.
struct TileWalk {
  int tiles_m, tiles_n, kt_count, tiles, dp_tiles;
  int step_m;  // rows between tile rows: BM, or BM - halo (tile rows overlap by the halo)
  // tile phase
  int first, count, stride;
  // stream phase
  int64_t total;
  int grid, sgrid, begin, end;  // sgrid: workgroups in the stream phase
  int dp_steps;

  int group_m;

  // halo > 0: tile row tm covers rows [tm (BM - halo), + BM), so the halo
  // rows before each tile row's outputs are computed in the same tile.
  __device__ TileWalk(int M, int N, int K, int BM, int BN, int BK, int dp, int group, int halo = 0) {
    group_m = max(1, group);
    step_m = BM - halo;
    tiles_m = M <= BM ? 1 : 1 + (M - BM + step_m - 1) / step_m;
    tiles_n = (N + BN - 1) / BN;
    kt_count = (K + BK - 1) / BK;
    tiles = tiles_m * tiles_n;
    dp_tiles = min(dp, tiles);
    grid = gridDim.x;
    // Workgroups are dispatched round-robin over the 8 XCDs; a grid smaller
    // than that deals the tiles over as many groups as it has workgroups.
    const int xcds = min(8, grid);
    const int xcd = blockIdx.x % xcds;
    const int slot = blockIdx.x / xcds;
    const int slots = grid / xcds + (xcd < grid % xcds ? 1 : 0);  // workgroups on this XCD
    const int per = dp_tiles / xcds, rem = dp_tiles % xcds;
    const int xbegin = xcd * per + min(xcd, rem);
    const int xcount = per + (xcd < rem ? 1 : 0);
    first = xbegin + slot;
    stride = slots;
    count = slot < xcount ? (xcount - slot + slots - 1) / slots : 0;
    dp_steps = count * kt_count;
    total = (int64_t)(tiles - dp_tiles) * kt_count;
    // At most one workgroup per iteration, so that every stream range is
    // non-empty (the arrival count of a split tile is its owner count).
    sgrid = (int)min<int64_t>(grid, total);
    begin = (int)blockIdx.x < sgrid ? start(blockIdx.x) : 0;
    end = (int)blockIdx.x < sgrid ? start(blockIdx.x + 1) : 0;
  }
  __device__ int start(int g) const { return (int)((int64_t)g * total / sgrid); }
  __device__ int row0(int tm) const { return tm * step_m; }

  // Tile index -> coordinates (grouped raster).
  __device__ void tile_coords(int t, int& tm, int& tn) const {
    const int group = t / (group_m * tiles_n);
    const int first_m = group * group_m;
    const int gm = min(group_m, tiles_m - first_m);
    const int in = t - group * group_m * tiles_n;
    tm = first_m + in % gm;
    tn = in / gm;
  }
  __device__ int steps() const { return dp_steps + (end - begin); }
  // The segment whose first k-tile is step `pos` of this workgroup.
  __device__ Segment segment_at(int pos) const {
    Segment sg;
    if (pos < dp_steps) {
      const int j = pos / kt_count;
      tile_coords(first + j * stride, sg.tm, sg.tn);
      sg.kt0 = 0;
      sg.kt1 = kt_count;
      sg.st = -1;
      sg.spos = 0;
    } else {
      const int sp = begin + (pos - dp_steps);
      const int t = sp / kt_count;
      tile_coords(dp_tiles + t, sg.tm, sg.tn);
      sg.kt0 = sp - t * kt_count;
      sg.kt1 = min(kt_count, sg.kt0 + (end - sp));
      sg.st = t;
      sg.spos = sp;
    }
    sg.pos = pos;
    return sg;
  }
  __device__ Segment first_segment() const { return segment_at(0); }
  __device__ Segment next_segment(const Segment& sg) const {
    return segment_at(sg.pos + (sg.kt1 - sg.kt0));
  }
  __device__ bool complete(const Segment& sg) const { return sg.kt0 == 0 && sg.kt1 == kt_count; }
  // Stream phase: the workgroups whose ranges overlap stream tile st, [g_lo, g_hi].
  __device__ void tile_owners(int st, int& g_lo, int& g_hi) const {
    const int64_t lo = (int64_t)st * kt_count, hi = lo + kt_count;  // [lo, hi)
    int g = (int)(lo * sgrid / total);
    while (g > 0 && start(g) > lo) --g;
    while (start(g + 1) <= lo) ++g;
    g_lo = g;
    g = (int)((hi - 1) * sgrid / total);
    while (g > 0 && start(g) > hi - 1) --g;
    while (start(g + 1) <= hi - 1) ++g;
    g_hi = g;
  }
};

// STREAMK: stream-K schedule (the weight-streaming shapes); the large-M
// shapes compile the tile schedule only.
// OCC: resident workgroups per CU the register allocation must allow.
// PW: producer waves.  0: every wave issues its share of the refills between
// its MFMAs.  PW > 0: PW extra waves issue all of them and do nothing else,
// so a refill instruction that stalls issue while the load path drains
// stalls no matrix work.  Under stream-K the compute waves then also wait
// for their partial stores (before the arrival counter) without draining
// the refills in flight: a wave's vmcnt covers every vector memory access
// it issued, and with producer waves those are its stores alone.
// PW < 0: the ping-pong schedule (see below), STAGES its ring's slots.
constexpr int producer_waves(int pw) { return pw > 0 ? pw : 0; }
template <int BM, int BN, int WM, int WN, int STAGES_, int BK_, int OCC, bool STREAMK, int EPI, int PW_ = 0>
__global__ __launch_bounds__((WM * WN + producer_waves(PW_)) * 64)
__attribute__((amdgpu_waves_per_eu(((WM * WN + producer_waves(PW_)) * OCC + 3) / 4))) void gemm_tile_kernel(GemmArgs a) {
  constexpr bool kPP = PW_ < 0;
  constexpr int PW = producer_waves(PW_);
  constexpr int STAGES = kPP ? 2 : STAGES_;
  using S = TileShape<BM, BN, WM, WN, STAGES, BK_>;
  constexpr int BK = S::BK;
  // Residual epilogues of producer-wave tile kernels whose LDS budget has
  // room: the producers copy each tile's residual block into LDS while its
  // k-loop runs, so the epilogue does not wait on a read from HBM.
  constexpr bool kResLds = PW > 0 && !STREAMK && epi_has_resid<epi_base(EPI)>() &&
                           (S::kLdsBytes + BM * BN * 2) * OCC <= 160 * 1024 && (BM * BN * 2 / 1024) % PW == 0;
  constexpr int kResBytes = kResLds ? BM * BN * 2 : 0;
  // Row statistics of a fused pre-norm: under stream-K each compute wave sums
  // the squares of the rows it multiplies for RMSNorm (RowSums); the others
  // read those of a pass before them: LayerNorm's variance is taken about the
  // mean, which no sum over one walk of K gives (layer_stats).  The tile
  // kernels were built with sums of their own, both ways, and lost
  // what the pass costs: in the producer waves, from the landed stages, the
  // sums delayed the refills (ModernBERT-base Wi+LN at 8109 tokens 48.9 us
  // against 49.3 with the pass, Qwen3.5-small in_proj at 8192 409.6 against
  // 378.5); in the compute waves they spilled (58.0 and 459.4 us).
  constexpr bool kStatPass = !STREAMK || epi_base(EPI) == kEpiConvSilu || epi_norm(EPI) == kNormLayer;
  constexpr int kOwnNorm = kStatPass ? kNormNone : epi_norm(EPI);
  // (the ping-pong ring: STAGES_ slots of half the x or half the w rows)
  constexpr int kSlotBytes = (BM > BN ? BM : BN) / 2 * S::kRowBytes;
  static_assert(!kPP || STAGES_ * kSlotBytes <= 160 * 1024, "LDS budget of one gfx950 CU");
  __shared__ __attribute__((aligned(1024))) char lds[kPP ? STAGES_ * kSlotBytes : S::kLdsBytes + kResBytes];
  char* const res_lds = lds + S::kLdsBytes;
  // (every k-tile loop needs two k-steps per tile, so that a tile's copy,
  // issued after its first barrier, lands before its last)
  const bool res_in_lds = kResLds && a.K > BK_ && a.Nout >= 8 && a.Nout % 8 == 0 && a.ldr % 8 == 0 &&
                          (reinterpret_cast<uintptr_t>(a.resid) & 15) == 0 &&
                          (int64_t)a.M * a.ldr * 2 < 0x7ffffff0ll;

  constexpr bool kConv = epi_base(EPI) == kEpiConvSilu;
  static_assert(!kConv || WM == 1, "conv epilogue: one wave row per tile");
  static_assert(PW == 0 || !kConv, "producer waves: no conv epilogue");
  const TileWalk walk(a.M, a.N, a.K, BM, BN, BK, STREAMK ? a.dp_tiles : 1 << 30, a.group_m,
                      kConv ? kConvHalo : 0);
  if (walk.steps() == 0) return;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: keep in SGPRs
  const int wm = wave / WN;
  const int wn = wave % WN;

  // ---- DMA.  The issue cursor walks the segments in stream order.
  // Instruction u = i * waves + wave of a k-tile: u < XT covers x rows
  // RPI*u .. RPI*u + RPI-1, else w rows RPI*(u-XT) ..; either way its 1 KB
  // lands at stage offset u * 1 KB.  Lane -> row + lane/CPR, position
  // lane%CPR, source chunk position ^ swz(row).  Rows past M / N clamp to
  // the last row; chunks past K read zeros through an out-of-range buffer
  // offset.
  const int lrow = lane / S::CPR, lpos = lane % S::CPR;
  // A wave's first kXDma instructions read x, the rest w.  Row, chunk and
  // swizzle of each instruction depend only on the lane, so the per-lane
  // source offsets (row clamp included) are computed when the issue cursor
  // enters a tile; a k-tile then costs only the scalar base advance, and the
  // K-tail test runs on a tile's last, partial k-tile only.
  constexpr int kDW = PW ? PW : S::kWaves;  // waves that issue refills
  constexpr int kDma = S::DT / kDW;          // refill instructions per issuing wave per k-tile
  static_assert(S::XT % kDW == 0 && S::DT % kDW == 0, "x and w instructions deal evenly over the waves");
  static_assert(kDma * (STAGES - 1) < 64, "vmcnt field");
  constexpr int kXDma = S::XT / kDW;
  const int dwave = PW ? wave - S::kWaves : wave;
  auto dma_row = [&](int i) {
    const int u = i * kDW + dwave;
    return (i < kXDma ? u : u - S::XT) * S::RPI + lrow;
  };
  unsigned src_off[kDma];
  auto set_offsets = [&](const Segment& sg) {
    const int x_left = a.M - 1 - walk.row0(sg.tm), w_left = a.N - 1 - sg.tn * BN;
#pragma unroll
    for (int i = 0; i < kDma; ++i) {
      const int r = dma_row(i);
      const int c = lpos ^ lds_swz<BK>(r);
      const int rw = min(r, w_left);  // (tile rows start on a 32-row block: BN % 32 == 0)
      src_off[i] = i < kXDma ? (unsigned)(min(r, x_left) * (int)a.ldx * 2 + c * 16)
                   : a.w_kt ? (unsigned)((rw / kBlkRows) * a.w_kt * kBlkBytes + (rw % kBlkRows) * (kBlkK * 2) + c * 16)
                            : (unsigned)(rw * (int)a.ldw * 2 + c * 16);
    }
  };
  Segment isg = walk.first_segment();
  int is_kt = isg.kt0;
  set_offsets(isg);
  // A refill of one stage from the cursor's k-tile, prepared once (scalar
  // descriptors, stage base, K-tail extent); dma_one(r, i) issues its
  // instruction i and issue_advance() then moves the cursor on, so that the
  // refill can be spread between MFMAs (mma_dma below).  A refill that is
  // not live gets descriptors of zero size: its instructions read zeros into
  // a stage that is never read again (the end of the stream), so the main
  // loop issues the same instruction sequence every k-tile.
  struct Refill {
    rsrc_t xr, wr;
    char* base;
    int kleft;  // valid K elements in the k-tile
  };
  auto refill_at = [&](int stage, bool live) {
    Refill r;
    const int m0 = walk.row0(isg.tm), n0 = isg.tn * BN;
    const int bytes = live ? 0x7ffffff0 : 0;
    r.base = lds + stage * S::kStageBytes;
    r.xr = make_rsrc_uniform(reinterpret_cast<const char*>(a.x + (int64_t)m0 * a.ldx) + is_kt * BK * 2, bytes);
    r.wr = make_rsrc_uniform(
        a.w_kt ? reinterpret_cast<const char*>(a.w) + ((int64_t)(n0 / kBlkRows) * a.w_kt + is_kt) * kBlkBytes
               : reinterpret_cast<const char*>(a.w + (int64_t)n0 * a.ldw) + is_kt * BK * 2,
        bytes);
    r.kleft = a.K - is_kt * BK;
    return r;
  };
  auto dma_one = [&](const Refill& r, int i) {
    unsigned off = src_off[i];
    if (r.kleft < BK && (lpos ^ lds_swz<BK>(dma_row(i))) * 8 >= r.kleft) off = kOutOfRange;
    // Stream-K reads each weight byte once per call: its weight loads are
    // non-temporal (nt), measured 4-8% faster on the weight streams than
    // the default policy.
    if (i < kXDma || !STREAMK) dma16(i < kXDma ? r.xr : r.wr, off, (lds_void*)(r.base + (i * kDW + dwave) * 1024));
    else dma16_pol<kCachePolicyNt>(r.wr, off, (lds_void*)(r.base + (i * kDW + dwave) * 1024));
  };
  auto issue_advance = [&]() {
    if (++is_kt == isg.kt1) {
      isg = walk.next_segment(isg);
      is_kt = isg.kt0;
      set_offsets(isg);
    }
  };
  auto issue = [&](int stage) {  // issue the cursor's k-tile, then advance the cursor
    const Refill r = refill_at(stage, true);
#pragma unroll
    for (int i = 0; i < kDma; ++i) dma_one(r, i);
    issue_advance();
  };

  // ---- producer waves: the prologue's requests, then per k-tile: wait for
  // the next k-tile's loads, the barrier that retires the current one (the
  // compute waves' barrier, one per k-tile on both sides), then the refill
  // of the stage it freed.
  if constexpr (PW > 0) {
    if (wave >= S::kWaves) {
      const int steps = walk.steps();
      // The residual copy of tile `sg`: instruction i fills LDS bytes
      // [1024 i, 1024 i + 1024) of the row-major [BM][BN] block.  Rows past
      // M and columns past Nout read clamped (their outputs are not stored).
      auto issue_res = [&](const Segment& sg) {
        if constexpr (kResLds) {
          const rsrc_t rr = make_rsrc_uniform(a.resid, 0x7ffffff0);
          const int m0 = walk.row0(sg.tm), n0 = sg.tn * BN;
#pragma unroll
          for (int q = 0; q < BM * BN * 2 / 1024 / PW; ++q) {
            const int i = q * PW + dwave;
            const int e = i * 512 + lane * 8;
            const int row = min(m0 + e / BN, a.M - 1), col = min(n0 + e % BN, a.Nout - 8);
            dma16(rr, (unsigned)(((int64_t)row * a.ldr + col) * 2), (lds_void*)(res_lds + i * 1024));
          }
        }
      };
      Segment psg = walk.first_segment();  // the tile of step s
      int pkt = psg.kt0;
      for (int t = 0; t < STAGES; ++t)
        if (t < steps) issue(t);
      if (steps >= STAGES) vm_wait<(STAGES - 1) * kDma>();
      else vm_wait<0>();
      if (res_in_lds) issue_res(psg);
      __syncthreads();
      int stage = 0;
      asm volatile(".p2align 7");  // (the loop's place in its lines: see align_loop)
      for (int s = 0; s < steps; ++s) {
        // Before the barrier after which the tile's epilogue runs, its
        // residual copy has landed too.
        const bool tile_end = kResLds && pkt + 1 == psg.kt1;
        if (res_in_lds && tile_end) {
          vm_wait<0>();
        } else if (s + 1 < steps) {
          if (s + STAGES - 1 < steps) vm_wait<(STAGES - 2) * kDma>();
          else vm_wait<0>();
        }
        __syncthreads();
        const int freed = stage;
        stage = stage + 1 == STAGES ? 0 : stage + 1;
        if (s + STAGES < steps) issue(freed);
        // A tile's copy goes out after its first barrier: the compute waves
        // have finished the previous tile's epilogue to get there.
        if constexpr (kResLds) {
          if (res_in_lds && s > 0 && pkt == psg.kt0) issue_res(psg);
          if (tile_end && s + 1 < steps) {
            psg = walk.next_segment(psg);
            pkt = psg.kt0;
          } else {
            ++pkt;
          }
        }
      }
      vm_wait<0>();
      return;
    }
  }

  // ---- fragment sets in registers (see the main loop):
  //   kDeep: one set per k-step of a k-tile;  otherwise two (ping-pong).
  constexpr int kReads = S::FM + S::FN;  // LDS reads per fragment set
  constexpr int kWavesPerSimd = ((S::kWaves + PW) * OCC + 3) / 4;  // register budget 512 / this
  constexpr bool kDeep = S::KS == 4 && kReads * 4 * 4 <= 64 && kWavesPerSimd <= 3;
  static_assert(kDeep || S::FM * S::FN * 16 + 2 * kReads * 4 + 24 <= 512 / kWavesPerSimd,
                "two fragment sets fit beside the accumulators");

  // ---- fragment addressing (byte offsets within a stage): lane reads row
  // (base + lane%32) of chunk 2*ks + lane/32.
  const int frow = lane & 31;
  const int fk = lane >> 5;
  int xrow_off[S::FM], xrow_swz[S::FM], wrow_off[S::FN], wrow_swz[S::FN];
#pragma unroll
  for (int j = 0; j < S::FM; ++j) {
    const int r = wm * S::TM + j * 32 + frow;
    xrow_off[j] = r * S::kRowBytes;
    xrow_swz[j] = lds_swz<BK>(r);
  }
#pragma unroll
  for (int i = 0; i < S::FN; ++i) {
    const int r = wn * S::TN + i * 32 + frow;
    wrow_off[i] = S::kXBytes + r * S::kRowBytes;
    wrow_swz[i] = lds_swz<BK>(r);
  }

  struct Frags {
    i32x4 x[S::FM];
    i32x4 w[S::FN];
  };
  auto read = [&](Frags& f, int stage, int ks) {
    const char* base = lds + stage * S::kStageBytes;
    const int c = ks * 2 + fk;
#pragma unroll
    for (int j = 0; j < S::FM; ++j)
      f.x[j] = *reinterpret_cast<const i32x4*>(base + xrow_off[j] + ((c ^ xrow_swz[j]) << 4));
#pragma unroll
    for (int i = 0; i < S::FN; ++i)
      f.w[i] = *reinterpret_cast<const i32x4*>(base + wrow_off[i] + ((c ^ wrow_swz[i]) << 4));
  };

  // Row sums taken by the compute waves: lane l holds row l % 32 of each x
  // block over the k-chunks of its half (l / 32).  Every wave sums the rows
  // it multiplies, so nothing is exchanged between waves.
  RowSums<kOwnNorm> sums[S::FM];
  f32x16 acc[S::FN][S::FM];
  auto zero_acc = [&]() {
#pragma unroll
    for (int j = 0; j < S::FM; ++j) sums[j] = RowSums<kOwnNorm>();
#pragma unroll
    for (int i = 0; i < S::FN; ++i)
#pragma unroll
      for (int j = 0; j < S::FM; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  };
  zero_acc();

  auto mma = [&](const Frags& f) {
#pragma unroll
    for (int i = 0; i < S::FN; ++i)
#pragma unroll
      for (int j = 0; j < S::FM; ++j) {
        acc[i][j] = mfma32(f.w[i], f.x[j], acc[i][j]);
        if (i == 0) sums[j].add(f.x[j]);
      }
  };
  // The same MFMAs with DMA instructions [I0, I0 + N) of refill `r` spread
  // evenly between them (after MFMA q go instructions I0 + q*N/Q ..
  // I0 + (q+1)*N/Q - 1, Q MFMAs in all), so that the load path drains while
  // the matrix unit works.
  auto mma_dma = [&](const Frags& f, const Refill& r, auto i0c, auto nc) {
    constexpr int I0 = decltype(i0c)::value, N = decltype(nc)::value;
    constexpr int Q = S::FN * S::FM;
#pragma unroll
    for (int i = 0; i < S::FN; ++i)
#pragma unroll
      for (int j = 0; j < S::FM; ++j) {
        const int q = i * S::FM + j;
        acc[i][j] = mfma32(f.w[i], f.x[j], acc[i][j]);
        if (i == 0) sums[j].add(f.x[j]);
#pragma unroll
        for (int d = I0 + q * N / Q; d < I0 + (q + 1) * N / Q; ++d) dma_one(r, d);
        __builtin_amdgcn_sched_barrier(0);
      }
  };

  // ---- epilogue of one tile, straight from registers.  A lane's
  // accumulator block (i, j) holds token m = lane%32 and, in register
  // 4g + e, feature 8g + 4h + e (h = lane/32).  For a register-group pair
  // (g, g+1), lanes l and l+32 hold the two 8-byte halves of token l's
  // features 8g .. 8g+7 and 8(g+1) .. 8(g+1)+7 crosswise; one
  // v_permlane32_swap per dword turns that into 16 contiguous bytes per lane
  // (lane l: features 8g.., lane l+32: 8(g+1)..), stored with one 16-byte
  // store.  Rounding mirrors the unfused reference: the projection (or the
  // gated product) is rounded to bf16 in registers; bias, gelu and the
  // residual add then apply in f32 on the stored layout, each rounded.
  auto pair16 = [](bf16x4 lo, bf16x4 hi) -> bf16x8 {
    const i32x2 a = __builtin_bit_cast(i32x2, lo), b = __builtin_bit_cast(i32x2, hi);
    const auto s0 = __builtin_amdgcn_permlane32_swap((unsigned)a[0], (unsigned)b[0], false, false);
    const auto s1 = __builtin_amdgcn_permlane32_swap((unsigned)a[1], (unsigned)b[1], false, false);
    const i32x4 v = {(int)s0[0], (int)s1[0], (int)s0[1], (int)s1[1]};
    return __builtin_bit_cast(bf16x8, v);
  };
  // Pre-norm epilogues scale the accumulators of row m first: r_m (acc -
  // mu_m c_n) for LayerNorm, r_m acc for RMSNorm (the norm weight is folded
  // into w, c_n = sum_k of folded row n); then the base epilogue E runs.
  constexpr int E = epi_base(EPI);
  constexpr int NORM = epi_norm(EPI);
  // (A tile's column sums, and the statistics of a pass before, are all
  // loaded before any of them is used, so the epilogue waits for one round
  // trip, not one per block.)
  auto normalize_tile = [&](int m0, int n0) {
    float mu[S::FM], rs[S::FM];
#pragma unroll
    for (int j = 0; j < S::FM; ++j) {
      const int row0 = m0 + wm * S::TM + j * 32;
      if constexpr (kStatPass) {
        const int m = min(row0 + frow, a.M - 1);
        mu[j] = a.stats[2 * (int64_t)m];
        rs[j] = a.stats[2 * (int64_t)m + 1];
      } else {
        // both halves of the row's k-chunks
        const float var = (float)((sums[j].q + __shfl_xor(sums[j].q, 32, 64)) / a.K);
        mu[j] = 0.0f;
        rs[j] = 1.0f / sqrtf(var + a.eps);
      }
    }
    if constexpr (NORM == kNormLayer) {
      // acc - mu_m c_n as one more MFMA per block: A holds c_n's bf16 split
      // (hi, hi, lo) and B -mu_m's (hi, lo, hi) in k = 0..2 (lanes 0-31;
      // zeros elsewhere), so the block gains c_hi mu_hi + c_hi mu_lo +
      // c_lo mu_hi, each product exact in f32 (relative error ~2^-16 of
      // mu c, the c_lo mu_lo term).  Two values per lane instead of the
      // block's 16 column sums.
      i32x4 ca[S::FN], mb[S::FM];
#pragma unroll
      for (int i = 0; i < S::FN; ++i) {
        const float c = a.colsum[min(n0 + wn * S::TN + i * 32 + frow, a.N - 1)];
        const __bf16 hi = to_bf16(c), lo = to_bf16(c - to_f32(hi));
        bf16x8 v = {};
        if (fk == 0) v[0] = hi, v[1] = hi, v[2] = lo;
        ca[i] = __builtin_bit_cast(i32x4, v);
      }
#pragma unroll
      for (int j = 0; j < S::FM; ++j) {
        const float nm = -mu[j];
        const __bf16 hi = to_bf16(nm), lo = to_bf16(nm - to_f32(hi));
        bf16x8 v = {};
        if (fk == 0) v[0] = hi, v[1] = lo, v[2] = hi;
        mb[j] = __builtin_bit_cast(i32x4, v);
      }
#pragma unroll
      for (int i = 0; i < S::FN; ++i)
#pragma unroll
        for (int j = 0; j < S::FM; ++j) acc[i][j] = mfma32(ca[i], mb[j], acc[i][j]);
    }
#pragma unroll
    for (int i = 0; i < S::FN; ++i)
#pragma unroll
      for (int j = 0; j < S::FM; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] *= rs[j];
  };
  // DeltaNet causal conv + SiLU over the in_proj qkv columns
  // (src/archs/qwen35_text.rs:515-526,632-650; src/kernels/qwen35.cu:3-29):
  // out[r, n] = silu(sum over taps t = 3..0 of w[n, 3 - t] * p[r - t, n]),
  // p = the bf16-rounded projection, taps before the row's sequence start
  // (pos[r] < t) reading zeros; columns from conv_ch on are the plain
  // projection (z, b, a).  The taps accumulate in f32 and the SiLU uses the
  // hardware exp and reciprocal (as the SwiGLU epilogue), rounded once to
  // bf16: the reference rounds
  // every product and partial sum to bf16 instead, which costs three times
  // the VALU work in this epilogue and agrees to the projection tolerance.  The wave
  // holds all rows of the tile (WM = 1): row R = 32 j + lane % 32 of block
  // j, so row R - t is lane - t of block j, or lane + 32 - t of block j - 1.
  // One ds_bpermute per tap moves a bf16 pair: each lane offers block j's
  // value, or block j - 1's when it is among the last t lanes of its half.
  // Rows below `skip` are the tile's halo (computed, not stored).
  auto conv_epilogue = [&](int m0, int n0, int skip) {
    const int h = fk;
    int pos[S::FM];
#pragma unroll
    for (int j = 0; j < S::FM; ++j) {
      const int m = m0 + j * 32 + frow;
      pos[j] = m < a.M ? a.pos[m] : 0;
    }
#pragma unroll
    for (int i = 0; i < S::FN; ++i) {
      bf16x4 o[S::FM][4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n = n0 + wn * S::TN + i * 32 + 8 * g + 4 * h;  // features n .. n+3 (conv_ch % 4 == 0)
        float p[S::FM][4];
#pragma unroll
        for (int j = 0; j < S::FM; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) p[j][e] = round_bf16(acc[i][j][4 * g + e]);
        if (n < a.conv_ch) {
          // taps of features n .. n+3: 16 bf16, row-major [feature][tap]
          const bf16x8 w01 = *reinterpret_cast<const bf16x8*>(a.conv_w + (int64_t)n * kConvTaps);
          const bf16x8 w23 = *reinterpret_cast<const bf16x8*>(a.conv_w + (int64_t)n * kConvTaps + 8);
          float cw[4][kConvTaps];
#pragma unroll
          for (int q = 0; q < kConvTaps; ++q) {
            cw[0][q] = to_f32(w01[q]);
            cw[1][q] = to_f32(w01[4 + q]);
            cw[2][q] = to_f32(w23[q]);
            cw[3][q] = to_f32(w23[4 + q]);
          }
          // packed bf16 pairs of each block: (e0, e1), (e2, e3)
          unsigned pk[S::FM][2];
#pragma unroll
          for (int j = 0; j < S::FM; ++j)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
              bf16x4 b4;
#pragma unroll
              for (int e = 0; e < 4; ++e) b4[e] = to_bf16(p[j][e]);
              pk[j][u] = __builtin_bit_cast(i32x2, b4)[u];
            }
          float val[S::FM][4];
#pragma unroll
          for (int j = 0; j < S::FM; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) val[j][e] = 0.0f;
#pragma unroll
          for (int t = kConvTaps - 1; t >= 0; --t) {  // oldest tap first, as the reference adds them
            float x[S::FM][4];
            if (t == 0) {
#pragma unroll
              for (int j = 0; j < S::FM; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) x[j][e] = p[j][e];
            } else {
              const int src = (lane & 32) | (((lane & 31) - t) & 31);
              const bool late = (lane & 31) >= 32 - t;  // offers the previous block's row
#pragma unroll
              for (int j = 0; j < S::FM; ++j)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                  const unsigned prev = j > 0 ? pk[j > 0 ? j - 1 : 0][u] : 0u;
                  const unsigned offer = late ? prev : pk[j][u];
                  const unsigned got = (unsigned)__shfl((int)offer, src, 64);
                  const i32x2 g2 = {(int)(u == 0 ? got : 0), (int)(u == 1 ? got : 0)};
                  const bf16x4 b4 = __builtin_bit_cast(bf16x4, g2);
                  x[j][2 * u] = to_f32(b4[2 * u]);
                  x[j][2 * u + 1] = to_f32(b4[2 * u + 1]);
                }
            }
            const int tap = kConvTaps - 1 - t;
#pragma unroll
            for (int j = 0; j < S::FM; ++j) {
              const float keep = pos[j] >= t ? 1.0f : 0.0f;  // taps before the sequence start read zeros
#pragma unroll
              for (int e = 0; e < 4; ++e) val[j][e] = fmaf(x[j][e] * keep, cw[e][tap], val[j][e]);
            }
          }
#pragma unroll
          for (int j = 0; j < S::FM; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float v = val[j][e];
              o[j][g][e] = to_bf16(silu(v));
            }
        } else {
#pragma unroll
          for (int j = 0; j < S::FM; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[j][g][e] = to_bf16(p[j][e]);
        }
      }
#pragma unroll
      for (int j = 0; j < S::FM; ++j) {
        const int r = j * 32 + frow;
        const int m = m0 + r;
        const bool row_ok = m < a.M && r >= skip;
#pragma unroll
        for (int gp = 0; gp < 2; ++gp) {
          const bf16x8 v = pair16(o[j][2 * gp], o[j][2 * gp + 1]);
          const int n = n0 + wn * S::TN + i * 32 + 16 * gp + 8 * h;
          if (row_ok && n < a.Nout) store8(a.y + (int64_t)m * a.ldy + n, v, a.Nout - n);
        }
      }
    }
  };
  auto epilogue = [&](int m0, int n0, int skip) {
    if constexpr (NORM != kNormNone) normalize_tile(m0, n0);
    if constexpr (kConv) {
      conv_epilogue(m0, n0, skip);
      return;
    }
    // (opaque, so that no address formed of them is kept, or spilled, across
    // the k-loop: on the 256x160 tiles with bias and GELU it reloaded up to
    // four a k-tile, 5% of 4096 x 4999 x 3200; the gated epilogues, of few
    // addresses, spill more this way)
    int row = frow, h = fk;
    if constexpr (!epi_gated(E)) asm volatile("" : "+v"(row), "+v"(h));
    const int out_n0 = epi_gated(E) ? (n0 + wn * S::TN) / 2 : n0 + wn * S::TN;
    // Outputs, residuals and biases of calls whose rows are all 16-byte
    // aligned and within 2 GiB move by buffer instructions: a 32-bit row
    // offset per row block, the column in the instruction, rows past M
    // dropped by the descriptor's size.  The others take the element-wise
    // checks of store8 and load8, which cost a 64-bit address, an alignment
    // test and a divergent branch per 16 bytes (the vision tower's fc1 at 3001
    // rows 43.7 -> 39.8 us, 27B gate_up at 4096 tokens 1162 -> 1128, where the
    // ping-pong groups' epilogues follow each other; 256x160 plans 0-2%).
    // (At three and four waves per SIMD not for bias and residual together,
    // whose descriptors spill into the k-loop: vision fc2 on 256x160 104 ->
    // 112 us.  Nor beside the residual's LDS copy: 15 registers spill, not 4.)
    constexpr bool kVec = kWavesPerSimd <= 2 || !(E == kEpiBiasResidual || kResLds);
    const bool vec_n = kVec && a.Nout % 8 == 0;
    const bool vec_y = vec_n && a.ldy % 8 == 0 && (reinterpret_cast<uintptr_t>(a.y) & 15) == 0 &&
                       ((int64_t)a.M + BM) * a.ldy * 2 < 0x7ffffff0ll;  // (no row of a tile wraps 32 bits)
    const bool vec_r = epi_has_resid<E>() && vec_n && a.ldr % 8 == 0 &&
                       (reinterpret_cast<uintptr_t>(a.resid) & 15) == 0 &&
                       ((int64_t)a.M + BM) * a.ldr * 2 < 0x7ffffff0ll;
    const bool vec_b = epi_has_bias<E>() && vec_n && (reinterpret_cast<uintptr_t>(a.bias) & 15) == 0;
    const rsrc_t yr = make_rsrc(a.y, vec_y ? (int)((int64_t)a.M * a.ldy * 2) : 0);
    const rsrc_t rr = make_rsrc(a.resid, vec_r ? (int)((int64_t)a.M * a.ldr * 2) : 0);
    const rsrc_t br = make_rsrc(a.bias, vec_b ? a.Nout * 2 : 0);
    auto put = [&](int m, int n, bf16x8 v) {
      if (vec_y)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4, v), yr,
                                               n < a.Nout ? (int)(m * (int)a.ldy * 2 + n * 2) : (int)kOutOfRange, 0, 0);
      else if (m < a.M && n < a.Nout)
        store8(a.y + (int64_t)m * a.ldy + n, v, a.Nout - n);
    };
    auto get_resid = [&](int m, int n) -> bf16x8 {
      if (vec_r)
        return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(
            rr, n < a.Nout ? (int)(m * (int)a.ldr * 2 + n * 2) : (int)kOutOfRange, 0, 0));
      return m < a.M && n < a.Nout ? load8_bf16(a.resid + (int64_t)m * a.ldr + n, a.Nout - n) : bf16x8{};
    };
    auto get_bias = [&](int n) -> bf16x8 {
      if (vec_b) return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(br, n * 2, 0, 0));
      return n < a.Nout ? load8_bf16(a.bias + n, a.Nout - n) : bf16x8{};
    };
    // The residual of every element this lane stores, loaded before any
    // store: y may alias it (the in-place update of the hidden state), and a
    // load behind a store to a possibly aliasing address would wait a whole
    // round trip each.  A lane reads exactly the elements it then writes, so
    // reading them all first is correct in place too.
    // (Only for wave tiles of at most three 32x32 blocks, or four with two
    // waves per SIMD (256 registers): the larger ones have no registers to
    // spare for the batch and would spill.)
    constexpr bool kResRegs = epi_has_resid<E>() && !epi_gated(E) && E != kEpiRopeQkv &&
                              (S::FM * S::FN <= 3 || (S::FM * S::FN <= 4 && kWavesPerSimd <= 2));
    bf16x8 rres[kResRegs ? S::FM : 1][kResRegs ? S::FN : 1][2];
    if constexpr (kResRegs) {
      if (!(kResLds && res_in_lds)) {
#pragma unroll
        for (int j = 0; j < S::FM; ++j) {
          const int m = m0 + wm * S::TM + j * 32 + row;
#pragma unroll
          for (int i = 0; i < S::FN; ++i)
#pragma unroll
            for (int gp = 0; gp < 2; ++gp) {
              const int n = out_n0 + i * 32 + 16 * gp + 8 * h;
              rres[j][i][gp] = get_resid(m, n);
            }
        }
      }
    }
    // The bias of every column this lane stores, likewise loaded before
    // any store (the bias does not depend on the row: FN x 2 vectors).
    // (Only where the accumulators and the batched vectors take at most half
    // of a wave's registers: beyond that the batch spills.  The ping-pong
    // kernel's fragment sets are free by then: with the bias of each row
    // block read behind the last one's stores, the vision tower's fc1 at 8192
    // rows ran 132 us, batched 119.)
    constexpr bool kBiasRegs = epi_has_bias<E>() && !epi_gated(E) && E != kEpiRopeQkv &&
                               (kPP || S::FM * S::FN * 16 + S::FN * 8 + (kResRegs ? S::FM * S::FN * 8 : 0) <=
                                           512 / kWavesPerSimd / 2);
    bf16x8 rbias[kBiasRegs ? S::FN : 1][2];
    if constexpr (kBiasRegs) {
#pragma unroll
      for (int i = 0; i < S::FN; ++i)
#pragma unroll
        for (int gp = 0; gp < 2; ++gp) {
          const int n = out_n0 + i * 32 + 16 * gp + 8 * h;
          rbias[i][gp] = get_bias(n);
        }
    }
    // A block (i, j); cbias and cres are its bias and residual vectors where
    // they were read in a batch of the column blocks' rows (kPipe).
    constexpr bool kPipe = kWavesPerSimd <= 2 && !epi_gated(E) && E != kEpiRopeQkv &&
                           ((epi_has_bias<E>() && !kBiasRegs) || (epi_has_resid<E>() && !kResRegs));
    auto block = [&](int j, int i, const bf16x8* cbias, const bf16x8* cres) {
      const int m = m0 + wm * S::TM + j * 32 + row;
      const bool row_ok = m < a.M;
      if constexpr (E == kEpiRopeQkv) {
        // Blocks i (even) and i+1 are the two halves of one 64-wide head
        // (the plan guarantees 64-wide, head-aligned wave columns), so a
        // lane holds columns c and c+32 of the same token: the rotation
        // of src/kernels/modernbert.cu:31-74 happens in registers on the
        // bf16-rounded projection, rounded once, and q, k and v go to
        // their planes.
        if (i % 2 == 0) {
          const int nw = out_n0 + i * 32;  // head start column in qkv
          const int H = a.Nout / 3;
          const int p = nw / H;
          const int col = nw - p * H;
          const int pos = row_ok ? min(max(a.pos[m], 0), a.rope_rows - 1) : 0;  // stay inside the tables
          bf16x4 lo[4], hi[4];
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            float x0[4], x1[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              x0[e] = round_bf16(acc[i][j][4 * g + e]);
              x1[e] = round_bf16(acc[i + 1][j][4 * g + e]);
            }
            if (p < 2) {
              const int c = 8 * g + 4 * h;  // column within the half head
              const f32x4 cs = *reinterpret_cast<const f32x4*>(a.rope_cos + (int64_t)pos * 32 + c);
              const f32x4 sn = *reinterpret_cast<const f32x4*>(a.rope_sin + (int64_t)pos * 32 + c);
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const float r0 = x0[e] * cs[e] - x1[e] * sn[e];
                const float r1 = x0[e] * sn[e] + x1[e] * cs[e];
                x0[e] = r0;
                x1[e] = r1;
              }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              lo[g][e] = to_bf16(x0[e]);
              hi[g][e] = to_bf16(x1[e]);
            }
          }
          __bf16* dst = a.y + p * a.plane + (int64_t)m * a.ldy + col;
#pragma unroll
          for (int gp = 0; gp < 2; ++gp) {
            const bf16x8 vlo = pair16(lo[2 * gp], lo[2 * gp + 1]);
            const bf16x8 vhi = pair16(hi[2 * gp], hi[2 * gp + 1]);
            if (row_ok) {
              store8(dst + 16 * gp + 8 * h, vlo, 8);
              store8(dst + 32 + 16 * gp + 8 * h, vhi, 8);
            }
          }
        }
      } else if constexpr (epi_gated(E)) {
        // A 32-row block of the packed weight is 16 gate rows then the 16
        // up rows of the same 16 output columns: registers 4g+e (g = 0, 1)
        // hold gate rows, 4(g+2)+e the matching up rows.
        bf16x4 o[2];
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            o[g][e] = to_bf16(epi_gate<E>(acc[i][j][4 * g + e], acc[i][j][4 * (g + 2) + e]));
        const bf16x8 v = pair16(o[0], o[1]);
        put(m, out_n0 + i * 16 + 8 * h, v);
      } else {
#pragma unroll
        for (int gp = 0; gp < 2; ++gp) {
          bf16x4 p[2];
#pragma unroll
          for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) p[q][e] = to_bf16(acc[i][j][4 * (2 * gp + q) + e]);
          bf16x8 v = pair16(p[0], p[1]);
          const int n = out_n0 + i * 32 + 16 * gp + 8 * h;
          if constexpr (E != kEpiNone) {
            bf16x8 b = {}, r = {};
            if constexpr (kBiasRegs) b = rbias[i][gp];
            else if constexpr (kPipe && epi_has_bias<E>()) b = cbias[gp];
            else if constexpr (epi_has_bias<E>()) b = get_bias(n);
            if constexpr (epi_has_resid<E>()) {
              if (kResLds && res_in_lds) r = *reinterpret_cast<const bf16x8*>(res_lds + ((m - m0) * BN + (n - n0)) * 2);
              else if constexpr (kResRegs) r = rres[j][i][gp];
              else if constexpr (kPipe) r = cres[gp];
              else r = get_resid(m, n);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              float t = epi_pre<E>(to_f32(v[e]), to_f32(b[e]));
              if constexpr (epi_has_resid<E>()) t = round_bf16(t + to_f32(r[e]));
              v[e] = to_bf16(t);
            }
          }
          put(m, n, v);
        }
      }
    };
    if constexpr (!kVec) {
#pragma unroll
      for (int j = 0; j < S::FM; ++j) {
        const int m = m0 + wm * S::TM + j * 32 + row;
        const bool row_ok = m < a.M;
#pragma unroll
        for (int i = 0; i < S::FN; ++i)
#pragma unroll
          for (int gp = 0; gp < 2; ++gp) {
            bf16x4 p[2];
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
              for (int e = 0; e < 4; ++e) p[q][e] = to_bf16(acc[i][j][4 * (2 * gp + q) + e]);
            bf16x8 v = pair16(p[0], p[1]);
            const int n = out_n0 + i * 32 + 16 * gp + 8 * h;
            if (row_ok && n < a.Nout) {
              const int valid = a.Nout - n;
              float b[8] = {0, 0, 0, 0, 0, 0, 0, 0};
              if constexpr (kBiasRegs) {
#pragma unroll
                for (int e = 0; e < 8; ++e) b[e] = to_f32(rbias[i][gp][e]);
              } else if constexpr (epi_has_bias<E>()) {
                load8(a.bias + n, b, valid);
              }
              float r[8];
              if (kResLds && res_in_lds) {
                const bf16x8 rv = *reinterpret_cast<const bf16x8*>(res_lds + ((m - m0) * BN + (n - n0)) * 2);
#pragma unroll
                for (int e = 0; e < 8; ++e) r[e] = to_f32(rv[e]);
              } else if constexpr (kResRegs) {
#pragma unroll
                for (int e = 0; e < 8; ++e) r[e] = to_f32(rres[j][i][gp][e]);
              } else {
                load8(a.resid + (int64_t)m * a.ldr + n, r, valid);
              }
#pragma unroll
              for (int e = 0; e < 8; ++e) v[e] = to_bf16(round_bf16(epi_pre<E>(to_f32(v[e]), b[e]) + r[e]));
              store8(a.y + (int64_t)m * a.ldy + n, v, valid);
            }
          }
      }
    } else if constexpr (kPipe) {
      // All rows of a column block are read before its first store: one round
      // trip per column block, not one per 32x32 block (Qwen3.5-small out_proj
      // and down at 8192 tokens 124 -> 120 and 173 -> 169 us, ModernBERT-large
      // mlp.Wo there 49.8 -> 46.3).
#pragma unroll
      for (int i = 0; i < S::FN; ++i) {
        bf16x8 cbias[2] = {}, cres[S::FM][2] = {};
#pragma unroll
        for (int gp = 0; gp < 2; ++gp) {
          const int n = out_n0 + i * 32 + 16 * gp + 8 * h;
          if constexpr (epi_has_bias<E>() && !kBiasRegs) cbias[gp] = get_bias(n);
          if constexpr (epi_has_resid<E>() && !kResRegs)
            if (!(kResLds && res_in_lds))  // (block() takes it from the LDS copy)
#pragma unroll
              for (int j = 0; j < S::FM; ++j) cres[j][gp] = get_resid(m0 + wm * S::TM + j * 32 + row, n);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < S::FM; ++j) block(j, i, cbias, cres[j]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < S::FM; ++j)
#pragma unroll
        for (int i = 0; i < S::FN; ++i) block(j, i, nullptr, nullptr);
    }
  };

  // ---- stream-K partials: f32 accumulators in lane-native order, two
  // slots (head, tail) per workgroup: [wave][block i][block j][4 x f32x4][64].
  // Each XCD has its own L2 and the L2s are not coherent with each other, so
  // a device-scope fence would write back and invalidate the whole L2 (and
  // with it the cached x panel every workgroup on the XCD is using).  The
  // partials instead move with the agent-coherent cache policy (sc1: stores
  // write through, loads bypass stale L2 lines): the writer waits for its
  // stores to be acknowledged before a relaxed agent-scope counter
  // increment, and the last arriving workgroup reads them back coherently.
  constexpr int kWaveF4 = S::FN * S::FM * 4 * 64;     // f32x4 per wave per slot
  constexpr int kTileF4 = S::kWaves * kWaveF4;        // f32x4 per slot
  constexpr int kCoherent = 16;                       // cache policy: sc1
  const rsrc_t wsr = make_rsrc(a.ws);
  auto slot_off = [&](int g, int slot) -> unsigned {  // byte offset of this lane's first f32x4
    return (unsigned)((((int64_t)g * 2 + slot) * kTileF4 + wave * kWaveF4 + lane) * 16);
  };
  // The row sums of a fused pre-norm go the same way, to a.stats:
  // [workgroup][slot][wave][block j][64 lanes].
  const rsrc_t ssr = make_rsrc(a.stats);
  auto sums_off = [&](int g, int slot) -> unsigned {
    return (unsigned)(((((int64_t)g * 2 + slot) * S::kWaves + wave) * S::FM * 64 + lane) * 8);
  };
  // A partial segment: write this workgroup's partial; returns true when it
  // is the tile's last segment to arrive, with acc then holding the full sum
  // (the caller runs the epilogue).
  auto finish_partial = [&](const Segment& sg) -> bool {
    const int t = sg.st;
    const int slot = sg.spos == walk.begin ? 0 : 1;
    const unsigned mine = slot_off(blockIdx.x, slot);
    // (sched_barrier keeps the scheduler from hoisting the whole partial's
    // memory traffic together: that would raise the register peak of the
    // kernel, and with it cost occupancy in the main loop.)
#pragma unroll
    for (int i = 0; i < S::FN; ++i)
#pragma unroll
      for (int j = 0; j < S::FM; ++j) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x4 v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                           acc[i][j][4 * q + 3]};
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(i32x4, v), wsr,
                                                 (int)(mine + ((i * S::FM + j) * 4 + q) * 64 * 16), 0,
                                                 kCoherent);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    if constexpr (kOwnNorm != kNormNone) {
#pragma unroll
      for (int j = 0; j < S::FM; ++j)
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(i32x2, sums[j].q), ssr,
                                              (int)(sums_off(blockIdx.x, slot) + j * 64 * 8), 0, kCoherent);
    }
    int g_lo, g_hi;
    walk.tile_owners(t, g_lo, g_hi);
    // Each wave arrives on its own counter (tile, wave): its slice of the
    // tile (its accumulators, its epilogue) is independent of the other
    // waves', so the last owner of each slice sums and stores that slice
    // alone -- no barrier and no LDS.  Waves of one workgroup may disagree
    // about being last; every slice still has exactly one last owner.
    unsigned* counter = a.counters + (int64_t)t * S::kWaves + wave;
    __builtin_amdgcn_s_waitcnt(0);  // this wave's partial stores are acknowledged
    unsigned prev = 0;
    if (lane == 0) prev = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    prev = __builtin_amdgcn_readfirstlane(prev);
    if (prev != (unsigned)(g_hi - g_lo)) return false;
    zero_acc();
    const int64_t tile_lo = (int64_t)t * walk.kt_count;
    for (int g = g_lo; g <= g_hi; ++g) {
      // g's segment in this tile is its head iff g's range starts inside the tile.
      const int gslot = walk.start(g) >= tile_lo ? 0 : 1;
      const unsigned src = slot_off(g, gslot);
      if constexpr (kOwnNorm != kNormNone) {
#pragma unroll
        for (int j = 0; j < S::FM; ++j)
          sums[j].q += __builtin_bit_cast(
              double, __builtin_amdgcn_raw_buffer_load_b64(ssr, (int)(sums_off(g, gslot) + j * 64 * 8), 0, kCoherent));
      }
      // All of one owner's loads are in flight together (these coherent
      // reads come from beyond the L2: one round trip per owner, not one
      // per block), then added in the same order as always.
      f32x4 v[S::FN][S::FM][4];
#pragma unroll
      for (int i = 0; i < S::FN; ++i)
#pragma unroll
        for (int j = 0; j < S::FM; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            v[i][j][q] = __builtin_bit_cast(
                f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                           wsr, (int)(src + ((i * S::FM + j) * 4 + q) * 64 * 16), 0, kCoherent));
#pragma unroll
      for (int i = 0; i < S::FN; ++i)
#pragma unroll
        for (int j = 0; j < S::FM; ++j)
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][j][4 * q + e] += v[i][j][q][e];
      __builtin_amdgcn_sched_barrier(0);
    }
    if (lane == 0) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
  };

  // ---- ping-pong main loop (PW < 0), for large tiles and long streams.
  //
  // Two groups of four waves (one per SIMD each) run half a phase apart: in
  // one barrier interval a wave reads the fragments of its next quadrant and
  // issues its share of a refill, in the next it runs the quadrant's MFMAs
  // (8 of 32 cycles at 256x256) while the SIMD's other wave loads.  A load
  // that stalls its wave's issue then never stands in front of that wave's
  // MFMAs, without producer waves and the third of the registers they hold.
  //
  // LDS is a ring of SLOTS slots of 16 KB.  A phase reads one unit (half of
  // one operand's rows of a k-tile) and requests the unit kAhead phases on
  // into the slot that the last phase freed: each operand byte is read from
  // LDS once per wave, its slot is free a quarter of a k-tile later, and 2 1/4
  // k-tiles are on their way at any time, against one in the two-stage
  // 256x256 kernel that this replaces (its barrier waited for loads issued
  // one k-tile before).
  //
  // Hazards.  A unit's readers wait for their reads (lgkmcnt(0)) before the
  // barrier that ends their load interval; the first request into its slot
  // is issued after the later group's.  A unit's requests have landed before
  // it is read: each wave waits for its own share (vmcnt) one phase earlier,
  // in front of a barrier that both groups pass before the first read.
  //
  // Measured, 8192 x 8192 x 8192: 1200 -> 1340-1397 TFLOP/s against the
  // two-stage kernel, same boxes; 2010 with operands of zeros, so the rest is
  // what the card's power allows for the data.
  // Without its refills the loop reaches 2150, without its LDS reads 1730.
  // Slower: the refills issued between the MFMAs (1163), before the fragment
  // reads (1258), or half of each unit later (1220-1306); eight slots instead
  // of ten lose up to 1%; the raster group (2 to 8 tile rows) changes nothing.
  if constexpr (kPP) {
    static_assert(WM == 2 && WN == 4 && BK == 64 && OCC == 1 && !STREAMK && !kConv, "ping-pong: 2 x 4 waves");
    static_assert(S::FM % 2 == 0 && S::FN % 2 == 0, "ping-pong: wave tiles in quadrants");
    constexpr int SLOTS = STAGES_;
    constexpr int HM = S::FM / 2, HN = S::FN / 2;            // blocks of half a wave tile
    constexpr int kXI = BM / 2 / S::RPI / S::kWaves;         // refill instructions per wave: half of x
    constexpr int kWI = BN / 2 / S::RPI / S::kWaves;         // half of w
    static_assert(kXI == kWI, "every unit is the same number of refill instructions");
    static_assert(kXI * S::RPI * S::kWaves * 2 == BM && kWI * S::RPI * S::kWaves * 2 == BN, "refills deal evenly");
    constexpr int kAhead = SLOTS - 1;                        // units requested ahead of the one read
    // Unit u of the stream is half of one operand's rows of a k-tile, in the
    // order x0, w0, w1, x1; the half h of x holds every wave row's blocks
    // [h HM, (h + 1) HM), of w every wave column's [h HN, (h + 1) HN).
    auto unit_row = [&](bool is_w, int h, int r) {  // unit row -> tile row
      constexpr int hx = S::TM / 2, hw = S::TN / 2;
      return is_w ? r / hw * S::TN + h * hw + r % hw : r / hx * S::TM + h * hx + r % hx;
    };
    unsigned soff[2 * (kXI + kWI)];
    auto pp_offsets = [&](const Segment& sg) {
      const int x_left = a.M - 1 - walk.row0(sg.tm), w_left = a.N - 1 - sg.tn * BN;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < kXI; ++i) {
          const int r = (i * S::kWaves + wave) * S::RPI + lrow;
          soff[h * kXI + i] = (unsigned)(min(unit_row(false, h, r), x_left) * (int)a.ldx * 2 + ((lpos ^ lds_swz<BK>(r)) << 4));
        }
#pragma unroll
        for (int i = 0; i < kWI; ++i) {
          const int r = (i * S::kWaves + wave) * S::RPI + lrow, c = (lpos ^ lds_swz<BK>(r)) << 4;
          const int rw = min(unit_row(true, h, r), w_left);
          soff[2 * kXI + h * kWI + i] =
              a.w_kt ? (unsigned)((rw / kBlkRows) * a.w_kt * kBlkBytes + (rw % kBlkRows) * (kBlkK * 2) + c)
                     : (unsigned)(rw * (int)a.ldw * 2 + c);
        }
      }
    };
    const int steps = walk.steps();
    // The request cursor: the descriptors of its k-tile, moved on by a
    // scalar add per k-tile (in the shadow of a quadrant's MFMAs, not in
    // front of a request).  Past the end of the stream a size of zero keeps
    // the instruction count.
    Segment qsg = walk.first_segment();
    int qkt = qsg.kt0, qstep = 0;
    const char *qx, *qw;
    const int wstep = a.w_kt ? kBlkBytes : BK * 2;
    auto enter_segment = [&]() {
      const int n0 = qsg.tn * BN;
      pp_offsets(qsg);
      qx = reinterpret_cast<const char*>(a.x + (int64_t)walk.row0(qsg.tm) * a.ldx) + qsg.kt0 * BK * 2;
      qw = a.w_kt ? reinterpret_cast<const char*>(a.w) + (int64_t)(n0 / kBlkRows) * a.w_kt * kBlkBytes
                  : reinterpret_cast<const char*>(a.w + (int64_t)n0 * a.ldw);
      qw += (int64_t)qsg.kt0 * wstep;
    };
    enter_segment();
    int qbytes = 0x7ffffff0;
    const int ktail = a.K % BK;  // valid k of a partial last k-tile
    bool qtail = ktail && qsg.kt0 == walk.kt_count - 1;
    // Request the cursor's unit of type T into `slot`.
    auto request = [&](auto tc, int slot) {
      constexpr int T = decltype(tc)::value;
      constexpr bool is_w = T == 1 || T == 2;
      constexpr int h = T >= 2 ? 1 : 0;
      const rsrc_t r = make_rsrc_uniform(is_w ? qw : qx, qbytes);
      unsigned off[kXI];
#pragma unroll
      for (int i = 0; i < kXI; ++i) off[i] = soff[is_w ? 2 * kXI + h * kWI + i : h * kXI + i];
      if (qtail) {  // (wave-uniform) chunks past K read zeros
#pragma unroll
        for (int i = 0; i < kXI; ++i)
          if ((lpos ^ lds_swz<BK>((i * S::kWaves + wave) * S::RPI + lrow)) * 8 >= ktail) off[i] = kOutOfRange;
      }
#pragma unroll
      for (int i = 0; i < kXI; ++i)
        dma16(r, off[i], (lds_void*)(lds + slot * kSlotBytes + (i * S::kWaves + wave) * 1024));
    };
    auto advance = [&](auto tc) {  // behind the request of type T
      if constexpr (decltype(tc)::value == 3) {
        qx += BK * 2;
        qw += wstep;
        if (++qstep >= steps) {
          qbytes = 0;
        } else if (++qkt == qsg.kt1) {
          qsg = walk.next_segment(qsg);
          qkt = qsg.kt0;
          enter_segment();
        }
        qtail = ktail && qkt == walk.kt_count - 1;
      }
    };
    constexpr int kInFlight = kXI * (kAhead - 1);  // refill instructions that may be outstanding at a barrier
    static_assert(kInFlight < 64, "vmcnt field");

    // Fragments: chunk 2 ks + fk of unit row r at ((fk ^ swz) << 4) ^ (ks << 5).
    i32x4 xf[2][HM][S::KS], wf[2][HN][S::KS];
    const int xr0 = wm * (S::TM / 2) + frow, wr0 = wn * (S::TN / 2) + frow;
    const int xb = xr0 * S::kRowBytes + ((fk ^ lds_swz<BK>(xr0)) << 4);
    const int wb = wr0 * S::kRowBytes + ((fk ^ lds_swz<BK>(wr0)) << 4);
    // (32 rows further on, lds_swz flips its bit 2: the chunk of k-step ks ^ 2)
    auto read_x = [&](int h, int slot) {
      const int b = xb + slot * kSlotBytes;
#pragma unroll
      for (int j = 0; j < HM; ++j)
#pragma unroll
        for (int ks = 0; ks < S::KS; ++ks)
          xf[h][j][ks] = *reinterpret_cast<const i32x4*>(lds + (b ^ ((ks ^ (j % 2 * 2)) << 5)) + j * 32 * S::kRowBytes);
    };
    auto read_w = [&](int h, int slot) {
      const int b = wb + slot * kSlotBytes;
#pragma unroll
      for (int i = 0; i < HN; ++i)
#pragma unroll
        for (int ks = 0; ks < S::KS; ++ks)
          wf[h][i][ks] = *reinterpret_cast<const i32x4*>(lds + (b ^ ((ks ^ (i % 2 * 2)) << 5)) + i * 32 * S::kRowBytes);
    };
    auto quadrant = [&](int hx, int hw) {
#pragma unroll
      for (int ks = 0; ks < S::KS; ++ks)
#pragma unroll
        for (int i = 0; i < HN; ++i)
#pragma unroll
          for (int j = 0; j < HM; ++j)
            acc[hw * HN + i][hx * HM + j] = mfma32(wf[hw][i][ks], xf[hx][j][ks], acc[hw * HN + i][hx * HM + j]);
    };
    auto bar = [&]() {
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    };
    int slot = 0, freed = SLOTS - 1;
    auto next_slot = [&]() {
      freed = slot;
      slot = slot + 1 == SLOTS ? 0 : slot + 1;
    };
    const bool second = wave >= S::kWaves / 2;  // the group half a phase behind
    // One phase of unit type T: its fragments, a request into the slot the
    // last phase freed, the wait for the next phase's unit; the barrier; the
    // quadrant that the fragments complete; the barrier.  (Not the second
    // group's last one, which would have the first group's last epilogue in
    // front of its own; each group then passes as many.)
    auto phase = [&](auto tc, bool load, bool mul) {
      constexpr int T = decltype(tc)::value;
      if (load) {
        if constexpr (T == 0) read_x(0, slot);
        if constexpr (T == 1) read_w(0, slot);
        if constexpr (T == 2) read_w(1, slot);
        if constexpr (T == 3) read_x(1, slot);
        __builtin_amdgcn_sched_barrier(0);
        request(std::integral_constant<int, (T + kAhead) % 4>(), freed);
        __builtin_amdgcn_sched_barrier(0);
        next_slot();
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the slot just read may be refilled after the barrier
        vm_wait<kInFlight>();
      }
      bar();
      __builtin_amdgcn_s_setprio(1);
      if (mul) {
        if constexpr (T == 0) quadrant(1, 0);
        if constexpr (T == 1) quadrant(0, 0);
        if constexpr (T == 2) quadrant(0, 1);
        if constexpr (T == 3) quadrant(1, 1);
      }
      if (load) advance(std::integral_constant<int, (T + kAhead) % 4>());
      __builtin_amdgcn_s_setprio(0);
      if (load || !second) bar();
    };
    using std::integral_constant;
    // Prologue: the first kAhead units, the first of them landed.
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
      if (u % 4 == 0) request(integral_constant<int, 0>(), u);
      if (u % 4 == 1) request(integral_constant<int, 1>(), u);
      if (u % 4 == 2) request(integral_constant<int, 2>(), u);
      if (u % 4 == 3) request(integral_constant<int, 3>(), u);
      if (u % 4 == 3) advance(integral_constant<int, 3>());
    }
    vm_wait<kInFlight>();
    bar();
    if (second) bar();
    Segment csg = walk.first_segment();
    int ckt = csg.kt0;
    for (int s = 0; s < steps; ++s) {
      phase(integral_constant<int, 0>(), true, s > 0);
      if (s > 0 && ++ckt == csg.kt1) {
        epilogue(walk.row0(csg.tm), csg.tn * BN, 0);
        zero_acc();
        csg = walk.next_segment(csg);
        ckt = csg.kt0;
      }
      phase(integral_constant<int, 1>(), true, true);
      phase(integral_constant<int, 2>(), true, true);
      phase(integral_constant<int, 3>(), true, true);
    }
    phase(integral_constant<int, 0>(), false, true);
    epilogue(walk.row0(csg.tm), csg.tn * BN, 0);
    vm_wait<0>();  // the zero-size refills of the last units write LDS too
    return;
  }

  // ---- main loop over this workgroup's k-tile stream.  Step s lives in
  // stage s % STAGES.  The prologue requests steps 0..STAGES-1; after the
  // barrier that retires step s, step s + STAGES is requested into the stage
  // just freed -- across item boundaries, so the next item's first k-tiles
  // land while this item finishes and stores.  Before that barrier step s+1
  // must have landed while s+2 .. s+STAGES-1 may still be in flight:
  // vmcnt((STAGES-2) * DMAs per step).  sched_barrier(0) pins the order
  // below: the next k-step's fragment reads are issued before the current
  // k-step's MFMAs, so LDS latency hides behind a full k-step of matrix work.
  const int steps = walk.steps();
  constexpr bool kIssue = PW == 0;  // this wave issues refills
  if constexpr (kIssue) {
    for (int t = 0; t < STAGES; ++t)
      if (t < steps) issue(t);
    if (steps >= STAGES) vm_wait<(STAGES - 1) * kDma>();
    else vm_wait<0>();
  }
  __syncthreads();

  Segment csg = walk.first_segment();  // compute cursor
  int ckt = csg.kt0;
  // Schedules of a k-tile's KS k-steps of MFMAs (fragment reads one k-step
  // ahead of their MFMAs):
  //   kDeep (one fragment set per k-step, when they fit in registers): the
  //     barrier that frees the stage comes after the k-tile's last two
  //     fragment sets are in registers, so two k-steps of MFMAs run after it,
  //     covering the next stage's first fragment reads, with the freed
  //     stage's refill issued between them;
  //   otherwise (ping-pong sets): one k-step of MFMAs after the barrier.
  constexpr int kSets = kDeep ? 4 : 2;
  Frags fr[kSets];
  if (steps > 0) {
    read(fr[0], 0, 0);
    if constexpr (kDeep) read(fr[1], 0, 1);
  }
  // A tile's end is followed by the loop's first instruction; it is put on a
  // 128-byte line, wherever the code in front of it ends (the accumulators
  // are operands so that nothing else comes between).  Left to chance, a
  // change of the epilogue moved it to where the 128x192 tiles' loop, the
  // same instructions, ran 5% slower: 1024 x 3072 x 1024 14.9 us, now 14.1,
  // 1024 x 5120 x 17408 with a residual 179 -> 171.  (Not for RoPE, which
  // spills more with it.)
  auto align_loop = [&]() {
    if constexpr (E != kEpiRopeQkv) {
#pragma unroll
      for (int i = 0; i < S::FN; ++i)
#pragma unroll
        for (int j = 0; j < S::FM; ++j) asm volatile("" : "+v"(acc[i][j]));
      asm volatile(".p2align 7");
    }
  };
  int stage = 0;
  for (int s = 0; s < steps; ++s) {
    if constexpr (kDeep) {
      // fr[0] (and fr[1], one set later) of this k-tile were read after the
      // previous barrier.  Waiting for them explicitly keeps the compiler
      // from resolving its merged loop-header state with a full LDS wait
      // after the next reads.
      __builtin_amdgcn_s_waitcnt(0xc07f | (kReads << 8));  // lgkmcnt(kReads): fr[0] is in
      __builtin_amdgcn_sched_barrier(0);
      read(fr[2], stage, 2);
      __builtin_amdgcn_sched_barrier(0);
      mma(fr[0]);
      __builtin_amdgcn_sched_barrier(0);
      read(fr[3], stage, 3);
      __builtin_amdgcn_sched_barrier(0);
      mma(fr[1]);
      __builtin_amdgcn_sched_barrier(0);
    } else {
      // As above: the k-tile's first fragments are in.
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0), vmcnt/expcnt unconstrained
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 1; ks < S::KS; ++ks) {
        read(fr[ks % 2], stage, ks);
        __builtin_amdgcn_sched_barrier(0);
        mma(fr[(ks - 1) % 2]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (kIssue && s + 1 < steps) {
      if (s + STAGES - 1 < steps) vm_wait<(STAGES - 2) * kDma>();
      else vm_wait<0>();
    }
    __syncthreads();
    // Next k-tile's first fragments, this k-tile's last MFMAs, then the
    // refill of the stage just freed: the refill's load instructions can
    // stall issue while the load path drains, and issued behind the MFMAs
    // that stall overlaps matrix work instead of delaying it.
    const int freed = stage;
    stage = stage + 1 == STAGES ? 0 : stage + 1;
    // One workgroup per CU (OCC == 1): the refill's instructions go between
    // the MFMAs that follow the barrier.  With two workgroups per CU the
    // other workgroup's MFMAs cover the refill, and one burst after the
    // first MFMA group measured faster.
    using std::integral_constant;
    constexpr bool kSpread = OCC == 1 && kIssue;
    const Refill r = refill_at(freed, s + STAGES < steps);
    auto refill_all = [&]() {
#pragma unroll
      for (int i = 0; i < kDma; ++i) if constexpr (kIssue) dma_one(r, i);
    };
    if constexpr (kDeep && kSpread) {
      constexpr int kHalf = kDma / 2;
      if (s + 1 < steps) {
        read(fr[0], stage, 0);
        read(fr[1], stage, 1);
      }
      __builtin_amdgcn_sched_barrier(0);
      mma_dma(fr[2], r, integral_constant<int, 0>(), integral_constant<int, kHalf>());
      mma_dma(fr[3], r, integral_constant<int, kHalf>(), integral_constant<int, kDma - kHalf>());
    } else if constexpr (kDeep) {
      if (s + 1 < steps) read(fr[0], stage, 0);
      __builtin_amdgcn_sched_barrier(0);
      mma(fr[2]);
      __builtin_amdgcn_sched_barrier(0);
      refill_all();
      __builtin_amdgcn_sched_barrier(0);
      if (s + 1 < steps) read(fr[1], stage, 1);
      __builtin_amdgcn_sched_barrier(0);
      mma(fr[3]);
    } else if constexpr (kSpread) {
      if (s + 1 < steps) read(fr[0], stage, 0);
      __builtin_amdgcn_sched_barrier(0);
      mma_dma(fr[(S::KS - 1) % 2], r, integral_constant<int, 0>(), integral_constant<int, kDma>());
    } else {
      if (s + 1 < steps) read(fr[0], stage, 0);
      __builtin_amdgcn_sched_barrier(0);
      mma(fr[(S::KS - 1) % 2]);
      __builtin_amdgcn_sched_barrier(0);
      refill_all();
    }
    if (kIssue && s + STAGES < steps) issue_advance();
    __builtin_amdgcn_sched_barrier(0);
    if (++ckt == csg.kt1) {
      if constexpr (STREAMK) {
        if (walk.complete(csg) || finish_partial(csg))
          epilogue(walk.row0(csg.tm), csg.tn * BN, csg.tm ? kConvHalo : 0);
      } else {
        epilogue(walk.row0(csg.tm), csg.tn * BN, csg.tm ? kConvHalo : 0);
      }
      zero_acc();
      if (s + 1 < steps) {
        csg = walk.next_segment(csg);
        ckt = csg.kt0;
      }
      align_loop();
    }
  }
  vm_wait<0>();  // the zero-size refills of the last k-tiles write LDS too
}

}  // namespace sys1
