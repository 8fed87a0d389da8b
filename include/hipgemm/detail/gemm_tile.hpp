// hipgemm -- FP8 GEMM on tiles between 128 x 128 and 256 x 256 (gfx950).
//
// C[M x N] = scale_a * scale_b * A[M x K] . B_T[N x K]^T, the same contract
// and the same GemmArgs as the 4-wave schedule (gemm_4wave.hpp).  Where the
// 256 x 256 tiles of that schedule fill half the CUs or leave a short last
// round, and the 128 x 128 ones (gemm_t128.hpp) need two rounds, a tile in
// between fills the CUs in one.  No reference counterpart:
// fp8_4wave.hpp:334-567 has 256 x 256 tiles only.
//
// Work decomposition: one workgroup = 4 waves (one per SIMD), persistent over
// the tiles (tile_walk / grouped_tile, layout.hpp).  Wave w owns the BM / 2 x
// BN / 2 part (w / 2, w % 2) of a tile as FA x FB blocks of 16 x 16
// (v_mfma_f32_16x16x128_f8f6f4, FA * FB per 128-byte K-step).
//
// What bounds it: per step a CU moves (BM + BN) * 128 bytes L2 -> LDS (a
// DMA-only loop of these tiles reaches 100 GB/s per CU), writes and reads
// them in LDS (BM + BN rows in, 2 (BM + BN) out) and issues FA * FB MFMA of
// 32 cycles per wave; on 128 x 128 these take 0.33, 0.35 and 0.23 us, a step
// 0.39 us.  With one select and one address computation per DMA and per
// read in the loop, and the wave's scalar work after the barrier, a step was
// 0.47 us (one set of operands: 2048 x 2048 x 8192 34.2 -> 29.9 us, 1536 x 4096 x
// 4096 33.0 -> 28.9, 1024^3 7.45 -> 7.10, MXFP4 2048 x 2048 x 8192 25.0 -> 22.9,
// with row and column scales, bias and silu 2048 x 2048 x 4096 23.0 -> 19.2;
// operands from memory: the first two 39.0 -> 36.8 and 35.0 -> 31.8): the steady
// loop now has four address additions per step and nothing else.
//
// Pipeline: S LDS stages of BM + BN rows x 128 bytes, DMA'd (buffer_load_dwordx4
// ... lds) S steps ahead of the reads, and two register sets: the fragments
// of step k + 1 are read while the MFMA of step k run, so that a stage is
// free for the DMA of step k + S as soon as step k starts.  Step k:
//   wait for the wave's own LDS reads of step k (done during step k - 1) and
//   its own DMA of step k + 1; barrier; the last MFMA of step k - 1 (they
//   read registers only, and keep the matrix unit busy while the waves
//   meet); then the MFMA of step k, each followed by one LDS read of step
//   k + 1 and, evenly spread, the DMA of step k + S into step k's stage.
// The step sequence runs on across tiles: the DMA and the reads past a tile's
// last step are the next tile's first steps.  Steps per tile are padded to an
// even count >= S (padding steps read zeros).
//
// DMA that fetch whole steps of the tile take the lanes' offsets as they are;
// the others (the step K ends inside, padding, the next tile's steps) go
// through a per-lane select, in a copy of the step of their own.
//
// K order: the workgroups of XCD x (blockIdx % 8) start a unit's whole steps
// at step x * whole / 8 of them and wrap around; a step that the unit's K range
// ends inside comes last (no start but 0 with MX scales, whose scale words
// follow the plain order).  Started together at step 0, every workgroup's DMA
// of a step falls at the same offset of each operand row, and with row strides
// that are a multiple of 4096 bytes all those rows meet at one offset within
// 4 KiB -- which measured as an HBM-bound stall; one start per XCD keeps the
// workgroups of an XCD (which share operand panels in their L2) in step.  Same
// process, 128 x 128 tiles, against starting at step 0: 40 x 28672 x 4096 +19 %,
// 16 x 28672 x 4096 +24 %, 64 x 16384 x 8192 +29 %, 4096 x 1536 x 4096 +5 %, 512 x
// 4096 x 8192 and 2048 x 2048 x 8192 within 1 %; K-slices that are not all whole
// steps 407 x 3072 x 11648 +9 %, 1006 x 3072 x 5824 +7 %.  The fp32 sums run in
// that rotated order (deterministic per launch shape).
//
// LDS layout: 128-byte rows with the slot_xor swizzle, lane group g reading
// slots 2g and 2g + 1 before the XOR (layout.hpp: conflict-free; A and B_T
// share the K order).  kMx needs the instruction's own K order: chunks g and
// g + 4 under strip_xor, conflict-free too.
//
// kSplit (128 x 128 and 64-column tiles): work units are (tile, K-slice) pairs
// (g.split); each writes its fp32 partial tile (written through to the coherent
// level, sc1: the slices of a tile run on several XCDs, whose L2s are not coherent
// with each other).  With g.split.arrivals, each wave then waits for its own
// partial stores, counts its quadrant's arrival (a relaxed agent-scope atomic),
// and the wave that arrives last at a quadrant sums the quadrant's partials in
// slice order (its own from its accumulators, the others read back with sc1) and
// runs the epilogue on the sum: no waiting on other workgroups and no barrier, so
// waves of one workgroup may take different paths here.  Without it,
// gemm_t128_reduce_body sums them in a kernel of its own; both add +0 + slice 0 +
// slice 1 + ... in fp32, so their outputs are the same.
//
// kNt: B_T's DMA carry the non-temporal hint, for one row of tiles, where each
// B_T line is read by one workgroup (64 x 14336 x 4096 on 64 x 64 tiles 14.9 ->
// 13.8 us, 128 x 14336 x 4096 18.5 -> 17.7; with K-slices level to 10 %
// slower), in one step: with rows that do not start on 128-byte lines each line
// belongs to two steps, and the hint cost 8 % at the median of 167 such shapes
// (30 % at most).
//
// kMx: MX block scales from g.mx (the packed layout of MxArgs; per-tensor
// epilogue).  Each step also loads, two steps ahead, each operand's 16 scale
// bytes of the lane into registers (one buffer load per operand).
//
// Epilogue: acc * scale (or the extended epilogue, kExt), 16 rows of C at a
// time through the wave's own LDS stage, then 16-byte stores, consecutive
// lanes along a row; without 16-byte alignment (kVec false), 2-byte stores
// straight from the registers.  fp32 and e4m3 outputs go straight from the
// accumulators.  Lanes outside M x N get out-of-range offsets.
#pragma once

#include <type_traits>

#include "arch.hpp"
#include "epilogue.hpp"
#include "gemm_4wave.hpp"
#include "layout.hpp"

namespace hipgemm {
namespace detail {

template <int BM, int BN, int S>
struct CfgTile {
  static constexpr int kThreads = 256;
  static constexpr int kBM = BM, kBN = BN, kBK = 128;
  static constexpr int kStages = S;
  static constexpr int kWM = BM / 2, kWN = BN / 2;      // a wave's part
  static constexpr int kFA = kWM / 16, kFB = kWN / 16;  // 16-row fragments
  static constexpr int kAStage = kBM * kBK;
  static constexpr int kStage = kAStage + kBN * kBK;
  // Staging per wave: 16 rows of C, or kExt's vectors (1.5 KiB).
  static constexpr int kRows16 = 16 * kWN * 2;
  static constexpr int kStoreStage = kRows16 > 1536 ? kRows16 : 1536;
  static constexpr int kStoreBase = kStages * kStage;
  static constexpr int kPartial = BM * BN * 4;  // a K-slice's fp32 tile
  static constexpr int kLdsBytes = kStoreBase + 4 * kStoreStage;
  static constexpr int kDmaA = BM / 32, kDmaB = BN / 32;  // per wave per step
  static constexpr int kDma = kDmaA + kDmaB;
  static_assert(kLdsBytes <= 160 * 1024, "LDS");
};

template <class Cfg, bool kVec, bool kExt = false, int kFmt = 0,
          int kAct = kActNone, int kOut = kOutBf16, bool kSplit = false,
          bool kMx = false, bool kNt = false>
__device__ __forceinline__ void gemm_tile_body(const GemmArgs& g, lds_u8* lds) {
  constexpr int S = Cfg::kStages, FA = Cfg::kFA, FB = Cfg::kFB;
  constexpr int kDma = Cfg::kDma;           // DMA per wave per step
  constexpr int kD = kDma + (kMx ? 2 : 0);  // memory operations per step
  constexpr bool k4 = is_fp4(kFmt), k6 = is_fp6(kFmt);
  // fp6 operands: a step is 128 elements, 96 bytes of a row, held in LDS
  // slots 0-5 of the 128-byte row (slots 6 and 7 stay unfetched).
  constexpr int kStepBytes = k6 ? 96 : Cfg::kBK;
  // LDS reads per fragment: two 16-byte halves, fp6 three 8-byte pieces.
  constexpr int kPieces = k6 ? 3 : 2;
  constexpr int kReads = kPieces * (FA + FB);
  // MFMA of a step issued after the next step's barrier (none, one and two
  // measured within 1 %; none where every MFMA is needed to carry its reads).
  constexpr int kMfma = FA * FB;
  constexpr int kTail = kReads <= 2 * (kMfma - 1) ? 1 : 0, kHead = kMfma - kTail;
  // Reads go one per MFMA, two for the first kReads - kHead of them.
  constexpr int kTwo = kReads > kHead ? kReads - kHead : 0;
  static_assert(kReads <= 2 * kHead && kDma <= kHead, "one DMA per MFMA");
  static_assert(!kMx || (!kExt && !k6), "MX: per-tensor epilogue, 8-bit and fp4");
  static_assert(!kMx || (Cfg::kBM == 128 && Cfg::kBN == 128),
                "MX: 128 x 128 tiles");
  // Stores of C per wave per tile (16-byte path), or of a partial or of wide
  // outputs (one per block straight from the accumulators).
  constexpr int kStores = kSplit || (kExt && kOut >= kOutF32)
                              ? FA * FB
                              : FA * (Cfg::kRows16 / 1024);
  static_assert((S - 2) * kD + kStores < 64, "vmcnt range");
  const int lane = lane_id();
  const int wave = wave_id();
  const int wm = wave >> 1, wn = wave & 1;
  const int M = g.M, N = g.N, K = g.K;
  const int tiles_m = (M + Cfg::kBM - 1) / Cfg::kBM;
  const int tiles_n = (N + Cfg::kBN - 1) / Cfg::kBN;
  const int tiles = tiles_m * tiles_n;
  const int units = kSplit ? tiles * g.split.slices : tiles;
  const int steps = kSplit ? g.split.slice_steps : (K + kStepBytes - 1) / kStepBytes;
  const int steps_pad = max((S + 1) & ~1, (steps + 1) & ~1);
  const int workers = g.workers > 0 ? min((int)gridDim.x, g.workers)
                                    : (int)gridDim.x;
  if ((int)blockIdx.x >= workers) return;
  // Work unit u: tile u % tiles, K-slice u / tiles (one slice unless kSplit),
  // so that units running together share A rows or B columns.
  const TileWalk walk = tile_walk(blockIdx.x, workers, units);
  int t = walk.first;
  if (t >= walk.end) return;

  const float sa = g.scale_a ? *g.scale_a : 1.0f;
  const float sb = g.scale_b ? *g.scale_b : 1.0f;
  const float scale = sa * sb;

  // ---- DMA lane geometry: instruction q of wave w covers rows (4q + w) * 8
  // .. + 8 of A (or B_T); lane l takes row + l / 8, 16-byte slot l % 8, which
  // holds K-chunk (l % 8) ^ slot_xor(row). ----------------------------------
  const int drow = lane >> 3;
  const int dchunk =
      (lane & 7) ^ (kMx ? strip_xor(drow) : slot_xor(8 * (wave & 1) + drow));
  // fp6: the lanes of slots 6 and 7 always read zero.
  const uint32_t pad6 = k6 && dchunk >= 6 ? kOobOffset : 0u;
  uint32_t voff_a[Cfg::kDmaA], voff_b[Cfg::kDmaB];
#pragma unroll
  for (int q = 0; q < Cfg::kDmaA; ++q)
    voff_a[q] = ((uint32_t)((4 * q + wave) * 8 + drow) * (uint32_t)g.lda + dchunk * 16) | pad6;
#pragma unroll
  for (int q = 0; q < Cfg::kDmaB; ++q)
    voff_b[q] = ((uint32_t)((4 * q + wave) * 8 + drow) * (uint32_t)g.ldb + dchunk * 16) | pad6;

  // Buffer resources of a unit's A rows and B_T rows (rows past M / N read
  // zero; none past the walk's end), its K range [k0, kend), the whole steps
  // of it, and the one it starts at (K order, above).
  struct Src {
    __amdgpu_buffer_rsrc_t a, b;
    int k0, kend, full, rot;
    int tm, tn;  // tile coordinates (kMx); tm = -1: no unit
  };
  auto src_of = [&](int unit) {
    if (unit >= walk.end)
      return Src{make_rsrc(g.A, 0u), make_rsrc(g.B, 0u), 0, 0, 0, 0, -1, 0};
    const int tile = kSplit ? unit % tiles : unit;
    const int slice = kSplit ? unit / tiles : 0;
    const TileCoord c = grouped_tile_u(tile, tiles_m, tiles_n, g.group_m);
    const int ra = min(Cfg::kBM, M - c.m * Cfg::kBM);
    const int rb = min(Cfg::kBN, N - c.n * Cfg::kBN);
    const int k0 = __builtin_amdgcn_readfirstlane(slice * steps * kStepBytes);
    const int kend = min(K, k0 + steps * kStepBytes);
    const int full = max(0, kend - k0) / kStepBytes;
    const int rot = kMx ? 0 : (int)((blockIdx.x & 7u) * (unsigned)full / 8u);
    return Src{make_rsrc(g.A + (size_t)c.m * Cfg::kBM * g.lda,
                         (uint32_t)ra * (uint32_t)g.lda),
               make_rsrc(g.B + (size_t)c.n * Cfg::kBN * g.ldb,
                         (uint32_t)rb * (uint32_t)g.ldb),
               k0, kend, full, rot, c.m, c.n};
  };
  Src cur = src_of(t);
  Src nxt = src_of(t + walk.stride);

  // DMA source of step d of the unit (d >= steps_pad: step d - steps_pad of
  // the next one).  kEdge: it may not be a whole step of the unit; lanes
  // whose chunk lies at or past its K range read zero.
  struct DmaSrc {
    __amdgpu_buffer_rsrc_t a, b;
    uint32_t k0, oob;
  };
  auto dma_src = [&](int d, auto edge) {
    constexpr bool kEdge = decltype(edge)::value;
    const bool next = kEdge && d >= steps_pad;
    const int dd = next ? d - steps_pad : d;
    const int full = next ? nxt.full : cur.full;
    int dr = dd + (next ? nxt.rot : cur.rot);
    if (dr >= full) dr -= full;
    if (kEdge && dd >= full) dr = dd;  // the step K ends inside, padding
    uint32_t k0 = (uint32_t)((next ? nxt.k0 : cur.k0) + dr * kStepBytes);
    asm volatile("" : "+s"(k0));
    uint32_t oob = 0;
    if constexpr (kEdge)
      oob = (int)(k0 + dchunk * 16) < (next ? nxt.kend : cur.kend) ? 0u : kOobOffset;
    return DmaSrc{next ? nxt.a : cur.a, next ? nxt.b : cur.b, k0, oob};
  };
  // Instruction n of a step (A rows first) into the stage at `dst`.
  auto dma_one = [&](const DmaSrc& s, int dst, int n, auto edge) {
    constexpr bool kEdge = decltype(edge)::value;
    const bool is_a = n < Cfg::kDmaA;
    const int q = is_a ? n : n - Cfg::kDmaA;
    const uint32_t vo = is_a ? voff_a[q] : voff_b[q];
    lds_u8* to = lds + dst + (is_a ? 0 : Cfg::kAStage) + (4 * q + wave) * 1024;
    if (kNt && !is_a)
      dma16_nt(s.b, to, kEdge ? vo | s.oob : vo, s.k0);
    else
      dma16(is_a ? s.a : s.b, to, kEdge ? vo | s.oob : vo, s.k0);
  };

  // ---- fragment reads: rows 16 f + l % 16 of the wave's part.  Lane group
  // g = l / 16 reads slots 2g and 2g + 1 before the XOR; kMx (the MFMA's own
  // K order) chunks g and g + 4 under strip_xor. ----------------------------
  const int r16 = lane & 15, grp = lane >> 4;
  const uint32_t row_a = (uint32_t)((wm * Cfg::kWM + r16) * Cfg::kBK);
  const uint32_t row_b =
      (uint32_t)(Cfg::kAStage + (wn * Cfg::kWN + r16) * Cfg::kBK);
  // Offset of piece q of a fragment in its row.  fp6: lane group g holds
  // bytes 24 g .. 24 g + 23 of the step (element boundaries fall on 3-byte
  // multiples) as three 8-byte pieces; byte b of row r sits in slot
  // (b / 16) ^ slot_xor(r), half (b / 8) % 2: conflict-free.
  uint32_t piece[kPieces];
#pragma unroll
  for (int q = 0; q < kPieces; ++q) {
    if constexpr (k6) {
      const int b = 24 * grp + 8 * q;
      piece[q] = (uint32_t)((((b >> 4) ^ slot_xor(r16)) << 4) + (((b >> 3) & 1) << 3));
    } else if constexpr (kMx) {
      piece[q] = (uint32_t)(((grp + 4 * q) ^ strip_xor(r16)) * 16);
    } else {
      piece[q] = (uint32_t)(((2 * grp + q) ^ slot_xor(r16)) * 16);
    }
  }
  // (The 8-byte pieces as integers: the optimiser widened loads of two-element
  // vectors to the operand's eight, and the array stayed in memory.)
  using Piece = std::conditional_t<k6, uint64_t, i32x4>;
  // Read n of a step, in the order the MFMA use the fragments: A0, every B,
  // A1 ..; every piece of each.
  struct Ptrs {
    const lds_u8 *a[kPieces], *b[kPieces];
  };
  auto ptrs = [&](int stage) {
    Ptrs p;
#pragma unroll
    for (int q = 0; q < kPieces; ++q) {
      p.a[q] = lds + row_a + piece[q] + stage;
      p.b[q] = lds + row_b + piece[q] + stage;
    }
    return p;
  };
  auto read_one = [&](const Ptrs& p, int n) -> Piece {
    const int f = n / kPieces, q = n % kPieces;
    const lds_u8* r = f == 0    ? p.a[q]
                      : f <= FB ? p.b[q] + (f - 1) * 16 * Cfg::kBK
                                : p.a[q] + (f - FB) * 16 * Cfg::kBK;
    if constexpr (k6) return __builtin_bit_cast(uint64_t, lds_read8(r));
    else return lds_read16(r);
  };
  // The six registers of an fp6 operand (the MFMA reads no more).
  auto join6 = [](uint64_t a, uint64_t b, uint64_t c) {
    return i32x8{(int)a, (int)(a >> 32), (int)b, (int)(b >> 32), (int)c, (int)(c >> 32), 0, 0};
  };
  i32x8 fa[2][FA], fb[2][FB];
  auto frag = [&](const Piece* rd) {
    if constexpr (k6) return join6(rd[0], rd[1], rd[2]);
    else return join(rd[0], rd[1]);
  };
  auto set_frags = [&](int set, const Piece (&rd)[kReads]) {
    fa[set][0] = frag(rd);
#pragma unroll
    for (int j = 0; j < FB; ++j) fb[set][j] = frag(rd + kPieces * (1 + j));
#pragma unroll
    for (int i = 1; i < FA; ++i) fa[set][i] = frag(rd + kPieces * (FB + i));
  };

  // kMx: the lane's 16 scale bytes of A and of B_T for the step of each
  // register set.  The packed layout holds, per 128-row group W and per pair
  // p of 128-element MFMA steps, 16 bytes per lane (step 0 of the pair, then
  // step 1; 8 fragments of 16 rows each): for fp4 a 128-byte step is one pair
  // (its two MFMA take halves 0 and 1), for 8-bit operands half of one.  W =
  // the tile's row (A) or column (B_T) index.  Pairs past K and missing units
  // read zero.
  i32x4 mxa[2] = {}, mxb[2] = {};
  auto mx_load = [&](int d, int set) {
    const bool next = d >= steps_pad;
    const int gs = (next ? nxt.k0 : cur.k0) / Cfg::kBK + (next ? d - steps_pad : d);
    const int kel = k4 ? 2 * K : K;  // K in elements
    const int P = mx_pairs(kel);
    const int p = k4 ? gs : gs / 2;
    const MxArgs mx = kernel_mx();
    const int tm = next ? nxt.tm : cur.tm, tn = next ? nxt.tn : cur.tn;
    const bool live = tm >= 0 && p < P;
    const uint32_t vo = (uint32_t)lane * 16u;
    const __amdgpu_buffer_rsrc_t ra =
        make_rsrc(mx.a, live ? (uint32_t)mx_packed_bytes(M, kel) : 0u);
    const __amdgpu_buffer_rsrc_t rb =
        make_rsrc(mx.b, live ? (uint32_t)mx_packed_bytes(N, kel) : 0u);
    mxa[set] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(
        ra, vo + (uint32_t)(live ? (tm * P + p) * 1024 : 0), 0, 0));
    mxb[set] = __builtin_bit_cast(i32x4, __builtin_amdgcn_raw_buffer_load_b128(
        rb, vo + (uint32_t)(live ? (tn * P + p) * 1024 : 0), 0, 0));
  };
  // The wave's scale words of a step (fp4: halves 0 and 1; 8-bit: half `set`
  // of the pair: units start on even steps): A, B_T of the first MFMA, then
  // of fp4's second.
  struct MxWords {
    uint32_t a0, b0, a1, b1;
  };
  auto mx_words = [&](int set) {
    const int h0 = k4 ? 0 : 2 * set;
    MxWords w{};
    w.a0 = (uint32_t)(wm ? mxa[set][h0 + 1] : mxa[set][h0]);
    w.b0 = (uint32_t)(wn ? mxb[set][h0 + 1] : mxb[set][h0]);
    if constexpr (k4) {
      w.a1 = (uint32_t)(wm ? mxa[set][3] : mxa[set][2]);
      w.b1 = (uint32_t)(wn ? mxb[set][3] : mxb[set][2]);
    }
    return w;
  };

  f32x4 acc[FA][FB];
  // MFMA n of a step: blocks row by row, odd rows right to left (the MFMA
  // after a row change shares its B fragment with the one before).
  auto mfma = [&](int set, int n, const MxWords& w) {
    const int i = n / FB, j = i % 2 ? FB - 1 - n % FB : n % FB;
    const i32x8 &x = fb[set][j], &y = fa[set][i];
    f32x4& c = acc[i][j];
    if constexpr (k4) {
      // fp4: 256 elements per 128-byte step, two MFMA per block, on the low
      // and the high 16 bytes of the fragments.
      const i32x8 xh = __builtin_shufflevector(x, x, 4, 5, 6, 7, 0, 1, 2, 3);
      const i32x8 yh = __builtin_shufflevector(y, y, 4, 5, 6, 7, 0, 1, 2, 3);
      if constexpr (kMx) {
        c = mfma_16x16x128_mx<kFmtFp4, kFmtFp4>(x, y, c, w.b0, w.a0, j, i);
        c = mfma_16x16x128_mx<kFmtFp4, kFmtFp4>(xh, yh, c, w.b1, w.a1, j, i);
      } else {
        c = mfma_16x16x128<kFmtFp4, kFmtFp4>(x, y, c);
        c = mfma_16x16x128<kFmtFp4, kFmtFp4>(xh, yh, c);
      }
    } else if constexpr (kMx) {
      c = mfma_16x16x128_mx<fmt_b(kFmt), fmt_a(kFmt)>(x, y, c, w.b0, w.a0, j, i);
    } else {
      c = mfma_16x16x128<fmt_b(kFmt), fmt_a(kFmt)>(x, y, c);
    }
  };
  MxWords mxw{};  // of the step whose tail MFMA are still to come
  auto tail = [&](int set) {
#pragma unroll
    for (int n = kHead; n < kMfma; ++n) mfma(set, n, mxw);
  };
  auto next_stage = [](int s) {
    s += Cfg::kStage;
    return s == S * Cfg::kStage ? 0 : s;
  };
  // One step after its barrier: register set `set`, its own stage at `st`
  // (refilled with step d), the next step's at `rst`.
  auto step = [&](int set, int st, int rst, int d, bool with_tail, auto edge) {
    if (with_tail) tail(set ^ 1);
    if constexpr (kMx) mxw = mx_words(set);
    const DmaSrc src = dma_src(d, edge);
    const Ptrs p = ptrs(rst);
    sched_fence();
    Piece rd[kReads];
#pragma unroll
    for (int n = 0; n < kHead; ++n) {
      mfma(set, n, mxw);
      __builtin_amdgcn_sched_group_barrier(0x008, k4 ? 2 : 1, 0);
      const int r0 = n < kTwo ? 2 * n : n + kTwo;
      if (r0 < kReads) {
        rd[r0] = read_one(p, r0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
      if (n < kTwo) {
        rd[r0 + 1] = read_one(p, r0 + 1);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      }
#pragma unroll
      for (int q = 0; q < kDma; ++q)
        if (q * kHead / kDma == n) {
          dma_one(src, st, q, edge);
          __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
      sched_fence();
    }
    // kMx: the scales of the step after next, into this step's set (its head
    // MFMA are issued and its words copied): two steps ahead, so that they
    // retire with DMA the waits cover anyway.
    if constexpr (kMx) mx_load(d - (S - 2), set);
    set_frags(set ^ 1, rd);
  };

  // kExt: the wave's row scales, column scales and biases into its staging
  // area (rows at +0, columns at +512, bias at +1024), one float per lane
  // and 64; zero past M / N.
  lds_u8* stg = lds + Cfg::kStoreBase + wave * Cfg::kStoreStage;
  auto scale_dma = [&](int tile) {
    const TileCoord c = grouped_tile_u(tile, tiles_m, tiles_n, g.group_m);
    const EpiArgs ea = kernel_epi();
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const __amdgpu_buffer_rsrc_t rr =
        make_rsrc(ea.row_scale, ea.row_scale ? (uint32_t)M * 4u : 0u);
    const __amdgpu_buffer_rsrc_t rc =
        make_rsrc(ea.col_scale, ea.col_scale ? (uint32_t)N * 4u : 0u);
    const __amdgpu_buffer_rsrc_t rb =
        make_rsrc(ea.bias, ea.bias ? (uint32_t)N * 4u : 0u);
    const uint32_t ro = (uint32_t)(c.m * Cfg::kBM + wm * Cfg::kWM + ln) * 4u;
    const uint32_t co = (uint32_t)(c.n * Cfg::kBN + wn * Cfg::kWN + ln) * 4u;
#pragma unroll
    for (int h = 0; h < (Cfg::kWM + 63) / 64; ++h)
      dma4(rr, stg + 256 * h, ro + 256 * h);
#pragma unroll
    for (int h = 0; h < (Cfg::kWN + 63) / 64; ++h) {
      dma4(rc, stg + 512 + 256 * h, co + 256 * h);
      dma4(rb, stg + 1024 + 256 * h, co + 256 * h);
    }
  };

  bool stores = false;     // the previous tile's C stores are in flight
  bool first_tile = true;  // its first steps' DMA came from the prologue
  int st = 0;              // stage of the step about to start
  // Steps k, k + 1 of the tile (register sets 0, 1).  first: the tile's
  // first pair; warm: no tail before its first step (the workgroup's first).
  auto step_pair = [&](int k, bool first, bool warm, auto edge) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // Step k + h's reads are done (every wave's, after the barrier: its
      // stage may be refilled).  Step k + h + 1 landed: newer than it are
      // S - 2 steps' DMA and, in the first S - 1 steps of a tile after the
      // first, the previous tile's stores (kExt's vector loads only make
      // the wait longer).
      wait_lgkmcnt<0>();
      if (stores && k + h < S - 1) wait_vmcnt<(S - 2) * kD + kStores>();
      else if (kMx && first_tile && k + h < S - 1) wait_vmcnt<(S - 2) * kDma>();
      else wait_vmcnt<(S - 2) * kD>();
      barrier();
      if constexpr (kExt)
        if (first && h == 0) scale_dma(kSplit ? t % tiles : t);
      const int rst = next_stage(st);
      step(h, st, rst, k + h + S, !(warm && h == 0), edge);
      st = rst;
    }
  };

  // Prologue of the first tile: (kMx: the scales of steps 0 and 1,) steps
  // 0 .. S - 1, then the reads of step 0.
  if constexpr (kMx) {
    mx_load(0, 0);
    mx_load(1, 1);
  }
#pragma unroll
  for (int d = 0; d < S; ++d) {
    const DmaSrc src = dma_src(d, std::true_type{});
#pragma unroll
    for (int n = 0; n < kDma; ++n) dma_one(src, d * Cfg::kStage, n, std::true_type{});
  }
  wait_vmcnt<(S - 1) * kDma>();
  barrier();
  {
    const Ptrs p = ptrs(0);
    Piece rd[kReads];
#pragma unroll
    for (int r = 0; r < kReads; ++r) rd[r] = read_one(p, r);
    set_frags(0, rd);
  }

  for (;;) {
#pragma unroll
    for (int i = 0; i < FA; ++i)
#pragma unroll
      for (int j = 0; j < FB; ++j) acc[i][j] = f32x4{};
    // The first pair apart: no tail MFMA of this tile before it.
    step_pair(0, true, true, std::true_type{});
    // Pairs k whose DMA (steps k + S, k + S + 1) are whole steps of the unit.
    const int k_edge = max(0, (cur.full - S) & ~1);
    int k = 2;
    for (; k < k_edge; k += 2) step_pair(k, false, false, std::false_type{});
    for (; k < steps_pad; k += 2) step_pair(k, false, false, std::true_type{});
    tail(1);

    // ---- epilogue ---------------------------------------------------------
    bool write_c = !kSplit;
    if constexpr (kSplit) {
      // The unit's fp32 partial: wave w's FA x FB blocks at ((t * 4 + w) * FA *
      // FB + FB i + j) KiB of g.split.partial, lane l's 16 bytes at + 16 l (unit
      // t = slice * tiles + tile).
      constexpr int kCoherent = 16;  // cache policy: sc1
      const int slices = g.split.slices;
      const __amdgpu_buffer_rsrc_t rp = make_rsrc(
          g.split.partial, (uint32_t)tiles * (uint32_t)slices * (uint32_t)Cfg::kPartial);
      const uint32_t lo = (uint32_t)lane * 16u;
      // Wave-uniform offsets in scalar registers (t's division ran on the
      // VALU): a buffer instruction whose scalar operand sits in a VGPR is
      // wrapped in a readfirstlane loop.
      const uint32_t own_off =
          (uint32_t)__builtin_amdgcn_readfirstlane((t * 4 + wave) * (Cfg::kPartial / 4));
#pragma unroll
      for (int i = 0; i < FA; ++i)
#pragma unroll
        for (int j = 0; j < FB; ++j)
          store_b128<kCoherent>(__builtin_bit_cast(i32x4, acc[i][j]), rp,
                                lo + (uint32_t)((FB * i + j) * 1024), own_off);
      if (g.split.arrivals) {
        const int tile = __builtin_amdgcn_readfirstlane(t % tiles);
        const int own = __builtin_amdgcn_readfirstlane(t / tiles);
        int* const ctr = g.split.arrivals + tile * 4 + wave;
        // This wave's partial stores (and every other operation of it) are
        // complete before its arrival is counted.
        wait_vmcnt<0>();
        int before = 0;
        if (lane == 0)
          before = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
        before = __builtin_amdgcn_readfirstlane(before);
        if (before == slices - 1) {
          // Last arrival: +0 + slice 0 + slice 1 + ..., two slices' loads
          // in flight at a time; the own slice comes from the accumulators,
          // slices past the last read zero (offset out of range: +0, which
          // leaves every sum unchanged).
          f32x4 sum[FA][FB];
#pragma unroll
          for (int i = 0; i < FA; ++i)
#pragma unroll
            for (int j = 0; j < FB; ++j) sum[i][j] = f32x4{};
          for (int q0 = 0; q0 < slices; q0 += 2) {
            f32x4 v[2][FA][FB];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
              const int q = q0 + b;
              const uint32_t so =
                  (uint32_t)(((q < slices ? q : 0) * tiles + tile) * 4 + wave) * (uint32_t)(Cfg::kPartial / 4);
              const uint32_t oob = q < slices && q != own ? 0u : kOobOffset;
#pragma unroll
              for (int i = 0; i < FA; ++i)
#pragma unroll
                for (int j = 0; j < FB; ++j)
                  v[b][i][j] = __builtin_bit_cast(
                      f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                 rp, (lo + (uint32_t)((FB * i + j) * 1024)) | oob, so,
                                 kCoherent));
            }
#pragma unroll
            for (int b = 0; b < 2; ++b) {
              const bool is_own = q0 + b == own;
#pragma unroll
              for (int i = 0; i < FA; ++i)
#pragma unroll
                for (int j = 0; j < FB; ++j)
                  sum[i][j] += is_own ? acc[i][j] : v[b][i][j];
            }
          }
#pragma unroll
          for (int i = 0; i < FA; ++i)
#pragma unroll
            for (int j = 0; j < FB; ++j) acc[i][j] = sum[i][j];
          // Every lane stores the same zero: no branch on the lane.
          __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          write_c = true;
        }
      }
    }
    if (write_c) {
    const TileCoord tc =
        grouped_tile_u(kSplit ? t % tiles : t, tiles_m, tiles_n, g.group_m);
    const int rows_left = M - tc.m * Cfg::kBM - wm * Cfg::kWM;  // from wave row 0
    const int cols_left = N - tc.n * Cfg::kBN - wn * Cfg::kWN;  // from wave col 0
    auto oob_unless = [](int x, int limit) -> uint32_t {
      return (uint32_t)((limit - 1 - x) >> 31) & kOobOffset;
    };
    int elane = lane;
    asm volatile("" : "+v"(elane));
    const int er16 = elane & 15, egrp = elane >> 4;
    EpiVec<FA, FB> ev;
    if constexpr (kExt) ev.read_lds(stg, kernel_epi(), scale, elane);
    auto pack = [&](const f32x4& a, int i, int j) -> u32x2 {
      if constexpr (kExt)
        return ev.template pack4<kAct, kOut>(a[0], a[1], a[2], a[3], i, j);
      else
        return u32x2{pack_bf16x2(a[0] * scale, a[1] * scale),
                     pack_bf16x2(a[2] * scale, a[3] * scale)};
    };
    // C window of this wave; the range ends at its last valid element.
    constexpr int es = kExt ? out_bytes(kOut) : 2;  // bytes per C element
    const int wrows = min(Cfg::kWM, rows_left), wcols = min(Cfg::kWN, cols_left);
    uint8_t* cw = reinterpret_cast<uint8_t*>(g.C) +
                  ((size_t)(tc.m * Cfg::kBM + wm * Cfg::kWM) * g.ldc +
                   tc.n * Cfg::kBN + wn * Cfg::kWN) * es;
    const bool any = wrows > 0 && wcols > 0;
    const __amdgpu_buffer_rsrc_t rsrc_c = make_rsrc(
        cw, any ? (uint32_t)(((wrows - 1) * g.ldc + wcols) * es) : 0u);
    if constexpr (kExt && kOut >= kOutF32) {
      // 4 consecutive elements per lane and block: one 16- or 4-byte store,
      // or one per element.
#pragma unroll
      for (int i = 0; i < FA; ++i)
#pragma unroll
        for (int j = 0; j < FB; ++j) {
          const int r = 16 * i + er16, col = 16 * j + 4 * egrp;
          const uint32_t off = (uint32_t)((r * g.ldc + col) * es) |
                               oob_unless(r, rows_left);
          const f32x4& a = acc[i][j];
          const f32x4 v = ev.template value4<kAct>(a[0], a[1], a[2], a[3], i, j);
          if constexpr (kOut == kOutF32) {
            if constexpr (kVec) {
              store_b128<kStoreCPart>(__builtin_bit_cast(i32x4, v), rsrc_c,
                                      off | oob_unless(col, cols_left), 0);
            } else {
              const i32x4 vb = __builtin_bit_cast(i32x4, v);
#pragma unroll
              for (int e = 0; e < 4; ++e)
                __builtin_amdgcn_raw_buffer_store_b32(
                    (uint32_t)vb[e], rsrc_c,
                    (off | oob_unless(col + e, cols_left)) + 4 * e, 0, kStoreCPart);
            }
          } else {
            const uint32_t w = ev.e4m3x4(v);
            if constexpr (kVec) {
              __builtin_amdgcn_raw_buffer_store_b32(
                  w, rsrc_c, off | oob_unless(col, cols_left), 0, kStoreCPart);
            } else {
#pragma unroll
              for (int e = 0; e < 4; ++e)
                __builtin_amdgcn_raw_buffer_store_b8(
                    (uint8_t)(w >> (8 * e)), rsrc_c,
                    (off | oob_unless(col + e, cols_left)) + e, 0, kStoreCPart);
            }
          }
        }
    } else if constexpr (kVec) {
      // 8-byte piece p (columns 4p .. 4p + 3) of staged row r at slot
      // p ^ (r % 16) (p ^ (r % 8) where a row's pieces are not a multiple of
      // 16); read back as 16-byte units (pieces 2c, 2c + 1: halves swapped on
      // odd rows).  One wave's LDS operations complete in order: no barrier.
      constexpr int kRow = Cfg::kWN * 2;    // bytes of a staged row
      constexpr int kUnits = Cfg::kWN / 8;  // 16-byte units of a row
      constexpr int kX = (Cfg::kWN / 4) % 16 == 0 ? 15 : 7;
      // Row segments that are not whole 128-byte lines go out cached: the
      // L2 merges the lines (kStoreCPart).
      constexpr int kAux = kRow % 128 == 0 ? kStoreC : kStoreCPart;
#pragma unroll
      for (int i = 0; i < FA; ++i) {
#pragma unroll
        for (int j = 0; j < FB; ++j)
          lds_write8(stg + er16 * kRow + (((4 * j + egrp) ^ (er16 & kX)) * 8),
                     pack(acc[i][j], i, j));
        compiler_fence();
#pragma unroll
        for (int q = 0; q < Cfg::kRows16 / 1024; ++q) {
          const int x = 64 * q + elane, r = x / kUnits, c = x % kUnits;
          i32x4 v = lds_read16(stg + r * kRow + (((2 * c) ^ (r & kX)) >> 1) * 16);
          if (r & 1) v = i32x4{v[2], v[3], v[0], v[1]};
          const uint32_t off = (uint32_t)(((16 * i + r) * g.ldc + 8 * c) * 2) |
                               oob_unless(16 * i + r, rows_left) |
                               oob_unless(8 * c, cols_left);
          store_b128<kAux>(v, rsrc_c, off, 0);
        }
        compiler_fence();
      }
    } else {
#pragma unroll
      for (int i = 0; i < FA; ++i)
#pragma unroll
        for (int j = 0; j < FB; ++j) {
          const u32x2 pk = pack(acc[i][j], i, j);
          const int r = 16 * i + er16, col = 16 * j + 4 * egrp;
          const uint32_t rb = (uint32_t)((r * g.ldc + col) * 2) | oob_unless(r, rows_left);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const uint32_t w = (e < 2 ? pk.x : pk.y) >> (16 * (e & 1));
            __builtin_amdgcn_raw_buffer_store_b16(
                (unsigned short)w, rsrc_c,
                (rb | oob_unless(col + e, cols_left)) + 2 * e, 0, kStoreCPart);
          }
        }
    }

    }  // write_c

    t += walk.stride;
    if (t >= walk.end) break;
    cur = nxt;
    nxt = src_of(t + walk.stride);
    stores = kSplit || kVec || (kExt && kOut >= kOutF32);
    first_tile = false;
  }
  // The last tile's look-ahead DMA (empty ranges) still count in vmcnt.
  wait_vmcnt<0>();
}

}  // namespace detail
}  // namespace hipgemm
