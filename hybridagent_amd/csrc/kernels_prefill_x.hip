// Prefill-shaped W4A16 MoE expert GEMMs, exact form, for group sizes that are
// powers of two >= 32 (the released checkpoints' 32 and the benchmark's 128):
//
//   MODE = gateup : inter[s] = gelu(x[tok(s)] Wg^T) * (x[tok(s)] Wu^T)
//                   (quantization.py:112-120), rows s in expert-segment order
//   MODE = down   : dn[sorted_pos[s]] = inter[s] W_d^T   (quantization.py:122-127)
//
// Work item = (m-tile of up to 256 rows of one expert's segment, n-tile of
// 256 weight rows; gate_up: 128 gate rows + the matching 128 up rows).  A
// persistent grid of one 512-thread workgroup per CU takes the items from a
// work queue (the tile list lists the large tiles first): for down, XCD x
// (workgroups are dealt to the 8 XCDs in turn) owns m-tiles x, x + 8, ...
// with all their n-tiles and a queue of its own; gate_up has one queue for
// the chip.  Each of the eight wavefronts owns 32
// weight rows (gate_up: 16 gate + their 16 up rows) for all the item's
// rows: MB m-blocks of v_mfma_f32_32x32x16_bf16 accumulators, MB = the item's
// 32-row blocks, 1 .. 8 (gate_up's half n-tile: 1 .. 4 per wavefront half).
//
// The small tails (most of them are whole experts of few rows) give a stage
// little MFMA work, so what a stage costs whatever its rows decides.
//  - They run as tail items (px_run_t): stages of 128 k, the item's scales
//    read once as one contiguous block.  128 experts of 64 rows at the Gemma
//    shape, G = 128, tiled: gate_up 144 -> 116 us, down 90 -> 76 us; packed
//    layers of 257 tokens x top-8 at G = 32 / 128 322 -> 162 / 173 -> 157 us
//    (with a 16-byte scale chunk per row and stage the 768 rows of a
//    three-n-tile stage touched more cache lines than an XCD's L2 holds).
//  - On the tiled weights, where nearly all m-tiles are tails of at most 32
//    rows, each is a wide item of three n-tiles (px_run_w): one stage's cost
//    for three n-tiles' weights.
// Each output is the one-n-tile item's bit for bit.
//
// Per 64-wide k stage, all by direct global -> LDS loads of 16 bytes per
// lane (one instruction fills 1 KiB).  Every load of the main loop is one,
// all of one size, so they complete in the order they were issued and a
// partial vmcnt wait proves a stage landed (direct loads of 4 bytes were
// seen to finish ahead of 16-byte ones issued before them):
//   A  the item's activation rows, 8 rows x 128 bytes per instruction, rows
//      128 bytes apart with the 16-byte chunks XOR-swizzled by (row / 2) % 8
//      so that the fragment reads of 16 consecutive rows cover all LDS banks
//      once;
//   B  the packed words of the 256 weight rows (32 bytes each) and, per
//      row, the aligned 16 bytes of its scales that hold this stage's
//      group(s) (an aligned pair of bf16).
// A ring of three stages keeps two in flight while one is multiplied, and
// runs on across items: a workgroup issues its next item's first two stages
// before the current item's epilogue, which runs while they land.  Each
// lane dequantises the four packed words of its weight row that its four
// MFMA steps need exactly as the reference does -- bf16_RNE(q * s),
// q = u - 8 -- in registers; one B fragment feeds the MB MFMAs of its step.
// The lane layout of an MFMA step: lane l holds row (col) l % 32 and the
// 8 k of chunk 4 (l / 32) + s of the stage, for A and B alike.
//
// The MFMAs compute D[weight row][activation row] (dequantised weights as
// the A operand), so each lane ends with four consecutive output columns of
// one activation row per register quad: the epilogue stores 8 bytes per
// lane straight from registers; gate_up finds each gate column's up column
// in the same lane and applies gelu_tanh(gate) * up with the reference's
// bf16 rounding points.
//
// While direct LDS loads are in flight the kernel issues no other vector
// memory load: row indices (gate_up: the next item's gathered token rows;
// down: the current item's output rows) come into an LDS table by a direct
// load of their own with the item's second-to-last stage.  (A direct LDS
// load and an ordinary load issued after it need not complete in that
// order, so a vmcnt wait counted for one could pass while the other is
// outstanding.)  Each wavefront issues only the loads it needs; a stage's
// wait counts the loads that wavefront issued after it.
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "lds_pipe.hpp"

namespace w4a16 {

namespace {

constexpr int kPxWaves = 8;
constexpr int kPxThreads = 64 * kPxWaves;
constexpr int kPxBM = kPrefillXBM;           // 256 rows
constexpr int kPxBN = 32 * kPxWaves;         // 256 weight rows per item
constexpr int kPxKT = 64;                    // k per stage
constexpr int kPxStages = 3;
// LDS: the ring of stages, each A [256 rows][128 B] | B words [256 tile
// rows][32 B] | scale chunks [256 tile rows][16 B]; the row-index table
// (512 ints from a 16-byte-aligned start: sorted_pos[s & ~3 ..] for a
// segment starting at s); down's epilogue rows
constexpr int kPxBOff = kPxBM * kPxKT * 2;
constexpr int kPxSOff = kPxBOff + kPxBN * kPxKT / 2;
constexpr int kPxStageBytes = kPxSOff + kPxBN * 16;
constexpr int kPxTable = kPxStages * kPxStageBytes;  // 512 row indices
// down's epilogue rows: 32 rows x 32 bf16 per wavefront, rows 80 bytes
// apart (the 8-byte writes of 32 rows spread over the banks)
constexpr int kPxEpiOff = kPxTable + 2048;
constexpr int kPxEpiPitch = 80;
constexpr int kPxEpiBytes = 32 * kPxEpiPitch;
constexpr int kPxEpiEnd = kPxEpiOff + kPxWaves * kPxEpiBytes;
// the item index a workgroup takes from its queue (one int), last in LDS
constexpr int kPxLds = 160 * 1024;
constexpr int kPxQSlot = kPxLds - 16;
static_assert(kPxEpiEnd <= kPxQSlot, "LDS of a CU");
// at most four direct A loads per wavefront and stage (fewer for tiles of
// fewer rows), then one B-word load and one scale-chunk load (wavefronts
// 0..3)
constexpr int kPxNA = 4;
// Wide items (tiled weights): a segment tail of at most kPrefillTinyRows rows
// (one m-block) takes kPxWide n-tiles at once, so its per-stage latency is
// paid once for three n-tiles' weights.  Its stage holds 32
// activation rows (4 KiB of the A region); the other n-tiles' words and
// scale chunks go in the rest of that region: n-tile b of the item has its
// words at px_wide_b(b) and its scale chunks at px_wide_s(b).
constexpr int kPxWide = 3;
constexpr int px_wide_b(int b) { return b == 0 ? kPxBOff : 4096 + 8192 * (b - 1); }
constexpr int px_wide_s(int b) { return b == 0 ? kPxSOff : 4096 + 8192 * (kPxWide - 1) + 4096 * (b - 1); }
static_assert(px_wide_s(kPxWide - 1) + 4096 <= kPxBOff, "a wide stage's blocks fit in the A region");
static_assert(kPrefillTinyRows == 32, "a wide item is one 32-row m-block");
// Tail items (px_run_t): a segment tail of at most 64 rows (MBT = 1 or 2
// m-blocks).  Its stage holds 128 k: A [2 halves][32 MBT rows][128 B] | B
// words, 16 KiB ([256 rows][64 B] from the packed layout, [2][256 rows][32 B]
// from the tiled copy); the item's scales, whole, follow the ring of three
// such stages (gate_up: the gate rows', the up rows' at PrefillArgs::tail_s1).
constexpr int kPxTailMaxBlocks = 2;
constexpr int kPxTailRing = 3;
constexpr int px_tail_b(int mbt) { return mbt * 8192; }
constexpr int px_tail_stage(int mbt) { return px_tail_b(mbt) + kPxBN * kPxKT; }

}  // namespace


// One work item: (m-tile, first n-tile, n-tiles nb) and what that fixes.
struct PxItem {
  int nt, e, seg0, nrows, mb, nb;
};

// Item `item` of a queue of n_local m-tiles, tile list entries x0, x0 + xs,
// ...; [t0, t1) are the tails of at most kPrefillTinyRows rows.  With n_wide
// > 0 these are wide items, n_wide of kPxWide n-tiles each (n-tiles past the
// matrix compute on its last rows and store nothing), where they stand in the
// list: a wide item is longer than the tails after it.  Else every m-tile has
// n_nt items, the tails [t0, t1) last: they are the shortest.
__device__ __forceinline__ PxItem px_item_info(const PrefillArgs& a, int x0, int xs, int n_local, int t0, int t1,
                                               int n_wide, int item) {
  PxItem it;
  int lm;
  it.nb = 1;
  const int i0 = t0 * a.n_nt, i1 = i0 + (t1 - t0) * n_wide;
  if (n_wide > 0 && item >= i0) {
    if (item < i1) {
      const int j = item - i0;
      const int q = j / n_wide;
      lm = t0 + q;
      it.nt = kPxWide * (j - q * n_wide);
      it.nb = kPxWide;
    } else {
      const int j = item - i1;
      const int q = j / a.n_nt;
      lm = t1 + q;
      it.nt = j - q * a.n_nt;
    }
  } else {
    lm = item / a.n_nt;
    it.nt = item - lm * a.n_nt;
    if (n_wide == 0 && lm >= t0) lm = lm - t0 < n_local - t1 ? lm - t0 + t1 : lm - (n_local - t1);
  }
  const int tile = ld_uniform(a.tiles, x0 + xs * lm);
  it.e = tile >> 16;
  it.seg0 = ld_uniform(a.offsets, it.e) + (tile & 0xFFFF) * kPxBM;
  it.nrows = min(kPxBM, ld_uniform(a.offsets, it.e + 1) - it.seg0);
  it.mb = (it.nrows + 31) >> 5;  // 32-row blocks
  return it;
}

// whether a one-n-tile item runs as a tail item (px_run_t): one or two
// m-blocks
__device__ __forceinline__ bool px_is_tail(const PrefillArgs& a, const PxItem& it) {
  return it.mb <= kPxTailMaxBlocks && a.tail_s1[it.mb == 2 ? 1 : 0] >= 0;
}

// A lane's load sources for one item; na = the wavefront's A loads per
// stage, n = all its loads per stage (both wavefront-uniform).
struct PxLoads {
  __amdgpu_buffer_rsrc_t wsrc, ssrc;
  int avoff[kPxNA];
  int bvoff, bstride, svoff;
  int na, n;
};

// weight row of tile row tr of n-tile nt (gate_up: wavefront w's tile rows
// 32 w .. 32 w + 31 are gate rows 128 nt + 16 w .. + 15, then the matching
// up rows; rows past the matrix repeat its last row, their results are
// dropped)
template <int MODE>
__device__ __forceinline__ int px_weight_row(const PrefillArgs& a, int nt, int tr) {
  if (MODE == kModeGateUp) {
    const int w = tr >> 5, cc = tr & 31;
    const int col = min(128 * nt + 16 * w + (cc & 15), a.I - 1);
    return cc < 16 ? col : a.I + col;
  }
  return min(kPxBN * nt + tr, a.N - 1);
}

// gate_up reads the item's gathered rows from the LDS table, which must
// hold this item's rows (row r at entry seg0 % 4 + r)
template <int MODE, bool TILED>
__device__ __forceinline__ PxLoads px_loads(const PrefillArgs& a, const PxItem& it, const unsigned char* smem) {
  PxLoads L;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // A: instruction j = wave + 8 i brings rows 8 j .. 8 j + 7; lane l takes
  // row 8 j + l / 8 into LDS slot l % 8, i.e. chunk (l % 8) ^ ((row / 2) % 8)
  // of the row (rows past the segment repeat its last row).
  const int* table = reinterpret_cast<const int*>(smem + kPxTable);
  L.na = 0;
#pragma unroll
  for (int i = 0; i < kPxNA; ++i) {
    const int j = wave + 8 * i;
    const bool real = j < 4 * it.mb;
    L.na += real ? 1 : 0;
    const int r = 8 * j + (lane >> 3);
    const int rr = min(r, it.nrows - 1);
    const int64_t src = MODE == kModeGateUp ? (real ? table[(it.seg0 & 3) + rr] : 0) / a.topk : it.seg0 + rr;
    const int chunk = (lane & 7) ^ ((r >> 1) & 7);
    L.avoff[i] = real ? (int)(src * a.lda * 2) + 16 * chunk : 0;
  }
  L.n = L.na + 1 + (wave < 4 ? 1 : 0);
  // B words: instruction `wave` brings tile rows 32 wave .. + 31, lane l row
  // 32 wave + l / 2, bytes 16 (l % 2) of the stage's 32
  const int K2 = a.K >> 1;  // packed bytes per weight row
  if (TILED) {
    // tiled copy: the item's stage kt is the 8 KiB block (nt, kt) of the
    // expert, tile rows in order, so instruction `wave` reads one KiB
    const int nkt = a.K / kPxKT;
    const int64_t per_e = (int64_t)a.n_nt * nkt * 2048;  // int32 words
    L.wsrc = make_rsrc(reinterpret_cast<const uint32_t*>(a.wt) + (int64_t)it.e * per_e, (uint32_t)(per_e * 4));
    L.bvoff = it.nt * nkt * 8192 + wave * 1024 + 16 * lane;
    L.bstride = 8192;
  } else {
    L.wsrc = make_rsrc(reinterpret_cast<const uint32_t*>(a.wp) + (int64_t)it.e * a.N * (a.K >> 3),
                       (uint32_t)a.N * K2);
    L.bvoff = px_weight_row<MODE>(a, it.nt, 32 * wave + (lane >> 1)) * K2 + 16 * (lane & 1);
    L.bstride = kPxKT / 2;
  }
  // scale chunks: waves 0..3 bring tile rows 64 wave + l, the aligned 16
  // bytes holding the stage's scale pair (the stage adds 2 x the pair's
  // group index, the lane rounds down to 16 bytes).  The descriptor starts
  // at the expert's scales rounded down to 16 bytes; svoff carries the
  // difference.
  const uintptr_t sbase = reinterpret_cast<uintptr_t>(a.ws + (int64_t)it.e * a.N * a.ng);
  L.ssrc = make_rsrc(reinterpret_cast<const void*>(sbase & ~uintptr_t(15)), (uint32_t)a.N * a.ng * 2u + 16u);
  const bool sreal = wave < 4;
  L.svoff = sreal ? (int)(sbase & 15) + px_weight_row<MODE>(a, it.nt, 64 * wave + lane) * a.ng * 2 : 0;
  return L;
}

// Part `part` (0..3, issued before MFMA step `part`) of the direct loads of
// stage kt of an item into ring slot `slot`, L.n loads in all: part p brings
// A load p (if this wavefront has one), part 0 also the B words, part 1 the
// scale chunks.
__device__ __forceinline__ void px_issue(const PrefillArgs& a, const PxLoads& L, unsigned char* smem, int kt,
                                         int slot, int part) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  unsigned char* st = smem + slot * kPxStageBytes;
  if (part < L.na)
    px_dma16(make_rsrc(a.act, (uint32_t)a.act_bytes), L.avoff[part], kt * (kPxKT * 2),
             st + (wave + 8 * part) * 1024);
  if (part == 0) px_dma16(L.wsrc, L.bvoff, kt * L.bstride, st + kPxBOff + wave * 1024);
  if (part == 1 && wave < 4) {
    const int gpair = ((kt * kPxKT) >> a.gshift) & ~1;
    px_dma16(L.ssrc, (L.svoff + 2 * gpair) & ~15, 0, st + kPxSOff + 1024 * wave);
  }
}

__device__ __forceinline__ void px_issue_all(const PrefillArgs& a, const PxLoads& L, unsigned char* smem, int kt,
                                             int slot) {
#pragma unroll
  for (int p = 0; p < 4; ++p) px_issue(a, L, smem, kt, slot, p);
}

// One direct load per wavefront: the row indices sorted_pos[tseg & ~3 ..]
// (512 entries; past the routed rows they read as zero, readers clamp to the
// segment) into the LDS table; wavefronts w and w + 2 bring the same part.
__device__ __forceinline__ void px_issue_table(const PrefillArgs& a, unsigned char* smem, int tseg) {
  const int lane = threadIdx.x & 63;
  const int half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) & 1;
  px_dma16(make_rsrc(a.sorted_pos, (uint32_t)a.rows_total * 4u), 4 * ((tseg & ~3) + 256 * half + 4 * lane), 0,
           smem + kPxTable + 1024 * half);
}

// A wide item's load sources: wavefronts 0..3 bring its 32 activation rows
// (one A load each, as a one-m-block item's); every wavefront the words of
// its 32 tile rows of each n-tile, wavefronts 0..3 the scale chunks of each.
struct PxLoadsW {
  __amdgpu_buffer_rsrc_t wsrc, ssrc;
  int avoff;
  int bvoff[kPxWide], svoff[kPxWide];
  int na, n;
};

template <int MODE>
__device__ __forceinline__ PxLoadsW px_loads_w(const PrefillArgs& a, const PxItem& it, const unsigned char* smem) {
  PxLoadsW L;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int* table = reinterpret_cast<const int*>(smem + kPxTable);
  const bool areal = wave < 4;
  const int r = 8 * wave + (lane >> 3);
  const int rr = min(r, it.nrows - 1);
  const int64_t src = MODE == kModeGateUp ? (areal ? table[(it.seg0 & 3) + rr] : 0) / a.topk : it.seg0 + rr;
  const int chunk = (lane & 7) ^ ((r >> 1) & 7);
  L.avoff = areal ? (int)(src * a.lda * 2) + 16 * chunk : 0;
  L.na = areal ? 1 : 0;
  L.n = L.na + kPxWide + (wave < 4 ? kPxWide : 0);
  // tiled copy: n-tiles past the expert's read past the descriptor's range
  // (zeros); their results are not stored
  const int nkt = a.K / kPxKT;
  const int64_t per_e = (int64_t)a.n_nt * nkt * 2048;
  L.wsrc = make_rsrc(reinterpret_cast<const uint32_t*>(a.wt) + (int64_t)it.e * per_e, (uint32_t)(per_e * 4));
#pragma unroll
  for (int b = 0; b < kPxWide; ++b) L.bvoff[b] = (it.nt + b) * nkt * 8192 + wave * 1024 + 16 * lane;
  const uintptr_t sbase = reinterpret_cast<uintptr_t>(a.ws + (int64_t)it.e * a.N * a.ng);
  L.ssrc = make_rsrc(reinterpret_cast<const void*>(sbase & ~uintptr_t(15)), (uint32_t)a.N * a.ng * 2u + 16u);
#pragma unroll
  for (int b = 0; b < kPxWide; ++b)
    L.svoff[b] = wave < 4 ? (int)(sbase & 15) + px_weight_row<MODE>(a, it.nt + b, 64 * wave + lane) * a.ng * 2 : 0;
  return L;
}

// Part `part` (0..3, issued before MFMA step `part`) of a wide item's stage
// kt into ring slot `slot`: part 0 the A load, part p < kPxWide the words of
// n-tile p, part p >= 1 the scale chunks of n-tile p - 1.
__device__ __forceinline__ void px_issue_w(const PrefillArgs& a, const PxLoadsW& L, unsigned char* smem, int kt,
                                           int slot, int part) {
  static_assert(kPxWide <= 3, "four parts carry the loads of three n-tiles");
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  unsigned char* st = smem + slot * kPxStageBytes;
  if (part == 0 && L.na > 0)
    px_dma16(make_rsrc(a.act, (uint32_t)a.act_bytes), L.avoff, kt * (kPxKT * 2), st + wave * 1024);
  if (part < kPxWide) px_dma16(L.wsrc, L.bvoff[part < kPxWide ? part : 0], kt * 8192, st + px_wide_b(part) + wave * 1024);
  if (part >= 1 && part <= kPxWide && wave < 4) {
    const int b = part >= 1 ? part - 1 : 0;
    const int gpair = ((kt * kPxKT) >> a.gshift) & ~1;
    px_dma16(L.ssrc, (L.svoff[b] + 2 * gpair) & ~15, 0, st + px_wide_s(b) + 1024 * wave);
  }
}

// A tail item's load sources (MBT m-blocks): MBT A loads and two B loads per
// wavefront and stage of 128 k.
struct PxLoadsT {
  __amdgpu_buffer_rsrc_t asrc, wsrc;
  int avoff, bvoff[2];
  int bback[2];          // from a B piece past the row to the one before it
  int bstage, bw0, bw1;  // B: bytes per stage; LDS place of load i: wave bw0 + i bw1
};

// columns of a group of 32 weight rows lie inside the matrix
template <int MODE>
__device__ __forceinline__ bool px_group_real(const PrefillArgs& a, int nt, int g) {
  return MODE == kModeGateUp ? 128 * nt + 16 * g < a.I : kPxBN * nt + 32 * g < a.N;
}

template <int MODE, bool TILED, int MBT>
__device__ __forceinline__ PxLoadsT px_loads_t(const PrefillArgs& a, const PxItem& it, const unsigned char* smem) {
  PxLoadsT L;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int* table = reinterpret_cast<const int*>(smem + kPxTable);
  // A: instructions of 8 rows of one 64-wide half; MBT = 1: wavefront w
  // brings rows 8 (w % 4) .. of half w / 4, MBT = 2: rows 8 w .. of both
  const int r = 8 * (MBT == 1 ? wave & 3 : wave) + (lane >> 3);
  const int rr = min(r, it.nrows - 1);
  const int64_t src = MODE == kModeGateUp ? table[(it.seg0 & 3) + rr] / a.topk : it.seg0 + rr;
  L.avoff = (int)(src * a.lda * 2) + 16 * ((lane & 7) ^ ((r >> 1) & 7));
  L.asrc = make_rsrc(a.act, (uint32_t)a.act_bytes);
  const int K2 = a.K >> 1;
  if (TILED) {
    // load i: the wavefront's KiB of k block 2 st + i
    const int nkt = a.K / kPxKT;
    const int64_t per_e = (int64_t)a.n_nt * nkt * 2048;
    L.wsrc = make_rsrc(reinterpret_cast<const uint32_t*>(a.wt) + (int64_t)it.e * per_e, (uint32_t)(per_e * 4));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      L.bvoff[i] = (it.nt * nkt + i) * 8192 + wave * 1024 + 16 * lane;
      L.bback[i] = i * 8192;
    }
    L.bstage = 16384;
    L.bw0 = 1024;
    L.bw1 = 8192;
  } else {
    // load i: rows 32 wave + 16 i .., 64 bytes (four 16-byte pieces) each,
    // piece XOR-swizzled by (row / 4) % 4
    L.wsrc = make_rsrc(reinterpret_cast<const uint32_t*>(a.wp) + (int64_t)it.e * a.N * (a.K >> 3),
                       (uint32_t)a.N * K2);
    const int piece = (lane & 3) ^ ((lane >> 4) & 3);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      L.bvoff[i] = px_weight_row<MODE>(a, it.nt, 32 * wave + 16 * i + (lane >> 2)) * K2 + 16 * piece;
      L.bback[i] = piece >= 2 ? 32 : 0;
    }
    L.bstage = kPxKT;
    L.bw0 = 2048;
    L.bw1 = 1024;
  }
  return L;
}

// The loads of a tail item's stage st (k blocks 2 st and 2 st + 1 of 64) into
// ring slot `slot`.  When K / 64 is odd the last stage has only the first of
// the two: what would come from past the row comes from the first again.
template <int MBT>
__device__ __forceinline__ void px_issue_t(const PrefillArgs& a, const PxLoadsT& L, unsigned char* smem, int st,
                                           int slot) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  unsigned char* dst = smem + slot * px_tail_stage(MBT);
  const int two = 2 * st + 1 < a.K / kPxKT ? 1 : 0;
  if (MBT == 1) {
    const int hf = wave >> 2;
    px_dma16(L.asrc, L.avoff, (2 * st + hf * two) * (kPxKT * 2), dst + hf * 4096 + (wave & 3) * 1024);
  } else {
#pragma unroll
    for (int hf = 0; hf < 2; ++hf)
      px_dma16(L.asrc, L.avoff, (2 * st + hf * two) * (kPxKT * 2), dst + hf * 8192 + wave * 1024);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
    px_dma16(L.wsrc, L.bvoff[i] - (two ? 0 : L.bback[i]), st * L.bstage,
             dst + px_tail_b(MBT) + wave * L.bw0 + i * L.bw1);
}

// One contiguous block of scales (rows row0 .. of expert e) into LDS at dst,
// from the 16-byte boundary at or before it.
__device__ __forceinline__ void px_issue_scale_block(const PrefillArgs& a, int e, int row0, int rows,
                                                     unsigned char* dst) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uintptr_t p = reinterpret_cast<uintptr_t>(a.ws + ((int64_t)e * a.N + row0) * a.ng);
  const int bytes = (int)(p & 15) + rows * a.ng * 2;
  const __amdgpu_buffer_rsrc_t src = make_rsrc(reinterpret_cast<const void*>(p & ~uintptr_t(15)), (uint32_t)(bytes + 15) & ~15u);
  for (int i = wave; i * 1024 < bytes; i += kPxWaves) px_dma16(src, i * 1024 + 16 * lane, 0, dst + i * 1024);
}

// Issues a tail item's scales and its stages 0 and 1; returns the wavefront's
// loads per stage.
template <int MODE, bool TILED, int MBT>
__device__ __forceinline__ int px_issue_first_t(const PrefillArgs& a, const PxItem& it, unsigned char* smem) {
  const PxLoadsT L = px_loads_t<MODE, TILED, MBT>(a, it, smem);
  unsigned char* s0 = smem + kPxTailRing * px_tail_stage(MBT);
  if (MODE == kModeGateUp) {
    const int cols = min(128, a.I - 128 * it.nt);
    px_issue_scale_block(a, it.e, 128 * it.nt, cols, s0);
    px_issue_scale_block(a, it.e, a.I + 128 * it.nt, cols, smem + a.tail_s1[MBT - 1]);
  } else {
    px_issue_scale_block(a, it.e, kPxBN * it.nt, min(kPxBN, a.N - kPxBN * it.nt), s0);
  }
  px_issue_t<MBT>(a, L, smem, 0, 0);
  px_issue_t<MBT>(a, L, smem, 1, 1);
  return MBT + 2;
}

// Issues an item's stages 0 and 1 (into the first two ring slots); returns
// the wavefront's loads per stage.  Gate_up: the LDS table holds the item's
// rows.  Every wavefront is past its last LDS read of the item before.
template <int MODE, bool TILED>
__device__ __forceinline__ int px_issue_first(const PrefillArgs& a, const PxItem& it, unsigned char* smem) {
  if (TILED && it.nb > 1) {
    const PxLoadsW L = px_loads_w<MODE>(a, it, smem);
#pragma unroll
    for (int p = 0; p < 4; ++p) px_issue_w(a, L, smem, 0, 0, p);
#pragma unroll
    for (int p = 0; p < 4; ++p) px_issue_w(a, L, smem, 1, 1, p);
    return L.n;
  }
  if (px_is_tail(a, it)) {
    if (it.mb == 1) return px_issue_first_t<MODE, TILED, 1>(a, it, smem);
    return px_issue_first_t<MODE, TILED, 2>(a, it, smem);
  }
  const PxLoads L = px_loads<MODE, TILED>(a, it, smem);
  px_issue_all(a, L, smem, 0, 0);
  px_issue_all(a, L, smem, 1, 1);
  return L.n;
}

// The output of one group of 32 weight rows (wg) of an item for MB m-blocks
// from block mo on.  Lane l holds, for activation row 32 mb + c of block mb,
// the group's weight rows 8 J + 4 h + i in acc[mb][4 J + i] (J, i = 0..3):
// four consecutive output columns per J.  gate_up stores them as 8 bytes from
// registers: weight rows 0..15 are the gate rows and 16..31 their up rows, so
// acc[mb][q] (gate) pairs with acc[mb][q + 8] (up).
template <int MODE, int MB>
__device__ __forceinline__ void px_store(const PrefillArgs& a, unsigned char* smem, const PxItem& it, int wg, int mo,
                                         const f32x16_t* acc) {
  int lane = threadIdx.x & 63;
  // what the epilogue derives from the lane is formed here: hoisted out of
  // the item loop for every form of item it took registers that spilled in
  // down (3 tiled, 8 packed), and a reload here waits for every load and
  // store in flight (777 packed tokens, G = 32, skewed: 222.2 -> 215.7 us)
  asm volatile("" : "+v"(lane));
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 5, c = lane & 31;
  if (MODE == kModeGateUp) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int grow = 32 * (mo + mb) + c;
      if (grow >= it.nrows) continue;
      uint16_t* orow = a.out + (int64_t)(it.seg0 + grow) * a.ldo + 128 * it.nt + 16 * wg + 4 * h;
#pragma unroll
      for (int J = 0; J < 2; ++J) {
        float hv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float g = round_bf16(acc[mb][4 * J + i]);
          const float u = round_bf16(acc[mb][4 * J + i + 8]);
          hv[i] = round_bf16(gelu_tanh_f32(g)) * u;
        }
        *reinterpret_cast<uint2*>(orow + 8 * J) = make_uint2(pack_bf16x2(hv[0], hv[1]), pack_bf16x2(hv[2], hv[3]));
      }
    }
  } else {
    // dn rows are long (N columns, rows scattered by sorted_pos): the
    // group's 32 columns of each row go out as 16-byte stores, through LDS
    // one m-block at a time (the wavefront reads only what it wrote: no
    // barrier)
    const int* table = reinterpret_cast<const int*>(smem + kPxTable);
    unsigned char* ob = smem + kPxEpiOff + wave * kPxEpiBytes;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
      for (int J = 0; J < 4; ++J)
        *reinterpret_cast<uint2*>(ob + c * kPxEpiPitch + 2 * (8 * J + 4 * h)) =
            make_uint2(pack_bf16x2(acc[mb][4 * J], acc[mb][4 * J + 1]), pack_bf16x2(acc[mb][4 * J + 2], acc[mb][4 * J + 3]));
#pragma unroll
      for (int itr = 0; itr < 2; ++itr) {
        const int idx = lane + 64 * itr;
        const int row = idx >> 2, q4 = idx & 3;
        const int grow = 32 * (mo + mb) + row;
        if (grow < it.nrows) {
          const u32x4_t v = *reinterpret_cast<const u32x4_t*>(ob + row * kPxEpiPitch + 16 * q4);
          st16(a.out + (int64_t)table[(it.seg0 & 3) + grow] * a.N + kPxBN * it.nt + 32 * wg + 8 * q4, v);
        }
      }
    }
  }
}

// Multiply one item.  On entry its stages 0 and 1 are issued into slots 0
// and 1 (this wavefront's n_inflight loads each; gate_up: the LDS table
// holds the item's rows).  After its last stage it issues the next item's
// stages 0 and 1 (when has_next) and returns their per-stage load count;
// the epilogue runs while they land.
// SPLIT (gate_up's last n-tile when I % 128 == 64: only wavefronts 0..3
// have columns): wavefront w multiplies the weight rows of wavefront w % 4
// with m-blocks MB (w / 4) .. + MB - 1 of the item's 2 MB, so all eight
// wavefronts share the work instead of four idling.
// With fetch_q (non-null) wavefront 0 takes an index from that queue
// counter during the last stage (no stage load is issued after it, so the
// stage's vmcnt(0) wait covers it) and leaves it in LDS at kPxQSlot.
template <int MODE, bool TILED, int MB, bool SPLIT = false>
__device__ __forceinline__ int px_run(const PrefillArgs& a, unsigned char* smem, const PxItem& it,
                                      const PxItem& nx, bool has_next, int n_inflight,
                                      int* fetch_q) {
  static_assert(!SPLIT || MODE == kModeGateUp, "only gate_up has half n-tiles");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wg = SPLIT ? (wave & 3) : wave;      // weight rows 32 wg .. of the tile
  const int mo = SPLIT ? (wave >> 2) * MB : 0;   // first m-block
  const int nkt = a.K / kPxKT;
  const int h = lane >> 5;  // which half of the step's 16 k this lane holds
  const int c = lane & 31;  // row (A) / column (B) inside a 32-block
  const int gshift = a.gshift;
  const int nt = it.nt, seg0 = it.seg0;

  // this lane's reads: A fragment of block mb, step s -> row 32 mb + c,
  // chunk 4 h + s at slot chunk ^ ((c / 2) % 8); B words and scale pair of
  // tile row 32 wave + c
  int aoff[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) aoff[s] = mo * 4096 + c * 128 + 16 * ((4 * h + s) ^ ((c >> 1) & 7));
  const int boff = kPxBOff + (32 * wg + c) * 32 + 16 * h;
  // the scale chunk of tile row 32 wave + c; the pair sits at byte
  // (2 (row ng + pair group)) % 16 of it
  const int soff = kPxSOff + (32 * wg + c) * 16;
  const int srow2 = (int)(reinterpret_cast<uintptr_t>(a.ws + (int64_t)it.e * a.N * a.ng) & 15) +
                    px_weight_row<MODE>(a, nt, 32 * wg + c) * a.ng * 2;
  auto soff_of = [&](int t) -> int { return soff + ((srow2 + 2 * (((t * kPxKT) >> gshift) & ~1)) & 15); };
  // wavefronts whose columns lie past the matrix (gate_up's last n-tile
  // when I % 128 == 64) do no MFMA work and store nothing
  const bool work = SPLIT || (MODE == kModeGateUp ? 128 * nt + 16 * wave < a.I : kPxBN * nt + 32 * wave < a.N);

  f32x16_t acc[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[i][q] = 0.f;

  auto scale_of = [&](int t, uint32_t sp) -> float {
    const int g = (t * kPxKT + 32 * h) >> gshift;
    const int sel = g - (((t * kPxKT) >> gshift) & ~1);  // 0 or 1
    return bf16_bits_to_f32((sp >> (16 * sel)) & 0xFFFFu);
  };
  auto read_a = [&](const unsigned char* st, int s, u32x4_t* af) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) af[mb] = *reinterpret_cast<const u32x4_t*>(st + mb * 4096 + aoff[s]);
  };
  // D[weight row][activation row]: the dequantised weights are the MFMA's A
  // operand, the activation rows its B operand
  auto mfmas = [&](const u32x4_t* af, u32x4_t bf) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[mb] = mfma32(bf, af[mb], acc[mb]);
  };
  auto stage_ptr = [&](int sl) -> const unsigned char* { return smem + sl * kPxStageBytes; };
  // the loads issued after the awaited stage: those of the stage issued in
  // this iteration (n of them)
  auto no_hook = [] {};
  // hook: runs after the wait, before the barrier (its LDS writes are seen
  // by every wavefront after it)
  auto wait_and_sync = [&](int n, auto hook) {
    __builtin_amdgcn_sched_barrier(0);
    px_wait_vm(n);
    __builtin_amdgcn_sched_barrier(0);
    hook();
    px_barrier();
  };

  wait_and_sync(n_inflight, no_hook);  // stage 0 landed (stage 1 may still be loading)
  // Software pipeline: each A fragment register is reloaded with the next
  // step's fragment right after the MFMA that reads it, and the next step's
  // B fragment is dequantised while the current step's MFMAs run.  Stage
  // t's last-step fragments are in registers before the barrier that ends
  // the stage, so after it each MFMA of that step is followed by the read
  // of stage t + 1's first fragment for the same block.
  u32x4_t af[MB];
  u32x4_t bw = {0u, 0u, 0u, 0u};
  float sc = 0.f;
  const ExactRegs kr = exact_regs();
  if (work) {
    read_a(stage_ptr(0), 0, af);
    bw = *reinterpret_cast<const u32x4_t*>(stage_ptr(0) + boff);
    sc = scale_of(0, *reinterpret_cast<const uint32_t*>(stage_ptr(0) + soff_of(0)));
  }
  int slot = 0;
  int slot2 = 2;
  // one k stage: refill the slot stage t - 1 used (issue(slot2)), multiply
  // stage t, wait for stage t + 1 and meet the other wavefronts
  auto iter = [&](int t, int n, auto issue, auto hook) {
    const int nslot = slot == kPxStages - 1 ? 0 : slot + 1;
    if (work) {
      const unsigned char* st = stage_ptr(slot);
      const ExactScale es = exact_scale(sc);
      const uint32_t wv[4] = {bw.x, bw.y, bw.z, bw.w};
      u32x4_t bf = unpack_exact<false>(wv[0], es, kr);
#pragma unroll
      for (int s2 = 0; s2 < 3; ++s2) {
        issue(slot2, s2);
        const u32x4_t bfn = unpack_exact<false>(wv[s2 + 1], es, kr);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          acc[mb] = mfma32(bf, af[mb], acc[mb]);
          af[mb] = *reinterpret_cast<const u32x4_t*>(st + mb * 4096 + aoff[s2 + 1]);
        }
        bf = bfn;
      }
      issue(slot2, 3);
      wait_and_sync(n, hook);  // stage t + 1 landed (stage t + 2 may still be loading)
      if (t + 1 < nkt) {
        const unsigned char* sn = stage_ptr(nslot);
        bw = *reinterpret_cast<const u32x4_t*>(sn + boff);
        const uint32_t sp = *reinterpret_cast<const uint32_t*>(sn + soff_of(t + 1));
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          acc[mb] = mfma32(bf, af[mb], acc[mb]);
          af[mb] = *reinterpret_cast<const u32x4_t*>(sn + mb * 4096 + aoff[0]);
        }
        sc = scale_of(t + 1, sp);
      } else {
        mfmas(af, bf);
      }
    } else {
#pragma unroll
      for (int p = 0; p < 4; ++p) issue(slot2, p);
      wait_and_sync(n, hook);
    }
    slot = nslot;
    slot2 = slot2 == kPxStages - 1 ? 0 : slot2 + 1;
  };
  {
    const PxLoads lc = px_loads<MODE, TILED>(a, it, smem);
    for (int t = 0; t + 2 < nkt; ++t)
      iter(t, lc.n, [&](int sl, int p) { px_issue(a, lc, smem, t + 2, sl, p); }, no_hook);
  }
  // the last two stages issue no stage loads; the second-to-last brings the
  // row-index table (gate_up: the next item's rows, for its load sources;
  // down: this item's output rows, for its epilogue)
  const int tseg = MODE == kModeGateUp ? (has_next ? nx.seg0 : seg0) : seg0;
  iter(nkt - 2, 1, [&](int, int p) {
    if (p == 0) px_issue_table(a, smem, tseg);
  }, no_hook);
  const bool fetch = fetch_q != nullptr && wave == 0;  // wavefront-uniform
  int fv = 0;
  iter(nkt - 1, 0,
       [&](int, int p) {
         if (p == 0 && fetch && lane == 0) fv = __hip_atomic_fetch_add(fetch_q, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
       },
       [&] {
         if (fetch && lane == 0) *reinterpret_cast<int*>(smem + kPxQSlot) = fv;
       });
  // every wavefront is past its last LDS read: the next item's first stages
  const int n_next = has_next ? px_issue_first<MODE, TILED>(a, nx, smem) : 0;
  if (work) px_store<MODE, MB>(a, smem, it, wg, mo, acc);
  return n_next;
}

// Multiply one wide item (kPxWide n-tiles of a tail of at most 32 rows), in
// px_run's stage protocol.  Each n-tile's outputs are px_run<MODE, TILED, 1>'s for
// that n-tile bit for bit: the same MFMA on the same operands, one k step
// after the other.
template <int MODE, bool TILED>
__device__ __forceinline__ int px_run_w(const PrefillArgs& a, unsigned char* smem, const PxItem& it,
                                        const PxItem& nx, bool has_next, int n_inflight,
                                        int* fetch_q) {
  constexpr int NB = kPxWide;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nkt = a.K / kPxKT;
  const int h = lane >> 5;
  const int c = lane & 31;
  const int gshift = a.gshift;
  const int nt0 = it.nt, seg0 = it.seg0;

  int aoff[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) aoff[s] = c * 128 + 16 * ((4 * h + s) ^ ((c >> 1) & 7));
  int boff[NB], soffb[NB], srow2[NB];
  const int sb15 = (int)(reinterpret_cast<uintptr_t>(a.ws + (int64_t)it.e * a.N * a.ng) & 15);
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    boff[b] = px_wide_b(b) + (32 * wave + c) * 32 + 16 * h;
    soffb[b] = px_wide_s(b) + (32 * wave + c) * 16;
    srow2[b] = sb15 + px_weight_row<MODE>(a, nt0 + b, 32 * wave + c) * a.ng * 2;
  }
  f32x16_t acc[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[b][q] = 0.f;
  auto scale_of = [&](int t, uint32_t sp) -> float {
    const int g = (t * kPxKT + 32 * h) >> gshift;
    const int sel = g - (((t * kPxKT) >> gshift) & ~1);  // 0 or 1
    return bf16_bits_to_f32((sp >> (16 * sel)) & 0xFFFFu);
  };
  auto stage_ptr = [&](int sl) -> const unsigned char* { return smem + sl * kPxStageBytes; };
  auto no_hook = [] {};
  auto wait_and_sync = [&](int n, auto hook) {
    __builtin_amdgcn_sched_barrier(0);
    px_wait_vm(n);
    __builtin_amdgcn_sched_barrier(0);
    hook();
    px_barrier();
  };
  const ExactRegs kr = exact_regs();

  wait_and_sync(n_inflight, no_hook);  // stage 0 landed
  int slot = 0;
  int slot2 = 2;
  // one k stage: read its words and scales, refill the slot stage t - 1 used
  // (issue(slot2)) while multiplying, wait for stage t + 1 and meet
  auto iter = [&](int t, int n, auto issue, auto hook) {
    const unsigned char* st = stage_ptr(slot);
    u32x4_t bw[NB];
    ExactScale es[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      bw[b] = *reinterpret_cast<const u32x4_t*>(st + boff[b]);
      const int so = soffb[b] + ((srow2[b] + 2 * (((t * kPxKT) >> gshift) & ~1)) & 15);
      es[b] = exact_scale(scale_of(t, *reinterpret_cast<const uint32_t*>(st + so)));
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      issue(slot2, s);
      const u32x4_t af = *reinterpret_cast<const u32x4_t*>(st + aoff[s]);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const uint32_t w = s == 0 ? bw[b].x : s == 1 ? bw[b].y : s == 2 ? bw[b].z : bw[b].w;
        acc[b] = mfma32(unpack_exact<false>(w, es[b], kr), af, acc[b]);
      }
    }
    wait_and_sync(n, hook);  // stage t + 1 landed (stage t + 2 may still be loading)
    slot = slot == kPxStages - 1 ? 0 : slot + 1;
    slot2 = slot2 == kPxStages - 1 ? 0 : slot2 + 1;
  };
  {
    const PxLoadsW lc = px_loads_w<MODE>(a, it, smem);
    for (int t = 0; t + 2 < nkt; ++t)
      iter(t, lc.n, [&](int sl, int p) { px_issue_w(a, lc, smem, t + 2, sl, p); }, no_hook);
  }
  const int tseg = MODE == kModeGateUp ? (has_next ? nx.seg0 : seg0) : seg0;
  iter(nkt - 2, 1, [&](int, int p) {
    if (p == 0) px_issue_table(a, smem, tseg);
  }, no_hook);
  const bool fetch = fetch_q != nullptr && wave == 0;  // wavefront-uniform
  int fv = 0;
  iter(nkt - 1, 0,
       [&](int, int p) {
         if (p == 0 && fetch && lane == 0) fv = __hip_atomic_fetch_add(fetch_q, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
       },
       [&] {
         if (fetch && lane == 0) *reinterpret_cast<int*>(smem + kPxQSlot) = fv;
       });
  const int n_next = has_next ? px_issue_first<MODE, TILED>(a, nx, smem) : 0;

  // n-tiles past the matrix, and gate_up columns past I, store nothing
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    PxItem one = it;
    one.nt = nt0 + b;
    if (px_group_real<MODE>(a, one.nt, wave)) px_store<MODE, 1>(a, smem, one, wave, 0, &acc[b]);
  }
  return n_next;
}

// Multiply one tail item of MBT = MB WM m-blocks (WM = 2: gate_up's last
// n-tile when I % 128 == 64, its four groups shared by the two wavefront
// halves, a row block each), in px_run's protocol with stages of 128 k.  Few
// rows give the matrix cores little work per weight, so what counts is that
// the weights' stream and the dequantisation seldom wait: the item's scales
// are read once, as one contiguous block (a stage's own 16-byte chunks would
// touch a cache line per weight row and stage), and a stage takes 64
// consecutive bytes of each packed row.  Each output is the sum px_run forms,
// in the same order, bit for bit.
template <int MODE, bool TILED, int MB, int WM = 1>
__device__ __forceinline__ int px_run_t(const PrefillArgs& a, unsigned char* smem, const PxItem& it,
                                        const PxItem& nx, bool has_next, int* fetch_q) {
  constexpr int MBT = MB * WM;
  constexpr int n = MBT + 2;  // loads per stage
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wg = WM == 2 ? (wave & 3) : wave;
  const int mo = WM == 2 ? (wave >> 2) * MB : 0;
  const int h = lane >> 5, c = lane & 31;
  const int nkt = a.K / kPxKT, nst = (nkt + 1) >> 1;
  const bool work = px_group_real<MODE>(a, it.nt, wg);
  const PxLoadsT lc = px_loads_t<MODE, TILED, MBT>(a, it, smem);

  // step s (0..7) of a stage: half s / 4, chunk 4 h + s % 4 of row c
  int aoff[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) aoff[s] = mo * 4096 + c * 128 + 16 * ((4 * h + s) ^ ((c >> 1) & 7));
  int boff[2];
#pragma unroll
  for (int hf = 0; hf < 2; ++hf)
    boff[hf] = px_tail_b(MBT) + (TILED ? hf * 8192 + (32 * wg + c) * 32 + 16 * h
                                                 : (32 * wg + c) * 64 + 16 * ((2 * hf + h) ^ ((c >> 2) & 3)));
  // this lane's row of scales
  const int row0 = MODE == kModeGateUp ? (c < 16 ? 0 : a.I) + 128 * it.nt : kPxBN * it.nt;
  const unsigned char* srow =
      smem + (int)(reinterpret_cast<uintptr_t>(a.ws + ((int64_t)it.e * a.N + row0) * a.ng) & 15) +
      (px_weight_row<MODE>(a, it.nt, 32 * wg + c) - row0) * a.ng * 2 +
      (MODE == kModeGateUp && c >= 16 ? a.tail_s1[MBT - 1] : kPxTailRing * px_tail_stage(MBT));

  f32x16_t acc[MB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[i][q] = 0.f;
  const ExactRegs kr = exact_regs();
  u32x4_t af[MB], bw[2], bf;
  float sc[2];
  auto read_a = [&](const unsigned char* p, int s, int mb) {
    return *reinterpret_cast<const u32x4_t*>(p + (s >> 2) * MBT * 4096 + mb * 4096 + aoff[s & 3]);
  };
  // a stage's words and scales (past K: the last group's, not used)
  auto read_b = [&](const unsigned char* p, int st) {
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
      bw[hf] = *reinterpret_cast<const u32x4_t*>(p + boff[hf]);
      const int g = min(((2 * st + hf) * kPxKT + 32 * h) >> a.gshift, a.ng - 1);
      sc[hf] = bf16_bits_to_f32(*reinterpret_cast<const uint16_t*>(srow + 2 * g));
    }
  };
  auto word = [&](int s) {
    const u32x4_t v = bw[s >> 2];
    return (s & 3) == 0 ? v.x : (s & 3) == 1 ? v.y : (s & 3) == 2 ? v.z : v.w;
  };
  auto stage_ptr = [&](int sl) -> const unsigned char* { return smem + sl * px_tail_stage(MBT); };
  int slot = 0, slot2 = 2;
  // one stage of NS steps: issue() fills slot2, the wait leaves VM loads in
  // flight
  auto stage = [&](int t, auto ns, auto vm, auto issue, auto hook) {
    constexpr int NS = decltype(ns)::value;
    const int nslot = slot == kPxTailRing - 1 ? 0 : slot + 1;
    issue(slot2);
    if (work) {
      const unsigned char* p = stage_ptr(slot);
#pragma unroll
      for (int s = 0; s < NS - 1; ++s) {
        const u32x4_t bn = unpack_exact<false>(word(s + 1), exact_scale(sc[(s + 1) >> 2]), kr);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
          acc[mb] = mfma32(bf, af[mb], acc[mb]);
          af[mb] = read_a(p, s + 1, mb);
        }
        bf = bn;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(px_vm_wait(decltype(vm)::value));
    hook();
    px_barrier();
    if (work) {
      const unsigned char* p = stage_ptr(nslot);
      if (t + 1 < nst) read_b(p, t + 1);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        acc[mb] = mfma32(bf, af[mb], acc[mb]);
        if (t + 1 < nst) af[mb] = read_a(p, 0, mb);
      }
      if (t + 1 < nst) bf = unpack_exact<false>(word(0), exact_scale(sc[0]), kr);
    }
    slot = nslot;
    slot2 = slot2 == kPxTailRing - 1 ? 0 : slot2 + 1;
  };
  const std::integral_constant<int, 8> full;
  const std::integral_constant<int, 4> half;
  const std::integral_constant<int, 0> all;
  auto no_hook = [] {};

  __builtin_amdgcn_s_waitcnt(px_vm_wait(n));
  px_barrier();  // the scales and stage 0 landed (stage 1 may still be loading)
  if (work) {
    read_b(stage_ptr(0), 0);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) af[mb] = read_a(stage_ptr(0), 0, mb);
    bf = unpack_exact<false>(word(0), exact_scale(sc[0]), kr);
  }
  for (int t = 0; t + 2 < nst; ++t)
    stage(t, full, std::integral_constant<int, n>{}, [&](int sl) { px_issue_t<MBT>(a, lc, smem, t + 2, sl); }, no_hook);
  // the last two stages refill nothing; the first of them brings the row
  // indices (gate_up: the next item's rows, for its load sources; down: this
  // item's output rows), the last takes the queue's next index
  stage(nst - 2, full, std::integral_constant<int, 1>{}, [&](int) {
    px_issue_table(a, smem, MODE == kModeGateUp && has_next ? nx.seg0 : it.seg0);
  }, no_hook);
  const bool fetch = fetch_q != nullptr && wave == 0;  // wavefront-uniform
  int fv = 0;
  auto take = [&](int) {
    if (fetch && lane == 0) fv = __hip_atomic_fetch_add(fetch_q, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  auto put = [&] {
    if (fetch && lane == 0) *reinterpret_cast<int*>(smem + kPxQSlot) = fv;
  };
  if (nkt & 1)
    stage(nst - 1, half, all, take, put);
  else
    stage(nst - 1, full, all, take, put);
  const int n_next = has_next ? px_issue_first<MODE, TILED>(a, nx, smem) : 0;
  if (work) px_store<MODE, MB>(a, smem, it, wg, mo, acc);
  return n_next;
}

template <int MODE, bool TILED>
__device__ __forceinline__ int px_dispatch(const PrefillArgs& a, unsigned char* smem, const PxItem& it,
                                           const PxItem& nx, bool has_next, int n_inflight, int* fetch_q) {
  if constexpr (TILED)
    if (it.nb > 1) return px_run_w<MODE, TILED>(a, smem, it, nx, has_next, n_inflight, fetch_q);
  // gate_up's half n-tile: eight wavefronts on four wavefronts' columns
  const bool half = MODE == kModeGateUp && a.I - 128 * it.nt == 64;
  if (px_is_tail(a, it)) {
    if (it.mb == 1) return px_run_t<MODE, TILED, 1>(a, smem, it, nx, has_next, fetch_q);
    if constexpr (MODE == kModeGateUp)
      if (half) return px_run_t<MODE, TILED, 1, 2>(a, smem, it, nx, has_next, fetch_q);
    return px_run_t<MODE, TILED, 2>(a, smem, it, nx, has_next, fetch_q);
  }
  if constexpr (MODE == kModeGateUp) {
    if (half && it.mb >= 2) {
      if (it.mb >= 7) return px_run<MODE, TILED, 4, true>(a, smem, it, nx, has_next, n_inflight, fetch_q);
      if (it.mb >= 5) return px_run<MODE, TILED, 3, true>(a, smem, it, nx, has_next, n_inflight, fetch_q);
      if (it.mb >= 3) return px_run<MODE, TILED, 2, true>(a, smem, it, nx, has_next, n_inflight, fetch_q);
      return px_run<MODE, TILED, 1, true>(a, smem, it, nx, has_next, n_inflight, fetch_q);
    }
  }
  switch (it.mb) {
    case 8: return px_run<MODE, TILED, 8>(a, smem, it, nx, has_next, n_inflight, fetch_q);
    case 7: return px_run<MODE, TILED, 7>(a, smem, it, nx, has_next, n_inflight, fetch_q);
    case 6: return px_run<MODE, TILED, 6>(a, smem, it, nx, has_next, n_inflight, fetch_q);
    case 5: return px_run<MODE, TILED, 5>(a, smem, it, nx, has_next, n_inflight, fetch_q);
    case 4: return px_run<MODE, TILED, 4>(a, smem, it, nx, has_next, n_inflight, fetch_q);
    case 3: return px_run<MODE, TILED, 3>(a, smem, it, nx, has_next, n_inflight, fetch_q);
    case 2: return px_run<MODE, TILED, 2>(a, smem, it, nx, has_next, n_inflight, fetch_q);
    default: return px_run<MODE, TILED, 1>(a, smem, it, nx, has_next, n_inflight, fetch_q);
  }
}

// Persistent grid, one workgroup per CU.  down: local item i of XCD x is
// n-tile i % n_nt of the XCD's m-tile i / n_nt, tile list entry x + 8 (i /
// n_nt), so an m-tile's activation rows are read into one L2 for its 11
// n-tiles; workgroup b of XCD x = b % 8 takes local items b / 8 and b / 8 +
// P (P = workgroups per XCD), then the items that XCD's queue counter
// (queues[x]) hands out, 2 P, 2 P + 1, ...  gate_up: item i is n-tile i %
// n_nt of tile list entry i / n_nt, workgroup b takes items b and b + P (P
// = all workgroups), then those of the one queue (queues[0]): its items
// differ more in cost (segment tails, the half n-tile) and the XCDs in
// speed, and the whole chip draining one queue ends them closer together
// than the rows kept in one L2 save.  The list runs from large tiles to
// small but for the tails of at most kPrefillTinyRows rows, which stand before
// the other tails: as wide items they are the longer ones and are taken there,
// as tail items last (px_item_info).  Workgroups ask in the order they get
// there, during the last stage of the item before their next one, so the
// index is known one item ahead (the next item's rows and first stages are
// loaded during the current one).  queues[8] counts the workgroups that
// have left; the expert sort zeroes the counters and the last workgroup to
// leave resets them.  Without queues the deal is fixed: items b + r P.
template <int MODE, bool TILED>
__global__ __launch_bounds__(kPxThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_prefill_x(PrefillArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int ntiles = ld_uniform(a.counters, 1);
  const int tiny0 = ld_uniform(a.counters, 2), tiny1 = ld_uniform(a.counters, 3);  // the smallest tails
  constexpr bool kChip = MODE == kModeGateUp;  // one queue for the chip
  const int x0 = kChip ? 0 : (int)(blockIdx.x & 7);
  const int xs = kChip ? 1 : 8;
  const int n_local = kChip ? ntiles : (ntiles > x0 ? (ntiles - x0 + 7) >> 3 : 0);  // the queue's m-tiles
  // the queue's m-tiles before list entry b
  auto local = [&](int b) { return kChip ? b : (b > x0 ? (b - x0 + 7) >> 3 : 0); };
  const int t0 = local(tiny0), t1 = local(tiny1);
  // Wide items where the m-tiles are smallest tails but for one in fifty: of
  // like length, they go round once.  Among other items their own length (two
  // to three times a tail's) shows at the end: at the Gemma shape, tiled, G =
  // 128 / 32, as wide / tail items, 257 tokens of flat routing 139/155,
  // 160/163 us; 400 tokens 167/158, 191/166; 257 tokens skewed 182/173,
  // 206/178; 1536 tokens skewed 311/280, 325/283.
  const int n_wide = TILED && 50 * (tiny1 - tiny0) >= 49 * ntiles ? (a.n_nt + kPxWide - 1) / kPxWide : 0;
  const int it_end = (n_local - (t1 - t0)) * a.n_nt + (t1 - t0) * (n_wide > 0 ? n_wide : a.n_nt);
  const int P = kChip ? (int)gridDim.x : (int)(gridDim.x >> 3);
  int* const queue = a.queues != nullptr ? a.queues + x0 : nullptr;
  // the last workgroup to leave resets the counters for the next launch
  // (every other one has taken its last index before counting itself out)
  auto leave = [&] {
    if (a.queues == nullptr || threadIdx.x != 0) return;
    const int d = __hip_atomic_fetch_add(a.queues + 8, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (d == (int)gridDim.x - 1) {
#pragma unroll
      for (int x = 0; x < 9; ++x) __hip_atomic_store(a.queues + x, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  };
  int item = kChip ? (int)blockIdx.x : (int)(blockIdx.x >> 3);
  if (item >= it_end) {
    leave();
    return;
  }
  PxItem cur = px_item_info(a, x0, xs, n_local, t0, t1, n_wide, item);
  if (MODE == kModeGateUp) {
    // the first item's gathered rows into the table (nothing else in flight)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const __amdgpu_buffer_rsrc_t tsrc = make_rsrc(a.sorted_pos, (uint32_t)a.rows_total * 4u);
    if (wave < 2) px_dma16(tsrc, 4 * ((cur.seg0 & ~3) + 256 * wave + 4 * lane), 0, smem + kPxTable + 1024 * wave);
    __builtin_amdgcn_s_waitcnt(px_vm_wait(0));
    px_barrier();
  }
  int n_inflight = px_issue_first<MODE, TILED>(a, cur, smem);
  int nitem = item + P;
  for (;;) {
    const bool has_next = nitem < it_end;
    const PxItem nxt = has_next ? px_item_info(a, x0, xs, n_local, t0, t1, n_wide, nitem) : cur;
    // with a next item, take the index of the one after it during this item
    n_inflight = px_dispatch<MODE, TILED>(a, smem, cur, nxt, has_next, n_inflight, has_next ? queue : nullptr);
    if (!has_next) break;
    item = nitem;
    nitem = queue != nullptr ? 2 * P + __builtin_amdgcn_readfirstlane(*reinterpret_cast<volatile int*>(smem + kPxQSlot))
                             : item + P;
    cur = nxt;
  }
  // the loads issued past the last stage land before the workgroup leaves
  __builtin_amdgcn_s_waitcnt(px_vm_wait(0));
  leave();
}

// The tiled weight copy: piece (e, nt, kt, tr, h) = 16 bytes of weight row
// px_weight_row(nt, tr) at byte 32 kt + 16 h, so stage kt of n-tile nt is
// 8 KiB in the order the kernel's B loads fill LDS (tile row tr at 32 tr).
template <int MODE>
__global__ __launch_bounds__(256) void k_tile_prefill(const uint32_t* __restrict__ packed,
                                                      uint32_t* __restrict__ tiled, PrefillArgs a,
                                                      int64_t pieces) {
  const int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (p >= pieces) return;
  const int nkt = a.K / kPxKT;
  const int h = (int)(p & 1);
  const int tr = (int)((p >> 1) & 255);
  int64_t q = p >> 9;
  const int kt = (int)(q % nkt);
  q /= nkt;
  const int nt = (int)(q % a.n_nt);
  const int64_t e = q / a.n_nt;
  const int row = px_weight_row<MODE>(a, nt, tr);
  const int64_t src = (e * a.N + row) * (int64_t)(a.K / 2) + 32 * kt + 16 * h;
  *reinterpret_cast<u32x4_t*>(tiled + p * 4) = *reinterpret_cast<const u32x4_t*>(packed + src / 4);
}

size_t prefill_tiled_bytes_per_expert(int mode, int64_t H, int64_t I) {
  if (H % kPxKT != 0 || I % kPxKT != 0 || H < 3 * kPxKT || I < 3 * kPxKT) return 0;
  const int64_t K = mode == kModeGateUp ? H : I;
  const int64_t n_nt = mode == kModeGateUp ? (I + 127) / 128 : (H + 255) / 256;
  return (size_t)(n_nt * (K / kPxKT) * 8192);
}

hipError_t launch_tile_prefill(int mode, const int32_t* packed, int E, int H, int I, int32_t* tiled,
                               hipStream_t s) {
  if (prefill_tiled_bytes_per_expert(mode, H, I) == 0) return hipErrorInvalidValue;
  PrefillArgs a{};
  a.I = I;
  a.N = mode == kModeGateUp ? 2 * I : H;
  a.K = mode == kModeGateUp ? H : I;
  a.n_nt = mode == kModeGateUp ? (I + 127) / 128 : (H + 255) / 256;
  const int64_t pieces = (int64_t)E * a.n_nt * (a.K / kPxKT) * 512;
  if (pieces == 0) return hipSuccess;
  const dim3 grid((unsigned)((pieces + 255) / 256));
  const uint32_t* src = reinterpret_cast<const uint32_t*>(packed);
  uint32_t* dst = reinterpret_cast<uint32_t*>(tiled);
  if (mode == kModeGateUp)
    hipLaunchKernelGGL(k_tile_prefill<kModeGateUp>, grid, dim3(256), 0, s, src, dst, a, pieces);
  else
    hipLaunchKernelGGL(k_tile_prefill<kModeDown>, grid, dim3(256), 0, s, src, dst, a, pieces);
  return hipGetLastError();
}

// persistent grid: the workgroups that fit on the device at once (a multiple
// of the 8 XCDs), at most one per item
int prefill_grid_size(const void* kern, int threads, size_t lds, int max_items) {
  int per_cu = 1;
  // more than half of a CU's LDS: one workgroup, nothing to ask the runtime
  if (2 * lds <= 160 * 1024 &&
      (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, threads, lds) != hipSuccess || per_cu <= 0))
    per_cu = 1;
  int g = device_cus() * per_cu;
  if (max_items < g) g = max_items;
  return ((g + 7) / 8) * 8;
}

size_t prefill_x_lds_bytes() { return (size_t)kPxLds; }

// H and I multiples of the 64-wide stage, at least three stages; G a power of two >= 32 whose
// group counts per row are even for both matrices (a stage's scale pair is
// one aligned dword)
bool prefill_x_supported(int64_t H, int64_t I, int64_t G) {
  if (H % kPxKT != 0 || I % kPxKT != 0 || H < 3 * kPxKT || I < 3 * kPxKT || G < 32 || (G & (G - 1)) != 0)
    return false;
  const int64_t ng_h = (H + G - 1) / G, ng_i = (I + G - 1) / G;
  return ng_h % 2 == 0 && ng_i % 2 == 0;
}

hipError_t launch_prefill_x(int mode, PrefillArgs a, int max_mtiles, hipStream_t s) {
  if (max_mtiles <= 0) return hipSuccess;
  // tail items where the ring leaves room for the item's scales (gate_up's
  // second block in the LDS that only down's epilogue uses if it fits there,
  // else behind the first) and K has three stages of 128; else px_run's
  // stages bring their own scales
  const int sb = (((mode == kModeGateUp ? 128 : kPxBN) * a.ng * 2 + 16) + 1023) / 1024 * 1024;
  for (int mbt = 1; mbt <= kPxTailMaxBlocks; ++mbt) {
    const int s0 = kPxTailRing * px_tail_stage(mbt);
    const bool apart = mode != kModeGateUp || sb <= kPxQSlot - kPxEpiOff;
    a.tail_s1[mbt - 1] = mode != kModeGateUp ? 0 : apart ? kPxEpiOff : s0 + sb;
    if (s0 + (apart ? 1 : 2) * sb > kPxTable || a.K <= 4 * kPxKT) a.tail_s1[mbt - 1] = -1;
  }
  const size_t lds = prefill_x_lds_bytes();
  auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(prefill_grid_size(reinterpret_cast<const void*>(kern), kPxThreads, lds,
                                                    max_mtiles * a.n_nt)),
                       dim3(kPxThreads), lds, s, a);
  };
  if (mode == kModeGateUp) {
    if (a.wt != nullptr)
      launch(k_prefill_x<kModeGateUp, true>);
    else
      launch(k_prefill_x<kModeGateUp, false>);
  } else {
    if (a.wt != nullptr)
      launch(k_prefill_x<kModeDown, true>);
    else
      launch(k_prefill_x<kModeDown, false>);
  }
  return hipGetLastError();
}

}  // namespace w4a16
