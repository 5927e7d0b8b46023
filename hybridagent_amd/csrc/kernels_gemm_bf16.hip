// bf16 x bf16 GEMMs at prefill sizes, for the weights that are not quantised:
//
//   grouped (the BF16 experts, backends.py:209-283, on the expert segments of
//   the MoE plan)
//     gate/up : inter[s] = bf16(bf16(gelu_tanh(bf16(x[tok(s)] Wg^T))) * bf16(x[tok(s)] Wu^T))
//     plain   : dn[sorted_pos[s]] = bf16(inter[s] Wd^T)
//   dense (the FFN block's shared MLP, backends.py:105-108)
//     gate/up : the same on all rows, gate rows from W and up rows from W2
//     plain   : out = bf16(x W^T)
//
// The streaming kernels (k_bf16_expert, k_linear_bf16) read a 16-column
// block's weights once per 64 rows and each activation row once per 16
// columns; past a few dozen rows per weight that traffic, through L2, is what
// they spend their time on.  Here a workgroup of eight wavefronts owns a tile
// of 256 weight rows (gate/up: 128 gate rows and the matching 128 up rows) x
// up to 160 activation rows, so a weight is read once per 160 rows (an
// expert's segment: once per 128) and an activation row once per 256 columns.
//
// k advances in stages of 64, both operands by direct global -> LDS loads of
// 16 bytes per lane through a ring of three stages (two in flight while one
// is multiplied), rows 128 bytes apart with the 16-byte chunks XOR-swizzled
// by (row / 2) % 8: the fragment reads of 16 consecutive rows cover all LDS
// banks once.  The multiply is v_mfma_f32_32x32x16_bf16 with the weights as
// the A operand (each lane ends with four consecutive output columns of one
// row per register quad).  Step s of a stage takes k = 16 s .. 16 s + 15, so
// a last half stage (K % 64 == 32) is two steps, and its loads of chunks
// past K are turned to the row's chunk four before.  Each fragment register
// is reloaded for the next step right after its last MFMA.  WM = 1: every
// wavefront has 32 weight rows x all MB blocks of 32 activation rows; WM = 2:
// 64 weight rows x half of the rows, which reads (MB + 2) fragments for 2 MB
// MFMAs instead of (MB + 1) for MB.
//
// The dense kernels are built per tile height.  The accumulators of a range
// and of the ranges before it are 160 registers at five blocks; they fit (no
// spills) because one path leads through the last stage, whole or half: two
// paths made the compiler hold a third set across their join.
//
// A workgroup goes from tile to tile without draining the ring: the next
// tile's first two stages are issued before the current one's epilogue.
// Grouped tiles come from one queue for the chip (the expert sort's list of
// 128-row tiles, each with all its column tiles); the dense launch deals
// every XCD a contiguous run of tiles, ordered so that the tiles running at
// once on an XCD share rows and columns.
//
// Every output is the streaming kernels' sum, bit for bit, whatever tile it
// falls in: K in the same ranges (GemmBf16Args::ranges), each range one fp32
// chain, the ranges added in order -- so a row's result does not change where a
// larger batch takes this kernel.  One 32x32x16 MFMA on chunks 0, 1 and one on
// chunks 2, 3 of 32 k give the bits of the 16x16x32 MFMA on all four (compared
// on 65,536 sums; every other order of the chunks differs).  A range's end
// costs 32 VALU per block of 32 rows and group of 32 weight rows: against one
// chain over all of K the FFN block at 2048 rows takes 492.8 us, not 490.4,
// and 1031 tokens of BF16 experts 380.5, not 379.5.
//
// Bound: the experts by their weights' stream (1031 tokens x top-8 over 128
// experts of 11.9 MB, flat routing: the call 1316 us streamed per 64 rows, 332
// here, 4.6 TB/s; skewed, Zipf 1.1: 1510 .. 1860 and 380).  The dense form by
// no one unit: gate/up of 2048 rows x 2 x 2112 (58 us, five blocks) has the
// MFMAs busy 35 % of the time and LDS 21 %, without bank conflicts; its
// wavefronts wait for loads and at the stage barrier for 30 % of theirs and to
// issue for 31 % (shared MLP of 2048 rows, 73 GFLOP: 830 us streamed, about 95
// here).
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "lds_pipe.hpp"
#include "rules.hpp"

namespace w4a16 {

namespace {

constexpr int kGxWaves = 8;
constexpr int kGxThreads = 64 * kGxWaves;
constexpr int kGxBN = 256;  // weight rows per tile
constexpr int kGxKT = 64;   // k per stage
constexpr int kGxMaxBlocks = kGemmMaxBlocks;  // 32-row blocks per tile
constexpr int kGxStages = 3;
// a stage: A [160 rows][128 B] | B [256 rows][128 B]; after the ring the row
// indices of a grouped tile (256 ints from a 16-byte-aligned start) and the
// tile index taken from the queue
constexpr int kGxB = 32 * kGxMaxBlocks * kGxKT * 2;
constexpr int kGxStageBytes = kGxB + kGxBN * kGxKT * 2;
constexpr int kGxTable = kGxStages * kGxStageBytes;
constexpr int kGxQSlot = kGxTable + 1024;
constexpr int kGxLds = kGxQSlot + 16;
static_assert(kGxLds <= 160 * 1024, "LDS of a CU");
// plain epilogue: 32 rows x 32 bf16 per wavefront, rows 80 bytes apart (the
// 8-byte writes of 32 rows spread over the banks), in the ring slot of the
// tile's last stage
constexpr int kGxEpiPitch = 80;
static_assert(kGxWaves * 32 * kGxEpiPitch <= kGxStageBytes, "epilogue rows fit in a slot");
constexpr int kGxNA = (4 * kGxMaxBlocks + kGxWaves - 1) / kGxWaves;  // A loads per wavefront and stage
constexpr int kGxNB = 4;                                             // B loads
// dense: m-tiles whose column tiles run together on an XCD
constexpr int kGxGroupM = 4;

}  // namespace

struct GxItem {
  int nt, e, seg0, nrows, mb;
};

// a lane's load sources for one tile; na = this wavefront's A loads per stage
struct GxLoads {
  __amdgpu_buffer_rsrc_t asrc, wsrc[2];
  int avoff[kGxNA], bvoff[kGxNB];
  int na;
};

template <bool GROUPED>
__device__ __forceinline__ GxItem gx_item(const GemmBf16Args& a, int item) {
  GxItem it;
  if (GROUPED) {
    const int lm = item / a.n_nt;
    it.nt = item - lm * a.n_nt;
    const int tile = ld_uniform(a.tiles, lm);
    it.e = tile >> 16;
    it.seg0 = ld_uniform(a.offsets, it.e) + (tile & 0xFFFF) * kPrefillBM;
    it.nrows = min(kPrefillBM, ld_uniform(a.offsets, it.e + 1) - it.seg0);
    it.mb = (it.nrows + 31) >> 5;
  } else {
    const int n_mt = (a.M + 32 * a.mb - 1) / (32 * a.mb);
    const int g = item / (kGxGroupM * a.n_nt);
    const int rem = item - g * kGxGroupM * a.n_nt;
    const int gm = min(kGxGroupM, n_mt - g * kGxGroupM);
    it.nt = rem / gm;
    it.e = 0;
    it.seg0 = (g * kGxGroupM + rem - it.nt * gm) * 32 * a.mb;
    it.nrows = min(32 * a.mb, a.M - it.seg0);
    it.mb = a.mb;
  }
  return it;
}

// GATHER: the tile's rows are gathered through the LDS table, which must hold
// them (row r at entry seg0 % 4 + r)
template <int EPI, bool GROUPED>
__device__ __forceinline__ GxLoads gx_loads(const GemmBf16Args& a, const GxItem& it, const unsigned char* smem) {
  constexpr bool GU = EPI == kGemmGateUp;
  constexpr bool GATHER = GU && GROUPED;
  GxLoads L;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K2 = a.K * 2;
  const int* table = reinterpret_cast<const int*>(smem + kGxTable);
  // instruction j = wave + 8 i brings rows 8 j .. 8 j + 7: lane l row 8 j +
  // l / 8, the chunk its LDS slot l % 8 holds (rows past the tile repeat its
  // last row: their results are not stored)
  L.na = 0;
#pragma unroll
  for (int i = 0; i < kGxNA; ++i) {
    const int j = wave + kGxWaves * i;
    const bool real = j < 4 * it.mb;
    L.na += real ? 1 : 0;
    const int r = 8 * j + (lane >> 3);
    const int rr = min(r, it.nrows - 1);
    const int src = GATHER ? (real ? table[(it.seg0 & 3) + rr] : 0) / a.topk : rr;
    L.avoff[i] = src * K2 + 16 * ((lane & 7) ^ ((r >> 1) & 7));
  }
  // one descriptor per tile: offsets inside it stay below 2^31
  L.asrc = GATHER ? make_rsrc(a.act, (uint32_t)a.M * (uint32_t)K2)
                  : make_rsrc(a.act + (int64_t)it.seg0 * a.K, (uint32_t)it.nrows * (uint32_t)K2);
  // B: wavefront w brings tile rows 32 w .. 32 w + 31, instruction i rows
  // 8 i .. of them (gate/up: 0, 1 gate rows, 2, 3 their up rows).  Rows past
  // the matrix repeat its last row.
  const int n0 = it.nt * (GU ? kGxBN / 2 : kGxBN);
  const int left = a.cols - n0;  // output columns from this tile on
  const uint32_t wbytes = (uint32_t)min(left, kGxBN) * (uint32_t)K2;
  const int64_t wofs = ((int64_t)it.e * a.wrows + n0) * a.K;
  L.wsrc[0] = make_rsrc(a.W + wofs, wbytes);
  L.wsrc[1] = GU ? make_rsrc(a.W2 + wofs, wbytes) : L.wsrc[0];
#pragma unroll
  for (int i = 0; i < kGxNB; ++i) {
    const int tr = 32 * wave + 8 * i + (lane >> 3);
    const int row = GU ? 16 * wave + 8 * (i & 1) + (lane >> 3) : tr;
    L.bvoff[i] = min(row, left - 1) * K2 + 16 * ((lane & 7) ^ ((tr >> 1) & 7));
  }
  return L;
}

// part p (0..3) of the loads of stage kt into ring slot `slot`.  In a last
// half stage the lanes of chunks 4..7 (past K) load the chunk four before
// instead: a row's last chunks may be the last bytes of its tensor.  The
// chunk's upper half is bit 2 of (lane % 8) ^ ((row / 2) % 8): row / 8 is odd
// for odd A instructions (wave + 8 p) and odd B instructions (4 wave + p).
template <int EPI>
__device__ __forceinline__ void gx_issue(const GemmBf16Args& a, const GxLoads& L, unsigned char* smem, int kt,
                                         int slot, int p) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  unsigned char* st = smem + slot * kGxStageBytes;
  const int back = (kt + 1) * kGxKT > a.K ? 64 : 0;
  const int hi = (lane >> 2) & 1;
  if (p < kGxNA && p < L.na)
    px_dma16(L.asrc, L.avoff[p < kGxNA ? p : 0] - back * (hi ^ (wave & 1)), kt * (kGxKT * 2),
             st + (wave + kGxWaves * p) * 1024);
  px_dma16(L.wsrc[EPI == kGemmGateUp ? p >> 1 : 0], L.bvoff[p] - back * (hi ^ (p & 1)), kt * (kGxKT * 2),
           st + kGxB + wave * 4096 + p * 1024);
}

// a tile's stages 0 and 1 into ring slots q0 and q0 + 1; returns the
// wavefront's loads per stage
template <int EPI, bool GROUPED>
__device__ __forceinline__ int gx_issue_first(const GemmBf16Args& a, const GxItem& it, unsigned char* smem, int q0) {
  const GxLoads L = gx_loads<EPI, GROUPED>(a, it, smem);
  const int q1 = q0 == kGxStages - 1 ? 0 : q0 + 1;
#pragma unroll
  for (int p = 0; p < 4; ++p) gx_issue<EPI>(a, L, smem, 0, q0, p);
#pragma unroll
  for (int p = 0; p < 4; ++p) gx_issue<EPI>(a, L, smem, 1, q1, p);
  return L.na + kGxNB;
}

// One tile.  On entry its stages 0 and 1 are issued into slots p0 and p0 + 1
// (n_inflight loads of this wavefront each).  After its last stage it issues
// the next tile's first two stages (when has_next) and returns their load
// count; the epilogue runs while they land.  With fetch_q wavefront 0 takes
// an index from that counter during the last stage (whose wait is for all
// loads) and leaves it at kGxQSlot.
template <int EPI, bool GROUPED, int MB, int WM>
__device__ __forceinline__ int gx_run(const GemmBf16Args& a, unsigned char* smem, const GxItem& it, const GxItem& nx,
                                      bool has_next, int p0, int n_inflight, int* fetch_q) {
  constexpr bool GU = EPI == kGemmGateUp;
  constexpr int NB = WM;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = WM == 1 ? 0 : wave >> 2;       // the wavefront's row blocks wm MB ..
  const int wn = WM == 1 ? wave : wave & 3;     // and 32-row weight groups wn NB ..
  const int h = lane >> 5, c = lane & 31;
  const int nkt = (a.K + kGxKT - 1) / kGxKT;
  // chunk 2 s + h of row c of a 32-row block (A and B alike)
  int off[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) off[s] = c * 128 + 16 * ((2 * s + h) ^ ((c >> 1) & 7));
  const int a0 = wm * MB * 4096, b0 = kGxB + wn * NB * 4096;
  // a weight group past the matrix multiplies nothing
  const int ncol0 = GU ? (kGxBN / 2) * it.nt : kGxBN * it.nt;
  constexpr int GC = GU ? 16 : 32;  // output columns of a 32-row weight group
  const bool work = ncol0 + GC * NB * wn < a.cols;

  // acc: the current range of k, tot: the ranges before it
  f32x16_t acc[NB][MB], tot[NB][MB];
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[n][m][q] = tot[n][m][q] = 0.f;
  int left = a.krange;
  auto add_range = [&] {
#pragma unroll
    for (int n = 0; n < NB; ++n)
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          tot[n][m][q] += acc[n][m][q];
          acc[n][m][q] = 0.f;
        }
    left = a.krange;
  };
  u32x4_t af[MB], bf[NB], bn[NB];
  auto wait_and_sync = [&](int n, auto hook) {
    __builtin_amdgcn_sched_barrier(0);
    px_wait_vm(n);
    __builtin_amdgcn_sched_barrier(0);
    hook();
    px_barrier();
  };
  auto no_hook = [] {};

  wait_and_sync(n_inflight, no_hook);  // stage 0 landed
  int slot = p0;
  int slot2 = p0 + 2 >= kGxStages ? p0 + 2 - kGxStages : p0 + 2;
  if (work) {
    const unsigned char* st = smem + slot * kGxStageBytes;
#pragma unroll
    for (int n = 0; n < NB; ++n) bf[n] = *reinterpret_cast<const u32x4_t*>(st + b0 + n * 4096 + off[0]);
#pragma unroll
    for (int m = 0; m < MB; ++m) af[m] = *reinterpret_cast<const u32x4_t*>(st + a0 + m * 4096 + off[0]);
  }
  // one step: multiply the fragments at hand, reading the next step's (o: its
  // place in the stage at st) behind the MFMAs that used them
  auto step = [&](const unsigned char* st, int o) {
#pragma unroll
    for (int nn = 0; nn < NB; ++nn) bn[nn] = *reinterpret_cast<const u32x4_t*>(st + b0 + nn * 4096 + o);
#pragma unroll
    for (int m = 0; m < MB; ++m) {
#pragma unroll
      for (int nn = 0; nn < NB; ++nn) acc[nn][m] = mfma32(bf[nn], af[m], acc[nn][m]);
      af[m] = *reinterpret_cast<const u32x4_t*>(st + a0 + m * 4096 + o);
    }
#pragma unroll
    for (int nn = 0; nn < NB; ++nn) bf[nn] = bn[nn];
  };
  // one stage: refill the slot the stage before used (issue(slot2, part)),
  // multiply, wait until at most n loads are in flight and meet the other
  // wavefronts; the last step runs beside the next stage's first reads
  auto stage = [&](int n, auto issue) {
    const int nslot = slot == kGxStages - 1 ? 0 : slot + 1;
    if (work) {
      const unsigned char* st = smem + slot * kGxStageBytes;
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        issue(slot2, s);
        step(st, off[s + 1]);
        if (s == 1 && --left == 0) add_range();
      }
      issue(slot2, 3);
      wait_and_sync(n, no_hook);
      step(smem + nslot * kGxStageBytes, off[0]);
      if (--left == 0) add_range();
    } else {
#pragma unroll
      for (int p = 0; p < 4; ++p) issue(slot2, p);
      wait_and_sync(n, no_hook);
    }
    slot = nslot;
    slot2 = slot2 == kGxStages - 1 ? 0 : slot2 + 1;
  };
  {
    const GxLoads lc = gx_loads<EPI, GROUPED>(a, it, smem);
    for (int t = 0; t + 2 < nkt; ++t)
      stage(lc.na + kGxNB, [&](int sl, int p) { gx_issue<EPI>(a, lc, smem, t + 2, sl, p); });
  }
  // no stage loads are left for the last two stages: the first of them brings
  // the row indices (gate/up: the next tile's rows, for its load sources;
  // plain: this tile's output rows)
  const bool tab = GROUPED && wave == 0;  // wavefront-uniform
  stage(tab ? 1 : 0, [&](int, int p) {
    if (p == 0 && tab) {
      const int tseg = GU && has_next ? nx.seg0 : it.seg0;
      px_dma16(make_rsrc(a.sorted_pos, (uint32_t)a.rows_total * 4u), 4 * ((tseg & ~3) + 4 * lane), 0, smem + kGxTable);
    }
  });
  // the last stage, whole or half: where it is whole its first two steps, then
  // the two steps both have (one path for the accumulators)
  const bool whole = a.K % kGxKT == 0;
  const bool fetch = GROUPED && fetch_q != nullptr && wave == 0;  // wavefront-uniform
  int fv = 0;
  if (fetch && lane == 0) fv = __hip_atomic_fetch_add(fetch_q, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (work) {
    const unsigned char* st = smem + slot * kGxStageBytes;
    if (whole) {
      step(st, off[1]);
      step(st, off[2]);
      if (--left == 0) add_range();
    }
    step(st, whole ? off[3] : off[1]);
  }
  wait_and_sync(0, [&] {
    if (fetch && lane == 0) *reinterpret_cast<int*>(smem + kGxQSlot) = fv;
  });
  if (work) {
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int nn = 0; nn < NB; ++nn) acc[nn][m] = mfma32(bf[nn], af[m], acc[nn][m]);
  }
  const int n_next = has_next ? gx_issue_first<EPI, GROUPED>(a, nx, smem, (p0 + nkt) % kGxStages) : 0;
  if (!work) return n_next;
#pragma unroll
  for (int n = 0; n < NB; ++n)
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int q = 0; q < 16; ++q) tot[n][m][q] += acc[n][m][q];

  // ---- epilogue: lane (h, c) holds, for row 32 m + c of its block, weight
  // rows 8 J + 4 h + i of group n in acc[n][m][4 J + i]
  if (GU) {
    // rows 0..15 of a group are gate rows, 16..31 their up rows
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const int row = 32 * (wm * MB + m) + c;
      if (row >= it.nrows) continue;
#pragma unroll
      for (int n = 0; n < NB; ++n) {
        const int col = ncol0 + 16 * (wn * NB + n);
        if (col >= a.cols) continue;
        uint16_t* orow = a.out + (int64_t)(it.seg0 + row) * a.cols + col + 4 * h;
#pragma unroll
        for (int J = 0; J < 2; ++J) {
          float hv[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float g = round_bf16(tot[n][m][4 * J + i]);
            const float u = round_bf16(tot[n][m][4 * J + i + 8]);
            hv[i] = round_bf16(gelu_tanh_f32(g)) * u;
          }
          *reinterpret_cast<uint2*>(orow + 8 * J) = make_uint2(pack_bf16x2(hv[0], hv[1]), pack_bf16x2(hv[2], hv[3]));
        }
      }
    }
  } else {
    // 16-byte stores of a row's 32 columns, through the slot of the last
    // stage (every wavefront is past its reads; the next tile's stage 2 goes
    // there after the barrier that starts that tile)
    const int* table = reinterpret_cast<const int*>(smem + kGxTable);
    unsigned char* ob = smem + ((p0 + nkt - 1) % kGxStages) * kGxStageBytes + wave * 32 * kGxEpiPitch;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
#pragma unroll
      for (int n = 0; n < NB; ++n) {
#pragma unroll
        for (int J = 0; J < 4; ++J)
          *reinterpret_cast<uint2*>(ob + c * kGxEpiPitch + 2 * (8 * J + 4 * h)) =
              make_uint2(pack_bf16x2(tot[n][m][4 * J], tot[n][m][4 * J + 1]),
                         pack_bf16x2(tot[n][m][4 * J + 2], tot[n][m][4 * J + 3]));
        const int col = ncol0 + 32 * (wn * NB + n);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int idx = lane + 64 * i;
          const int r = 32 * (wm * MB + m) + (idx >> 2), q4 = idx & 3;
          if (r < it.nrows && col < a.cols) {
            const u32x4_t v = *reinterpret_cast<const u32x4_t*>(ob + (idx >> 2) * kGxEpiPitch + 16 * q4);
            const int64_t orow = GROUPED ? table[(it.seg0 & 3) + r] : it.seg0 + r;
            st16(a.out + orow * a.cols + col + 8 * q4, v);
          }
        }
      }
    }
  }
  return n_next;
}

// MBD: dense, the launch's row blocks per tile (0: grouped)
template <int EPI, int MBD>
__device__ __forceinline__ int gx_dispatch(const GemmBf16Args& a, unsigned char* smem, const GxItem& it,
                                           const GxItem& nx, bool has_next, int p0, int n_inflight, int* fetch_q) {
  constexpr bool GROUPED = MBD == 0;
  if constexpr (!GROUPED) {
    // wavefronts by rows where that reads fewer fragments per MFMA
    constexpr int WM = MBD == 2 || MBD == 4 ? 2 : 1;
    return gx_run<EPI, GROUPED, MBD / WM, WM>(a, smem, it, nx, has_next, p0, n_inflight, fetch_q);
  }
  switch (it.mb) {
    case 1: return gx_run<EPI, GROUPED, 1, 1>(a, smem, it, nx, has_next, p0, n_inflight, fetch_q);
    case 2: return gx_run<EPI, GROUPED, 1, 2>(a, smem, it, nx, has_next, p0, n_inflight, fetch_q);
    case 3: return gx_run<EPI, GROUPED, 3, 1>(a, smem, it, nx, has_next, p0, n_inflight, fetch_q);
    default: return gx_run<EPI, GROUPED, 2, 2>(a, smem, it, nx, has_next, p0, n_inflight, fetch_q);
  }
}

// Persistent grid.  Grouped: item i is column tile i % n_nt of list entry i /
// n_nt; workgroup b takes items b and b + P, then those that the queue hands
// out (2 P, 2 P + 1, ...), one ahead.  queue[8] counts the workgroups that
// have left; the sort zeroes the counters and the last to leave resets them.
// Dense: XCD x has tiles [x per, x per + per) in order, its workgroups every
// P-th of them.
template <int EPI, int MBD>
__global__ __launch_bounds__(kGxThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_gemm_bf16(GemmBf16Args a) {
  constexpr bool GROUPED = MBD == 0;
  extern __shared__ __align__(16) unsigned char smem[];
  int item, end, step;
  if (GROUPED) {
    end = ld_uniform(a.counters, 1) * a.n_nt;
    item = (int)blockIdx.x;
    step = (int)gridDim.x;
  } else {
    const int total = ((a.M + 32 * a.mb - 1) / (32 * a.mb)) * a.n_nt;
    const int per = (total + 7) >> 3, x = (int)(blockIdx.x & 7);
    end = min(total, (x + 1) * per);
    item = x * per + (int)(blockIdx.x >> 3);
    step = (int)(gridDim.x >> 3);
  }
  auto leave = [&] {
    if (!GROUPED || threadIdx.x != 0) return;
    const int d = __hip_atomic_fetch_add(a.queue + 8, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (d == (int)gridDim.x - 1) {
      __hip_atomic_store(a.queue, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(a.queue + 8, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  };
  if (item >= end) {
    leave();
    return;
  }
  const int nkt = (a.K + kGxKT - 1) / kGxKT;
  GxItem cur = gx_item<GROUPED>(a, item);
  if (GROUPED && EPI == kGemmGateUp) {
    // the first tile's gathered rows (nothing else in flight)
    if (threadIdx.x < 64)
      px_dma16(make_rsrc(a.sorted_pos, (uint32_t)a.rows_total * 4u), 4 * ((cur.seg0 & ~3) + 4 * (int)threadIdx.x), 0,
               smem + kGxTable);
    __builtin_amdgcn_s_waitcnt(px_vm_wait(0));
    px_barrier();
  }
  int n_inflight = gx_issue_first<EPI, GROUPED>(a, cur, smem, 0);
  int p0 = 0;
  int nitem = item + step;
  for (;;) {
    const bool has_next = nitem < end;
    const GxItem nxt = has_next ? gx_item<GROUPED>(a, nitem) : cur;
    n_inflight = gx_dispatch<EPI, MBD>(a, smem, cur, nxt, has_next, p0, n_inflight, has_next ? a.queue : nullptr);
    if (!has_next) break;
    nitem = GROUPED ? 2 * step + __builtin_amdgcn_readfirstlane(*reinterpret_cast<volatile int*>(smem + kGxQSlot))
                    : nitem + step;
    cur = nxt;
    p0 = (p0 + nkt) % kGxStages;
  }
  leave();
}

bool gemm_bf16_supported(int64_t K, int64_t cols) {
  // three stages at least; whole 32-row weight groups (the gate/up form's 16
  // columns of a group among them) and 16-byte rows
  return K % 32 == 0 && K > 2 * kGxKT && cols % 32 == 0 && cols > 0 && K <= (1 << 20);
}

hipError_t launch_gemm_bf16(int epi, GemmBf16Args a, int max_items, hipStream_t s) {
  const bool grouped = a.tiles != nullptr;
  a.n_nt = (a.cols + (epi == kGemmGateUp ? kGxBN / 2 : kGxBN) - 1) / (epi == kGemmGateUp ? kGxBN / 2 : kGxBN);
  if (!gemm_bf16_supported(a.K, a.cols) || (grouped && a.queue == nullptr)) return hipErrorInvalidValue;
  int64_t items = (int64_t)max_items * a.n_nt;
  if (!grouped) {
    if (a.mb < 1 || a.mb > kGxMaxBlocks) return hipErrorInvalidValue;
    items = (((int64_t)a.M + 32 * a.mb - 1) / (32 * a.mb)) * a.n_nt;
  }
  if (items <= 0) return hipSuccess;
  if (a.ranges < 1) return hipErrorInvalidValue;
  a.krange = (a.K / 32 + a.ranges - 1) / a.ranges;
  if (items > (int64_t(1) << 30)) return hipErrorInvalidValue;
  auto launch = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(prefill_grid_size(reinterpret_cast<const void*>(kern), kGxThreads, kGxLds, (int)items)),
                       dim3(kGxThreads), kGxLds, s, a);
  };
#define W4A16_GX(EPI_)                              \
  switch (grouped ? 0 : a.mb) {                     \
    case 0: launch(k_gemm_bf16<EPI_, 0>); break;    \
    case 1: launch(k_gemm_bf16<EPI_, 1>); break;    \
    case 2: launch(k_gemm_bf16<EPI_, 2>); break;    \
    case 3: launch(k_gemm_bf16<EPI_, 3>); break;    \
    case 4: launch(k_gemm_bf16<EPI_, 4>); break;    \
    default: launch(k_gemm_bf16<EPI_, 5>); break;   \
  }
  if (epi == kGemmGateUp)
    W4A16_GX(kGemmGateUp)
  else
    W4A16_GX(kGemmPlain)
#undef W4A16_GX
  return hipGetLastError();
}

}  // namespace w4a16
