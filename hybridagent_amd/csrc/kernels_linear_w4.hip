// Linear4Bit at prefill sizes (quantization.py:171-175):
//   y[m, n] = bf16(sum_k x[m, k] bf16_RNE((u[n, k] - 8) s[n, k / G]) + bias[n])
//
// The decode streamer (k_decode<dense>) streams and dequantises every weight
// once per 16 rows of x.  Here a workgroup of eight wavefronts owns a tile of
// 256 weight rows x 32 MB rows of x, one tile per workgroup, so a weight is
// dequantised once per 32 MB rows: each wavefront has 32 weight rows against
// all the tile's rows, dequantises one packed word per lane and MFMA step
// (17 VALU) and multiplies it into MB accumulators of
// v_mfma_f32_32x32x16_bf16, the weights as the A operand.
//
// Every output is the decode streamer's sum, bit for bit (decode_shape in
// rules.hpp: ranges of 128-wide k tiles, each range one fp32 chain, the ranges
// added in order), so a row's result does not change where a larger batch
// takes this kernel.  The streamer's 16x16x32 MFMA on word s of the tile's four
// 32-wide chunks is two 32x32x16 ones here, on chunks 0, 1 and on 2, 3; the
// words follow in order.  So a stage of 64 k holds half of the words of all
// four chunks, not two chunks whole: stage p of a tile words 2 p and 2 p + 1.
//
// The rows' stages go through a ring of three (two in flight), all by direct
// global -> LDS loads of 16 bytes per lane, which complete in issue order: of
// each row four pieces of 32 bytes, 16-byte chunks XOR-swizzled by (row / 2) %
// 8.  A tile's words come whole, 64 bytes a row, every second stage (two tiles
// in LDS; pieces swizzled by (row / 4) % 4).  The tile's scales are one
// contiguous block of the scale tensor; they are read whole, before the first
// stage, and stay in LDS (2-byte reads, so any group count and alignment).  In
// a last tile of fewer than four chunks the lanes past K multiply zeros, and
// their loads are turned to the tile's first chunk of the row.
//
// Bound: no one unit.  2816 x 2816 at 2048 rows (three blocks, 242 tiles, one
// round): 8.7 VALU per MFMA, issued for 37 % of the time, the MFMAs busy for 29
// %, LDS for 20 %; the wavefronts wait for loads and at the stage barrier for
// 32 % of theirs and to issue for 26 %.  2816 x 2816, G = 32, at 512 / 1024 /
// 2048 / 4096 rows: streamed 33 / 54 / 99 / 186 us, here 26 / 30 / 41 / 67 us
// (795 TFLOP/s at 2048; one chain over all of K 24.5 / 28.4 / 40.7 / 66.1).
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "lds_pipe.hpp"
#include "rules.hpp"

namespace w4a16 {

namespace {

constexpr int kLwWaves = 8;
constexpr int kLwThreads = 64 * kLwWaves;
constexpr int kLwBN = 256;        // weight rows per tile
constexpr int kLwStages = 3;      // ring of the rows' stages (64 k each)
constexpr int kLwPair = 16384;    // the words of a k tile (two stages)
constexpr int lw_stage(int mb) { return mb * 4096; }
constexpr int lw_ring(int mb) { return kLwStages * lw_stage(mb) + 2 * kLwPair; }
// output rows staged for 16-byte stores: 32 rows x 32 bf16 per wavefront, 80
// bytes apart, in the ring once the tile is done
constexpr int kLwEpiPitch = 80;
static_assert(kLwWaves * 32 * kLwEpiPitch <= lw_ring(1), "output rows fit in the ring");
// m-tiles whose column tiles run together on an XCD
constexpr int kLwGroupM = 4;

inline int lw_scale_bytes(int ng) { return (kLwBN * ng * 2 + 16 + 1023) / 1024 * 1024; }

}  // namespace

struct LinearW4Args {
  const uint16_t* x;
  const int32_t* wp;
  const uint16_t* ws;
  const uint16_t* bias;  // nullable
  uint16_t* y;
  int M, N, K, ng, gshift;
  int tpw, skip;  // k tiles of a range taken in a row, and from there to its next ones
  int n_mt, n_nt;
  int vec;        // rows of y are 16-byte aligned
};

template <int MB>
__global__ __launch_bounds__(kLwThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_linear_w4(LinearW4Args a) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int kStage = lw_stage(MB), kBOff = kLwStages * kStage;
  constexpr int NA = (4 * MB + kLwWaves - 1) / kLwWaves;  // A loads per wavefront and stage, at most
  // fragments of rows read ahead (six would not fit beside six blocks' sums)
  constexpr int R = MB == 6 ? 3 : MB;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = lane >> 5, c = lane & 31;
  // XCD x (workgroups are dealt in turn) has the tiles [x per, x per + per),
  // ordered so that the tiles running at once share rows and columns
  const int total = a.n_mt * a.n_nt, per = (total + 7) >> 3;
  const int item = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (item >= min(total, ((int)(blockIdx.x & 7) + 1) * per)) return;
  const int grp = item / (kLwGroupM * a.n_nt);
  const int rem = item - grp * kLwGroupM * a.n_nt;
  const int gm = min(kLwGroupM, a.n_mt - grp * kLwGroupM);
  const int nt = rem / gm;
  const int m0 = (grp * kLwGroupM + rem - nt * gm) * 32 * MB, n0 = nt * kLwBN;
  const int nrows = min(32 * MB, a.M - m0), ncols = min(kLwBN, a.N - n0);
  const int T = (a.K + 127) >> 7;           // k tiles
  const int nq = ((a.K - 1) >> 5 & 3) + 1;  // 32-wide chunks of the last

  // load sources; rows past the tile or the matrix repeat the last one (their
  // results are not stored)
  const int K2 = a.K * 2, W2 = a.K >> 1;
  const __amdgpu_buffer_rsrc_t asrc = make_rsrc(a.x + (int64_t)m0 * a.K, (uint32_t)nrows * (uint32_t)K2);
  const __amdgpu_buffer_rsrc_t wsrc =
      make_rsrc(reinterpret_cast<const unsigned char*>(a.wp) + (int64_t)n0 * W2, (uint32_t)ncols * (uint32_t)W2);
  // (a load's rows are 8 apart per wavefront: (row / 2) % 8 by lane and wave % 2)
  const int ach = (lane & 7) ^ ((4 * wave + (lane >> 4)) & 7), bch = (lane & 3) ^ ((lane >> 4) & 3);
  int avoff[NA], na = 0;
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int j = wave + kLwWaves * i;
    na += j < 4 * MB ? 1 : 0;
    avoff[i] = min(8 * j + (lane >> 3), nrows - 1) * K2 + 64 * (ach >> 1) + 16 * (ach & 1);
  }
  int bvoff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) bvoff[i] = min(32 * wave + 16 * i + (lane >> 2), ncols - 1) * W2 + 16 * bch;
  // chunks past K in the last tile: its first chunk again, multiplied by zero as zero
  const int aback = (ach >> 1) < nq ? 0 : 64 * (ach >> 1), bback = bch < nq ? 0 : 16 * bch;
  // part i (0..NA) of the rows' loads of stage p of tile t into ring slot
  // `slot`; load i (0, 1) of a tile's words
  auto issue_a = [&](int t, int p, int slot, int i) {
    if (i < NA && wave + kLwWaves * i < 4 * MB)
      px_dma16(asrc, avoff[i < NA ? i : 0] - (t == T - 1 ? aback : 0), t * 256 + 32 * p,
               smem + slot * kStage + (wave + kLwWaves * i) * 1024);
  };
  auto issue_b = [&](int t, int half, int i) {
    px_dma16(wsrc, bvoff[i] - (t == T - 1 ? bback : 0), t * 64,
             smem + kBOff + half * kLwPair + wave * 2048 + i * 1024);
  };
  // the tile's scales, from the 16-byte boundary at or before the first
  const uintptr_t sp = reinterpret_cast<uintptr_t>(a.ws + (int64_t)n0 * a.ng);
  const int sbytes = (int)(sp & 15) + ncols * a.ng * 2;
  {
    const __amdgpu_buffer_rsrc_t ssrc =
        make_rsrc(reinterpret_cast<const void*>(sp & ~uintptr_t(15)), (uint32_t)(sbytes + 15) & ~15u);
    for (int i = wave; i * 1024 < sbytes; i += kLwWaves)
      px_dma16(ssrc, i * 1024 + 16 * lane, 0, smem + lw_ring(MB) + i * 1024);
  }
#pragma unroll
  for (int i = 0; i < NA; ++i) issue_a(0, 0, 0, i);
  issue_b(0, 0, 0);
  issue_b(0, 0, 1);
#pragma unroll
  for (int i = 0; i < NA; ++i) issue_a(0, 1, 1, i);

  // step e of a stage: piece e & 1 (chunks 2 (e & 1) + h), word 2 p + e / 2
  int aoff[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) aoff[e] = c * 128 + 16 * ((4 * (e & 1) + 2 * h + (e >> 1)) ^ ((c >> 1) & 7));
  int boff[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) boff[g] = kBOff + (32 * wave + c) * 64 + 16 * ((2 * g + h) ^ ((c >> 2) & 3));
  const unsigned char* srow = smem + lw_ring(MB) + (int)(sp & 15) + min(32 * wave + c, ncols - 1) * a.ng * 2;
  // acc: the current range of k, tot: the ranges before it
  f32x16_t acc[MB], tot[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[m][q] = tot[m][q] = 0.f;
  const ExactRegs kr = exact_regs();
  u32x4_t af[R], bw[2], bf;
  float sc[2];
  auto read_a = [&](const unsigned char* st, int e, int m) {
    return *reinterpret_cast<const u32x4_t*>(st + m * 4096 + aoff[e]);
  };
  auto read_b = [&](int t, int half) {
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      bw[g] = *reinterpret_cast<const u32x4_t*>(smem + boff[g] + half * kLwPair);
      const int grp = min((t * 128 + 64 * g + 32 * h) >> a.gshift, a.ng - 1);
      sc[g] = bf16_bits_to_f32(*reinterpret_cast<const uint16_t*>(srow + 2 * grp));
    }
  };
  auto unpack = [&](int p, int e) {
    const u32x4_t v = bw[e & 1];
    const uint32_t w = p == 0 ? (e < 2 ? v.x : v.y) : (e < 2 ? v.z : v.w);
    return unpack_exact<false>(w, exact_scale(sc[e & 1]), kr);
  };
  // zero in the lanes whose chunk is past K (step e of the last tile; one path
  // whether there are any: with two the compiler holds a second set of
  // accumulators, which does not fit)
  auto keep = [&](u32x4_t v, int e) { return 2 * (e & 1) + h < nq ? v : u32x4_t{0u, 0u, 0u, 0u}; };

  px_wait_vm(na);
  px_barrier();  // the scales, stage 0 and its words landed (stage 1 may still be loading)
  read_b(0, 0);
#pragma unroll
  for (int m = 0; m < R; ++m) af[m] = read_a(smem, 0, m);
  bf = unpack(0, 0);
  int slot = 0, slot2 = 2, half = 0;
  // stage P of a tile, whose next is tile tn (LAST: none); the software
  // pipeline: each A fragment is reloaded for the next step right after its
  // MFMA, the next step's word is dequantised beside the current step's MFMAs,
  // and the last step's MFMAs run after the barrier, beside the next stage's
  // first reads
  auto stage = [&](auto pc, auto last, int tn) {
    constexpr int P = decltype(pc)::value;
    constexpr bool LAST = decltype(last)::value;
    const unsigned char* st = smem + slot * kStage;
    const int nslot = slot == kLwStages - 1 ? 0 : slot + 1;
#pragma unroll
    for (int e = 0; e < 3; ++e) {
      if (!LAST) {
        issue_a(tn, P, slot2, e);
        if (P == 0 && e > 0) issue_b(tn, half ^ 1, e - 1);
      }
      const u32x4_t bn = unpack(P, e + 1);
      const u32x4_t b = LAST ? keep(bf, e) : bf;
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        acc[m] = mfma32(b, LAST ? keep(af[m % R], e) : af[m % R], acc[m]);
        af[m % R] = m + R < MB ? read_a(st, e, m + R) : read_a(st, e + 1, m + R - MB);
      }
      bf = bn;
    }
    const u32x4_t b = LAST ? keep(bf, 3) : bf;
#pragma unroll
    for (int m = 0; m + R < MB; ++m) {
      acc[m] = mfma32(b, LAST ? keep(af[m % R], 3) : af[m % R], acc[m]);
      af[m % R] = read_a(st, 3, m + R);
    }
    __builtin_amdgcn_sched_barrier(0);
    px_wait_vm(LAST ? 0 : P == 0 ? na + 2 : na);
    px_barrier();  // the next stage landed
    const unsigned char* sn = smem + nslot * kStage;
    if (!LAST && P == 1) {
      half ^= 1;
      read_b(tn, half);
    }
#pragma unroll
    for (int m = MB - R; m < MB; ++m) {
      acc[m] = mfma32(b, LAST ? keep(af[m % R], 3) : af[m % R], acc[m]);
      if (!LAST || P == 0) af[m % R] = read_a(sn, 0, m + R - MB);
    }
    if (!LAST || P == 0) bf = unpack(P ^ 1, 0);
    slot = nslot;
    slot2 = slot2 == kLwStages - 1 ? 0 : slot2 + 1;
  };
  const std::integral_constant<int, 0> p0;
  const std::integral_constant<int, 1> p1;
  int t = 0, range0 = 0, run = a.tpw;  // the tile, its range's first, tiles up to the range's next jump
  for (int i = 0; i + 1 < T; ++i) {
    int tn = t + 1;
    if (--run == 0) {
      tn += a.skip;
      run = a.tpw;
    }
    const bool end = tn >= T;
    if (end) tn = range0 += a.tpw, run = a.tpw;
    stage(p0, std::false_type{}, tn);
    stage(p1, std::false_type{}, tn);
    if (end) {
#pragma unroll
      for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int q = 0; q < 16; ++q) {
          tot[m][q] += acc[m][q];
          acc[m][q] = 0.f;
        }
    }
    t = tn;
  }
  stage(p0, std::true_type{}, 0);
  stage(p1, std::true_type{}, 0);
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[m][q] += tot[m][q];

  // Lane (h, c) holds, for row 32 m + c, weight rows 8 J + 4 h + i in
  // acc[m][4 J + i].  Every wavefront is past its last read of the ring, which
  // now takes the wavefront's 32 x 32 block so that rows go out 16 bytes at a
  // time.
  if (32 * wave >= ncols) return;
  float bb[16];
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int n = 32 * wave + 8 * (q >> 2) + 4 * h + (q & 3);
    bb[q] = a.bias != nullptr && n < ncols ? bf16_bits_to_f32(a.bias[n0 + n]) : 0.f;
  }
  unsigned char* ob = smem + wave * 32 * kLwEpiPitch;
#pragma unroll
  for (int m = 0; m < MB; ++m) {
#pragma unroll
    for (int J = 0; J < 4; ++J)
      *reinterpret_cast<uint2*>(ob + c * kLwEpiPitch + 2 * (8 * J + 4 * h)) =
          make_uint2(pack_bf16x2(acc[m][4 * J] + bb[4 * J], acc[m][4 * J + 1] + bb[4 * J + 1]),
                     pack_bf16x2(acc[m][4 * J + 2] + bb[4 * J + 2], acc[m][4 * J + 3] + bb[4 * J + 3]));
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int idx = lane + 64 * i;
      const int row = 32 * m + (idx >> 2), col = 32 * wave + 8 * (idx & 3);
      if (row >= nrows || col >= ncols) continue;
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(ob + (idx >> 2) * kLwEpiPitch + 16 * (idx & 3));
      uint16_t* o = a.y + (int64_t)(m0 + row) * a.N + n0 + col;
      if (a.vec && col + 8 <= ncols) {
        st16(o, v);
      } else {
        const uint32_t w4[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int q = 0; q < 8; ++q)
          if (col + q < ncols) o[q] = (uint16_t)(w4[q >> 1] >> (16 * (q & 1)));
      }
    }
  }
}

// most 32-row blocks per tile whose ring and scales fit in LDS (0: none)
static int linear_w4_max_blocks(int64_t ng) {
  int mb = kLinearW4MaxBlocks;
  while (mb > 0 && lw_ring(mb) + lw_scale_bytes((int)ng) > 160 * 1024) --mb;
  return mb;
}

bool linear_w4_supported(int64_t K, int64_t G) {
  const int64_t ng = (K + G - 1) / G;
  // at least two tiles, and a partial one last in the order of the ranges
  return K % 32 == 0 && K > 128 && (K % 128 == 0 || !decode_ranges_interleave(K)) && K <= (1 << 20) && ng <= 1024 &&
         linear_w4_max_blocks(ng) > 0;
}

hipError_t launch_linear_w4(const uint16_t* x, const int32_t* wp, const uint16_t* ws, const uint16_t* bias,
                            uint16_t* y, int64_t M, int64_t N, int64_t K, int64_t G, hipStream_t s) {
  if (M == 0) return hipSuccess;
  if (!linear_w4_supported(K, G)) return hipErrorInvalidValue;
  LinearW4Args a{x, wp, ws, bias, y, (int)M, (int)N, (int)K, (int)((K + G - 1) / G), 0, 0, 0, 0, 0, 0};
  const DecodeShape sh = decode_shape(K);
  a.tpw = sh.tpw;
  a.skip = (sh.ksplit - 1) * sh.tpw;
  while ((int64_t(1) << (a.gshift + 1)) <= G) ++a.gshift;
  const int mb = linear_w4_blocks(M, N, device_cus(), linear_w4_max_blocks(a.ng));
  a.n_mt = (int)((M + 32 * mb - 1) / (32 * mb));
  a.n_nt = (int)((N + kLwBN - 1) / kLwBN);
  a.vec = N % 8 == 0 && (reinterpret_cast<uintptr_t>(y) & 15u) == 0;
  const int64_t total = (int64_t)a.n_mt * a.n_nt;
  if (total > (int64_t(1) << 30)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((total + 7) / 8 * 8)), block(kLwThreads);
  const size_t lds = (size_t)(lw_ring(mb) + lw_scale_bytes(a.ng));
  switch (mb) {
    case 1: hipLaunchKernelGGL(k_linear_w4<1>, grid, block, lds, s, a); break;
    case 2: hipLaunchKernelGGL(k_linear_w4<2>, grid, block, lds, s, a); break;
    case 3: hipLaunchKernelGGL(k_linear_w4<3>, grid, block, lds, s, a); break;
    case 4: hipLaunchKernelGGL(k_linear_w4<4>, grid, block, lds, s, a); break;
    case 5: hipLaunchKernelGGL(k_linear_w4<5>, grid, block, lds, s, a); break;
    default: hipLaunchKernelGGL(k_linear_w4<6>, grid, block, lds, s, a); break;
  }
  return hipGetLastError();
}

}  // namespace w4a16
