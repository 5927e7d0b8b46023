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
// k advances in stages of 64 through a ring of three (two in flight), all by
// direct global -> LDS loads of 16 bytes per lane, which complete in issue
// order: A = the rows' 128 bytes each, 16-byte chunks XOR-swizzled by (row /
// 2) % 8, B = the 256 rows' 32 bytes of words.  The tile's scales are one
// contiguous block of the scale tensor; they are read whole, before the first
// stage, and stay in LDS (2-byte reads, so any group count and alignment).
// Step s of a stage takes chunk 4 h + s of it (h = lane / 32): a last half
// stage (K % 64 == 32) has only h = 0's, so the lanes of h = 1 multiply zeros
// there and their loads are turned to the row's bytes before.
//
// Bound: no one unit.  2816 x 2816 at 2048 rows (three blocks, 242 tiles, one
// round): 7.8 VALU per MFMA, issued for 34 % of the time, the MFMAs busy for 30
// %, LDS for 21 %; the wavefronts wait for loads and at the stage barrier for
// 40 % of theirs.  2816 x 2816, G = 32, at 512 / 1024 / 2048 / 4096 rows:
// streamed 33 / 54 / 99 / 186 us, here 24 / 28 / 40 / 64 us (815 TFLOP/s at 2048).
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"
#include "lds_pipe.hpp"
#include "rules.hpp"

namespace w4a16 {

namespace {

constexpr int kLwWaves = 8;
constexpr int kLwThreads = 64 * kLwWaves;
constexpr int kLwBN = 256;  // weight rows per tile
constexpr int kLwKT = 64;   // k per stage
constexpr int kLwStages = 3;
constexpr int lw_stage(int mb) { return mb * 4096 + kLwBN * kLwKT / 2; }
// output rows staged for 16-byte stores: 32 rows x 32 bf16 per wavefront, 80
// bytes apart, in the ring once the tile is done
constexpr int kLwEpiPitch = 80;
static_assert(kLwWaves * 32 * kLwEpiPitch <= kLwStages * lw_stage(1), "output rows fit in the ring");
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
  int n_mt, n_nt;
  int vec;  // rows of y are 16-byte aligned
};

template <int MB>
__global__ __launch_bounds__(kLwThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void k_linear_w4(LinearW4Args a) {
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int kStage = lw_stage(MB);
  constexpr int NA = (4 * MB + kLwWaves - 1) / kLwWaves;  // A loads per wavefront and stage, at most
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
  const int nkt = (a.K + kLwKT - 1) / kLwKT;
  const bool odd = a.K % kLwKT != 0;

  // load sources; rows past the tile or the matrix repeat the last one (their
  // results are not stored)
  const int K2 = a.K * 2, W2 = a.K >> 1;
  const __amdgpu_buffer_rsrc_t asrc = make_rsrc(a.x + (int64_t)m0 * a.K, (uint32_t)nrows * (uint32_t)K2);
  const __amdgpu_buffer_rsrc_t wsrc =
      make_rsrc(reinterpret_cast<const unsigned char*>(a.wp) + (int64_t)n0 * W2, (uint32_t)ncols * (uint32_t)W2);
  int avoff[NA], na = 0;
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int j = wave + kLwWaves * i;
    na += j < 4 * MB ? 1 : 0;
    const int r = 8 * j + (lane >> 3);
    avoff[i] = min(r, nrows - 1) * K2 + 16 * ((lane & 7) ^ ((r >> 1) & 7));
  }
  const int bvoff = min(32 * wave + (lane >> 1), ncols - 1) * W2 + 16 * (lane & 1);
  // part p (0..NA) of the loads of stage kt into ring slot `slot`: A load p,
  // part 0 also the words.  The upper half of a last half stage (chunks 4..7:
  // bit 2 of (lane % 8) ^ ((row / 2) % 8), row / 8 being wave + 8 p; words
  // 4..7) would lie past the row.
  auto issue = [&](int kt, int slot, int p) {
    unsigned char* st = smem + slot * kStage;
    const bool half = (kt + 1) * kLwKT > a.K;
    if (p < NA && wave + kLwWaves * p < 4 * MB)
      px_dma16(asrc, avoff[p < NA ? p : 0] - (half ? 64 * (((lane >> 2) & 1) ^ (wave & 1)) : 0), kt * (kLwKT * 2),
               st + (wave + kLwWaves * p) * 1024);
    if (p == 0) px_dma16(wsrc, bvoff - (half ? 16 * (lane & 1) : 0), kt * (kLwKT / 2), st + MB * 4096 + wave * 1024);
  };
  // the tile's scales, from the 16-byte boundary at or before the first
  const uintptr_t sp = reinterpret_cast<uintptr_t>(a.ws + (int64_t)n0 * a.ng);
  const int sbytes = (int)(sp & 15) + ncols * a.ng * 2;
  {
    const __amdgpu_buffer_rsrc_t ssrc =
        make_rsrc(reinterpret_cast<const void*>(sp & ~uintptr_t(15)), (uint32_t)(sbytes + 15) & ~15u);
    for (int i = wave; i * 1024 < sbytes; i += kLwWaves)
      px_dma16(ssrc, i * 1024 + 16 * lane, 0, smem + kLwStages * kStage + i * 1024);
  }
#pragma unroll
  for (int p = 0; p < 4; ++p) issue(0, 0, p);
#pragma unroll
  for (int p = 0; p < 4; ++p) issue(1, 1, p);

  int aoff[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) aoff[s] = c * 128 + 16 * ((4 * h + s) ^ ((c >> 1) & 7));
  const int boff = MB * 4096 + (32 * wave + c) * 32 + 16 * h;
  const unsigned char* srow =
      smem + kLwStages * kStage + (int)(sp & 15) + min(32 * wave + c, ncols - 1) * a.ng * 2;
  f32x16_t acc[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[m][q] = 0.f;
  const ExactRegs kr = exact_regs();
  u32x4_t af[MB], bw, bf;
  ExactScale es;
  auto read_a = [&](const unsigned char* st, int s, int m) {
    return *reinterpret_cast<const u32x4_t*>(st + m * 4096 + aoff[s]);
  };
  auto read_b = [&](const unsigned char* st, int t) {
    const int g = min((t * kLwKT + 32 * h) >> a.gshift, a.ng - 1);
    bw = *reinterpret_cast<const u32x4_t*>(st + boff);
    es = exact_scale(bf16_bits_to_f32(*reinterpret_cast<const uint16_t*>(srow + 2 * g)));
  };
  // zero in the lanes of h = 1 of a last half stage, which has no k for them
  const bool none = odd && h != 0;
  auto keep = [&](u32x4_t v) { return none ? u32x4_t{0u, 0u, 0u, 0u} : v; };

  px_wait_vm(na + 1);
  px_barrier();  // the scales and stage 0 landed (stage 1 may still be loading)
  read_b(smem, 0);
#pragma unroll
  for (int m = 0; m < MB; ++m) af[m] = read_a(smem, 0, m);
  bf = unpack_exact<false>(bw.x, es, kr);
  int slot = 0, slot2 = 2;
  // stage t; the software pipeline: each A fragment is reloaded for the next
  // step right after its MFMA, the next step's word is dequantised beside the
  // current step's MFMAs, and the last step's MFMAs run after the barrier,
  // beside the next stage's first reads
  // (LAST: the last stage, whole or half by a lane mask.  Two paths here made
  // the compiler hold a second set of accumulators, 16 registers spilled at
  // six blocks: 4096 rows of 704 x 2816 25.0 us against 22.1.)
  auto stage = [&](int t, auto last, bool fill, int left) {
    constexpr bool LAST = decltype(last)::value;
    const unsigned char* st = smem + slot * kStage;
    const int nslot = slot == kLwStages - 1 ? 0 : slot + 1;
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      if (fill) issue(t + 2, slot2, s);
      const u32x4_t bn = unpack_exact<false>(s == 0 ? bw.y : s == 1 ? bw.z : bw.w, es, kr);
      const u32x4_t b = LAST ? keep(bf) : bf;
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        acc[m] = mfma32(b, LAST ? keep(af[m]) : af[m], acc[m]);
        af[m] = read_a(st, s + 1, m);
      }
      bf = bn;
    }
    if (fill) issue(t + 2, slot2, 3);
    __builtin_amdgcn_sched_barrier(0);
    px_wait_vm(left);
    px_barrier();  // stage t + 1 landed
    const u32x4_t b = LAST ? keep(bf) : bf;
    if (!LAST) {
      const unsigned char* sn = smem + nslot * kStage;
      read_b(sn, t + 1);
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        acc[m] = mfma32(b, af[m], acc[m]);
        af[m] = read_a(sn, 0, m);
      }
      bf = unpack_exact<false>(bw.x, es, kr);
    } else {
#pragma unroll
      for (int m = 0; m < MB; ++m) acc[m] = mfma32(b, LAST ? keep(af[m]) : af[m], acc[m]);
    }
    slot = nslot;
    slot2 = slot2 == kLwStages - 1 ? 0 : slot2 + 1;
  };
  for (int t = 0; t + 2 < nkt; ++t) stage(t, std::false_type{}, true, na + 1);
  stage(nkt - 2, std::false_type{}, false, 0);
  stage(nkt - 1, std::true_type{}, false, 0);

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
  while (mb > 0 && kLwStages * lw_stage(mb) + lw_scale_bytes((int)ng) > 160 * 1024) --mb;
  return mb;
}

bool linear_w4_supported(int64_t K, int64_t G) {
  const int64_t ng = (K + G - 1) / G;
  // at least three stages
  return K % 32 == 0 && K > 2 * kLwKT && K <= (1 << 20) && ng <= 1024 && linear_w4_max_blocks(ng) > 0;
}

hipError_t launch_linear_w4(const uint16_t* x, const int32_t* wp, const uint16_t* ws, const uint16_t* bias,
                            uint16_t* y, int64_t M, int64_t N, int64_t K, int64_t G, hipStream_t s) {
  if (M == 0) return hipSuccess;
  if (!linear_w4_supported(K, G)) return hipErrorInvalidValue;
  LinearW4Args a{x, wp, ws, bias, y, (int)M, (int)N, (int)K, (int)((K + G - 1) / G), 0, 0, 0, 0};
  while ((int64_t(1) << (a.gshift + 1)) <= G) ++a.gshift;
  const int mb = linear_w4_blocks(M, N, device_cus(), linear_w4_max_blocks(a.ng));
  a.n_mt = (int)((M + 32 * mb - 1) / (32 * mb));
  a.n_nt = (int)((N + kLwBN - 1) / kLwBN);
  a.vec = N % 8 == 0 && (reinterpret_cast<uintptr_t>(y) & 15u) == 0;
  const int64_t total = (int64_t)a.n_mt * a.n_nt;
  if (total > (int64_t(1) << 30)) return hipErrorInvalidValue;
  const dim3 grid((unsigned)((total + 7) / 8 * 8)), block(kLwThreads);
  const size_t lds = (size_t)(kLwStages * lw_stage(mb) + lw_scale_bytes(a.ng));
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
