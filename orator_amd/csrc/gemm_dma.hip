// bf16 GEMM with fp32 accumulation whose tiles go from memory straight into LDS, gfx950:
// out[M][N] (=|+=) act(in[M][K] W[N][K]^T + bias), and the gate|up form with SwiGLU.
//
// Serves the M > 1 products of gemm_bf16.hip's entry points whose K is a multiple of 64 (all of the
// decoder's and the audio tower's), but for short K with many outputs (gemm_dma_store_bound).
//
// What bounds it: the matrix cores and LDS bandwidth at once.  A 64 x 64 wave tile reads LDS as
// long as its MFMAs run (4 KB and 4 MFMAs of 32 cycles per 16 of K, 128 bytes a cycle for 4 waves),
// and the tile's own arrival comes on top.  Hence:
//  * Buffer loads with an LDS destination: no staging registers and no ds_write.  The register-
//    staged kernel ran at 760 TFLOP/s on 2048 x 2048 -> 12288, this one at 1118 (135.6 -> 92.2 us).
//  * NS stages with one barrier per 64 of K; NS - 1 stages are in flight, which is what cold
//    weights need (390 x 1024 -> 4096 from HBM: 20.0 -> 14.7 us).  Loads past the last stage are
//    issued all the same (its tile again): with a branch around them the compiler cannot count what
//    is in flight and waits for all of it at some stages (2048 x 6144 -> 2048, 1500 rows: 53.4 ->
//    44.3 us; 200 x 2048 -> 12288 21.3 -> 17.7).
//  * Rows of 128 bytes, unpadded (a load writes consecutive LDS bytes); the 16-byte chunk c of row r
//    lies at c ^ (r / 2) % 8, so the 16 rows a quarter-wave reads cover all banks once.  The
//    permutation is applied to the addresses the lanes load from.
//  * W is the MFMA's row operand: a lane ends with 4 consecutive columns of one output row and
//    stores them as they are (no LDS pass at the end).  For SwiGLU a 32-row block of the W tile
//    holds 8 gate rows, the same 8 columns' up rows, and so on, so gate and up meet in one lane.
//  * Fragments of the next 16 of K are read under the current ones' MFMAs.
#include <algorithm>

#include "common.hpp"
#include "internal.hpp"
#include "mfma_tile.hpp"

namespace orator_hip {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

enum GemmEpi : int { kDmaStore = 0, kDmaPartial = 1, kDmaAct = 2, kDmaSwiglu = 3 };

struct GemmDmaArgs {
  const void* A;  // bf16, or fp32 (the F32 kernels)
  const uint16_t* W;
  const float* bias;
  void* out;    // fp32 [M][N]; SwiGLU: bf16 [M][N / 2]
  float* part;  // split-K partials [split][M][N]
  int M, K, N, act, accumulate, k_split;
};

__device__ __forceinline__ float gemm_act(float v, int act) {
  if (act == 1) return 0.5f * v * (1.0f + erff(v * 0.70710678118654752440f));
  if (act == 2) return fmaxf(v, 0.0f);
  return v;
}

// Eight fp32 values as bf16 (v_cvt_pk_bf16_f32: to nearest even, as the cast kernel; a NaN stays one
// whatever its payload).
__device__ __forceinline__ bf16x8_t cvt_bf16x8(const f32x4_t lo, const f32x4_t hi) {
  return as_bf16x8(make_uint4(cvt_bf16x2(lo[0], lo[1]), cvt_bf16x2(lo[2], lo[3]),
                              cvt_bf16x2(hi[0], hi[1]), cvt_bf16x2(hi[2], hi[3])));
}

// F32: A is fp32 and lies in LDS as such, 256-byte rows with chunk c at c ^ r % 16; it is rounded as
// the fragments are read.
template <int BM, int BN, int WGM, int WGN, int NS, int MINW, int EPI, bool F32>
__global__ __launch_bounds__(64 * WGM * WGN, MINW) void gemm_bf16_dma_kernel(GemmDmaArgs a) {
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass has no LDS loads; it needs the launch stub only
  constexpr int BK = 64, CH = BK / 8;          // 16-byte chunks per tile row
  constexpr int NW = WGM * WGN;
  constexpr int TM = BM / WGM, TN = BN / WGN;  // wave tile
  constexpr int FM = TM / 32, FN = TN / 32;
  constexpr int CHA = F32 ? 2 * CH : CH;       // the same of an A row
  constexpr int RPA = 64 / CHA, RPW = 64 / CH;  // tile rows per load instruction of a wave
  constexpr int LA = BM / RPA;                 // load instructions of the A tile
  constexpr int L = (LA + BN / RPW) / NW;      // load instructions per wave and stage
  static_assert(LA % NW == 0 && BN / RPW % NW == 0 && BM % RPA == 0 && BN % RPW == 0);
  static_assert(TM % 32 == 0 && TN % 32 == 0 && NS >= 2 && NS <= 4);
  constexpr int kA = BM * CHA * 8;             // the A tile's part of a stage, in 2-byte units
  constexpr int kStage = kA + BN * BK;
  // One array per stage: the compiler's own waits before an LDS read then count the loads into
  // that stage only, and the later stages' loads stay in flight.
  __shared__ __align__(1024) uint16_t s0[kStage], s1[kStage];
  __shared__ __align__(1024) uint16_t s2[NS > 2 ? kStage : 8], s3[NS > 3 ? kStage : 8];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WGN, wn = wave % WGN;
  const int tiles_n = gridDim.x, tiles_m = gridDim.y;
  const int total = tiles_n * tiles_m;
  int lin = blockIdx.x + tiles_n * blockIdx.y;
  if ((total & 7) == 0) lin = (lin & 7) * (total >> 3) + (lin >> 3);
  constexpr int kGroup = 4;
  const int group = lin / (kGroup * tiles_n);
  const int first_m = group * kGroup;
  const int gm = min(tiles_m - first_m, kGroup);
  const int in_group = lin - group * kGroup * tiles_n;
  const int m0 = (first_m + in_group % gm) * BM, tn = in_group / gm;

  const int M = a.M, N = a.N, K = a.K;
  const int kb = blockIdx.z * a.k_split;
  const int n_k = min(K - kb, a.k_split) / BK;
  const __amdgpu_buffer_rsrc_t rs_a = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void*>(a.A), 0, static_cast<uint32_t>(M) * K * (F32 ? 4 : 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rs_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(a.W), 0, static_cast<uint32_t>(N) * K * 2, 0x00020000);
  // W row of tile row j
  auto w_row = [&](int j) {
    if constexpr (EPI == kDmaSwiglu) {
      const int I = N / 2, c = tn * (BN / 2) + (j >> 5) * 16 + ((j >> 4) & 1) * 8 + (j & 7);
      return min(c, I - 1) + ((j >> 3) & 1) * I;
    } else {
      return min(tn * BN + j, N - 1);
    }
  };
  auto swz = [](int r) { return (r >> 1) & (CH - 1); };
  uint32_t voff[L];
#pragma unroll
  for (int i = 0; i < L; ++i) {
    const int ins = wave + NW * i;
    if (i < LA / NW) {
      const int r = ins * RPA + lane / CHA;
      const int chunk = (lane % CHA) ^ (F32 ? r & (CHA - 1) : swz(r));
      voff[i] = (static_cast<uint32_t>(min(m0 + r, M - 1)) * K + kb) * (F32 ? 4 : 2) + 16 * chunk;
    } else {
      const int r = (ins - LA) * RPW + lane / CH;
      voff[i] = (static_cast<uint32_t>(w_row(r)) * K + kb) * 2 + 16 * ((lane % CH) ^ swz(r));
    }
  }
  auto issue = [&](uint16_t* st, int t) {
#pragma unroll
    for (int i = 0; i < L; ++i) {
      const int ins = wave + NW * i;
      const bool is_a = i < LA / NW;  // known at compile time: a branch here or in the addresses
      // above costs the stages' separation (the compiler then waits for every load in flight)
      const __amdgpu_buffer_rsrc_t rs = is_a ? rs_a : rs_w;
      // every load instruction fills 1024 bytes (512 units), A's first
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs, (__attribute__((address_space(3))) void*)(st + ins * 512), 16, voff[i],
          t * (F32 && is_a ? BK * 4 : BK * 2), 0, 0);
    }
  };

  // One block per wave: the four k-steps of a stage add up apart, which shortens every chain of fp32
  // additions to a quarter of K (the sums are then no further from 64 bits than K split
  // by four left them).
  constexpr int NA = FM * FN == 1 ? BK / 16 : 1;
  f32x16_t part_acc[NA][FM][FN];
#pragma unroll
  for (int h = 0; h < NA; ++h)
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) part_acc[h][i][j][e] = 0.0f;
  const int fr = lane & 31, hi = lane >> 5;
  const int fx = swz(fr);

  auto compute = [&](const uint16_t* st) {
    const uint16_t* pa = st + (wm * TM + fr) * (kA / BM);
    const uint16_t* pw = st + (kA / BK + wn * TN + fr) * BK;
    bf16x8_t fa[2][FM], fb[2][FN];
    [[maybe_unused]] f32x4_t ra[2][FM][2];
    auto read = [&](int ks, int s) {
      const int c = 8 * ((2 * ks + hi) ^ fx);
#pragma unroll
      for (int j = 0; j < FN; ++j)
        fb[s][j] = *reinterpret_cast<const bf16x8_t*>(pw + 32 * j * BK + c);
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        if constexpr (F32) {
          const uint16_t* row = pa + 32 * i * (kA / BM);
          const int c2 = 4 * ks + 2 * hi, x = fr & (CHA - 1);
          ra[s][i][0] = *reinterpret_cast<const f32x4_t*>(row + 8 * (c2 ^ x));
          ra[s][i][1] = *reinterpret_cast<const f32x4_t*>(row + 8 * ((c2 + 1) ^ x));
        } else {
          fa[s][i] = *reinterpret_cast<const bf16x8_t*>(pa + 32 * i * BK + c);
        }
      }
    };
    read(0, 0);
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      const int s = ks & 1;
      if (ks + 1 < BK / 16) read(ks + 1, s ^ 1);
      __builtin_amdgcn_sched_barrier(0);  // the next fragments are on their way under these MFMAs
      if constexpr (F32) {
#pragma unroll
        for (int i = 0; i < FM; ++i) fa[s][i] = cvt_bf16x8(ra[s][i][0], ra[s][i][1]);
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          part_acc[ks % NA][i][j] = mfma32(fb[s][j], fa[s][i], part_acc[ks % NA][i][j]);
    }
  };
  auto ready = [&] {  // stage t has arrived for every wave, stage t - 1 is read out
    // builtins, not asm: the compiler then knows what has arrived and adds no wait of its own
    constexpr int kLater = (NS - 2) * L;  // vmcnt bits 3:0 and 15:14, expcnt 6:4 and lgkmcnt 11:8
    __builtin_amdgcn_s_waitcnt(0x0070 | (kLater & 15) | (kLater >> 4) << 14);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto stage = [&](int i) -> uint16_t* {
    const int k = i % NS;
    return k == 0 ? s0 : k == 1 ? s1 : k == 2 ? s2 : s3;
  };
#pragma unroll
  for (int i = 0; i < NS - 1; ++i)
    issue(stage(i), min(i, n_k - 1));  // unconditional (a branch costs a wait for every load in flight)
  for (int t = 0; t < n_k; t += NS) {
#pragma unroll
    for (int u = 0; u < NS; ++u) {
      if (t + u < n_k) {
        ready();
        issue(stage(u + NS - 1), min(t + u + NS - 1, n_k - 1));
        compute(stage(u));
      }
    }
  }

  __builtin_amdgcn_s_waitcnt(0x0070);  // LDS is given back only when nothing is on its way to it
  auto& acc = part_acc[0];
#pragma unroll
  for (int h = 1; h < NA; h *= 2)
#pragma unroll
    for (int g = 0; g + h < NA; g += 2 * h) part_acc[g][0][0] += part_acc[g + h][0][0];
  // Lane: output row fr of each block row, columns 8 (e / 4) + 4 hi + e % 4 of each block column.
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + wm * TM + 32 * i + fr;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if constexpr (EPI == kDmaSwiglu) {
        const int I = N / 2;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const int col = tn * (BN / 2) + (wn * FN + j) * 16 + 8 * p + 4 * hi;
          float y[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float g = acc[i][j][8 * p + q], u = acc[i][j][8 * p + 4 + q];
            y[q] = (g / (1.0f + expf(-g))) * u;
          }
          if (col < I)  // I is a multiple of 4
            *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out) + static_cast<long>(m) * I +
                                      col) =
                make_uint2(pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3]));
        }
      } else {
        float* out = EPI == kDmaPartial ? a.part + static_cast<long>(blockIdx.z) * M * N
                                        : static_cast<float*>(a.out);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int n = tn * BN + wn * TN + 32 * j + 8 * g + 4 * hi;
          if (n >= N) continue;  // N is a multiple of 4
          float4 v = make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2],
                                 acc[i][j][4 * g + 3]);
          float4* dst = reinterpret_cast<float4*>(out + static_cast<long>(m) * N + n);
          if constexpr (EPI == kDmaAct) {
            if (a.bias) {
              v.x += a.bias[n], v.y += a.bias[n + 1], v.z += a.bias[n + 2], v.w += a.bias[n + 3];
            }
            v.x = gemm_act(v.x, a.act), v.y = gemm_act(v.y, a.act);
            v.z = gemm_act(v.z, a.act), v.w = gemm_act(v.w, a.act);
            if (a.accumulate) {
              const float4 o = *dst;
              v.x += o.x, v.y += o.y, v.z += o.z, v.w += o.w;
            }
          }
          *dst = v;
        }
      }
    }
  }
#endif
}

// out (=|+=) act(sum_z part[z] + bias), z ascending, 4 columns per thread.
__global__ __launch_bounds__(256) void gemm_dma_reduce_kernel(GemmDmaArgs a, int splits) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x;  // M N < 2^31
  const uint32_t MN = static_cast<uint32_t>(a.M) * a.N;
  if (4 * i >= MN) return;
  const float4* part = reinterpret_cast<const float4*>(a.part);
  float4 v = part[i];
  for (int z = 1; z < splits; ++z) {
    const float4 p = part[static_cast<size_t>(z) * (MN / 4) + i];
    v.x += p.x, v.y += p.y, v.z += p.z, v.w += p.w;
  }
  if (a.bias) {
    const float* b = a.bias + 4 * i % a.N;
    v.x += b[0], v.y += b[1], v.z += b[2], v.w += b[3];
  }
  v.x = gemm_act(v.x, a.act), v.y = gemm_act(v.y, a.act);
  v.z = gemm_act(v.z, a.act), v.w = gemm_act(v.w, a.act);
  float4* dst = static_cast<float4*>(a.out) + i;
  if (a.accumulate) {
    const float4 o = *dst;
    v.x += o.x, v.y += o.y, v.z += o.z, v.w += o.w;
  }
  *dst = v;
}

template <int BM, int BN, int WGM, int WGN, int NS, int MINW, bool SWIGLU, bool F32 = false>
int launch_tile(GemmDmaArgs a, int splits, hipStream_t s) {
  const int steps = a.K / 64;
  const int per = (steps + splits - 1) / splits;
  splits = (steps + per - 1) / per;
  a.k_split = 64 * per;
  const dim3 grid((a.N + BN - 1) / BN, (a.M + BM - 1) / BM, splits), block(64 * WGM * WGN);
  if constexpr (SWIGLU) {
    hipLaunchKernelGGL((gemm_bf16_dma_kernel<BM, BN, WGM, WGN, NS, MINW, kDmaSwiglu, F32>), grid, block,
                       0, s, a);
    return check_launch("gemm_bf16_dma_kernel (swiglu)");
  } else {
    if (splits > 1) {
      const size_t bytes = static_cast<size_t>(splits) * a.M * a.N * sizeof(float);
      a.part = static_cast<float*>(workspace(s, bytes, kWsGemm));
      if (!a.part) return ORATOR_ERR_HIP;
      hipLaunchKernelGGL((gemm_bf16_dma_kernel<BM, BN, WGM, WGN, NS, MINW, kDmaPartial, F32>), grid,
                         block, 0, s, a);
      if (int rc = check_launch("gemm_bf16_dma_kernel")) return rc;
      const unsigned quads = static_cast<unsigned>(static_cast<long>(a.M) * a.N / 4);
      hipLaunchKernelGGL(gemm_dma_reduce_kernel, dim3((quads + 255) / 256), dim3(256), 0, s, a,
                         splits);
      return check_launch("gemm_dma_reduce_kernel");
    }
    if (a.bias || a.act || a.accumulate)
      hipLaunchKernelGGL((gemm_bf16_dma_kernel<BM, BN, WGM, WGN, NS, MINW, kDmaAct, F32>), grid, block,
                         0, s, a);
    else
      hipLaunchKernelGGL((gemm_bf16_dma_kernel<BM, BN, WGM, WGN, NS, MINW, kDmaStore, F32>), grid, block,
                         0, s, a);
    return check_launch("gemm_bf16_dma_kernel");
  }
}

// Tile by the time its rounds over the chip take, in us per 2048 of K (every candidate scales with
// K alike), constants fitted on 256 CUs:
//   256 x 192, 8 waves, 1 workgroup per CU:             46 a round
//   128 x 128, 4 waves, 2 stages, 2 workgroups per CU:  36.6 a round, 22 with one per CU
//   128 x 128, 8 waves, 4 stages, 1 workgroup per CU:   20.1 (the same tile when one per CU is all)
//   64 x 64, 4 waves, 4 stages, 2 workgroups per CU:    14.4 a round, 11.3 with one per CU
// Every tile at each shape, us of replayed launches on one card, in that order, the rule's last:
//   2048 x 2048 -> 12288   98.9  103.4  117.6  177.7    99.5
//   2048 x 2048 -> 4096    44.2   37.2   42.2   57.7    37.1
//   2048 x 6144 -> 2048    97.8   65.1   52.3   76.5    52.5
//   1500 x 6144 -> 2048    98.1   62.7   44.4   60.6    44.8
//   503 x 2048 -> 12288    40.4   31.9   36.7   41.5    32.0
//   200 x 2048 -> 12288    36.5   24.2   19.2   23.3    18.9
//   503 x 2048 -> 4096     37.6   21.0   17.5   16.4    16.3
//   390 x 1024 -> 4096     22.5   12.8   11.4    9.4     9.4
enum class Tile { k256x192, k128x128, k128x128Deep, k64x64 };
struct Shape {
  Tile tile;
  int splits;
};
Shape pick_shape(int M, int K, int N) {
  const long cus = device_cu_count() > 0 ? device_cu_count() : 256;
  auto tiles = [&](int bm, int bn) {
    return static_cast<long>((M + bm - 1) / bm) * ((N + bn - 1) / bn);
  };
  auto cost = [&](long t, long slots, double round, double single) {
    const long rest = t % slots;
    return t / slots * round + (rest == 0 ? 0 : rest <= cus ? single : round);
  };
  const long t128 = tiles(128, 128), t64 = tiles(64, 64);
  const double c256 = cost(tiles(256, 192), cus, 46, 46);
  const double c128 = cost(t128, 2 * cus, 36.6, t128 <= cus ? 20.1 : 22);
  const double c64 = cost(t64, 2 * cus, 14.4, 11.3);
  if (c256 < c128 && c256 < c64) return {Tile::k256x192, 1};
  if (c128 < c64) return {t128 <= cus ? Tile::k128x128Deep : Tile::k128x128, 1};
  // A grid of at most half the CUs: K split until every CU has a workgroup, 512 of K each at least, or
  // two, 1024 each (us: 100 x 2048 -> 2048 10.1 unsplit, 5.0 and a reduction of 4 split by 4; 200 x
  // 2048 -> 2048 13.8 by 2, 14.5 by 4; 200 x 6144 -> 2048 24.3 by 2, 21.2 by 4).  One workgroup per CU
  // over a long K: split by two (503 x 6144 -> 2048 31.8 unsplit, 23.4 + 4; 503 x 2048 -> 2048, 11.3
  // and 10.1 + 4, stays whole; a third part would start another round: 390 x 6144 -> 2048 3 us slower).
  long splits = 1;
  if (2 * t64 <= cus)
    splits = std::max({std::min<long>(cus / t64, K / 512), std::min<long>(2 * cus / t64, K / 1024), 1L});
  else if (t64 <= cus && K >= 4096)
    splits = 2;
  return {Tile::k64x64, static_cast<int>(splits)};
}

template <bool SWIGLU>
int launch_shape(const GemmDmaArgs& a, hipStream_t s) {
  const Shape sh = pick_shape(a.M, a.K, a.N);
  switch (sh.tile) {
    case Tile::k256x192: return launch_tile<256, 192, 4, 2, 2, 2, SWIGLU>(a, 1, s);
    case Tile::k128x128: return launch_tile<128, 128, 2, 2, 2, 2, SWIGLU>(a, 1, s);
    case Tile::k128x128Deep: return launch_tile<128, 128, 2, 4, 4, 2, SWIGLU>(a, 1, s);
    default: return launch_tile<64, 64, 2, 2, 4, 2, SWIGLU>(a, sh.splits, s);
  }
}

// Sizes whose byte offsets fit the buffers' 32 bits.
bool fits32(int M, int K, int N) {
  const long lim = (1L << 31) - 1;
  return 2L * M * K <= lim && 2L * N * K <= lim && static_cast<long>(M) * N <= lim;
}

}  // namespace

// An output over an operand stays with the register-staged kernel, whose short grids write it from
// a second launch; here workgroups may still be reading what others write.
bool gemm_dma_takes(const void* in, const void* W, const void* out, size_t out_bytes, int M, int K,
                    int N) {
  const uintptr_t i = reinterpret_cast<uintptr_t>(in), w = reinterpret_cast<uintptr_t>(W),
                  o = reinterpret_cast<uintptr_t>(out);
  auto apart = [&](uintptr_t p, long rows) {
    return p + 2 * rows * K <= o || o + out_bytes <= p;
  };
  return K % 64 == 0 && N % 4 == 0 && ((i | w | o) & 15u) == 0 && fits32(M, K, N) && apart(i, M) &&
         apart(w, N);
}

int launch_gemm_dma(const uint16_t* in, const uint16_t* W, const float* bias, float* out, int M,
                    int K, int N, int act, bool accumulate, hipStream_t s) {
  return launch_shape<false>(
      GemmDmaArgs{in, W, bias, out, nullptr, M, K, N, act, accumulate ? 1 : 0, K}, s);
}

// fp32 activations of up to 128 rows: the cast pass is a launch and a round trip through memory, which
// the fused form saves (us with cold operands, cast + GEMM against fused: 2048 -> 2048 15.3 and 12.8
// at 2 rows, 16.9 and 14.4 at 128; 1024 -> 4096 17.1 and 14.6 at 128).  The A tile takes twice the LDS
// bandwidth and two of three stages' room, so with more rows the pass is cheaper (2048 -> 4096 at 200
// rows 24.0 and 26.3, at 512 30.6 and 34.0; 6144 -> 2048 at 200 29.1 and 34.0).
bool gemm_dma_takes_f32(const float* in, const void* W, const float* out, int M, int K, int N) {
  const uintptr_t ib = reinterpret_cast<uintptr_t>(in), ob = reinterpret_cast<uintptr_t>(out);
  const bool apart = ib + 4 * static_cast<uintptr_t>(M) * K <= ob ||
                     ob + 4 * static_cast<uintptr_t>(M) * N <= ib;
  const size_t out_bytes = 4 * static_cast<size_t>(M) * N;
  return M > 1 && M <= 128 && apart && gemm_dma_takes(in, W, out, out_bytes, M, K, N) &&
         fits32(M, 2 * K, N) && pick_shape(M, K, N).tile == Tile::k64x64;
}

int launch_gemm_dma_f32(const float* in, const uint16_t* W, const float* bias, float* out, int M,
                        int K, int N, int act, hipStream_t s) {
  return launch_tile<64, 64, 2, 2, 3, 2, false, true>(
      GemmDmaArgs{in, W, bias, out, nullptr, M, K, N, act, 0, K}, pick_shape(M, K, N).splits, s);
}

// Short K and many outputs on the larger tiles, whose waves have nothing to do while the tile's stores
// drain, 32 bytes of 32 rows at a time: the register-staged kernel's are faster as long as rows are
// whole 128-byte lines, and its sums are in the same order (us, this kernel and that one: 2048 x 64 ->
// 2048 8.0 and 6.7, 8192 x 128 -> 4096 37.3 and 29.6, 2048 x 192 -> 4096 13.6 and 12.1, 8192 x 256 ->
// 2048 26.6 and 22.2; 717 x 256 -> 4096 8.1 and 8.0, 8192 x 256 -> 1000 12.7 and 14.0; at K = 512
// 15 % either way from card to card).
bool gemm_dma_store_bound(int M, int K, int N) {
  return K <= 256 && N % 32 == 0 && static_cast<long>(M) * N >= 8192L * K &&
         pick_shape(M, K, N).tile != Tile::k64x64;
}

bool gemm_dma_splits(int M, int K, int N) { return pick_shape(M, K, N).splits > 1; }

int launch_gemm_dma_swiglu(const uint16_t* in, const uint16_t* W, uint16_t* out, int M, int K,
                           int I, hipStream_t s) {
  return launch_shape<true>(GemmDmaArgs{in, W, nullptr, out, nullptr, M, K, 2 * I, 0, 0, K}, s);
}

}  // namespace orator_hip
