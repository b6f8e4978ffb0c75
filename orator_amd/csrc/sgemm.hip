// fp32 GEMM (gfx950): out[M,N] = act(sum_k in[m,k] * W[n,k] (+ bias[n])).
//
// Replaces gemm::LaunchSgemm / LaunchSgemmBatched (include/model/gemm.cuh:47-268): the same
// nn.Linear "NT" contract (both operands K-contiguous), activation codes 0 none, 1 SiLU,
// 2 ReLU, 3 sigmoid (gemm.cuh:38-45), strided batches, arbitrary M/N/K and alignment.
//
// fp32 products on the bf16 matrix cores: every operand is split in registers into three bf16
// terms, whose sum is the fp32 value exactly from 2^-103 on, and the six products of terms that
// reach fp32's precision are accumulated in fp32 (what is dropped is below 2^-24 of |x w|, and the
// MFMA adds 32 products per rounding where an fp32 chain rounds at each).  Six bf16 MFMAs take 96
// cycles per 16 x 16 x 32 block, the fp32 MFMA's 256.  Measured against 64 bits (random normal
// operands, relative 2-norm; the fp32 MFMA in parentheses): K = 64 4.7e-8 (1.4e-7), 255 1.6e-7
// (2.9e-7), 512 1.6e-7 (4.1e-7), 2048 2.4e-7 whole and 1.7e-7 split over workgroups (2.9e-7 in
// eight parts), 4096 split 1.7e-7 (4.4e-7).
//
// Results that the terms cannot carry are formed again by the wave on the fp32 MFMA: those that are
// not finite, those so small that operands below 2^-103 may show in them, and all after an operand
// of 2^32 or more.  One more MFMA per fragment finds the large operands (2-4 % of the time; a
// class test of every element's third remainder found the small ones directly and took 12-25 %).
// 717 x 512 -> 2048: 24 us with a NaN in one row, 19 with every second row zero, 36 with every
// operand near 2^-118, against 26, 24 and 26 when every product was formed on the fp32 MFMA.
//
// Workgroup = BM x BN tile of one batch entry; its WK waves share the tile and split K: wave w
// takes the 32-float slices w, w + WK, ..., accumulates the whole tile in registers, and the WK
// partial tiles are added in LDS in wave order (deterministic).  So every element is loaded and
// split by exactly one wave of the workgroup, and the k loop has no barrier: a wave's slice comes
// by buffer loads straight into the wave's own LDS area (8 lanes per 128-byte row piece; read as
// fragments directly from memory, 16 rows per instruction, the same loads ran at 16 bytes per
// clock and CU), goes to registers whole, and the next slice's loads run under the MFMAs.  What
// bounds it: the splitting (about 3.7 VALU instructions per MFMA at 64 x 64) and the MFMAs share
// the issue slots -- a slice of a 64 x 64 tile takes ~2700 cycles per SIMD against 1536 of MFMA
// alone, with the loads removed 9 % less -- and, at the Conformer's sizes, the ~4 us of launch,
// first loads and epilogue.  The bf16 dot product in place of the unpack + subtraction saves a
// fifth of the VALU work but occupies the matrix cores: no faster.  Interleaving VALU and MFMA by
// scheduling groups and wave priorities: no effect.
//
// Measured (us, replayed launches; before: the fp32-MFMA kernel with split K and its reduction):
//   717 x 512 -> 2048   24.9 -> 15.5    717 x 2048 -> 512   25.1 -> 18.2
//   717 x 512 -> 512    12.4 -> 8.0     717 x 512 -> 1536   24.5 -> 14.6
//   1433 x 512 -> 512   15.6 -> 10.6    717 x 512 -> 1024   15.3 -> 10.3
//   126 x 512 -> 2048   11.6 -> 6.1     126 x 2048 -> 512   12.7 -> 10.1
//   126 x 512 -> 512    10.5 -> 5.7     8 x (717 x 717 -> 64)  20.3 -> 13.6
//   8 x (717 x 64 -> 717)  14.2 -> 13.2
//   8 x (1000 x 64 -> 1999)  33.1 -> 28.9 (64 MB of unaligned rows written)
// Behind it still: a few rows at K < 32, which take element loads (8 x (16 x 16 -> 64) 4.2 -> 4.8),
// and 8 x (503 x 64 -> 1005), 11.2 -> 11.7.
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "internal.hpp"
#include "mfma_tile.hpp"

namespace orator_hip {
namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kSK = 32;  // K per slice (floats)

__device__ __forceinline__ float apply_act(float v, int act) {
  if (act == 1) return v / (1.0f + expf(-v));
  if (act == 2) return fmaxf(v, 0.0f);
  if (act == 3) return 1.0f / (1.0f + expf(-v));
  return v;
}

struct SgemmArgs {
  const float* in;
  const float* W;
  const float* bias;
  float* out;
  int M, K, N, act;
  int batch;
  int slices;  // K split over workgroups: batch entry z takes slices z * slices on; 0: not split
  int tiles_n, tiles_m;        // of one batch entry
  uint32_t rec_tiles, rec_run;  // floor(2^32 / d) of their product and of the faster running one
  long s_in, s_w, s_out;
  bool vec;  // K % 32 == 0 and 16-byte aligned operands: 16-byte loads
  // Grouped products (group > 0): `group` problems share `in`; problem z uses weight Wg[z],
  // bias bg[z] and output og[z] (batch = group, blockIdx.z selects the problem).
  int group;
  const float* Wg[3];
  const float* bg[3];
  float* og[3];
  // Residual update (residual != 0): out = out + res_scale * (in W^T + bias), act 0.
  int residual;
  float res_scale;
  // GLU (the GLU epilogue): W has 2 glu_c rows (value rows, then gate rows); out[m][c] =
  // a * (1 / (1 + exp(-b))) with a, b the value and gate outputs (bias added), 0 for rows
  // m >= glu_valid; out is [M][glu_c].
  int glu_c, glu_valid;
  // LayerNorm of the updated rows (ln_g non-null), a launch of its own after the product:
  // ln_out[m] = LayerNorm(out[m]) g + b; ln_out may be out.
  const float* ln_g;
  const float* ln_b;
  float* ln_out;
  float ln_eps;
  // fp16 outputs: bit z set stores problem z's output (group products; bit 0 otherwise) as
  // fp16, each value rounded to nearest even once; products without residual only.
  int h16;
};

// Eight fp32 values as three bf16 terms each (8 + 8 + 8 significant bits, each term the rest
// rounded to nearest): x = h + m + l exactly for |x| >= 2^-103 and within 2^-134 below (half the
// spacing of bf16's subnormals, which the MFMA takes and gives as they are).  Where |x| rounds past
// bf16's range, h is infinite and m and l are NaN.
struct Split {
  bf16x8_t h, m, l;
};
__device__ __forceinline__ Split split_bf16x3(float4 u, float4 v) {
  const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
  uint32_t h[4], m[4], l[4];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    h[w] = cvt_bf16x2(x[2 * w], x[2 * w + 1]);
    const float r0 = x[2 * w] - bf16_lo(h[w]), r1 = x[2 * w + 1] - bf16_hi(h[w]);
    m[w] = cvt_bf16x2(r0, r1);
    l[w] = cvt_bf16x2(r0 - bf16_lo(m[w]), r1 - bf16_hi(m[w]));
  }
  return {as_bf16x8(make_uint4(h[0], h[1], h[2], h[3])),
          as_bf16x8(make_uint4(m[0], m[1], m[2], m[3])),
          as_bf16x8(make_uint4(l[0], l[1], l[2], l[3]))};
}

// LONG: K from 2^24 on, where 64 rows no longer fit 32-bit byte offsets: the same loads by 64-bit
// addresses.
template <int BM, int BN, int WK, bool VEC, bool GLU, bool LONG>
__global__ __launch_bounds__(64 * WK, 2) void sgemm_nt_kernel(SgemmArgs a) {
  constexpr int NT = 64 * WK;
  constexpr int FM = BM / 16, FN = BN / 16;
  // per wave: a slice of BM + BN rows of 128 bytes while k runs, then its fp32 output tile (rows
  // padded by 4 floats: the 16 rows a quarter-wave writes 16 bytes of land on distinct bank
  // groups)
  constexpr int kCLd = BN + 4;
  constexpr int kSliceFloats = (BM + BN) * kSK, kTileFloats = BM * kCLd;
  constexpr int kWaveFloats = kSliceFloats > kTileFloats ? kSliceFloats : kTileFloats;
  __shared__ __align__(16) float smem[WK][kWaveFloats];

  // Workgroups are dealt to the 8 XCDs in turn: give each a contiguous piece of the tile order
  // (batch entries, then tiles with the operand of more rows running slowest), so the tiles that
  // share an L2 share rows of it, and the lines that neighbours write in part meet there.
  const uint32_t total = gridDim.x * gridDim.y * gridDim.z;
  const uint32_t lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  const uint32_t xcd = lin & 7;
  const uint32_t at = xcd * (total >> 3) + min(xcd, total & 7) + (lin >> 3);
  const bool n_slow = a.N > a.M;
  // n / d by its reciprocal, at most one short (scalar instructions; the compiler's own division
  // is a chain of vector ones)
  auto div = [](uint32_t n, uint32_t d, uint32_t rec) {
    const uint32_t q = __umulhi(n, rec);
    return q + (n - q * d >= d);
  };
  const uint32_t per_batch = a.tiles_n * a.tiles_m, run = n_slow ? a.tiles_m : a.tiles_n;
  const int batch = a.batch == 1 ? 0 : div(at, per_batch, a.rec_tiles);
  const uint32_t in_batch = at - batch * per_batch;
  const int slow = div(in_batch, run, a.rec_run), fast = in_batch - slow * run;
  const int tile_n = n_slow ? slow : fast, tile_m = n_slow ? fast : slow;
  const float* A = a.in + batch * a.s_in;
  const float* B = a.group ? a.Wg[batch] : a.W + batch * a.s_w;
  const int M = a.M, N = a.N, K = a.K;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = tile_m * BM, n0 = tile_n * BN;
  // GLU: tile rows [0, BN/2) are value rows from c0 on, [BN/2, BN) the matching gate rows
  constexpr int BW = GLU ? BN / 2 : BN;  // rows of one block of W rows
  const int w0 = tile_n * BW, w_last = (GLU ? a.glu_c : N) - 1;
  // Rows behind tile rows, clamped into range (outputs past M and N are never stored)
  auto a_row = [&](int t) { return A + static_cast<long>(min(m0 + t, M - 1)) * K; };
  auto w_row = [&](int t) {
    const long r = min(w0 + t % BW, w_last) + (t >= BW ? a.glu_c : 0);
    return B + r * K;
  };
  // the slice's rows through buffer loads straight into LDS; offsets count from the tile's
  // first row, so they fit 32 bits whatever the matrix's size
  const uint32_t row_bytes = static_cast<uint32_t>(K) * 4;
  auto rsrc = [&](const float* p, int rows) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, rows * row_bytes,
                                             0x00020000);
  };
  const int rows_a = min(BM, M - m0), rows_w = min(BW, w_last + 1 - w0);
  const __amdgpu_buffer_rsrc_t rs_a = rsrc(A + static_cast<long>(m0) * K, rows_a);
  const __amdgpu_buffer_rsrc_t rs_w = rsrc(B + static_cast<long>(w0) * K, rows_w);
  const __amdgpu_buffer_rsrc_t rs_g =
      GLU ? rsrc(B + (static_cast<long>(a.glu_c) + w0) * K, rows_w) : rs_w;
  // LDS row = 8 chunks of 16 bytes, chunk c in slot c ^ swz(row): fragment reads (16 rows, one
  // chunk) then hit distinct banks
  auto swz = [](int row) { return (row & 7) ^ ((row >> 3) & 1); };
  float* const mine = smem[wave];
  auto dma = [&](int s) {
    // VEC: 8 rows per instruction, 8 lanes x 16 bytes each; else 2 rows, 32 lanes x 4 bytes,
    // elements past K as zeros (an offset past the buffer)
    constexpr int RPI = VEC ? 8 : 2, LPR = 64 / RPI;
#pragma unroll
    for (int q = 0; q < (BM + BN) / RPI; ++q) {
      const int t = q * RPI;  // tile row of the instruction: A rows, then W rows
      const bool is_a = t < BM;
      const int r = (is_a ? t : (t - BM) % BW) + lane / LPR;
      const int row = min(r, (is_a ? rows_a : rows_w) - 1);
      const int lds_row = t + lane / LPR;
      uint32_t off, soff = 0;
      if constexpr (VEC) {
        off = row * row_bytes + 16 * ((lane % LPR) ^ swz(lds_row));
        soff = static_cast<uint32_t>(s) * (kSK * 4);
      } else {
        const int e = lane % LPR, k = s * kSK + 4 * ((e >> 2) ^ swz(lds_row)) + (e & 3);
        off = k < K ? row * row_bytes + 4 * k : 0xfffffffcu;
      }
      const __amdgpu_buffer_rsrc_t rs = is_a ? rs_a : t - BM < BW ? rs_w : rs_g;
      const auto dst = (__attribute__((address_space(3))) void*)(mine + t * kSK);
      if constexpr (LONG) {
        const int c = (lane % LPR) / (VEC ? 1 : 4) ^ swz(lds_row);
        const int k = s * kSK + (VEC ? 4 * c : 4 * c + lane % 4);
        const float* src =
            (is_a ? a_row(row) : w_row(row + (t - BM) / BW * BW)) + min(k, K - 1);
        const auto from = (__attribute__((address_space(1))) void*)(src);
        if constexpr (VEC)
          __builtin_amdgcn_global_load_lds(from, dst, 16, 0, 0);
        else
          __builtin_amdgcn_global_load_lds(from, dst, 4, 0, 0);
      } else if constexpr (VEC)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 16, off, soff, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, dst, 4, off, soff, 0, 0);
    }
  };
  // Fragment: lane = (row lane % 16, group lane / 16); group g takes floats 4g .. 4g + 3 and
  // 16 + 4g .. of the slice (the same k for A and W, so any assignment serves)
  const int fr = lane & 15, fg = lane >> 4;
  f32x4_t acc[FM][FN];
  [[maybe_unused]] f32x4_t sum[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) sum[i][j] = acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int n_all = K / kSK + (K % kSK != 0);
  const int first = a.slices ? batch * a.slices + wave : wave;  // this wave's: first, + WK, ...
  const int n_sl = a.slices ? min(n_all, (batch + 1) * a.slices) : n_all;
  // Sum of h * 2^96 over every operand of the wave, one MFMA per fragment: not finite once an
  // operand reaches 2^32 (or the sum does): a product that overflows stays infinite or becomes NaN,
  // also beside its opposite in one MFMA (measured for every pair of places).
  f32x4_t guard = {0.f, 0.f, 0.f, 0.f};
  constexpr uint32_t kGuard = 0x6f806f80u;
  const bf16x8_t big = as_bf16x8(make_uint4(kGuard, kGuard, kGuard, kGuard));
  if (first < n_sl) dma(first);
  for (int s = first; s < n_sl; s += WK) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // The whole slice to registers as bf16 terms, then the next slice's loads under the MFMAs:
    // the six products of terms that reach fp32's precision (the dropped m l, l m and l l are
    // below 2^-24 of |x w|), smallest first.  The W fragment is the MFMA's row operand, so a
    // lane ends up with 4 consecutive columns of one output row.
    float4 raw_a[FM][2], raw_w[FN][2];
    auto fetch = [&](float4(&raw)[2], int t) {
      const float* row = mine + (t + fr) * kSK;
      const int x = swz(t + fr);
      raw[0] = *reinterpret_cast<const float4*>(row + 4 * (fg ^ x));
      raw[1] = *reinterpret_cast<const float4*>(row + 4 * ((4 + fg) ^ x));
    };
#pragma unroll
    for (int j = 0; j < FN; ++j) fetch(raw_w[j], BM + 16 * j);
#pragma unroll
    for (int i = 0; i < FM; ++i) fetch(raw_a[i], 16 * i);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (n_sl - s > WK) dma(s + WK);
    if (LONG && !VEC && s >= K / kSK) {  // elements past K came as copies of the last one
      auto mask = [&](float4(&raw)[2]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int left = K - (s * kSK + 16 * h + 4 * fg);
          raw[h] = make_float4(left > 0 ? raw[h].x : 0.f, left > 1 ? raw[h].y : 0.f,
                               left > 2 ? raw[h].z : 0.f, left > 3 ? raw[h].w : 0.f);
        }
      };
#pragma unroll
      for (int j = 0; j < FN; ++j) mask(raw_w[j]);
#pragma unroll
      for (int i = 0; i < FM; ++i) mask(raw_a[i]);
    }
    Split sa[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      sa[i] = split_bf16x3(raw_a[i][0], raw_a[i][1]);
      guard = __builtin_amdgcn_mfma_f32_16x16x32_bf16(big, sa[i].h, guard, 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const Split w = split_bf16x3(raw_w[j][0], raw_w[j][1]);
      guard = __builtin_amdgcn_mfma_f32_16x16x32_bf16(big, w.h, guard, 0, 0, 0);
      auto mma = [&](const bf16x8_t& x, auto term) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, sa[i].*term, acc[i][j], 0, 0, 0);
      };
      mma(w.l, &Split::h);
      mma(w.h, &Split::l);
      mma(w.m, &Split::m);
      mma(w.m, &Split::h);
      mma(w.h, &Split::m);
      mma(w.h, &Split::h);
    }
    if constexpr (WK == 1) {  // (two slices at most) as two waves would add them
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          sum[i][j] += acc[i][j];
          acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
  if constexpr (WK == 1) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = sum[i][j];
  }
  // Per-wave partial tiles to LDS, then the sum over the waves (in wave order) and the
  // epilogue, a thread per 4 columns
  float low = INFINITY, odd = 0.0f;  // the smallest magnitude; NaN where a value is not finite
  auto part = [&](int i, int j) -> f32x4_t& {
    return *reinterpret_cast<f32x4_t*>(mine + (16 * i + fr) * kCLd + 16 * j + 4 * fg);
  };
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      part(i, j) = acc[i][j];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        low = fminf(low, fabsf(acc[i][j][e]));
        odd = fmaf(acc[i][j][e], 0.0f, odd);
      }
    }
  float wide = 0.0f;  // NaN after an operand of 2^32 or more
#pragma unroll
  for (int e = 0; e < 4; ++e) wide = fmaf(guard[e], 0.0f, wide);
  // Operands below 2^-103, whose terms do not sum to them, cost a value at most K 2^-101 while the
  // others stay below 2^32: below 2^-26 of it from `small` on.  Smaller ones, ones that are not
  // finite and, after an operand of 2^32 or more, all are formed again from the fp32 operands.
  const float small = static_cast<float>(K) * 0x1p-75f;
  if (first < n_sl && __any(odd + wide != 0.0f || low < small)) [[unlikely]] {
    // straight from memory; group fg takes floats 4 fg .. 4 fg + 3 of half a slice
    auto load = [&](const float* row, int k) {
      if (VEC) return *reinterpret_cast<const float4*>(row + k);
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = row[min(k + e, K - 1)];  // no branch: the loads are all in flight together
        v[e] = k + e < K ? v[e] : 0.0f;
      }
      return make_float4(v[0], v[1], v[2], v[3]);
    };
    const bool all = __any(wide != 0.0f);
    float least = INFINITY;  // of the values other than zero
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float v = fabsf(part(i, j)[e]);
          least = v != 0.0f ? fminf(least, v) : least;
        }
    bool again = LONG || all || __any(odd != 0.0f || least < small);
    if (!again) {  // zeros: right unless there are operands below 2^-103 other than zero
      uint32_t key = 0xffffffffu;  // least 2 |bits| - 1: zeros last
      constexpr int RPI = VEC ? 8 : 2, LPR = 64 / RPI, Q = (BM + BN) / RPI;
#pragma unroll 1
      for (int s = first; s < n_sl; s += WK) {
        // past the last row a buffer load gives zero; past K the last element serves
        const uint32_t off =
            lane / LPR * row_bytes +
            (VEC ? s * (4 * kSK) + 16 * (lane % LPR) : 4 * min(s * kSK + lane % LPR, K - 1));
        typename std::conditional_t<VEC, u32x4_t, uint32_t> x[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          const int t = q * RPI;  // tile row of the instruction: A rows, then W rows
          const __amdgpu_buffer_rsrc_t rs = t < BM ? rs_a : t - BM < BW ? rs_w : rs_g;
          const uint32_t at = off + (t < BM ? t : (t - BM) % BW) * row_bytes;
          if constexpr (VEC)
            x[q] = __builtin_amdgcn_raw_buffer_load_b128(rs, at, 0, 0);
          else
            x[q] = __builtin_amdgcn_raw_buffer_load_b32(rs, at, 0, 0);
        }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
          if constexpr (VEC) {
#pragma unroll
            for (int e = 0; e < 4; ++e) key = min(key, 2 * x[q][e] - 1);
          } else {
            key = min(key, 2 * x[q] - 1);
          }
        }
      }
      again = __any(key < 2 * __float_as_uint(0x1p-103f) - 1);
    }
    if (again) {
      f32x4_t ex[FM][FN];
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) ex[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      // the next half on its way under the current one's MFMAs
      float4 next_a[FM], next_w[FN];
      auto fetch = [&](int k) {
#pragma unroll
        for (int i = 0; i < FM; ++i) next_a[i] = load(a_row(16 * i + fr), k + 4 * fg);
#pragma unroll
        for (int j = 0; j < FN; ++j) next_w[j] = load(w_row(16 * j + fr), k + 4 * fg);
      };
      fetch(first * kSK);
#pragma unroll 1
      for (int h = 0, s = first; s < n_sl; s += WK * h, h ^= 1) {
        float4 va[FM], vw[FN];
#pragma unroll
        for (int i = 0; i < FM; ++i) va[i] = next_a[i];
#pragma unroll
        for (int j = 0; j < FN; ++j) vw[j] = next_w[j];
        if (h == 0)
          fetch(s * kSK + kSK / 2);
        else if (n_sl - s > WK)
          fetch((s + WK) * kSK);
        auto mma = [&](auto f) {
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
              ex[i][j] =
                  __builtin_amdgcn_mfma_f32_16x16x4f32(vw[j].*f, va[i].*f, ex[i][j], 0, 0, 0);
        };
        mma(&float4::x), mma(&float4::y), mma(&float4::z), mma(&float4::w);
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          f32x4_t v = part(i, j);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (all || !(fabsf(v[e]) >= small && fabsf(v[e]) < INFINITY)) v[e] = ex[i][j][e];
          part(i, j) = v;
        }
    }
  }
  __syncthreads();
  auto total_of = [&](int r, int c, float (&v)[4]) {
    f32x4_t t = *reinterpret_cast<const f32x4_t*>(smem[0] + r * kCLd + c);
#pragma unroll
    for (int w = 1; w < WK; ++w) t += *reinterpret_cast<const f32x4_t*>(smem[w] + r * kCLd + c);
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = t[q];
  };
  if constexpr (GLU) {
    // columns [0, BN/2) of the tile are the value outputs of channels c0 .., [BN/2, BN) the
    // gate outputs of the same channels; the same fp32 values and formula as a plain product
    // followed by the GLU pass (its bias added, then a * (1 / (1 + exp(-b))))
    constexpr int HB = BN / 2, TPRg = HB / 4, RPIg = NT / TPRg;
    const int Cg = a.glu_c, c0 = tile_n * HB;
    const int orow = tid / TPRg, j = 4 * (tid % TPRg);
    float ba[4] = {0.f, 0.f, 0.f, 0.f}, bg[4] = {0.f, 0.f, 0.f, 0.f};
    if (a.bias) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        ba[q] = a.bias[min(c0 + j + q, Cg - 1)];
        bg[q] = a.bias[Cg + min(c0 + j + q, Cg - 1)];
      }
    }
    const bool vec_out = (Cg % 4) == 0 && ((reinterpret_cast<uintptr_t>(a.out)) & 15) == 0;
    for (int r = orow; r < BM; r += RPIg) {
      const int m = m0 + r;
      if (m >= M) continue;
      float av[4], gv[4], o[4];
      total_of(r, j, av);
      total_of(r, HB + j, gv);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float x = av[q] + ba[q], g = gv[q] + bg[q];
        o[q] = m < a.glu_valid ? x * (1.0f / (1.0f + __expf(-g))) : 0.0f;
      }
      float* dst = a.out + static_cast<long>(m) * Cg + c0 + j;
      if (vec_out && c0 + j + 3 < Cg) {
        *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (c0 + j + q < Cg) dst[q] = o[q];
      }
    }
    return;
  }
  float* C = a.group ? a.og[batch] : a.out + batch * a.s_out;
  const float* bias = a.group ? a.bg[batch] : a.bias;
  const bool h16 = (a.h16 >> (a.group ? batch : 0)) & 1;
  // The rows in two forms: without options, and with every option looked at per element (8 x (717 x
  // 64 -> 1433): 22.8 us, 19.4 without, scalar division included).
  const bool plain = !a.act && !a.residual && !h16;
  auto finish = [&](float v, float b, const float* old, auto simple) {
    if constexpr (simple) return v + b;
    v = apply_act(v + b, a.act);
    return a.residual ? fmaf(a.res_scale, v, *old) : v;
  };
  const int rows = min(BM, M - m0);
  if ((N % 4) == 0 && (reinterpret_cast<uintptr_t>(C) & (h16 ? 7 : 15)) == 0) {
    // 4 columns per thread, one 16-byte (fp16: 8-byte) store
    constexpr int TPRo = BN / 4, RPIo = NT / TPRo;
    const int orow = tid / TPRo, ocol = 4 * (tid % TPRo);
    const int n = n0 + ocol;
    if (n >= N) return;
    float bv[4] = {0.f, 0.f, 0.f, 0.f};
    if (bias) {
#pragma unroll
      for (int q = 0; q < 4; ++q) bv[q] = bias[n + q];
    }
    auto store = [&](auto simple) {
      for (int r = orow; r < rows; r += RPIo) {
        const long at = static_cast<long>(m0 + r) * N + n;
        float v[4];
        total_of(r, ocol, v);
#pragma unroll
        for (int q = 0; q < 4; ++q) v[q] = finish(v[q], bv[q], C + at + q, simple);
        if (!simple && h16) {
          typedef _Float16 h4_t __attribute__((ext_vector_type(4)));
          const h4_t hv = {static_cast<_Float16>(v[0]), static_cast<_Float16>(v[1]),
                           static_cast<_Float16>(v[2]), static_cast<_Float16>(v[3])};
          *reinterpret_cast<h4_t*>(reinterpret_cast<_Float16*>(C) + at) = hv;
        } else {
          *reinterpret_cast<float4*>(C + at) = make_float4(v[0], v[1], v[2], v[3]);
        }
      }
    };
    plain ? store(std::true_type{}) : store(std::false_type{});
    return;
  }
  // other row lengths and alignments: a column per thread, so that a store instruction still
  // writes whole row pieces
  constexpr int RPS = NT / BN;  // rows per pass
  const int c = tid % BN, n = n0 + c;
  if (n >= N) return;
  const float b = bias ? bias[n] : 0.0f;
  constexpr int U = BM / RPS < 4 ? BM / RPS : 4;
  auto store = [&](auto simple) {
    for (int r0 = tid / BN; r0 < rows; r0 += U * RPS) {
      float v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int r = r0 + u * RPS;
        v[u] = smem[0][r * kCLd + c];
#pragma unroll
        for (int w = 1; w < WK; ++w) v[u] += smem[w][r * kCLd + c];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int r = r0 + u * RPS;
        if (r >= rows) break;
        const long at = static_cast<long>(m0 + r) * N + n;
        const float x = finish(v[u], b, C + at, simple);
        if (!simple && h16)
          reinterpret_cast<_Float16*>(C)[at] = static_cast<_Float16>(x);
        else
          C[at] = x;
      }
    }
  };
  plain ? store(std::true_type{}) : store(std::false_type{});
}

template <int BM, int BN, int WK, bool VEC, bool GLU, bool LONG = false>
int launch_tile(SgemmArgs a, hipStream_t s) {
  const int bn = GLU ? BN / 2 : BN, cols = GLU ? a.glu_c : a.N;
  a.tiles_n = (cols + bn - 1) / bn;
  a.tiles_m = (a.M + BM - 1) / BM;
  auto rec = [](uint64_t d) {
    return static_cast<uint32_t>(std::min<uint64_t>((1ull << 32) / d, 0xffffffffu));
  };
  a.rec_tiles = rec(static_cast<uint64_t>(a.tiles_n) * a.tiles_m);
  a.rec_run = rec(a.N > a.M ? a.tiles_m : a.tiles_n);
  const dim3 grid(a.tiles_n, a.tiles_m, a.batch);
  hipLaunchKernelGGL((sgemm_nt_kernel<BM, BN, WK, VEC, GLU, LONG>), grid, dim3(64 * WK), 0, s, a);
  return check_launch("sgemm_nt_kernel");
}

// Tile and waves by K and grid.  Many small tiles keep every CU busy where the grid is short;
// larger tiles split fewer elements per MFMA.  Eight waves per tile shorten a short grid's time
// (126 x 512 -> 512: 5.8 us, 6.1 with four) and, for long K, keep the partial sums short; four let
// two to five workgroups share a CU, so that one's first loads and epilogue run under the others'
// MFMAs (717 x 512 -> 2048: 32 x 64 tiles, four waves 17.5 us, eight 20.8; 2000 x 512 -> 2048: 64 x
// 64, four waves 34.6, eight 43.3, 32 x 64 38.3; 717 x 512 -> 1536: 32 x 32, four waves 15.8, eight
// 17.3, 32 x 64 16.2; 717 x 2048 -> 512: 32 x 64, eight waves 17.6, 32 x 32 20.0, 64 x 64 25.6).
// Short K: the instructions around the few slices and the outputs bound it, so 32 x 32 tiles with a
// wave per slice while the grid is short, then wave tiles of 32 x 64, from 15 tiles per CU on one
// wave for both slices (8 x (600 x 64 -> 600): 32 x 32 with two waves 9.5 us, 32 x 64 with two 8.4;
// 8 x (1000 x 64 -> 1999): 32 x 32 two waves 31.6, 32 x 64 two 32.4, one 28.5; 1999 x 30 -> 2048:
// 13.9 and, one wave, 10.7).
template <bool VEC, bool GLU>
int launch_sized(const SgemmArgs& a, hipStream_t s) {
  const long cus = device_cu_count() > 0 ? device_cu_count() : 256;
  auto tiles = [&](int bm, int bn) {
    return static_cast<long>((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn) * a.batch;
  };
  if (a.K >= 1 << 24) return launch_tile<32, 32, 8, VEC, GLU, true>(a, s);
  if (a.K >= 1024) {
    if (tiles(32, 32) <= cus) return launch_tile<32, 32, 8, VEC, GLU>(a, s);
    if (tiles(32, 64) <= 2 * cus) return launch_tile<32, 64, 8, VEC, GLU>(a, s);
    return launch_tile<64, 64, 8, VEC, GLU>(a, s);
  }
  if (a.K >= 256) {
    if (2 * tiles(32, 32) <= 3 * cus) return launch_tile<32, 32, 8, VEC, GLU>(a, s);
    if (tiles(32, 32) <= 5 * cus) return launch_tile<32, 32, 4, VEC, GLU>(a, s);
    if (tiles(32, 64) <= 4 * cus) return launch_tile<32, 64, 4, VEC, GLU>(a, s);
    return launch_tile<64, 64, 4, VEC, GLU>(a, s);
  }
  const long t = tiles(32, 32);
  if (a.K <= kSK) {
    if (t <= 8 * cus) return launch_tile<32, 32, 1, VEC, GLU>(a, s);
    return launch_tile<32, 64, 1, VEC, GLU>(a, s);
  }
  if (t <= 4 * cus) return launch_tile<32, 32, 4, VEC, GLU>(a, s);
  if (a.K <= 2 * kSK && t > 15 * cus) return launch_tile<32, 64, 1, VEC, GLU>(a, s);
  if (a.K <= 2 * kSK && t > 8 * cus) return launch_tile<32, 64, 2, VEC, GLU>(a, s);
  return launch_tile<32, 32, 2, VEC, GLU>(a, s);
}

// out_b[i] = act(sum_z part[z][b][i] + bias), z ascending, or the residual update.
__global__ __launch_bounds__(256) void sgemm_reduce_kernel(SgemmArgs a, const float* part,
                                                           int splits) {
  const long MN = static_cast<long>(a.M) * a.N, all = MN * a.batch;
  const long i = static_cast<long>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= all) return;
  float v = part[i];
  for (int z = 1; z < splits; ++z) v += part[z * all + i];
  v = apply_act(v + (a.bias ? a.bias[i % a.N] : 0.0f), a.act);
  float* out = a.out + (a.batch > 1 ? i / MN * a.s_out + i % MN : i);
  *out = a.residual ? fmaf(a.res_scale, v, *out) : v;
}

// Through partial products in memory, for one of two reasons.  Long K on a short grid: parts of K,
// 1024 each at least, on workgroups of their own, as many as the CUs take in one round, and a
// second launch that adds them (us, whole and split: 126 x 2048 -> 512 12.0 and 10.1, 1 x 4096 ->
// 1024 19.0 and 10.7, 64 x 16384 -> 64 65.7 and 13.4; one row and two columns at K = 2^24 63 ms and
// 0.32).  And outputs that lie over an operand, which other workgroups may still be reading.
int run_parts(const SgemmArgs& a, int splits, float* part, hipStream_t s) {
  SgemmArgs p = a;
  if (splits > 1) {
    const int n_sl = a.K / kSK + (a.K % kSK != 0);
    p.slices = (n_sl + splits - 1) / splits;
    splits = (n_sl + p.slices - 1) / p.slices;
    p.batch = splits;
  }
  const long MN = static_cast<long>(a.M) * a.N, all = MN * a.batch;
  p.out = part;
  p.s_out = MN;
  p.bias = nullptr;
  p.act = p.residual = 0;
  const bool far = a.K >= 1 << 24;
  int rc;
  if (splits == 1)
    rc = a.vec ? launch_sized<true, false>(p, s) : launch_sized<false, false>(p, s);
  else if (a.vec)
    rc = far ? launch_tile<32, 32, 8, true, false, true>(p, s)
             : launch_tile<32, 32, 8, true, false>(p, s);
  else
    rc = far ? launch_tile<32, 32, 8, false, false, true>(p, s)
             : launch_tile<32, 32, 8, false, false>(p, s);
  if (rc) return rc;
  hipLaunchKernelGGL(sgemm_reduce_kernel, dim3(static_cast<unsigned>((all + 255) / 256)),
                     dim3(256), 0, s, a, part, splits);
  return check_launch("sgemm_reduce_kernel");
}

// Whether [p, p + n) and [q, q + m) floats share memory.
bool overlap(const float* p, long n, const float* q, long m) { return p < q + m && q < p + n; }

int run_sgemm(SgemmArgs a, int batch, bool glu, hipStream_t s) {
  a.batch = batch;
  const long cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const long tiles = static_cast<long>((a.M + 31) / 32) * ((a.N + 31) / 32);
  long splits = std::min<long>(cus / tiles, a.K / 1024);
  if (splits < 1 || batch > 1) splits = 1;
  // operands and outputs of the plain product (of all its batch entries)
  const bool plain = !glu && !a.group && !a.h16;
  auto span = [&](long stride, long rows, long cols) { return (batch - 1) * stride + rows * cols; };
  const long out_n = span(a.s_out, a.M, a.N);
  const bool over = plain && (overlap(a.out, out_n, a.in, span(a.s_in, a.M, a.K)) ||
                              overlap(a.out, out_n, a.W, span(a.s_w, a.N, a.K)));
  float* part = nullptr;
  if (plain && (splits > 1 || over)) {
    const size_t bytes = splits * batch * sizeof(float) * a.M * a.N;
    // without room, as in a capture before the first call, a split product stays whole
    if (over || workspace_at_hand(s, bytes, kWsGemm)) {
      part = static_cast<float*>(workspace(s, bytes, kWsGemm));
      if (!part && over) return ORATOR_ERR_HIP;
    }
  }
  const int rc = part ? run_parts(a, static_cast<int>(splits), part, s)
                 : glu ? launch_sized<true, true>(a, s)
                 : a.vec ? launch_sized<true, false>(a, s) : launch_sized<false, false>(a, s);
  if (rc || !a.ln_g) return rc;
  return launch_layer_norm(a.out, a.ln_g, a.ln_b, a.ln_out, a.M, a.N, a.ln_eps, s);
}

}  // namespace

int launch_sgemm(const float* in, const float* W, const float* bias, float* out, int M, int K,
                 int N, int act, int batch, long stride_in, long stride_w, long stride_out,
                 hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0 || batch <= 0) return ORATOR_OK;
  if (!in || !W || !out) return fail(ORATOR_ERR_INVALID, "sgemm: null pointer");
  if (act < 0 || act > 3) return fail(ORATOR_ERR_INVALID, "sgemm: act must be 0..3");
  if (batch > 65535) return fail(ORATOR_ERR_UNSUPPORTED, "sgemm: at most 65535 batches");
  SgemmArgs a{};
  a.in = in;
  a.W = W;
  a.bias = bias;
  a.out = out;
  a.M = M;
  a.K = K;
  a.N = N;
  a.act = act;
  a.s_in = batch > 1 ? stride_in : 0;
  a.s_w = batch > 1 ? stride_w : 0;
  a.s_out = batch > 1 ? stride_out : 0;
  a.vec = (K % kSK) == 0 && ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(W) |
                            (batch > 1 ? (stride_in | stride_w) * 4 : 0)) & 15) == 0;
  return run_sgemm(a, batch, false, stream);
}

int launch_sgemm_residual_ln(const float* in, const float* W, const float* bias, float* out,
                             int M, int K, int N, float res_scale, const float* ln_g,
                             const float* ln_b, float* ln_out, float eps, hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0) return ORATOR_OK;
  if (!in || !W || !out || !ln_g || !ln_b || !ln_out)
    return fail(ORATOR_ERR_INVALID, "sgemm_residual_ln: null pointer");
  SgemmArgs a{};
  a.in = in;
  a.W = W;
  a.bias = bias;
  a.out = out;
  a.M = M;
  a.K = K;
  a.N = N;
  a.residual = 1;
  a.res_scale = res_scale;
  a.ln_g = ln_g;
  a.ln_b = ln_b;
  a.ln_out = ln_out;
  a.ln_eps = eps;
  a.vec = (K % kSK) == 0 &&
          ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(W)) & 15) == 0;
  return run_sgemm(a, 1, false, stream);
}

int launch_sgemm_glu(const float* in, const float* W, const float* bias, float* out, int M, int K,
                     int C, int valid, hipStream_t stream) {
  if (M <= 0 || C <= 0 || K <= 0) return ORATOR_OK;
  if (!in || !W || !out) return fail(ORATOR_ERR_INVALID, "sgemm_glu: null pointer");
  if ((K % kSK) != 0 ||
      ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(W)) & 15) != 0)
    return ORATOR_ERR_UNSUPPORTED;  // no 16-byte loads: the caller takes the two-pass path
  SgemmArgs a{};
  a.in = in;
  a.W = W;
  a.bias = bias;
  a.out = out;
  a.M = M;
  a.K = K;
  a.N = 2 * C;
  a.vec = true;
  a.glu_c = C;
  a.glu_valid = valid;
  return run_sgemm(a, 1, true, stream);
}

int launch_sgemm_group3(const float* in, const float* const W[3], const float* const bias[3],
                        void* const out[3], int M, int K, int N, int h16_mask,
                        hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0) return ORATOR_OK;
  if (!in) return fail(ORATOR_ERR_INVALID, "sgemm: null pointer");
  SgemmArgs a{};
  a.in = in;
  a.M = M;
  a.K = K;
  a.N = N;
  a.group = 3;
  a.h16 = h16_mask & 7;
  uintptr_t align = reinterpret_cast<uintptr_t>(in);
  for (int g = 0; g < 3; ++g) {
    if (!W[g] || !out[g]) return fail(ORATOR_ERR_INVALID, "sgemm: null pointer");
    a.Wg[g] = W[g];
    a.bg[g] = bias[g];
    a.og[g] = static_cast<float*>(out[g]);
    align |= reinterpret_cast<uintptr_t>(W[g]);
  }
  a.W = a.Wg[0];
  a.vec = (K % kSK) == 0 && (align & 15) == 0;
  return run_sgemm(a, 3, false, stream);
}

int launch_sgemm_f16_out(const float* in, const float* W, void* out, int M, int K, int N,
                         hipStream_t stream) {
  if (M <= 0 || N <= 0 || K <= 0) return ORATOR_OK;
  if (!in || !W || !out) return fail(ORATOR_ERR_INVALID, "sgemm: null pointer");
  SgemmArgs a{};
  a.in = in;
  a.W = W;
  a.out = static_cast<float*>(out);
  a.M = M;
  a.K = K;
  a.N = N;
  a.h16 = 1;
  a.vec = (K % kSK) == 0 &&
          ((reinterpret_cast<uintptr_t>(in) | reinterpret_cast<uintptr_t>(W)) & 15) == 0;
  return run_sgemm(a, 1, false, stream);
}

}  // namespace orator_hip

using namespace orator_hip;

extern "C" {

int orator_sgemm(const float* in, const float* W, const float* bias, float* out, int M, int K,
                 int N, int act, void* stream) {
  return launch_sgemm(in, W, bias, out, M, K, N, act, 1, 0, 0, 0, static_cast<hipStream_t>(stream));
}

int orator_sgemm_batched(const float* in, const float* W, float* out, int M, int K, int N, int act,
                         int batch, long stride_in, long stride_w, long stride_out, void* stream) {
  return launch_sgemm(in, W, nullptr, out, M, K, N, act, batch, stride_in, stride_w, stride_out,
                      static_cast<hipStream_t>(stream));
}

}  // extern "C"
