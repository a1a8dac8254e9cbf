// W4A8 product for 2..64 tokens on the gfx950 matrix cores, groups of 32, 64
// or 128 and any number of them: the same exact lane sums and the same f32
// epilogue order as the other W4A8 kernels (gemm.rs:458-784), so the outputs
// equal the CPU path bit for bit.
//
// Work split.  A wave owns 16 weight rows and 16 tokens and walks K four
// groups a step: lane (j = lane % 16, h = lane / 16) streams row j's codes and
// parameters of group 4q + h, and token j's scale and input sum of that group.
// For reference lane l, v_mfma_f32_16x16x4_4b_f16 multiplies four independent
// 16 x 16 x 4 products, one per group: two of them (columns 0, 4, 1, 5 and 2,
// 6, 3, 7 of the 8-column block l), or four at group 128 (blocks l and l + 8),
// give S_l of the 16 tokens and rows for all four groups with no padding in
// K.  Lane (j, h) then holds, in registers 4g + r, token 4h + r of row j, group
// 4q + g, and runs f_l += fl(S_l * cs) group by group; cs = fl(ws * as) and
// fl(wz * xsum) come from v_mfma_f32_16x16x1_4b_f32 (one product and +0: one
// rounding).  The operands enter as in gemm_mm.hip: codes as f16 subnormals
// with the scales times 2^24, or, in a step whose scales include a finite
// 2^88 or more, as 1024 + n minus 1024.
//
// Everything streams through registers, NQ steps ahead: the activations
// ("qa", written by the quantizing kernels in the lane order of this
// kernel) are 1 KB per block and step, which the waves of a CU share through
// its L1, so there is no LDS staging and no barrier before the end.  Lanes of
// tokens past the tile's last read that last token's data, and lanes of groups
// past the row's last read that group's with zero parameters and scales, so
// nothing outside the inputs enters.
//
// CW: the eight (four at group 32) lane chains of a row are independent until
// the final sum, so CW waves may share a row tile, NL / CW chains each, where
// too few row tiles would leave SIMDs idle; they read disjoint parts of the
// codes and activations.  The VALU epilogue bounds large shapes (9 operations
// per row, token and group of 32, 17 per group of 64 or 128, on 16 token
// slots); latency the small ones.  Measured (whole calls): @@.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "kernels.h"

namespace rai {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <int GS, int CW>
struct StreamCfg {
  static constexpr int NL = GS == 32 ? 4 : 8;      // reference lanes
  static constexpr int LW = NL / CW;               // of them in a wave
  static constexpr int BPL = GS == 128 ? 2 : 1;    // 8-column blocks per reference lane
  static constexpr int NB = GS / 8, NBW = LW * BPL;  // blocks of a group, of a wave
  static constexpr int NQ = NBW >= 16 ? 1 : NBW >= 8 ? 2 : NBW >= 4 ? 4 : 8;  // ring depth in steps
  static constexpr int WR = 4 / CW;                // row tiles per block (four waves)
};

// N dwords of a buffer.
template <int N>
__device__ __forceinline__ void load_dwords(uint32_t *d, const __amdgpu_buffer_rsrc_t r, int voff, int soff) {
  if constexpr (N == 1) {
    d[0] = __builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, 0);
  } else if constexpr (N == 2) {
    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, 0);
    d[0] = v[0];
    d[1] = v[1];
  } else {
#pragma unroll
    for (int i = 0; i < N / 4; ++i) {
      const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, voff + 16 * i, soff, 0);
#pragma unroll
      for (int k = 0; k < 4; ++k) d[4 * i + k] = v[k];
    }
  }
}

// A block dword's codes, columns (0, 4, 1, 5) and (2, 6, 3, 7), the odd ones
// at 16 times their value: f16 subnormals (SUB) or exact integers.
template <bool SUB>
__device__ __forceinline__ h4 codes_half(uint32_t t) {
  if constexpr (SUB) {
    const u32x2 d = {t & 0x000F000Fu, t & 0x00F000F0u};
    return __builtin_bit_cast(h4, d);
  }
  const h2 bias = {(_Float16)1024.0f, (_Float16)1024.0f};
  const h2 e0 = __builtin_bit_cast(h2, (t & 0x000F000Fu) | 0x64006400u) - bias;
  const h2 e1 = __builtin_bit_cast(h2, (t & 0x00F000F0u) | 0x64006400u) - bias;
  return h4{e0[0], e0[1], e1[0], e1[1]};
}

template <int GS, int CW>
__global__ __launch_bounds__(256, 2) void k_gemv_stream(float *out, const float *add, const uint8_t *__restrict__ nib,
                                                        const uint8_t *__restrict__ params,
                                                        const _Float16 *__restrict__ qa,
                                                        const float *__restrict__ scales,
                                                        const float *__restrict__ sums, int rows, int cols, int m) {
  using C = StreamCfg<GS, CW>;
  constexpr int NL = C::NL, LW = C::LW, BPL = C::BPL, NB = C::NB, NBW = C::NBW, NQ = C::NQ, WR = C::WR;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cw = wave % CW, wr = wave / CW;
  const int j = lane & 15, h = lane >> 4;
  const int groups = cols / GS, nq = (groups + 3) / 4;
  const int t0 = 16 * blockIdx.y, mt = min(16, m - t0);
  const int row = (blockIdx.x * WR + wr) * 16 + j, rowc = min(row, rows - 1);
  const int jt = min(j, mt - 1);
  const __amdgpu_buffer_rsrc_t rcs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(nib), 0, rows * (cols / 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rps =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(params), 0, rows * groups * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t rss =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(scales), 0, m * groups * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t rxs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(sums), 0, m * groups * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t ras = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<_Float16 *>(qa), 0, (int)gridDim.y * nq * (NB * 1024), 0x00020000);
  // Lane offsets of a step; in the last step the lanes past the groups take
  // the last group.
  const int hl = min(h, groups - 1 - 4 * (nq - 1));
  const bool past = hl < h;
  auto off = [&](int hh, int &vc, int &vp, int &vs, int &va) {
    vc = rowc * (cols / 2) + hh * (GS / 2) + cw * LW * 4;
    vp = (rowc * groups + hh) * 4;
    vs = ((t0 + jt) * groups + hh) * 4;
    va = (hh * 16 + jt) * 16;
  };
  int vc, vp, vs, va, vcl, vpl, vsl, val;
  off(h, vc, vp, vs, va);
  off(hl, vcl, vpl, vsl, val);
  const int a0 = ((int)blockIdx.y * nq * NB + cw * NBW) * 1024;

  uint32_t rc[NQ][NBW], rp[NQ], ra[NQ][NBW][4];
  float rs[NQ], rx[NQ];
  // Step q's weights and scales, and its activations; a step past the end
  // reads the last one again (unused).
  auto load_w = [&](int s, int q) {
    const bool last = q >= nq - 1;
    const int qc = min(q, nq - 1);
    const int c = last ? vcl : vc, p = last ? vpl : vp, a = last ? vsl : vs;
    load_dwords<LW>(rc[s], rcs, c, qc * (2 * GS));
    if constexpr (BPL == 2) load_dwords<LW>(rc[s] + LW, rcs, c + 32, qc * (2 * GS));
    rp[s] = __builtin_amdgcn_raw_buffer_load_b32(rps, p, qc * 16, 0);
    rs[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rss, a, qc * 16, 0));
    if (cw == 0) rx[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rxs, a, qc * 16, 0));
  };
  auto load_a = [&](int s, int b, int q) {
    const int qc = min(q, nq - 1);
    load_dwords<4>(ra[s][b], ras, q >= nq - 1 ? val : va, a0 + qc * (NB * 1024) + b * 1024);
  };
#pragma unroll
  for (int s = 0; s < NQ; ++s) {
    rx[s] = 0.0f;
    load_w(s, s);
#pragma unroll
    for (int b = 0; b < NBW; ++b) load_a(s, b, s);
  }

  float f[LW][4], zc[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
#pragma unroll
    for (int l = 0; l < LW; ++l) f[l][r] = 0.0f;
    zc[r] = 0.0f;
  }
  const f16v zero = {};
  // The lane sums of reference lane l of the wave from ring slot s.
  auto lane_sums = [&](int s, int l, auto sub) __attribute__((always_inline)) {
    constexpr bool SUB = decltype(sub)::value;
    f16v D = zero;
#pragma unroll
    for (int k = 0; k < BPL; ++k) {
      const uint32_t w = rc[s][k * LW + l];
      const uint32_t(&a)[4] = ra[s][l * BPL + k];
      const u32x2 alo = {a[0], a[1]}, ahi = {a[2], a[3]};
      D = __builtin_amdgcn_mfma_f32_16x16x4f16(__builtin_bit_cast(h4, alo), codes_half<SUB>(w), D, 0, 0, 0);
      D = __builtin_amdgcn_mfma_f32_16x16x4f16(__builtin_bit_cast(h4, ahi), codes_half<SUB>(w >> 8), D, 0, 0, 0);
    }
    return D;
  };
  auto step = [&](int s, int q, auto sub) __attribute__((always_inline)) {
    constexpr bool SUB = decltype(sub)::value;
    const bool none = q == nq - 1 && past;
    const float as = none ? 0.0f : SUB ? rs[s] * 16777216.0f : rs[s];
    const uint32_t pw = none ? 0u : rp[s];
    const float ws = (float)__builtin_bit_cast(_Float16, (uint16_t)(pw & 0xFFFF));
    const f16v cs = __builtin_amdgcn_mfma_f32_16x16x1f32(as, ws, zero, 0, 0, 0);
    f16v D[2];
    D[0] = lane_sums(s, 0, sub);
    if constexpr (LW > 1) D[1] = lane_sums(s, 1, sub);
    if (cw == 0) {
      const float wz = (float)__builtin_bit_cast(_Float16, (uint16_t)(pw >> 16));
      const f16v z = __builtin_amdgcn_mfma_f32_16x16x1f32(none ? 0.0f : rx[s], wz, zero, 0, 0, 0);
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int r = 0; r < 4; ++r) zc[r] = zc[r] + z[4 * g + r];
    }
#pragma unroll
    for (int l = 0; l < LW; ++l) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int r = 0; r < 4; ++r) f[l][r] = f[l][r] + D[l & 1][4 * g + r] * cs[4 * g + r];
      if (l + 2 < LW) D[l & 1] = lane_sums(s, l + 2, sub);
    }
  };
  for (int q0 = 0; q0 < nq; q0 += NQ) {
#pragma unroll
    for (int s = 0; s < NQ; ++s) {
      const int q = q0 + s;
      if (q < nq) {
        const float av = fabsf(rs[s]);
        if (__builtin_amdgcn_ballot_w64(av >= 0x1p88f && av < INFINITY) != 0)
          step(s, q, std::false_type{});
        else
          step(s, q, std::true_type{});
      }
      load_w(s, q + NQ);
#pragma unroll
      for (int b = 0; b < NBW; ++b) load_a(s, b, q + NQ);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // hsum8 of the row tile's chains (lanes 4..7 are +0 at group 32), which the
  // CW waves hold.
  float all[NL][4];
  if constexpr (CW == 1) {
#pragma unroll
    for (int l = 0; l < NL; ++l)
#pragma unroll
      for (int r = 0; r < 4; ++r) all[l][r] = f[l][r];
  } else {
    __shared__ float fin[WR][NL][4][64];
#pragma unroll
    for (int l = 0; l < LW; ++l)
#pragma unroll
      for (int r = 0; r < 4; ++r) fin[wr][cw * LW + l][r][lane] = f[l][r];
    __syncthreads();
    if (cw != 0) return;
#pragma unroll
    for (int l = 0; l < NL; ++l)
#pragma unroll
      for (int r = 0; r < 4; ++r) all[l][r] = fin[wr][l][r][lane];
  }
  if (row < rows) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 4 * h + r;
      if (t < mt) {
        const size_t oi = (size_t)(t0 + t) * rows + row;
        float v;
        if constexpr (NL == 4)
          v = ((all[0][r] + all[1][r]) + (all[2][r] + all[3][r])) + zc[r];
        else
          v = (((all[0][r] + all[4][r]) + (all[1][r] + all[5][r])) +
               ((all[2][r] + all[6][r]) + (all[3][r] + all[7][r]))) + zc[r];
        out[oi] = add ? add[oi] + v : v;
      }
    }
  }
}

template <int GS>
void launch_stream_t(float *out, const float *add, const uint8_t *nib, const uint8_t *params, const _Float16 *qa,
                     const float *scales, const float *sums, int rows, int cols, int m, hipStream_t s) {
  const int rt = (rows + 15) / 16, tt = (m + 15) / 16;
  auto go = [&](auto cw) {
    constexpr int CW = decltype(cw)::value;
    const dim3 grid((rt + 4 / CW - 1) / (4 / CW), tt);
    hipLaunchKernelGGL((k_gemv_stream<GS, CW>), grid, dim3(256), 0, s, out, add, nib, params, qa, scales, sums, rows,
                       cols, m);
  };
  // The chains of a row tile split until the chip's 1024 SIMDs have two waves.
  if (rt * tt >= 2048)
    go(std::integral_constant<int, 1>{});
  else if (rt * tt >= 1024)
    go(std::integral_constant<int, 2>{});
  else
    go(std::integral_constant<int, 4>{});
}

}  // namespace

bool gemv_stream_path(int rows, int cols, int m, int gs) {
  return (gs == 32 || gs == 64 || gs == 128) && m >= 2 && m <= kMfmaMaxTokens && rows > 0 && cols % gs == 0 &&
         (int64_t)rows * (cols / 2) < ((int64_t)1 << 31) && qa_bytes(m, cols, gs) < ((size_t)1 << 31);
}

size_t qa_bytes(int m, int cols, int gs) {
  return (size_t)((m + 15) / 16) * ((cols / gs + 3) / 4) * (gs / 8) * 1024;
}

void launch_gemv_stream(float *out, const float *add, const uint8_t *nib, const uint8_t *params, const _Float16 *qa,
                        const float *scales, const float *sums, int rows, int cols, int m, int gs, hipStream_t s) {
  if (gs == 32)
    launch_stream_t<32>(out, add, nib, params, qa, scales, sums, rows, cols, m, s);
  else if (gs == 64)
    launch_stream_t<64>(out, add, nib, params, qa, scales, sums, rows, cols, m, s);
  else
    launch_stream_t<128>(out, add, nib, params, qa, scales, sums, rows, cols, m, s);
}

}  // namespace rai
