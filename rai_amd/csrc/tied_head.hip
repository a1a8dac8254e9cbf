// Tied 8-bit lm_head (gemm.rs:804-1047, 1981-2076) for whole groups of 32, 64
// or 128: logits[t][v] = hsum8(f) + zc over the vocabulary rows of the
// embedding table, codes 0..255 against the hidden row quantized to +-63.
//
// Reference order.  Lane l (0..7) of a group sums code x activation over
// columns 4l..4l+3 of each of the group's 32-column chunks (exact in int32);
// f_l += fl(float(s_l) * fl(ws * hs)) group by group; zc += fl(wz * hsum) is a
// chain of its own.
//
// The table is read once per kTiedTokens tokens and bounds the kernel at one
// token (65.5 MB for 32000 x 2048), so a load instruction of a wave covers
// 2048 consecutive bytes of a row: lane u holds 32-column unit u of the
// chunk (two 16-byte loads) for each of the wave's R rows, the next chunk's
// loads in flight while this one computes.  v_dot4_i32_i8 is signed, so codes
// enter as code - 128 and 128 * sum(activations) is added back (exact).  The
// GS / 32 lanes of a group add their units by DPP and share its eight
// products; these go through a wave-private LDS area and come back
// transposed: lane c = r * 9 + l runs chain l of row r over the chunk's
// groups in order.  Four rows a wave: 9 R chains fit the 64 lanes, and 32000
// rows give 8000 waves, eight a SIMD.
//
// One thread per row with byte loads, as the general kernel in kernels.hip
// (other group sizes, partial groups, misaligned tables) does it, took 41.7 us
// at 32000 x 2048 and 17.9 us for the quantization (the whole call 73.7 us,
// now 29.5).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels.h"
#include "quant_dev.h"

namespace rai {

namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kTiedRows = 4;    // rows per wave
constexpr int kTiedWaves = 4;   // waves per block
constexpr int kTiedTokens = 4;  // tokens per pass over the table

// quantize_hidden_i8 (gemm.rs:924-1047): +-63 per group, and the input sums;
// eight lanes per group as k_quant.  Grid (ceil(groups / 32), m).
template <int GS>
__global__ __launch_bounds__(256) void k_quant63(const float *__restrict__ x, int n, int8_t *__restrict__ q,
                                                 float *__restrict__ scales, float *__restrict__ sums) {
  constexpr int NB = GS / 8;
  const int t = blockIdx.y, groups = n / GS;
  const int g = blockIdx.x * 32 + threadIdx.x / 8, j = threadIdx.x & 7;
  const bool ok = g < groups;
  const float *xr = x + (size_t)t * n + (size_t)(ok ? g : 0) * GS;
  float v[NB], a = 0.0f, amax = 0.0f;
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    v[c] = ok ? xr[8 * c + j] : 0.0f;
    a = a + v[c];
    amax = fmaxf(amax, fabsf(v[c]));
  }
  const float b = a + dpp_mov<kDppShl4>(a);
  const float c2 = b + dpp_mov<kDppShl1>(b);
  const float total = c2 + dpp_mov<kDppShl2>(c2);
  amax = fmaxf(amax, dpp_mov<kDppHalfMirror>(amax));
  amax = fmaxf(amax, dpp_mov<kDppXor1>(amax));
  amax = fmaxf(amax, dpp_mov<kDppXor2>(amax));
  const float scale = amax > 1e-10f ? amax / 63.0f : 1.0f;
  const float inv = 1.0f / scale;
  if (!ok) return;
  int8_t *qo = q + (size_t)t * n + (size_t)g * GS;
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    float r = rintf(v[c] * inv);
    r = fminf(fmaxf(r, -63.0f), 63.0f);
    qo[8 * c + j] = (int8_t)(int)r;
  }
  if (j == 0) {
    scales[(size_t)t * groups + g] = scale;
    sums[(size_t)t * groups + g] = total;
  }
}

template <int CTRL>
__device__ __forceinline__ int add_dpp(int v) {
  return v + __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, true);
}

template <int GS, int MT>
__global__ __launch_bounds__(64 * kTiedWaves) void k_tied_head_w(float *__restrict__ logits,
                                                                 const uint8_t *__restrict__ codes,
                                                                 const uint8_t *__restrict__ params,
                                                                 const int8_t *__restrict__ hq,
                                                                 const float *__restrict__ hscales,
                                                                 const float *__restrict__ hsums, int vocab, int n,
                                                                 int m) {
  constexpr int R = kTiedRows, LPG = GS / 32;  // lanes per group
  constexpr int GPC = 64 / LPG;                // groups per chunk
  constexpr int STR = GPC + 8;                 // product row stride (16-byte rows, spread over the banks)
  constexpr int NP = 8 / LPG;                  // products per lane and row
  static_assert(9 * R <= 64, "one chain per lane");
  __shared__ __align__(16) float lds[kTiedWaves][9 * R * STR];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row0 = (blockIdx.x * kTiedWaves + wave) * R;
  const int t0 = blockIdx.y * MT;
  const int groups = n / GS, units = n / 32, nch = (units + 63) / 64;
  float *pl = lds[wave];
  const int k = lane % LPG, gl = lane / LPG;
  const bool chain = lane < 9 * R;
  const float4 *pc = reinterpret_cast<const float4 *>(pl + (chain ? lane : 0) * STR);

  u32x4 cw[R][2];
  uint32_t pw[R];
  auto load = [&](int ch) {
    const int u = min(ch * 64 + lane, units - 1), g = min(ch * GPC + gl, groups - 1);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const size_t row = min(row0 + r, vocab - 1);
      const u32x4 *src = reinterpret_cast<const u32x4 *>(codes + row * n + (size_t)u * 32);
      cw[r][0] = src[0];
      cw[r][1] = src[1];
      pw[r] = reinterpret_cast<const uint32_t *>(params)[row * groups + g];
    }
  };
  load(0);
  float acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = 0.0f;
  for (int ch = 0; ch < nch; ++ch) {
    const int u = ch * 64 + lane, g = ch * GPC + gl;
    const bool in = u < units;
    u32x4 cc[R][2];
    uint32_t pp[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
      // Lanes past the row: zero parameters and scales, so that their
      // products are +-0, which no chain sees.
      cc[r][0] = cw[r][0] ^ 0x80808080u;
      cc[r][1] = cw[r][1] ^ 0x80808080u;
      pp[r] = in ? pw[r] : 0u;
    }
    if (ch + 1 < nch) load(ch + 1);
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int tok = min(t0 + t, m - 1);
      const u32x4 *hsrc = reinterpret_cast<const u32x4 *>(hq + (size_t)tok * n + (size_t)min(u, units - 1) * 32);
      const u32x4 h0 = hsrc[0], h1 = hsrc[1];
      const float hs = in ? hscales[(size_t)tok * groups + g] : 0.0f;
      const float hx = in ? hsums[(size_t)tok * groups + g] : 0.0f;
      int bias[8];
#pragma unroll
      for (int l = 0; l < 8; ++l)
        bias[l] = __builtin_amdgcn_sdot4((int)(l < 4 ? h0[l] : h1[l - 4]), 0x01010101, 0, false) * 128;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        int s[8];
#pragma unroll
        for (int l = 0; l < 8; ++l) {
          s[l] = __builtin_amdgcn_sdot4((int)(l < 4 ? cc[r][0][l] : cc[r][1][l - 4]),
                                        (int)(l < 4 ? h0[l] : h1[l - 4]), bias[l], false);
          if constexpr (LPG >= 2) s[l] = add_dpp<kDppXor1>(s[l]);
          if constexpr (LPG >= 4) s[l] = add_dpp<kDppXor2>(s[l]);
        }
        const float ws = (float)__builtin_bit_cast(_Float16, (uint16_t)(pp[r] & 0xFFFF));
        const float wz = (float)__builtin_bit_cast(_Float16, (uint16_t)(pp[r] >> 16));
        const float cs = ws * hs;
        float *pr = pl + r * 9 * STR + gl;
        // Lane k of the group keeps products k * NP .. + NP - 1.
#pragma unroll
        for (int i = 0; i < NP; ++i) {
          int si = s[i];
#pragma unroll
          for (int kk = 1; kk < LPG; ++kk) si = k == kk ? s[kk * NP + i] : si;
          pr[(k * NP + i) * STR] = (float)si * cs;
        }
        if (k == 0) pr[8 * STR] = wz * hx;
      }
      // The wave's LDS operations complete in order; the fences only keep the
      // compiler from moving the reads above the writes.
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int q = 0; q < GPC / 4; ++q) {
        const float4 p = pc[q];
        acc[t] = acc[t] + p.x;
        acc[t] = acc[t] + p.y;
        acc[t] = acc[t] + p.z;
        acc[t] = acc[t] + p.w;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    float *fin = pl + t * 64;
    if (chain) fin[lane] = acc[t];
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (lane < R * MT) {
    const int t = lane / R, r = lane % R;
    const float *f = pl + t * 64 + r * 9;
    const float v = (((f[0] + f[4]) + (f[1] + f[5])) + ((f[2] + f[6]) + (f[3] + f[7]))) + f[8];
    if (row0 + r < vocab && t0 + t < m) logits[(size_t)(t0 + t) * vocab + row0 + r] = v;
  }
}

template <int GS>
void launch_tied_t(float *logits, const float *hidden, const uint8_t *codes, const uint8_t *params, int vocab, int n,
                   int m, int8_t *hq, float *hscales, float *hsums, hipStream_t s) {
  hipLaunchKernelGGL(k_quant63<GS>, dim3((n / GS + 31) / 32, m), dim3(256), 0, s, hidden, n, hq, hscales, hsums);
  const int rb = kTiedRows * kTiedWaves, blocks = (vocab + rb - 1) / rb;
  if (m == 1)
    hipLaunchKernelGGL((k_tied_head_w<GS, 1>), dim3(blocks), dim3(64 * kTiedWaves), 0, s, logits, codes, params, hq,
                       hscales, hsums, vocab, n, m);
  else
    hipLaunchKernelGGL((k_tied_head_w<GS, kTiedTokens>), dim3(blocks, (m + kTiedTokens - 1) / kTiedTokens),
                       dim3(64 * kTiedWaves), 0, s, logits, codes, params, hq, hscales, hsums, vocab, n, m);
}

}  // namespace

// Dword loads of the table and 16-byte ones of the quantized row (hq is 256
// bytes aligned by its owners).
bool tied_head_wave_path(int n, int gs, const void *codes, const void *params) {
  return (gs == 32 || gs == 64 || gs == 128) && n > 0 && n % gs == 0 &&
         ((uintptr_t)codes | (uintptr_t)params) % 4 == 0;
}

void launch_tied_head_wave(float *logits, const float *hidden, const uint8_t *codes, const uint8_t *params, int vocab,
                           int n, int gs, int m, int8_t *hq, float *hscales, float *hsums, hipStream_t s) {
  if (gs == 32)
    launch_tied_t<32>(logits, hidden, codes, params, vocab, n, m, hq, hscales, hsums, s);
  else if (gs == 64)
    launch_tied_t<64>(logits, hidden, codes, params, vocab, n, m, hq, hscales, hsums, s);
  else
    launch_tied_t<128>(logits, hidden, codes, params, vocab, n, m, hq, hscales, hsums, s);
}

}  // namespace rai
