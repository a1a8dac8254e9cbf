// Prefill attention's scores and PV on the matrix cores, bit for bit the
// reference's f32 order (attention_head_avx2, layers.rs:1266-1380).
//
// Both are FMA chains: lane c (0..7) of a score accumulates q[8i + c] k[8i + c]
// over i, and out[d] accumulates p_s v_s[d] over the positions.  One step of
// such a chain for 16 tokens x 16 columns is an outer product, and
// v_mfma_f32_16x16x1_4b_f32 adds four of them (one product each, one rounding)
// to four independent 16 x 16 accumulators: four of a score's lanes, or four
// 16-dimension slices of a head.  1024 FMAs take 32 matrix cycles, half of what
// the VALU needs for them, and the VALU stays free.
//
// Against the DPP-FMA score kernel and the streamed PV kernel (one lane per
// chain, fused.hip), 256 tokens, 32 heads of 128 on 8 kv heads, 3072 to 4096
// positions: scores 204 -> 108 us, PV 214 -> 143 (counters: a SIMD finishes a
// matrix instruction every 64 cycles in the scores, whose two or three waves each
// run a chain, and every 93 in PV's one chain, not the 32 of its passes).  PV's chain is as long for one tile of
// tokens as for sixteen, so it takes over only past kPvMmTokens of them.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "kernels.h"

namespace rai {

namespace {

typedef float f16v __attribute__((ext_vector_type(16)));

constexpr int kTT = 16;    // tokens per tile
constexpr int kSP = 64;    // positions per score block: four waves of 16
constexpr int kPP = 64;    // positions per PV stage
constexpr int kPS = kPP + 4;

// Block (64-position tile, kv head, share of the units): wave w holds the keys
// of positions 16 w.. in registers (lane (s, j): chains j and j + 4 of position
// s) and every unit's query rows - 16 tokens of one query head - pass through
// LDS, where a row lies chain by chain (row stride 4 mod 64 floats: the 16
// tokens' reads fall on different banks).  Unit u = token tile * G + head.
template <int HD>
__global__ __launch_bounds__(256) void k_scores_mm(const float *__restrict__ q, int q_ld,
                                                   const float *__restrict__ kc, int cap, int pos0, int m, int nh,
                                                   int nkv, float scale, float *__restrict__ S, int sstride) {
  constexpr int NI = HD / 8, QS = HD + 4, QV = kTT * HD / 4 / 256;  // query float4 per thread and unit
  __shared__ __align__(16) float ks[kSP * QS];
  __shared__ __align__(16) float qs[2][kTT * QS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kv = blockIdx.y, G = nh / nkv, s0 = blockIdx.x * kSP, npos = pos0 + m;
  const int units = (m + kTT - 1) / kTT * G;
  const int share = (units + gridDim.z - 1) / gridDim.z;
  int u = blockIdx.z * share;
  const int uend = min(units, u + share);
  // Token tiles whose last token ends before this tile of positions see none
  // of it.
  if (s0 > pos0) u = max(u, (s0 - pos0) / kTT * G);
  if (u >= uend) return;
  // Element 4 e4 .. + 3 of a row: chains 4 (e4 % 2).., step e4 / 2.
  auto put = [&](float *row, int e4, float4 v) {
    float *d = row + 4 * (e4 & 1) * NI + (e4 >> 1);
    d[0] = v.x;
    d[NI] = v.y;
    d[2 * NI] = v.z;
    d[3 * NI] = v.w;
  };
  float4 qv[QV];
  auto load_q = [&](int uu) {
    const int t0 = uu / G * kTT, hq = kv * G + uu % G;
#pragma unroll
    for (int i = 0; i < QV; ++i) {
      const int e = tid + 256 * i, t = e / (HD / 4), e4 = e % (HD / 4);
      qv[i] = *reinterpret_cast<const float4 *>(q + (size_t)min(t0 + t, m - 1) * q_ld + hq * HD + 4 * e4);
    }
  };
  auto put_q = [&](float *b) {
#pragma unroll
    for (int i = 0; i < QV; ++i) {
      const int e = tid + 256 * i;
      put(b + e / (HD / 4) * QS, e % (HD / 4), qv[i]);
    }
  };
  load_q(u);
  for (int e = tid; e < kSP * HD / 4; e += 256) {
    const int s = e / (HD / 4), e4 = e % (HD / 4);
    const float4 v =
        *reinterpret_cast<const float4 *>(kc + ((size_t)kv * cap + min(s0 + s, npos - 1)) * HD + 4 * e4);
    put(ks + s * QS, e4, v);
  }
  put_q(qs[0]);
  __syncthreads();
  const int col = lane & 15, j = lane >> 4;
  float kr[2][NI];
  auto chains = [&](const float *row, float (&r)[2][NI]) {
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int i = 0; i < NI / 4; ++i) {
        const float4 v = reinterpret_cast<const float4 *>(row + (j + 4 * c) * NI)[i];
        r[c][4 * i] = v.x;
        r[c][4 * i + 1] = v.y;
        r[c][4 * i + 2] = v.z;
        r[c][4 * i + 3] = v.w;
      }
  };
  chains(ks + (16 * wave + col) * QS, kr);
  const int s = s0 + 16 * wave + col;
  for (int b = 0; u < uend; ++u, b ^= 1) {
    if (u + 1 < uend) load_q(u + 1);
    const int t0 = u / G * kTT, hq = kv * G + u % G;
    float qr[2][NI];
    chains(qs[b] + col * QS, qr);
    f16v D0 = {}, D1 = {};
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      D0 = __builtin_amdgcn_mfma_f32_16x16x1f32(qr[0][i], kr[0][i], D0, 0, 0, 0);
      D1 = __builtin_amdgcn_mfma_f32_16x16x1f32(qr[1][i], kr[1][i], D1, 0, 0, 0);
    }
    if (u + 1 < uend) put_q(qs[b ^ 1]);
    // Lane (s, j) holds tokens 4 j + r, chains c of D0 and c + 4 of D1 in
    // register 4 c + r.
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = t0 + 4 * j + r;
      const float d = ((D0[r] + D1[r]) + (D0[4 + r] + D1[4 + r])) +
                      ((D0[8 + r] + D1[8 + r]) + (D0[12 + r] + D1[12 + r]));
      if (t < m && s < npos) S[((size_t)t * nh + hq) * sstride + s] = d * scale;
    }
    __syncthreads();
  }
}

// Block (four units of a kv head, kv head, 64-dimension slice): wave w runs
// unit 4 x + w (16 tokens of one query head, as above) over all its positions, a
// stage of 64 at a time: the slice's V rows (d-major, read by all four waves)
// and the units' probabilities e * (1 / sum) pass through LDS.  Positions that
// some token of the tile does not see (at most 15, and up to three before them)
// run on the VALU, token by token, so that no product with a masked position
// enters a chain.
template <int HD>
__global__ __launch_bounds__(256) void k_pv_mm(const float *__restrict__ S, const float *__restrict__ vc, int vstride,
                                               int pos0, int m, int nh, int nkv, int sstride,
                                               float *__restrict__ out) {
  __shared__ __align__(16) float vs[64 * kPS];
  __shared__ __align__(16) float ps[4][kTT * kPS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kv = blockIdx.y, G = nh / nkv, d0 = blockIdx.z * 64;
  const int units = (m + kTT - 1) / kTT * G;
  const int row = tid >> 4, c4 = 4 * (tid & 15);  // this thread's V / P row and columns
  auto unit_of = [&](int w) { return min(4 * (int)blockIdx.x + w, units - 1); };
  const float *pr[4];
  float inv[4];
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    const int u = unit_of(w), t = min(u / G * kTT + row, m - 1);
    pr[w] = S + ((size_t)t * nh + kv * G + u % G) * sstride;
    inv[w] = pr[w][sstride - 1];
  }
  const float *vr = vc + ((size_t)kv * HD + d0 + row) * vstride;
  const int u = unit_of(wave), t0 = u / G * kTT;
  const int nfull = pos0 + t0 + 1, nlast = pos0 + min(t0 + kTT, m);  // seen by every token, by the last
  const int nblk = pos0 + min(unit_of(3) / G * kTT + kTT, m);        // by the block
  float4 vv[4], pv[4];
  auto load = [&](int s0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      vv[i] = *reinterpret_cast<const float4 *>(vr + (size_t)16 * i * vstride + s0 + c4);
      pv[i] = *reinterpret_cast<const float4 *>(pr[i] + min(s0 + c4, sstride - 4));
    }
  };
  f16v acc = {};
  const int col = lane & 15, j = lane >> 4;
  load(0);
  for (int s0 = 0; s0 < nblk; s0 += kPP) {
    __syncthreads();  // the stage before is read
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *reinterpret_cast<float4 *>(vs + (row + 16 * i) * kPS + c4) = vv[i];
      float4 p = pv[i];
      p.x = p.x * inv[i];
      p.y = p.y * inv[i];
      p.z = p.z * inv[i];
      p.w = p.w * inv[i];
      *reinterpret_cast<float4 *>(ps[i] + row * kPS + c4) = p;
    }
    __syncthreads();
    if (s0 + kPP < nblk) load(s0 + kPP);
    const float *pa = ps[wave] + col * kPS, *vb = vs + lane * kPS;
    const int full = max(0, min(kPP, nfull - s0)) & ~3, end = min(kPP, nlast - s0);
    auto four = [&](const float4 a, const float4 b) __attribute__((always_inline)) {
      acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a.x, b.x, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a.y, b.y, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a.z, b.z, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x1f32(a.w, b.w, acc, 0, 0, 0);
    };
    auto at = [](const float *p, int k) { return *reinterpret_cast<const float4 *>(p + k); };
    if (full == kPP) {
      // Sixteen positions' operands requested before the sixteen ahead of
      // them multiply.
      float4 a[2][4], b[2][4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        a[0][i] = at(pa, 4 * i);
        b[0][i] = at(vb, 4 * i);
      }
#pragma unroll
      for (int g = 0; g < kPP / 16; ++g) {
        if (g + 1 < kPP / 16) {
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            a[(g + 1) & 1][i] = at(pa, 16 * (g + 1) + 4 * i);
            b[(g + 1) & 1][i] = at(vb, 16 * (g + 1) + 4 * i);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) four(a[g & 1][i], b[g & 1][i]);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      for (int k = 0; k < full; k += 4) four(at(pa, k), at(vb, k));
      // Register 4 c + r: token 4 j + r, dimension 16 c + col.
      for (int k = full; k < end; ++k) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = ps[wave][(4 * j + r) * kPS + k];
          const bool sees = s0 + k <= pos0 + t0 + 4 * j + r;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const float f = __fmaf_rn(p, vs[(16 * c + col) * kPS + k], acc[4 * c + r]);
            acc[4 * c + r] = sees ? f : acc[4 * c + r];
          }
        }
      }
    }
  }
  if (4 * (int)blockIdx.x + wave < units) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = t0 + 4 * j + r;
      if (t < m) {
#pragma unroll
        for (int c = 0; c < 4; ++c) out[((size_t)t * nh + kv * G + u % G) * HD + d0 + 16 * c + col] = acc[4 * c + r];
      }
    }
  }
}

template <int HD>
void scores_t(const float *q, int q_ld, const float *kc, int cap, int pos0, int m, int nh, int nkv, float scale,
              float *S, int sstride, hipStream_t s) {
  const int tiles = (pos0 + m + kSP - 1) / kSP, units = (m + kTT - 1) / kTT * (nh / nkv);
  // The units in shares of at least four, up to about eight blocks a CU (three
  // run at a time), so that no CU is left with a block more than the others.
  const int z = std::max(1, std::min(units / 4, 2048 / std::max(1, tiles * nkv)));
  hipLaunchKernelGGL(k_scores_mm<HD>, dim3(tiles, nkv, z), dim3(256), 0, s, q, q_ld, kc, cap, pos0, m, nh, nkv, scale,
                     S, sstride);
}

}  // namespace

// Head sizes of 64 and 128 with the d-major V cache; 16-byte loads of the query
// rows and both caches.
bool attn_mm_path(const float *q, int q_ld, const float *kc, const float *vc, int vstride, int m, int nh, int nkv,
                  int hd) {
  return m >= kAttnMmTokens && (hd == 64 || hd == 128) && nh % nkv == 0 && vstride > 0 && vstride % 64 == 0 &&
         q_ld % 4 == 0 && (((uintptr_t)q | (uintptr_t)kc | (uintptr_t)vc) & 15) == 0;
}

void launch_scores_mm(const float *q, int q_ld, const float *kc, int cap, int pos0, int m, int nh, int nkv, int hd,
                      float scale, float *S, int sstride, hipStream_t s) {
  if (hd == 64)
    scores_t<64>(q, q_ld, kc, cap, pos0, m, nh, nkv, scale, S, sstride, s);
  else
    scores_t<128>(q, q_ld, kc, cap, pos0, m, nh, nkv, scale, S, sstride, s);
}

void launch_pv_mm(const float *S, const float *vc, int vstride, int pos0, int m, int nh, int nkv, int hd, int sstride,
                  float *out, hipStream_t s) {
  const int units = (m + kTT - 1) / kTT * (nh / nkv);
  const dim3 grid((units + 3) / 4, nkv, hd / 64);
  if (hd == 64)
    hipLaunchKernelGGL(k_pv_mm<64>, grid, dim3(256), 0, s, S, vc, vstride, pos0, m, nh, nkv, sstride, out);
  else
    hipLaunchKernelGGL(k_pv_mm<128>, grid, dim3(256), 0, s, S, vc, vstride, pos0, m, nh, nkv, sstride, out);
}

}  // namespace rai
