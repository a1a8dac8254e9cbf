// W4A8 product for small batches (w4a8_route) on the gfx950 matrix cores, groups of 32, 64
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
// with the scales times 2^24, or, where a scale of the tile is finite and 2^88
// or more, as 1024 + n minus 1024 (a second run over K).
//
// Loads.  The L1 serves one 64-byte piece per cycle however many lanes ask
// for it, so no load goes out in the operand order, where neighbouring lanes lie
// in different rows (14336x4096 at group 64, 9 tokens, took 39.5 us that way, 21.4
// this way; at group 128 a wave makes 111 accesses a step): the activations, their scales
// and their sums ("qa", written by the quantizing kernels) lie in lane order
// and are read a few steps ahead; the codes are read as whole row pieces, four
// steps (a stage) at a time, and the parameters likewise, a stage or two ahead,
// and reach their lanes through LDS (16-byte units, the unit index XORed with
// the row so that the 16 rows' reads fall on different banks).  One barrier a
// stage.  Lanes of tokens past the tile's last read that last token's data,
// and lanes of groups past the row's last read that group's codes with zero
// parameters and scales, so nothing outside the inputs enters; no load leaves
// the arrays (stream_addr.h).
//
// CW: the eight (four at group 32) lane chains of a row are independent until
// the final sum, so CW waves may share a row tile, NL / CW chains each, where
// too few row tiles would leave SIMDs idle (a lone wave issues a VALU
// operation every eight cycles, two waves nearly twice as many); they share
// the loads of a stage's codes.  The VALU epilogue bounds large shapes (9
// operations per row, token and group of 32, 17 per group of 64 or 128, on 16
// token slots), the latency of the weights in flight the small ones.  Device
// time at 9 tokens, weights from HBM, against the VALU kernel that group 128
// took before: 4096x14336 65 -> 19.1 us (whole call 100.8 -> 21.5).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "kernels.h"
#include "quant_dev.h"
#include "stream_addr.h"

namespace rai {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <int GS, int CW>
struct StreamCfg {
  static constexpr int NL = GS == 32 ? 4 : 8;      // reference lanes
  static constexpr int LW = NL / CW;               // of them in a wave
  static constexpr int BPL = GS == 128 ? 2 : 1;    // 8-column blocks per reference lane
  static constexpr int NB = GS / 8, NBW = LW * BPL;  // blocks of a group, of a wave
  // Activation ring in steps and code ring in stages.  Loads return in order, so
  // neither helps past the other's depth.
  static constexpr int NQ = NBW <= 2 ? 8 : NBW <= 4 ? 4 : 2;
  static constexpr int WR = 4 / CW;                // row tiles per block (four waves)
  static constexpr int REC = qa_rec_bytes(GS);     // bytes of a step's activations
  static constexpr int U = GS / 8;                 // 16-byte code units of a row and step
  static constexpr int NC = U / 4;                 // code loads per lane and step
  // A stage is four steps; each of a row tile's CW waves loads 4 / CW of them.
  static constexpr int SPW = 4 / CW, CL = SPW * NC;  // steps, code loads per lane and stage
  static constexpr int D = NQ == 2 ? 1 : 2;
  static_assert(4 * D % NQ == 0, "static ring slots");
  static constexpr int TILE_UNITS = 64 * U;          // LDS units of a row tile's stage
};

template <int GS, int CW>
__global__ __launch_bounds__(256, 2) void k_gemv_stream(float *out, const float *add, const uint8_t *__restrict__ nib,
                                                        const uint8_t *__restrict__ params,
                                                        const _Float16 *__restrict__ qa, int rows, int cols, int m) {
  using C = StreamCfg<GS, CW>;
  constexpr int NL = C::NL, LW = C::LW, BPL = C::BPL, NBW = C::NBW, NQ = C::NQ, WR = C::WR;
  constexpr int REC = C::REC, U = C::U, NC = C::NC;
  constexpr int SPW = C::SPW, CL = C::CL, DS = C::D;
  __shared__ __align__(16) u32x4 units[2][WR][C::TILE_UNITS];
  __shared__ __align__(16) u32x4 punits[2][4][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int cw = wave % CW, wr = wave / CW;
  const int j = lane & 15, h = lane >> 4;
  const int groups = cols / GS, nq = (groups + 3) / 4;
  const int t0 = 16 * blockIdx.y, mt = min(16, m - t0);
  const int row0 = (blockIdx.x * WR + wr) * 16, row = row0 + j;
  const __amdgpu_buffer_rsrc_t rcs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(nib), 0, rows * (cols / 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rps =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(params), 0, rows * groups * 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t ras =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<_Float16 *>(qa), 0, (int)gridDim.y * nq * REC, 0x00020000);

  // Code unit u (16 bytes) of a step's 4 groups of row r lies at LDS unit
  // r * U + (u ^ swz(r)) of the step's 16 U; lane i of load c moves unit
  // 64 c + i.
  auto swz = [](int r) { return (r / (16 / U)) & (U - 1); };
  const int nst = (nq + 3) / 4;
  int vc[NC], vcl[NC];  // and in the last step: units of groups past the row's take its last group
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int r = (64 * c + lane) / U, u = ((64 * c + lane) % U) ^ swz(r);
    const int rr = min(row0 + r, rows - 1);
    vc[c] = stream_code_off(rr, cols, GS, 0, u / NC, u % NC).v;
    vcl[c] = stream_code_off(rr, cols, GS, nq - 1, u / NC, u % NC).v;
  }
  // Parameters of stage S: lane i moves 16 bytes (one step) of row
  // i / 4.  Past the row's groups they are the next row's, or past the array
  // (zeros, which the range check of the VGPR offset answers); never used.
  const int pr = lane >> 2, ps = (lane & 3) ^ ((pr >> 2) & 3);
  const int prow = min(row0 + pr, rows - 1);
  const int jt = min(j, mt - 1);
  const int va = (h * 16 + jt) * 16, vs = (h * 16 + jt) * 4;
  // Groups past the row's have no activations: the last step's lanes read
  // those of its last group.
  const int hl = min(h, groups - 1 - 4 * (nq - 1));
  const bool past = hl < h;
  const int val = (hl * 16 + jt) * 16, vsl = (hl * 16 + jt) * 4;
  const int a0 = (int)blockIdx.y * nq * REC;

  u32x4 rc[DS][CL], rp[DS], ra[NQ][NBW];
  float rs[NQ], rx[NQ];
  // The wave's share of stage S's codes (steps 4 S + cw * SPW ..) and its
  // parameters; steps past the end read the last one again (unused).
  auto load_c = [&](int d, int S) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < SPW; ++i) {
      const int q = 4 * S + cw * SPW + i, qc = min(q, nq - 1);
      const bool last = q >= nq - 1;
#pragma unroll
      for (int c = 0; c < NC; ++c)
        rc[d][i * NC + c] = __builtin_amdgcn_raw_buffer_load_b128(rcs, last ? vcl[c] : vc[c], qc * (2 * GS), 0);
    }
    const BufOff po = stream_param_off(prow, groups, S, ps);
    rp[d] = __builtin_amdgcn_raw_buffer_load_b128(rps, po.v, po.s, 0);
  };
  // Step q's scales and activations.
  auto load_a = [&](int s, int q) __attribute__((always_inline)) {
    const bool last = q >= nq - 1;
    const int as = a0 + min(q, nq - 1) * REC;
    const int v = last ? vsl : vs;
    rs[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ras, v, as + C::NB * 1024, 0));
    rx[s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ras, v, as + C::NB * 1024 + 256, 0));
#pragma unroll
    for (int b = 0; b < NBW; ++b)
      ra[s][b] = __builtin_amdgcn_raw_buffer_load_b128(ras, last ? val : va, as + (cw * NBW + b) * 1024, 0);
  };

  float f[LW][4], zc[4];
  const f16v zero = {};
  // The wave's code dwords of lane (j, h): chains cw * LW.., at group 128 the
  // blocks 8 further as well; and its parameter dword.
  uint32_t wc[LW * BPL], par;
  auto codes = [&](const u32x4 *lc, const u32x4 *lp, int i, uint32_t (&w)[LW * BPL],
                   uint32_t &p) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < BPL; ++k) {
      constexpr int N = LW < 4 ? LW : 4;
#pragma unroll
      for (int t = 0; t < LW / N; ++t) {
        const int d = cw * LW + 8 * k + 4 * t;  // dword of the group
        const uint32_t *src =
            reinterpret_cast<const uint32_t *>(lc + i * (16 * U) + j * U + ((h * NC + d / 4) ^ swz(j))) + d % 4;
        if constexpr (N == 4) {
          const u32x4 v = *reinterpret_cast<const u32x4 *>(src);
#pragma unroll
          for (int e = 0; e < 4; ++e) w[k * LW + 4 * t + e] = v[e];
        } else if constexpr (N == 2) {
          const u32x2 v = *reinterpret_cast<const u32x2 *>(src);
          w[k * LW] = v[0];
          w[k * LW + 1] = v[1];
        } else {
          w[k * LW] = *src;
        }
      }
    }
    p = reinterpret_cast<const uint32_t *>(lp + j * 4 + (i ^ ((j >> 2) & 3)))[h];
  };
  // The lane sums of reference lane l of the wave from ring slot s.
  auto lane_sums = [&](int s, int l, auto sub) __attribute__((always_inline)) {
    constexpr bool SUB = decltype(sub)::value;
    f16v D = zero;
#pragma unroll
    for (int k = 0; k < BPL; ++k) {
      const uint32_t w = wc[k * LW + l];
      const u32x4 a = ra[s][l * BPL + k];
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
    const uint32_t pw = none ? 0u : par;
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
  bool big = false;
  auto run = [&](auto sub) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
      for (int l = 0; l < LW; ++l) f[l][r] = 0.0f;
      zc[r] = 0.0f;
    }
    auto put = [&](int d, int S) __attribute__((always_inline)) {
#pragma unroll
      for (int c = 0; c < CL; ++c)
        units[S & 1][wr][(cw * SPW + c / NC) * (16 * U) + 64 * (c % NC) + lane] = rc[d][c];
      punits[S & 1][wave][lane] = rp[d];
    };
    // Ring slot d holds stage S = d mod DS from the time stage S - DS went to
    // LDS.
#pragma unroll
    for (int d = 0; d < DS; ++d) load_c(d, d);
#pragma unroll
    for (int s = 0; s < NQ; ++s) load_a(s, s);
    put(0, 0);
    load_c(0, DS);
    for (int S0 = 0; S0 < nst; S0 += DS) {
#pragma unroll
      for (int d = 0; d < DS; ++d) {
        const int S = S0 + d;
        if (S < nst) {
          // Stage S is in LDS, and stage S - 1's buffer is free.
          __syncthreads();
          put((d + 1) % DS, S + 1);
          load_c((d + 1) % DS, S + 1 + DS);
          const u32x4 *lc = units[S & 1][wr], *lp = punits[S & 1][wave];
          codes(lc, lp, 0, wc, par);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int q = 4 * S + i, s = (4 * d + i) % NQ;
            uint32_t wn[LW * BPL], pn = 0;
            if (i < 3) codes(lc, lp, i + 1, wn, pn);
            const float av = fabsf(rs[s]);
            if (q < nq) {
              big = big || (av >= 0x1p88f && av < INFINITY);
              step(s, q, sub);
            }
            load_a(s, q + NQ);
            __builtin_amdgcn_sched_barrier(0);
            if (i < 3) {
              par = pn;
#pragma unroll
              for (int k = 0; k < LW * BPL; ++k) wc[k] = wn[k];
            }
          }
        }
      }
    }
    __syncthreads();  // every wave is done with the LDS stages
  };
  run(std::true_type{});
  // Some scale of the tile's tokens is finite and 2^88 or more (every wave
  // of the block sees the same scales): again in the other code form.
  if (__builtin_amdgcn_ballot_w64(big) != 0) run(std::false_type{});

  // hsum8 of the row tile's chains (lanes 4..7 are +0 at group 32), which the
  // CW waves hold.
  float all[NL][4];
  if constexpr (CW == 1) {
#pragma unroll
    for (int l = 0; l < NL; ++l)
#pragma unroll
      for (int r = 0; r < 4; ++r) all[l][r] = f[l][r];
  } else {
    float(*fin)[NL][4][64] = reinterpret_cast<float(*)[NL][4][64]>(&units[0][0][0]);
    static_assert(sizeof(units) >= sizeof(float) * WR * NL * 4 * 64, "the chains fit the stages");
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
                     int rows, int cols, int m, hipStream_t s) {
  const int rt = (rows + 15) / 16, tt = (m + 15) / 16;
  auto go = [&](auto cw) {
    constexpr int CW = decltype(cw)::value;
    const dim3 grid((rt + 4 / CW - 1) / (4 / CW), tt);
    hipLaunchKernelGGL((k_gemv_stream<GS, CW>), grid, dim3(256), 0, s, out, add, nib, params, qa, rows, cols,
                       m);
  };
  // CW from the number of row x token tiles, measured on 2048..28672 rows, K
  // 2048..14464 and 2..64 tokens with the weights from HBM (us, CW = 1 / 2 /
  // 4).  Group 32: 768 tiles 24.2 / 22.4 / 19.9, 1024 25.3 / 23.8 / 28.2, 1792
  // 40.0 / 47.1 / 49.5.  Group 64: 256 - / 14.1 / 10.8, 512 - / 8.3 / 8.2, 768
  // - / 18.2 / 20.4, 1792 - / 38.8 / 46.8.  Group 128: 256 - / 26.3 / 19.1, 512
  // equal, 768 - / 14.2 / 15.7.  (One wave per tile does not fit the registers
  // past group 32.)
  const int tiles = rt * tt;
  if (tiles <= (GS == 32 ? 800 : 512)) {
    go(std::integral_constant<int, 4>{});
    return;
  }
  if constexpr (GS == 32) {
    if (tiles >= 1200) {
      go(std::integral_constant<int, 1>{});
      return;
    }
  }
  go(std::integral_constant<int, 2>{});
}

}  // namespace

size_t qa_bytes(int m, int cols, int gs) {
  return (size_t)((m + 15) / 16) * ((cols / gs + 3) / 4) * qa_rec_bytes(gs);
}

void launch_gemv_stream(float *out, const float *add, const uint8_t *nib, const uint8_t *params, const _Float16 *qa,
                        int rows, int cols, int m, int gs, hipStream_t s) {
  if (gs == 32)
    launch_stream_t<32>(out, add, nib, params, qa, rows, cols, m, s);
  else if (gs == 64)
    launch_stream_t<64>(out, add, nib, params, qa, rows, cols, m, s);
  else
    launch_stream_t<128>(out, add, nib, params, qa, rows, cols, m, s);
}

}  // namespace rai
