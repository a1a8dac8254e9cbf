// W4A8 GEMM for prefill-sized token counts (w4a8_route) on the gfx950 matrix
// cores, groups of 32, 64 or 128: the reference's matmul_chunk_i8 /
// matmul_row_tile (gemm.rs:540-784) with the same per-lane integer sums and
// the same f32 epilogue order, so the outputs equal the CPU path bit for bit.
//
// Integer part.  The reference's lane l takes the 8-column blocks l, l + 4,
// ... of a group of 32 (four lanes) or l, l + 8, ... of a group of 64 or 128
// (eight lanes).  One matrix instruction takes exactly the K-slice of one
// lane: v_mfma_f32_32x32x8_f16 one block (groups 32 and 64),
// v_mfma_f32_32x32x16_f16 the two blocks l and l + 8 (group 128).  So
// D[token][row] is the lane sum S_l (the PMADDUBSW/PMADDWD sum of code x
// activation products, gemm.rs:606-614) for 32 tokens x 32 rows, with no
// block-diagonal padding.  Codes 0..15
// enter as f16 subnormals n 2^-24 (odd columns 16 n 2^-24: one mask per
// pair), activations as f16 a (odd columns a / 16); every product and
// partial sum is an integer times 2^-24 below 2^-9, so the f32
// accumulators hold S 2^-24 exactly in any order, and the records carry the
// activation scales times 2^24, so that fl(S 2^-24 * fl(ws * as 2^24)) =
// fl(S * fl(ws * as)) (power-of-two scaling commutes with rounding in the
// normal range; ws * as is zero or above 2^-24 * 1e-10 / 127).  A group
// whose 32 tokens include a scale of 2^88 or more (where as 2^24
// could overflow the product) keeps its scales as they are, is flagged,
// and runs with the codes as f16 1024 + n minus 1024 (S itself).  The
// f16 instruction is used rather than an int8 one because it returns S
// already as f32: an i32 result would cost one VALU conversion per S, and
// the VALU epilogue, not the matrix core, bounds this kernel.
//
// Scale products.  cs = fl(ws * as) and fl(wz * xsum) for 32 tokens x 32
// rows are outer products, which v_mfma_f32_32x32x1_2b_f32 rounds once
// (one product and +0): block 0 gives the 1024 cs, block 1 the 1024 zero
// terms, 64 matrix cycles against 128 VALU ones, from one LDS dword per
// lane.  (A product of -0 comes out as +0; neither chain sees a difference,
// since a sum that starts at +0 is never -0.)  What stays on the VALU is
// two operations per lane sum and one per zero term: 9 per (row, token,
// group of 32), 17 per group of 64 or 128.
//
// Lane roles: B = weights, lane l holds row j = l % 32 and the K-slice half
// h = l / 32; A = activations, token i = l % 32, half h; the
// lane's 16 results are tokens 8 (v / 4) + 4 h + v % 4 of row j.  K order
// of a half: columns (2h, 2h + 4, 2h + 1, 2h + 5) of the block (groups 32
// and 64); the whole block l + 8h, columns (0, 4, 1, 5, 2, 6, 3, 7) (128).
//
// Epilogue per lane, for its row and 16 tokens, in group order
// (gemm.rs:616-651): f_l += fl(S_l * cs); zc += fl(wz * xsum); at the end
// out = hsum8(f) + zc (the movehdup/movehl sum of gemm.rs:655-662; lanes
// 4..7 stay +0 at group 32).
//
// Data: activations are packed once per GEMM input by k_mm_pack into
// records per (32-token tile, group): GS / 8 512-byte A operands
// (lane-ordered), then 32 scales (times 2^24 unless flagged) and 32 input
// sums; after the records one int per (token tile, group), nonzero
// for a flagged group.  The groups of a tile are padded to the kernel's
// step (UG) with zero records, whose parameters are taken as zero: every
// term they add is +0.  A block of WR waves
// (32 rows each) shares one token tile; the records of P groups are copied
// to LDS by DMA (global_load_lds), double-buffered.  Each lane streams its
// row's codes and parameters through a register ring UG groups ahead.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "kernels.h"
#include "quant_dev.h"

namespace rai {

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f32v __attribute__((ext_vector_type(32)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

constexpr int kMmWR = 4;  // waves (32-row tiles) per block

template <int GS>
struct MmCfg {
  static constexpr int REC = GS * 64 + 256;           // bytes per (token tile, group)
  static constexpr int P = 512 / GS;                  // groups per LDS stage
  static constexpr int UG = GS == 32 ? 4 : 2;         // groups per unrolled step and ring slots
  static constexpr int NU = GS == 32 ? 1 : 2;         // 16-byte code loads per lane and group
  static constexpr int NL = GS == 32 ? 4 : 8;         // reference lanes
  static_assert(P % UG == 0, "whole steps per stage");
};

int mm_rec(int gs) { return gs * 64 + 256; }
int mm_pad_groups(int groups, int gs) {
  const int ug = gs == 32 ? 4 : 2;
  return (groups + ug - 1) / ug * ug;
}

// Token tile t of a packed input covers rows src[first + 0..count) of
// q_split (src null: rows first..); without a tile table, tile t is rows
// 32t..32t + 31 of m.
struct MmTile {
  int first, count;
};
__device__ __forceinline__ MmTile mm_tile(const MmMoe &moe, int tt, int m) {
  if (moe.tiles) return {moe.tiles[tt].y, moe.tiles[tt].z};
  return {tt * 32, min(32, m - tt * 32)};
}

// One block per (token tile, 128 columns of the padded row), 256 threads.
// The tile's 32 rows of those columns are read with whole-line loads (eight
// lanes of 16 bytes per row) into LDS; then each thread writes its lanes'
// f16 A values, and one thread per (group, token) its scale or input
// sum.  Tokens past the tile's count and columns past the row are zero.
template <int GS>
__global__ __launch_bounds__(256) void k_mm_pack(const int8_t *__restrict__ q_split,
                                                 const float *__restrict__ scales, const float *__restrict__ sums,
                                                 int m, int cols, int gpad, uint8_t *__restrict__ rec, MmMoe moe) {
  constexpr int QS = 128 + 16;  // LDS row stride (bytes)
  constexpr int REC = MmCfg<GS>::REC, GB = 128 / GS;  // groups per block
  __shared__ __align__(16) int8_t qs[32 * QS];
  const int tid = threadIdx.x, c0 = 128 * blockIdx.x, tt = blockIdx.y;
  const int groups = cols / GS, g0 = GB * blockIdx.x;
  int *flags = reinterpret_cast<int *>(rec + (size_t)gridDim.y * gpad * REC) + (size_t)tt * gpad;
  if (moe.tiles && tt >= *moe.ntiles) return;
  const MmTile tile = mm_tile(moe, tt, m);
  auto src_row = [&](int i) { return moe.tiles && moe.src ? moe.src[tile.first + i] : tile.first + i; };
  {
    const int i = tid >> 3, col = c0 + 16 * (tid & 7);
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if (i < tile.count && col < cols)
      v = *reinterpret_cast<const uint4 *>(q_split + (size_t)src_row(i) * cols + col);
    *reinterpret_cast<uint4 *>(qs + i * QS + 16 * (tid & 7)) = v;
  }
  __syncthreads();
  uint8_t *r0 = rec + ((size_t)tt * gpad + g0) * REC;
  const int l = tid & 63, i = l & 31, h = l >> 5, wave = tid >> 6;
  // q_split block: four even columns, then four odd ones.
  if constexpr (GS == 128) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int b = wave + 4 * u;  // reference lane b: block b (h = 0) or b + 8
      const int8_t *e = qs + i * QS + 8 * (b + 8 * h);
      h8 a;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        a[4 * k + 0] = (_Float16)(float)e[k];
        a[4 * k + 1] = (_Float16)(float)e[k + 2];
        a[4 * k + 2] = (_Float16)((float)e[4 + k] * 0.0625f);
        a[4 * k + 3] = (_Float16)((float)e[6 + k] * 0.0625f);
      }
      *reinterpret_cast<h8 *>(r0 + b * 1024 + l * 16) = a;
    }
  } else {
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int blk = wave + 4 * u;           // of the 16 blocks of these columns
      const int g = blk / (GS / 8), b = blk % (GS / 8);
      if (g0 + g < gpad) {
        const int8_t *e = qs + i * QS + 8 * blk;
        h4 a;
        a[0] = (_Float16)(float)e[h];
        a[1] = (_Float16)(float)e[h + 2];
        a[2] = (_Float16)((float)e[4 + h] * 0.0625f);
        a[3] = (_Float16)((float)e[6 + h] * 0.0625f);
        *reinterpret_cast<h4 *>(r0 + g * REC + b * 512 + l * 8) = a;
      }
    }
  }
  // Wave g writes group g's scales (lanes 0..31) and sums.
  if (wave < GB && g0 + wave < gpad) {
    const int g = wave;
    float v = 0.0f;
    if (i < tile.count && g0 + g < groups) v = (h ? sums : scales)[(size_t)src_row(i) * groups + g0 + g];
    const float av = fabsf(v);
    const bool huge = __builtin_amdgcn_ballot_w64(h == 0 && av >= 0x1p88f && av < INFINITY) != 0;
    reinterpret_cast<float *>(r0 + g * REC + GS * 64)[l] = (h == 0 && !huge) ? v * 0x1p24f : v;
    if (l == 0) flags[g0 + g] = huge;
  }
}

// The reference lanes' sums D = A_l x B_l of one group.
template <int GS, bool SUB>
__device__ __forceinline__ f16v mm_lane_sums(const uint8_t *rc, const u4v (&wq)[MmCfg<GS>::NU], int b, uint32_t sh,
                                             int lane) {
  const f16v zero = {};
  if constexpr (GS == 128) {
    const uint32_t w = wq[b >> 2][b & 3];
    const h4 lo = codes_half<SUB>(w), hi = codes_half<SUB>(w >> 8);
    const h8 bq = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const h8 *>(rc + b * 1024 + lane * 16), bq, zero,
                                                  0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x8f16(*reinterpret_cast<const h4 *>(rc + b * 512 + lane * 8),
                                                codes_half<SUB>(wq[b >> 2][b & 3] >> sh), zero, 0, 0, 0);
  }
}

template <int GS>
struct MmLane {
  float f[MmCfg<GS>::NL][16];
  float zc[16];
};

// One group: the scale products and the lane sums from the LDS record `rc`
// and the code ring slot `wq`, then the epilogue with parameter dword `pw`.
// Codes as f16 subnormals (SUB), or as 1024 + n with the record's scales
// times smul (2^-24 for those stored times 2^24: exact).
template <int GS, bool SUB>
__device__ __forceinline__ void mm_group(const uint8_t *rc, const u4v (&wq)[MmCfg<GS>::NU], uint32_t pw, uint32_t sh,
                                         int lane, float smul, MmLane<GS> &acc) {
  constexpr int NL = MmCfg<GS>::NL;
  // Lanes 0..31: token scale and weight scale; 32..63: input sum and zero.
  float as = reinterpret_cast<const float *>(rc + GS * 64)[lane];
  if constexpr (!SUB) as = as * (sh ? 1.0f : smul);
  const float wp = (float)__builtin_bit_cast(_Float16, (uint16_t)(pw >> (2 * sh)));
  const f32v zero = {};
  const f32v cz = __builtin_amdgcn_mfma_f32_32x32x1f32(as, wp, zero, 0, 0, 0);
  f16v D0 = mm_lane_sums<GS, SUB>(rc, wq, 0, sh, lane);
  f16v D1 = mm_lane_sums<GS, SUB>(rc, wq, 1, sh, lane);
#pragma unroll
  for (int v = 0; v < 16; ++v) acc.zc[v] = acc.zc[v] + cz[16 + v];
#pragma unroll
  for (int b = 0; b < NL; b += 2) {
#pragma unroll
    for (int v = 0; v < 16; ++v) acc.f[b][v] = acc.f[b][v] + D0[v] * cz[v];
    if (b + 2 < NL) D0 = mm_lane_sums<GS, SUB>(rc, wq, b + 2, sh, lane);
#pragma unroll
    for (int v = 0; v < 16; ++v) acc.f[b + 1][v] = acc.f[b + 1][v] + D1[v] * cz[v];
    if (b + 3 < NL) D1 = mm_lane_sums<GS, SUB>(rc, wq, b + 3, sh, lane);
  }
}

// Block: WR waves x 32 rows, one token tile (blockIdx.y).  Requires
// rows * cols / 2 < 2^31.
template <int GS, int WR>
__global__ __launch_bounds__(64 * WR, 2) void k_w4a8_mm(float *out, const float *add, const uint8_t *nib,
                                                        const uint8_t *params, const uint8_t *__restrict__ rec,
                                                        int rows, int cols, int m, int ld, MmMoe moe) {
  using C = MmCfg<GS>;
  constexpr int REC = C::REC, P = C::P, UG = C::UG, NU = C::NU;
  constexpr int STAGE = (P * REC + 1023) & ~1023;  // whole DMA pieces
  // Two arrays, so that the compiler can tell a stage's reads from the DMA
  // into the other buffer.
  __shared__ __align__(16) uint8_t bufA[STAGE];
  __shared__ __align__(16) uint8_t bufB[STAGE];
  if (moe.tiles && (int)blockIdx.y >= *moe.ntiles) return;  // the whole block
  const MmTile tile = mm_tile(moe, blockIdx.y, m);
  if (moe.tiles) {
    const int e = moe.tiles[blockIdx.y].x;
    nib = moe.nib_tab[(size_t)e * moe.tstride];
    params = moe.par_tab[(size_t)e * moe.tstride];
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, h = lane >> 5;
  const uint32_t sh = 8u * h;
  const int groups = cols / GS, gpad = (groups + UG - 1) / UG * UG, ntile = (gpad + P - 1) / P;
  const int row = blockIdx.x * 32 * WR + 32 * wave + j;
  const int rowc = min(row, rows - 1);
  const uint8_t *rtile = rec + (size_t)blockIdx.y * gpad * REC;
  const __amdgpu_buffer_rsrc_t rcs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(nib), 0, rows * (cols / 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rps =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(params), 0, rows * groups * 4, 0x00020000);
  // Group 128: lane half h multiplies the blocks 8h..8h + 7 only.
  const uint32_t vc0 = (uint32_t)rowc * (cols / 2) + (GS == 128 ? 32u * h : 0u);
  const uint32_t vp0 = (uint32_t)rowc * groups * 4;

  // Stage kt's records, 1 KB per instruction; the last piece may read past
  // the tile's records into the bytes behind them (mm_pack_bytes pads the
  // end), which no group uses.
  auto dma = [&](uint8_t *b, int kt) {
    const uint8_t *src = rtile + (size_t)kt * P * REC;
    const int n = min(P, gpad - kt * P) * REC;
    for (int c = wave * 1024; c < n; c += WR * 1024)
      __builtin_amdgcn_global_load_lds(src + c + lane * 16, (lds_void *)(b + c), 16, 0, 0);
  };
  // Ring: codes and parameters of groups g..g + UG - 1 (slot g % UG);
  // refills clamped to the last group.
  u4v wr[UG][NU];
  uint32_t pr[UG];
  auto load = [&](u4v (&w)[NU], uint32_t &p, int g) {
    const int gc = min(g, groups - 1);
#pragma unroll
    for (int u = 0; u < NU; ++u)
      w[u] = __builtin_amdgcn_raw_buffer_load_b128(rcs, (int)(vc0 + 16 * u), gc * (GS / 2), 0);
    p = __builtin_amdgcn_raw_buffer_load_b32(rps, (int)vp0, gc * 4, 0);
  };
#pragma unroll
  for (int s = 0; s < UG; ++s) load(wr[s], pr[s], s);
  dma(bufA, 0);
  MmLane<GS> acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
#pragma unroll
    for (int b = 0; b < C::NL; ++b) acc.f[b][v] = 0.0f;
    acc.zc[v] = 0.0f;
  }
  __syncthreads();

  // Flags of this token tile: any set (rare) runs the whole block with
  // the codes as 1024 + n, and the unflagged groups' scales times 2^-24.
  const int *gflag = reinterpret_cast<const int *>(rec + (size_t)gridDim.y * gpad * REC) + (size_t)blockIdx.y * gpad;
  int fl = 0;
  for (int i = lane; i < gpad; i += 64) fl |= gflag[i];
  const bool anybig = __builtin_amdgcn_ballot_w64(fl != 0) != 0;

  auto run = [&](auto sub) __attribute__((always_inline)) {
    constexpr bool SUB = decltype(sub)::value;
    auto stage = [&](const uint8_t *b, int kt) __attribute__((always_inline)) {
      const int cnt = min(P, gpad - kt * P);  // a multiple of UG
      for (int g0 = 0; g0 < cnt; g0 += UG) {
#pragma unroll
        for (int gi = 0; gi < UG; ++gi) {
          const int g = kt * P + g0 + gi;
          float smul = 1.0f;
          if constexpr (!SUB) smul = __builtin_amdgcn_readfirstlane(gflag[g]) ? 1.0f : 0x1p-24f;
          mm_group<GS, SUB>(b + (g0 + gi) * REC, wr[gi], g < groups ? pr[gi] : 0u, sh, lane, smul, acc);
          load(wr[gi], pr[gi], g + UG);
        }
      }
    };
    for (int kt = 0; kt < ntile; kt += 2) {
      if (kt + 1 < ntile) dma(bufB, kt + 1);
      stage(bufA, kt);
      __syncthreads();
      if (kt + 1 < ntile) {
        if (kt + 2 < ntile) dma(bufA, kt + 2);
        stage(bufB, kt + 1);
        __syncthreads();
      }
    }
  };
  if (anybig)
    run(std::false_type{});
  else
    run(std::true_type{});
  if (row < rows) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int t = 8 * (v >> 2) + 4 * h + (v & 3);
      if (t < tile.count) {
        const size_t oi = (size_t)(tile.first + t) * ld + row;
        float r;
        if constexpr (C::NL == 4)
          r = ((acc.f[0][v] + acc.f[1][v]) + (acc.f[2][v] + acc.f[3][v])) + acc.zc[v];
        else
          r = (((acc.f[0][v] + acc.f[4][v]) + (acc.f[1][v] + acc.f[5][v])) +
               ((acc.f[2][v] + acc.f[6][v]) + (acc.f[3][v] + acc.f[7][v]))) + acc.zc[v];
        out[oi] = add ? add[oi] + r : r;
      }
    }
  }
}

template <int GS>
void launch_mm_t(float *out, const float *add, const uint8_t *nib, const uint8_t *params, const int8_t *q_split,
                 const float *scales, const float *sums, int rows, int cols, int m, int ntt, int ld, uint8_t *pack,
                 const MmMoe &moe, hipStream_t s) {
  const int gpad = mm_pad_groups(cols / GS, GS);
  if (q_split)
    hipLaunchKernelGGL(k_mm_pack<GS>, dim3((gpad * GS + 127) / 128, ntt), dim3(256), 0, s, q_split, scales, sums, m,
                       cols, gpad, pack, moe);
  if (out)
    hipLaunchKernelGGL((k_w4a8_mm<GS, kMmWR>), dim3((rows + 32 * kMmWR - 1) / (32 * kMmWR), ntt), dim3(64 * kMmWR), 0,
                       s, out, add, nib, params, pack, rows, cols, m, ld, moe);
}

}  // namespace

// Against the VALU kernel that the shapes outside group 32 and K % 512 == 0
// took before, whole calls measured 14336x4096 at 512 tokens, group 128: 2084
// -> 176 us; 4096x11008 at 301 tokens, group 32: 1630 -> 228 us (1.25 waves
// per SIMD: the 1280 waves leave three quarters of the SIMDs with one).
static bool mm_ok(int rows, int cols, int gs) {
  return (gs == 32 || gs == 64 || gs == 128) && rows > 0 && cols > 0 && cols % gs == 0 &&
         (int64_t)rows * (cols / 2) < ((int64_t)1 << 31);
}

// Two to four tokens on the tiled VALU kernel, whose time grows with the tokens
// where the streamed kernel's (16 token slots) does not (device time, weights
// from HBM, us, VALU / streamed):
// - Two tokens: 28672x4096 group 64 26.2 / 36.1, group 128 26.1 / 29.7;
//   11008x4128 group 32 14.9 / 21.4; 256x2048 group 64 5.7 / 6.7.  One to four
//   groups of 64 or 128 in few rows: 4096x256 group 128 5.1 / 4.7.
// - Three, where the streamed kernel's blocks leave much of their last round
//   empty (5000 to 12288 rows: 384 or 344 blocks on 256 CUs) or K is short:
//   11008x4096 group 64 16.0 / 19.4, group 128 13.5 / 15.9; 6144x2048 group 64
//   8.1 / 9.2, 6144x14336 38.0 / 34.2; 28672x2048 group 64 19.1 / 22.3, group 128
//   18.3 / 19.0; 4096x2048 group 64 7.2 / 7.4; 14336x4096 23.6 / 20.5.
// - Four: 11008x2048 group 64 11.1 / 12.2, 11008x4096 27.1 / 19.5.
static bool small_path(int rows, int cols, int m, int gs) {
  if (m == 2) return gs == 32 || cols >= 1024 || rows > 5000;
  if (m == 3) return rows > 5000 && (rows <= 12288 ? cols <= 4096 || rows > 8192 : gs < 128 && cols < 4096);
  return m == 4 && rows > 8192 && rows <= 12288 && cols <= 2048;
}

// Where the lines lie (device time, weights from HBM):
// - The register-pipelined kernel, whose tiles are four tokens, where
//   gemv_rp_path says so; the VALU kernel for small_path's few tokens.
// - The streamed kernel has 16 x 16 tiles and splits a tile's chains over
//   waves, so it wins until the GEMM's 32 x 32 tiles alone fill the chip, at
//   about 4500 tiles of its own: group 32, K = 4096, 28672 rows, 32 tokens (3584
//   tiles) 68.2 against 70.0, 64 tokens (7168) 120.5 against 97.5; 4096 rows, 96
//   tokens (1536) 36 against 66.  Group 128, where the GEMM's two blocks per
//   instruction count: 14336 rows, 33 tokens (2688) 38.4 against 41.1, 64
//   (3584) 46.7 against 41.7.
// - Up to 16 tokens half of the GEMM's tile would be padding at any size.
W4Route w4a8_route(int rows, int cols, int m, int gs, bool tiled) {
  if (!mm_ok(rows, cols, gs)) return W4Route::kValu;
  if (gemv_rp_path(rows, cols, m, gs, tiled)) return W4Route::kRp;
  if (small_path(rows, cols, m, gs)) return W4Route::kSmall;
  const int64_t tiles = (int64_t)((rows + 15) / 16) * ((m + 15) / 16);
  if ((m <= 16 || tiles <= (gs == 128 ? 3000 : 4500)) && qa_bytes(m, cols, gs) < ((size_t)1 << 31))
    return W4Route::kStream;
  return W4Route::kMm;
}

// Records, flags and the bytes the last DMA piece may read past them.
size_t mm_pack_tiles_bytes(int tiles, int cols, int gs) {
  const size_t n = (size_t)tiles * mm_pad_groups(cols / gs, gs);
  return n * mm_rec(gs) + n * sizeof(int) + 1024;
}

size_t mm_pack_bytes(int m, int cols, int gs) { return mm_pack_tiles_bytes((m + 31) / 32, cols, gs); }

void launch_w4a8_mm(float *out, const float *add, const uint8_t *nib, const uint8_t *params, const int8_t *q_split,
                    const float *scales, const float *sums, int rows, int cols, int m, int gs, uint8_t *pack,
                    hipStream_t s) {
  const int ntt = (m + 31) / 32;
  auto go = [&](auto launch) {
    launch(out, add, nib, params, q_split, scales, sums, rows, cols, m, ntt, rows, pack, MmMoe{}, s);
  };
  if (gs == 32)
    go(launch_mm_t<32>);
  else if (gs == 64)
    go(launch_mm_t<64>);
  else
    go(launch_mm_t<128>);
}

bool moe_mm_path(int rows, int cols, int gs) { return mm_ok(rows, cols, gs); }

void launch_moe_mm(float *out, int ld, const MmMoe &moe, int max_tiles, const int8_t *q_split, const float *scales,
                   const float *sums, int rows, int cols, int gs, uint8_t *pack, hipStream_t s) {
  auto go = [&](auto launch) {
    launch(out, nullptr, nullptr, nullptr, q_split, scales, sums, rows, cols, 0, max_tiles, ld, pack, moe, s);
  };
  if (gs == 32)
    go(launch_mm_t<32>);
  else if (gs == 64)
    go(launch_mm_t<64>);
  else
    go(launch_mm_t<128>);
}

}  // namespace rai
