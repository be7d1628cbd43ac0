// r9k_moe_nvfp4.hip -- grouped (MoE) native-NVFP4-weight x fp8-activation GEMM for gfx950, routed through the
// moe_align_block_size tables (decode family: 16 * MT-row blocks).
//
//   out[r, n] = bf16( (sum_k A_q[r / a_row_div, k] * e2m1[n, k] * s16[n, k / 16]) * (Wg[n] * As[r / a_row_div]
//                     (* topk_w[r])) )
//
// with s16 the e4m3 scale of each 16-element group and Wg the fp32 per-row global multiplier: the checkpoint's NVFP4
// weight, exact, accumulated in fp32. Reference: kernels/r9k_moe_mxfp4a8.hip:89-96 and 300-340 (NVFP4 weight math),
// :469-482 (epilogue order), :641-647 (entry).
//
// The scaled MFMA applies only power-of-two (e8m0) block scales, so an e4m3 scale does not ride on it. Here the weights
// are widened to fp16: V_CVT_SCALEF32_PK_F16_FP4 (scale 1) gives e2m1, one V_CVT_SCALEF32_PK_F16_FP8 a lane's two group
// scales, and one packed fp16 multiply e2m1 * s16 (at most 6 significant bits and within [2^-10, 2688]: exact in fp16).
// The fp8 activations widen to fp16 exactly, and V_MFMA_F32_16X16X32_F16 accumulates the exact products in fp32 -- no
// per-group rescaling of partial sums. The widening's vector instructions bound these kernels next to the weight bytes
// (decode) and the matrix pipe (prefill): splitting s16 into the conversion's exponent operand and a mantissa factor
// took ~14 instructions a K-tile and column tile where this takes one.
// Operand layout of the instruction: A lane l holds row l % 16 and 8 K values, B lane l column l % 16 and the same 8
// K values, lane group g = l / 16 taking instruction K 8g .. 8g + 7; C lane l holds column l % 16, rows 4g .. 4g + 3.
// Step s (0..3) of a 128-wide K-tile gives lane group g the K values 32g + 8s .. + 7, so over the tile lane group g
// covers the 32 contiguous K values 32g .. 32g + 31 (groups 2g and 2g + 1): two 16-byte activation loads a row.
//
// Weight layout (per expert, produced by kernels/moe.py prepare_nvfp4_weights), nkt = ceil(K / 128):
//   codes  : N/16 column tiles of nkt K-tiles of 1 KB. Lane l = g * 16 + c of K-tile kt holds the 16 checkpoint bytes
//            W[16 nt + c, kt * 64 + 16 g .. + 16] at l * 16 (the MXFP4 fragment order), dword s feeding step s.
//   scales : N/16 column tiles of nkt K-tiles of 128 bytes. Lane l's 2 bytes at l * 2 are the e4m3 scales of groups
//            kt * 8 + 2g and kt * 8 + 2g + 1 of column c.
//   A partial last K-tile (K % 128 = 16 G) is stored whole, codes and scales zero past group G.
//   Wg     : fp32 [N] (wg_estride floats per expert).
#include "r9k_common.h"
#include "r9k_dma.h"
#include "r9k_rowquant.h"

namespace {

using namespace r9k;

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int NV_KT = 128;          // K per tile (8 groups)
constexpr int NV_G = 16;            // NVFP4 group

__device__ __forceinline__ u32x4 ld16_nt(const uint8_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
}
__device__ __forceinline__ uint32_t ld2_nt(const uint8_t* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const uint16_t*>(p));
}

// The two e4m3 group scales of a lane's K-tile (the low 16 bits of sw) as fp16, exact; NaN bytes stay NaN.
__device__ __forceinline__ h2 scales_f16(uint32_t sw) {
  return __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)sw, 1.0f, false);
}

// 8 e2m1 codes (one dword, low nibble first) -> e2m1 * s as 8 fp16, exact
__device__ __forceinline__ h8 e2m1x8_f16(uint32_t w, _Float16 s) {
  const h2 ss = {s, s};
  const h2 p0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 0) * ss;
  const h2 p1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 1) * ss;
  const h2 p2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 2) * ss;
  const h2 p3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 3) * ss;
  return (h8){p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// the two e2m1 codes of byte j (constant) of one dword as fp16
__device__ __forceinline__ h2 e2m1x2_f16(uint32_t w, int j) {
  return j == 0 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 0)
       : j == 1 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 1)
       : j == 2 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 2)
                : __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 3);
}

// 8 e4m3 codes (two dwords) -> 8 fp16, exact
__device__ __forceinline__ h8 e4m3x8_f16(uint32_t lo, uint32_t hi) {
  const h2 p0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)lo, 1.0f, false);
  const h2 p1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)lo, 1.0f, true);
  const h2 p2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)hi, 1.0f, false);
  const h2 p3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)hi, 1.0f, true);
  return (h8){p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// One workgroup: 16 * MT routed rows x NPW column tiles; SK waves split the K-tiles (SK > 1: partial tiles summed
// through LDS in wave order). Each wave walks its K range in batches of U K-tiles, all loads of a batch issued
// before its MFMAs; addresses past K are clamped and their groups skipped (uniform per tile).
template <int MT, int NPW, int SK, int U>
__global__ void __launch_bounds__(WAVE * SK) moe_nvfp4_kernel(
    const uint8_t* __restrict__ A, const float* __restrict__ As, const uint8_t* __restrict__ Wq,
    const uint8_t* __restrict__ Ws, const float* __restrict__ Wg, uint16_t* __restrict__ C,
    const int* __restrict__ sorted_ids, const int* __restrict__ expert_ids, const int* __restrict__ ntpp,
    const float* __restrict__ topk_w, long wq_estride, long ws_estride, long wg_estride, int numel, int a_row_div,
    int K, int N, int blk, int subs) {
  constexpr int BLK = 16 * MT;
  extern __shared__ float red[];

  const int rb = blockIdx.y / subs, sub = blockIdx.y - rb * subs;
  const int row0 = rb * blk + sub * BLK;
  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
  const int g = lane >> 4, c = lane & 15;
  const int np = ntpp[0];
  const int e = expert_ids[rb];
  const int first = sorted_ids[rb * blk];
  int fr_in[MT];
#pragma unroll
  for (int i = 0; i < MT; i++) fr_in[i] = sorted_ids[row0 + i * 16 + c];
  if (rb * blk >= np || e < 0) return;
  if (first < 0 || first >= numel || __shfl(fr_in[0], 0, WAVE) >= numel) return;   // padding: end of a block
  const int NT = N / 16;
  const int nkt = (K + NV_KT - 1) / NV_KT;
  const int kvalid_g = K - 32 * g;                          // K values of lane group g's run in tile kt: minus kt*128

  size_t arow[MT];
  float ras[MT], rtw[MT];                                  // row r of M-tile i (lane c's row): As, topk weight
#pragma unroll
  for (int i = 0; i < MT; i++) {
    int fr = fr_in[i];
    if (fr >= numel || fr < 0) fr = first;
    arow[i] = (size_t)(fr / a_row_div) * K;
    ras[i] = As[fr / a_row_div];
    rtw[i] = topk_w ? topk_w[fr] : 1.f;
  }
  const uint8_t* __restrict__ We = Wq + (size_t)e * wq_estride;
  const uint8_t* __restrict__ Se = Ws + (size_t)e * ws_estride;
  const float* __restrict__ Ge = Wg + (size_t)e * wg_estride;
  const uint8_t* wtile[NPW];
  const uint8_t* stile[NPW];
#pragma unroll
  for (int j = 0; j < NPW; j++) {
    int nt = (int)blockIdx.x * NPW + j;
    nt = nt < NT ? nt : NT - 1;                            // out-of-range tiles compute a copy, never stored
    wtile[j] = We + (size_t)nt * nkt * 1024;
    stile[j] = Se + (size_t)nt * nkt * 128;
  }

  v4f acc[NPW][MT];
#pragma unroll
  for (int j = 0; j < NPW; j++)
#pragma unroll
    for (int i = 0; i < MT; i++) acc[j][i] = (v4f){0.f, 0.f, 0.f, 0.f};

  const int kt0 = wave * nkt / SK, kt1 = (wave + 1) * nkt / SK;
  for (int kt = kt0; kt < kt1; kt += U) {
    u32x4 bw[U][NPW];
    uint32_t sw[U][NPW];
    uint4 alo[U][MT], ahi[U][MT];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = min(kt + u, kt1 - 1);
      // lane group g's 32 K values of this tile: 32, 16 (K % 32 == 16 at the end) or none; a missing half loads a
      // valid address and is zeroed below
      const int kv = kvalid_g - k * NV_KT;
      const int olo = kv >= 16 ? k * NV_KT + 32 * g : 0, ohi = kv >= 32 ? k * NV_KT + 32 * g + 16 : 0;
#pragma unroll
      for (int j = 0; j < NPW; j++) {
        bw[u][j] = ld16_nt(wtile[j] + (size_t)k * 1024 + lane * 16);
        sw[u][j] = ld2_nt(stile[j] + (size_t)k * 128 + lane * 2);
      }
#pragma unroll
      for (int i = 0; i < MT; i++) {
        alo[u][i] = *reinterpret_cast<const uint4*>(A + arow[i] + olo);
        ahi[u][i] = *reinterpret_cast<const uint4*>(A + arow[i] + ohi);
      }
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = kt + u;
      if (k < kt1) {
        const int kv = kvalid_g - k * NV_KT;
        const bool lo_ok = kv >= 16, hi_ok = kv >= 32;
        h8 a[MT][4];
#pragma unroll
        for (int i = 0; i < MT; i++) {
          const uint4 l = lo_ok ? alo[u][i] : make_uint4(0u, 0u, 0u, 0u);
          const uint4 h = hi_ok ? ahi[u][i] : make_uint4(0u, 0u, 0u, 0u);
          a[i][0] = e4m3x8_f16(l.x, l.y);
          a[i][1] = e4m3x8_f16(l.z, l.w);
          a[i][2] = e4m3x8_f16(h.x, h.y);
          a[i][3] = e4m3x8_f16(h.z, h.w);
        }
#pragma unroll
        for (int j = 0; j < NPW; j++) {
          const h2 gs = scales_f16(sw[u][j]);
#pragma unroll
          for (int st = 0; st < 4; st++) {
            const h8 b = e2m1x8_f16(bw[u][j][st], gs[st >> 1]);
#pragma unroll
            for (int i = 0; i < MT; i++) acc[j][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i][st], b, acc[j][i], 0, 0, 0);
          }
        }
      }
    }
  }

  if constexpr (SK == 1) {
    // lane holds column c of each tile, rows 4g .. 4g + 3; row factors come from the lanes that loaded them
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int fr = __shfl(fr_in[i], 4 * g + q, WAVE);
        const float as_ = __shfl(ras[i], 4 * g + q, WAVE), tw = __shfl(rtw[i], 4 * g + q, WAVE);
        if (fr < 0 || fr >= numel) continue;
#pragma unroll
        for (int j = 0; j < NPW; j++) {
          const int n = (blockIdx.x * NPW + j) * 16 + c;
          if (n < N) {
            float sc = Ge[n] * as_;
            if (topk_w) sc *= tw;
            C[(size_t)fr * N + n] = f2bf(acc[j][i][q] * sc);
          }
        }
      }
  } else {
    __shared__ int s_fr[MT * 16];
    __shared__ float s_as[MT * 16], s_tw[MT * 16];
    if (wave == 0 && g == 0) {
#pragma unroll
      for (int i = 0; i < MT; i++) {
        s_fr[i * 16 + c] = fr_in[i];
        s_as[i * 16 + c] = ras[i];
        s_tw[i * 16 + c] = rtw[i];
      }
    }
#pragma unroll
    for (int j = 0; j < NPW; j++)
#pragma unroll
      for (int i = 0; i < MT; i++) {
        float* t = red + (size_t)((wave * NPW + j) * MT + i) * 256;
#pragma unroll
        for (int q = 0; q < 4; q++) t[(4 * g + q) * 16 + c] = acc[j][i][q];
      }
    __syncthreads();
    constexpr int TOT = NPW * MT * 256;
    for (int idx = tid; idx < TOT; idx += WAVE * SK) {
      const int col = idx & 15, row = (idx >> 4) & 15, ti = idx >> 8;   // ti = j * MT + i
      const int j = ti / MT, i = ti - j * MT;
      const int n = (blockIdx.x * NPW + j) * 16 + col;
      if (n >= N) continue;
      const int fr = s_fr[i * 16 + row];
      if (fr < 0 || fr >= numel) continue;
      float v = 0.f;
#pragma unroll
      for (int s = 0; s < SK; s++) v += red[(size_t)s * TOT + idx];
      float sc = Ge[n] * s_as[i * 16 + row];
      if (topk_w) sc *= s_tw[i * 16 + row];
      C[(size_t)fr * N + n] = f2bf(v * sc);
    }
  }
}

struct NvPick { int NPW, SK, U; };

// Launch shape from the host-known shape: two column tiles a workgroup (one for a dense linear of up to 8 rows); K
// split over SK waves for long K; each wave issues its K range in as few load batches as 4 K-tiles a batch allow (5
// for a dense linear of more than 8 rows).
NvPick nv_pick(int N, int K, int max_blocks, int rows, int MT) {
  const int nkt = (K + NV_KT - 1) / NV_KT;
  const int NT = N / 16;
  const int NPW = NT >= 2 ? 2 : 1;
  const long tiles = (long)max_blocks * ((NT + NPW - 1) / NPW);
  const int SK = nkt >= 8 ? (tiles >= 12288 ? 2 : 4) : 1;
  const int per = (nkt + SK - 1) / SK;
  int U = per >= 4 ? 4 : (per >= 2 ? 2 : 1);
  int npw = NPW;
  if (MT == 1 && max_blocks <= 2 && SK == 4 && per >= 5) {
    // at most two 16-row routing blocks (a dense linear at decode widths: moe_gemm sizes the grid at ceil(numel / 16) +
    // min(numel, E) blocks): one column tile a workgroup up to 8 rows, two and 5-tile
    // batches above (config 4, [17408, 5120], quant + GEMM: M = 1 19.6 -> 18.4 us, M = 4 19.5 -> 18.8, M = 16
    // 23.6 -> 22.8; the K split is unchanged, so the bits are too)
    npw = rows > 8 ? 2 : 1;
    U = rows > 8 ? 5 : 4;
  }
  return {npw, SK, U};
}

template <int MT, int NPW, int SK, int U>
void nv_launch(dim3 grid, hipStream_t st, long a, long as, long wq, long ws, long wg, long c, long sorted_ids,
               long expert_ids, long ntpp, long topk_w, long wq_estride, long ws_estride, long wg_estride, int numel,
               int a_row_div, int K, int N, int blk, int subs) {
  const size_t smem = SK > 1 ? (size_t)SK * NPW * MT * 256 * sizeof(float) : 0;
  hipLaunchKernelGGL((moe_nvfp4_kernel<MT, NPW, SK, U>), grid, dim3(WAVE * SK), smem, st, (const uint8_t*)a,
                     (const float*)as, (const uint8_t*)wq, (const uint8_t*)ws, (const float*)wg, (uint16_t*)c,
                     (const int*)sorted_ids, (const int*)expert_ids, (const int*)ntpp, (const float*)topk_w,
                     wq_estride, ws_estride, wg_estride, numel, a_row_div, K, N, blk, subs);
}

// ------------------------------------------------------------------------------------------ prefill (tiles of 128)
// Routed rows in blocks of 128 (a routing block of 128 or 256 rows covered by 1 or 2 workgroups along grid.y) x 128
// output columns per workgroup; 4 waves in 2 x 2, each 64 rows x 64 columns = 4 x 4 tiles of the fp16 MFMA above.
// K runs in 128-wide tiles through a ring of three LDS slots (activations 16 KB, codes 8 KB, scales 1 KB) filled by
// direct global -> LDS DMA (every wave issues the same 7 DMA instructions a K-tile, so the waits are fixed vmcnt counts;
// no compiler-tracked load sits in the loop). Each wave widens its 4 column tiles' weights once per K-tile (codes and
// scales from LDS, as in the decode kernel) and reuses them over its 4 row tiles; the activation rows are widened per
// row tile. Bound: the matrix pipe and, nearly as long, the widening's vector instructions (two conversions and a
// multiply an MFMA, all at the full rate of 4 clocks a wave instruction). So they have to overlap within a wave: every
// MFMA carries one conversion pair of the next row tile's activations and one of the next K-tile's weights. Widening a
// K-tile's weights ahead of its MFMAs instead left that to the other wave of the SIMD. [17408, 5120], 2000 rows: 325 ->
// 313 us (1.14 PFLOP/s, where a plain bf16 matrix product of 8192^3 reaches 1.21 on the same card; matrix pipe busy 55%
// of the clocks); row-block groups on top, an L2-friendlier tile order, 0.7%: not kept.
// Activation row pieces sit XOR-swizzled (16-byte piece p of row r at position p ^ (r & 7)) so the 16 rows a fragment
// read touches land in different banks: the DMA lane that fills position p of row r fetches piece p ^ (r & 7). Past K
// (a partial last K-tile) an activation piece is fetched from the row's last valid piece; the weights' codes and scales
// there are zero, so those products are exact zeros.
constexpr int PV_BM = 128, PV_BN = 128, PV_THREADS = 256;
constexpr int PV_NS = 3;           // LDS stages
constexpr int PV_DMA = 7;          // DMA instructions per wave and stage: 4 activation, 2 code, 1 scale

struct PvStage {
  uint8_t a[PV_BM * NV_KT];        // fp8 activations, row-major, swizzled 16-byte pieces
  uint8_t b[8 * 1024];             // codes of the 8 column tiles, the global layout's K-tile
  uint8_t s[8 * 128];              // their scales
};
struct PvW { u32x4 k[4]; };           // a column tile's widened weights of one K-tile
constexpr size_t PV_SMEM = PV_NS * sizeof(PvStage) + PV_BM * (sizeof(int) + 2 * sizeof(float));

template <bool PIPE>
__global__ void __launch_bounds__(PV_THREADS, 2) nvfp4_prefill_kernel(
    const uint8_t* __restrict__ A, const float* __restrict__ As, const uint8_t* __restrict__ Wq,
    const uint8_t* __restrict__ Ws, const float* __restrict__ Wg, uint16_t* __restrict__ C,
    const int* __restrict__ sorted_ids, const int* __restrict__ expert_ids, const int* __restrict__ ntpp,
    const float* __restrict__ topk_w, long wq_estride, long ws_estride, long wg_estride, int numel, int a_row_div,
    int K, int N, int blk, int subs) {
  extern __shared__ __align__(16) uint8_t pv_smem[];
  PvStage* st = reinterpret_cast<PvStage*>(pv_smem);
  int* s_fr = reinterpret_cast<int*>(pv_smem + PV_NS * sizeof(PvStage));
  float* s_as = reinterpret_cast<float*>(s_fr + PV_BM);         // As of each tile row (read once, before the loop)
  float* s_tw = s_as + PV_BM;                                  // topk_w of each tile row
  const int rb = blockIdx.y / subs, sub = blockIdx.y - rb * subs;
  const int row0 = rb * blk + sub * PV_BM;
  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
  const int g = lane >> 4, c = lane & 15, wm = wave >> 1, wn = wave & 1;
  const int np = ntpp[0];
  const int e = expert_ids[rb];
  const int first = sorted_ids[row0];
  if (rb * blk >= np || e < 0 || first < 0 || first >= numel) return;     // uniform: a dead block or padding
  if (tid < PV_BM) {
    const int fr = sorted_ids[row0 + tid];
    s_fr[tid] = fr;
    const bool live = fr >= 0 && fr < numel;
    s_as[tid] = live ? As[fr / a_row_div] : 0.f;
    s_tw[tid] = live && topk_w ? topk_w[fr] : 1.f;
  }
  __syncthreads();
  const int NT = N / 16, nkt = (K + NV_KT - 1) / NV_KT;
  const int nt0 = blockIdx.x * (PV_BN / 16);
  const uint8_t* We = uniform_ptr(Wq + (size_t)e * wq_estride);
  const uint8_t* Se = uniform_ptr(Ws + (size_t)e * ws_estride);
  const float* __restrict__ Ge = Wg + (size_t)e * wg_estride;

  // DMA sources (32-bit offsets from uniform bases; the host keeps A and one expert's codes below 4 GiB).
  // Activations: instruction i of wave w fills LDS pieces q = (4 i + w) * 64 + lane, i.e. row r = 32 i + 8 w + lane / 8
  // at position lane % 8, which holds the row's piece (lane % 8) ^ (r & 7) = (lane % 8) ^ (lane / 8).
  const int gp16 = ((lane & 7) ^ (lane >> 3)) * 16;
  uint32_t arow[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int f = s_fr[32 * i + 8 * wave + (lane >> 3)];
    f = (f < 0 || f >= numel) ? first : f;                     // padding rows load a valid row, never stored
    arow[i] = (uint32_t)(f / a_row_div) * (uint32_t)K;
  }
  // codes: instruction i of wave w fills column tile t = 4 i + w (1 KB); scales: wave w's dword lanes fill tiles
  // 2 w and 2 w + 1 (128 bytes each)
  uint32_t boff[2];
#pragma unroll
  for (int i = 0; i < 2; i++) boff[i] = (uint32_t)min(nt0 + 4 * i + wave, NT - 1) * (uint32_t)(nkt * 1024) + lane * 16;
  const uint32_t soff = (uint32_t)min(nt0 + (tid >> 5), NT - 1) * (uint32_t)(nkt * 128) + (tid & 31) * 4;
  const uint32_t la0 = lds_addr(&st[0].a[wave * 1024]);
  const uint32_t lb0 = lds_addr(&st[0].b[wave * 1024]);
  const uint32_t ls0 = lds_addr(&st[0].s[wave * 256]);
  // K-tile k's activations (4 loads) and codes + scales (3 loads) into ring slot sl; k past the end re-reads the last
  // K-tile, so every step issues the same loads
  auto issue_a = [&](int k, uint32_t sl) {
    const uint32_t ka = (uint32_t)min(min(k, nkt - 1) * NV_KT + gp16, K - 16);
#pragma unroll
    for (int i = 0; i < 4; i++) dma16s(A, arow[i] + ka, la0 + sl + i * 4096);
  };
  auto issue_w = [&](int k, uint32_t sl) {
    const uint32_t kc = (uint32_t)min(k, nkt - 1);
#pragma unroll
    for (int i = 0; i < 2; i++) dma16s(We, boff[i] + kc * 1024u, lb0 + sl + i * 4096);
    dma4s(Se, soff + kc * 128u, ls0 + sl);
  };

  constexpr uint32_t SL = sizeof(PvStage);
  // this lane's fragments in slot 0: row tile i at + i * 16 * NV_KT, column tile j at + j * 1024 (codes), + j * 128
  const int r0 = wm * 64 + c;
  const uint8_t* const fl = st[0].a + r0 * NV_KT + ((2 * g) ^ (r0 & 7)) * 16;
  const uint8_t* const fh = st[0].a + r0 * NV_KT + ((2 * g + 1) ^ (r0 & 7)) * 16;
  const uint8_t* const fw = st[0].b + wn * 4096 + lane * 16;
  const uint8_t* const fs = st[0].s + wn * 512 + lane * 2;
  auto ld_lo = [&](uint32_t sl, int i) { return *reinterpret_cast<const u32x4*>(fl + sl + i * 16 * NV_KT); };
  auto ld_hi = [&](uint32_t sl, int i) { return *reinterpret_cast<const u32x4*>(fh + sl + i * 16 * NV_KT); };
  auto ld_w = [&](uint32_t sl, int j) { return *reinterpret_cast<const u32x4*>(fw + sl + j * 1024); };
  auto ld_s = [&](uint32_t sl, int j) { return (uint32_t)*reinterpret_cast<const uint16_t*>(fs + sl + j * 128); };

  v4f acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};

  if constexpr (PIPE) {
    // Ahead of the loop: K-tiles 0 and 1 of everything and 2 of the weights on their way, K-tile 0's weights widened, the
    // raw weights of K-tile 1's first two column tiles and the raw activations of row tile 1 in registers
    issue_a(0, 0);
    issue_w(0, 0);
    issue_w(1, SL);
    issue_a(1, SL);
    issue_w(2, 2 * SL);
    __builtin_amdgcn_s_waitcnt(0xC07F);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(PV_DMA) : "memory");
    PvW B[2][3], b3;                                             // column tile 3 is widened in place
    u32x4 a[4], rl = ld_lo(0, 0), rh = ld_hi(0, 0), rw[2];
    uint32_t rs;
    h2 gs;
  #pragma unroll
    for (int j = 0; j < 4; j++) {
      rw[1] = ld_w(0, j);
      gs = scales_f16(ld_s(0, j));
      PvW& d = j < 3 ? B[0][j] : b3;
  #pragma unroll
      for (int t = 0; t < 4; t++) d.k[t] = __builtin_bit_cast(u32x4, e2m1x8_f16(rw[1][t], gs[t >> 1]));
    }
    a[0] = __builtin_bit_cast(u32x4, e4m3x8_f16(rl.x, rl.y));
    a[1] = __builtin_bit_cast(u32x4, e4m3x8_f16(rl.z, rl.w));
    a[2] = __builtin_bit_cast(u32x4, e4m3x8_f16(rh.x, rh.y));
    a[3] = __builtin_bit_cast(u32x4, e4m3x8_f16(rh.z, rh.w));
    rl = ld_lo(0, 1);
    rw[0] = ld_w(SL, 0);
    rs = ld_s(SL, 0);
    __builtin_amdgcn_s_waitcnt(0xC07F);                          // K-tile 0's weights are read: slot 0 takes K-tile 3's
    asm volatile("s_barrier" ::: "memory");
    issue_a(2, 2 * SL);
    issue_w(3, 0);

    // One K-tile kt (slot c0; c1, c2 hold kt + 1, kt + 2) from the widened weights bc and b3. Row tile i's 16 MFMAs run
    // step by step (p / 4) over the 4 column tiles, and each carries one conversion pair of row tile i + 1's activations
    // and one of the next K-tile's column tile i, four MFMAs behind, so that activations and column tile 3 replace their
    // predecessors in the same registers right after their last use (step 3 of each in the next row tile's first four).
    // In row tile 2 a barrier publishes the activations of kt + 1 and the weights of kt + 2 (issued a K-tile ago; the 7
    // loads after them stay in flight); every wave has read the activations of kt and the weights of kt + 1 by then, so
    // their slots take those of kt + 3 and kt + 4.
    auto step = [&](int kt, uint32_t c0, uint32_t c1, uint32_t c2, PvW (&bc)[3], PvW (&bn)[3]) {
  #pragma unroll
      for (int i = 0; i < 4; i++) {
  #pragma unroll
        for (int p = 0; p < 16; p++) {
          if (i == 2 && p == 8) {
            __builtin_amdgcn_s_waitcnt(0xC07F);
            asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(PV_DMA) : "memory");
            issue_a(kt + 3, c0);
            issue_w(kt + 4, c1);
          }
          const int t = p >> 2, j = p & 3;
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              __builtin_bit_cast(h8, a[t]), __builtin_bit_cast(h8, (j < 3 ? bc[j] : b3).k[t]), acc[i][j], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (p == 4) {
            gs = scales_f16(rs);
            rh = i < 3 ? ld_hi(c0, i + 1) : ld_hi(c1, 0);
            rw[(i + 1) & 1] = i < 3 ? ld_w(c1, i + 1) : ld_w(c2, 0);
            rs = i < 3 ? ld_s(c1, i + 1) : ld_s(c2, 0);
          }
          if (p == 12) rl = i < 2 ? ld_lo(c0, i + 2) : ld_lo(c1, i - 2);
          const int u = p >= 4 ? t - 1 : 3;                      // the step converted here
          const int jc = p >= 4 ? i : (i + 3) & 3;               // and its column tile (i == 0: of this K-tile)
          const uint32_t av = u < 2 ? rl[2 * u + (j >> 1)] : rh[2 * u + (j >> 1) - 4];
          const h2 pa = j & 1 ? __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)av, 1.0f, true)
                              : __builtin_amdgcn_cvt_scalef32_pk_f16_fp8((int)av, 1.0f, false);
          a[u][j] = __builtin_bit_cast(uint32_t, pa);
          const h2 pw = e2m1x2_f16(rw[jc & 1][u], j) * (h2){gs[u >> 1], gs[u >> 1]};
          (jc < 3 ? bn[jc] : b3).k[u][j] = __builtin_bit_cast(uint32_t, pw);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    uint32_t c0 = 0, c1 = SL, c2 = 2 * SL;
    int kt = 0;
    for (; kt + 1 < nkt; kt += 2) {
      step(kt, c0, c1, c2, B[0], B[1]);
      step(kt + 1, c1, c2, c0, B[1], B[0]);
      const uint32_t x = c0;
      c0 = c2;
      c2 = c1;
      c1 = x;
    }
    if (kt < nkt) step(kt, c0, c1, c2, B[0], B[1]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // no DMA may outlive the workgroup's LDS
  } else {
    // few K-tiles: two ahead in the ring, each widened ahead of its MFMAs, nothing loaded past the last
    issue_a(0, 0);
    issue_w(0, 0);
    if (nkt > 1) {
      issue_a(1, SL);
      issue_w(1, SL);
    }
    uint32_t sl = 0;
    for (int kt = 0; kt < nkt; kt++) {
      if (kt + 1 < nkt) asm volatile("s_waitcnt vmcnt(%0)" ::"i"(PV_DMA) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (kt + 2 < nkt) {                                      // into the slot read in the iteration before
        const uint32_t s2 = sl == 0 ? 2 * SL : sl - SL;
        issue_a(kt + 2, s2);
        issue_w(kt + 2, s2);
      }
      h8 b[4][4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const u32x4 bw = ld_w(sl, j);
        const h2 gs = scales_f16(ld_s(sl, j));
#pragma unroll
        for (int t = 0; t < 4; t++) b[j][t] = e2m1x8_f16(bw[t], gs[t >> 1]);
      }
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const u32x4 lo = ld_lo(sl, i), hi = ld_hi(sl, i);
        const h8 a[4] = {e4m3x8_f16(lo.x, lo.y), e4m3x8_f16(lo.z, lo.w), e4m3x8_f16(hi.x, hi.y),
                         e4m3x8_f16(hi.z, hi.w)};
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
          for (int t = 0; t < 4; t++)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t], b[j][t], acc[i][j], 0, 0, 0);
      }
      sl = sl == 2 * SL ? 0 : sl + SL;
    }
  }

  // epilogue: lane holds column c of each column tile, rows 4g .. 4g + 3 of each row tile; out = bf16(v * ((Wg[n] *
  // As[row]) * topk_w[row])), the row factors from LDS and the lane's 4 column multipliers loaded together. Branch-free:
  // every lane issues its 64 two-byte stores through a raw buffer of numel * N * 2 bytes (the host keeps it below
  // 2 GiB), a padding row or a column past N going to offset `cbytes`, which the range check drops -- no store waits
  // behind another.
  float wgv[4];
#pragma unroll
  for (int j = 0; j < 4; j++) wgv[j] = Ge[min((nt0 + wn * 4 + j) * 16 + c, N - 1)];
  const uint32_t cbytes = (uint32_t)numel * (uint32_t)N * 2u;
  const auto crs = __builtin_amdgcn_make_buffer_rsrc(C, (short)0, (int)cbytes, 0x00020000);
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int row = (wm * 4 + i) * 16 + 4 * g + q;
      const int fr = s_fr[row];
      const bool live = fr >= 0 && fr < numel;
      const float ras = s_as[row], rtw = s_tw[row];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int n = (nt0 + wn * 4 + j) * 16 + c;
        float sc = wgv[j] * ras;
        if (topk_w) sc *= rtw;
        const uint16_t v = (uint16_t)(pack_bf16x2(acc[i][j][q] * sc, 0.f) & 0xffffu);
        const uint32_t off = (live && n < N) ? ((uint32_t)fr * (uint32_t)N + (uint32_t)n) * 2u : cbytes;
        __builtin_amdgcn_raw_buffer_store_b16(v, crs, (int)off, 0, 0);
      }
    }
}

// ------------------------------------------------------------------- dense linear at decode widths, one launch
// The native NVFP4 dense linear for M <= 2 rows with the per-row fp8 activation quant inside the GEMM launch: every
// workgroup quantises the rows into LDS (r9k_rowquant.h: quant_rows_fp8's bytes), then runs moe_nvfp4_kernel's
// weight stream for one routing block of identity rows -- its widening, MFMA order, K split over SK waves and partial-
// tile sum -- so the output equals r9k_quant_rows_fp8 + r9k_moe_nvfp4a8 over identity tables bit for bit. The weight
// loads of the wave's first batch go out before the quant, whose latency they overlap.
constexpr int NQ_APAD = 16;       // bytes of padding per LDS code row

template <int NPW, int SK, int U, int MG>
__global__ void __launch_bounds__(WAVE * SK) dense_nvfp4_qa_kernel(
    const uint16_t* __restrict__ x, long ldx, const uint8_t* __restrict__ Wq, const uint8_t* __restrict__ Ws,
    const float* __restrict__ Wg, uint16_t* __restrict__ out, long ldo, int M, int N, int K) {
  extern __shared__ __align__(16) uint8_t lds[];
  const int lda = K + NQ_APAD;
  uint8_t* A = lds;
  float* s_row = reinterpret_cast<float*>(lds + (size_t)M * lda);
  float* red = s_row + 16;
  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid % WAVE;
  const int g = lane >> 4, c = lane & 15;
  const int NT = N / 16, nkt = K / NV_KT;

  const uint8_t* wtile[NPW];
  const uint8_t* stile[NPW];
#pragma unroll
  for (int j = 0; j < NPW; j++) {
    const int nt = min((int)blockIdx.x * NPW + j, NT - 1);     // a tile past N computes a copy, never stored
    wtile[j] = Wq + (size_t)nt * nkt * 1024 + lane * 16;
    stile[j] = Ws + (size_t)nt * nkt * 128 + lane * 2;
  }
  const int kt0 = wave * nkt / SK, kt1 = (wave + 1) * nkt / SK;

  u32x4 bw[U][NPW];
  uint32_t sw[U][NPW];
  auto issue = [&](int kt) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = min(kt + u, kt1 - 1);
#pragma unroll
      for (int j = 0; j < NPW; j++) {
        bw[u][j] = ld16_nt(wtile[j] + (size_t)k * 1024);
        sw[u][j] = ld2_nt(stile[j] + (size_t)k * 128);
      }
    }
  };
  {
    constexpr int T = WAVE * SK, XC = row_chunks<T>();
    const int nvec = K / 8;
    uint4 xv[MG][XC];
    load_row_group<T, MG, XC>(x, ldx, 0, M, nvec, tid, xv);
    issue(kt0);
    quant_row_group<T, MG, XC>(xv, 0, M, nvec, A, lda, s_row, red, tid);
  }

  v4f acc[NPW];
#pragma unroll
  for (int j = 0; j < NPW; j++) acc[j] = (v4f){0.f, 0.f, 0.f, 0.f};
  const bool arow = c < M;
  const uint8_t* ar = A + (size_t)(arow ? c : 0) * lda + 32 * g;   // lane group g: K values 32 g .. + 31 of a tile
  for (int kt = kt0; kt < kt1; kt += U) {
    if (kt != kt0) issue(kt);
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int k = kt + u;
      if (k < kt1) {                                         // wave-uniform
        uint4 l = *reinterpret_cast<const uint4*>(ar + k * NV_KT);
        uint4 h = *reinterpret_cast<const uint4*>(ar + k * NV_KT + 16);
        if (!arow) l = h = make_uint4(0u, 0u, 0u, 0u);
        const h8 a[4] = {e4m3x8_f16(l.x, l.y), e4m3x8_f16(l.z, l.w), e4m3x8_f16(h.x, h.y), e4m3x8_f16(h.z, h.w)};
#pragma unroll
        for (int j = 0; j < NPW; j++) {
          const h2 gs = scales_f16(sw[u][j]);
#pragma unroll
          for (int st = 0; st < 4; st++) {
            const h8 b = e2m1x8_f16(bw[u][j][st], gs[st >> 1]);
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[st], b, acc[j], 0, 0, 0);
          }
        }
      }
    }
  }

  // partial tiles through LDS (the quant's scratch is free again after its closing barrier), summed in wave order;
  // out = bf16(v * (Wg[n] * s[m])), moe_nvfp4_kernel's epilogue
#pragma unroll
  for (int j = 0; j < NPW; j++) {
    float* t = red + (size_t)(wave * NPW + j) * 256;
#pragma unroll
    for (int q = 0; q < 4; q++) t[(4 * g + q) * 16 + c] = acc[j][q];
  }
  __syncthreads();
  constexpr int TOT = NPW * 256;
  for (int idx = tid; idx < TOT; idx += WAVE * SK) {
    const int col = idx & 15, m = (idx >> 4) & 15, j = idx >> 8;
    const int n = (blockIdx.x * NPW + j) * 16 + col;
    if (m >= M || n >= N) continue;
    float v = 0.f;
#pragma unroll
    for (int s = 0; s < SK; s++) v += red[(size_t)s * TOT + idx];
    const float sc = Wg[n] * s_row[m];
    out[(size_t)m * ldo + n] = f2bf(v * sc);
  }
}

// ------------------------------------------------------------------- dense linear at decode widths, codes given
// The native NVFP4 dense linear for M <= 16 rows already quantised: moe_nvfp4_kernel's weight stream for one routing
// block of identity rows without the tables -- the same widening, MFMA order, K split over SK waves and partial-tile
// sum, so the same bits. Bound by the weight bytes and the widening's issue slots. Against that kernel over identity
// tables it starts its weight loads with its first instructions (no ntpp -> expert -> row id chain before them) and
// refills a K-tile's registers as soon as the tile is widened instead of draining a batch before the next. One
// column tile a workgroup and two K-tiles in flight a wave: 80 registers, six waves a SIMD, which hide more than a
// deeper ring on fewer waves (MI355X, GEMM alone, [17408, 5120] at M = 4: 14.2 us; 3 tiles 15.2, 4 15.2, 5 15.5, 10
// 16.1). Decode kernel -> this one, us: [17408, 5120] M = 4 / 8 / 16 16.1 / 17.9 / 20.3 -> 14.2 / 15.0 / 18.3,
// [5120, 17408] 22.4 / 23.5 / 27.0 -> 19.2 / 18.9 / 21.9, [4096, 4096] 7.3 / 7.5 / 10.4 -> 6.6 / 6.5 / 7.0, [1024,
// 2048] 6.0 / 6.1 / 6.5 -> 4.6 / 4.7 / 4.9.
template <int SK>
__global__ void __launch_bounds__(WAVE * SK) dense_nvfp4_a8_kernel(
    const uint8_t* __restrict__ A, long lda, const float* __restrict__ As, const uint8_t* __restrict__ Wq,
    const uint8_t* __restrict__ Ws, const float* __restrict__ Wg, uint16_t* __restrict__ out, long ldo, int M, int K) {
  constexpr int U = 2;                                          // K-tiles in flight a wave
  __shared__ float red[SK * 256];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  const int g = lane >> 4, c = lane & 15;
  const int nt = blockIdx.x, nkt = K / NV_KT;
  const uint8_t* wtile = Wq + (size_t)nt * nkt * 1024 + lane * 16;
  const uint8_t* stile = Ws + (size_t)nt * nkt * 128 + lane * 2;
  const uint8_t* arow = A + (size_t)min(c, M - 1) * lda + 32 * g;   // rows past M compute a copy, never stored
  const int kt0 = wave * nkt / SK, kt1 = (wave + 1) * nkt / SK;

  u32x4 bw[U];
  uint32_t sw[U];
  uint4 lo[U], hi[U];
  auto issue = [&](int u, int k) {
    bw[u] = ld16_nt(wtile + (size_t)k * 1024);
    sw[u] = ld2_nt(stile + (size_t)k * 128);
    lo[u] = *reinterpret_cast<const uint4*>(arow + (size_t)k * NV_KT);
    hi[u] = *reinterpret_cast<const uint4*>(arow + (size_t)k * NV_KT + 16);
  };
#pragma unroll
  for (int u = 0; u < U; u++) issue(u, min(kt0 + u, nkt - 1));
  // this thread's outputs: column tid % 16 of the tile, row tid / 16 and on
  const int n = nt * 16 + (tid & 15);
  const float wgn = Wg[n];

  v4f acc = (v4f){0.f, 0.f, 0.f, 0.f};
  for (int kt = kt0; kt < kt1; kt += U) {
#pragma unroll
    for (int u = 0; u < U; u++) {
      if (kt + u < kt1) {                                    // wave-uniform
        const h8 a[4] = {e4m3x8_f16(lo[u].x, lo[u].y), e4m3x8_f16(lo[u].z, lo[u].w), e4m3x8_f16(hi[u].x, hi[u].y),
                         e4m3x8_f16(hi[u].z, hi[u].w)};
        const h2 gs = scales_f16(sw[u]);
        h8 b[4];
#pragma unroll
        for (int st = 0; st < 4; st++) b[st] = e2m1x8_f16(bw[u][st], gs[st >> 1]);
        if (kt + u + U < kt1) issue(u, kt + u + U);
#pragma unroll
        for (int st = 0; st < 4; st++) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[st], b[st], acc, 0, 0, 0);
      }
    }
  }

#pragma unroll
  for (int q = 0; q < 4; q++) red[wave * 256 + (4 * g + q) * 16 + c] = acc[q];
  __syncthreads();
  for (int m = tid >> 4; m < M; m += WAVE * SK / 16) {
    float v = 0.f;
#pragma unroll
    for (int s = 0; s < SK; s++) v += red[s * 256 + m * 16 + (tid & 15)];
    const float sc = wgn * As[m];
    out[(size_t)m * ldo + n] = f2bf(v * sc);
  }
}

}  // namespace

// The prefill entry's native-NVFP4 case (r9k_moe_4bit_prefill with nv = 1; reference kernels/r9k_moe_mxfp4a8.hip:
// 1205-1230): routing blocks of blk = 128 or 256 rows, weights as r9k_moe_nvfp4a8 takes them. 0 / -7 blk / -3 / -6.
int r9k_nvfp4_prefill_launch(long a, long as, long wq, long ws, long wg, long c, long sorted_ids, long expert_ids,
                             long ntpp, long topk_w, long ws_estride, long wg_estride, int max_blocks, int numel,
                             int a_row_div, int K, int N, int blk, long stream) {
  if (blk != PV_BM && blk != 2 * PV_BM) return -7;
  if (max_blocks <= 0 || numel <= 0) return 0;
  if (!a || !as || !wq || !ws || !wg || !c || !sorted_ids || !expert_ids || !ntpp || a_row_div < 1) return -3;
  const int subs = blk / PV_BM;
  const long ny = (long)max_blocks * subs;
  if (ny > 0x7fffffffL) return -3;
  const dim3 grid((N + PV_BN - 1) / PV_BN, (unsigned)ny);
  const long wq_estride = (long)N * ((K + NV_KT - 1) / NV_KT) * 64;
  // the DMA addresses activations and one expert's codes through 32-bit offsets
  if ((long)((numel + a_row_div - 1) / a_row_div) * K >= (1L << 32) || wq_estride >= (1L << 32)) return -3;
  if ((long)numel * N * 2 >= (1L << 31)) return -3;             // the epilogue's raw output buffer
  // The software pipeline loads three K-tiles past the last and pays a prologue. Up to two K-tiles that costs more than
  // it hides ([16384, 256] at 128 / 1024 / 4096 rows 7.50 / 19.6 / 60.9 us plain, 7.65 / 20.9 / 65.9 pipelined), and up to
  // four where the tiles fill the chip twice over, whose other workgroups hide the widening (512 K: [16384] at 4096 rows
  // 85.6 / 87.5, 288 experts x 2048 at 128 rows each 161 / 170; with fewer tiles [4096] at 1024 rows 10.7 / 10.4). From
  // five on the pipeline wins or is even up to ~100M outputs ([4096, 1024] at 1024 rows 15.3 / 14.4).
  const int nkt = (K + NV_KT - 1) / NV_KT;
  const bool pipe = nkt > 4 || (nkt > 2 && (long)grid.x * ny < 1024);
  static const hipError_t attr[2] = {
      hipFuncSetAttribute(reinterpret_cast<const void*>(nvfp4_prefill_kernel<false>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)PV_SMEM),
      hipFuncSetAttribute(reinterpret_cast<const void*>(nvfp4_prefill_kernel<true>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)PV_SMEM)};
  if (attr[pipe] != hipSuccess) return -6;
  hipLaunchKernelGGL(pipe ? nvfp4_prefill_kernel<true> : nvfp4_prefill_kernel<false>, grid, dim3(PV_THREADS), PV_SMEM,
                     (hipStream_t)stream, (const uint8_t*)a, (const float*)as, (const uint8_t*)wq, (const uint8_t*)ws,
                     (const float*)wg, (uint16_t*)c, (const int*)sorted_ids, (const int*)expert_ids,
                     (const int*)ntpp, (const float*)topk_w, wq_estride, ws_estride, wg_estride, numel, a_row_div, K, N,
                     blk, subs);
  return hipGetLastError() == hipSuccess ? 0 : -6;
}

// Reference: kernels/r9k_moe_mxfp4a8.hip:641-647 (r9k_moe_nvfp4a8): same arguments and routing contract. ws / wg as
// the layout above (ws_estride bytes, wg_estride floats per expert); the code stride is N * ceil(K / 128) * 64 bytes
// (N * K / 2 when K % 128 == 0). WV and NPW are the reference's gfx1201 knobs and are not used; SK must divide K / 16
// as there (K % (16 SK) == 0). MT 1 / 2 / 4 rows tiles of 16 (the reference's bit 3 LDS-A flag is ignored).
// 0, or -1 N % 16, -2 K % (16 SK) or K % 16, -3 bad pointer / argument, -7 MT, -6 launch error.
extern "C" int r9k_moe_nvfp4a8(long a, long as, long wq, long ws, long wg, long c, long sorted_ids, long expert_ids,
                               long ntpp, long topk_w, long ws_estride, long wg_estride, int max_blocks, int numel,
                               int a_row_div, int K, int N, int WV, int SK, int NPW, int MT, long stream) {
  (void)WV;
  (void)NPW;
  MT &= 7;
  if (N % 16 || N <= 0) return -1;
  if (K % NV_G || K <= 0 || SK < 1 || K % (NV_G * SK)) return -2;
  if (MT != 1 && MT != 2 && MT != 4) return -7;
  if (a_row_div < 1) return -3;
  if (max_blocks <= 0 || numel <= 0) return 0;
  if (!a || !as || !wq || !ws || !wg || !c || !sorted_ids || !expert_ids || !ntpp) return -3;
  const int blk = 16 * MT;
  const NvPick p = nv_pick(N, K, max_blocks, numel, MT);
  const dim3 grid((N / 16 + p.NPW - 1) / p.NPW, (unsigned)max_blocks);
  const long wq_estride = (long)N * ((K + NV_KT - 1) / NV_KT) * 64;
  const hipStream_t st = (hipStream_t)stream;
#define NVL(MTv, NPWv, SKv, Uv)                                                                                   \
  if (MT == MTv && p.NPW == NPWv && p.SK == SKv && p.U == Uv) {                                                 \
    nv_launch<MTv, NPWv, SKv, Uv>(grid, st, a, as, wq, ws, wg, c, sorted_ids, expert_ids, ntpp, topk_w,          \
                                  wq_estride, ws_estride, wg_estride, numel, a_row_div, K, N, blk, 1);           \
    return hipGetLastError() == hipSuccess ? 0 : -6;                                                            \
  }
#define NVU(MTv, NPWv, SKv) NVL(MTv, NPWv, SKv, 1) NVL(MTv, NPWv, SKv, 2) NVL(MTv, NPWv, SKv, 4)
#define NVS(MTv, NPWv) NVU(MTv, NPWv, 1) NVU(MTv, NPWv, 2) NVU(MTv, NPWv, 4)
  NVS(1, 1) NVS(1, 2) NVS(2, 1) NVS(2, 2) NVS(4, 1) NVS(4, 2)
  NVL(1, 2, 4, 5)
#undef NVS
#undef NVU
#undef NVL
  return -3;
}

// No counterpart as one entry in the reference: r9k_quant_rows_fp8 + r9k_moe_nvfp4a8 over identity tables (the native
// NVFP4 dense linear, r9700_vllm/ops.py:66-83) in one launch, for M <= 2 rows. x bf16 [M][K] (row stride ldx
// elements, rows 16-byte aligned); wq / ws / wg one expert in this kernel's layout (prepare_nvfp4_weights); out bf16
// [M][N] (row stride ldo). Served: 1 <= M <= 2, K % 128 == 0, K <= 8192, N % 16 == 0; 2 (nothing launched) otherwise.
// 0, -3 bad argument, -6 launch error. Bit-equal to the two launches (the decode kernel's launch shape for one block).
extern "C" int r9k_dense_nvfp4_qa(long x, long ldx, long wq, long ws, long wg, long out, long ldo, int M, int N, int K,
                                  long stream) {
  if (M <= 0) return 0;
  if (!x || !wq || !ws || !wg || !out || N <= 0 || K <= 0) return -3;
  if (M > 2 || K % NV_KT || K > 8192 || N % 16 || (x & 15) || (ldx & 7) || (wq & 15)) return 2;
  const NvPick p = nv_pick(N, K, 1, M, 1);
  if (p.SK != 1 && p.SK != 4) return 2;
  const int T = WAVE * p.SK;
  if (K / 8 > (p.SK == 4 ? row_chunks<256>() : row_chunks<64>()) * T) return 2;
  // LDS: codes, 16 row scales, then the partial tiles (which also hold the quant's SK x M row maxima before them)
  const size_t smem = (size_t)M * (K + NQ_APAD) + 16 * sizeof(float) + (size_t)p.SK * p.NPW * 256 * sizeof(float);
  const dim3 grid((N / 16 + p.NPW - 1) / p.NPW), block(T);
  const hipStream_t st = (hipStream_t)stream;
  const int MG = M;
#define NQ(NPWv, SKv, Uv, MGv)                                                                                     \
  if (p.NPW == NPWv && p.SK == SKv && p.U == Uv && MG == MGv) {                                                    \
    hipLaunchKernelGGL((dense_nvfp4_qa_kernel<NPWv, SKv, Uv, MGv>), grid, block, smem, st, (const uint16_t*)x, ldx, \
                       (const uint8_t*)wq, (const uint8_t*)ws, (const float*)wg, (uint16_t*)out, ldo, M, N, K);      \
    return hipGetLastError() == hipSuccess ? 0 : -6;                                                               \
  }
#define NQM(NPWv, SKv, Uv) NQ(NPWv, SKv, Uv, 1) NQ(NPWv, SKv, Uv, 2)
#define NQU(NPWv, SKv) NQM(NPWv, SKv, 1) NQM(NPWv, SKv, 2) NQM(NPWv, SKv, 4)
  NQU(1, 1) NQU(2, 1) NQU(1, 4) NQU(2, 4)
#undef NQU
#undef NQM
#undef NQ
  return 2;
}

// No counterpart as one entry in the reference: the GEMM half of r9k_quant_rows_fp8 + r9k_moe_nvfp4a8 over identity
// tables (the native NVFP4 dense linear, r9700_vllm/ops.py:66-83) for 1 <= M <= 16 pre-quantised rows. q fp8 [M][K]
// (row stride ldq bytes, rows 16-byte aligned), s fp32 [M]; wq / ws / wg one expert in this kernel's layout; out bf16
// [M][N] (row stride ldo). Served: 1 <= M <= 16, K % 128 == 0, N % 16 == 0; 2 (nothing launched) otherwise. 0, -3 bad
// argument, -6 launch error. Same K split as r9k_moe_nvfp4a8 for one block, so the same bits.
extern "C" int r9k_dense_nvfp4_a8(long q, long ldq, long s, long wq, long ws, long wg, long out, long ldo, int M,
                                  int N, int K, long stream) {
  if (M <= 0) return 0;
  if (!q || !s || !wq || !ws || !wg || !out || N <= 0 || K <= 0) return -3;
  if (M > 16 || K % NV_KT || N % 16 || (q & 15) || (ldq & 15) || (wq & 15) || (ws & 1)) return 2;
  const int SK = nv_pick(N, K, 1, M, 1).SK;
  const dim3 grid(N / 16), block(WAVE * SK);
#define NA(SKv)                                                                                                     \
  hipLaunchKernelGGL((dense_nvfp4_a8_kernel<SKv>), grid, block, 0, (hipStream_t)stream, (const uint8_t*)q, ldq,     \
                     (const float*)s, (const uint8_t*)wq, (const uint8_t*)ws, (const float*)wg, (uint16_t*)out, ldo, \
                     M, K)
  if (SK == 1) NA(1);
  else if (SK == 2) NA(2);
  else NA(4);
#undef NA
  return hipGetLastError() == hipSuccess ? 0 : -6;
}
