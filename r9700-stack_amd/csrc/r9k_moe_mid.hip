// r9k_moe_mid.hip -- grouped MXFP4 x fp8 GEMM over 64- and 128-row routing blocks on gfx950: the widths between the
// decode kernel's few rows and the 256-row prefill kernel, and the routed shapes whose K that kernel does not take.
//
// Same contract as the other grouped GEMMs (r9k_moe_gemm.hip, r9k_moe_prefill.hip): routed flat rows through the align
// tables, out[r, n] = bf16(acc * (As[r / a_row_div] * topk_w[r])) (reference kernels/r9k_moe_mxfp4a8.hip:469-482),
// the prepared weights' fragment order (1 KB per 16-column x 128-K tile, 64 exponent bytes), any K % 32 == 0.
//
// What bounds it: at these widths a routing block's weights are used for 16-128 rows, so the launch is a weight
// stream (HBM) with the activation rows re-read from L2 by every column block; a workgroup's steps are bounded by the
// global -> LDS path (64 bytes a clock a CU: 270 clocks for 64 x 128) and, beside it, by the waves' instruction count;
// from a few hundred rows by the MFMAs and by tiles that do not divide into whole rounds of the CUs. The decode kernel
// it replaces here read both operands into registers with no reuse across waves and nothing in flight during its MFMAs.
// Measured on MI355X, before -> after: routed gate_up [640, 2560] x 512 experts, top-10, 3001 tokens 243 -> 124 us, down
// [2560, 320] 244 -> 97 (220 MB of weights and 154 MB out: 3.9 TB/s); dense [17408, 5120] at 36 / 64 / 333 rows, weights
// cold in every cache, 24.5 / 37.7 / 126 -> 17.9 / 20.1 / 39 us, and 23.2 / 36 / 125 -> 14.9 / 15.4 / 33 with them in the
// 256 MB last-level cache (64 rows: 2.4 and 3.1 TB/s of weights; 333 rows: 1.5 and 1.8 PFLOP/s); dense [4096, 4096] at
// 1024 rows, from the 256-row kernel, 44 -> 20 us.
//
// Work split: a workgroup of 2 x WN waves (per K group) owns BM rows x BN columns, and walks `span` consecutive column
// blocks of its routing block. The (column block, 128-wide K chunk) steps run as one stream through a ring of NS LDS
// stages filled by direct global -> LDS DMA, NS - 1 steps ahead, across the column blocks' boundaries. Where the tiles
// fill the chip, two workgroups of 256 threads a CU (at most 80 KB of LDS each) cover each other's table reads and
// epilogues, except in the 256-column variant for short K: 512 threads and 83.75 KB, one a CU, where halving the
// activation re-reads is worth more. Where they do not, KS groups of waves in one workgroup split the K chunks and their
// partial sums meet in LDS, in group order. Each step every thread issues OPS DMA loads; an explicit vmcnt wait plus a
// barrier publishes the stage. The loop holds no compiler-tracked global load, so nothing else drains the ring, and each
// column block's ST output stores are counted in the waits of the steps after.
//
// Operands of V_MFMA_SCALE_F32_16X16X128_F8F6F4 (layout measured on gfx950, see r9k_moe_gemm.hip): the weights in the A
// slot (fp4, their e8m0 exponent as the A scale), the activations in the B slot (fp8, scale 2^0). A lane of the result
// then holds four consecutive columns of one row; the epilogue stages 16 rows x 32 columns through 1 KB of LDS a wave
// so that each store writes 64 contiguous bytes of 16 rows. One accumulator takes a group's K-tiles in ascending order.
#include "r9k_common.h"
#include "r9k_dma.h"

#include <algorithm>

namespace {

using namespace r9k;

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int KC = 128;                        // K per step
constexpr int NXCD = 8;
constexpr int E8M0_ONE = 127;

// MTW row tiles and CT column tiles (of 16) a wave, 2 x WN waves a K group, NS ring stages, KS groups splitting the K
// chunks.
template <int MTW, int CT, int WN, int NS, int KS>
struct Mid {
  static constexpr int BM = 32 * MTW, BN = 16 * CT * WN;
  static constexpr int NW = 2 * WN, GTH = WAVE * NW;           // waves and threads of a group
  static constexpr int MA = BM * 8 / GTH;                      // activation loads a thread and step
  static constexpr int A_BYTES = BM * KC;                      // 16-byte pieces, XOR-swizzled by row
  static constexpr int W_BYTES = BN / 16 * 1024;
  static constexpr int S_BYTES = (CT * WN / 4 + 1) * 256;      // a wave's 4 tiles are 256 bytes; the last 256 unused
  static constexpr int CHUNK = A_BYTES + W_BYTES + S_BYTES;    // one K chunk of one group
  static constexpr int STAGE = KS * CHUNK;
  static constexpr int OPS = MA + CT / 2 + 1;                  // DMA loads a thread and step
  static constexpr int ST = MTW * CT / 2;                      // output stores a wave and column block
  static constexpr size_t SMEM = (size_t)NS * STAGE + NW * 1024;
  static_assert(SMEM <= 160 * 1024 && NS >= 3 && MA >= 1, "LDS");
  static_assert(KS > 1 || NW > 4 || SMEM <= 80 * 1024, "two workgroups of 256 threads a CU");
  static_assert((KS - 1) * NW * MTW * CT * 1024 <= NS * STAGE, "partial sums fit the ring");
  static_assert((NS - 1) * OPS + ST < 64, "vmcnt");
};

// One step's operand fragments of a wave: CT weight fragments (fp4) with their exponent bytes, MTW activation
// fragments (fp8, low and high K halves).
template <int MTW, int CT>
struct Frag {
  u32x4 w[CT], lo[MTW], hi[MTW];
  int sb[CT];
};

template <int N>
__device__ __forceinline__ void wait_vm_barrier() {
  // lgkmcnt(0) through the builtin (0xC07F: no vmcnt, no expcnt), which the compiler's own wait tracking sees: the
  // fragments read before the barrier are then known to be there, and no wait is put in front of their MFMAs
  __builtin_amdgcn_s_waitcnt(0xC07F);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"(N) : "memory");
}

template <int MTW, int CT, int WN, int NS, int KS>
__global__ void __launch_bounds__(2 * WAVE * WN * KS, 2) moe_mid_kernel(
    const uint8_t* __restrict__ A, const float* __restrict__ As, const uint8_t* __restrict__ Wq,
    const uint8_t* __restrict__ Ws, uint16_t* __restrict__ C, const int* __restrict__ sorted_ids,
    const int* __restrict__ expert_ids, const int* __restrict__ ntpp, const float* __restrict__ topk_w,
    long wq_estride, long ws_estride, int numel, int a_row_div, int K, int N, int blk, int span, int grp) {
  using P = Mid<MTW, CT, WN, NS, KS>;
  extern __shared__ __align__(16) uint8_t smem[];

  // live tiles only; XCD x (dispatch goes round-robin over them) owns a contiguous range of the logical tiles, which
  // run in groups of grp routing blocks, column-major within a group: the blocks of one expert share its weights
  // through that XCD's L2, and the column blocks of a routing block its activation rows
  const int nnb = (N + P::BN - 1) / P::BN, nsp = (nnb + span - 1) / span;
  const int nblk = ntpp[0] / blk, total = nblk * nsp;
  const int L = blockIdx.x;
  if (L >= total) return;
  const int q = total / NXCD, rem = total % NXCD, x = L % NXCD;
  const int logical = x * q + min(x, rem) + L / NXCD;
  const int gi = logical / (grp * nsp), gr = logical - gi * grp * nsp, gb = min(grp, nblk - gi * grp);
  const int rb = gi * grp + gr % gb, nb0 = gr / gb * span, nb1 = min(nb0 + span, nnb);

  const int kg = __builtin_amdgcn_readfirstlane(threadIdx.x / P::GTH);
  const int tid = threadIdx.x % P::GTH, wave = __builtin_amdgcn_readfirstlane(tid / WAVE), lane = tid % WAVE;
  const int g = lane >> 4, r = lane & 15;
  const int wm = wave / WN, wn = wave % WN;
  const int* __restrict__ rows = sorted_ids + (size_t)rb * blk;
  // every table read goes out together (the block's BM entries are all inside the table), then the row scales
  const int e = expert_ids[rb], first = rows[0];
  int ida[P::MA], idr[MTW], ido[MTW], idl[(P::BM + WAVE - 1) / WAVE];
#pragma unroll
  for (int p = 0; p < P::MA; p++) ida[p] = rows[p * (P::GTH / 8) + (tid >> 3)];   // DMA source rows
#pragma unroll
  for (int i = 0; i < MTW; i++) {
    idr[i] = rows[wm * 16 * MTW + i * 16 + r];                 // this lane's accumulator rows
    ido[i] = rows[wm * 16 * MTW + i * 16 + (lane >> 2)];       // and the rows it stores
  }
  int nlive = 0;                                               // padding sits at the end of a block
#pragma unroll
  for (int u = 0; u < (P::BM + WAVE - 1) / WAVE; u++) idl[u] = rows[min(u * WAVE + lane, P::BM - 1)];
#pragma unroll
  for (int u = 0; u < (P::BM + WAVE - 1) / WAVE; u++)
    nlive += __popcll(__ballot(u * WAVE + lane < P::BM && idl[u] >= 0 && idl[u] < numel));
  if (e < 0 || nlive == 0 || first < 0 || first >= numel) return;
  auto a_row = [&](int fr) { return a_row_div == 1 ? fr : fr / a_row_div; };

  const int NTt = N / 16;
  const int nfull = K / KC, krem = K % KC, nchunk = nfull + (krem ? 1 : 0), nk = (nchunk + KS - 1) / KS;
  const uint8_t* We = uniform_ptr(Wq + (size_t)e * wq_estride);
  const uint8_t* Se = uniform_ptr(Ws + (size_t)e * ws_estride);

  // ---- DMA sources: 32-bit offsets from A, We and Se. A partial last K-tile re-reads valid bytes for its dead lanes
  // (their operands are zeroed after the LDS read).
  const int piece = (tid & 7) ^ ((tid >> 4) & 7);             // LDS slot tid & 7 of row tid >> 3
  uint32_t aoff[P::MA];
#pragma unroll
  for (int p = 0; p < P::MA; p++)
    aoff[p] = (uint32_t)a_row(p * (P::GTH / 8) + (tid >> 3) < nlive ? ida[p] : first) * (uint32_t)K;
  const uint32_t ap_full = piece * 16, ap_tail = piece * 16 < krem ? piece * 16 : 0;
  const uint32_t wl_full = lane * 16, wl_tail = (lane < krem / 2 ? lane : r) * 16;       // 16 * (krem / 32) live lanes
  const uint32_t sl_full = r * 4, sl_tail = r * 4 < krem / 2 ? r * 4 : 0;
  const uint32_t lds0 = lds_addr(smem + kg * P::CHUNK);
  const uint32_t la = lds0 + wave * 1024, lw = la + P::A_BYTES, ls = lds0 + P::A_BYTES + P::W_BYTES + min(wave, CT * WN / 4) * 256;

  // The step whose DMA goes out next: column block `in`, chunk index ic * KS + kg, its offsets from We, A and Se.
  int in = nb0, ic = 0;
  uint32_t wo[CT / 2], ao[P::MA], so;
  auto set_step = [&]() {
    const int c = min(ic * KS + kg, nchunk - 1);               // a group past K re-reads the last chunk
    const bool tail = c == nfull;
#pragma unroll
    for (int p = 0; p < CT / 2; p++)                           // columns past N compute a copy, never stored
      wo[p] = (uint32_t)min(in * (P::BN / 16) + p * P::NW + wave, NTt - 1) * (uint32_t)(8 * K) +
              (tail ? wl_tail : wl_full) + (uint32_t)c * 1024;
#pragma unroll
    for (int p = 0; p < P::MA; p++) ao[p] = aoff[p] + (tail ? ap_tail : ap_full) + (uint32_t)c * KC;
    so = (uint32_t)min(in * (P::BN / 16) + min(wave * 4 + g, P::BN / 16 - 1), NTt - 1) * (uint32_t)(K / 2) +
         (tail ? sl_tail : sl_full) + (uint32_t)c * 64;
  };
  auto next_step = [&]() {
    ic++;
    if (__builtin_expect(ic >= nk - 1, 0)) {                   // the last chunk (it may be partial), or a new column block
      if (ic == nk) {                                          // (past the last block: any valid one)
        ic = 0;
        in++;
      }
      set_step();
    } else {
#pragma unroll
      for (int p = 0; p < CT / 2; p++) wo[p] += KS * 1024;
#pragma unroll
      for (int p = 0; p < P::MA; p++) ao[p] += KS * KC;
      so += KS * 64;
    }
  };
  auto dma_op = [&](int k, uint32_t st) {                      // load k of the step's OPS, into the stage at st
    if (k < CT / 2) dma16s(We, wo[k], lw + st + k * P::GTH * 16);
    else if (k < CT / 2 + P::MA) dma16s(A, ao[k - CT / 2], la + st + (k - CT / 2) * P::GTH * 16);
    else dma4s(Se, so, ls + st);
  };

  // ---- this lane's rows: scale of row r of each row tile (its accumulators), output row of its stores
  float sc[MTW], tw[MTW];
  uint32_t trow[MTW];
#pragma unroll
  for (int i = 0; i < MTW; i++) {
    const int fr = wm * 16 * MTW + i * 16 + r < nlive ? idr[i] : first;
    sc[i] = As[a_row(fr)];
    tw[i] = topk_w ? topk_w[fr] : 1.f;
    trow[i] = wm * 16 * MTW + i * 16 + (lane >> 2) < nlive ? (uint32_t)ido[i] * (uint32_t)N : 0xffffffffu;
  }

  const int sw = r >> 1;
  const uint8_t* const base = smem + kg * P::CHUNK;            // fragment addresses in stage 0
  const uint8_t* const flo = base + (wm * 16 * MTW + r) * 128 + (g ^ sw) * 16;
  const uint8_t* const fhi = base + (wm * 16 * MTW + r) * 128 + ((4 + g) ^ sw) * 16;
  const uint8_t* const fw = base + P::A_BYTES + wn * CT * 1024 + lane * 16;
  const uint8_t* const fs = base + P::A_BYTES + P::W_BYTES + wn * CT * 64 + lane;
  uint8_t* ost = smem + NS * P::STAGE + wave * 1024;
  const uint32_t cbytes = (uint32_t)numel * (uint32_t)N * 2u;
  const auto crs = __builtin_amdgcn_make_buffer_rsrc(C, (short)0, (int)cbytes, 0x00020000);

  // read k of the RD that fetch this group's fragments of the stage at byte st
  auto read_op = [&](Frag<MTW, CT>& F, int k, int st) {
    if (k < CT) {
      F.w[k] = *reinterpret_cast<const u32x4*>(fw + st + k * 1024);
      F.sb[k] = fs[st + k * 64];
    } else {
      const int i = (k - CT) >> 1;
      if ((k - CT) & 1) F.hi[i] = *reinterpret_cast<const u32x4*>(fhi + st + i * 2048);
      else F.lo[i] = *reinterpret_cast<const u32x4*>(flo + st + i * 2048);
    }
  };

  const int nst = (nb1 - nb0) * nk;
  set_step();
#pragma unroll
  for (int s = 0; s < NS; s++) {
#pragma unroll
    for (int k = 0; k < P::OPS; k++) dma_op(k, (uint32_t)s * P::STAGE);
    next_step();
  }
#pragma unroll
  for (int i = 0; i < MTW; i++) {                              // the only compiler-tracked loads end here
    sc[i] *= tw[i];
    asm volatile("" ::"v"(sc[i]));
  }

  v4f acc[MTW][CT];
#pragma unroll
  for (int i = 0; i < MTW; i++)
#pragma unroll
    for (int j = 0; j < CT; j++) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};

  // Barrier t publishes stage t + 1 and, every wave's reads of stage t being complete there, frees stage t for the DMA
  // of step t + NS. The LDS reads of stage t + 1's fragments and those DMA loads are spread over step t's MFMAs. The
  // loop is unrolled so that every stage offset is a constant, and issues the same loads in every step (past the last
  // one they re-read valid bytes that nothing uses): with one or two waves a SIMD the step's instruction count is what
  // bounds it, so branches and address arithmetic are kept out of it.
  constexpr int RD = CT + 2 * MTW, NE = P::OPS + RD, NM = MTW * CT, UN = NS % 2 ? 2 * NS : NS;
  static_assert(RD >= P::OPS - 1, "the extras alternate");
  Frag<MTW, CT> F[2];
  wait_vm_barrier<(NS - 1) * P::OPS>();
#pragma unroll
  for (int k = 0; k < RD; k++) read_op(F[0], k, 0);

  int cn = nb0, cc = 0, t = 0, since = NS;                     // since: steps since the last epilogue's stores
  // one step from stage u's fragments `cur`; true after the last one
  auto step = [&](int u, Frag<MTW, CT>& cur, Frag<MTW, CT>& nxt) -> bool {
    const int st = u * P::STAGE, stn = (u + 1) % NS * P::STAGE;
    // DMA of step t + 1 done: younger are the DMA of steps t + 2 .. t + NS - 1 and the stores of an epilogue within the
    // last NS - 1 steps (one is counted; when there were more, the wait is only stricter)
    if (__builtin_expect(since < NS - 1, 0)) wait_vm_barrier<(NS - 2) * P::OPS + P::ST>();
    else wait_vm_barrier<(NS - 2) * P::OPS>();
    since++;
    const int c = cc * KS + kg;
    if (__builtin_expect(c >= nfull, 0)) {                     // a partial K-tile (or, of a group, none): zero past K
      const int kr = c == nfull ? krem : 0;
#pragma unroll
      for (int j = 0; j < CT; j++) {
        if (g * 32 >= kr) {
          cur.w[j] = (u32x4){0u, 0u, 0u, 0u};
          cur.sb[j] = E8M0_ONE;
        }
      }
#pragma unroll
      for (int i = 0; i < MTW; i++) {
        if (g * 16 >= kr) cur.lo[i] = (u32x4){0u, 0u, 0u, 0u};
        if (64 + g * 16 >= kr) cur.hi[i] = (u32x4){0u, 0u, 0u, 0u};
      }
    }
#pragma unroll
    for (int m = 0; m < NM; m++) {
      const int i = m / CT, j = m % CT;
      const v8i af = (v8i){(int)cur.lo[i].x, (int)cur.lo[i].y, (int)cur.lo[i].z, (int)cur.lo[i].w,
                           (int)cur.hi[i].x, (int)cur.hi[i].y, (int)cur.hi[i].z, (int)cur.hi[i].w};
      const v8i wf = (v8i){(int)cur.w[j].x, (int)cur.w[j].y, (int)cur.w[j].z, (int)cur.w[j].w, 0, 0, 0, 0};
      acc[i][j] =
          __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(wf, af, acc[i][j], 4, 0, 0, cur.sb[j], 0, E8M0_ONE);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = m * NE / NM; x < (m + 1) * NE / NM; x++) {
        if (x < 2 * P::OPS && (x & 1) == 0) dma_op(x >> 1, (uint32_t)st);
        else read_op(nxt, x < 2 * P::OPS ? x >> 1 : x - P::OPS, stn);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    next_step();
    if (__builtin_expect(++cc == nk, 0)) {
      if constexpr (KS > 1) {
        // the groups' partial sums meet in the ring (one column block a workgroup, every stage is read): group 0 adds
        // them in group order
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        v4f* part = reinterpret_cast<v4f*>(smem);
        if (kg > 0) {
#pragma unroll
          for (int i = 0; i < MTW; i++)
#pragma unroll
            for (int j = 0; j < CT; j++) part[((((kg - 1) * MTW + i) * CT + j) * P::NW + wave) * WAVE + lane] = acc[i][j];
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (kg > 0) return true;
#pragma unroll
        for (int k = 0; k < KS - 1; k++)
#pragma unroll
          for (int i = 0; i < MTW; i++)
#pragma unroll
            for (int j = 0; j < CT; j++) acc[i][j] += part[(((k * MTW + i) * CT + j) * P::NW + wave) * WAVE + lane];
      }
      // epilogue: lane (g, r) holds row r, columns 4 g .. 4 g + 3 of each 16 x 16 tile. Two column tiles of a row tile
      // go to the wave's 1 KB (16-byte piece q of row r at q ^ (r & 3)) and come back as 16 bytes of row lane / 4; a
      // wave's LDS operations execute in order. Rows past the live ones and columns past N store to the dropped offset.
      const int rr = lane >> 2, qq = lane & 3;
#pragma unroll
      for (int i = 0; i < MTW; i++)
#pragma unroll
        for (int jp = 0; jp < CT / 2; jp++) {
#pragma unroll
          for (int h = 0; h < 2; h++) {
            const v4f v = acc[i][2 * jp + h];
            const uint2 pk = make_uint2(pack_bf16x2(v[0] * sc[i], v[1] * sc[i]), pack_bf16x2(v[2] * sc[i], v[3] * sc[i]));
            *reinterpret_cast<uint2*>(ost + r * 64 + (((2 * h + (g >> 1)) ^ (r & 3)) * 16) + (g & 1) * 8) = pk;
            acc[i][2 * jp + h] = (v4f){0.f, 0.f, 0.f, 0.f};
          }
          const v4i w = *reinterpret_cast<const v4i*>(ost + rr * 64 + ((qq ^ (rr & 3)) * 16));
          const int col = cn * P::BN + (wn * CT + 2 * jp) * 16 + qq * 8;
          const uint32_t off = (trow[i] != 0xffffffffu && col < N) ? (trow[i] + (uint32_t)col) * 2u : cbytes;
          __builtin_amdgcn_raw_buffer_store_b128(w, crs, (int)off, 0, 0);
        }
      cc = 0;
      cn++;
      since = 0;
    }
    return ++t >= nst;
  };
  for (bool done = false; !done;) {
#pragma unroll
    for (int u = 0; u < UN; u++) {
      if (step(u % NS, F[u & 1], F[(u + 1) & 1])) {
        done = true;
        break;
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // no DMA may outlive the workgroup's LDS
}

template <int MTW, int CT, int WN, int NS, int KS>
int launch_mid(long a, long as, long wq, long ws, long c, long sorted_ids, long expert_ids, long ntpp, long topk_w,
               long ws_estride, int max_blocks, int numel, int a_row_div, int K, int N, int blk, int span, int grp,
               hipStream_t st) {
  using P = Mid<MTW, CT, WN, NS, KS>;
  static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(moe_mid_kernel<MTW, CT, WN, NS, KS>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)P::SMEM);
  if (attr != hipSuccess) return -4;
  const int nnb = (N + P::BN - 1) / P::BN;
  const long grid = (long)max_blocks * ((nnb + span - 1) / span);
  if (grid > 0x7fffffffL) return -3;
  hipLaunchKernelGGL((moe_mid_kernel<MTW, CT, WN, NS, KS>), dim3((unsigned)grid), dim3(P::GTH * KS), P::SMEM, st, (const uint8_t*)a,
                     (const float*)as, (const uint8_t*)wq, (const uint8_t*)ws, (uint16_t*)c, (const int*)sorted_ids,
                     (const int*)expert_ids, (const int*)ntpp, (const float*)topk_w, (long)N * K / 2, ws_estride,
                     numel, a_row_div, K, N, blk, span, grp);
  return hipGetLastError() == hipSuccess ? 0 : -6;
}

}  // namespace

// Internal entry of the prefill dispatch in r9k_moe_gemm.hip: tables with blocks of blk = 64 or 128 rows, K % 32 == 0.
// 2 (nothing launched): a shape for the register kernel -- addresses past the 32-bit offsets, or bases that are not
// 16-byte aligned.
int r9k_mid_launch(long a, long as, long wq, long ws, long c, long sorted_ids, long expert_ids, long ntpp, long topk_w,
                   long ws_estride, int max_blocks, int numel, int a_row_div, int K, int N, int blk, long stream) {
  if (blk != 64 && blk != 128) return 2;
  if (max_blocks <= 0 || numel <= 0) return 0;
  if (!a || !as || !wq || !ws || !c || !sorted_ids || !expert_ids || !ntpp || a_row_div < 1) return -3;
  if (((a | wq | c) & 15) || (ws & 3) || (ws_estride & 3)) return 2;
  const long a_rows = ((long)numel + a_row_div - 1) / a_row_div;
  if (a_rows * K >= (1L << 31) || (long)N * K / 2 >= (1L << 31) || (long)numel * N * 2 >= (1L << 31)) return 2;
  const hipStream_t st = (hipStream_t)stream;
  const int nchunk = (K + KC - 1) / KC;
  auto tiles = [&](int bn) { return (long)max_blocks * ((N + bn - 1) / bn); };
  // Column blocks a workgroup walks: about 16 steps of short K (the table reads and the first DMA round trip of a
  // workgroup are then paid once per 16 steps: E = 512, K = 320, N = 2560, 3001 tokens: 156 us with one column block a
  // workgroup, 107 with 5; K = 512, 288 experts, 2048 tokens: 77 against 57 with 4) and 32 of long K (K = 2048: 93 with
  // one, 82 with 2, 88 with 4; K = 2560: 124 with one, 131 with 3), as long as the launch keeps 1024 workgroups.
  auto span_of = [&](int steps, int bn) { return (int)std::max(1L, std::min((long)(steps / nchunk), tiles(bn) / 1024)); };
  // One expert's blocks only (a dense linear): groups of 8 blocks share a weight tile through an XCD's L2 ([17408,
  // 5120] on 128-row blocks, 2048 rows: 163 us ungrouped, 148 with 8, 154 with 16).
  const int grp = max_blocks == (numel + blk - 1) / blk ? 8 : 1;
#define R9K_MID(MTW, CT, WN, NS, KS, SPAN)                                                                          \
  return launch_mid<MTW, CT, WN, NS, KS>(a, as, wq, ws, c, sorted_ids, expert_ids, ntpp, topk_w, ws_estride,        \
                                         max_blocks, numel, a_row_div, K, N, blk, SPAN, grp, st)
  if (blk == 128) R9K_MID(4, 4, 2, 3, 1, span_of(32, 128));
  // 64-row blocks whose 64 x 64 or 64 x 128 tiles do not fill the CUs: two groups split K (4096 x 4096: 37 rows 12.9 ->
  // 9.9 us on 64 x 64 tiles; [17408, 5120]: 37 rows 16.1 -> 14.9 on 64 x 128, and up to 32 rows 13.1 on 32 x 128)
  if (numel <= 32 && tiles(128) <= 256) R9K_MID(1, 4, 2, 5, 2, 1);
  if (tiles(64) <= 256) R9K_MID(2, 2, 2, 3, 2, 1);
  if (tiles(128) <= 256) R9K_MID(2, 4, 2, 4, 2, 1);
  // short K (few steps a column block, the routed down products): 256 columns a workgroup re-read the block's
  // activations half as often (K = 320 above: 107 -> 97 us; K = 512: 57 -> 54; K = 2560 no faster, 124 against 131)
  if (nchunk <= 4 && N >= 1024) R9K_MID(2, 4, 4, 3, 1, span_of(16, 256));
  R9K_MID(2, 4, 2, 4, 1, span_of(nchunk <= 4 ? 16 : 32, 128));
#undef R9K_MID
}
