// r9k_prep.hip -- checkpoint MXFP4 weights to the gfx950 kernels' layout (kernels/moe.py permute_fragments / pack_scales),
// one launch for the codes, the exponents and the per-row maxima.
//
// A workgroup owns one 16-row column tile of one expert. Codes: output piece p (16 bytes) of the tile is K-tile p / 64,
// lane p % 64 = 16 g + r, and comes from row r's 16 checkpoint bytes at 64 (p / 64) + 16 g (a partial last K-tile keeps
// its first 16 G lanes, the same formula). Exponents: output byte q is K-tile q / 64, lane q % 64, from row r's byte
// 4 (q / 64) + g; the row maximum goes behind the expert's exponents.
// Bound: HBM, every byte read once and written once. Reads touch 64 contiguous bytes of 16 rows an instruction and the
// next K-tile the neighbouring 64, writes are linear; PREP_U pieces a thread are in flight. It replaces four torch
// launches (two strided copies, a maximum over the last dimension and a copy): [17408, 5120] 105 us -> 17.4 us (5.4
// TB/s of its 94.7 MB).
#include "r9k_common.h"

namespace {

using namespace r9k;

constexpr int PREP_T = 256, PREP_U = 5;

__global__ void __launch_bounds__(PREP_T) mxfp4_prep_kernel(const uint8_t* __restrict__ packed,
                                                            const uint8_t* __restrict__ scale,
                                                            uint8_t* __restrict__ wq, uint8_t* __restrict__ ws, int N,
                                                            int K) {
  const int nt = blockIdx.x, tid = threadIdx.x;
  const long e = blockIdx.y;
  const int KB = K / 32;
  if (packed) {
    const uint8_t* src = packed + ((e * N + nt * 16L) * (K / 2));
    uint4* dst = reinterpret_cast<uint4*>(wq + ((e * N + nt * 16L) * (K / 2)));
    const int np = K / 2;                                    // pieces of the tile: 16 rows x K/2 bytes / 16
    for (int p0 = tid; p0 < np; p0 += PREP_T * PREP_U) {
      uint4 v[PREP_U];
#pragma unroll
      for (int u = 0; u < PREP_U; u++) {
        const int p = min(p0 + u * PREP_T, np - 1);
        v[u] = *reinterpret_cast<const uint4*>(src + (size_t)(p & 15) * (K / 2) + (p >> 6) * 64 + ((p >> 4) & 3) * 16);
      }
#pragma unroll
      for (int u = 0; u < PREP_U; u++)
        if (p0 + u * PREP_T < np) dst[p0 + u * PREP_T] = v[u];
    }
  }
  if (scale) {
    const uint8_t* src = scale + (e * N + nt * 16L) * KB;
    uint8_t* exp = ws + e * (long)(KB + 1) * N;
    uint32_t* dst = reinterpret_cast<uint32_t*>(exp + (long)nt * 16 * KB);
    for (int q = tid; q < 4 * KB; q += PREP_T) {             // 4 output bytes: rows r0 .. r0 + 3 of one 32-block
      const int r0 = (q & 3) * 4, kb = q >> 2;               // byte 4 q = (kb / 4) * 64 + (kb % 4) * 16 + r0
      uint32_t w = 0u;
#pragma unroll
      for (int j = 0; j < 4; j++) w |= (uint32_t)src[(r0 + j) * KB + kb] << (8 * j);
      dst[q] = w;
    }
    const int row = tid >> 4;                                // 16 lanes a row
    uint32_t m = 0u;
    for (int kb = tid & 15; kb < KB; kb += 16) m = max(m, (uint32_t)src[row * KB + kb]);
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, o, 16));
    if ((tid & 15) == 0) exp[(long)KB * N + nt * 16 + row] = (uint8_t)m;
  }
}

}  // namespace

// New entry point (no reference C symbol: the reference lays its weights out with torch, r9700_vllm/kernels/moe.py).
// packed [E, N, K/2] u8 -> wq (E * N * K/2 bytes, fragment order), scale [E, N, K/32] u8 -> ws [E, K/32 + 1, N] u8; all
// contiguous, wq not overlapping packed. Either half is left out when its source is 0. Codes 16-byte aligned, ws 4-byte.
// 0 / -1 N % 16 / -2 K % 32 / -3 bad pointer or count / -6 launch error.
extern "C" int r9k_mxfp4_prep(long packed, long scale, long wq, long ws, int E, int N, int K, long stream) {
  if (E <= 0 || N == 0) return 0;
  if (N < 0 || N % 16) return -1;
  if (K <= 0 || K % 32) return -2;
  if (!packed && !scale) return 0;
  if ((packed && (!wq || (packed & 15) || (wq & 15))) || (scale && (!ws || (ws & 3))) || E > 65535) return -3;
  hipLaunchKernelGGL(mxfp4_prep_kernel, dim3(N / 16, E), dim3(PREP_T), 0, (hipStream_t)stream, (const uint8_t*)packed,
                     (const uint8_t*)scale, (uint8_t*)wq, (uint8_t*)ws, N, K);
  return hipGetLastError() == hipSuccess ? 0 : -6;
}
