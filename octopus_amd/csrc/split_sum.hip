// The sum of a split-K product's partial tiles (StoreArgs::split): C = rs[row] x sum over the runs (+ addend) (+ C),
// rounded once to C's type.
//
// Bound by memory: S partial tiles of 256 KB read per tile of C. One workgroup per 16 rows of a tile, 256 threads: each
// wave reads its accumulator blocks in the order the GEMM's wave left them (1 KB per load, the runs in order, so the
// sum is the same every time), and the 16 x 256 result goes through the LDS to be stored in whole rows. 225 rows at d
// 2560, V 151,936 (26 runs of 10 tiles, 68 MB): 16 us.
#include "gemm_nt.h"
#include "octo_internal.h"

namespace octo {

// NJ: 16-column blocks per wave, 4 waves across the tile (256 columns: 4; fp32 operands, 128 columns: 2). A
// lane's 4 values of a block are 4 columns of a row (Acc16T).
template <typename OT, int NJ>
__global__ __launch_bounds__(256) void split_sum_kernel(GemmShape s, StoreArgs e) {
  constexpr int NI = 8, NV = 4, TNX = 64 * NJ, WAVE = NI * NJ * NV * 64;
  constexpr int LDT = TNX + 4;  // floats per row of the LDS tile: rows 4 banks apart
  __shared__ __attribute__((aligned(16))) float tile[16 * LDT];
  int64_t mtiles, ntiles;
  bounded_tiles(s, mtiles, ntiles);
  const int64_t tiles = mtiles * ntiles, at = blockIdx.y;
  const int S = octo_tiles::k_splits((int)tiles, (int)cdiv(s.K, (int64_t)64), e.split_alone != 0, e.split_cap);
  if (S < 2 || at >= tiles) return;
  const int64_t nt = at / mtiles, mt = at - nt * mtiles, m0 = mt * TM, n0 = nt * TNX;
  int64_t mvalid = s.M - m0;
  const int64_t nvalid = min(s.N - n0, (int64_t)TNX);
  if (s.count_on == 1) mvalid = dev_count(s.count, s.count_off + m0, mvalid);
  const int wm = blockIdx.x >> 3, i = blockIdx.x & 7, row0 = wm * 128 + i * 16;
  if (row0 >= mvalid) return;

  const int lane = threadIdx.x & 63, wn = threadIdx.x >> 6;
  const f32x4 *p = (const f32x4 *)(e.split + at * (TM * TNX) + (wm * 4 + wn) * WAVE + i * (NJ * NV * 64)) + lane;
  f32x4 a[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) a[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int run = 0; run < S; ++run, p += tiles * (TM * TNX / 4)) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const f32x4 x = p[j * 64];
#pragma unroll
      for (int v = 0; v < NV; ++v) a[j][v] += x[v];
    }
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    *(f32x4 *)(tile + (lane & 15) * LDT + (wn * NJ + j) * 16 + 4 * (lane >> 4)) = a[j];
  __syncthreads();

  const int row = threadIdx.x >> 4;
  if (row0 + row >= mvalid) return;
  const int64_t r = m0 + row0 + row;
  const float sc = e.row_scale ? e.row_scale[r] : 1.f;
  OT *C = (OT *)e.C + r * e.ldc + n0;
  const float *add = e.addend ? e.addend + r * e.ld_add + n0 : nullptr;
  typedef OT OT4 __attribute__((ext_vector_type(4)));
  const bool whole = (uintptr_t)e.C % sizeof(OT4) == 0 && e.ldc % 4 == 0;  // 4 values of C in one store
#pragma unroll
  for (int q = 0; q < NJ; ++q) {
    const int c0 = q * 64 + (threadIdx.x & 15) * 4;
    if (c0 >= nvalid) continue;
    const f32x4 t = *(const f32x4 *)(tile + row * LDT + c0);
    float x[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      x[u] = t[u] * sc;
      if (c0 + u < nvalid) {
        if (add) x[u] += add[c0 + u];
        if (e.accumulate) x[u] += (float)C[c0 + u];
      }
    }
    if (whole && c0 + 4 <= nvalid) {
      OT4 o;
#pragma unroll
      for (int u = 0; u < 4; ++u) o[u] = (OT)x[u];
      *(OT4 *)(C + c0) = o;
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (c0 + u < nvalid) C[c0 + u] = (OT)x[u];
    }
  }
}

template <int NJ>
static int go_split_sum(GemmShape s, const StoreArgs &e, hipStream_t st) {
  s.ntiles = (int)cdiv(s.N, (int64_t)(64 * NJ));
  // the most tiles that any device count would split (mostly they are not: the launch then ends at once)
  const int nk = (int)cdiv(s.K, (int64_t)64);
  int64_t tiles = 0;
  for (int64_t m = 1; m <= s.mtiles && m * s.ntiles < e.split_cap; ++m)
    if (octo_tiles::k_splits((int)(m * s.ntiles), nk, e.split_alone != 0, e.split_cap) > 1) tiles = m * s.ntiles;
  if (tiles == 0) return OCTO_OK;
  const dim3 grid(16, (unsigned)tiles);
  switch (e.dtype) {
    case OCTO_BF16: hipLaunchKernelGGL((split_sum_kernel<__bf16, NJ>), grid, dim3(256), 0, st, s, e); break;
    case OCTO_F16: hipLaunchKernelGGL((split_sum_kernel<_Float16, NJ>), grid, dim3(256), 0, st, s, e); break;
    case OCTO_F32: hipLaunchKernelGGL((split_sum_kernel<float, NJ>), grid, dim3(256), 0, st, s, e); break;
    default: return octo_fail(OCTO_EUNSUPPORTED, "split_sum: output dtype %d", e.dtype);
  }
  OCTO_CHECK_LAUNCH("split_sum");
  return OCTO_OK;
}

int launch_split_sum(const GemmShape &s, const StoreArgs &e, bool f32, hipStream_t st) {
  if (!e.split) return OCTO_OK;
  return f32 ? go_split_sum<2>(s, e, st) : go_split_sum<4>(s, e, st);
}

}  // namespace octo
