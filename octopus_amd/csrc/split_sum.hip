// The sum of a split-K product's partial tiles (StoreArgs::split): C = rs[row] x sum over the runs (+ addend) (+ C),
// rounded once to C's type.
//
// Bound by memory: S partial tiles of 256 KB read per tile of C. One workgroup per 16 rows of a tile, 256 threads: each
// wave reads its accumulator blocks in the order the GEMM's wave left them (256 contiguous bytes per load, the runs in
// order, so the sum is the same every time), and the 16 x 256 result goes through the LDS to be stored 4 values a
// thread along the rows. 225 rows at d 2560, V 151,936 (26 runs of 10 tiles, 68 MB): 16 us.
#include "gemm_nt.h"
#include "octo_internal.h"

namespace octo {

template <typename OT>
__global__ __launch_bounds__(256) void split_sum_kernel(GemmShape s, StoreArgs e) {
  typedef Acc16N<4> L;
  constexpr int LDT = 260;  // floats per row of the LDS tile: rows 4 banks apart
  __shared__ __attribute__((aligned(16))) float tile[16 * LDT];
  int64_t mtiles, ntiles;
  bounded_tiles(s, mtiles, ntiles);
  const int64_t tiles = mtiles * ntiles, at = blockIdx.y;
  const int S = octo_tiles::k_splits((int)tiles, (int)cdiv(s.K, (int64_t)64), e.split_alone != 0, e.split_cap);
  if (S < 2 || at >= tiles) return;
  const int64_t nt = at / mtiles, mt = at - nt * mtiles, m0 = mt * TM, n0 = nt * TN;
  int64_t mvalid = s.M - m0;
  const int64_t nvalid = min(s.N - n0, (int64_t)TN);
  if (s.count_on == 1) mvalid = dev_count(s.count, s.count_off + m0, mvalid);
  const int wm = blockIdx.x >> 3, i = blockIdx.x & 7, row0 = wm * 128 + i * 16;
  if (row0 >= mvalid) return;

  const int lane = threadIdx.x & 63, wn = threadIdx.x >> 6;
  const float *p = e.split + (at << 16) + (wm * L::NWN + wn) * (L::NI * L::NJ * L::NV * 64) + i * (L::NJ * L::NV * 64) + lane;
  float a[L::NJ * L::NV];
#pragma unroll
  for (int k = 0; k < L::NJ * L::NV; ++k) a[k] = 0.f;
#pragma unroll 2
  for (int run = 0; run < S; ++run, p += tiles << 16) {
#pragma unroll
    for (int k = 0; k < L::NJ * L::NV; ++k) a[k] += p[k * 64];
  }
#pragma unroll
  for (int j = 0; j < L::NJ; ++j)
#pragma unroll
    for (int v = 0; v < L::NV; ++v) tile[(4 * (lane >> 4) + v) * LDT + L::col(wn, j, lane)] = a[j * L::NV + v];
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
  for (int q = 0; q < 4; ++q) {
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

int launch_split_sum(const GemmShape &s, const StoreArgs &e, hipStream_t st) {
  if (!e.split) return OCTO_OK;
  // the most tiles that any device count would split (mostly they are not: the launch then ends at once)
  const int nk = (int)cdiv(s.K, (int64_t)64);
  int64_t tiles = 0;
  for (int64_t m = 1; m <= s.mtiles && m * s.ntiles < e.split_cap; ++m)
    if (octo_tiles::k_splits((int)(m * s.ntiles), nk, e.split_alone != 0, e.split_cap) > 1) tiles = m * s.ntiles;
  if (tiles == 0) return OCTO_OK;
  const dim3 grid(16, (unsigned)tiles);
  switch (e.dtype) {
    case OCTO_BF16: hipLaunchKernelGGL(split_sum_kernel<__bf16>, grid, dim3(256), 0, st, s, e); break;
    case OCTO_F16: hipLaunchKernelGGL(split_sum_kernel<_Float16>, grid, dim3(256), 0, st, s, e); break;
    case OCTO_F32: hipLaunchKernelGGL(split_sum_kernel<float>, grid, dim3(256), 0, st, s, e); break;
    default: return octo_fail(OCTO_EUNSUPPORTED, "split_sum: output dtype %d", e.dtype);
  }
  OCTO_CHECK_LAUNCH("split_sum");
  return OCTO_OK;
}

}  // namespace octo
