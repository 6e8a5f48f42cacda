// The fp32 GEMMs of the LM-head path on the bf16 matrix cores: each fp32 operand is the exact sum of three bf16 values
// (its 24 significand bits, 8 at a time; the method of Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial
// intelligence datatype for higher-precision computations", ARITH 2019), and a product is the six partial products that
// reach fp32's last bit,
//     a b = a0 b0 + a0 b1 + a1 b0 + a1 b1 + a0 b2 + a2 b0   (+ a1 b2 + a2 b1 + a2 b2, below 2^-23 |a b|),
// summed by v_mfma_f32_16x16x32_bf16 in fp32. The matrix cores' fp32 rate is 1/16 of their bf16 rate, so six bf16
// products are 2.6 times as fast. What is left out and one rounding per 32 products (against one per 2 with
// v_mfma_f32_32x32x2_f32) leave the sums no less exact, measured against 64 bits on [512, 32,000] logits of d 1024: the
// columns 6.4e-7 off (relative) against 7.9e-7, the gradients 8e-7 against 3.2e-6. Time there: the logits and their
// statistics 279 us with the fp32 instructions (120 TFLOP/s), 178 here (188 TFLOP/s in fp32 terms).
// An infinite operand, or one that bf16 rounds to infinity (from 3.39e38 on), has no such parts: no sum that it enters
// is finite. A wave that finds such a sum makes its part of the tile again by v_mfma_f32_16x16x4_f32 from the operands
// as they are (mainloop_plain), infinities and NaN where those products have them; to look for one takes no time that
// shows (those logits 182.2 us, 183.0 without). Below 2^-110 the third part loses bits.
//
// One workgroup computes a 256 x 128 tile of C[m, n] = sum_k A[m, k] B[n, k] with 8 waves, two per SIMD, 2 x 4 of 128 x
// 32 (AccX: the 16 x 16 block layout of the 16-bit kernels, 8 x 2 blocks). A stage is K = 32: 48 KB of fp32 go from
// global memory to registers one stage ahead, are split there, and land in the LDS as three bf16 planes per operand
// (72 KB a stage, two stages). Bound by the matrix cores: 96 MFMAs per wave and stage (1,536 cycles) against 24 values
// per thread to split (5.5 instructions each, and two for infinities). One wave of each SIMD splits the next
// stage before its MFMAs and the other after them, so that one's vector instructions run beside the other's MFMAs. A
// 256 x 256 tile would need 96 KB a stage: no room for the second.
//
// Two operand layouts, neither needing a transposed copy: XRows, K-contiguous rows (optionally through a row map),
// and XCols, K down the matrix rows (grad_h reads W and grad_W reads dz so): a thread loads 8 K-values of one column,
// a dword each, 64 neighbouring columns per instruction, and holds the same 8 consecutive K-values as for XRows.
#include "gemm_nt.h"
#include "octo_internal.h"

namespace octo {

constexpr int XM = 256, XN = 128, XK = 32;   // tile, and K per stage
constexpr int XROWB = XK * 2;                // bytes of a row of one plane
constexpr int XPA = XM * XROWB, XPB = XN * XROWB;
constexpr int XSTAGE = 3 * (XPA + XPB);      // 72 KB
constexpr int XTHREADS = 512;
static_assert(2 * XSTAGE <= 160 * 1024, "LDS budget");

struct AccX {
  static constexpr int NI = 8, NJ = 2, NV = 4, NWN = 4;
  typedef f32x4 V;
  static __device__ __forceinline__ int row(int wm, int i, int v, int lane) {
    return wm * 128 + i * 16 + 4 * (lane >> 4) + v;
  }
  static __device__ __forceinline__ int col(int wn, int j, int lane) { return wn * 32 + j * 16 + (lane & 15); }
};
typedef f32x4 XAcc[AccX::NI][AccX::NJ];

// Byte of 16-byte chunk c (8 K-values) of a plane's row: the swizzle that keeps a 16-lane pass over 16 rows of one
// chunk on all 64 banks once, reading and writing.
__device__ __forceinline__ int xslot(int row, int c) { return row * XROWB + ((c ^ ((row >> 2) & 3)) << 4); }

// x = p0 + p1 + p2, 8 values at a time: p0 = x to the nearest bf16, p1 the (exact) remainder to the nearest, p2 what is
// left, at most 7 bits, a bf16 as it stands. To the nearest and not towards zero, so that the remainders, and with them
// the partial products left out, have either sign: cut off, they all lean one way, 2^-23 of every sum, and the logprobs
// of [512, 32,000] logits were a quarter further from 64 bits than the fp32 instructions' (1.1e-6 against 8.8e-7). A
// value whose p0 is not finite keeps p0 alone: nothing needs it to (mainloop_plain), but the loop is 1-2% slower
// without the select (those logits 182 and 186 us).
__device__ __forceinline__ void split8(const float (&x)[8], i32x4 (&p)[3]) {
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    float r[2] = {x[2 * h], x[2 * h + 1]};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
      bf16x2 t;
      t[0] = (__bf16)r[0];
      t[1] = (__bf16)r[1];
      const uint32_t u = __builtin_bit_cast(uint32_t, t);
      p[k][h] = (int)u;
      if (k == 2) break;
      const float f[2] = {__uint_as_float(u << 16), __uint_as_float(u & 0xffff0000u)};
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        r[e] -= f[e];
        if (k == 0) r[e] = __builtin_fabsf(f[e]) < INFINITY ? r[e] : 0.f;
      }
    }
  }
}

// K-contiguous rows: R rows of the tile, 4 chunks of 8 values each per stage; item q of thread t is row (512 q + t) /
// 4, chunk t % 4, so that 4 neighbouring lanes read a row's 128 bytes.
template <int R> struct XRows {
  static constexpr int Q = R * 4 / XTHREADS;
  __amdgpu_buffer_rsrc_t rs;
  uint32_t off[Q], kbytes;
  float x[Q][8];
  __device__ __forceinline__ void init(const Operand &op, int64_t row0, int64_t K) {
    const int64_t valid = dev_count(op.count, op.count_off + row0, op.rows - row0);
    kbytes = (uint32_t)(K * 4);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int r = (q * XTHREADS + (int)threadIdx.x) >> 2;
      off[q] = r >= valid ? 0x80000000u : op.map ? (uint32_t)(op.map[row0 + r] * op.ld) : (uint32_t)(r * op.ld);
    }
    if (op.map) rs = make_rsrc(uniform_ptr(op.base), op.extent);
    else rs = make_rsrc(uniform_ptr(op.base + row0 * op.ld), (uint32_t)(R * op.ld));
  }
  __device__ __forceinline__ void load(int k) {  // K-values past the end read zero, 4 at a time
    const uint32_t kb = (uint32_t)k * (XK * 4) + (threadIdx.x & 3) * 32;
#pragma unroll
    for (int q = 0; q < Q; ++q)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bool in = kb + 16 * h < kbytes && off[q] < 0x80000000u;
        const f32x4 v = __builtin_bit_cast(f32x4, buf_load16(rs, in ? (int)(off[q] + kb + 16 * h) : (int)0x80000000u));
#pragma unroll
        for (int e = 0; e < 4; ++e) x[q][4 * h + e] = v[e];
      }
  }
  __device__ __forceinline__ void store(lds_char *planes) const {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      i32x4 p[3];
      split8(x[q], p);
      lds_char *at = planes + xslot((q * XTHREADS + (int)threadIdx.x) >> 2, threadIdx.x & 3);
#pragma unroll
      for (int k = 0; k < 3; ++k) *(lds_i32x4 *)(at + k * R * XROWB) = p[k];
    }
  }
};

// K down the matrix rows: C columns of the tile; item q of thread t is column (512 q + t) % C, chunk (512 q + t) / C.
// Rows at or past K and columns past the matrix read zero.
template <int C> struct XCols {
  static constexpr int Q = C * 4 / XTHREADS;
  const char *base;
  uint32_t ld;
  int K;
  bool col_ok[Q];
  uint32_t lo[Q];
  float x[Q][8];
  __device__ __forceinline__ void init(const Operand &op, int64_t col0, int64_t K_) {
    base = uniform_ptr(op.base + col0 * 4);
    ld = (uint32_t)op.ld;
    K = (int)K_;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = q * XTHREADS + (int)threadIdx.x, col = i % C;
      col_ok[q] = col < op.rows - col0;
      lo[q] = (uint32_t)(i / C) * 8 * ld + col * 4;
    }
  }
  __device__ __forceinline__ void load(int k) {
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(base + (int64_t)k * XK * ld, XK * ld);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int k0 = k * XK + (q * XTHREADS + (int)threadIdx.x) / C * 8;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const bool in = col_ok[q] && k0 + e < K;
        const int off = in ? (int)(lo[q] + e * ld) : (int)0x80000000u;
        x[q][e] = __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
      }
    }
  }
  __device__ __forceinline__ void store(lds_char *planes) const {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = q * XTHREADS + (int)threadIdx.x;
      i32x4 p[3];
      split8(x[q], p);
      lds_char *at = planes + xslot(i % C, i / C);
#pragma unroll
      for (int k = 0; k < 3; ++k) *(lds_i32x4 *)(at + k * C * XROWB) = p[k];
    }
  }
};

__device__ __forceinline__ void xmfma(const i32x4 a, const i32x4 b, f32x4 &c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// This wave's MFMAs of one stage: the smaller products first. TR as ring5_stage's (gemm_nt.h): a lane's 4 values are 4
// columns of a row.
template <bool TR>
__device__ __forceinline__ void xstage(const lds_char *A, const lds_char *B, int wm, int wn, int lane, XAcc &acc) {
  constexpr int PA[6] = {2, 0, 1, 1, 0, 0}, PB[6] = {0, 2, 1, 0, 1, 0};
  i32x4 fb[3][AccX::NJ];
#pragma unroll
  for (int k = 0; k < 3; ++k)
#pragma unroll
    for (int j = 0; j < AccX::NJ; ++j)
      fb[k][j] = *(const lds_i32x4 *)(B + k * XPB + xslot(wn * 32 + j * 16 + (lane & 15), lane >> 4));
#pragma unroll
  for (int i = 0; i < AccX::NI; i += 2) {
    i32x4 fa[3][2];
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int u = 0; u < 2; ++u)
        fa[k][u] = *(const lds_i32x4 *)(A + k * XPA + xslot(wm * 128 + (i + u) * 16 + (lane & 15), lane >> 4));
#pragma unroll
    for (int t = 0; t < 6; ++t)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < AccX::NJ; ++j) {
          if constexpr (TR) xmfma(fb[PB[t]][j], fa[PA[t]][u], acc[i + u][j]);
          else xmfma(fa[PA[t]][u], fb[PB[t]][j], acc[i + u][j]);
        }
  }
}

// Every wave's LDS reads and writes so far are done (global loads may be in flight).
__device__ __forceinline__ void xbarrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(WAIT_LGKM0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// acc = the tile's sums over nk stages; smem holds two stages. Ends with every wave past its last LDS read.
template <bool TR, typename LA, typename LB>
__device__ __forceinline__ void mainloop_x(LA &a, LB &b, int nk, lds_char *smem, XAcc &acc) {
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wm = w >> 2, wn = w & 3;
#pragma unroll
  for (int i = 0; i < AccX::NI; ++i)
#pragma unroll
    for (int j = 0; j < AccX::NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (nk == 0) return;
  a.load(0);
  b.load(0);
  a.store(smem);
  b.store(smem + 3 * XPA);
  if (nk > 1) {
    a.load(1);
    b.load(1);
  }
  xbarrier();
  for (int k = 0; k < nk; ++k) {
    lds_char *cur = smem + (k & 1) * XSTAGE, *nxt = smem + (1 - (k & 1)) * XSTAGE;
    auto refill = [&]() {  // stage k + 1 from its registers into the other buffer, stage k + 2 into the registers
      if (k + 1 < nk) {
        a.store(nxt);
        b.store(nxt + 3 * XPA);
      }
      if (k + 2 < nk) {
        a.load(k + 2);
        b.load(k + 2);
      }
    };
    if (wm == 0) refill();
    xstage<TR>(cur, cur + 3 * XPA, wm, wn, lane, acc);
    if (wm != 0) refill();
    xbarrier();
  }
}

// An operand's value i (row, or column of a K-major one) at k, read by itself; 0 outside the matrix.
struct XPlain {
  const char *base;
  const int64_t *map;
  int64_t ld, rows, K;
  bool down;  // K down the matrix rows
  __device__ __forceinline__ XPlain(const Operand &op, int64_t row0, int64_t K_, bool down_)
      : base(op.base), map(op.map ? op.map + row0 : nullptr), ld(op.ld), K(K_), down(down_) {
    rows = down ? op.rows - row0 : dev_count(op.count, op.count_off + row0, op.rows - row0);
    if (down) base += row0 * 4;
    else if (!map) base += row0 * ld;
  }
  __device__ __forceinline__ float at(int i, int64_t k) const {
    if (i >= rows || k >= K) return 0.f;
    return *(const float *)(down ? base + k * ld + i * 4 : base + (map ? map[i] : i) * ld + k * 4);
  }
};

// This wave's acc made again without the split, 4 K-values at a time from global memory. Rare and slow: not tuned.
template <bool TR>
__device__ __forceinline__ void mainloop_plain(const XPlain &a, const XPlain &b, XAcc &acc) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wm = w >> 2, wn = w & 3;
#pragma unroll
  for (int i = 0; i < AccX::NI; ++i)
#pragma unroll
    for (int j = 0; j < AccX::NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int64_t k0 = 0; k0 < a.K; k0 += 4) {
    const int64_t k = k0 + (lane >> 4);
    float fb[AccX::NJ];
#pragma unroll
    for (int j = 0; j < AccX::NJ; ++j) fb[j] = b.at(wn * 32 + j * 16 + (lane & 15), k);
#pragma unroll
    for (int i = 0; i < AccX::NI; ++i) {
      const float fa = a.at(wm * 128 + i * 16 + (lane & 15), k);
#pragma unroll
      for (int j = 0; j < AccX::NJ; ++j)
        acc[i][j] = TR ? __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j], fa, acc[i][j], 0, 0, 0)
                       : __builtin_amdgcn_mfma_f32_16x16x4f32(fa, fb[j], acc[i][j], 0, 0, 0);
    }
  }
}

// Whether an operand of this wave's part of the tile had such a value: it leaves no finite sum in its row or column, so
// one row and one column of blocks tell.
template <bool TR> __device__ __forceinline__ bool xnonfinite(const XAcc &acc) {
  float z = 0.f;
#pragma unroll
  for (int i = 0; i < AccX::NI; ++i)
#pragma unroll
    for (int v = 0; v < (TR ? 1 : AccX::NV); ++v) z = __builtin_fmaf(acc[i][0][v], 0.f, z);  // 0 x inf and 0 x NaN: NaN
#pragma unroll
  for (int j = 0; j < AccX::NJ; ++j)
#pragma unroll
    for (int v = 0; v < (TR ? AccX::NV : 1); ++v) z = __builtin_fmaf(acc[0][j][v], 0.f, z);
  return __any(z != 0.f);
}

// The tile's sums over K of A's rows from m0 on and B's from n0 on; a K-major operand (KM_A, KM_B) as XCols.
template <bool TR, int KM>
__device__ __forceinline__ void xtile(const Operand &A, const Operand &B, int64_t m0, int64_t n0, int64_t K,
                                      lds_char *smem, XAcc &acc) {
  const int stages = __builtin_amdgcn_readfirstlane((int)cdiv(K, (int64_t)XK));
  {
    typename std::conditional<KM == KM_A, XCols<XM>, XRows<XM>>::type a;
    typename std::conditional<KM == KM_B, XCols<XN>, XRows<XN>>::type b;
    a.init(A, m0, K);
    b.init(B, n0, K);
    mainloop_x<TR>(a, b, stages, smem, acc);
  }
  if (xnonfinite<TR>(acc)) mainloop_plain<TR>(XPlain(A, m0, K, KM == KM_A), XPlain(B, n0, K, KM == KM_B), acc);
}

// Tiles of the 256 x 128 grid, shrunk by a device count that bounds M or N; the order is gemm_nt.h's.
__device__ __forceinline__ void xtiles(const GemmShape &s, int64_t &mtiles, int64_t &ntiles) {
  mtiles = s.mtiles;
  ntiles = s.ntiles;
  if (s.count_on == 1) mtiles = min(mtiles, cdiv(dev_count(s.count, s.count_off, s.M), (int64_t)XM));
  if (s.count_on == 2) ntiles = min(ntiles, cdiv(dev_count(s.count, s.count_off, s.N), (int64_t)XN));
}
__device__ __forceinline__ bool xtile_of(const GemmShape &s, int &mt, int &nt) {
  int64_t mtiles, ntiles;
  xtiles(s, mtiles, ntiles);
  return tile_at(s, (int)(blockIdx.x & 7), (int64_t)(blockIdx.x >> 3), mtiles, ntiles, mt, nt);
}
__device__ __forceinline__ int64_t xtokens(const GemmShape &s, int64_t n0) {  // the tile's valid columns
  return min(dev_count(s.count, s.count_off + n0, s.N - n0), (int64_t)XN);
}

#define XKERNEL __global__ __launch_bounds__(XTHREADS, 1) __attribute__((amdgpu_waves_per_eu(2, 2))) void

// ---- logits: softmax statistics -------------------------------------------------------------------------------------
// As gemm_stats8_kernel (head_gemm.hip) without exponentials: part[row][vocab tile] = (m_a, S, U, m_b).
template <bool TANH>
XKERNEL gemm_stats_x_kernel(Operand A, Operand B, GemmShape s, StatsArgs e) {
  typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
  __shared__ __attribute__((aligned(16))) char smem_[2 * XSTAGE];
  lds_char *smem = (lds_char *)smem_;
  int mt, nt;
  if (!xtile_of(s, mt, nt)) return;
  const int64_t m0 = (int64_t)mt * XM, n0 = (int64_t)nt * XN, nvalid = xtokens(s, n0);
  if (nvalid <= 0) return;
  XAcc acc;
  xtile<false, KM_NONE>(A, B, m0, n0, s.K, smem, acc);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wm = w >> 2, wn = w & 3;
  const int64_t ma = e.v0 + m0;                       // first vocabulary row of the tile
  const int valid = (int)min(e.V - ma, (int64_t)XM);  // its rows below V
  lds_f32x4 *red = (lds_f32x4 *)smem;
#pragma unroll
  for (int j = 0; j < AccX::NJ; ++j) {
    float mx = -INFINITY;
#pragma unroll
    for (int i = 0; i < AccX::NI; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        if constexpr (TANH) acc[i][j][v] = ftanh(e.pre * acc[i][j][v]);
        if (AccX::row(wm, i, v, lane) < valid) mx = fmaxf(mx, acc[i][j][v]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float m2 = mx * e.c;
    float S = 0.f, U = 0.f;
#pragma unroll
    for (int i = 0; i < AccX::NI; ++i)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float t = __builtin_fmaf(acc[i][j][v], e.c, -m2);
        const float x = AccX::row(wm, i, v, lane) < valid ? fexp2(t) : 0.f;
        S += x;
        U = __builtin_fmaf(x, t, U);
      }
    S += __shfl_xor(S, 16, 64);
    S += __shfl_xor(S, 32, 64);
    U += __shfl_xor(U, 16, 64);
    U += __shfl_xor(U, 32, 64);
    if (lane < 16) red[wm * XN + AccX::col(wn, j, lane)] = f32x4{m2, S, U, 0.f};
  }
  __syncthreads();
  const int t = threadIdx.x;
  if (t < nvalid) {
    const f32x4 a = red[t], b = red[XN + t];
    const Stat3 r = stat_merge(Stat3{a[0], a[1], a[2]}, Stat3{b[0], b[1], b[2]});
    e.part[(n0 + t) * e.mtiles + e.v0 / XM + mt] = f32x4{a[0], r.S, r.U, b[0]};
  }
}

// ---- logits: dz -----------------------------------------------------------------------------------------------------
// dz = g (onehot - p) / T x post'(z), token-major [token][chunk column] fp32, zero past V.
template <bool TANH>
XKERNEL gemm_dz_x_kernel(Operand A, Operand B, GemmShape s, DzArgs e) {
  __shared__ __attribute__((aligned(16))) char smem_[2 * XSTAGE];
  int mt, nt;
  if (!xtile_of(s, mt, nt)) return;
  const int64_t m0 = (int64_t)mt * XM, n0 = (int64_t)nt * XN, nvalid = xtokens(s, n0);
  if (nvalid <= 0) return;
  XAcc acc;
  xtile<false, KM_NONE>(A, B, m0, n0, s.K, (lds_char *)smem_, acc);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wm = w >> 2, wn = w & 3;
  const int64_t ma = e.v0 + m0;
  const int valid = (int)min(e.V - ma, (int64_t)XM);
#pragma unroll
  for (int j = 0; j < AccX::NJ; ++j) {
    const int t = AccX::col(wn, j, lane);
    if (t >= nvalid) continue;
    const int64_t r = e.row_off + n0 + t;  // compact row
    float m2, l2s;
    row_state(e.lse, e.lse_pair, r, m2, l2s);
    const float gs = e.g[r] * e.gmul;
    const int64_t y = e.labels[e.label_idx ? e.label_idx[r] : r] - ma;
    float *dst = (float *)e.dzA + (n0 + t) * e.ldA + m0;
#pragma unroll
    for (int i = 0; i < AccX::NI; ++i) {
      const int row = AccX::row(wm, i, 0, lane);
      f32x4 d;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float x = acc[i][j][v], slope = 1.f;
        if constexpr (TANH) {
          x = ftanh(e.pre * x);
          slope = 1.f - x * x;
        }
        const float p = fexp2(__builtin_fmaf(x, e.c, -m2) - l2s);
        d[v] = row + v < valid ? __builtin_fmaf(-gs, p, y == row + v ? gs : 0.f) * slope : 0.f;
      }
      *(f32x4 *)(dst + row) = d;
    }
  }
}

// ---- gradients ------------------------------------------------------------------------------------------------------
// C = rs[row] x acc (+ addend) (+ C when accumulate), one loop with the run-time choices inside. A lane's 4 values of a
// block are neighbours in C's row (TR). An fp32 C += acc is one no-return atomic per element (one tile adds to it per
// launch, so the sums keep launch order).
template <typename OT>
__device__ __forceinline__ void store_x(const XAcc &acc, const StoreArgs &e, int64_t m0, int64_t n0, int64_t mvalid,
                                        int64_t nvalid) {
  typedef OT OT4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, wm = w >> 2, wn = w & 3;
  const bool aligned = (uintptr_t)e.C % sizeof(OT4) == 0 && e.ldc % 4 == 0;
#pragma unroll
  for (int i = 0; i < AccX::NI; ++i) {
    const int rr = wm * 128 + i * 16 + (lane & 15);
    if (rr >= mvalid) continue;
    OT *crow = (OT *)e.C + (m0 + rr) * e.ldc + n0;
    const float *arow = e.addend ? e.addend + (m0 + rr) * e.ld_add + n0 : nullptr;
    const float sc = e.row_scale ? e.row_scale[m0 + rr] : 1.f;
#pragma unroll
    for (int j = 0; j < AccX::NJ; ++j) {
      const int cc = wn * 32 + j * 16 + 4 * (lane >> 4);
      f32x4 x = acc[i][j];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        x[v] *= sc;
        if (arow) x[v] += cc + v < nvalid ? arow[cc + v] : 0.f;
      }
      if (e.accumulate && std::is_same<OT, float>::value) {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (cc + v < nvalid)
            __hip_atomic_fetch_add((float *)crow + cc + v, x[v], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        continue;
      }
      if (e.accumulate)
#pragma unroll
        for (int v = 0; v < 4; ++v) x[v] += cc + v < nvalid ? (float)crow[cc + v] : 0.f;
      if (aligned && cc + 4 <= nvalid) {
        OT4 o;
#pragma unroll
        for (int v = 0; v < 4; ++v) o[v] = (OT)x[v];
        *(OT4 *)(crow + cc) = o;
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (cc + v < nvalid) crow[cc + v] = (OT)x[v];
      }
    }
  }
}

// KM_B: grad_h = dz . W, its K in runs where StoreArgs::split has room (tile_order.h; partial tiles of 256 x 128,
// summed by split_sum). KM_A: grad_W = dz^T . h from h^T.
template <int OT, int KM>
XKERNEL gemm_store_x_kernel(Operand A, Operand B, GemmShape s, StoreArgs e) {
  __shared__ __attribute__((aligned(16))) char smem_[2 * XSTAGE];
  int64_t mtiles, ntiles;
  xtiles(s, mtiles, ntiles);
  int mt, nt, run = 0, S = 1;
  const int nk = (int)cdiv(s.K, (int64_t)64), tiles = (int)(mtiles * ntiles);
  if (KM == KM_B && e.split)
    S = __builtin_amdgcn_readfirstlane(octo_tiles::k_splits(tiles, nk, true, e.split_cap));
  if (S > 1) {
    const bool in = octo_tiles::split_item_at((int)(blockIdx.x & 7), (int)(blockIdx.x >> 3), S, (int)mtiles,
                                              (int)ntiles, run, mt, nt);
    if (!__builtin_amdgcn_readfirstlane(in)) return;
    run = __builtin_amdgcn_readfirstlane(run);
    mt = __builtin_amdgcn_readfirstlane(mt);
    nt = __builtin_amdgcn_readfirstlane(nt);
  } else if (!tile_at(s, (int)(blockIdx.x & 7), (int64_t)(blockIdx.x >> 3), mtiles, ntiles, mt, nt)) {
    return;
  }
  if (pass_store(e) == 0) return;
  const int64_t m0 = (int64_t)mt * XM, n0 = (int64_t)nt * XN;
  int64_t mvalid = s.M - m0, K = s.K;
  const int64_t nvalid = s.N - n0;
  if (s.count_on == 1) mvalid = dev_count(s.count, s.count_off + m0, mvalid);
  if (s.count_on == 3) K = dev_count(s.count, s.count_off, s.K);
  if (mvalid <= 0 || nvalid <= 0 || adds_nothing(e, 1, K)) return;
  if (S > 1) {
    const int k0 = 64 * __builtin_amdgcn_readfirstlane(octo_tiles::split_stage(run, S, nk));
    const int k1 = 64 * __builtin_amdgcn_readfirstlane(octo_tiles::split_stage(run + 1, S, nk));
    A.base += (int64_t)k0 * 4;
    B.base += k0 * B.ld;
    K = __builtin_amdgcn_readfirstlane(min(k1, (int)s.K) - k0);
  }
  XAcc acc;
  xtile<true, KM>(A, B, m0, n0, K, (lds_char *)smem_, acc);
  if (S > 1) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t at = (int64_t)run * tiles + (int64_t)nt * mtiles + mt;
    f32x4 *p = (f32x4 *)(e.split + at * (XM * XN) + w * (XM * XN / 8)) + lane;
#pragma unroll
    for (int i = 0; i < AccX::NI; ++i)
#pragma unroll
      for (int j = 0; j < AccX::NJ; ++j) p[(i * AccX::NJ + j) * 64] = acc[i][j];
    return;
  }
  store_x<typename Elem<OT>::T>(acc, e, m0, n0, mvalid, nvalid);
}

// ---- host launchers -------------------------------------------------------------------------------------------------

// The shape over 256 x 128 tiles.
static GemmShape xshape(GemmShape s) {
  s.ntiles = (int)cdiv(s.N, (int64_t)XN);
  return s;
}
static dim3 xgrid(const GemmShape &s) { return dim3((unsigned)tile_grid(s.mtiles, s.ntiles)); }

int launch_gemm_stats_f32(bool tanh, const Operand &A, const Operand &B, const GemmShape &s0, const StatsArgs &e,
                          hipStream_t st) {
  if (e.ex || e.z) return octo_fail(OCTO_EUNSUPPORTED, "gemm_stats: exponentials or kept logits of fp32 operands");
  const GemmShape s = xshape(s0);
  if (tanh) hipLaunchKernelGGL(gemm_stats_x_kernel<true>, xgrid(s), dim3(XTHREADS), 0, st, A, B, s, e);
  else hipLaunchKernelGGL(gemm_stats_x_kernel<false>, xgrid(s), dim3(XTHREADS), 0, st, A, B, s, e);
  OCTO_CHECK_LAUNCH("gemm_stats");
  return OCTO_OK;
}

int launch_gemm_dz_f32(bool tanh, const Operand &A, const Operand &B, const GemmShape &s0, const DzArgs &e,
                       hipStream_t st) {
  const GemmShape s = xshape(s0);
  if (tanh) hipLaunchKernelGGL(gemm_dz_x_kernel<true>, xgrid(s), dim3(XTHREADS), 0, st, A, B, s, e);
  else hipLaunchKernelGGL(gemm_dz_x_kernel<false>, xgrid(s), dim3(XTHREADS), 0, st, A, B, s, e);
  OCTO_CHECK_LAUNCH("gemm_dz");
  return OCTO_OK;
}

template <int OT>
static void go_store_x(const Operand &A, const Operand &B, const GemmShape &s, const StoreArgs &e, hipStream_t st,
                       int kmajor) {
  int64_t blocks = tile_grid(s.mtiles, s.ntiles);
  if (e.split && round_up(e.split_cap, 8) > blocks) blocks = round_up(e.split_cap, 8);
  const dim3 grid((unsigned)blocks);
  if (kmajor == KM_A) hipLaunchKernelGGL((gemm_store_x_kernel<OT, KM_A>), grid, dim3(XTHREADS), 0, st, A, B, s, e);
  else hipLaunchKernelGGL((gemm_store_x_kernel<OT, KM_B>), grid, dim3(XTHREADS), 0, st, A, B, s, e);
}

int launch_gemm_store_f32(const Operand &A, const Operand &B, const GemmShape &s0, const StoreArgs &e, hipStream_t st,
                          int kmajor) {
  if (e.part || e.part_blocked || kmajor == KM_NONE || (e.split && kmajor != KM_B))
    return octo_fail(OCTO_EUNSUPPORTED, "gemm_store: this product of fp32 operands");
  const Operand &c = kmajor == KM_A ? A : B;  // the K-major operand's stage: 32 rows within 32-bit offsets
  if (c.map || c.ld > 0x7fffffffLL / XK || c.ld % 4)
    return octo_fail(OCTO_EINVAL, "gemm_store: K-major operand layout");
  const GemmShape s = xshape(s0);
  switch (e.dtype) {
    case OCTO_BF16: go_store_x<OCTO_BF16>(A, B, s, e, st, kmajor); break;
    case OCTO_F16: go_store_x<OCTO_F16>(A, B, s, e, st, kmajor); break;
    case OCTO_F32: go_store_x<OCTO_F32>(A, B, s, e, st, kmajor); break;
    default: return octo_fail(OCTO_EUNSUPPORTED, "gemm_store: output dtype %d", e.dtype);
  }
  OCTO_CHECK_LAUNCH("gemm_store");
  return OCTO_OK;
}

}  // namespace octo
