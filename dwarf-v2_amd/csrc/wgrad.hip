// The weight and bias gradients of a linear layer over many rows,
// dW = dY^T X and db = dY^T 1, from bf16 to fp32.
//
// The block's projections give few outputs from many rows (2,048 x 512 and
// 512 x 512 from 30,720 tokens): a GEMM tiled over its outputs alone has 32
// workgroups for 256 CUs (hipBLASLt: 196 and 149 us, and 37 us for the bias).
// Here the rows are split so that about one workgroup runs per CU; each
// writes an fp32 partial tile and a second launch adds the splits in order.
//
// A workgroup of eight waves owns 128 outputs x 256 inputs; wave (wo, wi) 64 x
// 64 of them as 2 x 2 v_mfma_f32_32x32x16_bf16 accumulators.  Rows come 64 at
// a time through registers (two steps ahead) into one of two LDS buffers, as
// they are in memory; both operands have the token index along k, so they are
// read transposed (ds_read_b64_tr_b16).  16-byte chunk c of row r sits at
// chunk c ^ 2 (r & 7), which spreads the four rows of a transposed read over
// different banks.  The bias sums are added up as the rows pass through the
// registers.  Both launches together, 2,048 x 512 and 512 x 512 from 30,720
// rows: 86 and 35 us (794 and 461 TFLOP/s; the partial sums are 33 MB each);
// four waves of 64 x 128 107 and 42 (nothing to issue while a wave waits for
// its operands), two workgroups of 128 x 128 per CU 107 and 43, the bias as
// dot products of the operands 100 and 38.
// One split (more than 128 tiles, or at most four 64-row steps) writes dW and
// db itself instead of a partial and a copy of it: 16,384 x 4,096 from 256
// rows 204 -> 89 us, 8,192 x 2,048 from 200, 2,048 and 8,192 rows 52 -> 32,
// 117 -> 97, 346 -> 312 (the library, to bf16, with the cast and the bias:
// 141, 53, 116, 297; it is ahead from there on, 1,142 against 972 at 30,720
// rows, and rounds dW to bf16).
#include "common.h"
#include "dsqg_internal.h"
#include "dwarf_block.h"
#include "gather.h"
#include "mfma.h"

namespace dwarf {
namespace {

constexpr int kWgThreads = 512;
constexpr int kTO = 128, kTI = 256, kTK = 64;    // outputs, inputs, rows of a step
constexpr int kRowO = kTO * 2, kRowI = kTI * 2;  // LDS row bytes
constexpr int kStageBytes = kTK * (kRowO + kRowI);
constexpr int kLoadO = kTK * kRowO / 16 / kWgThreads, kLoadI = kTK * kRowI / 16 / kWgThreads;   // 16-byte loads per thread: 2, 4

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef short i16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ f32x16 mfma32_bf16(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

struct WgradStep {
  uint4 o[kLoadO], i[kLoadI];
};

__global__ __launch_bounds__(kWgThreads, 1) void linear_wgrad_kernel(const dwarf_linear_wgrad_args a, int splits, int rows_per,
                                                                 int tiles_i, float* __restrict__ part,
                                                                 float* __restrict__ part_b) {
  extern __shared__ __align__(16) char w_smem[];   // [2][kTK rows of dY, kTK rows of X]
  const int split = blockIdx.x % splits, tile = blockIdx.x / splits;   // a split's tiles share an XCD's L2
  const int o0 = tile / tiles_i * kTO, i0 = tile % tiles_i * kTI;
  const int64_t m0 = static_cast<int64_t>(split) * rows_per;
  const int rows = static_cast<int>(a.M - m0 < rows_per ? a.M - m0 : rows_per);
  const int steps = (rows + kTK - 1) / kTK;
  const int tid = threadIdx.x, w = uniform(tid / kWave), l = tid % kWave;
  const int wo = w >> 2, wi = w & 3;
  const int ldo = static_cast<int>(a.dy_stride) * 2, ldi = static_cast<int>(a.x_stride) * 2;
  const __amdgpu_buffer_rsrc_t ro = rows_rsrc(static_cast<const bf16*>(a.dy) + m0 * a.dy_stride, ldo, rows, 2 * a.O);
  const __amdgpu_buffer_rsrc_t ri = rows_rsrc(static_cast<const bf16*>(a.x) + m0 * a.x_stride, ldi, rows, 2 * a.I);

  // This thread's 16-byte pieces of a step: chunk tid % 16 (tid % 32) of rows tid / 16 + 32 u (tid / 32 + 16 u).  Rows
  // past the split lie past the resource's end and read zeros, and so does a column past O or I, by an offset past
  // every row: no condition stands around a load.
  const int co = tid % (kTO / 8), ro0 = tid / (kTO / 8), ci = tid % (kTI / 8), ri0 = tid / (kTI / 8);
  const uint32_t vo = (o0 + 8 * co < a.O ? 2u * (o0 + 8 * co) : kOutOfRange) + static_cast<uint32_t>(ro0 * ldo);
  const uint32_t vi = (i0 + 8 * ci < a.I ? 2u * (i0 + 8 * ci) : kOutOfRange) + static_cast<uint32_t>(ri0 * ldi);
  const int po = ro0 * kRowO + 16 * (co ^ 2 * (ro0 & 7)), pi = kTK * kRowO + ri0 * kRowI + 16 * (ci ^ 2 * (ri0 & 7));
  auto fetch = [&](WgradStep& s, int step) {
#pragma unroll
    for (int u = 0; u < kLoadO; ++u) s.o[u] = buf_load16(ro, vo + static_cast<uint32_t>((step * kTK + 32 * u) * ldo));
#pragma unroll
    for (int u = 0; u < kLoadI; ++u) s.i[u] = buf_load16(ri, vi + static_cast<uint32_t>((step * kTK + 16 * u) * ldi));
  };
  float bsum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};   // this thread's rows of its eight outputs
  auto put = [&](const WgradStep& s, int buf) {   // rows 32 (16) apart share a swizzle
    char* b = w_smem + buf * kStageBytes;
#pragma unroll
    for (int u = 0; u < kLoadO; ++u) {
      *reinterpret_cast<uint4*>(b + po + 32 * u * kRowO) = s.o[u];
      const uint32_t x[4] = {s.o[u].x, s.o[u].y, s.o[u].z, s.o[u].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        bsum[2 * e] += bf16_lo(x[e]);
        bsum[2 * e + 1] += bf16_hi(x[e]);
      }
    }
#pragma unroll
    for (int u = 0; u < kLoadI; ++u) *reinterpret_cast<uint4*>(b + pi + 16 * u * kRowI) = s.i[u];
  };

  // Operand lane l: column l % 32 of a 32-column block, rows 8 (l / 32) + [0, 8) of 16.  Two transposed reads of four
  // rows each; in each, lane j = l % 16 points at row j / 4, columns 16 ((l / 16) % 2) + 4 (j % 4).
  const int j = l & 15, rowl = 8 * (l >> 5) + (j >> 2);
  const int chunk = 2 * ((l >> 4) & 1) + ((j & 3) >> 1), half = 8 * (j & 1);
  int ao[2][2], ai[2][2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = rowl + 4 * h, x = 2 * (r & 7);
#pragma unroll
    for (int t = 0; t < 2; ++t) ao[t][h] = r * kRowO + 16 * ((8 * wo + 4 * t + chunk) ^ x) + half;
#pragma unroll
    for (int t = 0; t < 2; ++t) ai[t][h] = kTK * kRowO + r * kRowI + 16 * ((8 * wi + 4 * t + chunk) ^ x) + half;
  }
  f32x16 acc[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[t][u][r] = 0.f;

  auto operand = [&](const char* base, const int* off) {
    const i16x4 lo = lds_read_tr16(base + off[0]), hi = lds_read_tr16(base + off[1]);
    const i16x8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8, v);
  };
  auto compute = [&](int buf) {
    const char* base = w_smem + buf * kStageBytes;
#pragma unroll
    for (int k = 0; k < kTK / 16; ++k) {
      bf16x8 xo[2], xi[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) xo[t] = operand(base + 16 * k * kRowO, ao[t]);
#pragma unroll
      for (int t = 0; t < 2; ++t) xi[t] = operand(base + 16 * k * kRowI, ai[t]);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u) acc[t][u] = mfma32_bf16(xo[t], xi[u], acc[t][u]);
    }
  };

  WgradStep s0, s1;
  fetch(s0, 0);
  fetch(s1, 1);   // rows past the split read zeros
  put(s0, 0);
  fetch(s0, 2);
  __syncthreads();
  for (int s = 0; s < steps; s += 2) {   // a step past the last adds zeros
    put(s1, 1);
    fetch(s1, s + 3);
    compute(0);
    __syncthreads();
    put(s0, 0);
    fetch(s0, s + 4);
    compute(1);
    __syncthreads();
  }

  // C: register 4 q + r of lane l is row 8 q + 4 (l / 32) + r, column l % 32
  float* p = part + static_cast<int64_t>(split) * a.O * a.I;
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int o = o0 + 64 * wo + 32 * t + 8 * q + 4 * (l >> 5) + r;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int i = i0 + 64 * wi + 32 * u + (l & 31);
          if (o < a.O && i < a.I) p[static_cast<int64_t>(o) * a.I + i] = acc[t][u][4 * q + r];
        }
      }
  if (a.db != nullptr && i0 == 0) {   // uniform; every wave is done with the tiles
    float* sb = reinterpret_cast<float*>(w_smem);
#pragma unroll
    for (int e = 0; e < 8; ++e) sb[ro0 * kTO + 8 * co + e] = bsum[e];
    __syncthreads();
    if (tid < kTO && o0 + tid < a.O) {
      float b = 0.f;
      for (int r = 0; r < kWgThreads / (kTO / 8); ++r) b += sb[r * kTO + tid];
      part_b[static_cast<int64_t>(split) * a.O + o0 + tid] = b;
    }
  }
}

// dW and db: the splits in order.
__global__ __launch_bounds__(kBlock) void linear_wgrad_sum(const float* __restrict__ part, const float* __restrict__ part_b,
                                                           int splits, int64_t n, int64_t nb, float* __restrict__ dw,
                                                           float* __restrict__ db) {
  const int64_t i = 4 * (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x);
  const bool w = i < n;
  const int64_t at = w ? i : i - n, len = w ? n : nb;
  if (at >= len) return;
  const float4* src = reinterpret_cast<const float4*>((w ? part : part_b) + at);
  float4 s = *src;
#pragma unroll 8
  for (int k = 1; k < splits; ++k) {
    const float4 x = src[k * (len / 4)];
    s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
  }
  *reinterpret_cast<float4*>((w ? dw : db) + at) = s;
}

struct WgradPlan {
  int tiles_o, tiles_i, splits, rows_per;
};
WgradPlan wgrad_plan(const dwarf_linear_wgrad_args& a) {
  WgradPlan p;
  p.tiles_o = (a.O + kTO - 1) / kTO;
  p.tiles_i = (a.I + kTI - 1) / kTI;
  const int tiles = p.tiles_o * p.tiles_i;
  // one workgroup per CU where a split keeps at least four steps; a split's rows are whole steps and are addressed
  // with 32-bit offsets
  int64_t want = 256 / tiles;
  if (want < 1) want = 1;
  const int64_t steps = (a.M + kTK - 1) / kTK;
  if (want > (steps + 3) / 4) want = (steps + 3) / 4;
  const int64_t ld = a.dy_stride > a.x_stride ? a.dy_stride : a.x_stride;
  const int64_t most = ((int64_t(1) << 30) / (2 * (ld > 0 ? ld : 1))) / kTK;   // steps of a split below 1 GiB
  if (most > 0 && want < (steps + most - 1) / most) want = (steps + most - 1) / most;
  const int64_t per = (steps + want - 1) / want + 1 & ~int64_t(1);   // the loop takes two steps a turn
  p.rows_per = static_cast<int>(per * kTK);
  p.splits = static_cast<int>((steps + per - 1) / per);
  return p;
}

}  // namespace

// One split writes dW and db itself: no partials, no second launch.
size_t linear_wgrad_workspace(const dwarf_linear_wgrad_args& a) {
  const WgradPlan p = wgrad_plan(a);
  if (p.splits == 1) return 0;
  return static_cast<size_t>(p.splits) * (static_cast<size_t>(a.O) * a.I + a.O) * sizeof(float);
}

hipError_t launch_linear_wgrad(const dwarf_linear_wgrad_args& a, hipStream_t stream) {
  const WgradPlan p = wgrad_plan(a);
  const int64_t n = static_cast<int64_t>(a.O) * a.I;
  float* part = p.splits > 1 ? static_cast<float*>(a.workspace) : a.dw;
  float* part_b = p.splits > 1 ? part + p.splits * n : a.db;
  hipLaunchKernelGGL(linear_wgrad_kernel, dim3(p.tiles_o * p.tiles_i * p.splits), dim3(kWgThreads), 2 * kStageBytes, stream, a,
                     p.splits, p.rows_per, p.tiles_i, part, part_b);
  if (p.splits == 1) return hipGetLastError();
  const int64_t quads = (n + (a.db ? a.O : 0)) / 4;
  hipLaunchKernelGGL(linear_wgrad_sum, dim3(static_cast<unsigned>((quads + kBlock - 1) / kBlock)), dim3(kBlock), 0, stream,
                     part, part_b, p.splits, n, a.db ? static_cast<int64_t>(a.O) : 0, a.dw, a.db);
  return hipGetLastError();
}

}  // namespace dwarf
