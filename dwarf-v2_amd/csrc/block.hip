// The DSQG block around the attention: its normalised phase probes, and its
// per-head gain and content gate (dsqg:3278-3284), forward and backward, one
// pass each.  PyTorch's chain for the same is six launches
// forward (fp32 product, permute copy, sigmoid, product, cast) and nine
// backward, most of them on fp32 tensors.
#include "common.h"
#include "dsqg_internal.h"
#include "dwarf_block.h"
#include "gather.h"

namespace dwarf {
namespace {

constexpr int kItemLanes = 8;                     // lanes per (b, n, h): 8 channels = 16 bytes each
constexpr int kItems = kBlock / kItemLanes;       // (b, n, h) items per workgroup step
constexpr int kMaxGateWgs = 2048;                 // eight per CU, all resident

__device__ __forceinline__ void unpack8(const uint4& w, float* x) {
  x[0] = bf16_lo(w.x); x[1] = bf16_hi(w.x); x[2] = bf16_lo(w.y); x[3] = bf16_hi(w.y);
  x[4] = bf16_lo(w.z); x[5] = bf16_hi(w.z); x[6] = bf16_lo(w.w); x[7] = bf16_hi(w.w);
}
__device__ __forceinline__ uint4 pack8(const float* x) {
  return uint4{pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]), pack_bf16x2(x[4], x[5]), pack_bf16x2(x[6], x[7])};
}
__device__ __forceinline__ float sigmoid_bf16(float x) { return round_bf16(__fdividef(1.f, 1.f + __expf(-x))); }

// <y, o> over the item's 64 dims in every lane, in the order of the DSQG backward's own delta (dsqg_bwd_dq.hip: 16
// dims to a lane as one chain, then four lanes), so both give the same bits: lane 2g + 1 goes on with lane 2g's chain.
__device__ __forceinline__ float item_delta(const uint4& y, const uint4& o) {
  auto chain = [&](float x) { return dot2bf(y.w, o.w, dot2bf(y.z, o.z, dot2bf(y.y, o.y, dot2bf(y.x, o.x, x)))); };
  float x = chain(dpp_f<0xA0>(chain(0.f)));   // quad_perm [0,0,2,2]
  x = dpp_f<0xF5>(x);                         // quad_perm [1,1,3,3]: lanes 2g and 2g + 1 hold slice g
  x += dpp_f<0x4E>(x);                        // slices 0 + 1 and 2 + 3
  return x + dpp_f<0x141>(x);                 // row_half_mirror: lane i of eight <-> 7 - i
}

// Sum over the item's eight lanes, in every lane.
__device__ __forceinline__ float item_sum(float x) {
  x = group_sum<4>(x);
  return x + dpp_f<0x141>(x);   // row_half_mirror: lane i of eight <-> 7 - i
}

struct Item {
  unsigned b, n, h;
};
__device__ __forceinline__ Item item_of(unsigned i, unsigned H, unsigned N) {
  const unsigned row = i / H, b = row / N;
  return {b, row - b * N, i - row * H};
}

// Memory bound: out, gate in and gated out, 94 MB at B15 H8 N2048.  Consecutive
// items are the heads of one token, so gate and gated move as whole lines, and
// so does out stored [B,N,H,64].
__global__ __launch_bounds__(kBlock) void head_gate_fwd_kernel(const dwarf_head_gate_fwd_args a, unsigned items) {
  const unsigned c = threadIdx.x % kItemLanes;
  for (unsigned i = blockIdx.x * kItems + threadIdx.x / kItemLanes; i < items; i += gridDim.x * kItems) {
    const Item t = item_of(i, a.H, a.N);
    const uint4 ow = *reinterpret_cast<const uint4*>(static_cast<const bf16*>(a.out) + t.b * a.out_stride[0] +
                                                     t.h * a.out_stride[1] + t.n * a.out_stride[2] + 8 * c);
    const int64_t ch = t.h * kHeadDim + 8 * c;
    const uint4 gw = *reinterpret_cast<const uint4*>(static_cast<const bf16*>(a.gate) + t.b * a.gate_stride[0] +
                                                     t.n * a.gate_stride[1] + ch);
    const float gain = a.gain[t.h];
    float o[8], x[8];
    unpack8(ow, o);
    unpack8(gw, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = (o[e] * gain) * sigmoid_bf16(x[e]);
    *reinterpret_cast<uint4*>(static_cast<bf16*>(a.gated) + t.b * a.gated_stride[0] + t.n * a.gated_stride[1] + ch) =
        pack8(x);
  }
}

// Memory bound: dgated, out, gate in and dout, dgate out, 157 MB at B15 H8
// N2048.  The grid's stride is a multiple of H, so a lane serves one head
// throughout and keeps its dgain term in a register; one partial per item
// slot at the end.  delta comes from the rounded dout the DSQG backward reads.
__global__ __launch_bounds__(kBlock) void head_gate_bwd_kernel(const dwarf_head_gate_bwd_args a, unsigned items,
                                                               float* __restrict__ part) {
  const dwarf_head_gate_fwd_args& f = a.fwd;
  const unsigned c = threadIdx.x % kItemLanes;
  const unsigned slot = blockIdx.x * kItems + threadIdx.x / kItemLanes;
  const float gain = f.gain[slot % f.H];
  float acc = 0.f;
  for (unsigned i = slot; i < items; i += gridDim.x * kItems) {
    const Item t = item_of(i, f.H, f.N);
    const int64_t ch = t.h * kHeadDim + 8 * c;
    const uint4 dw = *reinterpret_cast<const uint4*>(static_cast<const bf16*>(a.dgated) + t.b * a.dgated_stride[0] +
                                                     t.n * a.dgated_stride[1] + ch);
    const uint4 ow = *reinterpret_cast<const uint4*>(static_cast<const bf16*>(f.out) + t.b * f.out_stride[0] +
                                                     t.h * f.out_stride[1] + t.n * f.out_stride[2] + 8 * c);
    const uint4 gw = *reinterpret_cast<const uint4*>(static_cast<const bf16*>(f.gate) + t.b * f.gate_stride[0] +
                                                     t.n * f.gate_stride[1] + ch);
    float lse = 0.f;
    if (a.delta_pairs) lse = a.lse[t.b * a.lse_stride[0] + t.h * a.lse_stride[1] + t.n * a.lse_stride[2]];
    float d[8], o[8], x[8], y[8];
    unpack8(dw, d);
    unpack8(ow, o);
    unpack8(gw, x);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float s = sigmoid_bf16(x[e]);
      const float dm = d[e] * s;
      acc = fmaf(dm, o[e], acc);
      y[e] = dm * gain;
      x[e] = round_bf16(d[e] * (o[e] * gain)) * (1.f - s) * s;
    }
    const uint4 yw = pack8(y);
    *reinterpret_cast<uint4*>(static_cast<bf16*>(a.dout) + t.b * a.dout_stride[0] + t.h * a.dout_stride[1] +
                              t.n * a.dout_stride[2] + 8 * c) = yw;
    *reinterpret_cast<uint4*>(static_cast<bf16*>(a.dgate) + t.b * a.dgate_stride[0] + t.n * a.dgate_stride[1] + ch) =
        pack8(x);
    if (a.delta_pairs) {
      const bool mass = static_cast<int>(t.n) >= a.query_start && lse > -INFINITY;
      const float dlt = item_delta(yw, ow);
      if (c == 0)
        *reinterpret_cast<float2*>(a.delta_pairs + 2 * ((static_cast<int64_t>(t.b) * f.H + t.h) * f.N + t.n)) =
            make_float2(dlt, mass ? lse * kLog2e : INFINITY);
    }
  }
  acc = item_sum(acc);
  if (c == 0) part[slot] = acc;
}

// dgain[h]: the item slots of one head in a fixed order.
__global__ __launch_bounds__(kBlock) void head_gate_gain_kernel(const float* __restrict__ part, unsigned slots,
                                                                unsigned H, float* __restrict__ dgain) {
  __shared__ float s_sum[kBlock / kWave];
  float x = 0.f;
#pragma unroll 8
  for (unsigned i = blockIdx.x + threadIdx.x * H; i < slots; i += kBlock * H) x += part[i];
  x = wave_sum_to_last(x);
  if (threadIdx.x % kWave == kWave - 1) s_sum[threadIdx.x / kWave] = x;
  __syncthreads();
  if (threadIdx.x == 0) dgain[blockIdx.x] = (s_sum[0] + s_sum[1]) + (s_sum[2] + s_sum[3]);
}

// A wave per probe row (PyTorch's normalize of the two banks is eight launches,
// 20 us of the stream).
__global__ __launch_bounds__(8 * kWave) void normalize_probes_kernel(const float* __restrict__ q,
                                                                     const float* __restrict__ k,
                                                                     float* __restrict__ out) {
  const int row = threadIdx.x / kWave, d = threadIdx.x % kWave;
  const float x = (row < kPlanes ? q + row * kHeadDim : k + (row - kPlanes) * kHeadDim)[d];
  const float ss = __shfl(wave_sum_to_last(x * x), kWave - 1);
  out[row * kHeadDim + d] = __fdiv_rn(x, fmaxf(__fsqrt_rn(ss), 1e-12f));
}

// Workgroups whose item slots are a multiple of H.
unsigned gate_bwd_wgs(int H, unsigned items) {
  int a = H, b = kItems;   // H / gcd(H, kItems)
  while (b) { const int r = a % b; a = b; b = r; }
  const unsigned step = static_cast<unsigned>(H / a);
  unsigned want = (items + kItems - 1) / kItems;
  if (want > kMaxGateWgs) want = kMaxGateWgs;
  return (want + step - 1) / step * step;
}

}  // namespace

size_t head_gate_bwd_workspace(const dwarf_head_gate_bwd_args& a) {
  return static_cast<size_t>(gate_bwd_wgs(a.fwd.H, static_cast<unsigned>(a.fwd.B) * a.fwd.N * a.fwd.H)) * kItems *
         sizeof(float);
}

hipError_t launch_normalize_probes(const float* q, const float* k, float* out, hipStream_t stream) {
  hipLaunchKernelGGL(normalize_probes_kernel, dim3(1), dim3(8 * kWave), 0, stream, q, k, out);
  return hipGetLastError();
}

hipError_t launch_head_gate_fwd(const dwarf_head_gate_fwd_args& a, hipStream_t stream) {
  const unsigned items = static_cast<unsigned>(a.B) * a.N * a.H;
  const unsigned wgs = (items + kItems - 1) / kItems;
  hipLaunchKernelGGL(head_gate_fwd_kernel, dim3(wgs), dim3(kBlock), 0, stream, a, items);
  return hipGetLastError();
}

hipError_t launch_head_gate_bwd(const dwarf_head_gate_bwd_args& a, hipStream_t stream) {
  const unsigned items = static_cast<unsigned>(a.fwd.B) * a.fwd.N * a.fwd.H;
  const unsigned wgs = gate_bwd_wgs(a.fwd.H, items);
  float* part = static_cast<float*>(a.workspace);
  hipLaunchKernelGGL(head_gate_bwd_kernel, dim3(wgs), dim3(kBlock), 0, stream, a, items, part);
  hipLaunchKernelGGL(head_gate_gain_kernel, dim3(a.fwd.H), dim3(kBlock), 0, stream, part, wgs * kItems,
                     static_cast<unsigned>(a.fwd.H), a.dgain);
  return hipGetLastError();
}

}  // namespace dwarf
