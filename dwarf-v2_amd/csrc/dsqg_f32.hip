// The fp32 DSQG kernels: forward, dQ, the parameter-gradient products and
// dK/dV (reference kernels dsqg:698-860, 863-1044, 1263-1488, 1734-1955, with
// the eager oracle's fp32 numerics).  Device-library exp, log and sincos.
//
// Mapping.  A workgroup of four waves owns 16 consecutive rows (queries, or
// keys in dK/dV) of one (b, h); four lanes share a row, lane g holding dims
// 16 i + 4 g + c (i, c < 4) of it and of every gathered row, so a load
// instruction covers 64 contiguous bytes of 16 rows (16 contiguous dims to a
// lane touch four times the 64-byte segments: forward 631 instead of 460 us,
// dK/dV 500 instead of 435 at B15 H8 T2048).  The four waves hold the same 16
// rows and take every fourth entry of the tile's offset list; their sums (in
// the forward, their running maxima too) are joined through LDS in wave
// order.  Each step's rows are requested two steps ahead, in two register
// buffers.
//
// One sequence of 2,048 tokens and eight heads is 1,024 workgroups: forward
// 40, dQ 68, products and reductions 18, dK/dV 32 us.  Two lanes to a row and
// 128 rows to a workgroup, one row load in flight, took 194, 340, 9.5 and 250
// (128 or 256 workgroups, each walking the whole list); at B15 1,022, 2,098,
// 14 and 1,005 against 460, 857, 74 and 435.  What binds them is the gathered
// rows (512 bytes a pair, 13 TB/s in the forward there) and about 200 VALU
// instructions a step.  Four workgroups per CU in the forward (49 us with
// three); the others need their registers (dQ held to three per CU 88 us,
// dK/dV to four 70).
//
// Rows are addressed with 64-bit offsets from the lane's own row: a lane
// without a source for an entry reads its own row and uses nothing of it.
#include "common.h"
#include "dsqg_internal.h"
#include "gather.h"
#include "mfma.h"

namespace dwarf {
namespace {

constexpr int kRowsF = 16;                   // rows per workgroup
constexpr int kWavesF = kBlock / kWave;
constexpr int kDims = 16;                    // head dims per lane
constexpr int kJoinRow = kHeadDim + 4;       // floats per joined row
constexpr int kListPad = 32;                 // list entries past J: the last step and its prefetches

struct F32Layout {
  int JE, qe_row;
  size_t off_list, off_qe, off_ds, off_ph, off_join, bytes;
};
// [list int2[JE + pad]] [qe[16][qe_row]] [ds[16][qe_row]] [dphase[JL][8]] [join[4][16][kJoinRow]]
__host__ __device__ inline F32Layout f32_layout(int J, int J_large, bool backward) {
  F32Layout L;
  L.JE = (J + 1 + 15) / 16 * 16;
  L.qe_row = L.JE + 4;
  L.off_list = 0;
  L.off_qe = static_cast<size_t>(L.JE + kListPad) * 8;
  L.off_ds = L.off_qe + static_cast<size_t>(kRowsF * L.qe_row) * 4;
  L.off_ph = L.off_ds + (backward ? static_cast<size_t>(kRowsF * L.qe_row) * 4 : 0);
  L.off_join = L.off_ph + (backward ? static_cast<size_t>(J_large) * 2 * kPlanes * 4 : 0);
  L.bytes = L.off_join + static_cast<size_t>(kWavesF * kRowsF * kJoinRow) * 4;
  return L;
}

__device__ __forceinline__ void load16(const float* p, float* x) {
  const float4* v = reinterpret_cast<const float4*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4 w = v[i];
    x[4 * i] = w.x; x[4 * i + 1] = w.y; x[4 * i + 2] = w.z; x[4 * i + 3] = w.w;
  }
}
// A lane's dims of a row whose address is offset by 4 g: x[4 i + c] is dim 16 i + 4 g + c.
__device__ __forceinline__ void load_row(const float* p, float* x) {
  const float4* v = reinterpret_cast<const float4*>(p);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float4 w = v[4 * i];
    x[4 * i] = w.x; x[4 * i + 1] = w.y; x[4 * i + 2] = w.z; x[4 * i + 3] = w.w;
  }
}
__device__ __forceinline__ void join_row(float* p, const float* x) {
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *reinterpret_cast<float4*>(p + 16 * i) = make_float4(x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]);
}
__device__ __forceinline__ float dot16(const float* a, const float* b) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < kDims; ++i) s = fmaf(a[i], b[i], s);
  return group_sum<4>(s);
}

// The tile's offset list, by wave 0 (visible after the caller's barrier).
__device__ __forceinline__ void tile_list(int2* list, int* count, const int* offsets, int J, int lo, int hi, int N,
                                          int dir) {
  if (threadIdx.x >= kWave) return;
  const int l = threadIdx.x;
  int cnt = 0;
  for (int base = 0; base < J; base += kWave) {
    const int j = base + l;
    const int d = j < J ? offsets[j] : 0;
    const int sd = dir * d;
    const bool need = j < J && sd <= hi && sd >= lo - (N - 1);
    const uint64_t mask = __ballot(need);
    const int pos = cnt + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(mask >> 32),
                                                     __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(mask), 0));
    if (need) list[pos] = make_int2(j, d);
    cnt += __popcll(mask);
  }
  // the pad's offset puts every row's partner past N - 1
  for (int t = cnt + l; t < cnt + kListPad; t += kWave) list[t] = make_int2(J, dir * (lo - N));
  if (l == 0) *count = cnt;
}

// E rows as MFMA operand slices: dims [16 c, 16 c + 16) of row j (zeros for j >= J).
__device__ __forceinline__ void load_e16(const dwarf_dsqg_fwd_args& f, int j, int c, bool vec, float* x) {
  const float* p = f.scale_embed + (j < f.J ? j : f.J - 1) * f.se_stride[0] + 16 * c * f.se_stride[1];
  if (vec) {
    load16(p, x);
  } else {
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = p[i * f.se_stride[1]];
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float e = f.se_round_bf16 ? round_bf16(x[i]) : x[i];
    x[i] = j < f.J ? e : 0.f;
  }
}
__device__ __forceinline__ bool e_vec(const dwarf_dsqg_fwd_args& f) {
  return f.se_stride[1] == 1 && (f.se_stride[0] & 3) == 0 && (reinterpret_cast<uintptr_t>(f.scale_embed) & 15) == 0;
}

// s_qe[query][j] = <q, e_j> / 8 + pb_j for the tile's 16 queries and every
// offset, on v_mfma_f32_16x16x4_f32; wave w forms the 16-offset blocks w, w + 4, ...
__device__ __forceinline__ void fill_qe(const dwarf_dsqg_fwd_args& f, const float* qbase, int n0, int h,
                                        const F32Layout& lay, float* s_qe) {
  const int w = threadIdx.x / kWave, l = threadIdx.x % kWave;
  const int lr = l & 15, lc = l >> 4;
  const bool vec = e_vec(f);
  float qa[16];
  load16(qbase + static_cast<int64_t>(min(n0 + lr, f.N - 1)) * f.q_stride[2] + 16 * lc, qa);
  for (int bi = w; bi < lay.JE / 16; bi += kWavesF) {
    const int j = 16 * bi + lr;
    float e[16];
    load_e16(f, j, lc, vec, e);
    const float pb = f.pos_bias[(j < f.J ? j : f.J - 1) * f.pb_stride[0] + h * f.pb_stride[1]];
    f32x4 c = zero4();
#pragma unroll
    for (int i = 0; i < 16; ++i) c = mfma16_f32(qa[i], e[i], c);
#pragma unroll
    for (int r = 0; r < 4; ++r) s_qe[(4 * lc + r) * lay.qe_row + j] = fmaf(c[r], 0.125f, pb);
  }
}

// d rows in elements for a lane with a source, 0 (its own row) for one without; d is uniform, so the product is
// the scalar unit's.
__device__ __forceinline__ int64_t shift_rows(bool ok, int d, int64_t stride) { return ok ? d * stride : 0; }

// One list entry's rows for a lane: K and V (or q and dO), the far pair's z (or y), base and gain.
struct Step {
  float x[kDims], y[kDims];
  float z, base, gain;
  int j;
  bool ok;
};

// MOVT pairs.  Plane r turns dims (16 r + SHIFT, 16 r + SHIFT + 1): element
// SHIFT % 4 of part r of lane SHIFT / 4, and the element after it, which for
// SHIFT % 4 == 3 is the next lane's first.
template <int SHIFT>
struct Pair {
  static constexpr int lane = SHIFT / 4, elem = SHIFT % 4;
  static constexpr bool split = elem == 3;
  // the second element of plane r's pair, in the pair's lane
  static __device__ __forceinline__ float second(const float* x, int r) {
    return split ? dpp_f<0xF9>(x[4 * r]) : x[4 * r + (split ? 0 : elem + 1)];   // quad_perm [1,2,3,3]
  }
  // x's pairs turned by (cos, sn), lane r's angle for plane r; w: the turned pairs, in the pair's lane
  static __device__ __forceinline__ void turn(float* x, float cs, float sn, int g, float (*w)[2]) {
#pragma unroll
    for (int r = 0; r < kPlanes; ++r) {
      const float c = r == 0 ? dpp_f<0x00>(cs) : r == 1 ? dpp_f<0x55>(cs) : r == 2 ? dpp_f<0xAA>(cs) : dpp_f<0xFF>(cs);
      const float s = r == 0 ? dpp_f<0x00>(sn) : r == 1 ? dpp_f<0x55>(sn) : r == 2 ? dpp_f<0xAA>(sn) : dpp_f<0xFF>(sn);
      const float a = x[4 * r + elem], b = second(x, r);
      w[r][0] = c * a - s * b;
      w[r][1] = s * a + c * b;
      x[4 * r + elem] = g == lane ? w[r][0] : a;
      if constexpr (split) {
        const float t = dpp_f<0x90>(w[r][1]);   // quad_perm [0,0,1,2]
        x[4 * r] = g == lane + 1 ? t : x[4 * r];
      } else {
        x[4 * r + elem + 1] = g == lane ? w[r][1] : x[4 * r + elem + 1];
      }
    }
  }
  // plane g's value of four held by the pair's lane
  static __device__ __forceinline__ float plane(const float* t, int g) {
    return pick4(g, dpp_f<lane * 0x55>(t[0]), dpp_f<lane * 0x55>(t[1]), dpp_f<lane * 0x55>(t[2]), dpp_f<lane * 0x55>(t[3]));
  }
};

// This lane's column of a MOVT table; without far offsets (no entry is used) any four floats that exist.
__device__ __forceinline__ const float* plane_column(const dwarf_dsqg_fwd_args& f, const float* table, int64_t head,
                                                     int g) {
  return (f.J_large > 0 ? table + head : f.z_pre) + g;
}

template <int SHIFT, bool TWO_PASS>
__global__ __launch_bounds__(kBlock, 4) void dsqg_f32_fwd(const dwarf_dsqg_fwd_args a, int tiles, int total) {
  constexpr float kSlack = 8.f;   // the running maximum is raised only past this (natural log)
  const int J = a.J, N = a.N, J_small = a.J_small;
  const F32Layout lay = f32_layout(J, a.J_large, false);
  extern __shared__ __align__(16) char f32_smem[];
  int2* s_list = reinterpret_cast<int2*>(f32_smem + lay.off_list);
  float* s_qe = reinterpret_cast<float*>(f32_smem + lay.off_qe);
  float* s_join = reinterpret_cast<float*>(f32_smem + lay.off_join);
  __shared__ int s_cnt;
  __shared__ float2 s_ml[kWavesF][kRowsF];

  const int work = xcd_remap(blockIdx.x, total);
  const int bh = work / tiles;
  const int n0 = (tiles - 1 - (work - bh * tiles)) * kRowsF;   // late tiles (longer lists) first
  const int b = bh / a.H, h = bh - b * a.H, hk = h / (a.H / a.H_kv);
  const int w = uniform(threadIdx.x / kWave), l = threadIdx.x % kWave, g = l & 3, qi = l >> 2;
  const int n = n0 + qi;
  const bool live = n < N && n >= a.query_start;
  const float* qbase = reinterpret_cast<const float*>(a.q) + b * a.q_stride[0] + h * a.q_stride[1];
  const int64_t nc = min(n, N - 1);
  float q[kDims];
  load_row(qbase + nc * a.q_stride[2] + 4 * g, q);
  const float yg = a.y_pre[b * a.y_stride[0] + h * a.y_stride[1] + nc * a.y_stride[2] + g];
  tile_list(s_list, &s_cnt, a.offsets, J, n0, min(n0 + kRowsF - 1, N - 1), N, 1);
  fill_qe(a, qbase, n0, h, lay, s_qe);
  __syncthreads();
  const int cnt = uniform(s_cnt);

  const float* kb = reinterpret_cast<const float*>(a.k) + b * a.k_stride[0] + hk * a.k_stride[1] + nc * a.k_stride[2] + 4 * g;
  const float* vb = reinterpret_cast<const float*>(a.v) + b * a.v_stride[0] + hk * a.v_stride[1] + nc * a.v_stride[2] + 4 * g;
  const float* zb = a.z_pre + b * a.z_stride[0] + hk * a.z_stride[1] + nc * a.z_stride[2] + g;
  const float* pbase = plane_column(a, a.phase_base, h * a.pbase_stride[1], g);
  const float* pgain = plane_column(a, a.phase_gain, h * a.pgain_stride[1], g);
  const float* qe = s_qe + qi * lay.qe_row;
  auto fetch = [&](Step& s, int i, bool values) {
    const int2 e = s_list[w + kWavesF * i];
    const int j = uniform(e.x), d = uniform(e.y), src = n - d;
    s.j = j;
    s.ok = live && src >= 0 && src < N;
    load_row(kb - shift_rows(s.ok, d, a.k_stride[2]), s.x);
    if (values) {
      load_row(vb - shift_rows(s.ok, d, a.v_stride[2]), s.y);
      s.z = *(zb - shift_rows(s.ok, d, a.z_stride[2]));
      const int far = max(0, min(j - J_small, a.J_large - 1));
      s.base = pbase[far * a.pbase_stride[0]];
      s.gain = pgain[far * a.pgain_stride[0]];
    }
  };

  const int steps = (cnt - w + kWavesF - 1) / kWavesF;   // entries w, w + 4, ...
  float acc[kDims];
#pragma unroll
  for (int i = 0; i < kDims; ++i) acc[i] = 0.f;
  float m = -INFINITY, sum = 0.f;
  if constexpr (TWO_PASS) {   // offline softmax (dsqg:863-1044): this wave's maximum first
    Step s0, s1;
    auto top = [&](const Step& s) {
      const float score = fmaf(dot16(q, s.x), 0.125f, qe[s.j]);
      if (s.ok && score > m) m = score;
    };
    if (steps > 0) {
      fetch(s0, 0, false);
      fetch(s1, 1, false);
    }
    for (int i = 0; i < steps; i += 2) {
      top(s0);
      fetch(s0, i + 2, false);
      top(s1);
      fetch(s1, i + 3, false);
    }
  }
  auto use = [&](Step& s) {
    const float score = fmaf(dot16(q, s.x), 0.125f, qe[s.j]);
    if (s.j >= J_small) {   // uniform
      float cs, sn, turned[kPlanes][2];
      sincosf(s.base + s.gain * yg * s.z, &sn, &cs);
      Pair<SHIFT>::turn(s.y, cs, sn, g, turned);
    }
    if (s.ok) {
      if (!TWO_PASS && score > m + kSlack) {
        const float c = expf(m - score);   // 0 on the first entry
#pragma unroll
        for (int i = 0; i < kDims; ++i) acc[i] *= c;
        sum *= c;
        m = score;
      }
      const float p = score == -INFINITY ? 0.f : expf(score - m);
      sum += p;
#pragma unroll
      for (int i = 0; i < kDims; ++i) acc[i] = fmaf(p, s.y[i], acc[i]);
    }
  };
  {
    Step s0, s1;
    if (steps > 0) {
      fetch(s0, 0, true);
      fetch(s1, 1, true);
    }
    for (int i = 0; i < steps; i += 2) {   // an entry past the list is nobody's source
      use(s0);
      fetch(s0, i + 2, true);
      use(s1);
      fetch(s1, i + 3, true);
    }
  }

  // join the four waves: wave w finishes queries 4w .. 4w + 3, 16 lanes to a query
  join_row(s_join + (w * kRowsF + qi) * kJoinRow + 4 * g, acc);
  if (g == 0) s_ml[w][qi] = make_float2(m, sum);
  __syncthreads();
  const int qo = 4 * w + (l >> 4), c4 = 4 * (l & 15);
  if (n0 + qo >= N) return;
  float top = -INFINITY;
#pragma unroll
  for (int u = 0; u < kWavesF; ++u) top = fmaxf(top, s_ml[u][qo].x);
  float o[4] = {0.f, 0.f, 0.f, 0.f}, tot = 0.f;
#pragma unroll
  for (int u = 0; u < kWavesF; ++u) {
    const float2 ml = s_ml[u][qo];
    // a wave that met no finite score holds no weight; NaN and +inf sums pass through
    const float c = ml.x == -INFINITY ? 1.f : expf(ml.x - top);
    const float4 x = *reinterpret_cast<const float4*>(s_join + (u * kRowsF + qo) * kJoinRow + c4);
    tot = fmaf(ml.y, c, tot);
    o[0] = fmaf(x.x, c, o[0]); o[1] = fmaf(x.y, c, o[1]); o[2] = fmaf(x.z, c, o[2]); o[3] = fmaf(x.w, c, o[3]);
  }
  const float inv = tot > 0.f ? 1.f / tot : 0.f;
  float* op = reinterpret_cast<float*>(a.out) + b * a.out_stride[0] + h * a.out_stride[1] +
              static_cast<int64_t>(n0 + qo) * a.out_stride[2] + c4;
  *reinterpret_cast<float4*>(op) = make_float4(o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv);
  if (c4 == 0)
    a.lse[b * a.lse_stride[0] + h * a.lse_stride[1] + static_cast<int64_t>(n0 + qo) * a.lse_stride[2]] =
        tot > 0.f ? top + logf(tot) : -INFINITY;
}

// dQ, dY, dPhase partials and the P and dS matrices [b, h][j][NP] (NP: N
// rounded up to whole 64-row tiles; only pairs with a source are written).  A
// workgroup walks tpw consecutive tiles of one (b, h) and keeps its dPhase
// sums in LDS; entry j belongs to one wave per tile and tiles are separated by
// barriers, so the order of every sum is fixed.  dQ's e_j part is dS E on
// v_mfma_f32_16x16x4_f32 from the tile's dS in LDS, wave w forming dims
// [16w, 16w + 16).
template <int SHIFT>
__global__ __launch_bounds__(kBlock) void dsqg_f32_dq(const dwarf_dsqg_bwd_args a, float* __restrict__ ds_ws,
                                                      float* __restrict__ p_ws, float* __restrict__ part_ph, int tiles,
                                                      int tpw, int n_tg, int NP, int total) {
  const dwarf_dsqg_fwd_args& f = a.fwd;
  const int J = f.J, N = f.N, J_small = f.J_small, JL = f.J_large;
  const F32Layout lay = f32_layout(J, JL, true);
  extern __shared__ __align__(16) char f32_smem[];
  int2* s_list = reinterpret_cast<int2*>(f32_smem + lay.off_list);
  float* s_qe = reinterpret_cast<float*>(f32_smem + lay.off_qe);
  float* s_ds = reinterpret_cast<float*>(f32_smem + lay.off_ds);
  float* s_ph = reinterpret_cast<float*>(f32_smem + lay.off_ph);
  float* s_join = reinterpret_cast<float*>(f32_smem + lay.off_join);
  __shared__ int s_cnt;
  __shared__ float s_dy[kWavesF][kRowsF][kPlanes];

  const int work = xcd_remap(blockIdx.x, total);
  const int bh = work / n_tg;
  const int tg = work - bh * n_tg;
  const int b = bh / f.H, h = bh - b * f.H, hk = h / (f.H / f.H_kv);
  const int w = uniform(threadIdx.x / kWave), l = threadIdx.x % kWave, g = l & 3, qi = l >> 2;
  const int lr = l & 15, lc = l >> 4;
  const float* qbase = reinterpret_cast<const float*>(f.q) + b * f.q_stride[0] + h * f.q_stride[1];
  const float* dobase = reinterpret_cast<const float*>(a.dout) + b * a.dout_stride[0] + h * a.dout_stride[1] + 4 * g;
  const float* obase = reinterpret_cast<const float*>(f.out) + b * f.out_stride[0] + h * f.out_stride[1] + 4 * g;
  const float* kbase = reinterpret_cast<const float*>(f.k) + b * f.k_stride[0] + hk * f.k_stride[1] + 4 * g;
  const float* vbase = reinterpret_cast<const float*>(f.v) + b * f.v_stride[0] + hk * f.v_stride[1] + 4 * g;
  const float* zbase = f.z_pre + b * f.z_stride[0] + hk * f.z_stride[1] + g;
  const float* pbase = plane_column(f, f.phase_base, h * f.pbase_stride[1], g);
  const float* pgain = plane_column(f, f.phase_gain, h * f.pgain_stride[1], g);
  const int64_t mat = static_cast<int64_t>(bh) * J * NP;

  for (int i = threadIdx.x; i < JL * 2 * kPlanes; i += kBlock) s_ph[i] = 0.f;
  for (int t = tg * tpw; t < min((tg + 1) * tpw, tiles); ++t) {
    const int n0 = t * kRowsF, n = n0 + qi;
    const bool live = n < N && n >= f.query_start;
    const int64_t nc = min(n, N - 1);
    __syncthreads();   // the previous tile's tables have been read, s_ph is cleared
    tile_list(s_list, &s_cnt, f.offsets, J, n0, min(n0 + kRowsF - 1, N - 1), N, 1);
    float q[kDims], go[kDims], o[kDims];
    load_row(qbase + nc * f.q_stride[2] + 4 * g, q);
    load_row(dobase + nc * a.dout_stride[2], go);
    load_row(obase + nc * f.out_stride[2], o);
    const float yg = f.y_pre[b * f.y_stride[0] + h * f.y_stride[1] + nc * f.y_stride[2] + g];
    const float lse = f.lse[b * f.lse_stride[0] + h * f.lse_stride[1] + nc * f.lse_stride[2]];
    const bool mass = live && lse > -INFINITY;
    for (int i = threadIdx.x; i < kRowsF * lay.qe_row; i += kBlock) s_ds[i] = 0.f;
    fill_qe(f, qbase, n0, h, lay, s_qe);
    const float delta = dot16(go, o);
    __syncthreads();
    const int cnt = uniform(s_cnt);
    const int steps = (cnt - w + kWavesF - 1) / kWavesF;
    const float *kb = kbase + nc * f.k_stride[2], *vb = vbase + nc * f.v_stride[2], *zb = zbase + nc * f.z_stride[2];
    float *pcol = p_ws + mat + nc, *dscol = ds_ws + mat + nc;
    const float* qe = s_qe + qi * lay.qe_row;
    float* dsr = s_ds + qi * lay.qe_row;
    float gob[kPlanes];   // the second element of dO's pairs
#pragma unroll
    for (int r = 0; r < kPlanes; ++r) gob[r] = Pair<SHIFT>::second(go, r);
    float dq[kDims], dy = 0.f;
#pragma unroll
    for (int i = 0; i < kDims; ++i) dq[i] = 0.f;
    auto fetch = [&](Step& s, int i) {
      const int2 e = s_list[w + kWavesF * i];
      const int j = uniform(e.x), d = uniform(e.y), src = n - d;
      s.j = j;
      s.ok = n < N && src >= 0 && src < N;
      load_row(kb - shift_rows(s.ok, d, f.k_stride[2]), s.x);
      load_row(vb - shift_rows(s.ok, d, f.v_stride[2]), s.y);
      s.z = *(zb - shift_rows(s.ok, d, f.z_stride[2]));
      const int far = max(0, min(j - J_small, JL - 1));
      s.base = pbase[far * f.pbase_stride[0]];
      s.gain = pgain[far * f.pgain_stride[0]];
    };
    auto use = [&](Step& s) {
      const float score = fmaf(dot16(q, s.x), 0.125f, qe[s.j]);
      float turn = 0.f;   // plane g's dO . d(R v) / dtheta
      if (s.j >= J_small) {   // uniform
        float cs, sn, wv[kPlanes][2], t[kPlanes];
        sincosf(s.base + s.gain * yg * s.z, &sn, &cs);
        Pair<SHIFT>::turn(s.y, cs, sn, g, wv);
#pragma unroll
        for (int r = 0; r < kPlanes; ++r) t[r] = gob[r] * wv[r][0] - go[4 * r + Pair<SHIFT>::elem] * wv[r][1];
        turn = Pair<SHIFT>::plane(t, g);
      }
      const float gd = dot16(go, s.y);
      float dth = 0.f, ds = 0.f, p = 0.f;
      if (s.ok && mass) {
        p = expf(score - lse);
        ds = p * (gd - delta);
        const float c = 0.125f * ds;
#pragma unroll
        for (int i = 0; i < kDims; ++i) dq[i] = fmaf(c, s.x[i], dq[i]);
        dth = p * turn;
      }
      // P from lane 0 and dS from lane 1 of each query; dS stays in LDS for the e_j part
      if (s.ok && g < 2) (g == 0 ? pcol : dscol)[static_cast<int64_t>(s.j) * NP] = g == 0 ? p : ds;
      if (s.ok && g == 2) dsr[s.j] = ds;
      if (s.j >= J_small && s.j < J) {   // uniform
        const float yz = s.ok && mass ? yg * s.z : 0.f;   // nothing of a row that is no source
        if (s.ok && mass) dy = fmaf(dth * s.gain, s.z, dy);
        const float db = sum_over_queries16(dth), dg = sum_over_queries16(dth * yz);
        if (l < kPlanes) {
          float* ph = s_ph + (s.j - J_small) * 2 * kPlanes + 2 * l;
          ph[0] += db;
          ph[1] += dg;
        }
      }
    };
    {
      Step s0, s1;
      if (steps > 0) {
        fetch(s0, 0);
        fetch(s1, 1);
      }
      for (int i = 0; i < steps; i += 2) {
        use(s0);
        fetch(s0, i + 2);
        use(s1);
        fetch(s1, i + 3);
      }
    }
    join_row(s_join + (w * kRowsF + qi) * kJoinRow + 4 * g, dq);
    s_dy[w][qi][g] = dy;
    __syncthreads();
    // wave w: dims [16w, 16w + 16) of every query, lane (lr, lc) dim 16w + lr of queries 4 lc + r
    f32x4 c = zero4();
    for (int j0 = lc; j0 < lay.JE; j0 += 16) {
      float e[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int j = j0 + 4 * u;
        e[u] = f.scale_embed[(j < J ? j : J - 1) * f.se_stride[0] + (16 * w + lr) * f.se_stride[1]];
        if (f.se_round_bf16) e[u] = round_bf16(e[u]);
        if (j >= J) e[u] = 0.f;
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) c = mfma16_f32(s_ds[lr * lay.qe_row + j0 + 4 * u], e[u], c);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int qo = 4 * lc + r;
      float x = 0.125f * c[r];
#pragma unroll
      for (int u = 0; u < kWavesF; ++u) x += s_join[(u * kRowsF + qo) * kJoinRow + 16 * w + lr];
      if (n0 + qo < N)
        reinterpret_cast<float*>(a.dq)[b * a.dq_stride[0] + h * a.dq_stride[1] +
                                       static_cast<int64_t>(n0 + qo) * a.dq_stride[2] + 16 * w + lr] = x;
    }
    if (threadIdx.x < kRowsF * kPlanes && n < N)   // wave 0: lane (qi, g)
      a.dy_pre[(static_cast<int64_t>(bh) * N + n) * kPlanes + g] =
          (s_dy[0][qi][g] + s_dy[1][qi][g]) + (s_dy[2][qi][g] + s_dy[3][qi][g]);
  }
  __syncthreads();
  float* ph = part_ph + static_cast<int64_t>((h * f.B + b) * n_tg + tg) * JL * 2 * kPlanes;   // head-major partial row
  for (int i = threadIdx.x; i < JL * 2 * kPlanes; i += kBlock) ph[i] = s_ph[i];
}

// dSE = dS^T Q / 8 and dPB = dS^T 1 from the dS matrix on
// v_mfma_f32_16x16x4_f32: a workgroup walks tpw consecutive 64-query tiles of
// one (b, h) with its sums in registers, wave w the 16-offset blocks w, w + 4,
// ... (MB of them) against all 64 dims of the q tile in LDS.  k runs over the
// tile's queries in the order 16 lc + i, so a lane's dS are four 16-byte
// loads.  Entries of pairs without a source were not written and count as 0.
template <int MB>
__global__ __launch_bounds__(kBlock) void dsqg_f32_dse(const dwarf_dsqg_bwd_args a, const float* __restrict__ ds_ws,
                                                       float* __restrict__ part_se, float* __restrict__ part_pb,
                                                       int tiles, int tpw, int n_tg, int NP) {
  constexpr int kRow = 65;   // 16 kRow = 16 (mod 64): the four k groups read different banks
  __shared__ float s_q[64 * kRow];
  const dwarf_dsqg_fwd_args& f = a.fwd;
  const int J = f.J, N = f.N;
  const int bh = blockIdx.x / n_tg, tg = blockIdx.x - bh * n_tg;
  const int b = bh / f.H, h = bh - b * f.H;
  const int w = threadIdx.x / kWave, l = threadIdx.x % kWave, lr = l & 15, lc = l >> 4;
  const int slot = (h * f.B + b) * n_tg + tg;
  const float* qbase = reinterpret_cast<const float*>(f.q) + b * f.q_stride[0] + h * f.q_stride[1];
  const float* lbase = f.lse + b * f.lse_stride[0] + h * f.lse_stride[1];
  f32x4 acc[MB][4];
  float pb[MB];
  int off[MB];
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int j = 16 * (w + kWavesF * m) + lr;
    off[m] = j < J ? f.offsets[j] : 0;
    pb[m] = 0.f;
#pragma unroll
    for (int d = 0; d < 4; ++d) acc[m][d] = zero4();
  }
  for (int t = tg * tpw; t < min((tg + 1) * tpw, tiles); ++t) {
    const int n0 = 64 * t;
    float x[MB][16];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const int j = 16 * (w + kWavesF * m) + lr;
      load16(ds_ws + (static_cast<int64_t>(bh) * J + (j < J ? j : J - 1)) * NP + n0 + 16 * lc, x[m]);
    }
    // q as zeros for a row without mass: its dS are zeros, which do not keep a NaN or inf out of the products
    constexpr int kQRows = 64 * 16 / kBlock;   // row pieces per thread
    float4 qv[kQRows];
    bool mass[kQRows];
#pragma unroll
    for (int u = 0; u < kQRows; ++u) {
      const int n = n0 + (threadIdx.x >> 4) + u * (kBlock / 16);
      const int64_t nc = min(n, N - 1);
      qv[u] = *reinterpret_cast<const float4*>(qbase + nc * f.q_stride[2] + 4 * (threadIdx.x & 15));
      mass[u] = n < N && n >= f.query_start && lbase[nc * f.lse_stride[2]] > -INFINITY;
    }
    __syncthreads();   // the previous tile's q has been read
#pragma unroll
    for (int u = 0; u < kQRows; ++u) {
      float* d = s_q + ((threadIdx.x >> 4) + u * (kBlock / 16)) * kRow + 4 * (threadIdx.x & 15);
      d[0] = mass[u] ? qv[u].x : 0.f; d[1] = mass[u] ? qv[u].y : 0.f;
      d[2] = mass[u] ? qv[u].z : 0.f; d[3] = mass[u] ? qv[u].w : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const bool has = 16 * (w + kWavesF * m) + lr < J;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int n = n0 + 16 * lc + i, src = n - off[m];
        x[m][i] = has && n < N && src >= 0 && src < N ? x[m][i] : 0.f;
        pb[m] += x[m][i];
      }
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const float qv = s_q[(16 * lc + i) * kRow + 16 * d + lr];
#pragma unroll
        for (int m = 0; m < MB; ++m) acc[m][d] = mfma16_f32(x[m][i], qv, acc[m][d]);
      }
    }
  }
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int j0 = 16 * (w + kWavesF * m);
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (j0 + 4 * lc + r < J)
          part_se[(static_cast<int64_t>(slot) * J + j0 + 4 * lc + r) * kHeadDim + 16 * d + lr] = 0.125f * acc[m][d][r];
    const float s = add_xor32(add_xor16(pb[m]));
    if (lc == 0 && j0 + lr < J) part_pb[static_cast<int64_t>(slot) * J + j0 + lr] = s;
  }
}

// dK, dV and dZ, key-centric, from the P and dS matrices the dQ launch wrote:
// per pair the q and dO rows, dK += dS q / 8, dV += P R^T dO, and dZ from the
// angle's derivative P (v_a (R^T dO)_b - v_b (R^T dO)_a).  No score is formed
// again.  The waves share the (query head, offset) entries of the KV head's
// group; their sums are joined in wave order.
template <int SHIFT>
__global__ __launch_bounds__(kBlock) void dsqg_f32_dkdv(const dwarf_dsqg_bwd_args a, const float* __restrict__ ds_ws,
                                                        const float* __restrict__ p_ws, int tiles, int NP, int total) {
  const dwarf_dsqg_fwd_args& f = a.fwd;
  const int J = f.J, N = f.N, J_small = f.J_small;
  extern __shared__ __align__(16) char f32_smem[];
  int2* s_list = reinterpret_cast<int2*>(f32_smem);
  __shared__ __align__(16) float s_join[2][kWavesF][kRowsF][kJoinRow];
  __shared__ float s_dz[kWavesF][kRowsF][kPlanes];
  __shared__ int s_cnt;

  const int work = xcd_remap(blockIdx.x, total);
  const int bk = work / tiles;
  const int m0 = (work - bk * tiles) * kRowsF;   // early keys (longer lists) first
  const int b = bk / f.H_kv, hk = bk - b * f.H_kv, group = f.H / f.H_kv;
  const int w = uniform(threadIdx.x / kWave), l = threadIdx.x % kWave, g = l & 3, ki = l >> 2;
  const int m = m0 + ki;
  const int64_t mc = min(m, N - 1);
  const float* vrow = reinterpret_cast<const float*>(f.v) + b * f.v_stride[0] + hk * f.v_stride[1] + mc * f.v_stride[2];
  float va[kPlanes], vv[kPlanes];
#pragma unroll
  for (int r = 0; r < kPlanes; ++r) {
    va[r] = vrow[16 * r + SHIFT];
    vv[r] = vrow[16 * r + SHIFT + 1];
  }
  const float zg = f.z_pre[b * f.z_stride[0] + hk * f.z_stride[1] + mc * f.z_stride[2] + g];
  tile_list(s_list, &s_cnt, f.offsets, J, m0, min(m0 + kRowsF - 1, N - 1), N, -1);
  __syncthreads();
  const int cnt = uniform(s_cnt);
  const int steps = (cnt - w + kWavesF - 1) / kWavesF;
  float dk[kDims], dv[kDims], dz = 0.f;
#pragma unroll
  for (int i = 0; i < kDims; ++i) dk[i] = dv[i] = 0.f;

  for (int h = hk * group; h < (hk + 1) * group; ++h) {
    const float* qb = reinterpret_cast<const float*>(f.q) + b * f.q_stride[0] + h * f.q_stride[1] + mc * f.q_stride[2] + 4 * g;
    const float* dob = reinterpret_cast<const float*>(a.dout) + b * a.dout_stride[0] + h * a.dout_stride[1] +
                       mc * a.dout_stride[2] + 4 * g;
    const float* yb = f.y_pre + b * f.y_stride[0] + h * f.y_stride[1] + mc * f.y_stride[2] + g;
    const float* pbase = plane_column(f, f.phase_base, h * f.pbase_stride[1], g);
    const float* pgain = plane_column(f, f.phase_gain, h * f.pgain_stride[1], g);
    const int64_t mat = static_cast<int64_t>(b * f.H + h) * J * NP + mc;
    struct KvStep : Step {
      float p, ds;
    };
    auto fetch = [&](KvStep& s, int i) {
      const int2 e = s_list[w + kWavesF * i];
      const int j = uniform(e.x), d = uniform(e.y), nq = m + d;
      s.j = j;
      s.ok = m < N && nq >= 0 && nq < N;
      load_row(qb + shift_rows(s.ok, d, f.q_stride[2]), s.x);
      load_row(dob + shift_rows(s.ok, d, a.dout_stride[2]), s.y);
      s.z = *(yb + shift_rows(s.ok, d, f.y_stride[2]));
      const int far = max(0, min(j - J_small, f.J_large - 1));
      s.base = pbase[far * f.pbase_stride[0]];
      s.gain = pgain[far * f.pgain_stride[0]];
      const int64_t at = mat + static_cast<int64_t>(min(j, J - 1)) * NP + (s.ok ? d : 0);
      s.p = p_ws[at];
      s.ds = ds_ws[at];
    };
    auto use = [&](KvStep& s) {
      float turn = 0.f;
      if (s.j >= J_small) {   // uniform; R^T turns dO back
        float cs, sn, wv[kPlanes][2], t[kPlanes];
        sincosf(s.base + s.gain * s.z * zg, &sn, &cs);
        Pair<SHIFT>::turn(s.y, cs, -sn, g, wv);
#pragma unroll
        for (int r = 0; r < kPlanes; ++r) t[r] = va[r] * wv[r][1] - vv[r] * wv[r][0];
        turn = Pair<SHIFT>::plane(t, g);
      }
      // a query without mass has P = dS = 0, and nothing of its rows may pass (0 times a NaN or inf is NaN); where a
      // query with mass has both, its terms are zeros
      if (s.ok && ((__float_as_uint(s.p) | __float_as_uint(s.ds)) << 1) != 0u) {
        const float c = 0.125f * s.ds;
#pragma unroll
        for (int i = 0; i < kDims; ++i) {
          dk[i] = fmaf(c, s.x[i], dk[i]);
          dv[i] = fmaf(s.p, s.y[i], dv[i]);
        }
        if (s.j >= J_small) dz = fmaf(s.p * turn * s.gain, s.z, dz);
      }
    };
    KvStep s0, s1;
    if (steps > 0) {
      fetch(s0, 0);
      fetch(s1, 1);
    }
    for (int i = 0; i < steps; i += 2) {
      use(s0);
      fetch(s0, i + 2);
      use(s1);
      fetch(s1, i + 3);
    }
  }
  join_row(&s_join[0][w][ki][4 * g], dk);
  join_row(&s_join[1][w][ki][4 * g], dv);
  s_dz[w][ki][g] = dz;
  __syncthreads();
  const int ko = 4 * w + (l >> 4), c4 = 4 * (l & 15);
  const int64_t mo = m0 + ko;
  if (mo < N) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
      for (int u = 0; u < kWavesF; ++u) {
        const float4 x = *reinterpret_cast<const float4*>(&s_join[t][u][ko][c4]);
        s.x += x.x; s.y += x.y; s.z += x.z; s.w += x.w;
      }
      float* dst = t == 0 ? reinterpret_cast<float*>(a.dk) + b * a.dk_stride[0] + hk * a.dk_stride[1] + mo * a.dk_stride[2]
                          : reinterpret_cast<float*>(a.dv) + b * a.dv_stride[0] + hk * a.dv_stride[1] + mo * a.dv_stride[2];
      *reinterpret_cast<float4*>(dst + c4) = s;
    }
  }
  if (threadIdx.x < kRowsF * kPlanes && m < N)
    a.dz_pre[(static_cast<int64_t>(bk) * N + m) * kPlanes + g] =
        (s_dz[0][ki][g] + s_dz[1][ki][g]) + (s_dz[2][ki][g] + s_dz[3][ki][g]);
}

#define DWARF_F32_SHIFTS(X) X(0) X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12) X(13) X(14)

template <bool TWO_PASS>
hipError_t launch_fwd(const dwarf_dsqg_fwd_args& a, hipStream_t stream) {
  const int tiles = (a.N + kRowsF - 1) / kRowsF;
  const int total = tiles * a.B * a.H;
  const size_t lds = f32_layout(a.J, a.J_large, false).bytes;
  switch (a.plane_shift) {
#define DWARF_CASE(S)                                                                                              \
  case S:                                                                                                          \
    hipLaunchKernelGGL((dsqg_f32_fwd<S, TWO_PASS>), dim3(total), dim3(kBlock), lds, stream, a, tiles, total); break;
    DWARF_F32_SHIFTS(DWARF_CASE)
#undef DWARF_CASE
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace

F32Plan f32_plan(const dwarf_dsqg_fwd_args& f) {
  F32Plan p;
  const int64_t bh = static_cast<int64_t>(f.B) * f.H;
  // tiles per workgroup: whole (b, h) rows of tiles share a workgroup's dPhase (dSE) sums once there are enough
  // workgroups to fill the chip without sharing (2,048: eight per CU; 512 for the products, whose slots are J x 64)
  auto per = [&](int tiles, int64_t wgs) {
    const int64_t t = (tiles * bh + wgs - 1) / wgs;
    return static_cast<int>(t < 1 ? 1 : (t < tiles ? t : (tiles > 0 ? tiles : 1)));
  };
  p.dq_tiles = (f.N + kRowsF - 1) / kRowsF;
  p.dq_tpw = per(p.dq_tiles, 2048);
  p.dq_ntg = (p.dq_tiles + p.dq_tpw - 1) / p.dq_tpw;
  p.se_tiles = (f.N + 63) / 64;
  p.se_tpw = per(p.se_tiles, 512);
  p.se_ntg = (p.se_tiles + p.se_tpw - 1) / p.se_tpw;
  p.np = 64 * p.se_tiles;
  return p;
}

hipError_t launch_f32_fwd(const dwarf_dsqg_fwd_args& a, hipStream_t stream) {
  return (a.schedule & DWARF_SCHED_TWO_PASS) ? launch_fwd<true>(a, stream) : launch_fwd<false>(a, stream);
}

hipError_t launch_f32_dq(const dwarf_dsqg_bwd_args& a, const BwdWorkspace& ws, hipStream_t stream) {
  const dwarf_dsqg_fwd_args& f = a.fwd;
  const F32Plan p = f32_plan(f);
  const int total = p.dq_ntg * f.B * f.H;
  char* base = static_cast<char*>(a.workspace);
  float* ds = reinterpret_cast<float*>(base + ws.ds_off);
  float* pm = ds + static_cast<size_t>(f.B) * f.H * f.J * p.np;
  float* ph = reinterpret_cast<float*>(base + ws.part_ph_off);
  const size_t lds = f32_layout(f.J, f.J_large, true).bytes;
  switch (f.plane_shift) {
#define DWARF_CASE(S)                                                                                              \
  case S:                                                                                                          \
    hipLaunchKernelGGL((dsqg_f32_dq<S>), dim3(total), dim3(kBlock), lds, stream, a, ds, pm, ph, p.dq_tiles,        \
                       p.dq_tpw, p.dq_ntg, p.np, total);                                                           \
    break;
    DWARF_F32_SHIFTS(DWARF_CASE)
#undef DWARF_CASE
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_f32_dse(const dwarf_dsqg_bwd_args& a, const BwdWorkspace& ws, hipStream_t stream) {
  const dwarf_dsqg_fwd_args& f = a.fwd;
  const F32Plan p = f32_plan(f);
  char* base = static_cast<char*>(a.workspace);
  const float* ds = reinterpret_cast<const float*>(base + ws.ds_off);
  float* se = reinterpret_cast<float*>(base + ws.part_se_off);
  float* pb = reinterpret_cast<float*>(base + ws.part_pb_off);
  const dim3 grid(p.se_ntg * f.B * f.H);
  if (f.J <= 2 * 16 * kWavesF)
    hipLaunchKernelGGL(dsqg_f32_dse<2>, grid, dim3(kBlock), 0, stream, a, ds, se, pb, p.se_tiles, p.se_tpw, p.se_ntg, p.np);
  else
    hipLaunchKernelGGL(dsqg_f32_dse<4>, grid, dim3(kBlock), 0, stream, a, ds, se, pb, p.se_tiles, p.se_tpw, p.se_ntg, p.np);
  return hipGetLastError();
}

hipError_t launch_f32_dkdv(const dwarf_dsqg_bwd_args& a, const BwdWorkspace& ws, hipStream_t stream) {
  const dwarf_dsqg_fwd_args& f = a.fwd;
  const F32Plan p = f32_plan(f);
  const int tiles = (f.N + kRowsF - 1) / kRowsF;
  const int total = tiles * f.B * f.H_kv;
  const float* ds = reinterpret_cast<const float*>(static_cast<char*>(a.workspace) + ws.ds_off);
  const float* pm = ds + static_cast<size_t>(f.B) * f.H * f.J * p.np;
  const size_t lds = static_cast<size_t>(f.J + kListPad) * 8;
  switch (f.plane_shift) {
#define DWARF_CASE(S)                                                                                              \
  case S:                                                                                                          \
    hipLaunchKernelGGL((dsqg_f32_dkdv<S>), dim3(total), dim3(kBlock), lds, stream, a, ds, pm, tiles, p.np, total); break;
    DWARF_F32_SHIFTS(DWARF_CASE)
#undef DWARF_CASE
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace dwarf
