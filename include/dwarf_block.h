/*
 * Entry points for the DSQG block around the attention op (libdwarf_dsqg.so,
 * gfx950): the normalised phase probes, the backward's two streams in one
 * call, the per-head gain and content gate after the attention, forward and
 * backward, and the projections' weight gradients.  Conventions (status
 * codes, strides in elements, dwarf_stream_t) are those of dwarf_dsqg.h.
 */
#ifndef DWARF_BLOCK_H
#define DWARF_BLOCK_H

#include "dwarf_dsqg.h"

#ifdef __cplusplus
extern "C" {
#endif

/*
 * out [2][4][64]: the rows of query_probes and key_probes (fp32 [4,64], contiguous) over max(norm, 1e-12)
 * (dsqg:3231-3232).
 */
int dwarf_normalize_probes(const float* query_probes, const float* key_probes, float* out, dwarf_stream_t stream);

/*
 * The bf16 backward's stages on two streams: dq and params on `stream`, delta (left out where pairs_ready says
 * that the workspace already holds the pairs, written on `stream`) and dkdv on `side`, which starts after what
 * `stream` held before the call; `stream` then waits for `side`, also where a stage fails, so nothing that
 * later work on `stream` reuses is still in use on `side`.  args->fwd.schedule holds DWARF_SCHED_DELTA_STAGE.
 */
int dwarf_dsqg_bwd_two_streams(const dwarf_dsqg_bwd_args* args, int32_t pairs_ready, dwarf_stream_t stream,
                               dwarf_stream_t side);

/*
 * The weight and bias gradients of y = x W^T + b over M rows: dw[o][i] = sum_m dy[m][o] x[m][i] and
 * db[o] = sum_m dy[m][o], fp32 sums in a fixed order.  dy [M,O] and x [M,I] bf16, unit column stride, row strides
 * in elements; O, I and the strides multiples of 8, rows 16-byte aligned; dw [O,I] and db [O] (may be NULL) fp32,
 * contiguous, 16-byte aligned.
 */
typedef struct {
  int64_t M;
  int32_t O, I;
  const void* dy; int64_t dy_stride;
  const void* x; int64_t x_stride;
  float* dw;
  float* db;
  void* workspace; size_t workspace_bytes;   /* 16-byte aligned */
} dwarf_linear_wgrad_args;

size_t dwarf_linear_wgrad_workspace_bytes(const dwarf_linear_wgrad_args* args);
int dwarf_linear_wgrad(const dwarf_linear_wgrad_args* args, dwarf_stream_t stream);

/*
 * gated[b,n,h*64+d] = bf16((out[b,h,n,d] * gain[h]) * bf16(sigmoid(gate[b,n,h*64+d]))), the products in
 * fp32: the block's if_gain and content gate (dsqg:3278-3284) under bf16 autocast.  out [B,H,N,64], gate and
 * gated [B,N,H*64], all bf16 with unit last stride and 16-byte aligned rows; gain [H] fp32.
 */
typedef struct {
  int32_t B, H, N;
  const void* out; int64_t out_stride[4];
  const float* gain;
  const void* gate; int64_t gate_stride[3];
  void* gated; int64_t gated_stride[3];
} dwarf_head_gate_fwd_args;

int dwarf_head_gate_fwd(const dwarf_head_gate_fwd_args* args, dwarf_stream_t stream);

/*
 * The gradients of that expression: with s = bf16(sigmoid(gate)) and dm = dgated * s, dout = bf16(dm * gain),
 * dgate = bf16(bf16(dgated * out * gain) * (1 - s) * s) and dgain[h] = sum of dm * out in fp32 in a fixed
 * order, rounded where autograd rounds them but for dgate, whose last product autograd forms from
 * bf16(bf16(...) * (1 - s)).  fwd.gated is not used.
 *
 * delta_pairs (may be NULL): [B,H,N] pairs (sum_d dout * out, lse * log2 e; +inf where lse is -inf or
 * n < query_start), what dwarf_dsqg_bwd_delta writes at the start of the DSQG backward's workspace, summed in
 * its order and so with its bits (before query_start it writes 0, which is this sum over the zero rows of out);
 * a caller that passes the workspace's address here runs its stages under DWARF_SCHED_DELTA_STAGE without that
 * launch.
 * lse [B,H,N] fp32 is read then.
 */
typedef struct {
  dwarf_head_gate_fwd_args fwd;
  const void* dgated; int64_t dgated_stride[3];
  void* dout; int64_t dout_stride[4];
  void* dgate; int64_t dgate_stride[3];
  float* dgain;
  const float* lse; int64_t lse_stride[3];
  int32_t query_start;
  float* delta_pairs;
  void* workspace; size_t workspace_bytes;   /* 16-byte aligned */
} dwarf_head_gate_bwd_args;

size_t dwarf_head_gate_bwd_workspace_bytes(const dwarf_head_gate_bwd_args* args);
int dwarf_head_gate_bwd(const dwarf_head_gate_bwd_args* args, dwarf_stream_t stream);

#ifdef __cplusplus
}
#endif

#endif /* DWARF_BLOCK_H */
