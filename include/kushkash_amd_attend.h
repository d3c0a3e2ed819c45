/* kushkash_amd prefill attention (in kushkash_amd/libkushhip.so, csrc/kush_attend.hip): attention of query
 * rows over key / value rows in fp16 or bf16 on gfx950, with the conventions of kushkash_amd.h (device
 * pointers, hipStream_t as void*, 0 on success, -1 unsupported head_dim or dtype, -2 bad arguments, -3 a HIP
 * error, the message in kush_last_error()).
 */
#ifndef KUSHKASH_AMD_ATTEND_H
#define KUSHKASH_AMD_ATTEND_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Attention of n_seqs sequences' query rows over their keys; q head i reads kv head i / group.
 *
 * dtype 1 fp16, 2 bf16 (q, k, v); out is the same type, or fp32 when out_f32. strides: 15 element strides --
 * (batch, row, head) of q, k, v, out and lse; dims are adjacent. Every pointer and stride of q, k, v and out is a
 * multiple of 16 bytes. lse (optional, fp32): each row's log of the sum of exp(scale q . k).
 * cu_q, cu_k NULL: every sequence has n_q query rows and n_k keys. Else rows are packed end to end,
 * sequence b's at cu_q[b] .. cu_q[b + 1] (keys: cu_k) and n_q / n_k are the longest; total_q query rows in all.
 * causal: query row t of a sequence of T sees keys 0 .. N - T + t (N >= T). scale > 0.
 *
 * waves: 4 (128 query rows, times group heads folded in, per workgroup) or 8 (256; head_dim 64 and 128).
 * chunk: at most this many 64-key tiles per workgroup (0: all of them); a row tile with more keys is split, its
 * partials go to part_o [splits][total_q][hkv * group][head_dim] and part_ml [..][2] (fp32, splits =
 * ceil(ceil(n_k / 64) / chunk)), and a second launch merges them.
 * Contract: the varlen attention of vllm/backend.py:837-880, attention with log-sum-exp _ops.py:254-276. */
int kush_attend(int head_dim, int dtype, const void* q, const void* k, const void* v, void* out, float* lse,
                const int64_t* strides, const int32_t* cu_q, const int32_t* cu_k, int32_t n_q, int32_t n_k,
                int64_t total_q, int32_t n_seqs, int32_t hkv, int32_t group, float scale, int32_t causal,
                int32_t out_f32, int32_t waves, int32_t chunk, float* part_o, float* part_ml, void* stream);

#ifdef __cplusplus
}
#endif

#endif
