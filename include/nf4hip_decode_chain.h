/* C ABI of libnf4hip_decode.so, second part: a whole decode step in one call.
 *
 * No counterpart in the reference's bitsandbytes path, whose decode step is a graph of launches per layer
 * (thunder/transforms/cudagraph.py:47-226).  Conventions as in nf4hip_decode.h; errors through
 * nf4hip_decode_last_error().
 */
#ifndef NF4HIP_DECODE_CHAIN_H
#define NF4HIP_DECODE_CHAIN_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* A whole single-token step of a Llama decoder with 4-bit linears (NF4, blocksize 64, fp32 absmax, no bias), from the embedded
 * token to the logits, in two launches: every workgroup streams its share of all weights and the workgroups hand the
 * activations of one linear to the next through `workspace`.
 *   x[batch, d_model]   the embedded tokens          out[batch, vocab]  logits
 *   layers              14 device pointers per layer: (codes, absmax, code book[16] fp32) of the QKV projection
 *                       [(n_head + 2 n_kv_head) * 128, d_model], the output projection [d_model, d_model], the gate-up projection
 *                       [2 d_ff, d_model] (rows 2j / 2j+1 = gate j / up j) and the down projection [d_model, d_ff]; then the weight of the
 *                       norm ahead of the MLP and that of the next layer's first norm (the last layer: of the final norm)
 *   head                (codes, absmax, code book) of the output head [vocab, d_model]; norm_first: the first layer's first norm
 *   pos, cos, sin       as for nf4hip_decode_attention (tables [max_seq, 128])
 *   kcache, vcache      [n_layer, batch, n_kv_head, max_seq, 128]; row *pos is written.  *pos outside 0..max_seq-1: nothing is.
 * `layers` and `head` are host arrays and not referred to after the call.  `workspace`: at least
 * nf4hip_decode_chain_workspace_bytes() bytes (0: this shape or device is not served), 16-byte aligned, any contents, this
 * call's alone until it has run.  The workgroups wait for each other, and only for workgroups that are already running: the step ends
 * however few of them the device holds at a time, and those that find a CU later join at the next linear or layer.  max_workgroups > 0: at
 * most so many (a workgroup takes a whole CU; the answer is the same bit for bit).
 *
 * nf4hip_decode_chain_joined: the same with workgroups held back, as other work on the device holds them back by itself:
 * first_members (0: all) of them at most share the first linear, more_members more each one after it. */
size_t nf4hip_decode_chain_workspace_bytes(int64_t batch, int64_t n_layer, int64_t d_model, int n_head, int n_kv_head, int64_t d_ff,
                                           int64_t vocab, int64_t max_seq);
int nf4hip_decode_chain(const void* x, const void* const* layers, const void* const* head, const void* norm_first, float eps,
                        const int64_t* pos, const float* cos, const float* sin, void* kcache, void* vcache, int64_t batch,
                        int64_t n_layer, int64_t d_model, int n_head, int n_kv_head, int64_t d_ff, int64_t vocab, int64_t max_seq,
                        int max_workgroups, void* out, void* workspace, size_t workspace_bytes, void* stream);
int nf4hip_decode_chain_joined(const void* x, const void* const* layers, const void* const* head, const void* norm_first, float eps,
                               const int64_t* pos, const float* cos, const float* sin, void* kcache, void* vcache, int64_t batch,
                               int64_t n_layer, int64_t d_model, int n_head, int n_kv_head, int64_t d_ff, int64_t vocab,
                               int64_t max_seq, int max_workgroups, int first_members, int more_members, void* out,
                               void* workspace, size_t workspace_bytes, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* NF4HIP_DECODE_CHAIN_H */
