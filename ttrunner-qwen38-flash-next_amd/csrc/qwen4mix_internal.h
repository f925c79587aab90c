// Internal declarations shared by the qwen4mix translation units.
#pragma once

#include <stddef.h>

#include "qwen4mix.h"

// Record `msg` as the calling thread's last error and return `code`.
int qm_fail(int code, const char* msg);

inline size_t qm_align256(size_t n) { return (n + 255) & ~static_cast<size_t>(255); }

// Whether na bytes at a and nb bytes at b share memory: a caller may give an
// output the memory of inputs that an entry point is done with, and a path that
// reads them beside its output stores is then not taken.
inline bool qm_overlap(const void* a, size_t na, const void* b, size_t nb) {
  const char* x = static_cast<const char*>(a);
  const char* y = static_cast<const char*>(b);
  return x < y + nb && y < x + na;
}

// The delta-rule token loop over strided q/k/v rows (q/k head h % hk): shared
// by qm_dn_recurrent and the prefill path.
int qm_dn_recurrent_strided(int act_dtype, int batch, int seq, int heads, int hk, long q_stride, long v_stride,
                            const void* q, const void* k, const void* v, const float* g, const float* beta,
                            float* state, void* out, hipStream_t stream);

// The same for a short prefill chunk (1 to QM_DN_SHORT_SEQ tokens) from the raw
// inputs: the conv over [ring | chunk] and the gates are formed in the kernel.
// The ring is read, not written.
constexpr int QM_DN_SHORT_SEQ = 16;
int qm_dn_short(const qm_dn_geom* g, int seq, const void* qkv, const void* a, const void* b, const float* a_neg,
                const float* dt_bias, const void* conv_w, const int* positions, const void* conv_ring, float* state,
                void* out, hipStream_t stream);

// The delta rule over a chunk of tokens for the prefill path: the WY/UT chunked
// kernels (64-token chunks) for chunks of 33 tokens or more, the token loop for
// shorter ones. `ws` holds qm_dn_rule_chunk_workspace(batch, seq, heads) bytes.
size_t qm_dn_rule_chunk_workspace(int batch, int seq, int heads);
int qm_dn_rule_chunk(int act_dtype, int batch, int seq, int heads, int hk, long q_stride, long v_stride,
                     const void* q, const void* k, const void* v, const float* g, const float* beta, float* state,
                     void* out, void* ws, size_t ws_bytes, hipStream_t stream);

// Workgroups of `kernel` (launched with block_threads threads and dyn_lds bytes
// of dynamic LDS) that can be resident on the current device at once: the
// occupancy per compute unit times the compute units. Cached per device.
int qm_resident_workgroups(const void* kernel, int block_threads, size_t dyn_lds, int* out);

// Zero n_words 32-bit words at p with a fill kernel on `stream`.
int qm_zero_words(void* p, long n_words, hipStream_t stream);

// The hyper-connection mix over many token rows on the matrix cores
// (hc_rows.hip): the geometries its kernels cover, the scratch they need, and
// the launches (chosen by as_rows). hyper, norm_w, w_di, w_up, mixed and ws are
// 16-byte aligned.
bool qm_hc_rows_covers(const qm_hc_geom& g);
size_t qm_hc_rows_workspace(const qm_hc_geom& g);
int qm_hc_mix_rows(const qm_hc_geom& g, int as_rows, const void* hyper, const float* norm_w, const void* w_di,
                   int with_inject, const void* w_up, void* mixed, void* inject, void* ws, hipStream_t stream);
