// Shared between the Chord attention translation units.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "common.h"

namespace motif {

struct ChordArgs {
  const void *q; int64_t q_sb, q_sh, q_st;
  const void *k; int64_t k_sb, k_sh, k_st;
  const void *v; int64_t v_sb, v_sh, v_st;
  const float *alpha, *beta, *mu, *ssmax;
  const float *log_n; int64_t ln_sb, ln_st;
  void *out; int64_t o_sb, o_sh, o_st;
  float *lse;
  int B, H, Hkv, L, S, q_start;
  float scale, eps;
  const int32_t *cu;  // packed sequences (B == 1) or nullptr
  // split-K partials
  float *part;        // [B][Hkv][splits][L * group][D + 2]
  int splits;         // key-range splits (decode kernel)
  int nqc;            // row chunks per (batch, kv head) (decode kernel)
  // device cursor (decode kernels): when set, *len_dev positions are cached, the L
  // new keys sit at [*len_dev, *len_dev + L), S holds the cache capacity, and the
  // merge pass advances *len_dev by L
  int *len_dev;
  const float *log_tab;  // ln(1 .. n) when log_n is NULL: log_n[b, i] = log_tab[q_start + i]
};

__device__ __forceinline__ float ggd_bias(float dist, float alpha, float beta, float mu, float eps) {
  // -alpha * (|d - mu| + eps)^beta, the power through exp2(beta * log2(.)).
  const float x = fabsf(dist - mu) + eps;
  return -alpha * fast_exp2(beta * fast_log2(x));
}

// The fp32-accumulating flash kernel (chord_wide.hip) for what the bf16 head-dim-64 kernel does
// not take: fp32, fp16 and bf16 at head dims 16, 32, 64, 128, padded batches.
bool chord_wide_serves(const ChordArgs &a);
int launch_chord_wide(const ChordArgs &a, int dtype, int D, hipStream_t s);

// Chord decode over a device cursor, shared by the C-ABI entry points that take
// a caller workspace and those that use the library's own scratch.
// The body of motif_chord_decode (same arguments and status codes).
int chord_decode_run(
    const void *q, int64_t q_sb, int64_t q_sh, int64_t q_st,
    const void *k_cache, int64_t k_sb, int64_t k_sh, int64_t k_st,
    const void *v_cache, int64_t v_sb, int64_t v_sh, int64_t v_st,
    int *length_dev, int capacity,
    const float *alpha, const float *beta, const float *mu, const float *ssmax,
    const float *log_n, int64_t ln_sb, int64_t ln_st, const float *log_table, int log_table_len,
    void *out, int64_t o_sb, int64_t o_sh, int64_t o_st,
    int B, int H, int Hkv, int L, int D, float scale, float eps,
    void *workspace, size_t workspace_bytes, int dtype, void *stream);

}  // namespace motif
