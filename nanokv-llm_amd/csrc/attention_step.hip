// One layer's call of a step through one entry point: store, then attention. Host code only; a
// step of a few rows is bound by the host, and the separate calls' argument handling
// took longer than their launches.
//
// Reference: Attention.forward, nanokvllm/layers/attention.py:67-108.
#include "nkv_common.h"

extern "C" int nkv_attention(const nkv_attention_args* a) {
  using namespace nkv;
  clear_error();
  NKV_REQUIRE(a, NKV_EINVAL, "attention: null arguments");
  const bool fp8 = a->kv_type == NKV_KV_FP8, f16 = a->kv_type == NKV_KV_F16;
  NKV_REQUIRE(fp8 || f16 || a->kv_type == NKV_KV_BF16, NKV_EINVAL,
              "attention: kv_type %lld is none of NKV_KV_*", (long long)a->kv_type);
  // the 32-bit arguments of the entry points below
  NKV_REQUIRE(a->n_seqs >= 0 && a->max_seqlen_q >= 0 && a->n_q_heads > 0 && a->n_kv_heads > 0 &&
                  a->head_dim > 0 && a->block_size > 0 && a->max_blocks_per_seq >= 0 &&
                  a->n_blocks >= 0 &&
                  (a->n_seqs | a->max_seqlen_q | a->n_q_heads | a->n_kv_heads | a->head_dim |
                   a->block_size | a->max_blocks_per_seq) <= INT32_MAX,
              NKV_EINVAL, "attention: bad sizes");
  const int32_t n_seqs = (int32_t)a->n_seqs, hq = (int32_t)a->n_q_heads;
  const int32_t hk = (int32_t)a->n_kv_heads, d = (int32_t)a->head_dim;
  const int32_t block = (int32_t)a->block_size, width = (int32_t)a->max_blocks_per_seq;
  const int64_t row = a->n_kv_heads * a->head_dim;
  const int64_t n_rows = a->n_blocks * a->block_size;
  const size_t ws_bytes = a->workspace_bytes < 0 ? 0 : (size_t)a->workspace_bytes;
  if (a->decode) {
    const size_t need = nkv_paged_decode_workspace_bytes(n_seqs, hq, d, width, block);
    NKV_REQUIRE(ws_bytes >= need, NKV_EWORKSPACE,
                "attention: the decode workspace needs %zu bytes (got %zu)", need, ws_bytes);
  }
  int rc = fp8 ? nkv_store_kvcache_fp8(a->key, a->key_row_stride, a->value, a->value_row_stride,
                                       a->k_cache, a->v_cache, a->slot_mapping, a->n_tokens, hk,
                                       d, n_rows, (float)a->k_scale, (float)a->v_scale,
                                       a->stream)
               : nkv_store_kvcache(a->key, a->key_row_stride, a->value, a->value_row_stride,
                                   a->k_cache, a->v_cache, a->slot_mapping, a->n_tokens, hk, d,
                                   n_rows, a->stream);
  if (rc) return rc;
  if (a->decode) {
    if (fp8)
      return nkv_paged_decode_fp8(a->q, a->q_row_stride, a->k_cache, a->v_cache, a->block_tables,
                                  a->bt_row_stride, a->cu_or_lens, n_seqs, hq, hk, d, block,
                                  width, a->n_blocks, (float)a->scale, (float)a->k_scale,
                                  (float)a->v_scale, a->out, a->out_row_stride, a->workspace,
                                  ws_bytes, a->stream);
    return (f16 ? nkv_paged_decode_f16 : nkv_paged_decode)(
        a->q, a->q_row_stride, a->k_cache, a->v_cache, a->block_tables, a->bt_row_stride,
        a->cu_or_lens, n_seqs, hq, hk, d, block, width, a->n_blocks, (float)a->scale, a->out,
        a->out_row_stride, a->workspace, ws_bytes, a->stream);
  }
  const int32_t max_q = (int32_t)a->max_seqlen_q;
  return prefill_paged((int32_t)a->kv_type, a->q, a->q_row_stride, a->k_cache, a->v_cache, row,
                       a->cu_or_lens, a->cu_seqlens_k, a->block_tables, a->bt_row_stride, width,
                       n_seqs, a->n_tokens, max_q, hq, hk, d, block, n_rows, (float)a->scale,
                       fp8 ? (float)a->k_scale : 1.f, fp8 ? (float)a->v_scale : 1.f, a->out,
                       a->out_row_stride, a->workspace, ws_bytes, a->stream);
}
