// Paged decode attention (one new query token per sequence, GQA) over the
// [num_blocks, block_size, Hk, D] bf16 cache.
//
// Reference: flash_attn_with_kvcache(q.unsqueeze(1), k_cache, v_cache,
// cache_seqlens=context_lens, block_table=block_tables, softmax_scale,
// causal=True) at nanokvllm/layers/attention.py:104-107.
//
// MI355X design (HBM-bound: every K/V byte is read exactly once):
//  * Balanced split-K ("stream-K"): the K/V stream of the batch is cut into
//    16-token chunks ordered (sequence, KV head group, chunk). Persistent
//    one-wave workgroups, as many as are resident at once, each take an equal
//    contiguous range of C chunks, so every wave moves the same number of
//    bytes whatever the context-length mix. A range crosses at most a few
//    (sequence, head group) segments; each segment it touches yields one
//    partial (m, l, O) per query head.
//    A head group is one KV head, or two (HP = 2; four for fp8 rows, HP = 4)
//    whose parts of every token row are read as one contiguous piece.
//  * Within a segment the wave streams chunks through a register ring holding
//    16 KiB of K and V (one chunk of 512-byte rows, two of 256-byte rows): the
//    chunk one ring ahead is issued as soon as the current chunk's rows are
//    staged in LDS, before its products are computed. Loads are
//    non-temporal raw buffer loads whose per-chunk descriptor covers only the
//    chunk's valid rows: keys past the context,
//    padding chunks and invalid block-table entries read as zero without
//    touching memory. Each consumed chunk is staged row-major in LDS.
//  * Both contractions run on the matrix cores:
//      S^T = K q^T   v_mfma_f32_16x16x32_bf16, A = 16 keys (read back from
//                    LDS, one key row per lane), B = the g query heads of the
//                    KV head; lane l ends up with head l%16, keys 4(l/16)..+3.
//      O^T += V^T P^T v_mfma_f32_16x16x16_bf16 per 16-dim block; the B
//                    operand is exactly the lane's 4 softmax weights (bf16),
//                    the A operand V^T comes from LDS with ds_read_b64_tr_b16.
//    Every lane holds state for one head (its column): the online softmax
//    needs no cross-lane traffic except one xor-max over the 4 key groups.
//  * A combine kernel merges the few partials of each (sequence, query head).
// Scores are kept in the log2 domain (scale * log2 e folded in) so the
// exponentials are single v_exp_f32 instructions.
//
// Workspace (caller-owned, sized by what the grid can write, not by the batch
// times the table width): one descriptor per (sequence, KV head) -- first
// partial row, partial count, row stride -- then the partial rows. Within a
// head group, wave wi's partial of sequence b is row wi + b: a segment's
// partials come from consecutive waves, and the next segment's first wave is
// at least its last one, so wi + b never collides and stays below
// waves + batch. A row holds O (D floats), m, l and two pad floats.
//
// head_dim D is 64, 128 or 256 (a template parameter of both kernels).
#include "decode_stream.h"
#include "launch_rules.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace nkv {

template <bool F8, int HP, int D, bool H16 = false>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2)))
void paged_decode_split_kernel(
    const bf16_t* __restrict__ q, int64_t q_row_stride,
    const void* __restrict__ k_cache, const void* __restrict__ v_cache,
    const int32_t* __restrict__ block_tables, int64_t bt_row_stride,
    const int32_t* __restrict__ context_lens, int32_t batch, int32_t Hk, int32_t G,
    int32_t NCG, int32_t block_size, int32_t max_blocks, int64_t n_blocks, int32_t min_chunks,
    float scale_log2, float v_scale, float* __restrict__ part, i32x4v_t* __restrict__ desc) {
  __shared__ __attribute__((aligned(16))) bf16_t lbuf[decode_lds_elems<F8, HP, D>()];
  decode_stream<F8, HP, D, H16>(DecodeSeqs{context_lens, batch}, (int)blockIdx.x,
                                (int)gridDim.x, lbuf, q, q_row_stride, k_cache, v_cache,
                                block_tables, bt_row_stride, Hk, G, NCG, block_size, max_blocks,
                                n_blocks, min_chunks, scale_log2, v_scale, part, desc);
}

// One workgroup (of one wave, or four) per (sequence, query head).
template <int D, bool H16 = false, int WAVES = 1>
__global__ __launch_bounds__(64 * WAVES) void paged_decode_combine_kernel(
    const int32_t* __restrict__ context_lens, int32_t Hq, int32_t Hk, int32_t NCG,
    const float* __restrict__ part, const i32x4v_t* __restrict__ desc,
    bf16_t* __restrict__ out, int64_t out_row_stride) {
  decode_combine<D, H16, WAVES>(DecodeSeqs{context_lens, 0}, (int)blockIdx.x / Hq,
                                (int)blockIdx.x % Hq, Hq, Hk, NCG, part, desc, out,
                                out_row_stride);
}

static int decode_check(const void* q, const void* k_cache, const void* v_cache,
                        const int32_t* block_tables, const int32_t* context_lens, int32_t batch,
                        int32_t n_q_heads, int32_t n_kv_heads, int32_t head_dim,
                        int32_t block_size, int32_t max_blocks_per_seq, int64_t q_row_stride,
                        int64_t bt_row_stride) {
  NKV_REQUIRE(batch >= 0 && n_kv_heads > 0 && n_q_heads > 0, NKV_EINVAL,
              "paged_decode: bad sizes (batch=%d, Hq=%d, Hk=%d)", batch, n_q_heads, n_kv_heads);
  NKV_REQUIRE(decode_dim_ok(head_dim), NKV_EUNSUPPORTED,
              "paged_decode: head_dim must be 64, 128 or 256 (got %d)", head_dim);
  NKV_REQUIRE(n_q_heads % n_kv_heads == 0, NKV_EINVAL,
              "paged_decode: n_q_heads %% n_kv_heads != 0 (%d, %d)", n_q_heads, n_kv_heads);
  const int g = n_q_heads / n_kv_heads;
  NKV_REQUIRE(g <= kMaxGroup, NKV_EUNSUPPORTED, "paged_decode: GQA group %d above %d", g,
              kMaxGroup);
  NKV_REQUIRE(block_size > 0 && block_size % kChunk == 0, NKV_EUNSUPPORTED,
              "paged_decode: block_size must be a multiple of 16 (got %d)", block_size);
  NKV_REQUIRE(max_blocks_per_seq > 0 && bt_row_stride >= max_blocks_per_seq, NKV_EINVAL,
              "paged_decode: bad block table width/stride (%d, %lld)", max_blocks_per_seq,
              (long long)bt_row_stride);
  NKV_REQUIRE((int64_t)max_blocks_per_seq * block_size < (1ll << 30), NKV_EUNSUPPORTED,
              "paged_decode: max_blocks_per_seq * block_size too large");
  NKV_REQUIRE((int64_t)block_size * n_kv_heads * head_dim * 2 < (1ll << 31), NKV_EUNSUPPORTED,
              "paged_decode: cache block too large for 32-bit buffer offsets");
  NKV_REQUIRE(q_row_stride >= (int64_t)n_q_heads * head_dim && q_row_stride % 8 == 0,
              NKV_EINVAL, "paged_decode: q row stride must be >= Hq*D and a multiple of 8");
  NKV_REQUIRE(q && k_cache && v_cache && block_tables && context_lens, NKV_EINVAL,
              "paged_decode: null pointer");
  NKV_REQUIRE(aligned16(q) && aligned16(k_cache) && aligned16(v_cache), NKV_EINVAL,
              "paged_decode: q/k_cache/v_cache must be 16-byte aligned");
  return NKV_OK;
}

// Persistent grid: as many one-wave workgroups as are resident at once, at most
// kWavesPerCU per CU (the workspace bound assumes no more).
template <bool F8, int HP, int D>
static int decode_grid() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    int per_cu = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per_cu, reinterpret_cast<const void*>(paged_decode_split_kernel<F8, HP, D>), 64,
            0) != hipSuccess ||
        per_cu <= 0)
      per_cu = kWavesPerCU;
    n = device_cus() * std::min(per_cu, kWavesPerCU);
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// KV heads per wave at most for head_dim D: a 512-byte piece of every token row
// (bf16: 4 / 2 / 1 at D = 64 / 128 / 256; fp8: 4 / 4 / 2).
template <bool F8>
static constexpr int decode_max_hp(int D) {
  const int hp = 512 / (D * (F8 ? 1 : 2));
  return hp > 4 ? 4 : hp;
}

// The resident grid of instance (F8, hp, D) -- hp and D from the plan.
template <bool F8>
static int decode_grid_of(int hp, int D) {
  if (D == 64) {
    return hp == 4 ? decode_grid<F8, 4, 64>() : hp == 2 ? decode_grid<F8, 2, 64>()
                                                        : decode_grid<F8, 1, 64>();
  }
  if (D == 128) {
    if constexpr (F8) {
      if (hp == 4) return decode_grid<true, 4, 128>();
    }
    return hp == 2 ? decode_grid<F8, 2, 128>() : decode_grid<F8, 1, 128>();
  }
  if constexpr (F8) {
    if (hp == 2) return decode_grid<true, 2, 256>();
  }
  return decode_grid<F8, 1, 256>();
}

// The launch a decode call makes: KV heads per wave, the grid and the smallest range.
struct DecodePlan {
  int hp;          // KV heads per wave (1, 2 or 4)
  int ncg;         // column groups per KV head (1 unless G > 16; then hp = 1)
  unsigned grid;   // one-wave workgroups
  int32_t min_chunks;
};

// Waves per head group that full tables give ranges of kMinChunks (or more, see
// decode_min_chunks).
static int64_t decode_useful_waves(int32_t batch, int32_t max_blocks, int32_t block_size) {
  const int64_t max_chunks = decode_max_chunks(max_blocks, block_size);
  const int32_t min_chunks = decode_min_chunks(max_chunks, kMinChunks);
  return std::max<int64_t>(1, (batch * max_chunks + min_chunks - 1) / min_chunks);
}

template <bool F8>
static DecodePlan decode_plan(int32_t batch, int32_t Hq, int32_t Hk, int32_t max_blocks,
                              int32_t block_size, int32_t D) {
  const int g = Hq / Hk;
  const int64_t max_chunks = decode_max_chunks(max_blocks, block_size);
  // Several KV heads per wave (up to a 512-byte piece of every token row) when the heads
  // group evenly, the hp*G query heads fit the 16 MFMA columns and there is enough work
  // for every wave (upper bound from the table width: >= 32 chunks per head group per
  // resident wave of the two-head instance); otherwise one.
  const int64_t work = (int64_t)batch * max_chunks * Hk;
  int hp = 1;
  if (decode_max_hp<F8>(D) >= 2 && Hk % 2 == 0 && 2 * g <= kMaxCols &&
      work >= 32 * (int64_t)decode_grid_of<F8>(2, D)) {
    hp = 2;
    if (decode_max_hp<F8>(D) >= 4 && Hk % 4 == 0 && 4 * g <= kMaxCols) hp = 4;
  }
  DecodePlan p;
  p.hp = hp;
  p.ncg = decode_ncg(g);
  p.min_chunks = decode_min_chunks(max_chunks, decode_range_floor(batch, D, F8));
  // Resident waves per head group, but no more than the table width lets receive a range
  // of kMinChunks (small batches launch only the waves that can get work).
  const int resident = decode_grid_of<F8>(hp, D);
  const int np = Hk * p.ncg / p.hp;
  const int64_t per =
      std::min<int64_t>(std::max(1, resident / np),
                        decode_useful_waves(batch, max_blocks, block_size));
  p.grid = (unsigned)(per * np);
  return p;
}

// Bytes of the descriptors (one per sequence, KV head and column group; 16-byte aligned)
// and of the partial rows a plan writes: each head group (waves + batch) x its columns,
// i.e. (grid / head groups + batch) x Hq rows in all (grid * hp*g + batch * Hq for G <= 16;
// at most grid * 16 + batch * Hq).
static size_t decode_desc_bytes(int32_t batch, int32_t n_groups) {
  return (size_t)batch * n_groups * sizeof(i32x4v_t);
}
static size_t decode_part_bytes(int64_t waves, int32_t batch, int32_t Hq, int32_t D) {
  return (size_t)((waves + batch) * (int64_t)Hq) * part_row(D) * sizeof(float);
}
// Waves per head group of a plan.
static int64_t decode_waves(const DecodePlan& p, int32_t Hk) {
  return (int64_t)p.grid / (Hk * p.ncg / p.hp);
}

}  // namespace nkv

extern "C" size_t nkv_paged_decode_workspace_bytes(int32_t batch, int32_t n_q_heads,
                                                   int32_t head_dim, int32_t max_blocks_per_seq,
                                                   int32_t block_size) {
  using namespace nkv;
  if (batch <= 0 || n_q_heads <= 0 || max_blocks_per_seq <= 0 || block_size <= 0 ||
      !decode_dim_ok(head_dim))
    return 0;
  // Whatever the plan: waves per head group x Hq <= grid x min(16, Hq) (a group's columns
  // are at most 16 and the groups' columns add up to Hq), grid <= CUs * kWavesPerCU and
  // grid <= useful * (head groups); the descriptors (per KV head and column group) at most
  // batch * Hq.
  const int64_t resident = (int64_t)device_cus() * kWavesPerCU;
  const int64_t cols = std::min<int64_t>(
      resident * std::min(kMaxCols, n_q_heads),
      decode_useful_waves(batch, max_blocks_per_seq, block_size) * n_q_heads);
  return decode_desc_bytes(batch, n_q_heads) + decode_part_bytes(0, batch, n_q_heads, head_dim) +
         (size_t)cols * part_row(head_dim) * sizeof(float);
}

namespace nkv {
template <bool F8, bool H16 = false>
static int decode_split(const void* q, int64_t q_row_stride, const void* k_cache,
                        const void* v_cache, const int32_t* block_tables, int64_t bt_row_stride,
                        const int32_t* context_lens, int32_t batch, int32_t n_q_heads,
                        int32_t n_kv_heads, int32_t head_dim, int32_t block_size,
                        int32_t max_blocks_per_seq, int64_t n_blocks, float scale, float k_scale,
                        float v_scale, void* workspace, size_t workspace_bytes, void* stream) {
  int rc = decode_check(q, k_cache, v_cache, block_tables, context_lens, batch, n_q_heads,
                        n_kv_heads, head_dim, block_size, max_blocks_per_seq, q_row_stride,
                        bt_row_stride);
  if (rc) return rc;
  if (batch == 0) return NKV_OK;
  NKV_REQUIRE(k_scale > 0.f && v_scale > 0.f, NKV_EINVAL, "paged_decode: scales must be > 0");
  const int64_t max_chunks = ((int64_t)max_blocks_per_seq * block_size + kChunk - 1) / kChunk;
  NKV_REQUIRE(max_chunks * batch * n_kv_heads < (1ll << 31), NKV_EUNSUPPORTED,
              "paged_decode: too many chunks in one call");
  const int g = n_q_heads / n_kv_heads;
  const DecodePlan p = decode_plan<F8>(batch, n_q_heads, n_kv_heads, max_blocks_per_seq,
                                       block_size, head_dim);
  const size_t desc_b = decode_desc_bytes(batch, n_kv_heads * p.ncg);
  const int64_t waves = decode_waves(p, n_kv_heads);
  const size_t need = desc_b + decode_part_bytes(waves, batch, n_q_heads, head_dim);
  NKV_REQUIRE(workspace && workspace_bytes >= need, NKV_EWORKSPACE,
              "paged_decode: workspace needs %zu bytes (got %zu)", need, workspace_bytes);
  NKV_REQUIRE((waves + batch) * n_q_heads < (1ll << 31), NKV_EUNSUPPORTED,
              "paged_decode: too many partial rows");
  i32x4v_t* desc = static_cast<i32x4v_t*>(workspace);
  float* part = reinterpret_cast<float*>(static_cast<char*>(workspace) + desc_b);
  const float scale_log2 = scale * k_scale * kLog2e;
  hipStream_t s = as_stream(stream);
#define NKV_DECODE_LAUNCH(HP, D)                                                               \
  hipLaunchKernelGGL((paged_decode_split_kernel<F8, HP, D, H16>), dim3(p.grid), dim3(64), 0, s, \
                     (const bf16_t*)q, q_row_stride, k_cache, v_cache, block_tables,           \
                     bt_row_stride, context_lens, batch, n_kv_heads, g, p.ncg, block_size,     \
                     max_blocks_per_seq, n_blocks, p.min_chunks, scale_log2, v_scale, part,    \
                     desc)
  if (head_dim == 64) {
    if (p.hp == 4) NKV_DECODE_LAUNCH(4, 64);
    else if (p.hp == 2) NKV_DECODE_LAUNCH(2, 64);
    else NKV_DECODE_LAUNCH(1, 64);
  } else if (head_dim == 128) {
    if (p.hp == 4) {
      if constexpr (F8) NKV_DECODE_LAUNCH(4, 128);
    } else if (p.hp == 2) {
      NKV_DECODE_LAUNCH(2, 128);
    } else {
      NKV_DECODE_LAUNCH(1, 128);
    }
  } else {
    if (p.hp == 2) {
      if constexpr (F8) NKV_DECODE_LAUNCH(2, 256);
    } else {
      NKV_DECODE_LAUNCH(1, 256);
    }
  }
#undef NKV_DECODE_LAUNCH
  return check_launch("nkv_paged_decode_split");
}

// The combine of a split launched with the same arguments: the partial rows start after
// the descriptors, whatever the plan.
template <bool H16 = false>
static int decode_combine(const int32_t* context_lens, int32_t batch, int32_t n_q_heads,
                          int32_t n_kv_heads, int32_t head_dim, int32_t block_size,
                          int32_t max_blocks_per_seq, void* out, int64_t out_row_stride,
                          const void* workspace, size_t workspace_bytes, void* stream) {
  NKV_REQUIRE(decode_dim_ok(head_dim), NKV_EUNSUPPORTED,
              "paged_decode: head_dim must be 64, 128 or 256 (got %d)", head_dim);
  NKV_REQUIRE(batch >= 0 && n_q_heads > 0 && n_kv_heads > 0 && n_q_heads % n_kv_heads == 0 &&
                  n_q_heads / n_kv_heads <= kMaxGroup && block_size > 0 &&
                  max_blocks_per_seq > 0,
              NKV_EINVAL, "paged_decode_combine: bad sizes");
  const int ncg = decode_ncg(n_q_heads / n_kv_heads);
  if (batch == 0) return NKV_OK;
  NKV_REQUIRE(out && context_lens, NKV_EINVAL, "paged_decode_combine: null pointer");
  // each lane stores D/64 consecutive bf16 (2, 4 or 8 bytes)
  const int al = head_dim / 64;  // elements per lane store
  NKV_REQUIRE(out_row_stride >= (int64_t)n_q_heads * head_dim && out_row_stride % al == 0 &&
                  (reinterpret_cast<uintptr_t>(out) & (2 * al - 1)) == 0,
              NKV_EINVAL,
              "paged_decode_combine: out must be %d-byte aligned with a row stride >= Hq*D "
              "that is a multiple of %d", 2 * al, al);
  const size_t desc_b = decode_desc_bytes(batch, n_kv_heads * ncg);
  NKV_REQUIRE(workspace && workspace_bytes > desc_b, NKV_EWORKSPACE,
              "paged_decode_combine: workspace of %zu bytes holds no partials",
              workspace_bytes);
  const i32x4v_t* desc = static_cast<const i32x4v_t*>(workspace);
  const float* part = reinterpret_cast<const float*>(static_cast<const char*>(workspace) + desc_b);
  const dim3 grid((unsigned)(batch * n_q_heads));
  // (the ranges of a 16-bit pool: an fp8 one's are no shorter)
  const int64_t max_chunks = decode_max_chunks(max_blocks_per_seq, block_size);
  const int64_t min_chunks =
      decode_min_chunks(max_chunks, decode_range_floor(batch, head_dim, false));
  const bool wide = combine_wide(batch, n_kv_heads, ncg, max_chunks, min_chunks,
                                 (int64_t)device_cus() * kWavesPerCU);
#define NKV_COMBINE_LAUNCH_W(D, W)                                                             \
  hipLaunchKernelGGL((paged_decode_combine_kernel<D, H16, W>), grid, dim3(64 * W), 0,          \
                     as_stream(stream), context_lens, n_q_heads, n_kv_heads, ncg, part, desc,  \
                     (bf16_t*)out, out_row_stride)
#define NKV_COMBINE_LAUNCH(D)                                                                  \
  do {                                                                                         \
    if (wide) NKV_COMBINE_LAUNCH_W(D, 4);                                                      \
    else NKV_COMBINE_LAUNCH_W(D, 1);                                                           \
  } while (0)
  if (head_dim == 64) NKV_COMBINE_LAUNCH(64);
  else if (head_dim == 128) NKV_COMBINE_LAUNCH(128);
  else NKV_COMBINE_LAUNCH(256);
#undef NKV_COMBINE_LAUNCH
#undef NKV_COMBINE_LAUNCH_W
  return check_launch("nkv_paged_decode_combine");
}
}  // namespace nkv

extern "C" int nkv_paged_decode_split(const void* q, int64_t q_row_stride, const void* k_cache,
                                      const void* v_cache, const int32_t* block_tables,
                                      int64_t bt_row_stride, const int32_t* context_lens,
                                      int32_t batch, int32_t n_q_heads, int32_t n_kv_heads,
                                      int32_t head_dim, int32_t block_size,
                                      int32_t max_blocks_per_seq, int64_t n_blocks, float scale,
                                      void* workspace, size_t workspace_bytes, void* stream) {
  nkv::clear_error();
  return nkv::decode_split<false>(q, q_row_stride, k_cache, v_cache, block_tables,
                                  bt_row_stride, context_lens, batch, n_q_heads, n_kv_heads,
                                  head_dim, block_size, max_blocks_per_seq, n_blocks, scale, 1.f,
                                  1.f, workspace, workspace_bytes, stream);
}

extern "C" int nkv_paged_decode_combine(const int32_t* context_lens, int32_t batch,
                                        int32_t n_q_heads, int32_t n_kv_heads, int32_t head_dim,
                                        int32_t block_size, int32_t max_blocks_per_seq,
                                        void* out, int64_t out_row_stride, const void* workspace,
                                        size_t workspace_bytes, void* stream) {
  nkv::clear_error();
  return nkv::decode_combine(context_lens, batch, n_q_heads, n_kv_heads, head_dim, block_size,
                             max_blocks_per_seq, out, out_row_stride, workspace, workspace_bytes,
                             stream);
}

extern "C" int nkv_paged_decode(const void* q, int64_t q_row_stride, const void* k_cache,
                                const void* v_cache, const int32_t* block_tables,
                                int64_t bt_row_stride, const int32_t* context_lens, int32_t batch,
                                int32_t n_q_heads, int32_t n_kv_heads, int32_t head_dim,
                                int32_t block_size, int32_t max_blocks_per_seq, int64_t n_blocks,
                                float scale, void* out, int64_t out_row_stride, void* workspace,
                                size_t workspace_bytes, void* stream) {
  int rc = nkv_paged_decode_split(q, q_row_stride, k_cache, v_cache, block_tables, bt_row_stride,
                                  context_lens, batch, n_q_heads, n_kv_heads, head_dim,
                                  block_size, max_blocks_per_seq, n_blocks, scale, workspace,
                                  workspace_bytes, stream);
  if (rc) return rc;
  return nkv_paged_decode_combine(context_lens, batch, n_q_heads, n_kv_heads, head_dim,
                                  block_size, max_blocks_per_seq, out, out_row_stride, workspace,
                                  workspace_bytes, stream);
}

extern "C" int nkv_paged_decode_f16(const void* q, int64_t q_row_stride, const void* k_cache,
                                    const void* v_cache, const int32_t* block_tables,
                                    int64_t bt_row_stride, const int32_t* context_lens,
                                    int32_t batch, int32_t n_q_heads, int32_t n_kv_heads,
                                    int32_t head_dim, int32_t block_size,
                                    int32_t max_blocks_per_seq, int64_t n_blocks, float scale,
                                    void* out, int64_t out_row_stride, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  nkv::clear_error();
  int rc = nkv::decode_split<false, true>(q, q_row_stride, k_cache, v_cache, block_tables,
                                          bt_row_stride, context_lens, batch, n_q_heads,
                                          n_kv_heads, head_dim, block_size, max_blocks_per_seq,
                                          n_blocks, scale, 1.f, 1.f, workspace, workspace_bytes,
                                          stream);
  if (rc) return rc;
  return nkv::decode_combine<true>(context_lens, batch, n_q_heads, n_kv_heads, head_dim,
                                   block_size, max_blocks_per_seq, out, out_row_stride,
                                   workspace, workspace_bytes, stream);
}

extern "C" int nkv_paged_decode_fp8(const void* q, int64_t q_row_stride, const void* k_cache,
                                    const void* v_cache, const int32_t* block_tables,
                                    int64_t bt_row_stride, const int32_t* context_lens,
                                    int32_t batch, int32_t n_q_heads, int32_t n_kv_heads,
                                    int32_t head_dim, int32_t block_size,
                                    int32_t max_blocks_per_seq, int64_t n_blocks, float scale,
                                    float k_scale, float v_scale, void* out,
                                    int64_t out_row_stride, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  nkv::clear_error();
  int rc = nkv::decode_split<true>(q, q_row_stride, k_cache, v_cache, block_tables,
                                   bt_row_stride, context_lens, batch, n_q_heads, n_kv_heads,
                                   head_dim, block_size, max_blocks_per_seq, n_blocks, scale,
                                   k_scale, v_scale, workspace, workspace_bytes, stream);
  if (rc) return rc;
  return nkv_paged_decode_combine(context_lens, batch, n_q_heads, n_kv_heads, head_dim,
                                  block_size, max_blocks_per_seq, out, out_row_stride, workspace,
                                  workspace_bytes, stream);
}

// ------------------------------------------------------------------ no-allocation variant
// The decode workspace in a fixed device array: for callers that cannot allocate (code
// under graph capture, tight serving loops). Each device holds its own copy of the array
// for the life of the process. Host code never passes the array's name to a kernel (on
// the host it is only a stand-in): its device address comes from hipGetSymbolAddress,
// taken once per device on the first call there, with that device current.
namespace nkv {
constexpr size_t kScratchBytes = NKV_DECODE_NOALLOC_MAX_BYTES;  // batch*Hq up to ~94k heads
}  // namespace nkv

static __device__ __align__(256) unsigned char scratch[nkv::kScratchBytes];

namespace nkv {
// Device address of `scratch` on the current device, or nullptr (error text set).
static void* scratch_ptr() {
  static std::atomic<void*> ptrs[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) {
    set_error("paged_decode_noalloc: no current device");
    return nullptr;
  }
  void* p = ptrs[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    // threads that race here obtain the same address
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      set_error("paged_decode_noalloc: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
      return nullptr;
    }
    ptrs[dev].store(p, std::memory_order_release);
  }
  return p;
}
}  // namespace nkv

extern "C" int nkv_paged_decode_noalloc(const void* q, int64_t q_row_stride, const void* k_cache,
                                        const void* v_cache, const int32_t* block_tables,
                                        int64_t bt_row_stride, const int32_t* context_lens,
                                        int32_t batch, int32_t n_q_heads, int32_t n_kv_heads,
                                        int32_t head_dim, int32_t block_size,
                                        int32_t max_blocks_per_seq, int64_t n_blocks,
                                        float scale, void* out, int64_t out_row_stride,
                                        void* stream) {
  using namespace nkv;
  clear_error();
  int rc = decode_check(q, k_cache, v_cache, block_tables, context_lens, batch, n_q_heads,
                        n_kv_heads, head_dim, block_size, max_blocks_per_seq, q_row_stride,
                        bt_row_stride);
  if (rc) return rc;
  if (batch == 0) return NKV_OK;
  // the bytes this call's plan needs, against the array's fixed size
  const DecodePlan p = decode_plan<false>(batch, n_q_heads, n_kv_heads, max_blocks_per_seq,
                                          block_size, head_dim);
  const size_t need = decode_desc_bytes(batch, n_kv_heads * p.ncg) +
                      decode_part_bytes(decode_waves(p, n_kv_heads), batch, n_q_heads,
                                        head_dim);
  NKV_REQUIRE(need <= kScratchBytes, NKV_EUNSUPPORTED,
              "paged_decode_noalloc: batch %d x %d query heads needs %zu bytes of partials, "
              "above the fixed %zu-byte array; use nkv_paged_decode with a workspace",
              batch, n_q_heads, need, kScratchBytes);
  void* ws = scratch_ptr();
  if (ws == nullptr) return NKV_ELAUNCH;
  rc = decode_split<false>(q, q_row_stride, k_cache, v_cache, block_tables, bt_row_stride,
                           context_lens, batch, n_q_heads, n_kv_heads, head_dim, block_size,
                           max_blocks_per_seq, n_blocks, scale, 1.f, 1.f, ws, kScratchBytes,
                           stream);
  if (rc) return rc;
  return decode_combine(context_lens, batch, n_q_heads, n_kv_heads, head_dim, block_size,
                        max_blocks_per_seq, out, out_row_stride, ws, kScratchBytes, stream);
}
