// The decode stream: one new query row per sequence against its paged K/V, a wave's equal
// share of the batch's 16-token chunks at a time, and the merge of a row's partials. Device code
// of the decode kernels (paged_decode.hip, whose header describes the design) and of the
// decode rows among prompts (prefill.hip).
#pragma once

#include "nkv_common.h"

#include <type_traits>

namespace nkv {

constexpr int kChunk = 16;               // tokens per pipeline stage
constexpr int kMinChunks = 4;            // chunks per wave range that grids are sized for
// partials per (sequence, query head) at most: what four waves' combine has in flight at once
// (4 x 32), and one, so that a table of 512 chunks splits into ranges of 4
constexpr int kMaxSlots = 129;
constexpr int kWinBlocks = 64;           // block ids held per window (one per lane)
constexpr int kBufferFlags = 0x00020000; // raw buffer resource word 3 (dword data)
constexpr int kStreamPolicy = 2;         // cache policy "nt": K/V are read exactly once
constexpr int kWavesPerCU = 8;           // resident split waves per CU (2 per SIMD)
// floats per partial row: O, m, l, 2 pad (528 B at D = 128)
constexpr int part_row(int D) { return D + 4; }
constexpr bool decode_dim_ok(int D) { return D == 64 || D == 128 || D == 256; }
constexpr int kMaxCols = 16;             // MFMA columns: query heads per wave at most
constexpr int kMaxGroup = 256;           // GQA group at most (above 16: column groups)
// Column groups per KV head: its G query heads over ceil(G / 16) waves when G > 16.
constexpr int decode_ncg(int G) { return G > kMaxCols ? (G + kMaxCols - 1) / kMaxCols : 1; }

typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4_t lds_i16x4_t;
typedef __bf16 bf16x2v_t __attribute__((ext_vector_type(2)));
typedef int32_t i32x4v_t __attribute__((ext_vector_type(4)));

static inline int64_t decode_max_chunks(int32_t max_blocks, int32_t block_size) {
  return ((int64_t)max_blocks * block_size + kChunk - 1) / kChunk;
}
// The smallest range a wave takes. The grid and the workspace are sized for ranges of kMinChunks
// of full tables; contexts shorter than the table leave some of those waves idle, and shorter
// ranges use them. A range starts with its first ring slots in flight at once, two chunks of
// 256-byte row pieces: longer ranges add round trips, shorter ones partials to merge. Measured
// with 4 / 3 (split and combine in a graph, us): four sequences of 300-1000 12.8 / 11.2, eight
// 13.8 / 12.4, 24 of 50-250 13.1 / 11.4, 40 of 20-64 12.4 / 10.6, 100 of 50-500 17.9 / 17.1; one
// or two, whose table fits, gain nothing (11.0 / 11.4). Ranges of two are slower from three
// sequences on (16 of 100-900, 40 query heads: 13.8 / 15.0). Over 704 shapes of 3 - 200 sequences
// 3 takes 0.957 of 4's time on average, 24 of them over 1.05, at most 1.11 (five of up to 3000, 64
// query heads on 8: 13.5 / 15.0). fp8 and head_dim 64 hold four chunks and keep ranges of four.
static inline int32_t decode_range_floor(int32_t batch, int32_t D, bool f8) {
  return D == 128 && !f8 && batch > 2 ? 3 : kMinChunks;
}
// The smallest range: the floor, or longer where the table width allows segments that would
// otherwise have more than kMaxSlots partials (a segment of n chunks is touched by at most
// ceil(n / C) + 1 waves), which is as many as the combine holds.
static inline int32_t decode_min_chunks(int64_t max_chunks, int32_t floor) {
  const int64_t c = (max_chunks + kMaxSlots - 2) / (kMaxSlots - 1);
  return (int32_t)(c > floor ? c : floor);
}

// Cursor over sequences in batches of 64 (one per lane): in the chunk stream
// of one KV head, sequence s owns chunks [g_s, g_s + nc_s).
struct SeqCursor {
  int cb;    // first sequence of the loaded batch (uniform)
  int base;  // stream index of sequence cb's first chunk (uniform)
  int tot;   // chunks of the batch (uniform)
  int ctx;   // lane: context length of sequence cb + lane
  int nc;    // lane: chunks of that sequence
  int incl;  // lane: inclusive prefix of nc over the batch
};

// The sequences of a decode batch: context_lens[s] keys for row s of q and out. Keys past the
// table or in an invalid block are left out.
struct DecodeSeqs {
  static constexpr bool kZeroInvalid = false;
  const int32_t* __restrict__ context_lens;
  int32_t batch;
  __device__ __forceinline__ int keys(int s) const { return context_lens[s]; }
  __device__ __forceinline__ int64_t row(int s) const { return s; }
};
// The sequences of a variable-length batch that bring one new token (the others have no chunk
// here): row cu_q[s] of q and out. Keys past the table or in an invalid block are zeros that
// take their weight, as everywhere in such a batch: those in a block are chunks like the others,
// those past the table's max_tokens are weighed by the combine, so that no row has more
// partials than its table's width allows.
struct OneRowSeqs {
  static constexpr bool kZeroInvalid = true;
  const int32_t* __restrict__ cu_q;
  const int32_t* __restrict__ cu_k;
  int32_t batch;
  int32_t max_tokens;
  __device__ __forceinline__ int keys(int s) const {
    return cu_q[s + 1] - cu_q[s] == 1 ? cu_k[s + 1] - cu_k[s] : 0;
  }
  __device__ __forceinline__ int64_t row(int s) const { return cu_q[s]; }
};

// Chunks of a sequence of ctx keys.
__device__ __forceinline__ int seq_chunks(int ctx, int max_tokens) {
  NKV_DBG(ctx < 0 || ctx > max_tokens, NKV_DEBUG_LENGTH);
  return ctx > 0 ? (min(ctx, max_tokens) + kChunk - 1) / kChunk : 0;
}
template <typename Seqs>
__device__ __forceinline__ void seq_load(SeqCursor& c, const Seqs& seqs, int max_tokens) {
  const int s = c.cb + (int)(threadIdx.x & 63);
  c.ctx = s < seqs.batch ? seqs.keys(s) : 0;
  c.nc = seq_chunks(c.ctx, max_tokens);
  c.incl = wave_incl_scan(c.nc);
  c.tot = __builtin_amdgcn_readlane(c.incl, 63);
}

// Element offset of head dim `dim` (a multiple of 4) in a staged LDS row. bf16 rows are
// dense. fp8 rows are staged as 8-dim pieces with the even pieces first (piece 2c at slot
// c, piece 2c+1 at slot D/16 + c): a lane widens 16 codes into pieces 2c and 2c+1, and
// each of its two 16-byte writes then lands beside its neighbours' (the 32-byte stride of
// a dense row would leave half the banks idle and pair the others up).
template <bool F8, int D>
__device__ __forceinline__ int stage_off(int dim) {
  if constexpr (F8) {
    const int piece = dim >> 3;
    return ((piece >> 1) + (D / 16) * (piece & 1)) * 8 + (dim & 7);
  } else {
    return dim;
  }
}

// F8: the caches hold fp8 (OCP E4M3FN) codes; a chunk's rows are half as many
// bytes and are widened to bf16 (exact) when staged in LDS; the K scale is
// folded into scale_log2 and the V scale multiplies the partial O.
// HP: KV heads per wave. With HP = 2 a wave reads both heads' halves of every
// token row as one contiguous piece (512 B bf16, 256 B fp8) instead of one
// head's 256 B: on this part a stream of 256-byte pieces at 2 KiB stride runs
// unevenly (pieces at odd 256-byte offsets come back later), and the waves of
// the slow heads set the kernel's length. The HP*G query heads fill MFMA columns
// 0..HP*G-1; each head's scores use its own K, the softmax weights of a column
// are zero for the other heads, so all heads' PV products add into one O^T.
// fp8 rows (1 KiB at Hk = 8) take HP = 4 for 512-byte pieces, with K and V
// staged through one LDS buffer so two waves per SIMD still fit.
// G (query heads per KV head) is any value with HP*G <= 16: the columns past
// HP*G are computed and dropped. D: head_dim (64, 128 or 256); a wave's piece of
// a token row (HP*D elements) is 128 to 512 bytes.
//
// One wave's work: wave `wid` of `n_waves`; `lbuf` is its own LDS, decode_lds_elems of it.
template <bool F8, int HP, int D>
constexpr int decode_lds_elems() {
  constexpr int kRows = HP * kChunk * (D + 16);
  return 2 * kRows * 2 >= 20480 ? kRows : 2 * kRows;
}
template <bool F8, int HP, int D, bool H16, typename Seqs>
__device__ __forceinline__ void decode_stream(
    const Seqs seqs, const int wid, const int n_waves, bf16_t* lbuf,
    const bf16_t* __restrict__ q, int64_t q_row_stride,
    const void* __restrict__ k_cache, const void* __restrict__ v_cache,
    const int32_t* __restrict__ block_tables, int64_t bt_row_stride, int32_t Hk, int32_t G,
    int32_t NCG, int32_t block_size, int32_t max_blocks, int64_t n_blocks, int32_t min_chunks,
    float scale_log2, float v_scale, float* __restrict__ part, i32x4v_t* __restrict__ desc) {
  static_assert(decode_dim_ok(D), "head_dim 64, 128 or 256");
  static_assert(!(F8 && H16), "fp8 caches are read with bf16 queries");
  constexpr int kEl = F8 ? 1 : 2;              // bytes per cache element
  constexpr int kSeg = HP * D * kEl;           // bytes a wave reads of each token row
  static_assert(kSeg >= 64 && kSeg <= 512, "a wave's piece of a row is 64..512 bytes");
  constexpr int kKs = D / 32;                  // k-steps of S^T (32 dims each)
  constexpr int kDb = D / 16;                  // 16-dim blocks of O^T
  constexpr int kVRow = D + 16;                // LDS row stride of a staged chunk (elements)
  constexpr int kPartRow = part_row(D);
  constexpr int kLpr = kSeg / 16;              // lanes per row (16-byte loads)
  constexpr int kRpl = 64 / kLpr;              // rows per load instruction
  constexpr int kLoads = kChunk / kRpl;        // loads per lane per K (or V) chunk
  // ring depth: 16 KiB of K and V in flight per wave (one chunk of 512-byte pieces, two of
  // 256-byte ones ...); a chunk's slot is refilled as soon as its rows are staged in LDS
  constexpr int kRing = kLoads >= 8 ? 1 : kLoads >= 4 ? 2 : 4;
  constexpr int kLph = kLpr / HP;              // lanes per head within a row
  // K and V of a chunk share one staging buffer (V is written after the K reads of S^T)
  // where two would take 20 KiB or more (four heads at D <= 128, two at D = 256), which
  // keeps two waves per SIMD within the LDS
  constexpr bool kShared = 2 * HP * kChunk * kVRow * 2 >= 20480;
  using Rows = bf16_t[HP][kChunk * kVRow];
  auto& kbuf = *reinterpret_cast<Rows*>(lbuf);
  auto& vbuf = *reinterpret_cast<Rows*>(lbuf + (kShared ? 0 : HP * kChunk * kVRow));

  const int lane = threadIdx.x & 63;
  const int batch = seqs.batch;
  const int g4 = lane >> 4;   // key group: keys 4*g4 .. 4*g4+3 of a chunk
  const int col = lane & 15;  // MFMA column: query head (S^T, O^T) / key row (K)
  // Column groups: the G > 16 query heads of a KV head are split over NCG = ceil(G / 16)
  // waves of 16 MFMA columns (the last one fewer; HP = 1 then); NCG = 1 otherwise.
  const int row_b = Hk * D * kEl;  // bytes of one cache row (token)
  const int max_tokens = max_blocks * block_size;

  // ---- this wave's KV heads and chunk range. Every head group has the same
  // chunk stream (sequence-major); waves p, p+NP, p+2NP, ... split it into
  // equal ranges, so the NP waves i*NP .. i*NP+NP-1 read the Hk heads of the
  // same cache blocks at the same time.
  const int NP = Hk * NCG / HP;
  const int grp = wid % NP;
  const int kvh0 = (grp / NCG) * HP;
  const int cg = grp - (grp / NCG) * NCG;  // column group
  // MFMA columns that are query heads (= partial rows per wave and sequence)
  const int HPG = NCG > 1 ? min(kMaxCols, G - cg * kMaxCols) : HP * G;
  const int qh0 = kvh0 * G + cg * kMaxCols;  // query head of column 0
  const int wi = wid / NP;
  const int Wh = n_waves / NP;
  if (wi >= Wh) return;
  // partial rows of this head group: (wave + sequence) x HPG columns, after the groups of
  // the query heads before qh0 (so the groups' regions add up to (waves + batch) x Hq rows)
  float* gpart = part + (int64_t)(Wh + batch) * qh0 * kPartRow;
  // chunks of the whole batch: its lengths' loads in flight together, one reduction (the first
  // 64 sequences' cursor is loaded with them)
  SeqCursor cur;
  cur.cb = 0;
  cur.base = 0;
  seq_load(cur, seqs, max_tokens);
  int T = cur.tot;
  if (batch > 64) {
    int more = 0;
#pragma unroll 4
    for (int s = 64 + lane; s < batch; s += 64)
      more += seq_chunks(seqs.keys(s), max_tokens);
    T += __builtin_amdgcn_readlane(wave_incl_scan(more), 63);
  }
  // equal ranges over the resident waves, at least min_chunks (which keeps every
  // segment within its partial slots)
  const int C = max((T + Wh - 1) / Wh, min_chunks);
  const int k_begin = wi * C;
  if (k_begin >= T) return;
  const int k_end = min(T, k_begin + C);

  // per-lane load offset: lane l reads 16 bytes of row l / kLpr (+ kRpl per
  // load), byte 16 * (l % kLpr) of the wave's piece of the row; it stages them
  // in head sh's LDS rows at dim sd (fp8 codes widen to 16 bf16 there). K is
  // re-read from LDS in the MFMA A layout.
  const int roff = (lane / kLpr) * row_b + (lane % kLpr) * 16;
  const int rstep = kRpl * row_b;  // bytes between a lane's consecutive loads
  const int sh = (lane % kLpr) / kLph;
  const int sd = (lane % kLph) * (16 / kEl);
  const int tr_row = 4 * g4 + (col >> 2);  // ds_read_b64_tr_b16 source row / column
  const int tr_col = (col & 3) * 4;
  const int hsel = col / G;                // head (of the HP) of this lane's column

  for (int k = k_begin; k < k_end;) {
    // ---- locate the sequence holding stream chunk k (wave-uniform)
    while (k >= cur.base + cur.tot) {
      cur.base += cur.tot;
      cur.cb += 64;
      seq_load(cur, seqs, max_tokens);
    }
    const int ln =
        __builtin_amdgcn_readfirstlane(__builtin_ctzll(__ballot(cur.base + cur.incl > k)));
    const int b = cur.cb + ln;
    const int ctx = __builtin_amdgcn_readlane(cur.ctx, ln);
    const int nc = __builtin_amdgcn_readlane(cur.nc, ln);
    const int g0 = cur.base + __builtin_amdgcn_readlane(cur.incl, ln) - nc;
    const int c_lo = k - g0;
    const int n_seg = min(nc - c_lo, k_end - k);
    const int w_first = g0 / C;  // first wave of the segment

    // q^T as the MFMA B operand: lane l -> query head kvh0*G + l%16 (columns
    // >= HP*G re-read the first head and are discarded), dims 8*(l/16) + 32*ks
    u32x4_t qreg[kKs];
    {
      const int hc = col < HPG ? col : 0;
      const u32x4_t* qp = reinterpret_cast<const u32x4_t*>(
          q + seqs.row(b) * q_row_stride + (int64_t)(qh0 + hc) * D + g4 * 8);
#pragma unroll
      for (int ks = 0; ks < kKs; ++ks) qreg[ks] = qp[ks * 4];
    }
    const char* kbase = static_cast<const char*>(k_cache) + (int64_t)kvh0 * D * kEl;
    const char* vbase = static_cast<const char*>(v_cache) + (int64_t)kvh0 * D * kEl;
    const int32_t* bt_row = block_tables + (int64_t)b * bt_row_stride;

    f32x4_t acc[kDb];  // O^T: lane l -> column l%16, dims 16*db + 4*(l/16) .. +3
#pragma unroll
    for (int db = 0; db < kDb; ++db) acc[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;

    // windows of at most kWinBlocks cache blocks (block ids one per lane)
    const int win_cap = (kWinBlocks - 1) * (block_size / kChunk);
    for (int wc = 0; wc < n_seg; wc += win_cap) {
      const int wlo = c_lo + wc;                 // first chunk of the window
      const int wn = min(n_seg - wc, win_cap);   // chunks in the window
      const int blk0 = wlo * kChunk / block_size;
      int blk_id = -1;
      {
        const int bi = blk0 + lane;
        if (bi < max_blocks && bi * block_size < (wlo + wn) * kChunk) {
          const int id = bt_row[bi];
          NKV_DBG(id < 0 || id >= n_blocks, NKV_DEBUG_BLOCK);  // every block here is needed
          blk_id = (id >= 0 && id < n_blocks) ? id : -1;
        }
      }

      u32x4_t kreg[kRing][kLoads];
      u32x4_t vreg[kRing][kLoads];
      int nv[kRing];  // valid keys of the chunk in each ring slot (0: masked)
      auto issue = [&](int j, int s) {
        const int t0 = (wlo + j) * kChunk;
        const int pb = __builtin_amdgcn_readlane(blk_id, min(t0 / block_size - blk0, 63));
        const int keys = j < wn ? min(max(ctx - t0, 0), kChunk) : 0;
        const int n = pb >= 0 ? keys : 0;
        nv[s] = Seqs::kZeroInvalid ? keys : n;
        const int64_t r0 = (int64_t)(pb < 0 ? 0 : pb) * block_size + t0 % block_size;
        const uint32_t bytes = (uint32_t)(n * row_b);
        const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(kbase + r0 * row_b), (short)0, bytes, kBufferFlags);
        const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(vbase + r0 * row_b), (short)0, bytes, kBufferFlags);
#pragma unroll
        for (int r = 0; r < kLoads; ++r)
          kreg[s][r] = __builtin_bit_cast(
              u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rk, roff + r * rstep, 0,
                                                             kStreamPolicy));
#pragma unroll
        for (int r = 0; r < kLoads; ++r)
          vreg[s][r] = __builtin_bit_cast(
              u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rv, roff + r * rstep, 0,
                                                             kStreamPolicy));
      };

      auto consume = [&](int s, auto refill, int nxt) {
        constexpr bool kRefill = decltype(refill)::value;
        const int nv_cur = nv[s];  // the refill below overwrites the slot's count
        // stage the chunk's K and V rows (row-major per head, bf16) in LDS
#pragma unroll
        for (int r = 0; r < kLoads; ++r) {
          const int row = (kRpl * r + lane / kLpr) * kVRow;
          const int e = row + stage_off<F8, D>(sd);
          if constexpr (F8) {
            const int e2 = row + stage_off<F8, D>(sd + 8);
            u32x4_t lo, hi;
            fp8x16_to_bf16(kreg[s][r], lo, hi);
            *reinterpret_cast<u32x4_t*>(&kbuf[sh][e]) = lo;
            *reinterpret_cast<u32x4_t*>(&kbuf[sh][e2]) = hi;
            if constexpr (!kShared) {
              fp8x16_to_bf16(vreg[s][r], lo, hi);
              *reinterpret_cast<u32x4_t*>(&vbuf[sh][e]) = lo;
              *reinterpret_cast<u32x4_t*>(&vbuf[sh][e2]) = hi;
            }
          } else {
            *reinterpret_cast<u32x4_t*>(&kbuf[sh][e]) = kreg[s][r];
            if constexpr (!kShared) *reinterpret_cast<u32x4_t*>(&vbuf[sh][e]) = vreg[s][r];
          }
        }
        if constexpr (kRefill && !kShared) {
          __builtin_amdgcn_sched_barrier(0);
          issue(nxt, s);  // the slot's registers are staged: refill now
          __builtin_amdgcn_sched_barrier(0);
        }
        // S^T for 16 keys x 16 columns per head; A operand: lane l -> key l%16,
        // dims 8*(l/16) + 32*ks
        f32x4_t st[HP];
#pragma unroll
        for (int hh = 0; hh < HP; ++hh) {
          f32x4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ks = 0; ks < kKs; ++ks) {
            const u32x4_t ka =
                *reinterpret_cast<const u32x4_t*>(
                    &kbuf[hh][col * kVRow + stage_off<F8, D>(g4 * 8 + ks * 32)]);
            a = mfma_16x16x32<H16>(ka, qreg[ks], a);
          }
          st[hh] = a;
        }
        // online softmax for column `col` over keys 4*g4 .. +3 of the chunk
        float sv[4];
        float cmax = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float x = st[0][r];
#pragma unroll
          for (int hh = 1; hh < HP; ++hh) x = hsel == hh ? st[hh][r] : x;
          sv[r] = (4 * g4 + r < nv_cur) ? x * scale_log2 : -INFINITY;
          cmax = fmaxf(cmax, sv[r]);
        }
        cmax = fmaxf(cmax, __shfl_xor(cmax, 16, 64));
        cmax = fmaxf(cmax, __shfl_xor(cmax, 32, 64));
        const float m_new = fmaxf(m_run, cmax);
        const float alpha = (m_new == -INFINITY) ? 1.f : fast_exp2(m_run - m_new);
        float p[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) p[r] = (sv[r] == -INFINITY) ? 0.f : fast_exp2(sv[r] - m_new);
        l_run = l_run * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
        m_run = m_new;
        if (alpha != 1.f) {
#pragma unroll
          for (int db = 0; db < kDb; ++db) acc[db] *= alpha;
        }
        const uint2 pw = {cvt_pk16<H16>(p[0], p[1]), cvt_pk16<H16>(p[2], p[3])};
        if constexpr (kShared) {  // V over the K rows: the S^T reads above come first
#pragma unroll
          for (int r = 0; r < kLoads; ++r) {
            const int row = (kRpl * r + lane / kLpr) * kVRow;
            if constexpr (F8) {
              u32x4_t lo, hi;
              fp8x16_to_bf16(vreg[s][r], lo, hi);
              *reinterpret_cast<u32x4_t*>(&vbuf[sh][row + stage_off<F8, D>(sd)]) = lo;
              *reinterpret_cast<u32x4_t*>(&vbuf[sh][row + stage_off<F8, D>(sd + 8)]) = hi;
            } else {
              *reinterpret_cast<u32x4_t*>(&vbuf[sh][row + sd]) = vreg[s][r];
            }
          }
          if constexpr (kRefill) {
            __builtin_amdgcn_sched_barrier(0);
            issue(nxt, s);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        // P^T per head: a column's weights only in its own head's product
        i16x4_t pbh[HP];
#pragma unroll
        for (int hh = 0; hh < HP; ++hh)
          pbh[hh] = __builtin_bit_cast(i16x4_t, (HP == 1 || hsel == hh) ? pw : uint2{0u, 0u});
        // O^T[dims][cols] += V^T[dims][keys] P^T[keys][cols], 16 dims per MFMA
#pragma unroll
        for (int db = 0; db < kDb; ++db) {
#pragma unroll
          for (int hh = 0; hh < HP; ++hh) {
            const i16x4_t va = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (lds_i16x4_t*)&vbuf[hh][tr_row * kVRow + stage_off<F8, D>(db * 16 + tr_col)]);
            acc[db] = mfma_16x16x16<H16>(va, pbh[hh], acc[db]);
          }
        }
      };

      // Ring schedule over the window padded to a multiple of kRing: every
      // group but the last refills each slot once its rows are staged
      // (branch-free, so the wait counts stay exact); the last group drains.
      const int n_groups = (wn + kRing - 1) / kRing;
#pragma unroll
      for (int s = 0; s < kRing; ++s) issue(s, s);
      for (int gi = 0; gi + 1 < n_groups; ++gi) {
#pragma unroll
        for (int s = 0; s < kRing; ++s)
          consume(s, std::integral_constant<bool, true>{}, (gi + 1) * kRing + s);
      }
#pragma unroll
      for (int s = 0; s < kRing; ++s) consume(s, std::integral_constant<bool, false>{}, 0);
    }

    // ---- segment epilogue: l over the four key groups, then the partial
    l_run += __shfl_xor(l_run, 16, 64);
    l_run += __shfl_xor(l_run, 32, 64);
    if constexpr (F8) {
#pragma unroll
      for (int db = 0; db < kDb; ++db) acc[db] *= v_scale;
    }
    // partial row (wi + b) * HPG + col of the group; the wave that ends the segment
    // writes each of its KV heads' descriptor {first row, count, row stride}
    const int prow0 = (wi + b) * HPG;
    if (col < HPG) {
      float* pr = gpart + (int64_t)(prow0 + col) * kPartRow;
#pragma unroll
      for (int db = 0; db < kDb; ++db)
        *reinterpret_cast<f32x4_t*>(&pr[db * 16 + g4 * 4]) = acc[db];
      if (g4 == 0) *reinterpret_cast<float2*>(&pr[D]) = float2{m_run, l_run};
    }
    if (c_lo + n_seg == nc && lane < HP) {
      const int64_t first = (int64_t)(Wh + batch) * qh0 + (int64_t)(w_first + b) * HPG +
                            lane * G;
      desc[((int64_t)b * Hk + kvh0 + lane) * NCG + cg] =
          i32x4v_t{(int32_t)first, wi - w_first + 1, HPG, 0};
    }
    k += n_seg;
  }
}

// Merge the partials of one (sequence, query head): O = sum_s 2^(m_s-M) O_s /
// sum_s 2^(m_s-M) l_s. Lane l owns output dims N*l .. N*l+N-1. WAVES = 1: the calling wave
// alone. WAVES > 1: the waves of a workgroup share the partials, wave w those with
// s % WAVES == w (in its lane s / WAVES), and merge once more through LDS: a context that many
// waves shared has up to kMaxSlots, and one wave took 10.3 us over a 23001-token sequence's 120
// (a round trip for every eight rows), four waves with 32 rows in flight each 4.2 us.
template <int D, bool H16, int WAVES, typename Seqs>
__device__ __forceinline__ void decode_combine(
    const Seqs seqs, const int b, const int h, int32_t Hq, int32_t Hk, int32_t NCG,
    const float* __restrict__ part, const i32x4v_t* __restrict__ desc,
    bf16_t* __restrict__ out, int64_t out_row_stride) {
  static_assert(decode_dim_ok(D), "head_dim 64, 128 or 256");
  static_assert(WAVES == 1 || !Seqs::kZeroInvalid, "each wave would weigh the keys past the table");
  constexpr int N = D / 64;
  constexpr int kPartRow = part_row(D);
  constexpr int kPer = (kMaxSlots + 64 * WAVES - 1) / (64 * WAVES);  // (m, l) pairs a lane holds
  constexpr int kFirst = WAVES > 1 ? 32 : 16;  // rows in flight with the (m, l) pairs
  const int lane = threadIdx.x & 63;
  const int wave = WAVES > 1 ? __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) : 0;
  const int G = Hq / Hk;
  // The context length and the KV head's descriptor first (one round trip), then every
  // (m, l) pair and the first partial rows at once (the second).
  const int ctx = seqs.keys(b);
  const int hq = h % G;                         // query head within the KV head's group
  const int cg = NCG > 1 ? hq / kMaxCols : 0;    // its column group (0 unless G > 16)
  const i32x4v_t d = desc[((int64_t)b * Hk + h / G) * NCG + cg];
  bf16_t* op = out + seqs.row(b) * out_row_stride + (int64_t)h * D + N * lane;
  float o[N];
#pragma unroll
  for (int i = 0; i < N; ++i) o[i] = 0.f;
  // the descriptor is written by this call for every sequence with ctx > 0
  const int n_all = ctx > 0 ? min(d.y, kMaxSlots) : 0;
  if (n_all == 0) {  // uniform
    if (wave == 0) store_dims<N, H16>(op, o, 0.f);
    return;
  }
  // this wave's partials: s = wave + WAVES * j, j < ns
  const int ns = (n_all - wave + WAVES - 1) / WAVES;
  const int64_t stride = (int64_t)d.z * kPartRow * WAVES;  // floats between them
  const float* pbase = part + ((int64_t)d.x + hq - cg * kMaxCols) * kPartRow +
                       (int64_t)d.z * kPartRow * wave;
  const float* po = pbase + N * lane;
  float2 ml[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    ml[k] = float2{-INFINITY, 0.f};
    const int j = lane + 64 * k;
    if (j < ns) ml[k] = *reinterpret_cast<const float2*>(pbase + j * stride + D);
  }
  float v0[kFirst][N];
#pragma unroll
  for (int u = 0; u < kFirst; ++u) {
    if (u < ns) {
      load_dims<N>(po + u * stride, v0[u]);
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) v0[u][i] = 0.f;
    }
  }
  // the wave's max and the weights w_s = 2^(m_s - M) with two wave reductions, then each lane
  // accumulates its output dims over the partials in order (the first came with the
  // (m, l) pairs; the rest in batches of eight loads in flight)
  float M = ml[0].x;
#pragma unroll
  for (int k = 1; k < kPer; ++k) M = fmaxf(M, ml[k].x);
  M = wave_max(M);
  int past = 0;  // zero keys past the table: score 0
  if constexpr (Seqs::kZeroInvalid) {
    past = max(ctx - seqs.max_tokens, 0);
    if (past > 0) M = fmaxf(M, 0.f);
  }
  float w[kPer], L = 0.f;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    w[k] = (ml[k].x == -INFINITY) ? 0.f : fast_exp2(ml[k].x - M);
    L += w[k] * ml[k].y;
  }
  L = wave_sum(L);
  if (past > 0) L = fmaf((float)past, fast_exp2(-M), L);
#pragma unroll
  for (int u = 0; u < kFirst; ++u) {
    const float wu = __shfl(w[0], u, 64);
    if (u < ns) {  // uniform
#pragma unroll
      for (int i = 0; i < N; ++i) o[i] = fmaf(wu, v0[u][i], o[i]);
    }
  }
  for (int s = kFirst; s < ns; s += 8) {  // uniform
    float v[8][N];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (s + u < ns) load_dims<N>(po + (s + u) * stride, v[u]);
    }
    float wk = w[0];  // uniform select: eight rows never straddle two of a lane's weights
#pragma unroll
    for (int k = 1; k < kPer; ++k) wk = s >= 64 * k ? w[k] : wk;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float wu = __shfl(wk, (s + u) & 63, 64);
      if (s + u < ns) {
#pragma unroll
        for (int i = 0; i < N; ++i) o[i] = fmaf(wu, v[u][i], o[i]);
      }
    }
  }
  if constexpr (WAVES > 1) {
    __shared__ float so[WAVES][N][64];
    __shared__ float2 sml[WAVES];
#pragma unroll
    for (int i = 0; i < N; ++i) so[wave][i][lane] = o[i];
    if (lane == 0) sml[wave] = float2{M, L};
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int x = 1; x < WAVES; ++x) M = fmaxf(M, sml[x].x);
    L = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) o[i] = 0.f;
#pragma unroll
    for (int x = 0; x < WAVES; ++x) {
      const float2 p = sml[x];
      const float wx = p.x == -INFINITY ? 0.f : fast_exp2(p.x - M);
      L = fmaf(wx, p.y, L);
#pragma unroll
      for (int i = 0; i < N; ++i) o[i] = fmaf(wx, so[x][i][lane], o[i]);
    }
  }
  store_dims<N, H16>(op, o, L > 0.f ? 1.f / L : 0.f);
}

}  // namespace nkv
