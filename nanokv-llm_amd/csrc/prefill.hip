// Varlen causal prefill over the paged K/V cache (bf16 MFMA, fp32 softmax).
//
// Reference: flash_attn_varlen_func(q, k, v, max_seqlen_q, cu_seqlens_q,
// max_seqlen_k, cu_seqlens_k, softmax_scale, causal=True, block_table) at
// nanokvllm/layers/attention.py:96-102 (bottom-right causal alignment: query
// j of a sequence with Lq queries and Lk keys sees keys 0 .. Lk-Lq+j).
//
// MI355X design (MFMA-bound):
//  * Workgroup = (sequence, tile of floor(R/g) queries, KV head) x 4 waves.
//    The tile's R "rows" are its queries for all g query heads of the KV
//    head, query-major (row r = query r/g, head r%g; rows past the tile's
//    queries x g are computed and dropped), so one K/V tile in LDS serves g
//    heads (GQA sharing). Wave w owns up to three 16-row groups at head_dim 128
//    (R = 192), two at 64 and in the fp8 instance (R = 128), one at 256
//    (R = 64, and the 128 KiB ring leaves one workgroup per CU); fewer where
//    the batch has few tiles (plain_groups). head_dim D is 64, 128 or 256 (a
//    template parameter).
//  * Keys advance in 64-key steps. Each step's K and V tiles (2 x 16 KiB at
//    D = 128) go from HBM straight into LDS with gfx950's 16-byte buffer-load-to-LDS
//    (no staging registers, no LDS write instructions) through a ring of
//    kStages tiles, issued kStages-1 steps ahead; one barrier per step.
//    LDS rows are dense (2D bytes) with the 16-byte chunks of row r XOR-permuted
//    by chunk_swz(r), which keeps both the K row reads and the V transpose reads
//    free of bank conflicts; the permutation is applied on the global side
//    (each lane fetches the chunk that belongs at its fixed LDS slot).
//  * S^T = K Q^T  (v_mfma_f32_16x16x32_bf16: A = 16 keys from LDS, B = the
//    wave's Q^T held in registers for the whole sequence) puts, in lane l,
//    row l%16 and keys 4(l/16)..+3 of each 16-key quarter. Two quarters make
//    the B operand of  O^T += V^T P^T  (16x16x32 over 32 keys) once their
//    weights are packed to bf16; V^T (A operand) comes from LDS with two
//    ds_read_b64_tr_b16 per 16-dim block and 32-key chunk. Each lane owns one row: the
//    online softmax needs one max over the 4 key groups per step.
//  * Causal: a tile stops at its last visible key; masks are applied per
//    element only where needed. Tiles are dispatched largest-first and the
//    KV head is the fastest grid index, so with 8 KV heads each head's tiles
//    share one XCD's L2.
//  * F8 (paged fp8 pool): K/V tiles come as 1-byte E4M3FN codes through
//    registers instead of straight into LDS: the next step's codes are loaded
//    while this step computes, then widened to bf16 (exact) and written to the
//    same swizzled LDS rows, so the MFMA part is the bf16 kernel's. The K scale
//    is folded into the softmax scale, the V scale into the final 1/l.
//  * Split launch (nkv_prefill_varlen_split): where few tiles or one long context would leave
//    the chip idle, the resident workgroups take equal ranges of all (tile, key step) work and a
//    second kernel merges the cut tiles; decode rows (one new token) are streamed by waves of
//    workgroups of their own, as the decode kernel does.
#include "decode_stream.h"
#include "launch_rules.h"

#include <algorithm>
#include <type_traits>

namespace nkv {

constexpr int kStep = 64;                 // keys per step
constexpr int kStages = 2;                // LDS ring depth (steps)
constexpr bool prefill_dim_ok(int D) { return D == 64 || D == 128 || D == 256; }
// Most 16-row groups per wave: three at head_dim 128 (each K and V^T read from LDS serves three
// MFMAs; bit-identical to two, at par to 2% faster), two at 64 and in the fp8 instance (whose
// staging registers leave no room for a third), one at 256 (its O^T and Q^T registers
// would not fit two waves per SIMD otherwise)
constexpr int prefill_row_groups(int D, bool F8) {
  return D == 256 ? 1 : (D == 128 && !F8 ? 3 : 2);
}
// rows (query, head pairs) of the largest tile, the split launch's: 4 waves
constexpr int prefill_tile_rows(int D, bool F8) { return 64 * prefill_row_groups(D, F8); }
// largest GQA group, the same for every instance of a head_dim: each tile holds at least
// one query for all g heads of its KV head
constexpr int prefill_max_group(int D) { return D == 256 ? 64 : 128; }
// XOR applied to the 16-byte chunk index of LDS row r (even: chunk pairs stay together).
// Keeps the K row reads and the V transpose reads free of bank conflicts: 2*(r & 7) for
// 256- and 512-byte rows, 2*((r >> 1) & 3) for 128-byte rows (two rows per bank line).
template <int D>
__device__ __forceinline__ int chunk_swz(int r) {
  if constexpr (D == 64) return 2 * ((r >> 1) & 3);
  else return 2 * (r & 7);
}
constexpr float kLazy = 8.f;              // log2 headroom before the running max is raised

typedef __attribute__((address_space(3))) u32x4_t lds_u32x4_t;
typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));

// Output pair: bf16 with the round-to-nearest-even of pack_bf16x2, or fp16.
template <bool H16>
__device__ __forceinline__ uint32_t out_pack(float a, float b) {
  if constexpr (H16) return cvt_pk16<true>(a, b);
  else return pack_bf16x2(a, b);
}
// Raw buffer descriptor over [base, base + bytes): loads past `bytes` return 0.
__device__ __forceinline__ i32x4_t buffer_desc(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)(uintptr_t)base;
  return i32x4_t{__builtin_amdgcn_readfirstlane((int32_t)(uint32_t)a),
                 __builtin_amdgcn_readfirstlane((int32_t)((a >> 32) & 0xffffu)),
                 __builtin_amdgcn_readfirstlane((int32_t)bytes), kBufferFlags};
}
// 16 bytes per lane from desc+voff into LDS at lds_addr + 16 * lane. Written as
// asm so that the compiler does not add a wait for it before every barrier;
// the ring's own s_waitcnt (vmcnt) orders it.
__device__ __forceinline__ void load_to_lds(i32x4_t desc, uint32_t lds_addr, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               :
               : "s"(lds_addr), "v"(voff), "s"(desc)
               : "memory");
}

// ---------------------------------------------------------------- split keys
// What the split launch adds to the plain one's arguments.
struct SplitArgs {
  int32_t n_seqs;
  int32_t min_range;   // shortest range, in cost units
  i32x4_t* desc;       // one per workgroup: {parts, first row of q, queries, KV head}
  float* part;         // two tiles of partial rows per workgroup
  int32_t ncg;         // the decode rows' column groups, their shortest range in chunks,
  int32_t min_chunks;  // descriptors and partial rows (decode_stream.h)
  i32x4v_t* row_desc;
  float* row_part;
  int32_t max_tokens;  // keys that a table row holds
  float chunk_cost;    // row_cost
};
constexpr int kSnap = 2;  // a range never cuts a unit within this many steps of its ends

// Floats of a partial row: O, m, l, 2 pad.
constexpr int prefill_part_row(int D) { return D + 4; }

constexpr int kMinRange = 4 * kFullStep;
// Shortest range over all heads' T tile steps: sqrt(T) / 6 steps. A range's part costs about 7
// steps to write and merge (100 KB each way), so halving the ranges of a small call gains until
// its steps take as long: four chunks of 75 - 195 tokens on 2650 (Hq 16, Hk 2) 52.5 -> 46.4 us;
// no range of a call that fills the chip is touched.
constexpr float kRangeRoot = 1.f / 6.f;
// Cost of one key step of a tile with `rows` rows.
template <int D, bool F8>
__device__ __forceinline__ int step_cost(int rows) {
  constexpr int kWaveRows = 16 * prefill_row_groups(D, F8);
  return kStepBase + (rows + kWaveRows - 1) / kWaveRows;
}
// Key steps of tile t (at least one, which an empty tile masks whole).
__device__ __forceinline__ int tile_steps(int Lq, int Lk, int qt, int t) {
  const int last = Lk - Lq + min(Lq, (t + 1) * qt) - 1;
  return last >= 0 ? last / kStep + 1 : 1;
}

// The decode rows among prompts (sequences that bring one new token; HP > 0, the KV heads a
// wave reads at once) are no units of the stream below: waves of workgroups of their own
// stream them as the decode kernel does, bound by the K/V bytes, beside the workgroups that
// the prompts' tiles keep at the matrix cores. A 192-row tile for one row ran at 5.2 TB/s of
// K/V (a 256-byte piece of each row and 64 keys in flight a workgroup; decode_stream: 6.5).

// The ranges of the split launch. The units of a KV head (sequence, tile) stand in one
// stream, a unit as long as its cost; range w is [w*C, (w+1)*C), with a cut that falls near
// a unit's end moved to that end. Every workgroup finds its own range from cu_seqlens.
struct SplitCursor {
  int seq, tile, q0, Lq, kb0, Lk;  // the current unit
  int u0;                          // its position in the stream
  int C, T, x, x_end;              // range length, stream length, the range's begin and end
  int group;                       // this workgroup's index among those of the tiles
  int row_groups;                  // workgroups of the decode rows: the first of the grid
};

// false: nothing to do, or (row_groups > blockIdx.x) the decode rows.
template <int D, bool F8, int HP>
__device__ __forceinline__ bool split_begin(const SplitArgs& sa,
                                            const int32_t* __restrict__ cu_q,
                                            const int32_t* __restrict__ cu_k, int qt, int G,
                                            int Hk, SplitCursor& c) {
  constexpr bool ROWS = HP > 0;
  const int lane = threadIdx.x & 63;
  int Lq = 0, Lk = 0, cost = 0, incl = 0;
  int chunks = 0;  // lane: of the decode rows
  auto load = [&](int cb) {  // lane: sequence cb + lane
    const int s = cb + lane;
    Lq = 0;
    Lk = 0;
    if (s < sa.n_seqs) {
      Lq = cu_q[s + 1] - cu_q[s];
      Lk = cu_k[s + 1] - cu_k[s];
      NKV_DBG(blockIdx.x == 0 && (Lq < 0 || Lk < 0 || Lq > Lk), NKV_DEBUG_LENGTH);
    }
    if (ROWS && Lq == 1) {
      chunks += seq_chunks(Lk, sa.max_tokens);
      Lq = 0;
    }
    cost = 0;
    for (int t = 0; t * qt < Lq; ++t)
      cost += tile_steps(Lq, Lk, qt, t) * step_cost<D, F8>(min(qt, Lq - t * qt) * G);
    incl = wave_incl_scan(cost);
    return __builtin_amdgcn_readlane(incl, 63);
  };
  int T = 0;
  for (int cb = 0; cb < sa.n_seqs; cb += 64) T += load(cb);
  c.T = T;
  int n_ranges = (int)gridDim.x / Hk;  // of each KV head
  c.row_groups = 0;
  if constexpr (ROWS) {
    const SplitShare share =
        split_share(n_ranges, __builtin_amdgcn_readlane(wave_incl_scan(chunks), 63),
                    sa.chunk_cost, T, sa.ncg, HP);
    n_ranges = share.tiles;
    c.row_groups = share.rows * Hk;
    if ((int)blockIdx.x < c.row_groups) return false;
  }
  c.group = (int)blockIdx.x - c.row_groups;
  const float steps = (float)T * (float)Hk / kFullStep;
  c.C = max(max((T + n_ranges - 1) / max(n_ranges, 1), sa.min_range),
            (int)(sqrtf(steps) * (kRangeRoot * kFullStep)));
  const int x = c.group / Hk * c.C;
  if (x >= T) return false;
  c.x = x;
  c.x_end = x + c.C;
  int base = 0, cb = 0;
  int tot = load(0);
  while (x >= base + tot) {
    base += tot;
    cb += 64;
    tot = load(cb);
  }
  const int ln = __builtin_amdgcn_readfirstlane(__builtin_ctzll(__ballot(base + incl > x)));
  c.seq = cb + ln;
  c.Lq = __builtin_amdgcn_readlane(Lq, ln);
  c.Lk = __builtin_amdgcn_readlane(Lk, ln);
  c.u0 = base + __builtin_amdgcn_readlane(incl, ln) - __builtin_amdgcn_readlane(cost, ln);
  c.tile = 0;
  for (;;) {
    const int u = tile_steps(c.Lq, c.Lk, qt, c.tile) *
                  step_cost<D, F8>(min(qt, c.Lq - c.tile * qt) * G);
    if (x < c.u0 + u) break;
    c.u0 += u;
    ++c.tile;
  }
  c.q0 = cu_q[c.seq];
  c.kb0 = cu_k[c.seq];
  return true;
}

// The unit after the current one (false at the end of the stream).
template <bool ROWS>
__device__ __forceinline__ bool split_next(const int32_t* __restrict__ cu_q,
                                           const int32_t* __restrict__ cu_k, int qt, int u1,
                                           SplitCursor& c) {
  c.u0 = u1;
  if (u1 >= c.T) return false;
  if (++c.tile * qt < c.Lq) return true;
  c.tile = 0;
  do {  // ends: the stream has more units
    ++c.seq;
    c.q0 = cu_q[c.seq];
    c.Lq = cu_q[c.seq + 1] - c.q0;
  } while (c.Lq <= (ROWS ? 1 : 0));
  c.kb0 = cu_k[c.seq];
  c.Lk = cu_k[c.seq + 1] - c.kb0;
  return true;
}

// One workgroup's work: a whole tile of a sequence (plain), or its range of the stream of
// units, each unit's key steps [s_lo, s_end) of n_steps (SPLIT).
// HP (SPLIT, paged): KV heads a wave of the decode rows reads at once, 0 for decode rows as
// tiles of one query.
template <bool F8, int D, bool H16, bool PAGED, int RG, bool SPLIT, int HP = 0>
__device__ __forceinline__ void prefill_body(
    const bf16_t* __restrict__ q, int64_t q_row_stride, const void* __restrict__ k_cache,
    const void* __restrict__ v_cache, int64_t k_row_stride, int64_t v_row_stride,
    const int32_t* __restrict__ cu_seqlens_q, const int32_t* __restrict__ cu_seqlens_k,
    const int32_t* __restrict__ block_tables, int64_t bt_row_stride, int32_t Hk, int32_t G,
    int32_t block_size, int32_t max_blocks, int32_t n_limit, int32_t n_tiles, float scale_log2,
    float v_scale, bf16_t* __restrict__ out, int64_t out_row_stride, const SplitArgs sa) {
  static_assert(prefill_dim_ok(D), "head_dim 64, 128 or 256");
  static_assert(!(F8 && H16), "fp8 caches are read with bf16 queries");
  constexpr int kEl = F8 ? 1 : 2;          // bytes per cache element
  constexpr int kRB = D * 2;               // bytes of a staged (bf16) K or V row
  constexpr int kNC = D / 8;               // 16-byte chunks per staged row
  constexpr int kRG = RG;
  constexpr int kTileB = kStep * kRB;      // bytes of one K or V tile
  constexpr int kStageB = 2 * kTileB;      // K tile then V tile
  constexpr int kKs = D / 32;              // k-steps of S^T
  constexpr int kDb = D / 16;              // 16-dim blocks of O^T
  constexpr int kRpl = 1024 / kRB;         // rows per 1 KiB load into LDS
  constexpr int kNl = 16 / kRpl;           // such loads per wave per tile
  constexpr int kLpr8 = D / 16;            // F8: lanes per row (16 codes each)
  constexpr int kRpl8 = 64 / kLpr8;        // F8: rows per load
  constexpr int kNl8 = 16 / kRpl8;         // F8: loads per wave per tile
  const int QT = 64 * RG / G;  // queries per tile
  constexpr int kRowLds = 2 * decode_lds_elems<F8, HP == 0 ? 1 : HP, D>();  // bytes a wave
  constexpr int kRingB = kStages * kStageB;
  __shared__ __attribute__((aligned(1024))) char
      ring[HP > 0 && 4 * kRowLds > kRingB ? 4 * kRowLds : kRingB];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g4 = lane >> 4;
  const int col = lane & 15;

  SplitCursor cur;
  int kvh = blockIdx.x % Hk;
  if constexpr (SPLIT) {
    // no unit of this range is cut at its end, unless one below says so
    if (tid == 0) sa.desc[blockIdx.x] = i32x4_t{0, 0, 0, 0};
    if (!split_begin<D, F8, HP>(sa, cu_seqlens_q, cu_seqlens_k, QT, G, Hk, cur)) {
      if constexpr (HP > 0) {
        if ((int)blockIdx.x < cur.row_groups)
          decode_stream<F8, HP, D, H16>(
              OneRowSeqs{cu_seqlens_q, cu_seqlens_k, sa.n_seqs, sa.max_tokens},
              (int)blockIdx.x * 4 + wave, cur.row_groups * 4,
              reinterpret_cast<bf16_t*>(ring + wave * kRowLds), q, q_row_stride, k_cache, v_cache,
              block_tables, bt_row_stride, Hk, G, sa.ncg, block_size, max_blocks, n_limit,
              sa.min_chunks, scale_log2, v_scale, sa.row_part, sa.row_desc);
      }
      return;  // uniform
    }
    kvh = cur.group % Hk;
  } else {
    const int rest = blockIdx.x / Hk;
    cur.tile = n_tiles - 1 - rest % n_tiles;  // largest tiles first
    cur.seq = rest / n_tiles;
    cur.q0 = cu_seqlens_q[cur.seq];
    cur.Lq = cu_seqlens_q[cur.seq + 1] - cur.q0;
    cur.kb0 = cu_seqlens_k[cur.seq];
    cur.Lk = cu_seqlens_k[cur.seq + 1] - cur.kb0;
  }
  int u1 = 0;        // the unit's end in the stream
  int snap = 0;      // a cut this near to the unit's ends moves there
  bool cut = false;  // the range ends inside the unit
  do {  // plain: once
  // A uniform value into a scalar register. The empty asm hides that it is uniform: the
  // compiler would drop the readfirstlane and keep the step's bookkeeping in VALU code.
  const auto uni = [](int v) {
    if constexpr (SPLIT) {
      asm("" : "+v"(v));
      v = __builtin_amdgcn_readfirstlane(v);
    }
    return v;
  };
  const int seq = uni(cur.seq), tile = uni(cur.tile);
  const int q0 = uni(cur.q0), Lq = uni(cur.Lq), kb0 = uni(cur.kb0), Lk = uni(cur.Lk);
  const int j0 = tile * QT;
  if constexpr (!SPLIT) {
    NKV_DBG(tid == 0 && tile == 0 && (Lq < 0 || Lk < 0 || Lq > Lk), NKV_DEBUG_LENGTH);
    if (j0 >= Lq) return;  // uniform
  }
  const int diag = Lk - Lq;  // query j sees keys <= diag + j
  const int last_key = min(Lk - 1, diag + j0 + QT - 1);
  int n_steps = last_key >= 0 ? last_key / kStep + 1 : 0;
  int s_lo = 0, s_end = n_steps;
  if constexpr (SPLIT) {
    n_steps = max(n_steps, 1);
    const int sc = step_cost<D, F8>(min(QT, Lq - j0) * G);
    snap = kSnap * sc;
    u1 = cur.u0 + n_steps * sc;
    // the range's begin may lie in its first unit
    if (cur.x >= cur.u0 + snap) {
      if (cur.x > u1 - snap) continue;  // it belongs to the range before (the loop's condition
                                    // steps to the next unit)
      s_lo = (cur.x - cur.u0 + sc - 1) / sc;
    }
    cut = false;
    if (cur.x_end < u1 && cur.x_end < cur.T) {  // the range ends within this unit
      if (cur.x_end < cur.u0 + snap) return;    // near its begin: it is the next range's
      cut = cur.x_end <= u1 - snap;
    }
    s_lo = uni(s_lo);
    s_end = uni(cut ? (cur.x_end - cur.u0 + sc - 1) / sc : n_steps);
  }
  // A part of the unit goes to one of the workgroup's two slots: the end of a unit begun
  // before its range, and the beginning of one that goes on after it. The latter's
  // workgroup describes the unit to the merge.
  auto part_tile = [&]() {
    return sa.part + ((int64_t)blockIdx.x * 2 + (s_lo == 0)) *
                         (64 * RG * prefill_part_row(D));
  };
  auto describe = [&]() {
    const int w0 = (cur.u0 + snap + cur.C - 1) / cur.C;  // the unit's first cut
    sa.desc[blockIdx.x] = i32x4_t{(u1 - snap) / cur.C - w0 + 2, q0 + j0, min(QT, Lq - j0), kvh};
  };
  const int k_lim = SPLIT ? min(Lk, s_end * kStep) : Lk;  // keys to load

  // ---- K/V tile loads. Wave w fills rows 16w .. 16w+15 of a tile with 1 KiB
  // loads (kRpl rows each: 4 at head_dim 128); lane i of load h lands at row
  // 16w + kRpl*h + i/kNC, slot i%kNC, and fetches the row's chunk
  // (i%kNC) ^ chunk_swz(row). A wave's 16
  // keys are consecutive rows (one cache block, B % 16 == 0, or the contiguous
  // K/V), so each wave's share of a step is one uniform base row and a byte
  // window covering only its valid keys: keys past Lk and keys of invalid
  // blocks read as 0. vol[] are the K offsets; V rows may have another stride
  // (contiguous mode), and their offsets differ by r * (row_bv - row_b).
  const uint32_t row_b = (uint32_t)k_row_stride * kEl;
  const uint32_t row_bv = (uint32_t)v_row_stride * kEl;
  const int lrow = lane / kNC;
  const int slot = lane % kNC;
  uint32_t vol[kNl];
#pragma unroll
  for (int h = 0; h < kNl; ++h) {
    const int r = kRpl * h + lrow;  // row within the wave's 16 (16w + r within the tile)
    vol[h] = (uint32_t)r * row_b + (uint32_t)kvh * (D * 2) +
             (uint32_t)(slot ^ chunk_swz<D>(r)) * 16u;
  }
  const uint32_t ring_base =
      (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)ring +
      (uint32_t)wave * (16u * kRB);
  // F8: load f of the wave's K (or V) codes brings rows kRpl8*f + lane/kLpr8, bytes
  // 16*(lane%kLpr8) of the head's D-byte piece, i.e. logical bf16 chunks 2c, 2c+1
  // (c = lane%kLpr8) of that LDS row
  const int f8_row0 = lane / kLpr8;
  const int f8_c = lane % kLpr8;
  u32x4_t kq[kNl8], vq[kNl8];  // F8: the next step's codes

  // Block ids: lane i holds entry bt_base + i of the sequence's table row, read
  // by the uniform v_readlane of the wave's block (reloaded every 64 blocks).
  const int32_t* bt = PAGED ? block_tables + (int64_t)seq * bt_row_stride : nullptr;
  int bt_base = 0;
  int bt_lane = -1;
  auto load_window = [&]() {
    const int e = bt_base + lane;
    const int id = e < max_blocks ? bt[e] : -1;
    NKV_DBG((int64_t)e * block_size < Lk && (e >= max_blocks || id < 0 || id >= n_limit),
            e >= max_blocks ? NKV_DEBUG_LENGTH : NKV_DEBUG_BLOCK);
    bt_lane = (id >= 0 && id < n_limit) ? id : -1;
  };
  // cursor of this wave's rows in the step loaded next: first key c_t0,
  // block c_blk, offset c_off in it
  int c_t0 = 0, c_blk = 0, c_off = 0;
  int c_left = 0;  // SPLIT: steps to load
  auto seek = [&](int s) {
    c_t0 = s * kStep + 16 * wave;
    if constexpr (PAGED) {
      c_blk = uni(c_t0 / block_size);
      c_off = c_t0 - c_blk * block_size;
      bt_base = c_blk & ~63;
      load_window();
    }
  };
  // SPLIT: the part's first step. Its steps go round: from s_first to s_end, then from s_lo. At
  // any time the workgroups of a KV head are then at one of a few steps, those that are the
  // same modulo the range's length, and each K/V row that several tiles need is read while
  // the L2 holds it.
  int s_first = s_lo;
  if constexpr (SPLIT) {
    const int rl = cur.C / step_cost<D, F8>(QT * G);
    const int f = (s_lo + rl - 1) / rl * rl;
    if (f < s_end) s_first = f;
    s_first = uni(s_first);
    c_left = s_end - s_lo;
  }
  seek(s_first);
  // Scalar selects only (no branches), so that the compiler can spread it between the
  // MFMAs that follow its call.
  auto issue = [&](int stage) {
    int nv = uni(min(16, k_lim - c_t0));
    int64_t row0;
    if constexpr (PAGED) {
      const int pb = __builtin_amdgcn_readlane(bt_lane, c_blk - bt_base);
      nv = pb < 0 ? 0 : nv;
      row0 = (int64_t)pb * block_size + c_off;
    } else {
      const int r0 = kb0 + c_t0;
      NKV_DBG(nv > 0 && (r0 < 0 || r0 > n_limit - nv), NKV_DEBUG_BLOCK);
      nv = (r0 < 0 || r0 > n_limit - nv) ? 0 : nv;  // outside the K/V rows
      row0 = r0;
    }
    nv = max(nv, 0);
    row0 = nv > 0 ? row0 : 0;
    const char* kp = static_cast<const char*>(k_cache) + row0 * k_row_stride * kEl;
    const char* vp = static_cast<const char*>(v_cache) + row0 * v_row_stride * kEl;
    if constexpr (F8) {  // into registers; widened into the stage by commit()
      (void)stage;
      const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
          (void*)kp, (short)0, (uint32_t)nv * row_b, kBufferFlags);
      const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
          (void*)vp, (short)0, (uint32_t)nv * row_bv, kBufferFlags);
#pragma unroll
      for (int f = 0; f < kNl8; ++f) {
        const uint32_t r = (uint32_t)(kRpl8 * f + f8_row0);
        const uint32_t col = (uint32_t)kvh * D + (uint32_t)f8_c * 16u;
        kq[f] = __builtin_bit_cast(
            u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rk, r * row_b + col, 0, 0));
        vq[f] = __builtin_bit_cast(
            u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rv, r * row_bv + col, 0, 0));
      }
    } else {
      const i32x4_t dk = buffer_desc(kp, (uint32_t)nv * row_b);
      const i32x4_t dv = buffer_desc(vp, (uint32_t)nv * row_bv);
      const uint32_t at = ring_base + (uint32_t)stage * kStageB;
#pragma unroll
      for (int h = 0; h < kNl; ++h) load_to_lds(dk, at + 1024u * h, vol[h]);
#pragma unroll
      for (int h = 0; h < kNl; ++h)
        load_to_lds(dv, at + kTileB + 1024u * h,
                    vol[h] + (uint32_t)(kRpl * h + lrow) * (row_bv - row_b));
    }
    c_t0 += kStep;
    if constexpr (PAGED) {  // blocks crossed: at most 4 (c_off < block_size, a multiple of 16)
      const int v = c_off + kStep;
      const int n = (v >= block_size) + (v >= 2 * block_size) + (v >= 3 * block_size) +
                    (v >= 4 * block_size);
      c_off = v - n * block_size;
      c_blk = uni(__builtin_amdgcn_readfirstlane(c_blk + n));
    }
  };
  auto refill_window = [&]() {  // uniform; once per 64 blocks, and where the steps wrap
    if constexpr (SPLIT) {
      c_left = uni(c_left - 1);
      if (c_left <= 0) c_t0 = k_lim;  // the steps after the last bring no row
      else if (c_t0 >= s_end * kStep) seek(s_lo);
    }
    if constexpr (PAGED) {
      if (c_blk - bt_base >= 64) {
        bt_base = c_blk & ~63;
        load_window();
      }
    }
  };
  // F8: the codes of the last issue() (after their loads land) widened into LDS stage
  // `stage`, rows 16w .. 16w+15 of the K and V tiles, in the bf16 path's swizzled layout
  // Lanes in the second half of a row write their pair's second chunk first (their codes'
  // halves swapped before widening), so each 16-byte write instruction covers distinct
  // bank groups of a row instead of pairing them up.
  const bool f8_swap = f8_c >= kLpr8 / 2;
  auto commit = [&](int stage) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    char* at = ring + stage * kStageB + wave * (16 * kRB);
#pragma unroll
    for (int f = 0; f < kNl8; ++f) {
      const int r = kRpl8 * f + f8_row0;  // row within the wave's 16 (16w + r within the tile)
      const int off = r * kRB + ((2 * f8_c) ^ chunk_swz<D>(r)) * 16;  // chunks 2c, 2c+1: adjacent
      const int o1 = off + (f8_swap ? 16 : 0), o2 = off + (f8_swap ? 0 : 16);
      u32x4_t lo, hi;
      u32x4_t c = kq[f];
      if (f8_swap) c = u32x4_t{c[2], c[3], c[0], c[1]};
      fp8x16_to_bf16(c, lo, hi);
      *reinterpret_cast<u32x4_t*>(at + o1) = lo;
      *reinterpret_cast<u32x4_t*>(at + o2) = hi;
      c = vq[f];
      if (f8_swap) c = u32x4_t{c[2], c[3], c[0], c[1]};
      fp8x16_to_bf16(c, lo, hi);
      *reinterpret_cast<u32x4_t*>(at + kTileB + o1) = lo;
      *reinterpret_cast<u32x4_t*>(at + kTileB + o2) = hi;
    }
  };

  // ---- prologue: the first kStages-1 steps in flight, then Q
#pragma unroll
  for (int st = 0; st < kStages - 1; ++st) {
    issue(st);
    refill_window();
  }

  if constexpr (SPLIT) {
    // a wave past the tile's rows only brings its share of the K/V rows
    if (wave * (16 * kRG) >= min(QT, Lq - j0) * G) {
      for (int s = s_lo; s < s_end; ++s) {  // any order: only the count matters
        if constexpr (F8) commit((s - s_lo) % kStages);
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();  // step s's tile is whole, the stage of s - 1 free
        if (s + 1 < s_end) issue((s - s_lo + 1) % kStages);
        refill_window();
      }
      __syncthreads();
      continue;
    }
  }

  // ---- this wave's row groups: head and query of this lane's row (query-major;
  // rows past QT*G take query Lq: attended like the others, never stored)
  int head[kRG], jrow[kRG];
#pragma unroll
  for (int rr = 0; rr < kRG; ++rr) {
    const int r = (wave * kRG + rr) * 16 + col;
    const bool real = r < QT * G;
    head[rr] = real ? r % G : 0;
    jrow[rr] = real ? j0 + r / G : Lq;
  }
  // Q^T as the MFMA B operand: lane l -> row l%16, dims 8*(l/16) + 32*ks
  u32x4_t qreg[kRG][kKs];
#pragma unroll
  for (int rr = 0; rr < kRG; ++rr) {
    const int jc = jrow[rr] < Lq ? jrow[rr] : j0;  // rows past the sequence: discarded
    const u32x4_t* qp = reinterpret_cast<const u32x4_t*>(
        q + (int64_t)(q0 + jc) * q_row_stride + (int64_t)(kvh * G + head[rr]) * D + g4 * 8);
#pragma unroll
    for (int ks = 0; ks < kKs; ++ks) qreg[rr][ks] = qp[ks * 4];
  }

  // LDS read offsets (bytes from a tile's start). K A operand, 16-key half hh,
  // dims 32ks + 8*g4: row 16hh + col, logical chunk g4 + 4ks.
  uint32_t ko[kKs];
#pragma unroll
  for (int ks = 0; ks < kKs; ++ks)
    ko[ks] = (uint32_t)col * kRB + (uint32_t)((g4 + 4 * ks) ^ chunk_swz<D>(col)) * 16u;
  // V^T via ds_read_b64_tr_b16: lane 16g + 4r + c reads row 4g + r (and +16),
  // dims 16db + 4c .. +3 = logical chunk 2db + c/2, half c%2.
  const int vrow = 4 * g4 + (col >> 2);
  const int vc = col & 3;
  uint32_t vo[kDb];
#pragma unroll
  for (int db = 0; db < kDb; ++db)
    vo[db] = (uint32_t)vrow * kRB + (uint32_t)(db ^ (chunk_swz<D>(vrow) >> 1)) * 32u +
             (uint32_t)vc * 8u;

  f32x4_t acc[kRG][kDb];  // O^T: lane l -> row l%16, dims 16*db + 4*(l/16) .. +3
#pragma unroll
  for (int rr = 0; rr < kRG; ++rr)
#pragma unroll
    for (int db = 0; db < kDb; ++db) acc[rr][db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run[kRG], l_run[kRG];
  float mb_run[kRG];  // m_run, or 0 while the row has no visible key
#pragma unroll
  for (int rr = 0; rr < kRG; ++rr) {
    m_run[rr] = -INFINITY;
    l_run[rr] = 0.f;
    mb_run[rr] = 0.f;
  }

  // Q is in registers before the loop: the empty asm uses pin the loads'
  // completion here, so no wait for them (which would also wait for the ring's
  // loads) lands inside the loop.
#pragma unroll
  for (int rr = 0; rr < kRG; ++rr)
#pragma unroll
    for (int ks = 0; ks < kKs; ++ks) asm volatile("" ::"v"(qreg[rr][ks]));
  // first step's tile landed (each wave waits for its own loads; the barrier
  // publishes all of them)
  if constexpr (F8) {
    commit(0);
  } else {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 * (kStages - 2)) : "memory");
  }
  __syncthreads();

  const char* lds = (const char*)(__attribute__((address_space(3))) char*)ring;
  auto step = [&](auto stage_c, int s, bool more) {
    constexpr int ST = decltype(stage_c)::value;
    if constexpr (F8) issue((ST + kStages - 1) % kStages);  // step s + kStages - 1
    const char* kt = lds + ST * kStageB;
    const char* vt = kt + kTileB;

    // S^T for the four 16-key quarters and the wave's row groups
    f32x4_t st[kRG][4];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      u32x4_t ka[kKs];
#pragma unroll
      for (int ks = 0; ks < kKs; ++ks)
        ka[ks] = *reinterpret_cast<const u32x4_t*>(kt + h * (16 * kRB) + ko[ks]);
      // step s + kStages - 1 into the other stage, after the third quarter's K reads: its
      // scalar work spreads over the QK MFMAs around it (measured against quarters 0, 1 and
      // 3, the PV chunks and the step's start: 2-4% faster than the start)
      if constexpr (!F8) {
        if (h == 2) issue((ST + kStages - 1) % kStages);
      }
#pragma unroll
      for (int rr = 0; rr < kRG; ++rr) {
        f32x4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < kKs; ++ks)
          a = mfma_16x16x32<H16>(ka[ks], qreg[rr][ks], a);
        st[rr][h] = a;
      }
    }
    // online softmax (log2 domain, running max m_run kept scaled). The max is
    // only raised when a row's maximum grows by more than kLazy (log2 units):
    // weights then stay <= 2^kLazy, exact after the final 1/l. Both row groups'
    // maxima first (one rescale branch), then per 32-key chunk the weights,
    // packed as the P^T B operand (8 bf16 per lane), and that chunk's PV
    // MFMAs: chunk 1's exp work overlaps chunk 0's MFMAs. The row sum is taken
    // over the same bf16 weights that multiply V.
    const bool edge = (s * kStep + kStep - 1 > diag + j0) || (s * kStep + kStep > Lk);  // uniform
    float sv[kRG][16];
#pragma unroll
    for (int rr = 0; rr < kRG; ++rr)
#pragma unroll
      for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) sv[rr][4 * h + r] = st[rr][h][r];
    if (edge) {
#pragma unroll
      for (int rr = 0; rr < kRG; ++rr) {
        const int lim = min(diag + jrow[rr], Lk - 1);  // last visible key of this row
#pragma unroll
        for (int h = 0; h < 4; ++h)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (s * kStep + 16 * h + 4 * g4 + r > lim) sv[rr][4 * h + r] = -INFINITY;
      }
    }
    // Each lane first tests its own 16 scores of a row group against the headroom; only
    // when some lane's exceed it does the wave take the row maxima across the 4 lane groups
    // (two permlane swaps) and rescale. The decisions are those of testing the row maxima
    // every step, which rarely rise past the headroom after the first steps.
    float lmax[kRG];
    bool lraise = false;
#pragma unroll
    for (int rr = 0; rr < kRG; ++rr) {
      const float* v = sv[rr];
      lmax[rr] = fmax3(fmax3(fmax3(v[0], v[1], v[2]), fmax3(v[3], v[4], v[5]),
                             fmax3(v[6], v[7], v[8])),
                       fmax3(v[9], v[10], v[11]),
                       fmax3(fmax3(v[12], v[13], v[14]), v[15], -INFINITY));
      lraise = lraise || (lmax[rr] * scale_log2 > m_run[rr] + kLazy);
    }
    if (__builtin_amdgcn_ballot_w64(lraise) != 0) {
#pragma unroll
      for (int rr = 0; rr < kRG; ++rr) {
        const float cm = col_max4(lmax[rr]) * scale_log2;
        const bool raise = cm > m_run[rr] + kLazy;  // false while the row has no visible key
        const float alpha = raise ? fast_exp2(m_run[rr] - cm) : 1.f;  // exp2(-inf) = 0
        m_run[rr] = raise ? cm : m_run[rr];
        mb_run[rr] = m_run[rr] == -INFINITY ? 0.f : m_run[rr];
        l_run[rr] *= alpha;
#pragma unroll
        for (int db = 0; db < kDb; ++db) acc[rr][db] *= alpha;
      }
    }
    const float* mb = mb_run;
    // O^T[dims][rows] += V^T[dims][keys] P^T[keys][rows] per 32-key chunk c:
    // k-slot j of lane group g is key 32c+4g+j (j<4), or 32c+16+4g+(j-4)
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      u32x4_t pb[kRG];
#pragma unroll
      for (int rr = 0; rr < kRG; ++rr) {
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
          p[e] = fast_exp2(fmaf(sv[rr][8 * c + e], scale_log2, -mb[rr]));  // -inf -> 0
        pb[rr] = u32x4_t{cvt_pk16<H16>(p[0], p[1]), cvt_pk16<H16>(p[2], p[3]),
                         cvt_pk16<H16>(p[4], p[5]), cvt_pk16<H16>(p[6], p[7])};
        float l = l_run[rr];
#pragma unroll
        for (int e = 0; e < 4; ++e) l = sum2_16<H16>(pb[rr][e], l);
        l_run[rr] = l;
      }
#pragma unroll
      for (int db = 0; db < kDb; ++db) {
        const char* vc = vt + c * (32 * kRB) + vo[db];
        const i16x4_t v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)vc);
        const i16x4_t v1 =
            __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_t*)(vc + 16 * kRB));
        const u32x4_t va = {__builtin_bit_cast(uint2, v0).x, __builtin_bit_cast(uint2, v0).y,
                            __builtin_bit_cast(uint2, v1).x, __builtin_bit_cast(uint2, v1).y};
#pragma unroll
        for (int rr = 0; rr < kRG; ++rr)
          acc[rr][db] = mfma_16x16x32<H16>(va, pb[rr], acc[rr][db]);
      }
    }
    // next step's tile landed (own loads), then publish and free this stage
    if constexpr (F8) {
      if (more) commit((ST + 1) % kStages);  // uniform
    } else {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(8 * (kStages - 2)) : "memory");
    }
    __syncthreads();
    refill_window();
  };
  static_assert(kStages == 2, "the step loop below is unrolled for 2 stages");
  if constexpr (SPLIT) {
    for (int i = s_lo, s = s_first;;) {
      step(std::integral_constant<int, 0>{}, s, ++i < s_end);
      if (i >= s_end) break;
      s = s + 1 < s_end ? s + 1 : s_lo;
      step(std::integral_constant<int, 1>{}, s, ++i < s_end);
      if (i >= s_end) break;
      s = s + 1 < s_end ? s + 1 : s_lo;
    }
  } else {
    for (int s = 0;;) {
      if (s >= n_steps) break;
      step(std::integral_constant<int, 0>{}, s, s + 1 < n_steps);
      ++s;
      if (s >= n_steps) break;
      step(std::integral_constant<int, 1>{}, s, s + 1 < n_steps);
      ++s;
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into LDS outlives the workgroup

  if constexpr (SPLIT) {
    if (cut || s_lo > 0) {  // a part of the unit: O, m and l as they are (uniform)
      float* tile_part = part_tile();
#pragma unroll
      for (int rr = 0; rr < kRG; ++rr) {
        const float l = col_sum4(l_run[rr]);
        if (jrow[rr] >= Lq) continue;
        float* pr = tile_part + ((wave * kRG + rr) * 16 + col) * prefill_part_row(D);
#pragma unroll
        for (int db = 0; db < kDb; ++db)
          *reinterpret_cast<f32x4_t*>(pr + db * 16 + g4 * 4) = acc[rr][db];
        if (g4 == 0) *reinterpret_cast<float2*>(pr + D) = float2{m_run[rr], l};
      }
      if (s_lo == 0 && tid == 0) describe();
      continue;
    }
  }
  // ---- epilogue: normalise and store this lane's 4 dims of each 16-dim block
#pragma unroll
  for (int rr = 0; rr < kRG; ++rr) {
    const float l = col_sum4(l_run[rr]);
    if (jrow[rr] >= Lq) continue;
    const float inv = l > 0.f ? (F8 ? v_scale : 1.f) / l : 0.f;
    bf16_t* op = out + (int64_t)(q0 + jrow[rr]) * out_row_stride +
                 (int64_t)(kvh * G + head[rr]) * D + g4 * 4;
#pragma unroll
    for (int db = 0; db < kDb; ++db) {
      const uint2 w = {out_pack<H16>(acc[rr][db][0] * inv, acc[rr][db][1] * inv),
                       out_pack<H16>(acc[rr][db][2] * inv, acc[rr][db][3] * inv)};
      *reinterpret_cast<uint2*>(op + db * 16) = w;
    }
  }
  } while (SPLIT && !cut && split_next<(HP > 0)>(cu_seqlens_q, cu_seqlens_k, QT, u1, cur));
}

#define NKV_PREFILL_PARAMS                                                                      \
  const bf16_t *__restrict__ q, int64_t q_row_stride, const void *__restrict__ k_cache,         \
      const void *__restrict__ v_cache, int64_t k_row_stride, int64_t v_row_stride,             \
      const int32_t *__restrict__ cu_seqlens_q, const int32_t *__restrict__ cu_seqlens_k,       \
      const int32_t *__restrict__ block_tables, int64_t bt_row_stride, int32_t Hk, int32_t G,   \
      int32_t block_size, int32_t max_blocks, int32_t n_limit, int32_t n_tiles,                 \
      float scale_log2, float v_scale, bf16_t *__restrict__ out, int64_t out_row_stride
#define NKV_PREFILL_PASS                                                                       \
  q, q_row_stride, k_cache, v_cache, k_row_stride, v_row_stride, cu_seqlens_q, cu_seqlens_k,   \
      block_tables, bt_row_stride, Hk, G, block_size, max_blocks, n_limit, n_tiles, scale_log2, \
      v_scale, out, out_row_stride

template <bool F8, int D, bool H16, bool PAGED, int RG>
__global__ __launch_bounds__(256, D == 256 ? 1 : 2) void prefill_varlen_kernel(
    NKV_PREFILL_PARAMS) {
  prefill_body<F8, D, H16, PAGED, RG, false>(NKV_PREFILL_PASS, SplitArgs{});
}

template <bool F8, int D, bool H16, bool PAGED, int HP>
__global__ __launch_bounds__(256, D == 256 ? 1 : 2) void prefill_split_kernel(
    NKV_PREFILL_PARAMS, const SplitArgs sa) {
  prefill_body<F8, D, H16, PAGED, prefill_row_groups(D, F8), true, HP>(NKV_PREFILL_PASS, sa);
}

// Merges the parts of the units that ranges cut: descriptor x (of the workgroup that holds a
// unit's first part; part p > 0 is in the first slot of the workgroup p * Hk after it) and rows
// 32*y .. of its tile (block y * groups + x). The blocks after those merge the decode rows'
// partials, one (sequence, query head) a wave. A wave merges four rows at once, lane l output
// dims N*l .. N*l+N-1, eight parts' loads in flight. Where the rows leave waves idle (a decode
// row's tile has G) they take every n-th part each and merge once more through LDS.
constexpr int kMergeRows = 32;
constexpr int kMergeWaves = kMergeRows / 4;
template <int D, bool H16>
__global__ __launch_bounds__(64 * kMergeWaves) void prefill_merge_kernel(
    const SplitArgs sa, const int32_t* __restrict__ cu_q, const int32_t* __restrict__ cu_k,
    int32_t Hk, int32_t G, int32_t tile_rows, int32_t n_groups, float v_scale,
    bf16_t* __restrict__ out, int64_t out_row_stride) {
  constexpr int N = D / 64;
  constexpr int kRow = prefill_part_row(D);
  __shared__ float so[kMergeWaves][4][N][64];
  __shared__ float2 sml[kMergeWaves][4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int n_tile_blocks = (tile_rows + kMergeRows - 1) / kMergeRows * n_groups;
  if ((int)blockIdx.x >= n_tile_blocks) {
    const int Hq = Hk * G;
    const int id = ((int)blockIdx.x - n_tile_blocks) * kMergeWaves + wave;
    const int b = id / Hq;
    if (b < sa.n_seqs && cu_q[b + 1] - cu_q[b] == 1)  // uniform over the wave
      decode_combine<D, H16, 1>(OneRowSeqs{cu_q, cu_k, sa.n_seqs, sa.max_tokens}, b,
                                id - b * Hq, Hq, Hk, sa.ncg, sa.row_part, sa.row_desc, out,
                                out_row_stride);
    return;
  }
  const int x = blockIdx.x % n_groups;
  const i32x4_t d = sa.desc[x];
  const int n_parts = d[0];
  const int rows = d[2] * G;
  const int y0 = (int)blockIdx.x / n_groups * kMergeRows;
  if (n_parts < 2 || y0 >= rows) return;  // uniform over the workgroup
  // groups of four rows, rounded up to a power of two, and the waves that share one's parts
  const int left = rows - y0;
  const int groups = left > 16 ? 8 : left > 8 ? 4 : left > 4 ? 2 : 1;
  const int shares = kMergeWaves / groups;
  const int r0 = y0 + (wave % groups) * 4;
  const int share = wave / groups;
  const int64_t tile_f = (int64_t)tile_rows * kRow;
  const float* first = sa.part + ((int64_t)x * 2 + 1) * tile_f;
  const float* next = sa.part + (int64_t)x * 2 * tile_f;  // + p * 2 * Hk tiles
  float M[4], L[4], o[4][N];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    M[i] = -INFINITY;
    L[i] = 0.f;
#pragma unroll
    for (int e = 0; e < N; ++e) o[i][e] = 0.f;
  }
  // (m, l, o) of one more part into row i's
  auto add = [&](int i, float m, float l, const float (&v)[N]) {
    if (m == -INFINITY) return;  // none of its keys is visible to the row
    const float top = fmaxf(M[i], m);
    const float alpha = fast_exp2(M[i] - top);
    const float w = fast_exp2(m - top);
    M[i] = top;
    L[i] = fmaf(w, l, L[i] * alpha);
#pragma unroll
    for (int e = 0; e < N; ++e) o[i][e] = fmaf(w, v[e], o[i][e] * alpha);
  };
  if (r0 < rows) {
    for (int p0 = share; p0 < n_parts; p0 += 8 * shares) {
      float2 ml[8][4];
      float v[8][4][N];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int p = p0 + u * shares;
        if (p >= n_parts) break;  // uniform
        const float* t = p == 0 ? first : next + (int64_t)p * 2 * Hk * tile_f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float* row = t + (int64_t)min(r0 + i, rows - 1) * kRow;
          ml[u][i] = *reinterpret_cast<const float2*>(row + D);
          load_dims<N>(row + N * lane, v[u][i]);
        }
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
        if (p0 + u * shares < n_parts) {  // uniform
#pragma unroll
          for (int i = 0; i < 4; ++i) add(i, ml[u][i].x, ml[u][i].y, v[u][i]);
        }
    }
  }
  if (shares > 1) {  // uniform
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
      for (int e = 0; e < N; ++e) so[wave][i][e][lane] = o[i][e];
      if (lane == 0) sml[wave][i] = float2{M[i], L[i]};
    }
    __syncthreads();
    if (share > 0) return;
    for (int w = wave + groups; w < kMergeWaves; w += groups) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v[N];
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = so[w][i][e][lane];
        add(i, sml[w][i].x, sml[w][i].y, v);
      }
    }
  }
  const int kvh = d[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = r0 + i;
    if (r >= rows) break;
    bf16_t* op = out + (int64_t)(d[1] + r / G) * out_row_stride +
                 (int64_t)(kvh * G + r % G) * D + N * lane;
    store_dims<N, H16>(op, o[i], L[i] > 0.f ? v_scale / L[i] : 0.f);
  }
}

}  // namespace nkv

namespace nkv {
// Ranges per KV head of a split launch: the workgroups that are resident at once.
static int prefill_ranges(int32_t n_kv_heads, int32_t head_dim) {
  return std::max(1, device_cus() * (head_dim == 256 ? 1 : 2) / n_kv_heads);
}
// The split launch's workspace: a descriptor and two tiles of partial rows per workgroup; for
// the decode rows a descriptor per (sequence, KV head, column group) and a partial row per
// query head for every wave of a head group and every sequence.
struct SplitSizes {
  size_t groups, desc, part, row_desc, row_part;
  size_t bytes() const { return desc + part + row_desc + row_part; }
};
static SplitSizes prefill_split_sizes(int32_t n_seqs, int32_t n_q_heads, int32_t n_kv_heads,
                                      int32_t head_dim, bool f8) {
  SplitSizes z;
  z.groups = (size_t)prefill_ranges(n_kv_heads, head_dim) * n_kv_heads;
  z.desc = z.groups * sizeof(i32x4_t);
  const size_t row = prefill_part_row(head_dim) * sizeof(float);
  z.part = z.groups * 2 * prefill_tile_rows(head_dim, f8) * row;
  z.row_desc = (size_t)n_seqs * n_kv_heads * decode_ncg(n_q_heads / n_kv_heads) *
               sizeof(i32x4v_t);
  // waves of a head group x Hq <= 4 * groups x its columns (at most 16)
  z.row_part = (4 * z.groups * std::min(kMaxCols, n_q_heads) + (size_t)n_seqs * n_q_heads) * row;
  return z;
}
// KV heads a wave of the decode rows reads at once: up to a 512-byte piece of every row, as the
// decode kernel's plan takes them for batches that fill the chip (a step that has prompts too
// is long enough for it).
template <bool F8>
static int prefill_row_heads(int32_t n_kv_heads, int32_t G, int32_t head_dim) {
  const int most = head_dim == 256 ? (F8 ? 2 : 1) : (F8 && head_dim == 128 ? 4 : 2);
  for (int hp = most; hp > 1; hp /= 2)
    if (n_kv_heads % hp == 0 && hp * G <= kMaxCols) return hp;
  return 1;
}

// Tiles of qt queries that a batch can have at most (total_q < 0: its rows are not known).
static int64_t split_most_tiles(int64_t n_seqs, int64_t total_q, int64_t max_seqlen_q,
                                int64_t qt) {
  const int64_t most = n_seqs * ((max_seqlen_q + qt - 1) / qt);
  return total_q < 0 ? most : std::min(most, total_q / qt + n_seqs);
}

// Whether the split launch is the faster one, from what the host knows of the lengths and the
// batch's mix. In us, fitted to both sides' times of 200 random steps at head_dim 128 (1 - 104
// sequences, 1 - 3000 new tokens, contexts of up to 16k, every KV type), what other forms change
// and a decode row's cost to 663 of head_dim 64 - 256 and 1 - 128 query heads a KV head:
//  * plain, the workgroup of the longest sequence's last tile walks its keys alone, 1.0 a 64-key
//    step with the small tiles of a few workgroups; else every step of a tile costs its share
//    of the chip, 1.5, and of a decode row 2.5;
//  * split, the tiles' steps cost the same (2.1 at head_dim 256), the rows' (their bytes) 0.25, or
//    0.6 for each of several column groups (1 at head_dim 256), and the launch, the parts' writing
//    and the merge 35.
// The keys of a batch are taken as half of the longest sequence's. Of the 663 the rule splits 270,
// 3 of them over 10% slower than the plain launch (17% at most) and others up to 8x faster, and
// loses 3.2% against always knowing the faster. 512 tokens on 12288 (Hq 32, Hk 8): 172 us plain
// (344 with 192-row tiles), 126 split; 48 decode rows with two 512-token chunks: 202 and 118.
static bool prefill_split_wins(int32_t n_seqs, int64_t total_q, int32_t max_seqlen_q,
                               int32_t max_seqlen_k, int32_t n_q_heads, int32_t n_kv_heads,
                               int32_t head_dim, bool f8) {
  const int g = n_q_heads / n_kv_heads;
  const int64_t qt = prefill_tile_rows(head_dim, f8) / g;
  const int64_t tiles_max = (max_seqlen_q + qt - 1) / qt;
  // every range counts the tiles of the sequences before it: not for long prompts (whose
  // tiles fill the chip anyway)
  if (tiles_max > 96 || max_seqlen_k < max_seqlen_q ||
      !split_fits(n_seqs, split_most_tiles(n_seqs, total_q, max_seqlen_q, qt), max_seqlen_k))
    return false;
  const BatchMix m = batch_mix(n_seqs, total_q, max_seqlen_q);
  const int64_t tiles = std::min(m.prompts * tiles_max, m.prompt_rows / qt + m.prompts);
  const int64_t rows = m.rows;
  const double steps = (max_seqlen_k + kStep - 1) / kStep;
  const double per_range = 1.0 / prefill_ranges(n_kv_heads, head_dim);
  const double seen = 1.0 - 0.5 * max_seqlen_q / max_seqlen_k;  // causal: of a prompt's own keys
  const double tile_steps = tiles * steps * seen * per_range * (n_seqs == 1 ? 1.0 : 0.5);
  const double row_steps = rows * steps * 0.5 * per_range;
  const double dim = head_dim / 128.0;
  const int ncg = decode_ncg(g);
  const double tile_cost = head_dim == 256 ? 2.1 : 1.5;
  const double row_cost = ncg == 1 ? 0.25 : (head_dim == 256 ? 1.0 : 0.6) * ncg;
  return dim * std::max(steps, 1.5 * tile_steps + 2.5 * row_steps) >
         35.0 + dim * (tile_cost * tile_steps + row_cost * row_steps);
}

// `split`: a split launch over `workspace` where the lengths that a table row (or the K/V rows)
// can have leave its positions in 32 bits; a plain one otherwise.
template <bool F8, bool H16 = false>
static int prefill_launch(const void* q, int64_t q_row_stride, const void* k_cache,
                          const void* v_cache, int64_t k_row_stride, int64_t v_row_stride,
                          const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                          const int32_t* block_tables, int64_t bt_row_stride,
                          int32_t max_blocks_per_seq, int32_t n_seqs, int32_t max_seqlen_q,
                          int32_t n_q_heads, int32_t n_kv_heads, int32_t head_dim,
                          int32_t block_size, int64_t n_rows, float scale, float k_scale,
                          float v_scale, void* out, int64_t out_row_stride, void* stream,
                          int64_t total_q = -1, bool split = false, void* workspace = nullptr,
                          size_t workspace_bytes = 0) {
  constexpr int kEl = F8 ? 1 : 2;
  const char* what = F8 ? "prefill_varlen_fp8" : H16 ? "prefill_varlen_f16" : "prefill_varlen";
  NKV_REQUIRE(n_seqs >= 0 && max_seqlen_q >= 0 && n_q_heads > 0 && n_kv_heads > 0, NKV_EINVAL,
              "%s: bad sizes", what);
  if (n_seqs == 0 || max_seqlen_q == 0) return NKV_OK;
  NKV_REQUIRE(prefill_dim_ok(head_dim), NKV_EUNSUPPORTED,
              "%s: head_dim must be 64, 128 or 256 (got %d)", what, head_dim);
  NKV_REQUIRE(n_q_heads % n_kv_heads == 0, NKV_EINVAL, "%s: Hq %% Hk != 0", what);
  const int g = n_q_heads / n_kv_heads;
  // a tile holds at least one query for all g heads of its KV head
  NKV_REQUIRE(g <= prefill_max_group(head_dim), NKV_EUNSUPPORTED, "%s: GQA group %d above %d",
              what, g, prefill_max_group(head_dim));
  NKV_REQUIRE(q && k_cache && v_cache && cu_seqlens_q && cu_seqlens_k && out, NKV_EINVAL,
              "%s: null pointer", what);
  NKV_REQUIRE(aligned16(q) && aligned16(k_cache) && aligned16(v_cache) && aligned16(out),
              NKV_EINVAL, "%s: q/k/v/out must be 16-byte aligned", what);
  NKV_REQUIRE(q_row_stride >= (int64_t)n_q_heads * head_dim && q_row_stride % 8 == 0 &&
                  out_row_stride >= (int64_t)n_q_heads * head_dim && out_row_stride % 8 == 0 &&
                  k_row_stride >= (int64_t)n_kv_heads * head_dim &&
                  k_row_stride % (16 / kEl) == 0 &&
                  v_row_stride >= (int64_t)n_kv_heads * head_dim &&
                  v_row_stride % (16 / kEl) == 0,
              NKV_EINVAL, "%s: row strides must cover the heads, in 16-byte multiples", what);
  NKV_REQUIRE(n_rows > 0, NKV_EINVAL, "%s: empty K/V", what);
  NKV_REQUIRE(k_row_stride * kEl * kStep < (1ll << 31) && v_row_stride * kEl * kStep < (1ll << 31),
              NKV_EUNSUPPORTED, "%s: K/V row stride too large", what);
  NKV_REQUIRE(!block_tables || k_row_stride == v_row_stride, NKV_EINVAL,
              "%s: paged K and V caches share one row stride", what);
  NKV_REQUIRE(!F8 || block_tables, NKV_EINVAL, "%s: fp8 K/V are read from a paged pool", what);
  NKV_REQUIRE(k_scale > 0.f && v_scale > 0.f, NKV_EINVAL, "%s: scales must be > 0", what);
  int max_blocks = 0;
  if (block_tables) {
    NKV_REQUIRE(block_size > 0 && block_size % 16 == 0, NKV_EUNSUPPORTED,
                "%s: block_size must be a positive multiple of 16", what);
    NKV_REQUIRE(max_blocks_per_seq > 0 && bt_row_stride >= max_blocks_per_seq,
                NKV_EINVAL, "%s: paged mode needs block_size, max_blocks_per_seq "
                "and bt_row_stride >= max_blocks_per_seq", what);
    max_blocks = max_blocks_per_seq;
  }
  // paged: valid block ids are [0, n_rows / block_size); contiguous: valid rows
  const int32_t n_limit = (int32_t)std::min<int64_t>(block_tables ? n_rows / block_size : n_rows,
                                                     INT32_MAX);
  if (split)
    split = split_fits(n_seqs,
                       split_most_tiles(n_seqs, total_q, max_seqlen_q,
                                        prefill_tile_rows(head_dim, F8) / g),
                       block_tables ? (int64_t)max_blocks * block_size : n_rows);
  const int groups = split ? prefill_row_groups(head_dim, F8)
                           : plain_groups(n_seqs, total_q, max_seqlen_q, n_kv_heads, g,
                                          prefill_row_groups(head_dim, F8), device_cus());
  const int tile_rows = 64 * groups;
  const int qt = tile_rows / g;
  const int64_t tiles = plain_tiles(n_seqs, max_seqlen_q, qt);
  const float sl2 = scale * k_scale * kLog2e;
  int64_t grid = n_seqs * tiles * n_kv_heads;
  const int32_t n_tiles = (int32_t)tiles;
  int64_t merge_grid = 0;
  int row_heads = 0;
  SplitArgs sa = {};
  if (split) {
    const SplitSizes z = prefill_split_sizes(n_seqs, n_q_heads, n_kv_heads, head_dim, F8);
    const size_t need = z.bytes();
    NKV_REQUIRE(workspace && aligned16(workspace) && workspace_bytes >= need, NKV_EWORKSPACE,
                "%s: the split launch needs a 16-byte aligned workspace of %zu bytes (got %zu)",
                what, need, workspace_bytes);
    grid = (int64_t)z.groups;
    sa.n_seqs = n_seqs;
    sa.min_range = kMinRange;
    char* ws = static_cast<char*>(workspace);
    sa.desc = reinterpret_cast<i32x4_t*>(ws);
    sa.part = reinterpret_cast<float*>(ws + z.desc);
    sa.row_desc = reinterpret_cast<i32x4v_t*>(ws + z.desc + z.part);
    sa.row_part = reinterpret_cast<float*>(ws + z.desc + z.part + z.row_desc);
    sa.ncg = decode_ncg(g);
    sa.min_chunks = block_tables ? decode_min_chunks(decode_max_chunks(max_blocks, block_size),
                                                     kMinChunks)
                                 : 0;
    // dense cache rows, positions of the decode rows' chunks in 32 bits, and workgroups for each
    // kind of work (otherwise decode rows are tiles)
    if (block_tables && k_row_stride == (int64_t)n_kv_heads * head_dim &&
        (int64_t)max_blocks * block_size < (1ll << 30) &&
        (int64_t)block_size * k_row_stride * kEl < (1ll << 31)) {
      sa.max_tokens = max_blocks * block_size;
      sa.chunk_cost = row_cost(head_dim, F8, sa.ncg);
      row_heads = prefill_row_heads<F8>(n_kv_heads, g, head_dim);
      if (prefill_ranges(n_kv_heads, head_dim) <= row_ranges_least(sa.ncg, row_heads))
        row_heads = 0;
    }
    merge_grid = grid * ((tile_rows + kMergeRows - 1) / kMergeRows) +
                 (row_heads ? ((int64_t)n_seqs * n_q_heads + kMergeWaves - 1) / kMergeWaves : 0);
    NKV_REQUIRE(merge_grid < (1ll << 31), NKV_EUNSUPPORTED, "%s: grid too large", what);
  }
  NKV_REQUIRE(grid < (1ll << 31), NKV_EUNSUPPORTED, "%s: grid too large", what);
#define NKV_PREFILL_ARGS                                                                       \
  (const bf16_t*)q, q_row_stride, k_cache, v_cache, k_row_stride, v_row_stride, cu_seqlens_q,  \
      cu_seqlens_k, block_tables, bt_row_stride, n_kv_heads, g, block_size, max_blocks,        \
      n_limit, n_tiles, sl2, v_scale, (bf16_t*)out, out_row_stride
#define NKV_PREFILL_PLAIN(D, P, RG)                                                            \
  hipLaunchKernelGGL((prefill_varlen_kernel<F8, D, H16, P, RG>), dim3((unsigned)grid),         \
                     dim3(256), 0, as_stream(stream), NKV_PREFILL_ARGS)
#define NKV_PREFILL_SPLIT(D, P, HP)                                                            \
  hipLaunchKernelGGL((prefill_split_kernel<F8, D, H16, P, HP>), dim3((unsigned)grid), dim3(256), \
                     0, as_stream(stream), NKV_PREFILL_ARGS, sa)
#define NKV_PREFILL_LAUNCH_P(D, P)                                                             \
  do {                                                                                         \
    if (!split) {                                                                              \
      if (groups == 1) NKV_PREFILL_PLAIN(D, P, 1);                                             \
      else if (groups == 2) NKV_PREFILL_PLAIN(D, P, std::min(2, prefill_row_groups(D, F8)));   \
      else NKV_PREFILL_PLAIN(D, P, prefill_row_groups(D, F8));                                 \
      break;                                                                                   \
    }                                                                                          \
    if constexpr (P) {                                                                         \
      if (row_heads == 0) NKV_PREFILL_SPLIT(D, P, 0);                                          \
      else if (row_heads == 1) NKV_PREFILL_SPLIT(D, P, 1);                                     \
      else if constexpr (D < 256 || F8) {                                                      \
        if constexpr (D == 128 && F8) {                                                        \
          if (row_heads == 4) NKV_PREFILL_SPLIT(D, P, 4);                                      \
          else NKV_PREFILL_SPLIT(D, P, 2);                                                     \
        } else {                                                                               \
          NKV_PREFILL_SPLIT(D, P, 2);                                                          \
        }                                                                                      \
      }                                                                                        \
    } else {                                                                                   \
      NKV_PREFILL_SPLIT(D, P, 0);                                                              \
    }                                                                                          \
    hipLaunchKernelGGL((prefill_merge_kernel<D, H16>), dim3((unsigned)merge_grid),             \
                       dim3(64 * kMergeWaves), 0, as_stream(stream), sa, cu_seqlens_q,         \
                       cu_seqlens_k, n_kv_heads, g, tile_rows, (int32_t)grid, v_scale,         \
                       (bf16_t*)out, out_row_stride);                                          \
  } while (0)
#define NKV_PREFILL_LAUNCH(D)                                                                  \
  do {                                                                                         \
    if (block_tables) NKV_PREFILL_LAUNCH_P(D, true);                                           \
    else if constexpr (!F8) NKV_PREFILL_LAUNCH_P(D, false);                                    \
  } while (0)
  if (head_dim == 64) NKV_PREFILL_LAUNCH(64);
  else if (head_dim == 128) NKV_PREFILL_LAUNCH(128);
  else NKV_PREFILL_LAUNCH(256);
#undef NKV_PREFILL_LAUNCH
#undef NKV_PREFILL_LAUNCH_P
#undef NKV_PREFILL_PLAIN
#undef NKV_PREFILL_SPLIT
#undef NKV_PREFILL_ARGS
  return check_launch(F8 ? "nkv_prefill_varlen_fp8"
                         : H16 ? "nkv_prefill_varlen_f16" : "nkv_prefill_varlen");
}
}  // namespace nkv

namespace nkv {
int prefill_paged(int32_t kv_type, const void* q, int64_t q_row_stride, const void* k_cache,
                  const void* v_cache, int64_t row_stride, const int32_t* cu_seqlens_q,
                  const int32_t* cu_seqlens_k, const int32_t* block_tables,
                  int64_t bt_row_stride, int32_t max_blocks_per_seq, int32_t n_seqs,
                  int64_t total_q, int32_t max_seqlen_q, int32_t n_q_heads, int32_t n_kv_heads,
                  int32_t head_dim, int32_t block_size, int64_t n_rows, float scale,
                  float k_scale, float v_scale, void* out, int64_t out_row_stride,
                  void* workspace, size_t workspace_bytes, void* stream) {
#define NKV_PREFILL_ANY(...)                                                                   \
  prefill_launch<__VA_ARGS__>(q, q_row_stride, k_cache, v_cache, row_stride, row_stride,       \
                              cu_seqlens_q, cu_seqlens_k, block_tables, bt_row_stride,         \
                              max_blocks_per_seq, n_seqs, max_seqlen_q, n_q_heads, n_kv_heads, \
                              head_dim, block_size, n_rows, scale, k_scale, v_scale, out,      \
                              out_row_stride, stream, total_q, workspace_bytes > 0, workspace, \
                              workspace_bytes)
  if (kv_type == NKV_KV_FP8) return NKV_PREFILL_ANY(true);
  if (kv_type == NKV_KV_F16) return NKV_PREFILL_ANY(false, true);
  return NKV_PREFILL_ANY(false);
#undef NKV_PREFILL_ANY
}
}  // namespace nkv

extern "C" int nkv_prefill_varlen(const void* q, int64_t q_row_stride, const void* k_cache,
                                  const void* v_cache, int64_t k_row_stride,
                                  int64_t v_row_stride, const int32_t* cu_seqlens_q,
                                  const int32_t* cu_seqlens_k, const int32_t* block_tables,
                                  int64_t bt_row_stride, int32_t max_blocks_per_seq,
                                  int32_t n_seqs, int32_t max_seqlen_q, int32_t n_q_heads,
                                  int32_t n_kv_heads, int32_t head_dim, int32_t block_size,
                                  int64_t n_rows, float scale, void* out, int64_t out_row_stride,
                                  void* stream) {
  nkv::clear_error();
  return nkv::prefill_launch<false>(q, q_row_stride, k_cache, v_cache, k_row_stride,
                                    v_row_stride, cu_seqlens_q, cu_seqlens_k, block_tables,
                                    bt_row_stride, max_blocks_per_seq, n_seqs, max_seqlen_q,
                                    n_q_heads, n_kv_heads, head_dim, block_size, n_rows, scale,
                                    1.f, 1.f, out, out_row_stride, stream);
}

extern "C" int nkv_prefill_varlen_f16(const void* q, int64_t q_row_stride, const void* k_cache,
                                      const void* v_cache, int64_t k_row_stride,
                                      int64_t v_row_stride, const int32_t* cu_seqlens_q,
                                      const int32_t* cu_seqlens_k, const int32_t* block_tables,
                                      int64_t bt_row_stride, int32_t max_blocks_per_seq,
                                      int32_t n_seqs, int32_t max_seqlen_q, int32_t n_q_heads,
                                      int32_t n_kv_heads, int32_t head_dim, int32_t block_size,
                                      int64_t n_rows, float scale, void* out,
                                      int64_t out_row_stride, void* stream) {
  nkv::clear_error();
  return nkv::prefill_launch<false, true>(q, q_row_stride, k_cache, v_cache, k_row_stride,
                                          v_row_stride, cu_seqlens_q, cu_seqlens_k, block_tables,
                                          bt_row_stride, max_blocks_per_seq, n_seqs,
                                          max_seqlen_q, n_q_heads, n_kv_heads, head_dim,
                                          block_size, n_rows, scale, 1.f, 1.f, out,
                                          out_row_stride, stream);
}

extern "C" int nkv_prefill_varlen_fp8(const void* q, int64_t q_row_stride, const void* k_cache,
                                      const void* v_cache, const int32_t* cu_seqlens_q,
                                      const int32_t* cu_seqlens_k, const int32_t* block_tables,
                                      int64_t bt_row_stride, int32_t max_blocks_per_seq,
                                      int32_t n_seqs, int32_t max_seqlen_q, int32_t n_q_heads,
                                      int32_t n_kv_heads, int32_t head_dim, int32_t block_size,
                                      int64_t n_blocks, float scale, float k_scale,
                                      float v_scale, void* out, int64_t out_row_stride,
                                      void* stream) {
  nkv::clear_error();
  const int64_t row = (int64_t)n_kv_heads * head_dim;  // codes (bytes) per cache row
  return nkv::prefill_launch<true>(q, q_row_stride, k_cache, v_cache, row, row, cu_seqlens_q,
                                   cu_seqlens_k, block_tables, bt_row_stride, max_blocks_per_seq,
                                   n_seqs, max_seqlen_q, n_q_heads, n_kv_heads, head_dim,
                                   block_size, n_blocks * block_size, scale, k_scale, v_scale,
                                   out, out_row_stride, stream);
}

extern "C" size_t nkv_prefill_split_workspace_bytes(int32_t n_seqs, int32_t n_q_heads,
                                                    int32_t n_kv_heads, int32_t head_dim,
                                                    int32_t kv_type) {
  using namespace nkv;
  if (n_seqs <= 0 || n_q_heads <= 0 || n_kv_heads <= 0 || n_q_heads % n_kv_heads != 0 ||
      !prefill_dim_ok(head_dim))
    return 0;
  return prefill_split_sizes(n_seqs, n_q_heads, n_kv_heads, head_dim, kv_type == NKV_KV_FP8)
      .bytes();
}

extern "C" size_t nkv_prefill_split_plan(int32_t n_seqs, int64_t total_q, int32_t max_seqlen_q,
                                         int32_t max_seqlen_k, int32_t n_q_heads,
                                         int32_t n_kv_heads, int32_t head_dim,
                                         int32_t kv_type) {
  using namespace nkv;
  if (n_seqs <= 0 || total_q <= 0 || max_seqlen_q <= 0 || n_q_heads <= 0 || n_kv_heads <= 0 ||
      n_q_heads % n_kv_heads != 0 || !prefill_dim_ok(head_dim) ||
      n_q_heads / n_kv_heads > prefill_max_group(head_dim))
    return 0;
  const bool f8 = kv_type == NKV_KV_FP8;
  return prefill_split_wins(n_seqs, total_q, max_seqlen_q, max_seqlen_k, n_q_heads, n_kv_heads,
                            head_dim, f8)
             ? prefill_split_sizes(n_seqs, n_q_heads, n_kv_heads, head_dim, f8).bytes()
             : 0;
}

extern "C" int nkv_prefill_varlen_split(int32_t kv_type, const void* q, int64_t q_row_stride,
                                        const void* k_cache, const void* v_cache,
                                        int64_t k_row_stride, int64_t v_row_stride,
                                        const int32_t* cu_seqlens_q,
                                        const int32_t* cu_seqlens_k,
                                        const int32_t* block_tables, int64_t bt_row_stride,
                                        int32_t max_blocks_per_seq, int32_t n_seqs,
                                        int32_t max_seqlen_q, int32_t n_q_heads,
                                        int32_t n_kv_heads, int32_t head_dim,
                                        int32_t block_size, int64_t n_rows, float scale,
                                        float k_scale, float v_scale, void* out,
                                        int64_t out_row_stride, void* workspace,
                                        size_t workspace_bytes, void* stream) {
  using namespace nkv;
  clear_error();
  if (kv_type != NKV_KV_FP8) k_scale = v_scale = 1.f;
#define NKV_PREFILL_SPLIT(...)                                                                 \
  prefill_launch<__VA_ARGS__>(q, q_row_stride, k_cache, v_cache, k_row_stride, v_row_stride,   \
                              cu_seqlens_q, cu_seqlens_k, block_tables, bt_row_stride,         \
                              max_blocks_per_seq, n_seqs, max_seqlen_q, n_q_heads, n_kv_heads, \
                              head_dim, block_size, n_rows, scale, k_scale, v_scale, out,      \
                              out_row_stride, stream, -1, true, workspace, workspace_bytes)
  switch (kv_type) {
    case NKV_KV_BF16: return NKV_PREFILL_SPLIT(false);
    case NKV_KV_F16: return NKV_PREFILL_SPLIT(false, true);
    case NKV_KV_FP8: return NKV_PREFILL_SPLIT(true);
  }
#undef NKV_PREFILL_SPLIT
  set_error("prefill_varlen_split: kv_type %d is none of NKV_KV_*", kv_type);
  return NKV_EINVAL;
}
