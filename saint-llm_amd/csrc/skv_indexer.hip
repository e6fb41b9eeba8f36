// Lightning-indexer block scores over the paged compressed indexer keys.
//
// Reference: lightning_indexer_scores_reference (kernels/attention.py:33-50)
// and the cached decode path CSA._indexer_topk_cached (csa.py:405-409):
//   head_scores[b,t,h,s] = ReLU(q[b,t,h,:] . k[b,s,:])
//   scores[b,t,s]        = sum_h w[b,t,h] * head_scores[b,t,h,s]
// The head axis is reduced on the fly; no (B, T, H, S) tensor is formed.  The
// scores are unmasked (the top-k applies the causal block mask); the cached
// path takes no visual bias (csa.py:396-399) and neither does this kernel.
//
// The tile (MFMA mapping, operand staging) is in skv_indexer_tile.h.
#include <algorithm>

#include "skv_common.h"
#include "skv_indexer_tile.h"

namespace skv {

struct IndexerArgs {
  const uint8_t* q;  // [rows, H, c] bf16, rows = batch * t_per_seq
  const float* w;    // [rows, H]
  const uint8_t* pool;  // [n_pages, block_size, c] bf16
  const int32_t* block_table;  // nullptr: a chunk's keys, sequence b's in page b
  const int32_t* n_entries;    // nullptr with it: max_entries
  float* scores;  // [rows, score_stride]
  int64_t score_stride;
  int32_t bt_stride;
  int32_t n_heads, c, block_size, n_pages, t_per_seq, max_entries;
  int32_t offset, m;  // a chunk's token t sees the entries below (offset + t) / m
};

// Entries that token t of sequence b is scored against.
template <bool kChunk>
__device__ __forceinline__ int indexer_entries(const IndexerArgs& a, int b, int t) {
  return min(kChunk ? (a.offset + t) / a.m : a.n_entries[b], a.max_entries);
}

// One workgroup per (tile of kIdxTile entries, query row).
template <bool kChunk>
__global__ __launch_bounds__(kIdxThreads, 2) void k_indexer_scores(IndexerArgs a) {
  __shared__ IndexerSmem sm;
  const int row = blockIdx.y;  // query row
  const int b = static_cast<int>(udiv24(row, a.t_per_seq));
  const IndexerRow r{a.q + static_cast<int64_t>(row) * a.n_heads * a.c * 2,
                     a.w + static_cast<int64_t>(row) * a.n_heads,
                     a.pool,
                     kChunk ? nullptr : a.block_table + static_cast<int64_t>(b) * a.bt_stride,
                     a.bt_stride,
                     a.block_size,
                     a.n_pages,
                     a.n_heads,
                     a.c,
                     b};
  float* out = a.scores + static_cast<int64_t>(row) * a.score_stride;
  indexer_tile<!kChunk>(
      sm, r, static_cast<int>(blockIdx.x),
      [&] { return indexer_entries<kChunk>(a, b, row - b * a.t_per_seq); },  // the grid covers max_entries
      [&](int e, float v) { out[e] = v; });
}

// ---------------------------------------------------------------------------
// Several query tokens per sequence (a prompt chunk).  The product is a GEMM of
// the tokens' heads against the sequence's keys, bound by the matrix cores once
// the keys are shared: a workgroup takes kIrTokens tokens and a run of entries,
// kIrTile at a time through LDS, and each of its 8 waves keeps one token's query
// (64 heads x 128 channels) as A operands in registers, so an LDS read of a key
// operand feeds 4 products.  (k_indexer_scores reads the query from LDS for
// every 16 entries, one read per product: LDS-bound at 0.43 PFLOP/s.)  Products
// and head sums run in k_indexer_scores's order: the scores are the same bits.
// 2,048 tokens x 4,096 entries of 64 heads x 128: 156 us, 0.88 PFLOP/s (323 us
// before; a large bf16 product of the library runs at 1.27).  Two tokens per
// wave would halve the key reads but spill.
// ---------------------------------------------------------------------------
constexpr int kIrMinTokens = 6;  // fewer query tokens per sequence: k_indexer_scores, as for few tiles (see the launch)
constexpr int kIrThreads = 512;
constexpr int kIrTokens = kIrThreads / kWave;  // query tokens per workgroup, one per wave
constexpr int kIrTile = 128;                   // entries per LDS tile

struct IndexerRowsArgs {
  IndexerArgs a;
  int32_t groups;  // token groups per sequence
  int32_t run;     // entries per workgroup, a multiple of kIrTile
};

// What heads and channels past the query's, and entries without a page, read:
// no select follows a load.
__device__ __align__(16) uint8_t g_idx_zero[16];

// HB: 16-head blocks, KS: 32-channel steps (heads and channels past the
// query's are zero in both operands).
// kChunk: the entries up to those that the workgroup's last token sees.
template <int HB, int KS, bool kChunk>
__global__ __launch_bounds__(kIrThreads, 2) void k_indexer_scores_rows(IndexerRowsArgs ra) {
  const IndexerArgs& a = ra.a;
  constexpr int kRow = 32 * KS + 8;  // LDS row of a key (16 bytes of pad: distinct banks)
  constexpr int kChunks = 4 * KS;    // 16-byte pieces of a key
  constexpr int kPer = kIrTile * kChunks / kIrThreads;
  __shared__ alignas(16) uint16_t keys[2][kIrTile][kRow];
  __shared__ int64_t src_row[3][kIrTile];  // byte offset of each entry's key in the pool, -1 unmapped or past the run;
                                           // tile i of the run in row i % 3
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid) / kWave;
  const int col = lane & 15, grp = lane >> 4;
  const int b = blockIdx.y / ra.groups;
  const int t0 = (blockIdx.y - b * ra.groups) * kIrTokens;
  const int t = t0 + wave;  // this wave's token
  const int n_ent = indexer_entries<kChunk>(a, b, min(t0 + kIrTokens, a.t_per_seq) - 1);
  const int e_lo = blockIdx.x * ra.run, e_hi = min(n_ent, e_lo + ra.run);
  if (e_lo >= e_hi) return;  // uniform
  const int32_t* bt_row = a.block_table + static_cast<int64_t>(b) * a.bt_stride;
  // entry e's page (loaded a tile ahead of its key) and its key's offset
  const auto page_of = [&](int e) { return kChunk ? b : bt_row[min(static_cast<int>(udiv24(e, a.block_size)), a.bt_stride - 1)]; };
  const auto row_of = [&](int e, int32_t page) -> int64_t {
    const int pi = static_cast<int>(udiv24(e, a.block_size));
    const bool ok = e < e_hi && pi < a.bt_stride && page >= 0 && page < a.n_pages;
    return ok ? (static_cast<int64_t>(page) * a.block_size + (e - pi * a.block_size)) * a.c * 2 : -1;
  };
  if (tid < 2 * kIrTile) src_row[tid / kIrTile][tid % kIrTile] = row_of(e_lo + tid, page_of(e_lo + tid));
  // the token's query as A operands, its head weights by D row
  bf16x8 qa[KS][HB];
  float wv[HB][4];
  const int64_t row = static_cast<int64_t>(b) * a.t_per_seq + min(t, a.t_per_seq - 1);
  const uint8_t* q = a.q + row * a.n_heads * a.c * 2;
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
    for (int hb = 0; hb < HB; ++hb) {
      const int h = hb * 16 + col, ch = ks * 32 + grp * 8;
      const uint8_t* p = (h < a.n_heads && ch < a.c) ? q + (h * a.c + ch) * 2 : g_idx_zero;
      qa[ks][hb] = as_bf16x8(*reinterpret_cast<const u32x4*>(p));
    }
  }
#pragma unroll
  for (int hb = 0; hb < HB; ++hb) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int h = hb * 16 + grp * 4 + i;
      const float* p = h < a.n_heads ? a.w + row * a.n_heads + h : reinterpret_cast<const float*>(g_idx_zero);
      wv[hb][i] = *p;
    }
  }
  // key staging: thread i holds pieces i, i + 512, ... of a tile
  u32x4 kreg[kPer];
  const auto load_tile = [&](int slot) {
#pragma unroll
    for (int p = 0; p < kPer; ++p) {
      const int piece = tid + p * kIrThreads;
      const int64_t off = src_row[slot][piece / kChunks];
      const int ch = (piece % kChunks) * 8;
      const uint8_t* src = (off >= 0 && ch < a.c) ? a.pool + off + ch * 2 : g_idx_zero;
      kreg[p] = *reinterpret_cast<const u32x4*>(src);
    }
  };
  const auto store_tile = [&](int buf) {
#pragma unroll
    for (int p = 0; p < kPer; ++p) {
      const int piece = tid + p * kIrThreads;
      *reinterpret_cast<u32x4*>(&keys[buf][piece / kChunks][(piece % kChunks) * 8]) = kreg[p];
    }
  };
  lds_barrier();
  load_tile(0);
  store_tile(0);
  lds_barrier();
  float* const out = a.scores + row * a.score_stride;
  // ReLU as the median of x, 0 and infinity, one instruction where a maximum is
  // two (it quiets its operand first); the compiler must not see the constant
  float inf = __builtin_huge_valf();
  asm("" : "+v"(inf));
  int buf = 0, slot = 0;
  for (int e0 = e_lo; e0 < e_hi; e0 += kIrTile) {
    const bool more = e0 + kIrTile < e_hi;  // uniform
    const int next = slot == 2 ? 0 : slot + 1;
    int32_t page = 0;
    if (more) {  // in flight while this tile is multiplied: the next tile's keys, the pages of the one after
      load_tile(next);
      page = page_of(e0 + 2 * kIrTile + tid % kIrTile);
    }
    // 16-entry blocks in turn: the products of one beside the ReLU and head sum
    // of the one before and the LDS reads of the next.  The barriers keep that
    // order (the compiler would chain each accumulator's products, which then
    // wait for one another).
    constexpr int kBlocks = kIrTile / 16;
    bf16x8 kv[2][KS];
    f32x4 acc[2][HB];
    float v[kBlocks];
    const auto read_keys = [&](int j) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        kv[j & 1][ks] = as_bf16x8(*reinterpret_cast<const u32x4*>(&keys[buf][j * 16 + col][ks * 32 + grp * 8]));
      }
    };
    // terms [n0, n1) of block j's head sum: term 4hb + i is head 16hb + 4grp + i
    const auto head_sum = [&](int j, int n0, int n1) {
#pragma unroll
      for (int n = n0; n < n1; ++n) {
        const float term = __builtin_amdgcn_fmed3f(acc[j & 1][n / 4][n % 4], 0.f, inf);  // ReLU, 0 for NaN
        v[j] = fmaf(wv[n / 4][n % 4], term, n == 0 ? 0.f : v[j]);
      }
    };
    read_keys(0);
#pragma unroll
    for (int j = 0; j < kBlocks; ++j) {
      if (j + 1 < kBlocks) read_keys(j + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
        for (int hb = 0; hb < HB; ++hb) {
          const f32x4 from = ks == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[j & 1][hb];
          acc[j & 1][hb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa[ks][hb], kv[j & 1][ks], from, 0, 0, 0);
          if (j > 0) head_sum(j - 1, (ks * HB + hb) * 4 / KS, (ks * HB + hb + 1) * 4 / KS);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    head_sum(kBlocks - 1, 0, 4 * HB);
    // heads summed over the lane groups, four entry blocks at once: each
    // exchange halves the blocks a lane group still holds, so that group g ends
    // with block g and lane l with entry l of the 64
    const bool g0 = grp & 1, g1 = grp & 2;
#pragma unroll
    for (int r0 = 0; r0 < kIrTile; r0 += kWave) {
      const float* const w = v + r0 / 16;
      const float a0 = (g0 ? w[1] : w[0]) + __shfl_xor(g0 ? w[0] : w[1], 16);
      const float a2 = (g0 ? w[3] : w[2]) + __shfl_xor(g0 ? w[2] : w[3], 16);
      const float sum = (g1 ? a2 : a0) + __shfl_xor(g1 ? a0 : a2, 32);
      const int e = e0 + r0 + lane;
      const bool ok = src_row[slot][r0 + lane] >= 0;
      if (t < a.t_per_seq && e < e_hi) out[e] = ok ? sum : -__builtin_huge_valf();
    }
    if (more) {
      // the keys' and offsets' last readers passed the barrier of the tile before
      store_tile(buf ^ 1);
      if (tid < kIrTile) src_row[next == 2 ? 0 : next + 1][tid] = row_of(e0 + 2 * kIrTile + tid, page);
      lds_barrier();
    }
    slot = next;
    buf ^= 1;
  }
}

template <int HB, int KS, bool kChunk>
void launch_indexer_rows(const IndexerArgs& a, int64_t batch, hipStream_t s) {
  IndexerRowsArgs ra;
  ra.a = a;
  ra.groups = static_cast<int32_t>(ceil_div(a.t_per_seq, kIrTokens));
  // one workgroup per CU is resident: about four rounds of them, runs of at
  // least 2 tiles (each workgroup reads its queries once)
  const int64_t tiles = ceil_div(a.max_entries, kIrTile);
  const int64_t want = ceil_div(4 * static_cast<int64_t>(device_cus()), batch * ra.groups);
  const int64_t run = std::max<int64_t>(ceil_div(tiles, want), std::min<int64_t>(tiles, 2));
  ra.run = static_cast<int32_t>(run * kIrTile);
  const dim3 grid(static_cast<unsigned>(ceil_div(tiles, run)), static_cast<unsigned>(batch * ra.groups));
  hipLaunchKernelGGL((k_indexer_scores_rows<HB, KS, kChunk>), grid, dim3(kIrThreads), 0, s, ra);
}

template <bool kChunk>
void launch_indexer(const IndexerArgs& a, int64_t batch, hipStream_t s) {
  // The line: 16 x 16,384 entries and 64 heads take k_indexer_scores 42 us for 4
  // tokens and 10.5 us for each more, k_indexer_scores_rows 53 us for 4 to 8.  While
  // the tiles of k_indexer_scores are too few to fill the device, the long start of
  // the other's workgroups counts for more, the larger the query the longer (scores /
  // rows; 64 heads x 128: 1 tile a CU 8.4 / 12.4 us, 2 12.6 / 12.7, 3 18.4 / 14.1;
  // 64 x 64: 1 7.1 / 8.6, 2 10.2 / 8.8; 32 x 128: an eighth 6.7 / 7.9, three eighths
  // 8.0 / 8.0; smaller ones 6.5 / 4.2-6.3 from the first tile on).
  const int hb = a.n_heads <= 16 ? 1 : a.n_heads <= 32 ? 2 : 4, ks = a.c <= 32 ? 1 : a.c <= 64 ? 2 : 4;
  const int quarters = hb * ks == 16 ? 10 : hb == 4 && ks == 2 ? 6 : hb * ks == 8 ? 1 : 0;  // tiles per four CUs
  const int64_t tiles = batch * a.t_per_seq * ceil_div(a.max_entries, kIdxTile);
  if (a.t_per_seq >= kIrMinTokens && 4 * tiles >= quarters * static_cast<int64_t>(device_cus())) {
    switch (hb * 8 + ks) {
      case 9: launch_indexer_rows<1, 1, kChunk>(a, batch, s); break;
      case 10: launch_indexer_rows<1, 2, kChunk>(a, batch, s); break;
      case 12: launch_indexer_rows<1, 4, kChunk>(a, batch, s); break;
      case 17: launch_indexer_rows<2, 1, kChunk>(a, batch, s); break;
      case 18: launch_indexer_rows<2, 2, kChunk>(a, batch, s); break;
      case 20: launch_indexer_rows<2, 4, kChunk>(a, batch, s); break;
      case 33: launch_indexer_rows<4, 1, kChunk>(a, batch, s); break;
      case 34: launch_indexer_rows<4, 2, kChunk>(a, batch, s); break;
      default: launch_indexer_rows<4, 4, kChunk>(a, batch, s); break;
    }
    return;
  }
  const dim3 grid(static_cast<unsigned>(ceil_div(a.max_entries, kIdxTile)), static_cast<unsigned>(batch * a.t_per_seq));
  hipLaunchKernelGGL(k_indexer_scores<kChunk>, grid, dim3(kIdxThreads), 0, s, a);
}

int indexer_check_query(const char* what, int64_t n_heads, int64_t channels) {
  if (n_heads < 1 || n_heads > 16 * kIdxMaxHB) {
    return set_error(SKV_EINVAL, "%s: n_heads must be in [1, %d]; got %lld", what, 16 * kIdxMaxHB,
                     (long long)n_heads);
  }
  if (channels < 8 || channels > 32 * kIdxMaxKS || channels % 8) {
    return set_error(SKV_EINVAL, "%s: channels must be a multiple of 8 in [8, %d]; got %lld", what,
                     32 * kIdxMaxKS, (long long)channels);
  }
  return SKV_OK;
}

int launch_indexer_chunk(const IndexerChunk& x, hipStream_t s) {
  IndexerArgs a{};
  a.q = static_cast<const uint8_t*>(x.q);
  a.w = x.w;
  a.pool = static_cast<const uint8_t*>(x.keys);
  a.scores = x.scores;
  a.score_stride = x.n_blocks;
  a.bt_stride = 1;
  a.n_heads = static_cast<int32_t>(x.n_heads);
  a.c = static_cast<int32_t>(x.channels);
  a.block_size = static_cast<int32_t>(x.key_rows);
  a.n_pages = static_cast<int32_t>(x.batch);
  a.t_per_seq = static_cast<int32_t>(x.t_new);
  a.max_entries = static_cast<int32_t>(x.n_blocks);
  a.offset = static_cast<int32_t>(x.offset);
  a.m = static_cast<int32_t>(x.m);
  launch_indexer<true>(a, x.batch, s);
  return check_launch("skv_indexer_topk");
}

}  // namespace skv

using namespace skv;

extern "C" int skv_indexer_scores(const void* q, const float* w, const void* idx_pool, int64_t block_size,
                                  int64_t n_pages, const int32_t* block_table, int64_t bt_stride,
                                  const int32_t* n_entries, float* scores, int64_t score_stride,
                                  int64_t batch, int64_t t_per_seq, int64_t n_heads, int64_t channels,
                                  int64_t max_entries, void* stream) {
  const char* what = "skv_indexer_scores";
  if (batch < 0 || t_per_seq < 0 || max_entries < 0) return set_error(SKV_EINVAL, "%s: negative size", what);
  if (batch == 0 || t_per_seq == 0 || max_entries == 0) return SKV_OK;
  if (!q || !w || !idx_pool || !block_table || !n_entries || !scores) {
    return set_error(SKV_EINVAL, "%s: NULL pointer", what);
  }
  if (const int rc = indexer_check_query(what, n_heads, channels)) return rc;
  if (block_size <= 0 || n_pages <= 0 || n_pages > 0x7fffffff || bt_stride <= 0 || bt_stride >= (1 << 24)) {
    return set_error(SKV_EINVAL, "%s: bad page geometry", what);
  }
  if (max_entries > score_stride || max_entries >= (1 << 24) - kIdxTile) {
    return set_error(SKV_EINVAL, "%s: max_entries must be <= score_stride and < 2^24", what);
  }
  const int64_t rows = batch * t_per_seq;
  if (rows > 65535 || batch >= (1 << 24)) return set_error(SKV_EINVAL, "%s: at most 65535 query rows", what);
  IndexerArgs a;
  a.q = static_cast<const uint8_t*>(q);
  a.w = w;
  a.pool = static_cast<const uint8_t*>(idx_pool);
  a.block_table = block_table;
  a.n_entries = n_entries;
  a.scores = scores;
  a.score_stride = score_stride;
  a.bt_stride = static_cast<int32_t>(bt_stride);
  a.n_heads = static_cast<int32_t>(n_heads);
  a.c = static_cast<int32_t>(channels);
  a.block_size = static_cast<int32_t>(block_size);
  a.n_pages = static_cast<int32_t>(n_pages);
  a.t_per_seq = static_cast<int32_t>(t_per_seq);
  a.max_entries = static_cast<int32_t>(max_entries);
  launch_indexer<false>(a, batch, static_cast<hipStream_t>(stream));
  return check_launch(what);
}
