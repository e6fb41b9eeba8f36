// Token compression: softmax-weighted pooling of every m tokens into one
// compressed entry, written straight into the paged compressed cache (bf16, or
// FP8 e4m3fn with a 1x128 fp32 scale), plus staging of the incomplete block.
//
// Reference semantics:
//   TokenLevelCompressor.forward (csa.py:66-88):
//     z = z_b + bias_b ; w = softmax(z, dim=tokens) ; out = sum_tokens(w * c_b)
//   HCA/CSA append state machine (kv_cache.py:171-195, 291-315):
//     combined = cat(h_buffer[:, :cnt], h_new); n_complete = total // m;
//     blocks -> compressed[:, nb:nb+n_complete]; leftover -> h_buffer
//   FP8 quantize-on-write (quant/reference.py:75-110) on each 128-dim block.
// Here the buffered state of the incomplete block is the running online-softmax
// state of each channel (max, sum, weighted sum; fp32 [batch, 3, channels]),
// so a decode step costs O(channels) whatever m is, and a block emits the same
// bits whichever calls brought its m tokens.
#include <algorithm>
#include <type_traits>

#include "skv_pool_state.h"

namespace skv {

struct CompressArgs {
  uint8_t* pool;
  int64_t entry_bytes;
  int bs;
  int64_t n_pages;
  const int32_t* bt;
  int64_t bt_stride;
  float* state;  // [batch, 3, channels]: running max, sum of weights, weighted sum
  const uint8_t* c_new;
  const uint8_t* z_new;
  int64_t in_seq_stride;
  int64_t in_row_stride;
  int64_t in_len;
  const float* bias;
  const int32_t* lens;
  const int32_t* n_new;
  int n_uni;
  int m;
  int channels;
  int format;
  int fp8_main;  // main (quantized) channels in FP8 format
};

// Work split.  The pooling is independent per channel and serial over an entry's
// tokens, so a row of lanes takes 128 channels (one fp8 scale block) of one entry,
// kCh of them a lane, and the rows of a workgroup's 4 waves are shared out between
// entries and blocks of channels.
//   * kCh = 8 (16 lanes read 256 consecutive bytes of a token row) where a call
//     brings an entry at most 4 tokens, which are in flight at once.
//   * Of longer entries the chain of tokens sets the time, about 26 instructions a
//     token and channel: 0.1 us a token at one channel a lane (2 waves a row), which
//     is taken while the rows are too few to fill the SIMDs.  With 8 rows per CU and
//     more the loads count: 8 channels up to 15 tokens, then 2.
// HBM-bound where the device is full: c and z rows are read once.  bf16 rows of 576
// channels, against one wave per entry with a memory round trip a token: 4
// sequences of 8,192 tokens in entries of 4 tokens 31 us (2.7 TB/s; 145), of 32 28
// (121), of 128 33 (455; at 2 channels a lane 38); two of 300 tokens in entries of 4
// 7.5 (17.6), of 128 19 (515).  (An entry's tokens split over 16 rows of lanes took
// 9.4 us there and 24 above, but its sums hung on how the tokens came.)
constexpr int kCmThreads = 256;
constexpr int kCmBlock = 128;  // channels of a row of lanes
constexpr int kCmRows = 4;     // most rows of 1 or 2 channels a lane

// A lane's kCh channels of a row as they lie in memory (bf16 or fp32).
template <class Row, int kCh>
struct RawRow {
  static constexpr int kWords = (kCh * sizeof(Row) + 3) / 4;
  uint32_t w[kWords];
  __device__ __forceinline__ void load(const uint8_t* row, int grp) {
    const uint8_t* p = row + grp * static_cast<int>(kCh * sizeof(Row));
    if constexpr (kCh == 8) {
#pragma unroll
      for (int i = 0; i < kWords; i += 4) {
        const u32x4 x = *reinterpret_cast<const u32x4*>(p + 4 * i);
#pragma unroll
        for (int j = 0; j < 4; ++j) w[i + j] = x[j];
      }
    } else {
      using Piece = std::conditional_t<kCh * sizeof(Row) == 8, u32x2, std::conditional_t<kCh * sizeof(Row) == 4, uint32_t, uint16_t>>;
      const Piece x = *reinterpret_cast<const Piece*>(p);
      if constexpr (kWords == 2) {
        w[0] = x[0];
        w[1] = x[1];
      } else {
        w[0] = x;
      }
    }
  }
  __device__ __forceinline__ void get(float (&f)[kCh]) const {
#pragma unroll
    for (int j = 0; j < kCh; ++j) {
      if constexpr (sizeof(Row) == 2) {
        f[j] = __uint_as_float(j & 1 ? w[j / 2] & 0xffff0000u : w[j / 2] << 16);
      } else {
        f[j] = __uint_as_float(w[j]);
      }
    }
  }
};

// kFold tokens of an entry, their loads issued together (left to itself the
// compiler waits for each row in turn: 14.8 us for a call of a few entries).
template <class Row, int kCh>
struct FoldTurn {
  static constexpr int kFold = kCh == 8 ? 4 : 16 / kCh;
  static constexpr int kVec = kCh == 8 ? 4 : kCh;
  typedef float f32v __attribute__((ext_vector_type(kVec), aligned(4)));  // bias is 4-byte aligned
  RawRow<Row, kCh> c[kFold], z[kFold];
  f32v bias[kFold][kCh / kVec];

  // tokens p, p + 1, ... below p1 of entry e (sequence b), channels kCh grp on
  __device__ __forceinline__ void load(const CompressArgs& a, int b, int first_new, int e, int p, int p1, int grp) {
    const int64_t at = b * a.in_seq_stride + (p - first_new) * a.in_row_stride;
    const uint8_t *cp = a.c_new + at, *zp = a.z_new + at;
    const float* bp = a.bias + static_cast<int64_t>(p - e * a.m) * a.channels + grp * kCh;
#pragma unroll
    for (int u = 0; u < kFold; ++u) {  // past the last token: its row again
      z[u].load(zp, grp);
      c[u].load(cp, grp);
#pragma unroll
      for (int i = 0; i < kCh / kVec; ++i) bias[u][i] = reinterpret_cast<const f32v*>(bp)[i];
      const bool on = p + u + 1 < p1;
      zp += on ? a.in_row_stride : 0;
      cp += on ? a.in_row_stride : 0;
      bp += on ? a.channels : 0;
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  __device__ __forceinline__ void values(int u, float (&v)[kCh]) const {
    z[u].get(v);
#pragma unroll
    for (int j = 0; j < kCh; ++j) v[j] += bias[u][j / kVec][j % kVec];
  }
};

// Tokens [p, p1), at least one, of entry e (sequence b) folded into st, 8 channels a lane.
template <class Row>
__device__ __forceinline__ void fold_tokens(PoolLane<8>& st, const CompressArgs& a, int b, int first_new, int e, int p,
                                            int p1, int grp) {
  using Turn = FoldTurn<Row, 8>;
  for (; p < p1; p += Turn::kFold) {
    Turn t;
    t.load(a, b, first_new, e, p, p1, grp);
    const auto one = [&](int u) {
      float v[8], x[8];
      t.values(u, v);
      t.c[u].get(x);
      pool_fold_token(st, v, x);
    };
    if (__ballot(p1 - p < Turn::kFold)) {  // a turn past some lane's last token
#pragma unroll
      for (int u = 0; u < Turn::kFold; ++u) {
        if (u < p1 - p) one(u);
      }
    } else {
#pragma unroll
      for (int u = 0; u < Turn::kFold; ++u) one(u);
    }
  }
}

// The same, kCh = 1 or 2 channels a lane of a whole wave (p uniform).  A turn's
// weights come first, off the chain: the maximum that a token meets does not wait
// for the sums.  The next turn's loads are in flight meanwhile.
template <class Row, int kCh>
__device__ __forceinline__ void fold_tokens(PoolLane<kCh>& st, const CompressArgs& a, int b, int first_new, int e, int p,
                                            int p1, int grp) {
  using Turn = FoldTurn<Row, kCh>;
  Turn t;
  t.load(a, b, first_new, e, p, p1, grp);
  for (;;) {
    float v[Turn::kFold][kCh], x[Turn::kFold][kCh];
#pragma unroll
    for (int u = 0; u < Turn::kFold; ++u) {
      t.values(u, v[u]);
      t.c[u].get(x[u]);
    }
    const int n = p1 - p;
    p += Turn::kFold;
    if (p < p1) t.load(a, b, first_new, e, p, p1, grp);
    const auto fold = [&](auto live) {
      float w[Turn::kFold][kCh];
      bool up[Turn::kFold][kCh];
#pragma unroll
      for (int u = 0; u < Turn::kFold; ++u) {
#pragma unroll
        for (int j = 0; j < kCh; ++j) {
          const float vu = live(u) ? v[u][j] : -INFINITY;  // past the end: leaves the maximum as it is
          w[u][j] = pool_weight(vu, st.mx[j], up[u][j]);
          st.mx[j] = __builtin_elementwise_maximum(st.mx[j], vu);  // NaN stays
        }
      }
#pragma unroll
      for (int u = 0; u < Turn::kFold; ++u) {
        if (!live(u)) continue;
#pragma unroll
        for (int j = 0; j < kCh; ++j) pool_add(st.sum[j], st.acc[j], w[u][j], up[u][j], x[u][j]);
      }
    };
    if (n >= Turn::kFold) {
      fold([](int) { return true; });
    } else {
      fold([n](int u) { return u < n; });
    }
    if (p >= p1) return;
  }
}

// The block-table slot of entry e of sequence b (the caller reads it ahead of
// the fold, with the first round trip).
__device__ __forceinline__ int32_t entry_page(const CompressArgs& a, int b, int e) {
  return a.bt[b * a.bt_stride + min<int64_t>(e / a.bs, a.bt_stride - 1)];
}

// Entry e, in page `page` of its table, from its channels' states (16 lanes, 8 channels each).
__device__ __forceinline__ void emit_entry(const PoolLane<8>& st, const CompressArgs& a, int e, int32_t page, int grp) {
  const int page_idx = e / a.bs;
  if (page_idx >= a.bt_stride || page < 0 || page >= a.n_pages) return;  // uniform over the row of lanes
  uint8_t* entry = a.pool + (static_cast<int64_t>(page) * a.bs + (e - page_idx * a.bs)) * a.entry_bytes;
  const int groups = a.channels >> 3;
  float out[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) out[j] = grp < groups ? pool_out(st, j) : 0.f;
  if (a.format != SKV_FMT_F32) {
#pragma unroll
    for (int j = 0; j < 8; j += 2) bf16_round2(out[j], out[j + 1]);  // a bf16 compressor's entries
  }
  store_entry_group(entry, out, grp, groups, a.format, a.fp8_main);
}

// The blocks that a sequence's new tokens touch: blocks [e0, e1) complete in this
// call; block e0 continues from the stored state when the call before left it
// incomplete, and the tokens of block e1, when it stays incomplete, go to the
// state.  When one call does both for different blocks, workgroup 0 takes block e1
// in a turn of its own after block e0 (which is its first), so that the state is
// read before it is written.
struct CompressSpan {
  int L, first_new, e0, e1;
  bool resumes, leaves;  // block e0 has a stored state; block e1 leaves one
  int n_units;           // blocks without that last turn's
  __device__ __forceinline__ bool load(const CompressArgs& a, int b) {
    L = __builtin_amdgcn_readfirstlane(a.lens[b]);
    const int n = a.n_new ? __builtin_amdgcn_readfirstlane(a.n_new[b]) : a.n_uni;
    if (n <= 0 || n > L || n > a.in_len) return false;
    first_new = L - n;
    e0 = first_new / a.m;
    e1 = L / a.m;
    resumes = first_new > e0 * a.m;
    leaves = L > e1 * a.m;
    n_units = e1 - e0 + (leaves && !apart() ? 1 : 0);
    return true;
  }
  __device__ __forceinline__ bool apart() const { return resumes && leaves && e1 > e0; }
  __device__ __forceinline__ int from(const CompressArgs& a, int e) const { return max(first_new, e * a.m); }
  __device__ __forceinline__ int to(const CompressArgs& a, int e) const {
    return static_cast<int>(min<int64_t>(L, (e + 1) * static_cast<int64_t>(a.m)));
  }
};

struct CompressSmem {
  alignas(16) float state[kCmRows][3][kCmBlock];  // a completed entry's (max, sum, weighted sum)
};

// Workgroup bx of gx over the blocks of sequence b of a stream, the zz-th part of
// its channels; its rows of lanes are `slots` entries of as many 128-channel blocks
// as remain.
template <class Row, int kCh>
__device__ __forceinline__ void compress_workgroup(CompressSmem& sm, const CompressArgs& a, int bx, int gx, int b, int zz,
                                                   int slots) {
  constexpr int kLanes = kCmBlock / kCh, kRows = kCmThreads / kLanes;
  CompressSpan sp;
  if (!sp.load(a, b)) return;
  const bool last_turn = bx == 0 && sp.apart();
  // rows of whole waves: known uniform, so that their addresses are scalars
  const int row = (kCh == 8 ? static_cast<int>(threadIdx.x) : __builtin_amdgcn_readfirstlane(threadIdx.x)) / kLanes;
  const int zper = kRows / slots, slot = row / zper;
  const int grp0 = (zz * zper + row % zper) * kLanes, grp = grp0 + threadIdx.x % kLanes;
  const int groups = a.channels / kCh;
  const int gsafe = min(grp, groups - 1);  // lanes past the channels read the last group and store nothing
  float* sbase = a.state + static_cast<int64_t>(b) * 3 * a.channels + gsafe * kCh;
  int unit0 = bx * slots;
  while (unit0 < sp.n_units || last_turn) {
    const bool in_last = unit0 >= sp.n_units;
    if (in_last) __syncthreads();  // block e0's lanes have read the state
    const int e = in_last ? sp.e1 + slot : sp.e0 + unit0 + slot;
    const bool active = grp0 < groups && (in_last ? slot == 0 : unit0 + slot < sp.n_units);  // uniform over the row of lanes
    int32_t page = -1;
    if (active) {
      page = entry_page(a, b, e);
      PoolLane<kCh> st;
      pool_reset(st);
      if (e == sp.e0 && sp.resumes) {
#pragma unroll
        for (int j = 0; j < kCh; ++j) {
          st.mx[j] = sbase[j];
          st.sum[j] = sbase[a.channels + j];
          st.acc[j] = sbase[2 * a.channels + j];
        }
      }
      fold_tokens<Row>(st, a, b, sp.first_new, e, sp.from(a, e), sp.to(a, e), gsafe);
      if (e < sp.e1) {
        if constexpr (kCh == 8) {
          emit_entry(st, a, e, page, grp);
        } else {
          const int i = threadIdx.x % kLanes;
#pragma unroll
          for (int j = 0; j < kCh; ++j) {
            sm.state[row][0][kCh * i + j] = st.mx[j];
            sm.state[row][1][kCh * i + j] = st.sum[j];
            sm.state[row][2][kCh * i + j] = st.acc[j];
          }
        }
      } else if (grp < groups) {
#pragma unroll
        for (int j = 0; j < kCh; ++j) {
          sbase[j] = st.mx[j];
          sbase[a.channels + j] = st.sum[j];
          sbase[2 * a.channels + j] = st.acc[j];
        }
      }
    }
    if constexpr (kCh < 8) {  // the entry by 16 lanes of 8 channels
      __syncthreads();
      const int i = threadIdx.x % kLanes;
      if (active && e < sp.e1 && i < kCmBlock / 8) {
        PoolLane<8> st;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          st.mx[j] = sm.state[row][0][8 * i + j];
          st.sum[j] = sm.state[row][1][8 * i + j];
          st.acc[j] = sm.state[row][2][8 * i + j];
        }
        emit_entry(st, a, e, page, grp0 * kCh / 8 + i);
      }
      if (unit0 + gx * slots < sp.n_units) __syncthreads();  // the LDS is written again
    }
    if (in_last) break;
    unit0 += gx * slots;
  }
}

// The streams of one launch, their workgroups one after another: a stream of
// short blocks or few channels leaves the device partly idle at its end and a small
// one all along, and each call costs the host more than a small one takes.  Five
// streams (three layers; 4 prompts of 29,588 tokens in all, 235 MB of c and z rows):
// 84.5 us, 2.8 TB/s.
constexpr int kCmStreams = 16;
// Workgroups of a stream (65,535 sequences of 16 blocks of channels are fewer).  All
// streams together keep below the 2^32 threads of a launch, past which the runtime
// starts the remainder only and reports no error.
constexpr int64_t kCmMaxBlocks = (1 << 20) - 1;
static_assert(65535 * (kPoolWave * 8 * kMaxGroups / kCmBlock) <= kCmMaxBlocks &&
              kCmStreams * kCmMaxBlocks * kCmThreads < int64_t(1) << 32, "one launch");

struct CompressStreams {
  CompressArgs s[kCmStreams];
  int32_t first[kCmStreams];     // first workgroup
  int32_t turns[kCmStreams];     // workgroups over a sequence's blocks
  int32_t zparts[kCmStreams];    // workgroups over the channels
  int32_t slots[kCmStreams];     // entries of a workgroup at a time
  int32_t channels[kCmStreams];  // of a lane: 8, 2 or 1
  int32_t n;
};

template <class Row>
__global__ __launch_bounds__(kCmThreads, sizeof(Row) == 2 ? 3 : 2) void k_compress_append(CompressStreams cs) {
  __shared__ CompressSmem sm;
  int i = 0;
  while (i + 1 < cs.n && static_cast<int>(blockIdx.x) >= cs.first[i + 1]) ++i;  // uniform
  const CompressArgs& a = cs.s[i];
  const int l = blockIdx.x - cs.first[i];
  const int rest = l / cs.zparts[i], zz = l - rest * cs.zparts[i];
  const int b = rest / cs.turns[i], bx = rest - b * cs.turns[i];
  if (cs.channels[i] == 8) {  // uniform
    compress_workgroup<Row, 8>(sm, a, bx, cs.turns[i], b, zz, cs.slots[i]);
  } else if (cs.channels[i] == 2) {
    compress_workgroup<Row, 2>(sm, a, bx, cs.turns[i], b, zz, cs.slots[i]);
  } else {
    compress_workgroup<Row, 1>(sm, a, bx, cs.turns[i], b, zz, cs.slots[i]);
  }
}

}  // namespace skv

using namespace skv;

// One stream's arguments, checked; 0 or an error code.
static int compress_args(const char* what, const skv_compress_stream& x, int64_t batch, CompressArgs& a, bool& in_f32) {
  in_f32 = (x.format & SKV_FMT_IN_F32) || (x.format & ~SKV_FMT_IN_F32) == SKV_FMT_F32;
  const int32_t format = x.format & ~SKV_FMT_IN_F32;
  const int64_t m = x.m, channels = x.channels;
  if (m <= 0 || m > 4096) return set_error(SKV_EINVAL, "%s: compression_rate must be in [1, 4096]; got %lld", what, (long long)m);
  if (channels <= 0 || (channels & 7) || channels > kPoolWave * 8 * kMaxGroups) {
    return set_error(SKV_EINVAL, "%s: channels must be a multiple of 8 in [8, %d]; got %lld", what,
                     kPoolWave * 8 * kMaxGroups, (long long)channels);
  }
  if (x.block_size <= 0 || x.bt_stride <= 0 || batch < 0 || batch > 65535) {
    return set_error(SKV_EINVAL, "%s: bad block_size/bt_stride/batch", what);
  }
  const int fp8_main = (format == SKV_FMT_F32) ? ((x.entry_bytes == channels * 4) ? 0 : -1)
                                               : entry_layout(format, channels, x.entry_bytes);
  if (fp8_main < 0) {
    return set_error(SKV_EINVAL,
                     "%s: entry_bytes %lld does not match format %d with %lld channels (bf16: 2*channels; "
                     "fp32: 4*channels; fp8: channels = 128*q + %d, entry_bytes = %lld)",
                     what, (long long)x.entry_bytes, format, (long long)channels, SKV_FP8_ROPE_DIMS,
                     (long long)SKV_FP8_ENTRY_BYTES(channels));
  }
  const uintptr_t align = reinterpret_cast<uintptr_t>(x.pool) | reinterpret_cast<uintptr_t>(x.tail_state) |
                          reinterpret_cast<uintptr_t>(x.c_new) |
                          reinterpret_cast<uintptr_t>(x.z_new) | static_cast<uintptr_t>(x.in_seq_stride) |
                          static_cast<uintptr_t>(x.in_row_stride);
  if (align & 15) return set_error(SKV_EINVAL, "%s: pointers and strides must be 16-byte aligned", what);
  if (!x.bias || (reinterpret_cast<uintptr_t>(x.bias) & 3)) return set_error(SKV_EINVAL, "%s: bias must be fp32", what);
  a = CompressArgs{};
  a.pool = static_cast<uint8_t*>(x.pool);
  a.entry_bytes = x.entry_bytes;
  a.bs = static_cast<int>(x.block_size);
  a.n_pages = x.n_pages;
  a.bt = x.block_table;
  a.bt_stride = x.bt_stride;
  a.state = x.tail_state;
  a.c_new = static_cast<const uint8_t*>(x.c_new);
  a.z_new = static_cast<const uint8_t*>(x.z_new);
  a.in_seq_stride = x.in_seq_stride;
  a.in_row_stride = x.in_row_stride;
  a.in_len = x.in_len;
  a.bias = x.bias;
  a.m = static_cast<int>(m);
  a.channels = static_cast<int>(channels);
  a.format = format;
  a.fp8_main = fp8_main;
  return SKV_OK;
}

static int launch_streams(const char* what, CompressStreams& cs, int64_t blocks, bool in_f32, void* stream) {
  if (cs.n == 0) return SKV_OK;
  const dim3 grid(static_cast<unsigned>(blocks));
  if (in_f32) {
    hipLaunchKernelGGL(k_compress_append<float>, grid, dim3(kCmThreads), 0, static_cast<hipStream_t>(stream), cs);
  } else {
    hipLaunchKernelGGL(k_compress_append<uint16_t>, grid, dim3(kCmThreads), 0, static_cast<hipStream_t>(stream), cs);
  }
  cs.n = 0;
  return check_launch(what);
}

static int compress_streams(const char* what, const skv_compress_stream* streams, int64_t n_streams,
                            const int32_t* seq_lens, const int32_t* n_new, int32_t n_new_uniform, int64_t batch,
                            void* stream) {
  CompressArgs a;
  bool f32 = false, run_f32 = false;
  for (int64_t i = 0; i < n_streams; ++i) {  // every stream before any launch
    if (const int rc = compress_args(what, streams[i], batch, a, f32)) return rc;
  }
  if (!n_new && n_new_uniform < 0) return set_error(SKV_EINVAL, "%s: n_new_uniform must be >= 0", what);
  if (batch == 0) return SKV_OK;
  CompressStreams cs{};
  int64_t blocks = 0;
  for (int64_t i = 0; i < n_streams; ++i) {
    if (streams[i].in_len <= 0) continue;
    if (const int rc = compress_args(what, streams[i], batch, a, f32)) return rc;
    a.lens = seq_lens;
    a.n_new = n_new;
    a.n_uni = n_new_uniform;
    if (cs.n == kCmStreams || (cs.n > 0 && f32 != run_f32)) {
      if (const int rc = launch_streams(what, cs, blocks, run_f32, stream)) return rc;
    }
    if (cs.n == 0) blocks = 0;
    run_f32 = f32;
    // a call's tokens lie in at most ceil((in_len - 1) / m) + 1 blocks
    const int64_t units = ceil_div(a.in_len - 1, a.m) + 1, zblocks = ceil_div(a.channels, kCmBlock);
    const int64_t tokens = std::min<int64_t>(a.m, a.in_len);  // most of an entry
    const int ch = tokens <= 4 ? 8 : units * batch * zblocks < 8 * device_cus() ? 1 : tokens < 16 ? 8 : 2;
    // Rows not needed for a sequence's entries take further blocks of channels, where
    // the device stays full that way: a token for each of 256 sequences 6.7 us (9.9
    // with a workgroup per block of channels, 8.8 with a wave per sequence), of 1,024
    // 11.6 (22.4, 19.3); of 4 sequences with 8 tokens it takes 10.2, not 7.8.
    const int rows = kCmThreads * ch / kCmBlock;
    int slots = 1;
    while (slots < rows && slots < units) slots *= 2;
    if (batch * ceil_div(units, slots) * ceil_div(zblocks, rows / slots) < device_cus()) slots = rows;
    const int64_t zparts = ceil_div(zblocks, rows / slots);
    // past its share of a launch's workgroups each of a stream's takes several turns
    const int64_t turns = std::min<int64_t>(ceil_div(units, slots), std::max<int64_t>(1, kCmMaxBlocks / (batch * zparts)));
    cs.s[cs.n] = a;
    cs.first[cs.n] = static_cast<int32_t>(blocks);
    cs.turns[cs.n] = static_cast<int32_t>(turns);
    cs.zparts[cs.n] = static_cast<int32_t>(zparts);
    cs.slots[cs.n] = slots;
    cs.channels[cs.n] = ch;
    ++cs.n;
    blocks += turns * batch * zparts;
  }
  return launch_streams(what, cs, blocks, run_f32, stream);
}

extern "C" int skv_compress_append(void* pool, int64_t entry_bytes, int64_t block_size,
                                   int64_t n_pages, const int32_t* block_table, int64_t bt_stride,
                                   float* tail_state, const void* c_new, const void* z_new,
                                   int64_t in_seq_stride, int64_t in_row_stride, int64_t in_len,
                                   const float* bias, const int32_t* seq_lens, const int32_t* n_new,
                                   int32_t n_new_uniform, int64_t m, int64_t channels,
                                   int32_t format, int64_t batch, void* stream) {
  const skv_compress_stream x{pool,  entry_bytes,   block_size,    n_pages, block_table, bt_stride, tail_state, c_new,
                              z_new, in_seq_stride, in_row_stride, in_len,  bias,        m,         channels,   format, 0};
  return compress_streams("skv_compress_append", &x, 1, seq_lens, n_new, n_new_uniform, batch, stream);
}

extern "C" int skv_compress_append_streams(const skv_compress_stream* streams, int64_t n_streams,
                                           const int32_t* seq_lens, const int32_t* n_new, int32_t n_new_uniform,
                                           int64_t batch, void* stream) {
  const char* what = "skv_compress_append_streams";
  if (n_streams < 0 || (n_streams > 0 && !streams)) return set_error(SKV_EINVAL, "%s: no streams", what);
  return compress_streams(what, streams, n_streams, seq_lens, n_new, n_new_uniform, batch, stream);
}
