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
// so a decode step costs O(channels) whatever m is, and a block emits from
// that state the same value a one-shot pooling of its m tokens gives.
#include <algorithm>

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

// Work split.  The pooling is independent per channel, so a workgroup takes a
// block of 128 channels (one fp8 scale block): 16 lanes of 8 channels read
// 256 consecutive bytes of a token row, and the 16 lane groups of its 4 waves
// are shared out between entries and token slices.  kSlices lane groups fold
// the tokens of one entry in turn, 4 tokens of a lane in flight at once, and
// are merged by lane shuffles (and through LDS for 16 slices); the other lane
// groups hold other entries.  A block of 4 tokens needs no slices (16 entries
// per workgroup); one of 128 takes all 16 lane groups, 8 tokens each.
// HBM-bound: c and z rows are read once.  One wave folding an entry's tokens one
// after another, with a memory round trip each, took 1.45 us per token.  4
// sequences of 6,700-8,192 tokens x 576 bf16 channels: entries of 4 tokens 33 us
// (2.6 TB/s; the call averaged 247 us before; 25 with the weights of a turn taken
// against its max at once, which moves the last bits of the sums and so codes of
// fp8 entries), of 128 tokens 26 us; 16 x 8,192 tokens in entries of 4 110 us; two
// sequences of 95 and 300 tokens 5.5 and, with blocks of 128, 8.3 us (186 before).
constexpr int kCmThreads = 256;
constexpr int kCmWaves = kCmThreads / kWave;
constexpr int kCmLanes = 16;                         // lanes per 128-channel token row
constexpr int kCmGroups = kCmThreads / kCmLanes;     // lane groups per workgroup
constexpr int kCmFold = 4;                           // tokens in flight per lane

struct CompressSmem {
  float mx[kCmWaves][8][kCmLanes];  // of 16 slices: each wave's max, then its sums from the common max
  float sum[kCmWaves - 1][8][kCmLanes], acc[kCmWaves - 1][8][kCmLanes];
};

// A lane's 8 channels of a row as they lie in memory (bf16 or fp32).
template <class Row>
struct RawRow {
  static constexpr int kVecs = sizeof(Row) / 2;  // 16-byte pieces
  u32x4 v[kVecs];
  __device__ __forceinline__ void load(const uint8_t* row, int grp) {
    const u32x4* p = reinterpret_cast<const u32x4*>(row + grp * 16 * kVecs);
#pragma unroll
    for (int i = 0; i < kVecs; ++i) v[i] = p[i];
  }
  __device__ __forceinline__ void get(float* f) const {
    if constexpr (kVecs == 1) {
      unpack8_bf16(v[0], f);
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) f[j] = __uint_as_float(v[j >> 2][j & 3]);
    }
  }
};

// Tokens first + slice + stride * i < p1 of entry e (sequence b) folded into
// st.  Every load of a turn is issued before any is used (left to itself the
// compiler waits for each row in turn: 14.8 us for a call of a few entries).
template <class Row, bool kSerial>
__device__ __forceinline__ void fold_tokens(PoolLane& st, const CompressArgs& a, int b, int first_new, int e, int first,
                                            int p1, int slice, int stride, int grp) {
  typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));  // bias is 4-byte aligned
  const uint8_t* cbase = a.c_new + b * a.in_seq_stride;
  const uint8_t* zbase = a.z_new + b * a.in_seq_stride;
  for (int p = first + slice; p < p1; p += kCmFold * stride) {
    RawRow<Row> cr[kCmFold], zr[kCmFold];
    f32x4u br[kCmFold][2];
    bool live[kCmFold];
#pragma unroll
    for (int u = 0; u < kCmFold; ++u) {
      const int pu = p + u * stride;
      live[u] = pu < p1;
      const int q = live[u] ? pu : p;  // a row that exists
      const int64_t off = (q - first_new) * a.in_row_stride;
      zr[u].load(zbase + off, grp);
      cr[u].load(cbase + off, grp);
      const f32x4u* bp = reinterpret_cast<const f32x4u*>(a.bias + static_cast<int64_t>(q - e * a.m) * a.channels + grp * 8);
      br[u][0] = bp[0];
      br[u][1] = bp[1];
    }
    __builtin_amdgcn_sched_barrier(0);
    float v[kCmFold][8], c[kCmFold][8];
#pragma unroll
    for (int u = 0; u < kCmFold; ++u) {
      zr[u].get(v[u]);
      cr[u].get(c[u]);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[u][j] += br[u][j >> 2][j & 3];
    }
    const bool part = __ballot(!live[kCmFold - 1]);  // a turn past some lane's last token
    if constexpr (kSerial) {
      if (part) {
#pragma unroll
        for (int u = 0; u < kCmFold; ++u) {
          if (live[u]) pool_fold_token(st, v[u], c[u]);
        }
      } else {
        pool_fold_serial<kCmFold>(st, v, c);
      }
    } else {
      if (part) {  // tokens past the end: value -inf whatever the bias, row -0: nothing is added
#pragma unroll
        for (int u = 1; u < kCmFold; ++u) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            v[u][j] = live[u] ? v[u][j] : -INFINITY;
            c[u][j] = live[u] ? c[u][j] : -0.f;
          }
        }
      }
      pool_fold<kCmFold>(st, v, c);
    }
  }
}

// The states of the lane groups of one entry, merged: every lane group holds
// the result for 1 and 4 slices (one lane group, one wave), wave 0 for 16.
// For 16 slices every thread of the workgroup must call it.
template <int kSlices>
__device__ __forceinline__ void merge_slices(CompressSmem& sm, PoolLane& st) {
  static_assert(kSlices == 1 || kSlices == 4 || kSlices == 16, "one lane group, one wave or the workgroup");
  if constexpr (kSlices == 1) return;
  float M[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    M[j] = __builtin_elementwise_maximum(st.mx[j], __shfl_xor(st.mx[j], 16));
    M[j] = __builtin_elementwise_maximum(M[j], __shfl_xor(M[j], 32));
  }
  pool_rebase(st, M);
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    st.sum[j] += __shfl_xor(st.sum[j], 16);
    st.acc[j] += __shfl_xor(st.acc[j], 16);
    st.sum[j] += __shfl_xor(st.sum[j], 32);
    st.acc[j] += __shfl_xor(st.acc[j], 32);
  }
  if constexpr (kSlices == 16) {
    const int wave = threadIdx.x / kWave, l = threadIdx.x % kCmLanes;
    if (threadIdx.x % kWave < kCmLanes) {
#pragma unroll
      for (int j = 0; j < 8; ++j) sm.mx[wave][j][l] = st.mx[j];
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      M[j] = sm.mx[0][j][l];
#pragma unroll
      for (int w = 1; w < kCmWaves; ++w) M[j] = __builtin_elementwise_maximum(M[j], sm.mx[w][j][l]);
    }
    pool_rebase(st, M);
    if (wave > 0 && threadIdx.x % kWave < kCmLanes) {
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        sm.sum[wave - 1][j][l] = st.sum[j];
        sm.acc[wave - 1][j][l] = st.acc[j];
      }
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
      for (int w = 0; w < kCmWaves - 1; ++w) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          st.sum[j] += sm.sum[w][j][l];
          st.acc[j] += sm.acc[w][j][l];
        }
      }
    }
  }
}

// The block-table slot of entry e of sequence b (the caller reads it ahead of
// the fold, with the first round trip).
__device__ __forceinline__ int32_t entry_page(const CompressArgs& a, int b, int e) {
  return a.bt[b * a.bt_stride + min<int64_t>(e / a.bs, a.bt_stride - 1)];
}

// Entry e, in page `page` of its table, from its channels' states (16 lanes, 8 channels each).
__device__ __forceinline__ void emit_entry(const PoolLane& st, const CompressArgs& a, int e, int32_t page, int grp,
                                           int groups) {
  const int page_idx = e / a.bs;
  if (page_idx >= a.bt_stride || page < 0 || page >= a.n_pages) return;  // uniform over the lane group
  uint8_t* entry = a.pool + (static_cast<int64_t>(page) * a.bs + (e - page_idx * a.bs)) * a.entry_bytes;
  float out[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) out[j] = grp < groups ? pool_out(st, j) : 0.f;
  if (a.format != SKV_FMT_F32) {
#pragma unroll
    for (int j = 0; j < 8; j += 2) bf16_round2(out[j], out[j + 1]);  // a bf16 compressor's entries
  }
  store_entry_group(entry, out, grp, groups, a.format, a.fp8_main);
}

// One workgroup of a stream: workgroup bx of gx over the blocks of sequence b,
// 128-channel block zb.  Blocks
// [e0, e1) of a sequence complete in this call; block e0 continues from the
// stored state when the call before left it incomplete, and the tokens of
// block e1, when it stays incomplete, go to the state.  When one call does
// both for different blocks, workgroup 0 takes block e1 in a turn of its own
// after block e0 (which is its first), so that the state is read before it
// is written.
template <class Row, int kSlices>
__device__ __forceinline__ void compress_workgroup(CompressSmem& sm, const CompressArgs& a, int bx, int gx, int b, int zb) {
  constexpr int kEntries = kCmGroups / kSlices;  // per workgroup and turn
  const int L = a.lens[b];
  const int n = a.n_new ? a.n_new[b] : a.n_uni;
  if (n <= 0 || n > L || n > a.in_len) return;
  const int first_new = L - n;
  const int e0 = first_new / a.m;
  const int e1 = L / a.m;
  const bool resumes = first_new > e0 * a.m;  // block e0 has a stored state
  const bool leaves = L > e1 * a.m;           // block e1 leaves one
  bool last_turn = bx == 0 && resumes && leaves && e1 > e0;
  const int n_units = e1 - e0 + (leaves && !(resumes && e1 > e0) ? 1 : 0);
  const int groups = a.channels >> 3;
  const int grp = zb * kCmLanes + threadIdx.x % kCmLanes;
  const int gsafe = min(grp, groups - 1);  // lanes past the channels read the last group and store nothing
  const int slot = threadIdx.x / kCmLanes / kSlices, slice = threadIdx.x / kCmLanes % kSlices;
  float* sbase = a.state + static_cast<int64_t>(b) * 3 * a.channels + gsafe * 8;
  int unit0 = bx * kEntries;
  while (unit0 < n_units || last_turn) {
    const bool in_last = unit0 >= n_units;
    if (in_last) __syncthreads();  // block e0's lanes have read the state
    const int unit = in_last ? e1 - e0 + slot : unit0 + slot;
    const int e = e0 + unit;
    const bool active = in_last ? slot == 0 : unit < n_units;
    PoolLane st;
    pool_reset(st);
    int32_t page = -1;
    if (active) {
      page = entry_page(a, b, e);
      if (e == e0 && slice == 0 && resumes) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          st.mx[j] = sbase[j];
          st.sum[j] = sbase[a.channels + j];
          st.acc[j] = sbase[2 * a.channels + j];
        }
      }
      fold_tokens<Row, kSlices == 1>(st, a, b, first_new, e, max(first_new, e * a.m), min(L, (e + 1) * a.m), slice, kSlices, gsafe);
    }
    merge_slices<kSlices>(sm, st);
    if (active && slice == 0) {
      if (e < e1) {
        emit_entry(st, a, e, page, grp, groups);
      } else if (grp < groups) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          sbase[j] = st.mx[j];
          sbase[a.channels + j] = st.sum[j];
          sbase[2 * a.channels + j] = st.acc[j];
        }
      }
    }
    if (in_last) break;
    unit0 += gx * kEntries;
    if constexpr (kSlices == 16) __syncthreads();  // the LDS is written again
  }
}

// The streams of one launch, their workgroups one after another: a stream of
// short blocks or few channels leaves the device partly idle at its end and a small
// one all along, and each call costs the host more than a small one takes.  Five
// streams (three layers; 4 prompts of 6,700-8,192 tokens): 112 us in five launches,
// 73 in one (3.1 TB/s).
constexpr int kCmStreams = 16;

struct CompressStreams {
  CompressArgs s[kCmStreams];
  int32_t first[kCmStreams];  // first workgroup
  int32_t turns[kCmStreams];  // workgroups over a sequence's blocks
  int32_t zblocks[kCmStreams];
  int32_t slices[kCmStreams];
  int32_t n, batch;
};

template <class Row>
__global__ __launch_bounds__(kCmThreads, sizeof(Row) == 2 ? 3 : 2) void k_compress_append(CompressStreams cs) {
  __shared__ CompressSmem sm;
  int i = 0;
  while (i + 1 < cs.n && static_cast<int>(blockIdx.x) >= cs.first[i + 1]) ++i;  // uniform
  const CompressArgs& a = cs.s[i];
  const int l = blockIdx.x - cs.first[i];
  const int rest = l / cs.zblocks[i], zb = l - rest * cs.zblocks[i];
  const int b = rest / cs.turns[i], bx = rest - b * cs.turns[i];
  switch (cs.slices[i]) {  // uniform
    case 1: compress_workgroup<Row, 1>(sm, a, bx, cs.turns[i], b, zb); break;
    case 4: compress_workgroup<Row, 4>(sm, a, bx, cs.turns[i], b, zb); break;
    default: compress_workgroup<Row, 16>(sm, a, bx, cs.turns[i], b, zb); break;
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
  cs.batch = static_cast<int32_t>(batch);
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
    // slices of an entry: at least 4 tokens per lane, which a turn of fold_tokens takes at once
    // (blocks of 8 over 4 slices: 54 us for 4 x 8192 tokens of 576 channels, over one: 24 us)
    const int slices = a.m < 16 ? 1 : a.m < 64 ? 4 : 16;
    const int64_t zblocks = ceil_div(a.channels, 8 * kCmLanes);
    // a call's tokens lie in at most ceil(in_len / m) + 1 blocks; past 2^26
    // workgroups of a stream each takes several turns
    const int64_t turns = std::min<int64_t>(ceil_div(ceil_div(a.in_len, a.m) + 1, kCmGroups / slices),
                                            std::max<int64_t>(1, (1 << 26) / (batch * zblocks)));
    cs.s[cs.n] = a;
    cs.first[cs.n] = static_cast<int32_t>(blocks);
    cs.turns[cs.n] = static_cast<int32_t>(turns);
    cs.zblocks[cs.n] = static_cast<int32_t>(zblocks);
    cs.slices[cs.n] = slices;
    ++cs.n;
    blocks += turns * batch * zblocks;
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
