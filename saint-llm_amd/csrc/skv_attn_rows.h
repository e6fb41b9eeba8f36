// Attention of many query rows (a prompt chunk, or a large decode batch): one
// workgroup per (query row, 64 heads) does the row's whole attention, both
// branches, and writes the output itself.  Included by skv_attention.hip, whose
// argument and fp8 definitions it uses.
//
// k_attn_part splits a row over units so that few rows fill the device, writes
// each unit's output and merges them in a second launch.  With a row per CU
// that costs more than the split gives: two units' outputs written and read
// back, and 4.5 us per 32-key tile, of which the products are 0.5, for its four
// barriers and a softmax that stands between the products.  Here the waves of a
// SIMD do different work:
//   * wave j < 4 holds the query of 16 heads (all dims) in registers and
//     computes each tile's scores and softmax: S = K Q^T, whole in the wave, to the
//     weights P in LDS;
//   * wave 4 + (hh, dh) holds the output of 32 heads x half of the dims and adds
//     P V of the tile before, so that one wave's softmax runs under the other's
//     products.  A V operand read from LDS feeds two products.
// One barrier ends a turn; the turns walk one stream of tiles through three LDS
// buffers: the window's keys (their scores are kept in LDS), the compressed
// entries (K = V, online softmax), the window's values, which waves 0-3 multiply
// themselves, the query's registers being free by then.  Their output, rounded
// to bf16 as the split path rounds its partial outputs, is handed over in LDS
// and added to the compressed branch's when that is written.
// 64 heads x 576, window 128: 512 rows over 512 picks 114 us (216 split), 1,000
// rows over 504 entries each 215 us (434): 1.66 us per tile, 25 us per row for the
// window, the start and the output.  A tile's LDS traffic (each of the 4 score waves
// reads its keys) is 1.0 of the 1.66; waves 0-3, a tile's scores then its softmax
// then their share of the staging one after another, end a turn last.  Loads
// issued between the products instead of at the turn's end: 134 us (spills).
#pragma once

namespace skv {

constexpr int kRowsWinTiles = 4;                          // window tiles whose scores LDS holds
constexpr int kRowsMaxWindow = kRowsWinTiles * kAtTile;

struct AttnRowsArgs {
  AttnArgs a;
  float* out;         // [rows, H, D]
  const float* sink;  // [H] or nullptr
  int32_t sink_comp;  // the compressed branch takes the sink (HCA)
};

template <int NKS>
struct RowsSmem {
  static constexpr int kD = NKS * 32;
  alignas(16) uint16_t tile[3][kAtTile * kD];  // rows of kD elements, chunks swizzled by rows_chunk
  u32x4 p[2][4][kWave];                        // [turn][16 heads][lane]: weights as the A operands of O += P V
  f32x4 sw[kRowsWinTiles][4][2][kWave];        // the window's scores as their wave holds them
  // per buffer and key: 1 / rms (1 for the window, 0 masked), it times the scores'
  // scale, and what is added to a scaled score (-inf masked)
  float rms[3][kAtTile], scale[3][kAtTile], mask[3][kAtTile];
  int64_t win_row[kRowsMaxWindow], row[kAtRun];  // source rows of the window's keys and of a run of the compressed
  float w[kAtMaxD];                            // k_norm weight
  alignas(16) float alpha[2][kAtHeads];        // [turn]: rescale of each head's O, where moved
  int moved[2][4];                             // [turn][16 heads]: a head's reference max moved
  alignas(16) float fin[kAtHeads];             // each head's factor of the compressed branch's O
};

// Chunk c (8 dims) of tile row r sits at chunk c ^ f(r), f(r) = 2 (r % 4) + (r / 4) % 2
// of its LDS row (rows start at the same bank).  The 8 lanes of a cycle of a K
// operand read (8 rows, one chunk) and the 16 lanes of a cycle of a V
// transposing read (rows 4g..4g+3, an aligned pair of chunks each) touch every
// bank once.
__device__ __forceinline__ int rows_chunk(int r, int c) { return c ^ (((r & 3) << 1) | ((r >> 2) & 1)); }

// Sum of the squares of two bf16 values, added to s (fp32).
__device__ __forceinline__ float dot2_sq(uint32_t v, float s) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  const bf16x2_t x = __builtin_bit_cast(bf16x2_t, v);
  return __builtin_amdgcn_fdot2_f32_bf16(x, x, s, false);
}

// The larger of x and the values 16 and 32 lanes away, and their sum (permutes
// of the vector unit: no LDS latency).
__device__ __forceinline__ float max_over_groups(float x) {
  const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(r16[0]), __uint_as_float(r16[1]));
  const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r32[0]), __uint_as_float(r32[1]));
}
__device__ __forceinline__ float sum_over_groups(float x) {
  const auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r16[0]) + __uint_as_float(r16[1]);
  const auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r32[0]) + __uint_as_float(r32[1]);
}

// The thread's index, computed from anew wherever it is asked for: addresses
// held from turn to turn would spill, and a spilled register's reload waits for
// every tile load issued before it.
__device__ __forceinline__ int fresh_tid() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

// A tile in flight: thread 16r + c0 holds chunks c0, c0 + 16, ... of key r, so
// that one row offset, one address and constant offsets serve all its loads
// and LDS stores.  Masked keys, and dims past D, read the zero row.  An fp8
// entry's codes are 8-code chunks c0 + 16k under scale k, its bf16 dims a chunk
// on the first 8 threads of a row; it is dequantized (fp32 product rounded to
// bf16, as the gathers do) when stored.
template <int NKS, bool kFp8>
struct RowsRaw {
  static constexpr int kChunks = NKS * 4;
  static constexpr int kPer = (kChunks + 15) / 16;
  static_assert(!kFp8 || (kFp8CodeChunks == 64 && kFp8RopeChunks == 8 && kFp8Main / 128 == 4 && kPer >= 4),
                "16 threads per 576-dim entry");
  u32x4 v[kPer];
  bool live;

  __device__ __forceinline__ void load(const int64_t* rows, const uint8_t* base, int D) {
    const int tid = fresh_tid(), c0 = tid & 15;
    const int64_t off = rows[tid >> 4];
    live = off >= 0;
    const uint8_t* p = live ? base + off : g_zero_row;
    if (D == NKS * 32) {  // uniform
#pragma unroll
      for (int k = 0; k < kPer; ++k) v[k] = *reinterpret_cast<const u32x4*>(p + 16 * min(c0 + 16 * k, kChunks - 1));
    } else {
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const int c = min(c0 + 16 * k, kChunks - 1);
        v[k] = *reinterpret_cast<const u32x4*>((8 * c < D ? p : g_zero_row) + 16 * c);
      }
    }
  }
  __device__ __forceinline__ void load_fp8(const int64_t* rows, const uint8_t* base) {
    const int tid = fresh_tid(), c0 = tid & 15;
    const int64_t off = rows[tid >> 4];
    live = off >= 0;
    const uint8_t* p = live ? base + off : g_zero_row;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const u32x2 lo = *reinterpret_cast<const u32x2*>(p + 8 * (c0 + 32 * k));
      const u32x2 hi = *reinterpret_cast<const u32x2*>(p + 8 * (c0 + 32 * k + 16));
      v[k] = u32x4{lo[0], lo[1], hi[0], hi[1]};
    }
    v[2] = *reinterpret_cast<const u32x4*>(p + kFp8Main);  // the four scales
    v[3] = *reinterpret_cast<const u32x4*>(p + kFp8Main + 16 + 16 * (c0 & 7));
  }

  // To LDS, with the key's factors (kNorm: k_norm's).
  template <bool kNorm>
  __device__ __forceinline__ void store(RowsSmem<NKS>& sm, int buf, float inv_d, float eps, float scale2) const {
    uint16_t* const dst = sm.tile[buf];
    const int tid = fresh_tid(), r = tid >> 4, c0 = tid & 15;
    uint16_t* d = dst + r * (NKS * 32) + 8 * rows_chunk(r, c0);
    float s = 0.f;
    const auto put = [&](int k, u32x4 x) {
      if (kChunks % 16 == 0 || c0 + 16 * k < kChunks) {
        *reinterpret_cast<u32x4*>(d + 128 * k) = x;
        if constexpr (kNorm) {
#pragma unroll
          for (int j = 0; j < 4; ++j) s = dot2_sq(x[j], s);
        }
      }
    };
    if constexpr (kNorm && kFp8) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float scale = __uint_as_float(v[2][k]);
        float f[8];
        e4m3fn_x4_to_f32(v[k >> 1][2 * (k & 1)], f);
        e4m3fn_x4_to_f32(v[k >> 1][2 * (k & 1) + 1], f + 4);
        u32x4 x;
#pragma unroll
        for (int h = 0; h < 4; ++h) x[h] = bf16_pack2(f[2 * h] * scale, f[2 * h + 1] * scale);
        put(k, x);
      }
      put(4, v[3]);
    } else {
#pragma unroll
      for (int k = 0; k < kPer; ++k) put(k, v[k]);
    }
    if constexpr (kNorm) {  // over the row's 16 threads
      s += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(s), 0x128, 0xf, 0xf, false));  // row_ror:8
      s += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(s), 0x124, 0xf, 0xf, false));
      s += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(s), 0x122, 0xf, 0xf, false));
      s += __uint_as_float(__builtin_amdgcn_update_dpp(0, __float_as_uint(s), 0x121, 0xf, 0xf, false));
    }
    if (c0 == 0) {
      const float rk = kNorm ? __builtin_amdgcn_rsqf(fmaf(s, inv_d, eps)) : 1.f;
      sm.rms[buf][r] = live ? rk : 0.f;
      sm.scale[buf][r] = rk * scale2;
      sm.mask[buf][r] = live ? 0.f : -__builtin_huge_valf();
    }
  }
};

// A query row, and where its tiles come from: tiles [0, n_w) are the window's
// keys, the next n_c the compressed entries, the last n_w the window's values.
struct RowsStream {
  int b, hg, cb, L;  // query row, head group, sequence, tokens the row sees
  int n_win, n_comp;  // keys
  int n_w, n_c;       // tiles
  float inv_d, scale2;  // 1 / D, log2(e) / sqrt(D)
  __device__ __forceinline__ int total() const { return 2 * n_w + n_c; }
  // turn t takes tile t; the output of the last compressed tile is the turn after's
  __device__ __forceinline__ int turns() const { return n_w > 0 ? total() : n_c + 1; }
};

// Source rows of compressed keys [k_lo, k_hi): byte offsets, -1 for masked
// ones.  pick0: the calling thread's pick of the first run, read ahead.
__device__ __forceinline__ void rows_resolve(int64_t* rows, const AttnArgs& a, const RowsStream& st, int k_lo, int k_hi,
                                             const int32_t* pick0 = nullptr) {
  for (int j = k_lo + static_cast<int>(threadIdx.x); j < k_hi; j += kAtThreads) {
    int64_t row = -1;
    if (j < st.n_comp) {
      int e = j;
      if (a.kind == SKV_LAYER_CSA) {
        e = pick0 ? *pick0 : a.picks[static_cast<int64_t>(st.b) * a.pick_stride + j];
        if (e >= max(a.n_entries[st.cb], 0)) e = -1;
      }
      if (e >= 0) {
        const int pi = static_cast<int>(udiv24(e, a.block_size));
        if (pi < a.bt_stride) {
          const int32_t page = a.block_table[static_cast<int64_t>(st.cb) * a.bt_stride + pi];
          if (page >= 0 && page < a.n_pages) {
            row = (static_cast<int64_t>(page) * a.block_size + (e - pi * a.block_size)) * a.entry_bytes;
          }
        }
      }
    }
    rows[j - k_lo] = row;
  }
}

// The loads of tile t of the stream.  Every thread of the workgroup calls it
// (a new run of compressed keys is resolved on the way).
template <int NKS, bool kFp8>
__device__ __forceinline__ void rows_load(RowsSmem<NKS>& sm, RowsRaw<NKS, kFp8>& raw, const AttnArgs& a,
                                          const RowsStream& st, int t) {
  const int c = t - st.n_w;
  if (c >= 0 && c < st.n_c) {
    constexpr int kRunTiles = kAtRun / kAtTile;
    if (c > 0 && c % kRunTiles == 0) {  // uniform; the rows of the run before have been read
      lds_barrier();
      rows_resolve(sm.row, a, st, c * kAtTile, min(st.n_c * kAtTile, c * kAtTile + kAtRun));
      lds_barrier();
    }
    const int64_t* rows = sm.row + (c % kRunTiles) * kAtTile;
    if constexpr (kFp8) {
      raw.load_fp8(rows, a.pool);
    } else {
      raw.load(rows, a.pool, a.D);
    }
  } else {
    const bool key = c < 0;
    raw.load(sm.win_row + (key ? t : c - st.n_c) * kAtTile, key ? a.win_k : a.win_v, a.D);
  }
}

// Tile t to its LDS buffer.
template <int NKS, bool kFp8>
__device__ __forceinline__ void rows_store(RowsSmem<NKS>& sm, const RowsRaw<NKS, kFp8>& raw, const AttnArgs& a,
                                           const RowsStream& st, int t) {
  if (t >= st.n_w && t < st.n_w + st.n_c) {
    raw.template store<true>(sm, t % 3, st.inv_d, a.eps, st.scale2);
  } else {
    raw.template store<false>(sm, t % 3, st.inv_d, a.eps, st.scale2);
  }
}

// The end of turn t, on every wave: tile t + 1, loaded since the turn before,
// goes to LDS (its buffer's last reader was turn t - 1), tile t + 2 is loaded.
template <int NKS, bool kFp8>
__device__ __forceinline__ void rows_next(RowsSmem<NKS>& sm, RowsRaw<NKS, kFp8>& raw, const AttnArgs& a,
                                          const RowsStream& st, int t) {
  if (t + 1 < st.total()) rows_store(sm, raw, a, st, t + 1);
  if (t + 2 < st.total()) rows_load(sm, raw, a, st, t + 2);
  lds_barrier();
}

// Waves 0-3: scores and softmax of heads 16 wave + col.
template <int NKS, bool kFp8>
__device__ __forceinline__ void rows_scores(RowsSmem<NKS>& sm, RowsRaw<NKS, kFp8>& raw, u32x4 (&q)[NKS],
                                            const AttnRowsArgs& ra, const RowsStream& st, int wave) {
  constexpr int kD = NKS * 32;
  const AttnArgs& a = ra.a;
  const int lane = threadIdx.x % kWave, col = lane & 15, grp = lane >> 4;
  const int head = wave * 16 + col;  // within the group
  const float ninf = -__builtin_huge_valf();
  const float inv_sqrt_d = rsqrtf(static_cast<float>(a.D));
  const float inv_cap = a.softcap > 0.f ? 1.f / a.softcap : 0.f;
  const float cap_log2e = a.softcap * kLog2e;
  const float sink = ra.sink ? ra.sink[min(st.hg * kAtHeads + head, a.H - 1)] * kLog2e : ninf;
  // K operand (A): row col (and 16 more), chunk 4m + grp: the swizzle sees 4 (m % 2)
  // + grp, two m further is 64 elements on
  int koff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) koff[i] = col * kD + 8 * rows_chunk(col, 4 * i + grp);
  float m_run = ninf, l_run = 0.f;    // compressed: reference max (log2), this lane's part of the sum
  float m_win = ninf, f_win = 0.f;    // window: max, then the factor of its weights
  // a head's factor, exp2(m - mb) / denominator with the sink: 0 without a live key
  const auto factor = [&](float m, float l, float sink2) {
    const float mb = fmaxf(m, sink2);
    const float e = __builtin_amdgcn_exp2f(m - mb);
    const float den = e * l + (sink2 != ninf ? __builtin_amdgcn_exp2f(sink2 - mb) : 0.f);
    return m != ninf ? e / den : 0.f;
  };
  const auto times_w = [&]() {  // q * w: k_norm's weight, as in k_attn_part
    if (st.n_c == 0) return;
#pragma unroll
    for (int m = 0; m < NKS; ++m) {
      const float* wp = sm.w + m * 32 + grp * 8;  // zero past D
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        q[m][h] = bf16_pack2(__uint_as_float(q[m][h] << 16) * wp[2 * h], __uint_as_float(q[m][h] & 0xffff0000u) * wp[2 * h + 1]);
      }
    }
  };
  if (st.n_w == 0) times_w();
  for (int t = 0; t < st.n_w + st.n_c; ++t) {
    {
      const uint16_t* kt = sm.tile[t % 3];
      // operands are read kAheadK steps of 32 dims ahead of the products
      constexpr int kAheadK = 2;
      u32x4 kv[NKS][2];
      const auto read_k = [&](int m) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) kv[m][kb] = *reinterpret_cast<const u32x4*>(kt + koff[m & 1] + 64 * (m >> 1) + kb * 16 * kD);
      };
#pragma unroll
      for (int m = 0; m < kAheadK; ++m) read_k(m);
      f32x4 s[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int m = 0; m < NKS; ++m) {
        if (m + kAheadK < NKS) read_k(m + kAheadK);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(kv[m][kb]), as_bf16x8(q[m]), s[kb], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      // scores of keys 16kb + 4grp + i, head col, in the log2 domain
      float mx = ninf;
      const auto key4 = [&](const float* x, int kb) { return *reinterpret_cast<const f32x4*>(x + 16 * kb + 4 * grp); };
      if (t < st.n_w) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const f32x4 scale = key4(sm.scale[t % 3], kb), mask = key4(sm.mask[t % 3], kb);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const float v = s[kb][i];
            s[kb][i] = a.softcap > 0.f ? cap_log2e * tanhf(v * inv_sqrt_d * inv_cap) + mask[i] : fmaf(v, scale[i], mask[i]);
            mx = fmaxf(mx, s[kb][i]);
          }
          sm.sw[t][wave][kb][lane] = s[kb];
        }
        m_win = fmaxf(m_win, max_over_groups(mx));
        if (t == st.n_w - 1) {
          float l = 0.f;
          for (int u = 0; u < st.n_w; ++u) {  // this lane's own scores
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
              const f32x4 x = sm.sw[u][wave][kb][lane];
#pragma unroll
              for (int i = 0; i < 4; ++i) l += m_win == ninf ? 0.f : __builtin_amdgcn_exp2f(x[i] - m_win);
            }
          }
          f_win = factor(m_win, sum_over_groups(l), sink);
          times_w();
        }
      } else {
        f32x4 rk[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          const f32x4 scale = key4(sm.scale[t % 3], kb), mask = key4(sm.mask[t % 3], kb);
          rk[kb] = key4(sm.rms[t % 3], kb);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            s[kb][i] = fmaf(s[kb][i], scale[i], mask[i]);
            mx = fmaxf(mx, s[kb][i]);
          }
        }
        mx = max_over_groups(mx);
        // the reference max moves only when a tile's max passes it by more than
        // kRescaleAt (log2): O and the sum are rescaled rarely
        const bool move = mx > m_run + kRescaleAt;
        const float al = move ? __builtin_amdgcn_exp2f(m_run - mx) : 1.f;
        if (move) m_run = mx;
        const uint64_t any = __ballot(al != 1.f);
        if (lane < 16) sm.alpha[t & 1][head] = al;
        if (lane == 0) sm.moved[t & 1][wave] = any != 0;
        const bool none = m_run == ninf;
        float psum = 0.f;
        u32x4 pa;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          float p[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            p[i] = none ? 0.f : __builtin_amdgcn_exp2f(s[kb][i] - m_run);
            psum += p[i];
            p[i] *= rk[kb][i];
          }
          pa[2 * kb] = bf16_pack2(p[0], p[1]);
          pa[2 * kb + 1] = bf16_pack2(p[2], p[3]);
        }
        l_run = l_run * al + psum;
        sm.p[t & 1][wave][lane] = pa;
      }
    }
    rows_next(sm, raw, a, st, t);
  }
  {  // the compressed branch is complete
    const float f = factor(m_run, sum_over_groups(l_run), ra.sink_comp ? sink : ninf);
    if (lane < 16) sm.fin[head] = f;
  }
  // the window's output: P V with the final weights, all dims
  int voff[4];  // as in rows_output
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 4 * grp + (col >> 2);
    voff[i] = r * kD + 8 * rows_chunk(r, 2 * i + ((col & 3) >> 1)) + 4 * (col & 1);
  }
  constexpr int kBlocks = kD / 16;
  f32x4 acc[kBlocks];
#pragma unroll
  for (int x = 0; x < kBlocks; ++x) acc[x] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int t = st.n_w + st.n_c; t < st.turns(); ++t) {
    if (t < st.total()) {
      const int u = t - st.n_w - st.n_c;
      u32x4 pa;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        const f32x4 x = sm.sw[u][wave][kb][lane];  // this lane's own scores
        float p[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = f_win == 0.f ? 0.f : __builtin_amdgcn_exp2f(x[i] - m_win) * f_win;
        pa[2 * kb] = bf16_pack2(p[0], p[1]);
        pa[2 * kb + 1] = bf16_pack2(p[2], p[3]);
      }
      const uint16_t* vt = sm.tile[t % 3];
      constexpr int kAheadV = 3;
      u32x4 vv[kBlocks];
      const auto read_v = [&](int x) {
        const uint16_t* v = vt + voff[x & 3] + 64 * (x >> 2);
        const u32x2 lo = read_tr(v), hi = read_tr(v + 16 * kD);
        vv[x] = u32x4{lo[0], lo[1], hi[0], hi[1]};
      };
#pragma unroll
      for (int x = 0; x < kAheadV; ++x) read_v(x);
#pragma unroll
      for (int x = 0; x < kBlocks; ++x) {
        if (x + kAheadV < kBlocks) read_v(x + kAheadV);
        acc[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(pa), as_bf16x8(vv[x]), acc[x], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    rows_next(sm, raw, a, st, t);
  }
  u32x2* park = reinterpret_cast<u32x2*>(&sm.tile[0][0]);  // no tile is read any more
#pragma unroll
  for (int x = 0; x < kBlocks; ++x) {
    park[(x * 4 + wave) * kWave + lane] = u32x2{bf16_pack2(acc[x][0], acc[x][1]), bf16_pack2(acc[x][2], acc[x][3])};
  }
  lds_barrier();
}

// Waves 4-7: O of heads 32hh + 16hb + 4grp + i, dims kD/2 dh + 16s + col, and
// the row's output.
template <int NKS, bool kFp8>
__device__ __forceinline__ void rows_output(RowsSmem<NKS>& sm, RowsRaw<NKS, kFp8>& raw, const AttnRowsArgs& ra,
                                            const RowsStream& st, int wave) {
  constexpr int kD = NKS * 32, kBlocks = NKS;  // 16-dim blocks of half the dims
  const AttnArgs& a = ra.a;
  const int lane = threadIdx.x % kWave, col = lane & 15, grp = lane >> 4;
  const int hh = (wave >> 1) & 1, dh = wave & 1;
  // V operand (B), transposing reads: rows 4grp + col/4 (and 16 more), chunk 2X + (col %
  // 4) / 2 of 16-dim block X = dh * kBlocks + s: four X further is 64 elements on
  int voff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 4 * grp + (col >> 2);
    voff[i] = r * kD + 8 * rows_chunk(r, 2 * (dh * kBlocks + i) + ((col & 3) >> 1)) + 4 * (col & 1);
  }
  const int d0 = 16 * dh * kBlocks + col;
  f32x4 acc[2][kBlocks];
#pragma unroll
  for (int hb = 0; hb < 2; ++hb) {
#pragma unroll
    for (int s = 0; s < kBlocks; ++s) acc[hb][s] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // P V of tile u, whose weights the turn before wrote
  const auto add_tile = [&](int u) {
    const uint16_t* vt = sm.tile[u % 3];
    bf16x8 pa[2];
#pragma unroll
    for (int hb = 0; hb < 2; ++hb) pa[hb] = as_bf16x8(sm.p[u & 1][2 * hh + hb][lane]);
    constexpr int kAheadV = 3;
    u32x4 vv[kBlocks];
    const auto read_v = [&](int s) {
      const uint16_t* v = vt + voff[s & 3] + 64 * (s >> 2);
      const u32x2 lo = read_tr(v), hi = read_tr(v + 16 * kD);
      vv[s] = u32x4{lo[0], lo[1], hi[0], hi[1]};
    };
#pragma unroll
    for (int s = 0; s < kAheadV && s < kBlocks; ++s) read_v(s);
#pragma unroll
    for (int s = 0; s < kBlocks; ++s) {
      if (s + kAheadV < kBlocks) read_v(s + kAheadV);
#pragma unroll
      for (int hb = 0; hb < 2; ++hb) acc[hb][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pa[hb], as_bf16x8(vv[s]), acc[hb][s], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // turn t adds compressed tile t - 1
  int t = 0;
  for (; t <= st.n_w && t < st.turns(); ++t) rows_next(sm, raw, a, st, t);
  for (; t <= st.n_w + st.n_c; ++t) {
    const int u = t - 1;
    if (sm.moved[u & 1][2 * hh] | sm.moved[u & 1][2 * hh + 1]) {  // rescale O where a head's reference max moved
#pragma unroll
      for (int hb = 0; hb < 2; ++hb) {
        const f32x4 al = *reinterpret_cast<const f32x4*>(&sm.alpha[u & 1][hh * 32 + hb * 16 + 4 * grp]);
#pragma unroll
        for (int s = 0; s < kBlocks; ++s) acc[hb][s] *= al;
      }
    }
    add_tile(u);
    rows_next(sm, raw, a, st, t);
  }
  for (; t < st.turns(); ++t) rows_next(sm, raw, a, st, t);
  lds_barrier();  // the window's output is in LDS
  // O times its factor and w, plus the window's
  const u32x2* park = reinterpret_cast<const u32x2*>(&sm.tile[0][0]);
  const int hg0 = st.hg * kAtHeads, D = a.D;
  const bool full = hg0 + kAtHeads <= a.H && D == kD;  // uniform
#pragma unroll
  for (int hb = 0; hb < 2; ++hb) {
    const int h0 = hg0 + hh * 32 + hb * 16 + 4 * grp;
    float* out = ra.out + (static_cast<int64_t>(st.b) * a.H + h0) * D + d0;
    f32x4 f = f32x4{0.f, 0.f, 0.f, 0.f};
    if (st.n_c > 0) f = *reinterpret_cast<const f32x4*>(&sm.fin[hh * 32 + hb * 16 + 4 * grp]);
#pragma unroll
    for (int s = 0; s < kBlocks; ++s) {
      const u32x2 o = park[((dh * kBlocks + s) * 4 + 2 * hh + hb) * kWave + lane];
      const f32x4 w = f32x4{__uint_as_float(o[0] << 16), __uint_as_float(o[0] & 0xffff0000u), __uint_as_float(o[1] << 16),
                            __uint_as_float(o[1] & 0xffff0000u)};
      const float wd = sm.w[d0 + 16 * s];
      f32x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = (f[i] != 0.f ? acc[hb][s][i] * f[i] * wd : 0.f) + w[i];
      if (full) {
#pragma unroll
        for (int i = 0; i < 4; ++i) out[i * kD + 16 * s] = v[i];
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (h0 + i < a.H && d0 + 16 * s < D) out[i * D + 16 * s] = v[i];
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

template <int NKS, bool kFp8>
__global__ __launch_bounds__(kAtThreads, 2) void k_attn_rows(AttnRowsArgs ra) {
  __shared__ RowsSmem<NKS> sm;
  const AttnArgs& a = ra.a;
  const int tid = threadIdx.x;
  // Block i runs on XCD i % X: the XCD takes consecutive rows, whose windows
  // overlap (and picks, where neighbours pick alike), so its L2 holds them.
  const int xs = __builtin_ctz(static_cast<uint32_t>(a.xcds));
  const int n_blocks = a.batch * a.n_hg, per_xcd = (n_blocks + a.xcds - 1) >> xs;
  const int turn = static_cast<int>(blockIdx.x) >> xs;
  const int item = (static_cast<int>(blockIdx.x) & (a.xcds - 1)) * per_xcd + turn;
  if (turn >= per_xcd || item >= n_blocks) return;  // uniform
  RowsStream st;
  st.b = item / a.n_hg;
  st.hg = item - st.b * a.n_hg;
  // query row b is token t of sequence cb, position L - n_q + t of its L tokens
  st.cb = st.b / a.n_q;
  st.L = min(max(a.lens[st.cb] - (a.n_q - 1 - (st.b - st.cb * a.n_q)), 0), (1 << 24) - 1);
  st.n_win = min(st.L, a.window);
  st.n_comp = 0;
  int32_t pick0 = -1;
  const bool comp = a.kind != SKV_LAYER_SWA;  // uniform
  if (comp) {
    st.n_comp = a.kind == SKV_LAYER_CSA ? a.top_k
                                        : min(static_cast<int>(udiv24(max(st.L - 1, 0), a.m)), max(a.n_entries[st.cb], 0));
    // the first run's picks ahead of the query
    if (a.kind == SKV_LAYER_CSA && st.n_comp > 0) {
      pick0 = a.picks[static_cast<int64_t>(st.b) * a.pick_stride + min(tid, st.n_comp - 1)];
    }
  }
  const auto uniform = [](float x) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(x))); };
  st.inv_d = uniform(1.f / static_cast<float>(a.D));
  st.scale2 = uniform(rsqrtf(static_cast<float>(a.D)) * kLog2e);
  st.n_w = (st.n_win + kAtTile - 1) / kAtTile;
  st.n_c = (st.n_comp + kAtTile - 1) / kAtTile;
  for (int j = tid; j < st.n_w * kAtTile; j += kAtThreads) {
    sm.win_row[j] = j < st.n_win ? (static_cast<int64_t>(st.cb) * a.ring +
                                   static_cast<int>(umod24(st.L - st.n_win + j, a.ring))) * a.win_row : -1;
  }
  const int wave = __builtin_amdgcn_readfirstlane(tid) / kWave;
  const int lane = tid % kWave;
  // the scores' waves: query of head 16 wave + col, all dims, zero past H and D
  u32x4 q[NKS];
  if (wave < 4) {
    const int h = st.hg * kAtHeads + wave * 16 + (lane & 15);
    const uint8_t* qrow = a.q + (static_cast<int64_t>(st.b) * a.H + min(h, a.H - 1)) * a.D * 2;
#pragma unroll
    for (int m = 0; m < NKS; ++m) {
      const int d0 = m * 32 + (lane >> 4) * 8;
      q[m] = *reinterpret_cast<const u32x4*>((h < a.H && d0 < a.D) ? qrow + d0 * 2 : g_zero_row);
    }
  }
  RowsRaw<NKS, kFp8> raw;
  lds_barrier();
  // a window tile comes first: its loads go out before the compressed rows are resolved
  if (st.n_w > 0) rows_load(sm, raw, a, st, 0);
  if (comp) {
    for (int d = tid; d < NKS * 32; d += kAtThreads) sm.w[d] = d < a.D ? a.knorm_w[d] : 0.f;
    static_assert(kAtRun == kAtThreads, "one key of the first run per thread");
    rows_resolve(sm.row, a, st, 0, min(st.n_c * kAtTile, kAtRun), &pick0);
    lds_barrier();
  }
  if (st.n_w == 0 && st.total() > 0) rows_load(sm, raw, a, st, 0);
  if (st.total() > 0) rows_store(sm, raw, a, st, 0);
  if (st.total() > 1) rows_load(sm, raw, a, st, 1);
  lds_barrier();
  if (wave < 4) {
    rows_scores(sm, raw, q, ra, st, wave);
  } else {
    rows_output(sm, raw, ra, st, wave);
  }
}

}  // namespace skv
