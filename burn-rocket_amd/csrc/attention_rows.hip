// Grouped-query attention of few query rows (decode steps, short queries and
// chunks) on gfx950, with the keys split over waves and workgroups.
//
// attn_fa_kernel (attention.hip) gives a workgroup 128 query rows and walks the
// keys between barriers, with V transposed by a launch of its own first. With a
// few rows that is one long serial walk on a handful of CUs: what bounds the
// call is its latency. Here a workgroup takes up to 16·RT rows of one kv head
// (row r ↔ query r / G, head r % G of the group) and one of S key ranges; its RW
// waves (8; 4 for head dim 256) walk the range's 32-key chunks on their own (wave
// w chunks w, w + RW, ...), with no barrier until their softmax states meet in LDS. With
// S > 1 the states then meet in a workspace: the workgroup that arrives last
// merges all S, in split order whichever it is, and nothing waits on another.
//
// Per wave and chunk (v_mfma_f32_16x16x32_f16):
//   Sᵀ = K·Qᵀ   K rows straight from memory into the operand registers (each
//               is read by one wave), Q held in registers; a lane owns one
//               query row (lane % 16) and keys 4·(lane/16)+e of each 16-key block;
//   P           as in attn_fa_kernel: exp2 in f32, split into two fp16 values;
//   Oᵀ += Vᵀ·Pᵀ V copied as it lies ([key][d]) into a wave-private LDS buffer
//               and read back through ds_read_b64_tr_b16, which hands lane l the
//               four keys 4·(lane/16)+e of column d = l % 16: the operand order
//               of P's registers, so V needs no transposing launch.
// The next chunk's K loads and V copies are in flight while a chunk is
// computed. V chunks of a row whose width is a power of two are stored with
// 32-byte pairs swizzled by the key, so that the 16 rows of a transposing read
// fall on different banks.
#include <algorithm>

#include "attn_common.hpp"

// Lambdas called once per row tile: left to the inliner, their captures went to
// scratch memory with two row tiles.
#define ALWAYS_INLINE __attribute__((always_inline))

namespace {
constexpr int CK = 32;  // keys per chunk
constexpr int MAX_SPLITS = 16;
// Waves per workgroup: their two V buffers each, and the merge, fit in LDS.
__host__ __device__ constexpr int rows_waves(int d) { return d <= 128 ? 8 : 4; }

template <int D, int RT>
struct RowsGeom {
  static constexpr int RW = rows_waves(D);
  static constexpr int NQC = (D + 31) / 32;     // 32-wide d chunks of QKᵀ
  static constexpr int NDB = (D + 15) / 16;     // 16-row d blocks of Oᵀ
  static constexpr int CH = D / 8;              // 16-byte chunks per V row
  static constexpr int V_INS = (CK * CH + 63) / 64;  // 1 KB copies per V chunk
  static constexpr int V_BYTES = V_INS * 1024;
  static constexpr int KL = 2 * NQC;            // K loads per chunk
  static constexpr bool POW2 = (D & (D - 1)) == 0;
  static constexpr int SWZ = POW2 ? (CH / 2 < 8 ? CH / 2 : 8) - 1 : 0;  // pair swizzle mask
  static constexpr int T = RT * NDB;            // 16x16 Oᵀ tiles per wave
  static constexpr int MERGE_BYTES = RW * (T * 64 * 16 + RT * 16 * 8);
  static constexpr int SMEM = MERGE_BYTES > RW * 2 * V_BYTES ? MERGE_BYTES : RW * 2 * V_BYTES;
  // one split's state in the workspace: Oᵀ tiles, then (m, l) per row
  static constexpr int SLOT_BYTES = T * 64 * 16 + RT * 16 * 8;
  static_assert(SMEM <= 160 * 1024 && KL + V_INS <= 63, "geometry");
};

// Four fp16 values of column l % 16 from four consecutive 16-value rows, see
// the header; p: this lane's 8 bytes of row (l % 16) / 4.
typedef __fp16 fp16x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ half4 lds_read_tr(const uint8_t *p) {
  return __builtin_bit_cast(half4, __builtin_amdgcn_ds_read_tr16_b64_v4f16(
                                       (__attribute__((address_space(3))) fp16x4 *)(p)));
}
}  // namespace

template <int D, int RT>
__global__ __launch_bounds__(rows_waves(D) * 64, 2) void attn_rows_kernel(AttnArgs a, const f16 *__restrict__ v,
                                                               int64_t v_tok_stride, int64_t v_head_stride, int G,
                                                               int S) {
  using Gm = RowsGeom<D, RT>;
  constexpr int KBUF = D > 128 ? 1 : 2;  // K register sets (two of head dim 256 spill)
  constexpr int NQC = Gm::NQC, NDB = Gm::NDB, CH = Gm::CH, V_INS = Gm::V_INS, KL = Gm::KL, T = Gm::T;
  constexpr int RW = Gm::RW;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  // Splits fastest: the S workgroups of one row group sit on different XCDs
  // and so does each one's key range.
  const int sp = blockIdx.x % S, tile = blockIdx.x / S;
  const int kvh = tile % a.n_kv_heads, rg = tile / a.n_kv_heads;
  const int R = G * a.n_q, r0 = rg * 16 * RT;

  // ---- key range: the chunks that some row of the group sees, S shares of it
  const TileKeys tk = tile_keys<CK>(a, r0 / G, (min(r0 + 16 * RT, R) - 1) / G);
  const int n_ch = tk.kt_end - tk.kt_begin;
  const int c_begin = tk.kt_begin + (int)((int64_t)n_ch * sp / S);
  const int c_end = tk.kt_begin + (int)((int64_t)n_ch * (sp + 1) / S);

  // ---- this lane's rows
  bool rok[RT];
  int klo[RT], khi[RT];
  half8 qf[RT][NQC];
  f16 *orow[RT];
  static_for<RT>([&](auto t_c) ALWAYS_INLINE {
    constexpr int t = decltype(t_c)::value;
    const int r = r0 + 16 * t + l16;
    rok[t] = r < R;
    const int q = rok[t] ? r / G : 0, h = kvh * G + (rok[t] ? r % G : 0);
    int64_t lo, hi;
    vis_range(a.mask_mode, a.window, a.q0 + q, lo, hi);
    lo = max(lo - a.k0, (int64_t)0);
    hi = min(hi - a.k0, (int64_t)a.n_kv - 1);
    klo[t] = rok[t] ? (int)min(lo, (int64_t)a.n_kv) : a.n_kv;
    khi[t] = rok[t] ? (int)max(hi, (int64_t)-1) : -1;
    const f16 *qrow = (const f16 *)a.q + (int64_t)q * a.q_tok_stride + (int64_t)h * a.q_head_stride;
#pragma unroll
    for (int c = 0; c < NQC; ++c) {
      const int d0 = 32 * c + 8 * lg;
      qf[t][c] = (rok[t] && d0 < D) ? *(const half8 *)(qrow + d0) : half8{};
    }
    orow[t] = (f16 *)a.out + (int64_t)q * a.o_tok_stride + (int64_t)h * a.o_head_stride;
  });
  const float masked_x = tk.degenerate ? MASKED_SCORE * LOG2E : -INFINITY;
  const bool softcap = a.softcap != 0.f;
  const float C = softcap ? LOG2E : a.scale * LOG2E;

  // ---- K loads and V copies of a chunk: the whole offset of every access is
  // in its vector offset, so keys past n_kv (and head columns past D) fall past
  // the buffer's end and read as zeros.
  const rsrc_t rk = make_rsrc((const f16 *)a.k + (int64_t)kvh * a.k_head_stride,
                              ((int64_t)(a.n_kv - 1) * a.k_tok_stride + D) * 2);
  const rsrc_t rv = make_rsrc(v + (int64_t)kvh * v_head_stride, ((int64_t)(a.n_kv - 1) * v_tok_stride + D) * 2);
  const uint32_t ks = (uint32_t)(a.k_tok_stride * 2), vs = (uint32_t)(v_tok_stride * 2);
  const uint32_t k_lane = (uint32_t)l16 * ks + (uint32_t)(lg * 16);
  uint8_t *const vbuf = smem + wave * (2 * Gm::V_BYTES);
  auto load_k = [&](half8(&kf)[2][NQC], int c) ALWAYS_INLINE {
    const uint32_t base = (uint32_t)c * (CK * ks) + k_lane;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
      for (int cc = 0; cc < NQC; ++cc) {
        const uint32_t off = 32 * cc + 8 * lg < D ? base + (uint32_t)(kb * 16) * ks + 64 * cc : OOB_OFFSET;
        kf[kb][cc] = __builtin_bit_cast(half8, __builtin_amdgcn_raw_buffer_load_b128(rk, off, 0, 0));
      }
  };
  auto copy_v = [&](int buf, int c) ALWAYS_INLINE {
#pragma unroll
    for (int i = 0; i < V_INS; ++i) {
      const int p = 64 * i + lane, row = p / CH, ch = p % CH;
      const int lch = Gm::SWZ ? ch ^ ((row & Gm::SWZ) << 1) : ch;  // logical chunk of this slot
      const uint32_t off = row < CK ? (uint32_t)(c * CK + row) * vs + (uint32_t)(lch * 16) : OOB_OFFSET;
      bdma16(rv, vbuf + buf * Gm::V_BYTES + i * 1024, off, 0);
    }
  };
  // Transposing reads: this lane's 8 bytes of key 4·lg + l16/4 (+ 16 per key
  // block), columns 16·db + 4·(l16%4)..; the swizzle moves 32-byte pairs.
  const int vkey = 4 * lg + (l16 >> 2);
  const uint32_t v_row = (uint32_t)(vkey * (D * 2) + (l16 & 3) * 8);
  const int vsw = vkey & Gm::SWZ;  // (16 keys on: the same swizzle, SWZ <= 7)

  floatx4 o[RT][NDB];
  float m_run[RT], l_run[RT];
  static_for<RT>([&](auto t_c) ALWAYS_INLINE {
    constexpr int t = decltype(t_c)::value;
    m_run[t] = -INFINITY;
    l_run[t] = 0.f;
#pragma unroll
    for (int db = 0; db < NDB; ++db) o[t][db] = floatx4{0.f, 0.f, 0.f, 0.f};
  });

  floatx4 s[RT][2];  // the chunk's scores
  auto scores = [&](const half8(&kf)[2][NQC]) ALWAYS_INLINE {
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        s[t][kb] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int cc = 0; cc < NQC; ++cc)
          s[t][kb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[kb][cc], qf[t][cc], s[t][kb], 0, 0, 0);
      }
  };
  auto softmax_pv = [&](int buf, int c) ALWAYS_INLINE {
    if (softcap) {
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int e = 0; e < 4; ++e) s[t][kb][e] = a.softcap * tanhf(s[t][kb][e] * a.scale / a.softcap);
    }
    const int kb0 = c * CK;
    half8 phi[RT], plo[RT];
    static_for<RT>([&](auto t_c) ALWAYS_INLINE {
      constexpr int t = decltype(t_c)::value;
      float x[8], mt = -INFINITY;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int key = kb0 + 16 * (i >> 2) + 4 * lg + (i & 3);
        // scaled first: a masked score is the masked value itself
        const float sc = s[t][i >> 2][i & 3] * C;
        x[i] = key >= a.n_kv ? -INFINITY : (key < klo[t] || key > khi[t]) ? masked_x : sc;
        mt = fmaxf(mt, x[i]);
      }
      mt = max4groups(mt);
      const float m_new = fmaxf(m_run[t], mt);
      const float mu = m_new == -INFINITY ? 0.f : m_new;
      if (__builtin_amdgcn_ballot_w64(m_new > m_run[t]) != 0) {
        const float alpha = __builtin_amdgcn_exp2f(m_run[t] - mu);
        l_run[t] *= alpha;
#pragma unroll
        for (int db = 0; db < NDB; ++db) o[t][db] *= alpha;
      }
      m_run[t] = m_new;
      uintx4 hw, lw;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e0 = __builtin_amdgcn_exp2f(x[2 * i] - mu), e1 = __builtin_amdgcn_exp2f(x[2 * i + 1] - mu);
        l_run[t] += e0 + e1;
        const unsigned int h = __builtin_bit_cast(unsigned int, __builtin_amdgcn_cvt_pkrtz(e0, e1));
        hw[i] = h;
        lw[i] = __builtin_bit_cast(unsigned int,
                                   __builtin_amdgcn_cvt_pkrtz(minus_half_lo(h, e0), minus_half_hi(h, e1)));
      }
      phi[t] = __builtin_bit_cast(half8, hw);
      plo[t] = __builtin_bit_cast(half8, lw);
    });
    const uint8_t *vb = vbuf + buf * Gm::V_BYTES + v_row;
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      const uint8_t *p = vb + ((db ^ vsw) << 5);
      const half4 a0 = lds_read_tr(p), a1 = lds_read_tr(p + 16 * D * 2);
      const half8 vf = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
      static_for<RT>([&](auto t_c) ALWAYS_INLINE {
        constexpr int t = decltype(t_c)::value;
        o[t][db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, phi[t], o[t][db], 0, 0, 0);
        o[t][db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf, plo[t], o[t][db], 0, 0, 0);
      });
    }
  };

  // ---- the wave's chunks c_begin + wave, + RW, ...
  half8 kf[KBUF][2][NQC];
  int c = c_begin + wave;
  auto step = [&](auto cur_c) ALWAYS_INLINE {
    constexpr int CUR = decltype(cur_c)::value;
    const bool more = c + RW < c_end;
    if constexpr (KBUF == 2) {
      if (more) {
        load_k(kf[CUR ^ 1], c + RW);
        copy_v(CUR ^ 1, c + RW);
        asm volatile("" ::: "memory");
        WAIT_VMCNT(KL + V_INS);  // this chunk's have landed
      } else {
        WAIT_VMCNT(0);
      }
      asm volatile("" ::: "memory");
      scores(kf[CUR]);
    } else {  // one K register set: refilled once the scores are formed
      WAIT_VMCNT(0);
      asm volatile("" ::: "memory");
      if (more) copy_v(CUR ^ 1, c + RW);
      scores(kf[0]);
      if (more) load_k(kf[0], c + RW);
    }
    softmax_pv(CUR, c);
    WAIT_LGKMCNT0();  // the V buffer's reads are done before it is refilled
    asm volatile("" ::: "memory");
    c += RW;
  };
  if (c < c_end) {
    load_k(kf[0], c);
    copy_v(0, c);
    while (true) {
      step(ic<0>{});
      if (c >= c_end) break;
      step(ic<1>{});
      if (c >= c_end) break;
    }
  }

  // ---- the waves' states meet in LDS: (m, l) per row, Oᵀ per lane
  __syncthreads();  // the V buffers are free
  floatx4 *x_o = (floatx4 *)smem;                       // [wave][tile][lane]
  float2 *x_ml = (float2 *)(smem + RW * T * 64 * 16);   // [wave][RT·16]
  static_for<RT>([&](auto t_c) ALWAYS_INLINE {
    constexpr int t = decltype(t_c)::value;
    const float l = sum4groups(l_run[t]);
    if (lg == 0) x_ml[wave * (RT * 16) + t * 16 + l16] = make_float2(m_run[t], l);
#pragma unroll
    for (int db = 0; db < NDB; ++db) x_o[(wave * T + t * NDB + db) * 64 + lane] = o[t][db];
  });
  __syncthreads();
  // wave w merges tiles w, w + RW, ...
  constexpr int SC1 = 16;  // cache policy bit: device scope
  const rsrc_t rp = make_rsrc((const uint8_t *)a.part + (S > 1 ? (size_t)tile * S * Gm::SLOT_BYTES : 0),
                              S > 1 ? (int64_t)S * Gm::SLOT_BYTES : 0);
  const uint32_t mine = (uint32_t)sp * Gm::SLOT_BYTES;
  float wa[RT][RW], m_all[RT], l_all[RT];
  static_for<RT>([&](auto t_c) ALWAYS_INLINE {
    constexpr int t = decltype(t_c)::value;
    float2 ml[RW];
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int w = 0; w < RW; ++w) {
      ml[w] = x_ml[w * (RT * 16) + t * 16 + l16];
      m = fmaxf(m, ml[w].x);
    }
    const float mu = m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int w = 0; w < RW; ++w) {
      wa[t][w] = __builtin_amdgcn_exp2f(ml[w].x - mu);
      l += ml[w].y * wa[t][w];
    }
    m_all[t] = m;
    l_all[t] = l;
  });
  auto store_o = [&](auto t_c, int db, floatx4 ov, float inv) ALWAYS_INLINE {
    constexpr int t = decltype(t_c)::value;
    const int d0 = db * 16 + 4 * lg;
    if (rok[t] && d0 < D) *(half4 *)(orow[t] + d0) = half4{(f16)(ov[0] * inv), (f16)(ov[1] * inv),
                                                          (f16)(ov[2] * inv), (f16)(ov[3] * inv)};
  };
  // Tile u = t·NDB + db of this wave: f(t, db, u), t known at compile time.
  auto my_tiles = [&](auto &&f) ALWAYS_INLINE {
    static_for<RT>([&](auto t_c) ALWAYS_INLINE {
      constexpr int t = decltype(t_c)::value;
      for (int db = wave; db < NDB; db += RW) f(t_c, db, t * NDB + db);
    });
  };
  my_tiles([&](auto t_c, int db, int u) ALWAYS_INLINE {
    constexpr int t = decltype(t_c)::value;
    floatx4 ov = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < RW; ++w) ov += x_o[(w * T + u) * 64 + lane] * wa[t][w];
    if (S > 1)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uintx4, ov), rp,
                                             rok[t] ? mine + (uint32_t)((u * 64 + lane) * 16) : OOB_OFFSET, 0, SC1);
    else
      store_o(t_c, db, ov, l_all[t] > 0.f ? 1.0f / l_all[t] : 0.f);
  });
  if (S == 1) return;
  if (wave == 0 && lg == 0) {
    static_for<RT>([&](auto t_c) ALWAYS_INLINE {
      constexpr int t = decltype(t_c)::value;
      const uintx2 w = {__float_as_uint(m_all[t]), __float_as_uint(l_all[t])};
      __builtin_amdgcn_raw_buffer_store_b64(w, rp, mine + (uint32_t)(T * 1024 + (t * 16 + l16) * 8), 0, SC1);
    });
  }
  WAIT_VMCNT(0);  // the state is stored before the arrival count
  __syncthreads();
  unsigned *flag = (unsigned *)smem;
  if (threadIdx.x == 0) {
    const unsigned prev = atomicAdd(a.cnt + tile, 1u);
    const unsigned last = prev == (unsigned)(S - 1);
    if (last) atomicExch(a.cnt + tile, 0u);  // every split is in: reset for the next launch
    *flag = last;
  }
  __syncthreads();
  if (!*flag) return;
  // One pass over the splits, in split order; the launch has at most MAX_SPLITS
  // of them, so that all loads are in flight together (each is a trip to memory).
  my_tiles([&](auto t_c, int db, int u) ALWAYS_INLINE {
    constexpr int t = decltype(t_c)::value;
    floatx4 x[MAX_SPLITS];
    uintx2 ml[MAX_SPLITS];
#pragma unroll
    for (int i = 0; i < MAX_SPLITS; ++i) {
      const uint32_t slot = rok[t] && i < S ? (uint32_t)i * Gm::SLOT_BYTES : OOB_OFFSET;  // past the end: zeros
      x[i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(
                                             rp, slot + (uint32_t)((u * 64 + lane) * 16), 0, SC1));
      ml[i] = __builtin_amdgcn_raw_buffer_load_b64(rp, slot + (uint32_t)(T * 1024 + (t * 16 + l16) * 8), 0, SC1);
    }
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int i = 0; i < MAX_SPLITS; ++i) m = fmaxf(m, i < S ? __uint_as_float(ml[i][0]) : -INFINITY);
    const float mu = m == -INFINITY ? 0.f : m;
    floatx4 ov = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < MAX_SPLITS; ++i) {
      const float w = i < S ? __builtin_amdgcn_exp2f(__uint_as_float(ml[i][0]) - mu) : 0.f;
      l += __uint_as_float(ml[i][1]) * w;
      ov += x[i] * w;
    }
    store_o(t_c, db, ov, l > 0.f ? 1.0f / l : 0.f);
  });
}

namespace {
// Rows per workgroup and the key split of a launch.
struct RowsPlan {
  int rt, tiles, splits;
};
// One row tile of 16 per workgroup while that leaves few workgroups or few
// keys: more workgroups then share the reads of K and V (16 query / 8 kv heads
// of 128 against 4096 keys, MI355X: 16 queries 13.4 us with one tile, 16.7 with
// two; 128 queries 28.0 against 24.3). Keys are split as far as each wave keeps
// one chunk and the launch fills the CUs once.
RowsPlan rows_plan(const AttnArgs &a) {
  const int G = a.n_head / a.n_kv_heads;
  const int64_t R = (int64_t)G * a.n_q;
  // Keys that a row tile can see. Causal counts them all, also where q0 leaves the
  // first queries fewer: their last ranges are empty then and merge with weight 0.
  int64_t keys = a.n_kv;
  if (a.mask_mode == RK_MASK_WINDOW) keys = std::min<int64_t>(keys, 2 * std::min<int64_t>(a.window, keys) + a.n_q);
  if (a.mask_mode == RK_MASK_CAUSAL_WINDOW) keys = std::min<int64_t>(keys, std::min<int64_t>(a.window, keys) + a.n_q);
  const int64_t chunks = (std::max<int64_t>(keys, 1) + CK - 1) / CK;
  const int64_t tiles1 = (R + 15) / 16 * a.n_kv_heads;
  RowsPlan p;
  p.rt = a.head_dim <= 128 && tiles1 >= 128 && tiles1 * chunks > 14000 ? 2 : 1;
  p.tiles = (int)((R + 16 * p.rt - 1) / (16 * p.rt)) * a.n_kv_heads;
  const int cus = a.num_cus > 0 ? a.num_cus : 256, RW = rows_waves(a.head_dim);
  const int64_t by_work = (chunks + RW - 1) / RW, by_cus = std::max(1, cus / p.tiles);
  p.splits = (int)std::min({by_work, by_cus, (int64_t)MAX_SPLITS});
  return p;
}

template <int D, int RT>
hipError_t launch_rows(const AttnArgs &a, const void *v, int64_t v_ts, int64_t v_hs, const RowsPlan &p,
                       hipStream_t st) {
  using Gm = RowsGeom<D, RT>;
  auto kern = attn_rows_kernel<D, RT>;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, Gm::SMEM);
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)(p.tiles * p.splits)), dim3(Gm::RW * 64), Gm::SMEM, st, a, (const f16 *)v, v_ts,
                     v_hs, a.n_head / a.n_kv_heads, p.splits);
  return hipGetLastError();
}

template <int D>
hipError_t launch_rows_d(const AttnArgs &a, const void *v, int64_t v_ts, int64_t v_hs, const RowsPlan &p,
                         hipStream_t st) {
  if constexpr (D <= 128)
    if (p.rt == 2) return launch_rows<D, 2>(a, v, v_ts, v_hs, p, st);
  return launch_rows<D, 1>(a, v, v_ts, v_hs, p, st);
}
}  // namespace

// By the number of 16-row tiles against the CUs: past two rounds (half a round
// for head dim 256) each tile's own read of K and V costs more than the 128-row
// kernel's serial walk. MI355X, causal, 4096 keys, the call with Vᵀ on
// attn_fa_kernel -> here: 32/4 heads of 128, 1 query 45.2 -> 10.0 us, 64 queries
// 47.1 -> 24, 256 queries (512 tiles) 48.4 -> 47.7, 512 queries 54 -> 89;
// 16/16 heads of 72, 1 query 42.5 -> 10.6, 512 queries (512 tiles) 46.5 -> 32.8,
// 1024 queries 48 -> 60; 3/1 heads of 256, 1 query 57 -> 16.1, 512 queries (96
// tiles) 61.9 -> 44.8, 1024 queries (192 tiles) 62 -> 75. A tile height or split
// forced by RK_ATTN_ROWS / RK_ATTN_SPLIT / RK_ATTN_SPLIT_TILES keeps
// attn_fa_kernel; RK_ATTN_FEW=0 turns this kernel off.
bool rk_attn_rows_fits(const AttnArgs &a, const void *v, int64_t v_tok_stride) {
  if (a.n_kv_heads <= 0 || a.n_head % a.n_kv_heads) return false;
  if (rk_knob("RK_ATTN_FEW", 1) == 0 || rk_knob("RK_ATTN_SPLIT", 0) != 0 || rk_knob("RK_ATTN_ROWS", 0) != 0 ||
      rk_knob("RK_ATTN_SPLIT_TILES", -1) >= 0)
    return false;
  // V is copied to LDS in 16-byte pieces, which attn_fa_kernel's own transposing
  // launch does not need to be aligned.
  if (((uintptr_t)v & 15) != 0 || v_tok_stride % 8 != 0) return false;
  // K and V of one kv head are addressed with 32-bit byte offsets.
  const int64_t reach = (int64_t)1 << 31, keys = (int64_t)a.n_kv + CK;
  if (keys * a.k_tok_stride * 2 >= reach || keys * v_tok_stride * 2 >= reach) return false;
  const int64_t tiles = ((int64_t)a.n_head / a.n_kv_heads * a.n_q + 15) / 16 * a.n_kv_heads;
  const int64_t cus = a.num_cus > 0 ? a.num_cus : 256;
  return a.head_dim > 128 ? 2 * tiles <= cus : tiles <= 2 * cus;
}

void rk_attn_rows_workspace(const AttnArgs &a, size_t *part_bytes, size_t *n_cnt) {
  const RowsPlan p = rows_plan(a);
  *part_bytes = *n_cnt = 0;
  if (p.splits <= 1) return;
  const size_t t = (size_t)p.rt * ((a.head_dim + 15) / 16);
  *part_bytes = (size_t)p.tiles * p.splits * (t * 1024 + (size_t)p.rt * 128);
  *n_cnt = (size_t)p.tiles;
}

hipError_t rk_launch_attention_rows(const AttnArgs &a, const void *v, int64_t v_ts, int64_t v_hs, hipStream_t st) {
  const RowsPlan p = rows_plan(a);
  if (p.splits > 1 && (!a.part || !a.cnt)) return hipErrorInvalidValue;
  switch (a.head_dim) {
    case 32: return launch_rows_d<32>(a, v, v_ts, v_hs, p, st);
    case 48: return launch_rows_d<48>(a, v, v_ts, v_hs, p, st);
    case 64: return launch_rows_d<64>(a, v, v_ts, v_hs, p, st);
    case 72: return launch_rows_d<72>(a, v, v_ts, v_hs, p, st);
    case 80: return launch_rows_d<80>(a, v, v_ts, v_hs, p, st);
    case 96: return launch_rows_d<96>(a, v, v_ts, v_hs, p, st);
    case 112: return launch_rows_d<112>(a, v, v_ts, v_hs, p, st);
    case 128: return launch_rows_d<128>(a, v, v_ts, v_hs, p, st);
    case 256: return launch_rows_d<256>(a, v, v_ts, v_hs, p, st);
  }
  return hipErrorInvalidValue;
}
