// GEMMs with few output tiles (decode steps, search queries, short batches) on
// gfx950: int8 with one scale per weight group, and fp16.
//
// What bounds these is latency, not bytes: the tiled kernels walk K stage by
// stage in each workgroup, with a barrier and an LDS round trip per stage, on
// a grid of a few dozen workgroups. Measured on MI355X (us per call, tiled
// kernel -> here):
//   int8 per token   12 rows, 1024->3072 8.7 -> 4.1;  3072->1024 19.8 -> 4.9;
//                    256 rows, 1024->3072 9.3 -> 7.0; 3072->1024 20.5 -> 7.9
//   int8 group 32    12 rows, 1024->3072 11.2 -> 4.4; 256 rows, 3072->1024 28.5 -> 8.8
//   fp16             1 row, 1024->3072 5.4 -> 3.4;    64 rows, 1024->1024 5.8 -> 3.9
#include "common.hpp"
#include "glu.hpp"
#include "kernels.hpp"

namespace {
constexpr int SNW = 8;  // waves per workgroup, the K split

__device__ __forceinline__ float glu_any(int glu, float g, float u) {
  return glu == GLU_SILU ? glu_apply<GLU_SILU>(g, u) : glu_apply<GLU_GELU>(g, u);
}
}  // namespace

// int8: C[m, n] = Σ_g (as[m, g]·)ws[n, g]·P_g (times as[m] per token), P_g the
// exact int32 product of a group of GB 32-value blocks, folded in ascending g
// with the formulas of gemm_i8_q8_kernel (fold, fold_group): the results are that
// kernel's bit for bit, so neither the number of rows nor a fused form changes a
// row's sums. Only the integer products are split over the waves: in a round of 8
// stages (128 K-values each) wave w forms stage w's products of the 16 x 16·TN
// tile (v_mfma_i32_16x16x32_i8, one block each) and hands them on through LDS,
// [element][stage][block or group]; then a thread per element folds the round's
// products in order. A stage is copied by its wave into an LDS slot of its own,
// whole 128-byte lines at a time, and refilled for the next round as soon as it
// is read. Tried for 3072->1024 at 12 rows, 4.9 us here: operands straight into
// registers, a wave per tile (9.1); four waves on a 32x32 tile with a barrier per
// stage (11.9); fold waves of their own (no gain).
namespace {
template <bool GROUPED, int GB, int TN>
struct SkinnyI8Geom {
  static constexpr int PB = TN == 1 ? 2 : 1;  // product buffers: two save a barrier per round
  // Codes of 16 rows or columns, and 64 bytes that keep the compiler from pairing
  // the reads of two tiles in one instruction: on the same banks, the pair would
  // take twice its time.
  static constexpr int TILE = 2048 + 64;
  static constexpr int SLOT = (1 + TN) * TILE;                   // a stage's codes: 16 rows, 16·TN columns
  static constexpr int SC = TN * 256 + (GROUPED ? 256 : 0);      // its scales, [column][4], [row][4]
  static constexpr int NS = 3;  // scale slots: a round's are folded while the next one's land
  // an element's products of a round, and 16 bytes that spread them over the banks
  static constexpr int PST = SNW * (4 / GB) * 4 + 16;
  static constexpr int P = TN * 256 * PST;
  static constexpr int SMEM = SNW * (SLOT + NS * SC) + PB * P;
  static_assert(SMEM <= 160 * 1024, "LDS");
};

template <bool GROUPED>
struct WaveI8Geom {
  static constexpr int ST = 2;
  // a stage: rows [16][128], column scales [16][4], columns (apart from the rows, as
  // above), row scales [group][16]
  static constexpr int WS_OFF = 2048, W_OFF = WS_OFF + 256, AS_OFF = W_OFF + 2048;
  static constexpr int SLOT = AS_OFF + (GROUPED ? 256 : 0);
  static constexpr int SMEM = 4 * ST * SLOT;
};
}  // namespace

template <bool GROUPED, bool WSF16, int GB, int TN, int GLU, bool OUT_F16>
__global__ __launch_bounds__(SNW * 64, 2) void skinny_i8_kernel(
    const int8_t *__restrict__ A, const float *__restrict__ AS, int as_stride, const int8_t *__restrict__ W,
    const float *__restrict__ WS, int ws_stride, void *__restrict__ C, int M, int N, int K, int tiles_m, int n_out) {
  using G = SkinnyI8Geom<GROUPED, GB, TN>;
  constexpr int GPS = 4 / GB;  // groups per stage
  static_assert(TN <= 2 && (!WSF16 || (GROUPED && GB == 1)) && (GLU == GLU_NONE || (TN == 2 && !GROUPED)), "form");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  // Row tiles fastest: the workgroups that read the same weights share an XCD.
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int m0 = id % tiles_m * 16, n0 = id / tiles_m * (16 * TN);
  const int rows = min(M - m0, 16), cols = min(N - n0, 16 * TN);
  const int KT = (K + 127) / 128, KB = K / 32;
  uint8_t *const slot = smem + wave * G::SLOT;
  uint8_t *const s_scale = smem + SNW * G::SLOT;  // [wave][NS]
  uint8_t *const s_p = s_scale + SNW * G::NS * G::SC;

  // Rows past M and N, and chunks past K, read as zeros (offsets past the end
  // of the buffers).
  const rsrc_t ra = make_rsrc(A + (size_t)m0 * K, (int64_t)rows * K);
  const rsrc_t rw = make_rsrc(W + (size_t)n0 * K, (int64_t)cols * K);
  const rsrc_t rs = make_rsrc(WS + (size_t)n0 * ws_stride, (int64_t)cols * ws_stride * 4);
  const rsrc_t ras = make_rsrc(AS + (size_t)m0 * as_stride, (int64_t)rows * as_stride * 4);
  // Copy q covers rows 8q..8q+7: lane → row 8q + lane/8, physical chunk lane%8,
  // which holds logical chunk (lane%8) ^ ((row >> 1) & 7), as in gemm_i8_q8_kernel.
  const int r8 = lane >> 3, p8 = lane & 7;
  const int ch[2] = {p8 ^ (r8 >> 1), p8 ^ (4 + (r8 >> 1))};  // q even, odd
  const uint32_t v_q[2] = {(uint32_t)(r8 * K + ch[0] * 16), (uint32_t)((8 + r8) * K + ch[1] * 16)};
  // scale copies: lane → row lane/4, block or group lane%4 of the stage
  const uint32_t v_ws = (uint32_t)(((lane >> 2) * ws_stride + (lane & 3)) * 4);
  const uint32_t v_as = (uint32_t)(((lane >> 2) * as_stride + (lane & 3)) * 4);
  auto issue = [&](int kt) {  // kt < KT
    uint8_t *sc = s_scale + (wave * G::NS + kt / SNW % G::NS) * G::SC;
    const uint32_t k0 = kt * 128;
    uint32_t v[2];
#pragma unroll
    for (int o = 0; o < 2; ++o) v[o] = (int)k0 + ch[o] * 16 < K ? v_q[o] : OOB_OFFSET;
#pragma unroll
    for (int q = 0; q < 2; ++q) bdma16(ra, slot + q * 1024, v[q], k0);
#pragma unroll
    for (int q = 0; q < 2 * TN; ++q) bdma16(rw, slot + (1 + (q >> 1)) * G::TILE + (q & 1) * 1024, v[q & 1], (q >> 1) * 16 * K + k0);
#pragma unroll
    for (int j = 0; j < TN; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, LDS_PTR(sc + j * 256), 4, v_ws,
                                               (uint32_t)(j * 16 * ws_stride * 4 + kt * 16), 0, 0);
    if constexpr (GROUPED)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          ras, LDS_PTR(sc + TN * 256), 4, (lane & 3) < GPS && kt * 4 + (lane & 3) * GB < KB ? v_as : OOB_OFFSET,
          (uint32_t)(kt * GPS * 4), 0, 0);
  };

  uint32_t f_off[4];  // the lane's 8 bytes of block b of its row
#pragma unroll
  for (int b = 0; b < 4; ++b)
    f_off[b] = (uint32_t)(l16 * 128 + (((2 * b + (lg >> 1)) ^ (l16 >> 1)) << 4) + (lg & 1) * 8);
  constexpr int GBIAS_BITS = 0x4B400000;  // 1.5·2^23, see gemm_i8_q8_kernel
  constexpr float GBIAS = 12582912.0f;
  constexpr int INIT = WSF16 ? GBIAS_BITS : 0;
  typedef int PV __attribute__((ext_vector_type(GPS)));
  // Stage kt's products: a lane has rows 4·lg + e of column l16 of each tile.
  auto produce = [&](int kt, uint8_t *pbuf) {
    WAIT_VMCNT(0);  // the stage has landed
    asm volatile("" ::: "memory");
    long a[4], w[TN][4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      a[b] = *(const long *)(slot + f_off[b]);
#pragma unroll
      for (int j = 0; j < TN; ++j) w[j][b] = *(const long *)(slot + (1 + j) * G::TILE + f_off[b]);
    }
    WAIT_LGKMCNT0();  // the slot is read: refilled while the products are formed
    asm volatile("" ::: "memory");
    if (kt + SNW < KT) issue(kt + SNW);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      intx4 p[GPS];
#pragma unroll
      for (int g = 0; g < GPS; ++g) {
        p[g] = intx4{INIT, INIT, INIT, INIT};
#pragma unroll
        for (int b = 0; b < GB; ++b)
          p[g] = __builtin_amdgcn_mfma_i32_16x16x32_i8(a[g * GB + b], w[j][g * GB + b], p[g], 0, 0, 0);
      }
      uint8_t *o = pbuf + (j * 256 + lg * 64 + l16) * G::PST + wave * (GPS * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        PV x;
#pragma unroll
        for (int g = 0; g < GPS; ++g) x[g] = p[g][e];
        *(PV *)(o + e * 16 * G::PST) = x;
      }
    }
  };

  // The thread's element: row f_row, column l16 of tile f_j.
  const bool folds = threadIdx.x < TN * 256;
  const int f_j = threadIdx.x >> 8, f_row = (threadIdx.x >> 4) & 15, m = m0 + f_row;
  float acc = 0.f;
  auto fold = [&](int p, float d, float as) {
    if constexpr (WSF16)
      acc = __builtin_fmaf(__builtin_fmaf(__int_as_float(p), d, -GBIAS * d), as, acc);
    else
      acc = __builtin_fmaf((float)p, GROUPED ? as * d : d, acc);
  };
  auto fold_round = [&](int r, const uint8_t *pbuf, auto whole_c) {
    const uint8_t *pp = pbuf + threadIdx.x * G::PST, *sc = s_scale + r % G::NS * G::SC;
    intx4 p[2 * GPS];  // [stage][group]; of stages past K whatever LDS holds, not folded
    floatx4 d[SNW], as[GROUPED ? SNW : 1];
#pragma unroll
    for (int q = 0; q < 2 * GPS; ++q) p[q] = *(const intx4 *)(pp + q * 16);
#pragma unroll
    for (int s = 0; s < SNW; ++s) {
      d[s] = *(const floatx4 *)(sc + s * (G::NS * G::SC) + f_j * 256 + l16 * 16);
      if constexpr (GROUPED) as[s] = *(const floatx4 *)(sc + s * (G::NS * G::SC) + TN * 256 + f_row * 16);
    }
#pragma unroll
    for (int s = 0; s < SNW; ++s)
#pragma unroll
      for (int g = 0; g < GPS; ++g) {
        if (!decltype(whole_c)::value && (r * SNW + s) * 4 + g * GB >= KB) return;
        fold(p[(s * GPS + g) / 4][(s * GPS + g) % 4], d[s][g * GB], as[GROUPED ? s : 0][g]);
      }
  };

  // A wave refills its slot and the next round's scales while others may still
  // fold this round or, with two product buffers, the one before: three scale
  // slots keep all of them apart.
  if (wave < KT) issue(wave);
  const float as_m = GROUPED || !folds ? 1.f : AS[(size_t)min(m, M - 1) * as_stride];
  for (int r = 0; r * SNW < KT; ++r) {
    uint8_t *const pbuf = s_p + (G::PB == 2 ? (r & 1) * G::P : 0);
    const int kt = r * SNW + wave;
    if (kt < KT) produce(kt, pbuf);
    WAIT_LGKMCNT0();
    BARRIER();  // the round's products and scales are in LDS
    if (folds) {
      if (4 * (r + 1) * SNW <= KB)
        fold_round(r, pbuf, std::true_type{});
      else
        fold_round(r, pbuf, std::false_type{});
    }
    if (G::PB == 1) {
      WAIT_LGKMCNT0();
      BARRIER();  // the products are read
    }
  }

  // (a per-token fp16 result is as·acc rounded once, as the compiler forms it in
  // gemm_i8_q8_kernel: v_fma_mixlo_f16)
  auto store = [&](int n, int ld, float y) {
    if (m < M && n < ld) {
      if constexpr (OUT_F16)
        ((f16 *)C)[(size_t)m * ld + n] = (f16)y;
      else
        ((float *)C)[(size_t)m * ld + n] = y;
    }
  };
  if constexpr (GLU != GLU_NONE) {  // tile 0: 16 gate columns, tile 1: the 16 up columns
    float *x = (float *)smem;       // (over the slots: every copy was waited for and read)
    if (f_j == 1) x[threadIdx.x & 255] = as_m * acc;
    __syncthreads();
    if (f_j == 0) store(n0 / 2 + l16, n_out, glu_apply<GLU>(as_m * acc, x[threadIdx.x]));
  } else if (folds) {
    if constexpr (GROUPED)
      store(n0 + f_j * 16 + l16, N, acc);
    else
      store(n0 + f_j * 16 + l16, N, as_m * acc);
  }
}

template <bool GROUPED, bool WSF16, int GB, int TN, int GLU, bool OUT_F16>
static hipError_t launch_skinny_i8_tn(const I8GemmArgs &g, hipStream_t st) {
  auto kern = skinny_i8_kernel<GROUPED, WSF16, GB, TN, GLU, OUT_F16>;
  constexpr int smem = SkinnyI8Geom<GROUPED, GB, TN>::SMEM;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  const int tm = (g.M + 15) / 16, tn = (g.N + 16 * TN - 1) / (16 * TN);
  hipLaunchKernelGGL(kern, dim3((unsigned)(tm * tn)), dim3(SNW * 64), smem, st, g.A, g.AS, g.as_stride, g.W, g.WS,
                     g.ws_stride, g.C, g.M, g.N, g.K, tm, g.n_out);
  return hipGetLastError();
}
// The same sums, a wave per 16x16 tile over all of K by itself, with no barrier:
// with more tiles than one round of the kernel above there are waves enough to
// hide a stage's issue and latency, and handing the products on costs more. A
// workgroup is 2x2 such waves (what they read in common hits the CU's cache),
// each with an LDS ring of two stages of its own (three to six are slower). While
// a stage's products are formed the next one is read and its slot refilled; then
// the stage is folded. Every wave copies its own operands: four waves ask a CU's
// cache for 17 KB a stage, 272 clocks of its 64 bytes per clock, of about 420 that
// a stage takes.
// gate|up: the left waves have gate, the right ones up.
template <bool GROUPED, bool WSF16, int GB, int GLU, bool OUT_F16>
__global__ __launch_bounds__(256, 2) void wave_i8_kernel(
    const int8_t *__restrict__ A, const float *__restrict__ AS, int as_stride, const int8_t *__restrict__ W,
    const float *__restrict__ WS, int ws_stride, void *__restrict__ C, int M, int N, int K, int tiles_m, int n_out) {
  using G = WaveI8Geom<GROUPED>;
  constexpr int GPS = 4 / GB, ST = G::ST;
  constexpr int L = 5 + (GROUPED ? 1 : 0);  // copies per stage
  static_assert((!WSF16 || (GROUPED && GB == 1)) && (GLU == GLU_NONE || !GROUPED), "form");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const int id = xcd_remap(blockIdx.x, gridDim.x);
  const int m0 = (id % tiles_m * 2 + (wave >> 1)) * 16, n0 = (id / tiles_m * 2 + (wave & 1)) * 16;
  const int rows = min(M - m0, 16), cols = min(N - n0, 16);
  if (GLU == GLU_NONE && (rows <= 0 || cols <= 0)) return;  // (gate|up: a barrier follows; empty buffers read zeros)
  const int KT = (K + 127) / 128, KB = K / 32;
  uint8_t *const ring = smem + wave * (ST * G::SLOT);

  const rsrc_t ra = make_rsrc(A + (size_t)m0 * K, (int64_t)rows * K);
  const rsrc_t rw = make_rsrc(W + (size_t)n0 * K, (int64_t)cols * K);
  const rsrc_t rs = make_rsrc(WS + (size_t)n0 * ws_stride, (int64_t)cols * ws_stride * 4);
  const rsrc_t ras = make_rsrc(AS + (size_t)m0 * as_stride, (int64_t)rows * as_stride * 4);
  const int r8 = lane >> 3, p8 = lane & 7;
  const int ch[2] = {p8 ^ (r8 >> 1), p8 ^ (4 + (r8 >> 1))};  // as in skinny_i8_kernel
  const uint32_t v_q[2] = {(uint32_t)(r8 * K + ch[0] * 16), (uint32_t)((8 + r8) * K + ch[1] * 16)};
  const uint32_t v_ws = (uint32_t)(((lane >> 2) * ws_stride + (lane & 3)) * 4);
  const uint32_t v_as = (uint32_t)((l16 * as_stride + lg) * 4);  // [group][row]
  auto issue = [&](int slot, int kt) {  // kt < KT
    uint8_t *sb = ring + slot * G::SLOT;
    const uint32_t k0 = kt * 128;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const uint32_t v = (int)k0 + ch[q] * 16 < K ? v_q[q] : OOB_OFFSET;
      bdma16(ra, sb + q * 1024, v, k0);
      bdma16(rw, sb + G::W_OFF + q * 1024, v, k0);
    }
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, LDS_PTR(sb + G::WS_OFF), 4, v_ws, (uint32_t)(kt * 16), 0, 0);
    if constexpr (GROUPED)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ras, LDS_PTR(sb + G::AS_OFF), 4,
                                               lg < GPS && kt * 4 + lg * GB < KB ? v_as : OOB_OFFSET,
                                               (uint32_t)(kt * GPS * 4), 0, 0);
  };
  struct Frags {
    long a[4], w[4];
    floatx4 ws, as[GROUPED ? GPS : 1];
  } fr[2];
  uint32_t f_off[4];  // the lane's 8 bytes of block b of its row
#pragma unroll
  for (int b = 0; b < 4; ++b)
    f_off[b] = (uint32_t)(l16 * 128 + (((2 * b + (lg >> 1)) ^ (l16 >> 1)) << 4) + (lg & 1) * 8);
  auto read = [&](Frags &f, int slot) {
    const uint8_t *sb = ring + slot * G::SLOT;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      f.a[b] = *(const long *)(sb + f_off[b]);
      f.w[b] = *(const long *)(sb + G::W_OFF + f_off[b]);
    }
    f.ws = *(const floatx4 *)(sb + G::WS_OFF + l16 * 16);
    if constexpr (GROUPED) {
#pragma unroll
      for (int g = 0; g < GPS; ++g) f.as[g] = *(const floatx4 *)(sb + G::AS_OFF + g * 64 + lg * 16);
    }
  };
  constexpr int GBIAS_BITS = 0x4B400000;  // 1.5·2^23, see gemm_i8_q8_kernel
  constexpr float GBIAS = 12582912.0f;
  constexpr int INIT = WSF16 ? GBIAS_BITS : 0;
  floatx4 facc = {0.f, 0.f, 0.f, 0.f};  // rows 4·lg + e of column l16
  auto fold = [&](const Frags &f, int g, intx4 p) {
    const float d = f.ws[g * GB];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int bits = p[e];
      if constexpr (WSF16)
        facc[e] = __builtin_fmaf(__builtin_fmaf(__int_as_float(bits), d, -GBIAS * d), f.as[g][e], facc[e]);
      else
        facc[e] = __builtin_fmaf((float)bits, GROUPED ? f.as[GROUPED ? g : 0][e] * d : d, facc[e]);
    }
  };
  // All copies but those of the `later` stages issued last have landed.
  auto landed = [&](auto later_c) {
    WAIT_VMCNT(decltype(later_c)::value * L);
    asm volatile("" ::: "memory");
  };
  int slot = 0;  // of the stage whose fragments were read last
  auto step = [&](const Frags &cur, Frags &nxt, int kt, auto steady_c) {
    constexpr bool STEADY = decltype(steady_c)::value;  // kt + 1 + ST < KT
    if (STEADY || kt + 1 < KT) {
      if (STEADY || kt + 1 + ST <= KT)
        landed(ic<ST - 1>{});
      else
        landed(ic<0>{});
      slot = slot + 1 == ST ? 0 : slot + 1;
      read(nxt, slot);
    }
    intx4 p[GPS];
#pragma unroll
    for (int g = 0; g < GPS; ++g) {
      p[g] = intx4{INIT, INIT, INIT, INIT};
#pragma unroll
      for (int b = g * GB; b < (g + 1) * GB; ++b)
        p[g] = __builtin_amdgcn_mfma_i32_16x16x32_i8(cur.a[b], cur.w[b], p[g], 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    WAIT_LGKMCNT0();  // stage kt + 1 is read: its slot is free
    asm volatile("" ::: "memory");
    if (STEADY || kt + 1 + ST < KT) issue(slot, kt + 1 + ST);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < GPS; ++g) {
      if (!STEADY && kt * 4 + g * GB >= KB) break;  // wave-uniform: K ends inside the stage
      fold(cur, g, p[g]);
    }
  };
#pragma unroll
  for (int i = 0; i < ST; ++i)
    if (i < KT) issue(i, i);
  float as_m[4];  // per token: the rows' scales
#pragma unroll
  for (int e = 0; e < 4; ++e) as_m[e] = GROUPED ? 1.f : AS[(size_t)min(m0 + 4 * lg + e, M - 1) * as_stride];
  if (KT >= ST)
    landed(ic<ST - 1>{});
  else
    landed(ic<0>{});
  read(fr[0], 0);
  WAIT_LGKMCNT0();
  asm volatile("" ::: "memory");
  if (ST < KT) issue(0, ST);
  int kt = 0;
  for (; kt + 2 + ST < KT; kt += 2) {
    step(fr[0], fr[1], kt, std::true_type{});
    step(fr[1], fr[0], kt + 1, std::true_type{});
  }
  for (; kt < KT; kt += 2) {
    step(fr[0], fr[1], kt, std::false_type{});
    if (kt + 1 < KT) step(fr[1], fr[0], kt + 1, std::false_type{});
  }

  auto store = [&](int m, int n, int ld, float y) {
    if (m < M && n < ld) {
      if constexpr (OUT_F16)
        ((f16 *)C)[(size_t)m * ld + n] = (f16)y;
      else
        ((float *)C)[(size_t)m * ld + n] = y;
    }
  };
  const int mr = m0 + 4 * lg;
  if constexpr (GLU != GLU_NONE) {  // the two waves swap, each finishes two of a lane's four rows
    float *x = (float *)(smem + (wave & 2) * (ST * G::SLOT));  // [gate, up][row][lane], over the pair's rings
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e) x[((wave & 1) * 4 + e) * 64 + lane] = as_m[e] * facc[e];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int e = 2 * (wave & 1) + i;
      store(mr + e, (n0 & ~31) / 2 + l16, n_out, glu_apply<GLU>(x[e * 64 + lane], x[(4 + e) * 64 + lane]));
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (GROUPED)
        store(mr + e, n0 + l16, N, facc[e]);
      else
        store(mr + e, n0 + l16, N, as_m[e] * facc[e]);
    }
  }
}

template <bool GROUPED, bool WSF16, int GB, int GLU, bool OUT_F16>
static hipError_t launch_wave_i8(const I8GemmArgs &g, hipStream_t st) {
  using G = WaveI8Geom<GROUPED>;
  static_assert(G::SMEM <= 64 * 1024, "LDS without an attribute");
  const int tm = (g.M + 31) / 32, tn = (g.N + 31) / 32;
  hipLaunchKernelGGL((wave_i8_kernel<GROUPED, WSF16, GB, GLU, OUT_F16>), dim3((unsigned)(tm * tn)), dim3(256), G::SMEM,
                     st, g.A, g.AS, g.as_stride, g.W, g.WS, g.ws_stride, g.C, g.M, g.N, g.K, tm, g.n_out);
  return hipGetLastError();
}

// skinny_i8_kernel while its tiles (16x16, or 16x32, which read the rows half as
// often) are one round of workgroups, wave_i8_kernel above (MI355X, per token:
// 3072->1024, 256 rows, two rounds, 11.3 us and 8.0; 1024->3072, 64 rows, two
// rounds, 5.8 and 4.9; within one round a wave that walks 3072 values alone takes
// 7 us and more at any number of rows).
template <bool GROUPED, bool WSF16, int GB, bool OUT_F16>
static hipError_t launch_skinny_i8_out(const I8GemmArgs &g, hipStream_t st) {
  const int64_t tm = (g.M + 15) / 16, n16 = (g.N + 15) / 16, n32 = (g.N + 31) / 32;
  const bool one16 = tm * n16 <= g.num_cus, one32 = tm * n32 <= g.num_cus;
  if constexpr (!GROUPED && GB == 1) {  // gate|up: pairs of 16x16
    if (g.glu == GLU_SILU)
      return one32 ? launch_skinny_i8_tn<false, false, 1, 2, GLU_SILU, OUT_F16>(g, st)
                   : launch_wave_i8<false, false, 1, GLU_SILU, OUT_F16>(g, st);
    if (g.glu == GLU_GELU)
      return one32 ? launch_skinny_i8_tn<false, false, 1, 2, GLU_GELU, OUT_F16>(g, st)
                   : launch_wave_i8<false, false, 1, GLU_GELU, OUT_F16>(g, st);
  }
  if (one16) return launch_skinny_i8_tn<GROUPED, WSF16, GB, 1, GLU_NONE, OUT_F16>(g, st);
  if (one32) return launch_skinny_i8_tn<GROUPED, WSF16, GB, 2, GLU_NONE, OUT_F16>(g, st);
  return launch_wave_i8<GROUPED, WSF16, GB, GLU_NONE, OUT_F16>(g, st);
}
template <bool GROUPED, bool WSF16, int GB>
static hipError_t launch_skinny_i8(const I8GemmArgs &g, hipStream_t st) {
  return g.out_f16 ? launch_skinny_i8_out<GROUPED, WSF16, GB, true>(g, st)
                   : launch_skinny_i8_out<GROUPED, WSF16, GB, false>(g, st);
}

// By the number of 16x16 output tiles against the CUs: past that the operands
// read again by every tile cost more than the tiled kernel's serial stages.
// MI355X, 256 CUs, tiled -> here. Per token, 16 tiles per CU: 1024->3072 15 tiles
// 9.4 -> 8.4, 18 tiles 9.4 -> 9.8; 2048->4096 16 tiles 15.0 -> 13.2, 20 tiles
// 15.2 -> 15.9; 4352->1152 13.5 tiles 28.0 -> 25.7; gate|up 1024->2x3072 12 tiles
// 10.6 -> 7.1, 19.5 tiles 11.0 -> 10.7; 3072->2x1024 16 tiles 22.6 -> 17.4, 24 tiles
// 22.8 -> 24.6. Group 32, 15 tiles: 1024->3072 15 tiles 12.0 -> 11.2, 18 tiles
// 12.0 -> 13.2; 4352->1152 13.5 tiles 39.5 -> 38.7; 2048->4096 16 tiles 20.3 ->
// 19.6. Groups of 64 and 128, 7 tiles: 1024->3072 in groups of 128, 6 tiles 6.3 ->
// 5.7, 9.8 tiles 6.5 -> 7.3; 4352->1152 6.8 tiles 16.5 -> 15.0, 9 tiles 16.7 ->
// 19.2. A tile forced by RK_Q8_TILE / RK_Q8G_TILE keeps the tiled kernel;
// RK_SKINNY=0 turns these kernels off.
bool rk_gemm_i8_skinny(const I8GemmArgs &g) {
  const bool token = g.mode == I8_PER_TOKEN, group = g.mode == I8_PER_GROUP && g.a_gb == g.gb;
  if (!(token || group) || (g.gb != 1 && g.gb != 2 && g.gb != 4)) return false;
  if (rk_knob("RK_SKINNY", 1) == 0 || rk_knob(token ? "RK_Q8_TILE" : "RK_Q8G_TILE", -1) >= 0) return false;
  const int64_t tiles = (int64_t)((g.M + 15) / 16) * ((g.N + 15) / 16);
  return tiles <= (g.gb > 1 ? 7 : group ? 15 : 16) * (int64_t)g.num_cus;
}

hipError_t rk_launch_gemm_i8_skinny(const I8GemmArgs &g, hipStream_t st) {
  if (g.mode == I8_PER_TOKEN) {
    if (g.gb == 1) return launch_skinny_i8<false, false, 1>(g, st);
    if (g.gb == 2) return launch_skinny_i8<false, false, 2>(g, st);
    if (g.gb == 4) return launch_skinny_i8<false, false, 4>(g, st);
  } else if (g.mode == I8_PER_GROUP) {
    if (g.gb == 1)
      return g.ws_f16 ? launch_skinny_i8<true, true, 1>(g, st) : launch_skinny_i8<true, false, 1>(g, st);
    if (g.gb == 2) return launch_skinny_i8<true, false, 2>(g, st);
    if (g.gb == 4) return launch_skinny_i8<true, false, 4>(g, st);
  }
  return hipErrorInvalidValue;
}

// fp16: operands straight from memory into registers (no other wave of the
// workgroup reads the same bytes; a stage's loads and the next one's are in
// flight together). A stage is 64 K-values (two v_mfma_f32_16x16x32_f16 steps),
// TM 16-row tiles, TN 16-row weight tiles (2: gate and up of 16 outputs). The MFMA forms
// Cᵀ tiles, so a lane holds 4 consecutive columns of one row.
template <int TM, int TN>
__global__ __launch_bounds__(SNW * 64, 2) void skinny_f16_kernel(const f16 *__restrict__ A, const f16 *__restrict__ B,
                                                                 void *__restrict__ C, int M, int N, int K,
                                                                 int out_f16, int glu, int n_out) {
  constexpr int T = TM * TN;
  __shared__ __attribute__((aligned(16))) float red[SNW * T * 256];  // [wave][tile][lane][4]
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15, lg = lane >> 4;
  const int n0 = blockIdx.x * (16 * TN), m0 = blockIdx.y * (16 * TM);
  const int rows = min(M - m0, 16 * TM), cols = min(N - n0, 16 * TN);
  const int KT = (K + 63) / 64;

  const rsrc_t ra = make_rsrc(A + (size_t)m0 * K, (int64_t)rows * K * 2);
  const rsrc_t rb = make_rsrc(B + (size_t)n0 * K, (int64_t)cols * K * 2);
  const uint32_t v_row = (uint32_t)((l16 * K + lg * 8) * 2);
  const bool ktail = (K % 64) != 0;

  struct Stage {
    half8 a[2][TM], b[2][TN];
  } st[2];
  auto load = [&](Stage &s, int kt) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      // chunks past K read as zeros
      const bool past = ktail && kt * 64 + u * 32 + lg * 8 >= K;
      const uint32_t v = past ? OOB_OFFSET : v_row + u * 64;
#pragma unroll
      for (int j = 0; j < TN; ++j)
        s.b[u][j] = __builtin_bit_cast(
            half8, __builtin_amdgcn_raw_buffer_load_b128(rb, past ? OOB_OFFSET : v + j * 32 * K, kt * 128, 0));
#pragma unroll
      for (int i = 0; i < TM; ++i)
        s.a[u][i] = __builtin_bit_cast(
            half8, __builtin_amdgcn_raw_buffer_load_b128(ra, past ? OOB_OFFSET : v + i * 32 * K, kt * 128, 0));
    }
  };
  floatx4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  auto stage = [&](const Stage &s) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(s.b[u][j], s.a[u][i], acc[i][j], 0, 0, 0);
  };
  if (wave < KT) load(st[0], wave);
  for (int kt = wave; kt < KT; kt += 2 * SNW) {
    if (kt + SNW < KT) load(st[1], kt + SNW);
    stage(st[0]);
    if (kt + SNW < KT) {
      if (kt + 2 * SNW < KT) load(st[0], kt + 2 * SNW);
      stage(st[1]);
    }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) *(floatx4 *)(red + ((wave * T + i * TN + j) * 64 + lane) * 4) = acc[i][j];
  __syncthreads();
  auto value = [&](int t, int e) {  // element e of tile t: row (e/4)%16, column 4·(e/64) + e%4
    float v = red[t * 256 + e];
#pragma unroll
    for (int w = 1; w < SNW; ++w) v += red[(w * T + t) * 256 + e];
    return v;
  };
  if (glu != GLU_NONE) {  // tile pairs: gate and up of 16 outputs
    for (int x = threadIdx.x; x < T * 128; x += SNW * 64) {
      const int p = x >> 8, i = p / (TN / 2 ? TN / 2 : 1), j = p % (TN / 2 ? TN / 2 : 1);
      const int c = x & 15, r = (x >> 4) & 15;  // columns fastest: coalesced stores
      const int e = (c >> 2) * 64 + r * 4 + (c & 3);
      const int m = m0 + i * 16 + r, oc = n0 / 2 + j * 16 + c;
      if (m < M && oc < n_out) {
        const float g = (float)(f16)value(i * TN + 2 * j, e), u = (float)(f16)value(i * TN + 2 * j + 1, e);
        const float y = glu_any(glu, g, u);
        if (out_f16)
          ((f16 *)C)[(size_t)m * n_out + oc] = (f16)y;
        else
          ((float *)C)[(size_t)m * n_out + oc] = y;
      }
    }
    return;
  }
  for (int x = threadIdx.x; x < T * 256; x += SNW * 64) {
    const int t = x >> 8, c = x & 15, r = (x >> 4) & 15;
    const int m = m0 + (t / TN) * 16 + r, n = n0 + (t % TN) * 16 + c;
    if (m < M && n < N) ((f16 *)C)[(size_t)m * N + n] = (f16)value(t, (c >> 2) * 64 + r * 4 + (c & 3));
  }
}

template <int TM, int TN>
static hipError_t launch_skinny_f16(const void *A, const void *B, void *C, int M, int N, int K, bool out_f16, int glu,
                                    int n_out, hipStream_t st) {
  hipLaunchKernelGGL((skinny_f16_kernel<TM, TN>), dim3((N + 16 * TN - 1) / (16 * TN), (M + 16 * TM - 1) / (16 * TM)),
                     dim3(SNW * 64), 0, st, (const f16 *)A, (const f16 *)B, C, M, N, K, (int)out_f16, glu, n_out);
  return hipGetLastError();
}

// Of a product whose K is split over eight waves (rk_gemm_f16_kwaves). n: the outputs
// of one product of a gate|up pair, whose tiles are twice as wide. Below K = 768:
// the smallest tile (1x1, 2x1 or 1x2 of 16x16) that one round of workgroups
// covers. From there gemm_f16_kwaves_kernel shares the reads of a 32x32 tile and
// these win only with a few rows, or while 1x1 tiles do for a short K (MI355X, here
// / there: 3072->1024 1 row 5.1 / 5.8 us, 8 rows 6.2 / 5.8, 16 rows 7.2 / 5.8;
// 2048->1024 8 rows 4.8 / 4.9, 16 rows 5.4 / 5.0; 4304->1152 8 rows 6.3 / 6.9;
// 1024->1024 64 rows 3.9 / 4.2; 1024->3072 32 rows, 2x1, 4.8 / 4.3; gate|up
// 1024->2x3072 8 rows 4.5 / 4.7, 16 rows 4.9 / 4.7).
static int f16_skinny_tile(int M, int n, int K, bool glu, int num_cus) {
  const int64_t m16 = (M + 15) / 16, m32 = (M + 31) / 32, n16 = (n + 15) / 16;
  if (K >= 768) {
    const bool few = glu ? K < 1536 && M <= 8 : K < 1536 || M <= 8;
    return few && M <= 128 && m16 * n16 <= num_cus ? 11 : 0;
  }
  return m16 * n16 <= num_cus ? 11 : m32 * n16 <= num_cus ? 21 : 12;
}

bool rk_gemm_f16_skinny(int kwaves, int M, int n, int K, bool glu, int num_cus) {
  return kwaves == 8 && rk_knob("RK_SKINNY", 1) != 0 && f16_skinny_tile(M, n, K, glu, num_cus) != 0;
}

hipError_t rk_launch_gemm_f16_skinny(const void *A, const void *B, void *C, int M, int N, int K, int glu, int n_out,
                                     bool out_f16, int num_cus, hipStream_t st) {
  if (!glu) n_out = N, out_f16 = true;
  const int tile = f16_skinny_tile(M, n_out, K, glu != 0, num_cus);
  if (glu) {
    if (tile == 11) return launch_skinny_f16<1, 2>(A, B, C, M, N, K, out_f16, glu, n_out, st);
    if (tile == 21) return launch_skinny_f16<2, 2>(A, B, C, M, N, K, out_f16, glu, n_out, st);
    if (tile == 12) return launch_skinny_f16<1, 4>(A, B, C, M, N, K, out_f16, glu, n_out, st);
  } else {
    if (tile == 11) return launch_skinny_f16<1, 1>(A, B, C, M, N, K, out_f16, glu, n_out, st);
    if (tile == 21) return launch_skinny_f16<2, 1>(A, B, C, M, N, K, out_f16, glu, n_out, st);
    if (tile == 12) return launch_skinny_f16<1, 2>(A, B, C, M, N, K, out_f16, glu, n_out, st);
  }
  return hipErrorInvalidValue;
}
