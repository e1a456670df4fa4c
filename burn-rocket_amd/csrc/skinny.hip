// GEMMs with few output tiles (decode steps, search queries, short batches) on
// gfx950: int8 with one scale per weight group, and fp16.
//
// What bounds these is latency, not bytes: the tiled kernels walk K stage by
// stage in each workgroup, with a barrier and an LDS round trip per stage, on
// a grid of a few dozen workgroups. Here a workgroup of 8 waves takes one
// output tile and the waves split K: wave w takes stages w, w + 8, ... on its
// own, with no barrier, and the partial sums meet once, in LDS, added in wave
// order. The order of the sums depends on K alone, so a fused gate|up product
// equals plain products that also run here bit for bit. Measured on MI355X (us
// per call, tiled kernel -> here):
//   int8 per token   12 rows, 1024->3072 8.7 -> 4.1;  3072->1024 20.0 -> 5.3;
//                    256 rows, 3072->1024 20.5 -> 6.0
//   int8 group 32    12 rows, 1024->3072 11.1 -> 4.5; 256 rows, 3072->1024 28.4 -> 7.7
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
// exact int32 product of a group of GB 32-value blocks. A stage is 128 K-values
// (4 blocks, one v_mfma_i32_32x32x32_i8 each) of 32 rows and 32 columns, copied
// by the wave into an LDS ring of its own, of I8_ST slots: whole 128-byte lines, where
// operands loaded straight into registers (32 rows of 32 bytes per load) are
// bound by the cache's line look-ups (3072->1024, 12 / 64 rows, MI355X: 7.3 /
// 8.7 us that way, 5.3 / 5.5 us here).
namespace {
constexpr int I8_A = 4096, I8_W = 4096, I8_WS = 1024;      // bytes of a slot: rows, columns, column scales
constexpr int I8_SLOT = I8_A + I8_W + I8_WS + 512;         // and row scales, [group][row]
}  // namespace

template <bool GROUPED, int GB, int I8_ST>
__global__ __launch_bounds__(SNW * 64, 2) void skinny_i8_kernel(
    const int8_t *__restrict__ A, const float *__restrict__ AS, int as_stride, const int8_t *__restrict__ W,
    const float *__restrict__ WS, int ws_stride, void *__restrict__ C, int M, int N, int K, int out_f16,
    int glu, int n_out) {
  constexpr int GPS = 4 / GB;  // groups per stage
  constexpr int AS_INS = GROUPED ? (GPS + 1) / 2 : 0;  // 64-value copies of row scales
  constexpr int L = 8 + 1 + AS_INS;                    // copies per stage
  constexpr int I8_RING = I8_ST * I8_SLOT;
  static_assert(SNW * I8_RING <= 160 * 1024, "LDS");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];

  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fcol = lane & 31, fh = lane >> 5;
  const int n0 = blockIdx.x * 32, m0 = blockIdx.y * 32;
  const int rows = min(M - m0, 32), cols = min(N - n0, 32);
  const int KT = (K + 127) / 128, KB = K / 32;
  uint8_t *const ring = smem + wave * I8_RING;

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
  auto issue = [&](int slot, int kt) {  // stages past the end copy zeros
    uint8_t *sb = ring + slot * I8_SLOT;
    const int k0 = kt * 128;
    uint32_t v[2];
#pragma unroll
    for (int o = 0; o < 2; ++o) v[o] = k0 + ch[o] * 16 < K ? (uint32_t)(r8 * K + ch[o] * 16) : OOB_OFFSET;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      bdma16(ra, sb + q * 1024, v[q & 1], (uint32_t)(q * 8 * K + k0));
      bdma16(rw, sb + I8_A + q * 1024, v[q & 1], (uint32_t)(q * 8 * K + k0));
    }
    const bool in = kt < KT;
    bdma16(rs, sb + I8_A + I8_W, in && lane < 32 ? (uint32_t)(lane * ws_stride * 4 + kt * 16) : OOB_OFFSET, 0);
#pragma unroll
    for (int c = 0; c < AS_INS; ++c) {
      const int g = 2 * c + fh;  // value 64c + lane: (group, row)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          ras, LDS_PTR(sb + I8_A + I8_W + I8_WS + c * 256), 4,
          in && g < GPS ? (uint32_t)((fcol * as_stride + kt * GPS + g) * 4) : OOB_OFFSET, 0, 0, 0);
    }
  };

  floatx16 facc;
#pragma unroll
  for (int r = 0; r < 16; ++r) facc[r] = 0.f;
  const int swz = (fcol >> 1) & 7;
  uint32_t f_off[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) f_off[b] = (uint32_t)(fcol * 128 + (((2 * b + fh) ^ swz) << 4));

#pragma unroll
  for (int i = 0; i < I8_ST; ++i) issue(i, wave + i * SNW);
  int slot = 0;
  for (int kt = wave; kt < KT; kt += SNW) {
    WAIT_VMCNT((I8_ST - 1) * L);  // this stage has landed (the next may be on its way)
    asm volatile("" ::: "memory");
    const uint8_t *sb = ring + slot * I8_SLOT;
    intx4 a[4], w[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      a[b] = *(const intx4 *)(sb + f_off[b]);
      w[b] = *(const intx4 *)(sb + I8_A + f_off[b]);
    }
    const floatx4 ws = *(const floatx4 *)(sb + I8_A + I8_W + fcol * 16);
    floatx4 as[GPS][4];  // the lane's 16 rows of each group: 8q + 4·fh + 0..3
#pragma unroll
    for (int g = 0; g < GPS; ++g)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        as[g][q] = GROUPED ? *(const floatx4 *)(sb + I8_A + I8_W + I8_WS + (g * 32 + q * 8 + fh * 4) * 4)
                           : floatx4{1.f, 1.f, 1.f, 1.f};
    WAIT_LGKMCNT0();  // the slot is read: refilled while the products are formed
    asm volatile("" ::: "memory");
    issue(slot, kt + I8_ST * SNW);
#pragma unroll
    for (int g = 0; g < GPS; ++g) {
      if (kt * 4 + g * GB >= KB) break;  // wave-uniform: K ends inside the stage
      const float d = ws[g * GB];
      intx16 p = {};
#pragma unroll
      for (int b = 0; b < GB; ++b)
        p = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[g * GB + b], w[g * GB + b], p, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float sc = GROUPED ? as[g][r >> 2][r & 3] * d : d;
        facc[r] = __builtin_fmaf((float)p[r], sc, facc[r]);
      }
    }
    slot = slot + 1 == I8_ST ? 0 : slot + 1;
  }
  WAIT_VMCNT(0);  // no copy may still be writing LDS

  float *mine = (float *)ring;
#pragma unroll
  for (int r = 0; r < 16; ++r) mine[r * 64 + lane] = facc[r];
  __syncthreads();
  // Element e = r·64 + lane: row 8·(r/4) + 4·(lane/32) + r%4,
  // column lane%32 (gate|up: columns 0..15 gate, 16..31 up).
  const float *red = (const float *)smem;
  auto value = [&](int e, int m) {
    float v = red[e];
#pragma unroll
    for (int w = 1; w < SNW; ++w) v += red[w * (I8_RING / 4) + e];
    return GROUPED ? v : AS[(size_t)m * as_stride] * v;
  };
  auto row_of = [&](int e) { return m0 + (e >> 8) * 8 + ((e >> 5) & 1) * 4 + ((e >> 6) & 3); };
  if (glu != GLU_NONE) {
    const int p = threadIdx.x;  // 512 gate|up pairs
    const int e = (p >> 4) * 32 + (p & 15);
    const int m = row_of(e), oc = n0 / 2 + (p & 15);
    if (m < M && oc < n_out) {
      const float y = glu_any(glu, value(e, m), value(e + 16, m));
      if (out_f16)
        ((f16 *)C)[(size_t)m * n_out + oc] = (f16)y;
      else
        ((float *)C)[(size_t)m * n_out + oc] = y;
    }
    return;
  }
  for (int e = threadIdx.x; e < 1024; e += SNW * 64) {
    const int m = row_of(e), n = n0 + (e & 31);
    if (m < M && n < N) {
      const float y = value(e, m);
      if (out_f16)
        ((f16 *)C)[(size_t)m * N + n] = (f16)y;
      else
        ((float *)C)[(size_t)m * N + n] = y;
    }
  }
}

template <bool GROUPED, int GB, int ST>
static hipError_t launch_skinny_i8_st(const I8GemmArgs &g, hipStream_t st) {
  auto kern = skinny_i8_kernel<GROUPED, GB, ST>;
  constexpr int smem = SNW * ST * I8_SLOT;
  static bool attr_set = false;
  if (!attr_set) {
    hipError_t e = hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) return e;
    attr_set = true;
  }
  hipLaunchKernelGGL(kern, dim3((g.N + 31) / 32, (g.M + 31) / 32), dim3(SNW * 64), smem, st, g.A, g.AS, g.as_stride,
                     g.W, g.WS, g.ws_stride, g.C, g.M, g.N, g.K, (int)g.out_f16, g.glu, g.glu ? g.n_out : g.N);
  return hipGetLastError();
}
// Two slots (one workgroup per CU) while the grid is one round of workgroups,
// one slot (two per CU) above: 1024->3072, 128 rows (384 tiles), 7.4 us with two
// slots, 5.2 with one.
template <bool GROUPED, int GB>
static hipError_t launch_skinny_i8(const I8GemmArgs &g, hipStream_t st) {
  const int64_t wgs = (int64_t)((g.N + 31) / 32) * ((g.M + 31) / 32);
  return wgs <= g.num_cus ? launch_skinny_i8_st<GROUPED, GB, 2>(g, st) : launch_skinny_i8_st<GROUPED, GB, 1>(g, st);
}

// By the number of 32x32 output tiles (of one product of a gate|up pair)
// against the CUs: past a few rounds of workgroups the weights and activations
// re-read by every tile cost more than the tiled kernel's serial stages.
// MI355X, 256 CUs, tiled -> here: per token 1024->3072 768 tiles 9.3 -> 7.1 us,
// 1152->4304 540 tiles 9.9 -> 7.1, 945 tiles 10.2 -> 11.0; group 32 1024->3072 768
// tiles 11.9 -> 10.8, 960 tiles 12.0 -> 13.6; gate|up 1024->2x4096 512 tiles
// 10.6 -> 8.0, 1152->2x4304 540 tiles 11.2 -> 12.5; group 128 1024->4096 512 tiles
// 6.1 -> 5.3, 1024->3072 576 tiles 6.2 -> 6.5. A tile forced by RK_Q8_TILE /
// RK_Q8G_TILE keeps the tiled kernel; RK_SKINNY=0 turns these kernels off.
bool rk_gemm_i8_skinny(const I8GemmArgs &g) {
  const bool token = g.mode == I8_PER_TOKEN, group = g.mode == I8_PER_GROUP && g.a_gb == g.gb;
  if (!(token || group) || (g.gb != 1 && g.gb != 2 && g.gb != 4)) return false;
  if (rk_knob("RK_SKINNY", 1) == 0 || rk_knob(token ? "RK_Q8_TILE" : "RK_Q8G_TILE", -1) >= 0) return false;
  const int64_t n = g.glu ? g.n_out : g.N;
  const int64_t tiles = ((g.M + 31) / 32) * ((n + 31) / 32);
  return tiles <= (g.gb == 1 && !g.glu ? 3 : 2) * (int64_t)g.num_cus;
}

hipError_t rk_launch_gemm_i8_skinny(const I8GemmArgs &g, hipStream_t st) {
  if (g.mode == I8_PER_TOKEN) {
    if (g.gb == 1) return launch_skinny_i8<false, 1>(g, st);
    if (g.gb == 2) return launch_skinny_i8<false, 2>(g, st);
    if (g.gb == 4) return launch_skinny_i8<false, 4>(g, st);
  } else if (g.mode == I8_PER_GROUP) {
    if (g.gb == 1) return launch_skinny_i8<true, 1>(g, st);
    if (g.gb == 2) return launch_skinny_i8<true, 2>(g, st);
    if (g.gb == 4) return launch_skinny_i8<true, 4>(g, st);
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
  if (glu != GLU_NONE) {
    for (int x = threadIdx.x; x < TM * 256; x += SNW * 64) {
      const int i = x >> 8, c = x & 15, r = (x >> 4) & 15;  // columns fastest: coalesced stores
      const int e = (c >> 2) * 64 + r * 4 + (c & 3);
      const int m = m0 + i * 16 + r, oc = n0 / 2 + c;
      if (m < M && oc < n_out) {
        const float g = (float)(f16)value(i * TN, e), u = (float)(f16)value(i * TN + TN - 1, e);
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

// n: the outputs of one product of a gate|up pair. Below K = 768: the smallest
// tile (1x1, 2x1 or 1x2 of 16x16; gate|up needs 1x2) that one round of
// workgroups covers, none if that takes larger ones. From there
// gemm_f16_kwaves_kernel shares the reads of a 32x32 tile and these win only
// with a few rows, or while 1x1 tiles do for a short K (MI355X, here / there:
// 3072->1024 1 row 5.1 / 5.8 us, 8 rows 6.2 / 5.8, 16 rows 7.2 / 5.8;
// 2048->1024 8 rows 4.8 / 4.9, 16 rows 5.4 / 5.0; 4304->1152 8 rows 6.3 / 6.9;
// 1024->1024 64 rows 3.9 / 4.2; 1024->3072 32 rows, 2x1, 4.8 / 4.3; gate|up
// 1024->2x3072 8 rows 4.5 / 4.7, 16 rows 4.9 / 4.7). A tile or split forced by
// RK_F16_TILE / RK_F16_KSPLIT keeps the tiled kernel.
static int f16_skinny_tile(int M, int n, int K, bool glu, int num_cus) {
  if (M > 128) return 0;
  const int64_t m16 = (M + 15) / 16, m32 = (M + 31) / 32, n16 = (n + 15) / 16, n32 = (n + 31) / 32;
  if (K >= 768) {
    if (m16 * n16 > num_cus) return 0;
    if (glu) return K < 1536 && M <= 8 ? 12 : 0;
    return K < 1536 || M <= 8 ? 11 : 0;
  }
  if (glu) return m16 * n16 <= num_cus ? 12 : 0;
  if (m16 * n16 <= num_cus) return 11;
  if (m32 * n16 <= num_cus) return 21;
  return m16 * n32 <= num_cus ? 12 : 0;
}

bool rk_gemm_f16_skinny(int M, int n, int K, bool glu, int num_cus) {
  if (rk_knob("RK_SKINNY", 1) == 0 || rk_knob("RK_F16_TILE", -1) >= 0 || rk_knob("RK_F16_KSPLIT", 1) != 1) return false;
  return f16_skinny_tile(M, n, K, glu, num_cus) != 0;
}

hipError_t rk_launch_gemm_f16_skinny(const void *A, const void *B, void *C, int M, int N, int K, int glu, int n_out,
                                     bool out_f16, int num_cus, hipStream_t st) {
  if (!glu) n_out = N, out_f16 = true;
  switch (f16_skinny_tile(M, n_out, K, glu != 0, num_cus)) {
    case 11: return launch_skinny_f16<1, 1>(A, B, C, M, N, K, out_f16, glu, n_out, st);
    case 21: return launch_skinny_f16<2, 1>(A, B, C, M, N, K, out_f16, glu, n_out, st);
    case 12: return launch_skinny_f16<1, 2>(A, B, C, M, N, K, out_f16, glu, n_out, st);
  }
  return hipErrorInvalidValue;
}
