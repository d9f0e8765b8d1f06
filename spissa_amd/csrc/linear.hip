// linear.hip -- the projections on either side of the attention path:
// out[M, N] = x[M, K] x W[N, K]^T + bias[N] with f32 activations and output
// and the weight resident in HBM as bf16, f16 or f32
// (crates/spissa-runtime/src/streaming/linear.rs:269-576,
// streaming_tile_linear_from_model, whose exact default accumulates each
// output as bias + a sequential f32 dot: streaming/kernels_raw16.rs:532-600,
// streaming/mod.rs:311-320; the plain form is ops.rs:62-105 linear).
//
// Five kernels here, and the tile kernel of linear_tile.hip for what lies
// between:
//  - linear_gemv_kernel (M <= 4 tokens, the decode projections): bound by the
//    weight bytes. A wave owns two weight rows; each lane streams 16-byte
//    pieces of them (8 bf16/f16 or 4 f32 weights) with the matching
//    activations from the cache, accumulates in f32, and the wave sums its
//    lanes with DPP and permlane exchanges.
//    linear_gemv_pass_kernel is its form for 16-bit weight rows of up to 4096: the
//    whole row is in flight before the first product, and x lies in LDS.
//  - linear_skinny_kernel (bf16 weights, 5 <= M <= 16, K % 32 == 0): 16x16x32
//    MFMAs, the activations split as below, K split over the workgroup's
//    eight waves.
//  - linear_short_kernel (bf16 weights, 5 <= M <= 64, short K, K % 128 == 0):
//    the same MFMAs on operands loaded straight in their order, K split over
//    four waves.
//  - linear_gemm_kernel (bf16 weights, large prompts, K % 32 == 0): MFMA
//    v_mfma_f32_32x32x16_bf16 on 256 x 320 or 128 x 256 output tiles, 32-deep
//    k tiles in LDS (weights copied global -> LDS with global_load_lds_dwordx4,
//    activations converted in registers). Each f32 activation is split into
//    bf16 hi = rne(x) and lo = rne(x - hi), and both halves meet the bf16
//    weight: the products are exact in f32 and the residual of the split is
//    below 2^-16 |x|, so the result carries f32-level error rather than bf16.
//  - linear_generic_kernel (everything else): one thread per output, the
//    reference's sequential f32 sum from the bias with separately rounded
//    products, so its results equal the reference's linear bit for bit.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "internal.hpp"

namespace spissa {

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
typedef __attribute__((address_space(3))) void lds_void;

// 16 bytes of weights -> f32 (exact for every dtype).
template <typename WT>
struct WChunk;
template <>
struct WChunk<float> {
  static constexpr int N = 4;
  __device__ static void get(const uint4 r, float (&f)[4]) {
    f[0] = __uint_as_float(r.x);
    f[1] = __uint_as_float(r.y);
    f[2] = __uint_as_float(r.z);
    f[3] = __uint_as_float(r.w);
  }
};
template <>
struct WChunk<__bf16> {
  static constexpr int N = 8;
  __device__ static void get(const uint4 r, float (&f)[8]) {
    const unsigned u[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = __uint_as_float(u[i] << 16);
      f[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
    }
  }
};
template <>
struct WChunk<_Float16> {
  static constexpr int N = 8;
  __device__ static void get(const uint4 r, float (&f)[8]) {
    const unsigned u[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = (float)__builtin_bit_cast(_Float16, (unsigned short)(u[i] & 0xffffu));
      f[2 * i + 1] = (float)__builtin_bit_cast(_Float16, (unsigned short)(u[i] >> 16));
    }
  }
};

template <int CTRL>
__device__ __forceinline__ float dpp0(float v) {
  return __builtin_amdgcn_update_dpp(0.0f, v, CTRL, 0xf, 0xf, false);
}

// Sum over the 64 lanes of a wave (every lane receives it).
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp0<0xB1>(v);   // lane ^ 1
  v += dpp0<0x4E>(v);   // lane ^ 2
  v += dpp0<0x141>(v);  // row_half_mirror
  v += dpp0<0x140>(v);  // row_mirror
  auto r16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(r16[0]) + __uint_as_float(r16[1]);
  auto r32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(r32[0]) + __uint_as_float(r32[1]);
}

constexpr int kGemvRowsPerWave = 2;

}  // namespace

// The rows of workgroup `block`: 4 * kGemvRowsPerWave of them. K is a
// multiple of the chunk width (8 for 16-bit weights, 4 for f32).
template <typename WT, int NB>
__device__ __forceinline__ void gemv_rows(const LinearArgs &a, int block) {
  using C = WChunk<WT>;
  constexpr int EPC = C::N, RW = kGemvRowsPerWave;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r0 = (block * 4 + wave) * RW;
  if (r0 >= a.N) return;  // uniform per wave
  const int nch = a.K / EPC;
  const char *wb = reinterpret_cast<const char *>(a.w);
  long roff[RW];
#pragma unroll
  for (int i = 0; i < RW; ++i) roff[i] = (long)min(r0 + i, a.N - 1) * a.K * (long)sizeof(WT);

  float acc[RW][NB], ss[NB];
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    ss[t] = 0.0f;
#pragma unroll
    for (int i = 0; i < RW; ++i) acc[i][t] = 0.0f;
  }
  const float *nw = a.norm_w;  // (uniform)

#pragma unroll 2
  for (int c = lane; c < nch; c += 64) {
    uint4 raw[RW];
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      // each weight byte is read once per call: the non-temporal hint keeps
      // the stream from displacing cached lines (5-8% faster measured)
      const u32x4 q = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(wb + roff[i] + (long)c * 16));
      raw[i] = make_uint4(q.x, q.y, q.z, q.w);
    }
    float xv[NB][EPC];
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const float *xp = a.x + (long)t * a.K + (long)c * EPC;
#pragma unroll
      for (int j = 0; j < EPC; j += 4) {
        const float4 v = *reinterpret_cast<const float4 *>(xp + j);
        xv[t][j] = v.x;
        xv[t][j + 1] = v.y;
        xv[t][j + 2] = v.z;
        xv[t][j + 3] = v.w;
      }
    }
    if (nw) {  // folded RMSNorm: sum of squares, then x * w
      float g[EPC];
#pragma unroll
      for (int j = 0; j < EPC; j += 4) *reinterpret_cast<float4 *>(&g[j]) = *reinterpret_cast<const float4 *>(nw + (long)c * EPC + j);
#pragma unroll
      for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int j = 0; j < EPC; ++j) {
          ss[t] = fmaf(xv[t][j], xv[t][j], ss[t]);
          xv[t][j] *= g[j];
        }
    }
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      float wf[EPC];
      C::get(raw[i], wf);
#pragma unroll
      for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int j = 0; j < EPC; ++j) acc[i][t] = fmaf(wf[j], xv[t][j], acc[i][t]);
    }
  }
#pragma unroll
  for (int i = 0; i < RW; ++i)
#pragma unroll
    for (int t = 0; t < NB; ++t) acc[i][t] = wave_sum(acc[i][t]);
  if (nw) {
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const float inv = 1.0f / sqrtf(wave_sum(ss[t]) / (float)a.K + a.norm_eps);
#pragma unroll
      for (int i = 0; i < RW; ++i) acc[i][t] *= inv;
    }
  }
  if (lane < RW * NB) {
    const int i = lane / NB, t = lane % NB;
    const int r = r0 + i;
    float v = 0.0f;
#pragma unroll
    for (int ii = 0; ii < RW; ++ii)
#pragma unroll
      for (int tt = 0; tt < NB; ++tt) v = (ii == i && tt == t) ? acc[ii][tt] : v;
    if (r < a.N) a.out[(long)t * a.N + r] = (a.bias ? a.bias[r] : 0.0f) + v;
  }
}


// Grid: ceil(N / (4 * kGemvRowsPerWave)) workgroups of 256 threads.
template <typename WT, int NB>
__global__ __launch_bounds__(256) void linear_gemv_kernel(const LinearArgs a) {
  gemv_rows<WT, NB>(a, blockIdx.x);
}

// Several projections of the same input in one launch (the q, k and v
// weights of a layer). Workgroup b belongs to the first segment whose
// cumulative workgroup count exceeds b; within it, the rows and arithmetic
// are those of linear_gemv_kernel, so the results are identical.
template <typename WT, int NB>
__global__ __launch_bounds__(256) void linear_gemv_multi_kernel(const LinearSegments m) {
  int b = blockIdx.x, seg = 0;
  while (seg + 1 < m.n && b >= m.blocks[seg]) b -= m.blocks[seg++];
  gemv_rows<WT, NB>(seg == 0 ? m.seg[0] : seg == 1 ? m.seg[1] : m.seg[2], b);
}

// NB tokens of 16-bit weight rows of at most U 16-byte pieces per lane. Bound by
// the weight bytes at large N and by one round of loads at small N: a wave
// issues every load of its rows before anything waits, where gemv_rows has two
// pieces of each row in flight. Meanwhile the workgroup forms x (times the norm's
// weights) in LDS once, where each wave of gemv_rows reads all of it, for one
// token already as many bytes as its weights, through the L1. The halves of a
// piece's eight activations lie apart, so that a wave's 16-byte reads are
// consecutive. Pieces past the row are read as zeros (range checks of the
// buffers) and add nothing: each lane's sum is gemv_rows' own, bit for bit.
// bf16, weights from HBM, us (gemv_rows against this): one token 512 x 2048
// 3.29 / 2.45, 5120 x 3072 7.58 / 6.86, 128256 x 3072 122.2 / 116.6 (6.8 TB/s);
// with the norm 1536 x 1152 4.05 / 3.17, 3072 x 2048 5.42 / 4.48; four tokens 512 x
// 2048 4.57 / 3.12, 5120 x 3072 12.68 / 9.48. Eight waves a workgroup measured
// the same but for small N (512 x 2048 2.69).
// Grid: the segments' workgroups of 4 * RW rows, as linear_gemv_multi_kernel's.
template <typename WT, int NB, int U, int RW, bool NORM>
__global__ __launch_bounds__(256) void linear_gemv_pass_kernel(const LinearSegments m) {
  static_assert(sizeof(WT) == 2, "8 weights per 16 bytes");
  constexpr int NW = 4, NT = 64 * NW, CH = 64 * U, CPT = (CH + NT - 1) / NT;
  __shared__ u32x4 xs[NB][2][CH];
  __shared__ float squares[NB][NW];
  int block = blockIdx.x, seg = 0;
  while (seg + 1 < m.n && block >= m.blocks[seg]) block -= m.blocks[seg++];
  const LinearArgs &a = seg == 0 ? m.seg[0] : seg == 1 ? m.seg[1] : m.seg[2];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r0 = (block * NW + wave) * RW;  // (rows past N are read clamped and not stored)
  const int row_bytes = a.K * 2;
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.x), 0, NB * a.K * 4, 0x00027000);
  const __amdgpu_buffer_rsrc_t gr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(NORM ? a.norm_w : a.x), 0, a.K * 4, 0x00027000);
  auto load16 = [](const __amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  };

  u32x4 xv[CPT][NB][2], gv[CPT][2], raw[U][RW];
#pragma unroll
  for (int q = 0; q < CPT; ++q) {
    const int c = (int)threadIdx.x + NT * q;
    const bool in = c * 8 < a.K;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int t = 0; t < NB; ++t) xv[q][t][j] = load16(xr, in ? t * a.K * 4 + c * 32 + 16 * j : 0x7ffffff0);
      if constexpr (NORM) gv[q][j] = load16(gr, c * 32 + 16 * j);
    }
  }
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char *>(reinterpret_cast<const char *>(a.w)) + (long)min(r0 + i, a.N - 1) * row_bytes, 0, row_bytes, 0x00027000);
#pragma unroll
    for (int u = 0; u < U; ++u)  // (2: non-temporal)
      raw[u][i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wr, (lane + 64 * u) * 16, 0, 2));
  }
  // (the compiler would sink the loads to their uses to save registers)
  __builtin_amdgcn_sched_barrier(0);

  float ss[NB];
#pragma unroll
  for (int t = 0; t < NB; ++t) ss[t] = 0.0f;
#pragma unroll
  for (int q = 0; q < CPT; ++q) {
    const int c = (int)threadIdx.x + NT * q;
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      if constexpr (NORM) {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float f = __uint_as_float(xv[q][t][j / 4][j % 4]);
          ss[t] = fmaf(f, f, ss[t]);
          xv[q][t][j / 4][j % 4] = __float_as_uint(f * __uint_as_float(gv[q][j / 4][j % 4]));
        }
      }
      if (CH % NT == 0 || c < CH) {
        xs[t][0][c] = xv[q][t][0];
        xs[t][1][c] = xv[q][t][1];
      }
    }
  }
  if constexpr (NORM) {
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      ss[t] = wave_sum(ss[t]);
      if (lane == 0) squares[t][wave] = ss[t];
    }
  }
  // (the weights stay in flight across the barrier)
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

  float acc[RW][NB];
#pragma unroll
  for (int i = 0; i < RW; ++i)
#pragma unroll
    for (int t = 0; t < NB; ++t) acc[i][t] = 0.0f;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float wf[RW][8];
#pragma unroll
    for (int i = 0; i < RW; ++i) WChunk<WT>::get(make_uint4(raw[u][i].x, raw[u][i].y, raw[u][i].z, raw[u][i].w), wf[i]);
#pragma unroll
    for (int t = 0; t < NB; ++t) {
      const u32x4 x0 = xs[t][0][lane + 64 * u], x1 = xs[t][1][lane + 64 * u];
#pragma unroll
      for (int i = 0; i < RW; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][t] = fmaf(wf[i][j], __uint_as_float(j < 4 ? x0[j % 4] : x1[j % 4]), acc[i][t]);
    }
  }
#pragma unroll
  for (int t = 0; t < NB; ++t) {
    float inv = 1.0f;
    if constexpr (NORM) {
      float sum = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; ++w) sum += squares[t][w];
      inv = 1.0f / sqrtf(sum / (float)a.K + a.norm_eps);
    }
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      acc[i][t] = wave_sum(acc[i][t]);
      if constexpr (NORM) acc[i][t] *= inv;
    }
  }
  if (lane < RW * NB) {
    const int i = lane / NB, t = lane % NB, r = r0 + i;
    float v = 0.0f;
#pragma unroll
    for (int ii = 0; ii < RW; ++ii)
#pragma unroll
      for (int tt = 0; tt < NB; ++tt) v = (ii == i && tt == t) ? acc[ii][tt] : v;
    if (r < a.N) a.out[(long)t * a.N + r] = (a.bias ? a.bias[r] : 0.0f) + v;
  }
}

namespace {
constexpr int kBK = 32;              // GEMM k tile
constexpr int kRowBytes = kBK * 2;  // one bf16 tile row: 64 bytes, four 16-byte chunks

// Chunk swizzle of a 64-byte LDS row: any 8 aligned consecutive rows reading
// the same chunk hit 8 distinct 16-byte groups modulo 128 bytes.
__device__ __forceinline__ int swz4(int row) { return ((row >> 1) ^ (row >> 2)) & 3; }

typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

// (rne(a), rne(b)) as bf16 bits, a in the low half.
__device__ __forceinline__ unsigned bf16x2_rne(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

// 16 bytes per lane global -> LDS (global_load_lds_dwordx4); the LDS address
// is the wave's base, lane l's bytes land at +16 l.
__device__ __forceinline__ void copy16_to_lds(const char *src, char *dst) {
  __builtin_amdgcn_global_load_lds(src, (lds_void *)dst, 16, 0, 0);
}
// s_waitcnt vmcnt(N) (N < 16; the other counters unconstrained).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  __builtin_amdgcn_s_waitcnt(0x0F70 | N);
}
}  // namespace

// WIDE: output rows of 2^21 floats and more, stored with 64-bit addresses and a
// test per element. Grid: ceil(M / BM) * ceil(N / BN) workgroups of 512 threads (WM x WN waves,
// each (BM / WM) x (BN / WN) outputs in 32 x 32 blocks). K % 32 == 0. Rows
// past M or N are read clamped and not stored. Two tile shapes
// (linear_prompt_path chooses):
//   256 x 320, 4 x 2 waves of 64 x 160: 104 KB of LDS, one workgroup per CU
//     (two waves per SIMD);
//   128 x 256, 2 x 4 waves of 64 x 64: 64 KB of LDS and at most 128 VGPRs, so
//     two workgroups share a CU and one's stores run beside the other's MFMAs.
// Pipeline, per 32-deep k tile t: the weight tile is copied into one of two
// LDS buffers one step ahead (issued in step t-1), and the activations are
// loaded into registers two steps ahead (issued in step t-2, split and written
// to one of two LDS buffers at the start of step t-1). Step t writes the
// activations of tile t+1, copies the weights of tile t+1, loads the
// activations of tile t+2, runs the MFMAs of tile t, then waits for
// everything but the activation loads it just issued.
// Measured on the 4096 x 5120 x 3072 projection (graph replay, weights from
// HBM): 216 us with 256 x 320 tiles, 251 with 128 x 256, the tile kernel 249;
// called by itself 225-228 (1.13-1.15 PFLOP/s of split products; a large product
// by the vendor's library, half this work per output, reaches 1.29 on this
// card). 4096 x 16384 x 3072: 775 / 721 / 770; 4096 x 16384 x 256: 138 / 95 /
// 127. Reading a step's first fragments before its copies, and an
// XCD-grouped tile order (each XCD a 4 x 8 block of tiles: 424 MB fetched
// beyond L2 for 81 MB of operands otherwise), measured within noise.
template <int BM, int BN, int WM, int WN, int MINWG, bool WIDE>
__global__ __launch_bounds__(WM * WN * 64, MINWG) void linear_gemm_kernel(const LinearArgs a) {
  static_assert(WM * WN == 8, "eight waves");
  constexpr int TM = BM / WM, TN = BN / WN;  // the wave's outputs
  constexpr int BI = TM / 32, BJ = TN / 32;  // its 32 x 32 blocks
  static_assert(BI * 32 == TM && BJ * 32 == TN, "32 x 32 blocks");
  constexpr int WCOPIES = BN * kRowBytes / 1024;  // 1 KB weight copies per k tile
  constexpr int WCW = (WCOPIES + 7) / 8;          // per wave (the last round partial)
  constexpr int XR = BM / 128;                    // activation rows per thread
  static_assert(XR * 128 == BM && WCOPIES * 1024 == BN * kRowBytes, "tile shape");
  __shared__ __attribute__((aligned(1024))) char w_lds0[BN * kRowBytes];
  __shared__ __attribute__((aligned(1024))) char w_lds1[BN * kRowBytes];
  __shared__ __attribute__((aligned(1024))) char xh_lds0[BM * kRowBytes];
  __shared__ __attribute__((aligned(1024))) char xh_lds1[BM * kRowBytes];
  __shared__ __attribute__((aligned(1024))) char xl_lds0[BM * kRowBytes];
  __shared__ __attribute__((aligned(1024))) char xl_lds1[BM * kRowBytes];

  const int tiles_n = (a.N + BN - 1) / BN;
  const int tm = blockIdx.x / tiles_n, tn = blockIdx.x % tiles_n;
  const int m0 = tm * BM, n0 = tn * BN;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wm = wave / WN, wn = wave % WN;  // the wave's TM x TN block
  const int lr = lane & 31, hl = lane >> 5;
  const int nk = a.K / kBK;

  // Weight copies: copy c = wave + 8 j fills LDS bytes [c * 1024, +1024);
  // lane l's 16 bytes land at +16 l, i.e. row R = byte / 64, position p, which
  // holds chunk p ^ swz4(R).
  const char *wg = reinterpret_cast<const char *>(a.w);
  long w_src[WCW];
#pragma unroll
  for (int j = 0; j < WCW; ++j) {
    const int c = min(wave + 8 * j, WCOPIES - 1);
    const int byte = c * 1024 + lane * 16;
    const int row = byte / kRowBytes, p = (byte % kRowBytes) / 16;
    const int n = min(n0 + row, a.N - 1);
    w_src[j] = (long)n * a.K * 2 + 16 * (p ^ swz4(row));
  }
  auto copy_w = [&](int kt, char *dst) {
#pragma unroll
    for (int j = 0; j < WCW; ++j)
      if (wave + 8 * j < WCOPIES) copy16_to_lds(wg + w_src[j] + (long)kt * kBK * 2, dst + (wave + 8 * j) * 1024);
  };
  // Activations: thread t loads rows t / 4 + 128 i, columns 8 (t % 4) + [0, 8)
  // of the k tile, splits them and writes 16 bytes of hi and of lo (chunk
  // t % 4 of the row).
  const int xr = tid >> 2, xc = tid & 3;
  const float *xg[XR];
#pragma unroll
  for (int i = 0; i < XR; ++i) xg[i] = a.x + (long)min(m0 + xr + 128 * i, a.M - 1) * a.K + 8 * xc;
  auto load_x = [&](int kt, float4 (&xv)[XR][2]) {
#pragma unroll
    for (int i = 0; i < XR; ++i)
#pragma unroll
      for (int e = 0; e < 2; ++e) xv[i][e] = *reinterpret_cast<const float4 *>(xg[i] + (long)kt * kBK + 4 * e);
  };
  auto store_x = [&](const float4 (&xv)[XR][2], char *hi, char *lo) {
#pragma unroll
    for (int r = 0; r < XR; ++r) {
      const float f[8] = {xv[r][0].x, xv[r][0].y, xv[r][0].z, xv[r][0].w, xv[r][1].x, xv[r][1].y, xv[r][1].z, xv[r][1].w};
      unsigned h[4], l[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // one v_cvt_pk_bf16_f32 per pair (round to nearest even), for hi and for lo
        h[i] = bf16x2_rne(f[2 * i], f[2 * i + 1]);
        const float r0 = f[2 * i] - __uint_as_float(h[i] << 16);
        const float r1 = f[2 * i + 1] - __uint_as_float(h[i] & 0xffff0000u);
        l[i] = bf16x2_rne(r0, r1);
      }
      const int row = xr + 128 * r;
      const int off = row * kRowBytes + 16 * (xc ^ swz4(row));
      *reinterpret_cast<uint4 *>(hi + off) = make_uint4(h[0], h[1], h[2], h[3]);
      *reinterpret_cast<uint4 *>(lo + off) = make_uint4(l[0], l[1], l[2], l[3]);
    }
  };

  // Fragment offsets: block b of the wave's block, 16-deep k step s: row
  // 32 b + lr of it, chunk 2 s + hl (TM, TN and 32 b are multiples of 32 and
  // leave swz4 unchanged).
  unsigned a_rd[BI][2], b_rd[BJ][2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int b = 0; b < BI; ++b) {
      const int ra = wm * TM + 32 * b + lr;
      a_rd[b][s] = ra * kRowBytes + 16 * ((2 * s + hl) ^ swz4(ra));
    }
#pragma unroll
    for (int b = 0; b < BJ; ++b) {
      const int rb = wn * TN + 32 * b + lr;
      b_rd[b][s] = rb * kRowBytes + 16 * ((2 * s + hl) ^ swz4(rb));
    }
  }

  f32x16 acc[BI][BJ];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  auto compute = [&](const char *wl, const char *xh, const char *xl) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      bf16x8 fa_h[BI], fa_l[BI], fb[BJ];
#pragma unroll
      for (int b = 0; b < BI; ++b) {
        fa_h[b] = *reinterpret_cast<const bf16x8 *>(xh + a_rd[b][s]);
        fa_l[b] = *reinterpret_cast<const bf16x8 *>(xl + a_rd[b][s]);
      }
#pragma unroll
      for (int b = 0; b < BJ; ++b) fb[b] = *reinterpret_cast<const bf16x8 *>(wl + b_rd[b][s]);
#pragma unroll
      for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int j = 0; j < BJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_h[i], fb[j], acc[i][j], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int j = 0; j < BJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa_l[i], fb[j], acc[i][j], 0, 0, 0);
    }
  };

  // One step on tile t; B selects the buffers (t % 2 computes, (t+1) % 2
  // receives): the weights of tile t+1 are copied one step ahead, the
  // activations loaded two ahead and written one ahead.
  auto step = [&](auto B_, int t, float4 (&xnext)[XR][2]) {
    constexpr int B = decltype(B_)::value;
    char *const w_cur = B ? w_lds1 : w_lds0, *const w_fill = B ? w_lds0 : w_lds1;
    char *const xh_cur = B ? xh_lds1 : xh_lds0, *const xl_cur = B ? xl_lds1 : xl_lds0;
    char *const xh_fill = B ? xh_lds0 : xh_lds1, *const xl_fill = B ? xl_lds0 : xl_lds1;
    if (t + 1 < nk) {
      store_x(xnext, xh_fill, xl_fill);
      copy_w(t + 1, w_fill);
    }
    const bool more = t + 2 < nk;
    if (more) load_x(t + 2, xnext);
    compute(w_cur, xh_cur, xl_cur);
    // everything but this step's activation loads is done
    if (more) wait_vmcnt<2 * XR>();
    else wait_vmcnt<0>();
    __syncthreads();
  };

  // Prologue: weights of tile 0 copied, activations of tile 0 in LDS, tile
  // 1's in registers.
  float4 xv[XR][2];
  copy_w(0, w_lds0);
  load_x(0, xv);
  store_x(xv, xh_lds0, xl_lds0);
  if (nk > 1) load_x(1, xv);
  wait_vmcnt<0>();
  __syncthreads();

  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  int t = 0;
  for (; t + 2 <= nk; t += 2) {
    step(I0(), t, xv);
    step(I1(), t + 1, xv);
  }
  if (t < nk) step(I0(), t, xv);

  // Accumulator layout: element e of lane l is row 8 (e / 4) + 4 hl + e % 4,
  // column lr of its 32 x 32 block. Stores go through a buffer that ends with
  // row M - 1: rows past it are dropped, columns past N get an offset past its
  // end, and no branch or argument read stands between the stores.
  const int M = a.M, N = a.N;
  if constexpr (WIDE) {
#pragma unroll
    for (int j = 0; j < BJ; ++j) {
      const int n = n0 + wn * TN + 32 * j + lr;
      const float bn = a.bias ? a.bias[min(n, N - 1)] : 0.0f;
#pragma unroll
      for (int i = 0; i < BI; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int m = m0 + wm * TM + 32 * i + 8 * (e >> 2) + 4 * hl + (e & 3);
          if (m < M && n < N) a.out[(long)m * N + n] = bn + acc[i][j][e];
        }
    }
    return;
  }
  const __amdgpu_buffer_rsrc_t ob = __builtin_amdgcn_make_buffer_rsrc(
      a.out + (long)m0 * N, 0, min(BM, M - m0) * N * 4, 0x00027000);
#pragma unroll
  for (int j = 0; j < BJ; ++j) {
    const int n = n0 + wn * TN + 32 * j + lr;
    const float bn = a.bias ? a.bias[min(n, N - 1)] : 0.0f;
    const unsigned o0 = n < N ? (unsigned)((wm * TM + 4 * hl) * N + n) * 4u : 0x80000000u;
#pragma unroll
    for (int i = 0; i < BI; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(bn + acc[i][j][e]), ob,
                                              (int)(o0 + (unsigned)((32 * i + 8 * (e >> 2) + (e & 3)) * N) * 4u), 0, 0);
  }
}

namespace {
typedef __attribute__((ext_vector_type(4))) float f32x4;
constexpr int kShortRows = 16;  // weight rows per workgroup of linear_short_kernel
}  // namespace

// For 5 to 16 tokens, bf16 weights, K % 8 == 0. A workgroup owns NB blocks of
// 16 weight rows and all tokens; its eight waves share K in contiguous ranges
// and run on their own, each with its own LDS and no barrier, until their sums
// meet at the end. Per 64-deep k tile a wave loads both operands row by row (a
// weight row's 128 bytes by eight lanes, an activation row's 256 by sixteen),
// splits the activations, and passes both through its LDS into
// v_mfma_f32_16x16x32_bf16 operands, two tiles in flight. Bound by the weight
// bytes and one latency. Against operands loaded straight into MFMA order (a
// quad of lanes on four rows: four cycles of address work for one), 16 tokens,
// weights from HBM: 5120 x 3072 20.0 -> 11.9 us (the tile kernel's two
// launches: 14.1), 3072 x 3072 14.8 -> 8.8 (12.4), 1536 x 1152 6.1 -> 5.1 (8.4).
// 64 bytes of a weight row per tile instead of 128: 5120 x 3072 13.6.
template <int NB>
__global__ __launch_bounds__(512, NB == 1 ? 4 : 2) void linear_skinny_kernel(const LinearSegments m) {
  // workgroup -> segment (projections of the same input) and its row block
  int block = blockIdx.x, seg = 0;
  while (seg + 1 < m.n && block >= m.blocks[seg]) block -= m.blocks[seg++];
  const LinearArgs &a = m.seg[seg];
  constexpr int NWV = 8, PD = 2;  // waves sharing K; tiles in flight
  constexpr int RB = 128;         // bytes of an LDS row: 64 k
  constexpr int XB = 16 * RB, WB = NB * 16 * RB;  // one piece of x; the weights
  constexpr int WAVE_LDS = 2 * XB + WB;
  constexpr int PART = NB * 64 * 16;
  constexpr int LDS = NWV * (WAVE_LDS > PART ? WAVE_LDS : PART);
  __shared__ __attribute__((aligned(1024))) char lds[LDS];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n0 = block * 16 * NB;
  const int K = a.K, steps = (K + 63) / 64, per = (steps + NWV - 1) / NWV;
  const int t0 = wave * per, t1 = min(steps, t0 + per);
  char *const mine = lds + wave * WAVE_LDS;

  // Rows past M or N and columns past K load as zeros.
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(a.x), 0, a.M * K * 4, 0x00027000);
  const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<char *>(reinterpret_cast<const char *>(a.w)) + (long)n0 * K * 2, 0, min(16 * NB, a.N - n0) * K * 2, 0x00027000);
  constexpr int XL = 4, WL = NB * 2;  // loads per tile: four x rows or eight weight rows each
  u32x4 xv[PD][XL], wv[PD][WL];
  const int kx = 4 * (lane & 15), kw = 8 * (lane & 7);
  auto load = [&](int t, u32x4 (&xs)[XL], u32x4 (&ws)[WL]) {
    const int k = t < t1 ? 64 * t : K;  // (past the range: zeros)
#pragma unroll
    for (int i = 0; i < WL; ++i)
      ws[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                  wr, k + kw < K ? ((8 * i + (lane >> 3)) * K + k + kw) * 2 : 0x7ffffff0, 0, 2 /* nt */));
#pragma unroll
    for (int i = 0; i < XL; ++i)
      xs[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                  xr, k + kx < K ? ((4 * i + (lane >> 4)) * K + k + kx) * 4 : 0x7ffffff0, 0, 0));
  };
  f32x4 acc[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) acc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto f7 = [](int row) { return (row >> 1) & 7; };
  const int r = lane & 15;
  const int frag[2] = {r * RB + 16 * ((lane >> 4) ^ f7(r)), r * RB + 16 * ((4 + (lane >> 4)) ^ f7(r))};
  auto compute = [&](const u32x4 (&xs)[XL], const u32x4 (&ws)[WL]) {
#pragma unroll
    for (int i = 0; i < WL; ++i) {
      const int row = 8 * i + (lane >> 3);
      *reinterpret_cast<u32x4 *>(mine + 2 * XB + row * RB + 16 * ((lane & 7) ^ f7(row))) = ws[i];
    }
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int row = 4 * i + (lane >> 4), c = lane & 15;
      const float f[4] = {__uint_as_float(xs[i].x), __uint_as_float(xs[i].y), __uint_as_float(xs[i].z), __uint_as_float(xs[i].w)};
      unsigned h[2], l[2];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        h[e] = bf16x2_rne(f[2 * e], f[2 * e + 1]);
        l[e] = bf16x2_rne(f[2 * e] - __uint_as_float(h[e] << 16), f[2 * e + 1] - __uint_as_float(h[e] & 0xffff0000u));
      }
      char *d = mine + row * RB + 16 * ((c >> 1) ^ f7(row)) + 8 * (c & 1);
      *reinterpret_cast<uint2 *>(d) = make_uint2(h[0], h[1]);
      *reinterpret_cast<uint2 *>(d + XB) = make_uint2(l[0], l[1]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    bf16x8 fw[2][NB], fh[2], fl[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int j = 0; j < NB; ++j) fw[s][j] = *reinterpret_cast<const bf16x8 *>(mine + 2 * XB + j * 16 * RB + frag[s]);
      fh[s] = *reinterpret_cast<const bf16x8 *>(mine + frag[s]);
      fl[s] = *reinterpret_cast<const bf16x8 *>(mine + XB + frag[s]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[s][j], fh[s], acc[j], 0, 0, 0);
        acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[s][j], fl[s], acc[j], 0, 0, 0);
      }
  };
#pragma unroll
  for (int u = 0; u < PD; ++u) load(t0 + u, xv[u], wv[u]);
  for (int t = t0; t < t1; t += PD) {
#pragma unroll
    for (int u = 0; u < PD; ++u) {  // (tiles past the range are zeros)
      compute(xv[u], wv[u]);
      load(t + u + PD, xv[u], wv[u]);
    }
  }
  __syncthreads();
  f32x4 *part = reinterpret_cast<f32x4 *>(lds);
#pragma unroll
  for (int j = 0; j < NB; ++j) part[(wave * NB + j) * 64 + lane] = acc[j];
  __syncthreads();
  // D layout: element e of lane l is weight row 4 (l / 16) + e, token l % 16.
  if (threadIdx.x < 64 * NB) {
    const int i = threadIdx.x, l = i & 63, j = i >> 6, t = l & 15;
    f32x4 s = part[i];
#pragma unroll
    for (int w = 1; w < NWV; ++w) s += part[w * NB * 64 + i];
    if (t < a.M) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = n0 + 16 * j + 4 * (l >> 4) + e;
        if (n < a.N) a.out[(long)t * a.N + n] = (a.bias ? a.bias[n] : 0.0f) + s[e];
      }
    }
  }
}

// For 5 to 64 tokens (MB blocks of 16), bf16 weights, K % 128 == 0, short K: the
// least work between launch and store. A workgroup owns 16 weight rows; wave w of
// its four covers k in [w K/4, (w+1) K/4). Per 32-deep k step a lane loads 16
// bytes of one weight row (the A operand of v_mfma_f32_16x16x32_bf16: row lane %
// 16, k 8 (lane / 16) + [0, 8)) straight from HBM, and 8 activations of one token
// (the B operand) from the cache, split into bf16 hi and lo; both meet the
// weights. The four waves' partial sums are added through LDS.
template <int MB>
__global__ __launch_bounds__(256) void linear_short_kernel(const LinearArgs a) {
  __shared__ f32x4 part[4][MB][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int n0 = blockIdx.x * kShortRows;
  const int r = lane & 15, kq = lane >> 4;  // operand row/column, k quarter (8 of 32)
  const int kw = a.K / 4;
  const int k_begin = wave * kw, k_end = k_begin + kw;
  const char *wrow = reinterpret_cast<const char *>(a.w) + (long)min(n0 + r, a.N - 1) * a.K * 2;
  const float *xrow[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) xrow[b] = a.x + (long)min(16 * b + r, a.M - 1) * a.K;

  f32x4 acc[MB];
#pragma unroll
  for (int b = 0; b < MB; ++b) acc[b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

  auto step = [&](int kk) {
    const bf16x8 wf = *reinterpret_cast<const bf16x8 *>(wrow + (long)(kk + 8 * kq) * 2);
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const float4 x0 = *reinterpret_cast<const float4 *>(xrow[b] + kk + 8 * kq);
      const float4 x1 = *reinterpret_cast<const float4 *>(xrow[b] + kk + 8 * kq + 4);
      const float f[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
      unsigned h[4], l[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        h[i] = bf16x2_rne(f[2 * i], f[2 * i + 1]);
        l[i] = bf16x2_rne(f[2 * i] - __uint_as_float(h[i] << 16), f[2 * i + 1] - __uint_as_float(h[i] & 0xffff0000u));
      }
      const bf16x8 xh = __builtin_bit_cast(bf16x8, make_uint4(h[0], h[1], h[2], h[3]));
      const bf16x8 xl = __builtin_bit_cast(bf16x8, make_uint4(l[0], l[1], l[2], l[3]));
      acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xh, acc[b], 0, 0, 0);
      acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf, xl, acc[b], 0, 0, 0);
    }
  };
  constexpr int U = MB <= 2 ? 8 : 4;  // k steps in flight (registers allowing)
  int kk = k_begin;
  for (; kk + 32 * U <= k_end; kk += 32 * U) {
#pragma unroll
    for (int u = 0; u < U; ++u) step(kk + 32 * u);
  }
  for (; kk < k_end; kk += 32) step(kk);

#pragma unroll
  for (int b = 0; b < MB; ++b) part[wave][b][lane] = acc[b];
  __syncthreads();
  // D layout: element e of lane l is row (weight) 4 (l / 16) + e, column
  // (token) l % 16 of its block. Thread t < 64 * MB finishes block t / 64.
  if (threadIdx.x < 64 * MB) {
    const int b = threadIdx.x >> 6, l = threadIdx.x & 63;
    const f32x4 s = part[0][b][l] + part[1][b][l] + part[2][b][l] + part[3][b][l];
    const int t = 16 * b + (l & 15);
    if (t < a.M) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int n = n0 + 4 * (l >> 4) + e;
        if (n < a.N) a.out[(long)t * a.N + n] = (a.bias ? a.bias[n] : 0.0f) + s[e];
      }
    }
  }
}

// One thread per output: the sum starts at the bias and adds x[m][k] * w[n][k]
// in index order, each product rounded first (ops.rs:94-103; also the exact
// batch-1 row-block loop of streaming/kernels_raw16.rs:640-672).
template <typename WT>
__global__ __launch_bounds__(256) void linear_generic_kernel(const LinearArgs a) {
#pragma clang fp contract(off)
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long)a.M * a.N) return;
  const int m = (int)(idx / a.N), n = (int)(idx % a.N);
  const WT *w = reinterpret_cast<const WT *>(a.w) + (long)n * a.K;
  const float *x = a.x + (long)m * a.K;
  float sum = a.bias ? a.bias[n] : 0.0f;
  for (int k = 0; k < a.K; ++k) {
    float wf;
    if constexpr (sizeof(WT) == 4) wf = (float)w[k];
    else if constexpr (__is_same(WT, __bf16)) wf = __uint_as_float((unsigned)__builtin_bit_cast(unsigned short, w[k]) << 16);
    else wf = (float)w[k];
    const float p = x[k] * wf;
    sum = sum + p;
  }
  a.out[idx] = sum;
}

namespace {
// Pieces per lane (U) of linear_gemv_pass_kernel, or 0: 16-bit weight rows of up to
// 8 x 64 pieces, which a wave holds whole in registers. Eight pieces are never
// slower than gemv_rows (one token, 4096 weights a row: 200 rows 3.0 us against 4.7,
// 4096 7.7 / 8.4, 128256 151 / 162; two tokens 4.2 / 5.6 at 1024 rows, 9.3 / 9.6 at
// 4096; four 11.2 / 12.8 at 4096, 177 / 288 at 128256); from nine on, about 4096
// rows of one or two tokens are, by up to 5 and 11% (5120 weights a row; other
// sizes still gain). Longer rows stay with gemv_rows (3000 x 8192, one token: 10.9
// us, in passes of six pieces 11.7). Rows
// of one piece a lane or less gain nothing by being in flight whole, and a wave
// here has one of them where it has two there: from 2048 rows on they stay with
// gemv_rows (one token, against this kernel: 2048 x 256 the same, 4096 x 256 8%
// less, 16384 x 256 3.9 / 5.3 us, 65536 x 128 8.8 / 14.5), until three or four
// tokens have two rows a wave here as well and enough of them (16384 x 256 the
// same, 65536 x 256 4 to 11% more). With the norm, two tokens or more (768 x 256,
// the sublayer's q, k and v: 0.4 to 1.2 us less).
int gemv_pass_pieces(const LinearArgs &a, long rows) {
  const long u = (a.K / 8 + 63) / 64;
  if (a.dtype == SPISSA_DTYPE_F32 || u > 8) return 0;
  if (u == 1 && (a.norm_w ? a.M >= 2 : rows > 2048 && !(a.M >= 3 && rows > 16384))) return 0;
  return (int)std::max(2L, u);
}

template <typename WT, int NB, int RW, bool NORM, int U = 2>
void launch_gemv_pass_as(hipStream_t st, const LinearSegments &m, int pieces, unsigned grid) {
  if constexpr (U <= 8) {
    if (pieces != U) return launch_gemv_pass_as<WT, NB, RW, NORM, U + 1>(st, m, pieces, grid);
    hipLaunchKernelGGL((linear_gemv_pass_kernel<WT, NB, U, RW, NORM>), dim3(grid), dim3(256), 0, st, m);
  }
}
// One row per wave: more waves cover the latency, and x is no longer read per
// wave (one token, two rows: 512 x 2048 2.73 us against 2.45, 128256 x 3072 119.0
// against 116.6). Three and four tokens read more of x from LDS than weights, and
// with the norm form it with more arithmetic: two rows there above 4096 rows
// (four tokens, 8000 x 2048: 8.86 against 9.52) or with the norm (5120 x 3072
// 12.0 against 13.0, but 512 x 2048 5.68 against 5.07; gemv_rows 6.76).
template <typename WT, int NB>
hipError_t launch_gemv_pass(hipStream_t st, LinearSegments &m, int pieces) {
  const bool norm = m.seg[0].norm_w != nullptr;
  long rows = 0, grid = 0;
  for (int i = 0; i < m.n; ++i) rows += m.seg[i].N;
  const int rw = NB >= 3 && (norm || rows > 4096) ? 2 : 1;
  for (int i = 0; i < m.n; ++i) grid += m.blocks[i] = (m.seg[i].N + 4 * rw - 1) / (4 * rw);
  if constexpr (NB >= 3) {
    if (norm)
      launch_gemv_pass_as<WT, NB, 2, true>(st, m, pieces, (unsigned)grid);
    else if (rw == 2)
      launch_gemv_pass_as<WT, NB, 2, false>(st, m, pieces, (unsigned)grid);
    else
      launch_gemv_pass_as<WT, NB, 1, false>(st, m, pieces, (unsigned)grid);
  } else if (norm) {
    launch_gemv_pass_as<WT, NB, 1, true>(st, m, pieces, (unsigned)grid);
  } else {
    launch_gemv_pass_as<WT, NB, 1, false>(st, m, pieces, (unsigned)grid);
  }
  return hipGetLastError();
}
template <typename WT>
hipError_t launch_gemv_pass(hipStream_t st, LinearSegments &m, int pieces) {
  switch (m.seg[0].M) {
    case 1: return launch_gemv_pass<WT, 1>(st, m, pieces);
    case 2: return launch_gemv_pass<WT, 2>(st, m, pieces);
    case 3: return launch_gemv_pass<WT, 3>(st, m, pieces);
    case 4: return launch_gemv_pass<WT, 4>(st, m, pieces);
    default: return hipErrorInvalidValue;
  }
}

template <typename WT>
hipError_t launch_gemv(hipStream_t st, const LinearArgs &a) {
  if constexpr (sizeof(WT) == 2) {
    if (const int pieces = gemv_pass_pieces(a, a.N)) {
      LinearSegments m{};
      m.n = 1;
      m.seg[0] = a;
      return launch_gemv_pass<WT>(st, m, pieces);
    }
  }
  const unsigned grid = (unsigned)((a.N + 4 * kGemvRowsPerWave - 1) / (4 * kGemvRowsPerWave));
  switch (a.M) {
    case 1: hipLaunchKernelGGL((linear_gemv_kernel<WT, 1>), dim3(grid), dim3(256), 0, st, a); break;
    case 2: hipLaunchKernelGGL((linear_gemv_kernel<WT, 2>), dim3(grid), dim3(256), 0, st, a); break;
    case 3: hipLaunchKernelGGL((linear_gemv_kernel<WT, 3>), dim3(grid), dim3(256), 0, st, a); break;
    case 4: hipLaunchKernelGGL((linear_gemv_kernel<WT, 4>), dim3(grid), dim3(256), 0, st, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
template <typename WT>
hipError_t launch_gemv_multi(hipStream_t st, LinearSegments &m) {
  long total = 0;
  if constexpr (sizeof(WT) == 2) {
    long rows = 0;
    for (int i = 0; i < m.n; ++i) rows += m.seg[i].N;
    if (const int pieces = gemv_pass_pieces(m.seg[0], rows)) return launch_gemv_pass<WT>(st, m, pieces);
  }
  for (int i = 0; i < m.n; ++i) total += m.blocks[i] = (m.seg[i].N + 4 * kGemvRowsPerWave - 1) / (4 * kGemvRowsPerWave);
  switch (m.seg[0].M) {
    case 1: hipLaunchKernelGGL((linear_gemv_multi_kernel<WT, 1>), dim3((unsigned)total), dim3(256), 0, st, m); break;
    case 2: hipLaunchKernelGGL((linear_gemv_multi_kernel<WT, 2>), dim3((unsigned)total), dim3(256), 0, st, m); break;
    case 3: hipLaunchKernelGGL((linear_gemv_multi_kernel<WT, 3>), dim3((unsigned)total), dim3(256), 0, st, m); break;
    case 4: hipLaunchKernelGGL((linear_gemv_multi_kernel<WT, 4>), dim3((unsigned)total), dim3(256), 0, st, m); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
template <typename WT>
hipError_t launch_generic_linear(hipStream_t st, const LinearArgs &a) {
  const long n = (long)a.M * a.N;
  hipLaunchKernelGGL((linear_generic_kernel<WT>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a);
  return hipGetLastError();
}
template <int BM, int BN, int WM, int WN, int MINWG, bool WIDE>
hipError_t launch_gemm(hipStream_t st, const LinearArgs &a) {
  const long grid = (((long)a.M + BM - 1) / BM) * (((long)a.N + BN - 1) / BN);
  hipLaunchKernelGGL((linear_gemm_kernel<BM, BN, WM, WN, MINWG, WIDE>), dim3((unsigned)grid), dim3(512), 0, st, a);
  return hipGetLastError();
}
template <typename WT>
hipError_t launch_typed(hipStream_t st, const LinearArgs &a, int path) {
  if (path == kLinearGemv) return launch_gemv<WT>(st, a);
  return launch_generic_linear<WT>(st, a);
}
}  // namespace

int linear_path(int dtype, long M, long N, long K) {
  const int epc = dtype == SPISSA_DTYPE_F32 ? 4 : 8;
  if (M <= 4) return K % epc == 0 ? kLinearGemv : kLinearGeneric;
  const bool bf16_tiles = dtype == SPISSA_DTYPE_BF16 && K % kBK == 0;
  // Up to 16 tokens the tile kernel would need K split over workgroups and a
  // second launch (5120 x 3072: 14.1 against 11.9 us; at 24 tokens it is the
  // other way round, 14.7 against 15.7). (The skinny kernel addresses 16 rows of
  // x and 32 of the weights with 32-bit byte offsets, the output with 64.)
  if (bf16_tiles && M <= 16 && K <= 1 << 21 && N <= 1 << 26) return kLinearSkinny;
  // The tile kernel addresses up to 128 rows of an operand and of the output
  // with 32-bit byte offsets. bf16 weights past that, whose K is whole 32-deep k
  // tiles, have the GEMM, which addresses with 64 bits. Sizes that are not such
  // tiles of bf16 weights take the tile kernel from 2^20 products. Below that they
  // keep the one-thread-per-output kernel for its result, the reference's sum bit
  // for bit, not for its time, which is one chain of K steps (f16 weights, against
  // the tile kernel: 8 x 200 x 8 2.5 / 3.5 us, 8 x 64 x 256 31 / 6.5, 8 x 40 x 2000
  // 245 / 8.6, 8 x 8 x 16384 1196 / 21).
  if (K % epc != 0 || K > 1 << 21 || N > 1 << 21) return bf16_tiles ? kLinearGemm : kLinearGeneric;
  return bf16_tiles || (double)M * N * K >= 1048576.0 ? kLinearTile : kLinearGeneric;
}

// Whether K is short enough for linear_short_kernel: it starts and ends sooner
// than the kernels that pass both operands through LDS, and has less in flight.
// 16 tokens or fewer, against the skinny kernel (us): 5 x 512 x 512 3.2 / 4.2, 16 x
// 16384 x 256 5.8 / 6.1, 5 x 262144 x 128 20.9 / 49.1 (its eight waves share K), 5
// x 200 x 1152 4.2 / 5.2 but 16 x 512 x 1024 5.0 / 4.7; 5 x 2048 x 768 the same, 16
// x 2048 x 1024 5.8 / 4.9. Up to 64, against the tile kernel: 17 x 512 x 512 4.5 /
// 6.7, 32 x 4096 x 1024 8.1 / 10.0, 48 x 2048 x 768 8.0 / 8.5, 64 x 4096 x 512 the
// same, 32 x 8192 x 512 the same, 17 x 16384 x 256 9% slower.
static bool linear_k_short(long M, long N, long K) {
  if (K % 128 != 0 || M > 64 || N > 1 << 26) return false;
  if (M <= 16) return K <= (M <= 8 && N <= 512 ? 1280 : 512);
  const long blocks = (M + 15) / 16;
  return K <= 1536 - 256 * blocks && N <= (blocks == 2 && K <= 512 ? 8192 : 4096);
}

int linear_few_path(int path, long M, long N, long K) {
  if (linear_k_short(M, N, K)) return kLinearShort;
  // Other short K on large N keep the skinny kernel's eight waves idle: 5 x
  // 65536 x 96 12.0 us against the tile kernel's 5.7; 16384 rows the same.
  // (Past the tile kernel's 32-bit offsets, the GEMM.)
  if (path == kLinearSkinny && K <= 512 && N > 24576) return N <= 1 << 21 ? kLinearTile : kLinearGemm;
  return path;
}

hipError_t launch_linear_multi(hipStream_t st, const LinearArgs *segs, int n, int path, int cus) {
  if (n < 1 || n > kMaxLinearSegments || (path != kLinearGemv && path != kLinearSkinny)) return hipErrorInvalidValue;
  LinearSegments m{};
  m.n = n;
  if (path == kLinearSkinny) {
    if (segs[0].dtype != SPISSA_DTYPE_BF16 || segs[0].K % 8 != 0 || segs[0].M > 16) return hipErrorInvalidValue;
    // 16 weight rows per workgroup while each gets a CU of its own, else 32
    // (3072 rows: 8.8 us against 11.3 with 32; 5120: 14.5 against 11.9)
    long rows = 0;
    for (int i = 0; i < n; ++i) rows += segs[i].N;
    const int nb = rows <= 16L * cus ? 1 : 2;
    long grid = 0;
    for (int i = 0; i < n; ++i) {
      m.seg[i] = segs[i];
      m.blocks[i] = (segs[i].N + 16 * nb - 1) / (16 * nb);
      grid += m.blocks[i];
    }
    if (nb == 1)
      hipLaunchKernelGGL(linear_skinny_kernel<1>, dim3((unsigned)grid), dim3(512), 0, st, m);
    else
      hipLaunchKernelGGL(linear_skinny_kernel<2>, dim3((unsigned)grid), dim3(512), 0, st, m);
    return hipGetLastError();
  }
  for (int i = 0; i < n; ++i) m.seg[i] = segs[i];
  switch (segs[0].dtype) {
    case SPISSA_DTYPE_F32: return launch_gemv_multi<float>(st, m);
    case SPISSA_DTYPE_BF16: return launch_gemv_multi<__bf16>(st, m);
    case SPISSA_DTYPE_F16: return launch_gemv_multi<_Float16>(st, m);
    default: return hipErrorInvalidValue;
  }
}

// Estimated times (us) of the two GEMM shapes and of the tile kernel's plan, as
// measured by graph replay with weights from HBM over 3824 shapes (17 to 8192
// tokens, 64 to 262144 rows, K 32 to 8192): launch, store of the output, and
// what a k tile's step takes at `load` workgroups a CU, a partly empty round
// included. Weights past the last-level cache cost the GEMMs, whose tile order
// runs along the weights, a further tenth. The shape so chosen is on average
// 0.1% and at most 12% above the fastest of the three, and in two of the shapes
// more than 3% above the choice between the GEMM shapes by rounds alone that
// came before the tile kernel.
int linear_prompt_path(const LinearTilePlan &tile, long M, long N, long K, int cus) {
  const double c = cus > 0 ? cus : 256, mb = 4e-6 * M * N, nk = (double)(K / kBK);
  const double far = 2e-6 * N * K > 200.0 ? 1.15 : 1.03;
  double load = (double)((M + 255) / 256) * ((N + 319) / 320) / c;
  const double wide = far * (6.0 + 0.11 * mb + nk * (load <= 1.0 ? std::max(1.68, 0.9 + 1.35 * load)
                                                                 : 1.2 * std::ceil(load) + 0.95 * load));
  load = (double)((M + 127) / 128) * ((N + 255) / 256) / c;
  const double half = far * (3.5 + 0.11 * mb + nk * (load <= 1.0   ? 0.72 + 0.47 * load
                                                        : load <= 2.0 ? 0.744 + 0.542 * load
                                                                      : 0.47 * (std::ceil(load) + load)));
  int rows, columns;
  linear_tile_dims(tile, &rows, &columns);
  const double tiles = tile.us * (rows == 32 ? 1.15 : 1.0) + 0.2 * mb - 1.0;
  if (tiles <= std::min(wide, half)) return kLinearTile;
  return half <= wide ? kLinearGemmHalf : kLinearGemm;
}

hipError_t launch_linear(hipStream_t st, const LinearArgs &a, int path, int cus) {
  if (a.M <= 0 || a.N <= 0) return hipSuccess;
  if (a.norm_w && path != kLinearGemv) return hipErrorInvalidValue;  // the folded norm is the GEMV's
  if (path == kLinearSkinny) return launch_linear_multi(st, &a, 1, path, cus);
  if (path == kLinearGemm || path == kLinearGemmHalf) {
    if (a.dtype != SPISSA_DTYPE_BF16 || a.K % kBK != 0) return hipErrorInvalidValue;
    // (256 rows of 2^21 floats are 2^31 bytes: the store buffer's range is an int)
    if (a.N >= 1 << 21) return launch_gemm<256, 320, 4, 2, 1, true>(st, a);
    return path == kLinearGemm ? launch_gemm<256, 320, 4, 2, 1, false>(st, a) : launch_gemm<128, 256, 2, 4, 2, false>(st, a);
  }
  if (path == kLinearShort) {
    if (a.dtype != SPISSA_DTYPE_BF16 || a.K % 128 != 0 || a.M > 64) return hipErrorInvalidValue;
    const dim3 grid((unsigned)((a.N + kShortRows - 1) / kShortRows));
    switch ((a.M + 15) / 16) {
      case 1: hipLaunchKernelGGL(linear_short_kernel<1>, grid, dim3(256), 0, st, a); break;
      case 2: hipLaunchKernelGGL(linear_short_kernel<2>, grid, dim3(256), 0, st, a); break;
      case 3: hipLaunchKernelGGL(linear_short_kernel<3>, grid, dim3(256), 0, st, a); break;
      default: hipLaunchKernelGGL(linear_short_kernel<4>, grid, dim3(256), 0, st, a); break;
    }
    return hipGetLastError();
  }
  switch (a.dtype) {
    case SPISSA_DTYPE_F32: return launch_typed<float>(st, a, path);
    case SPISSA_DTYPE_BF16: return launch_typed<__bf16>(st, a, path);
    case SPISSA_DTYPE_F16: return launch_typed<_Float16>(st, a, path);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace spissa
