// linear_tile.hip -- the projections between the decode GEMV and the
// large-prompt GEMM (linear.hip): batches, chunks and short prompts, weights
// stored as f16 or f32 at more than four tokens, and the q, k and v weights of
// a layer in one launch.
//
// out = x W^T on v_mfma_f32_32x32x16_bf16, both operands as sums of bf16
// pieces (piece 0 the nearest bf16, each next one the nearest bf16 of what is
// left), accumulated in f32:
//   bf16 weights: x as two pieces, products x0 w + x1 w (the split leaves
//     2^-18 of x), as the other kernels of bf16 weights above four tokens have
//     it; three (exact) when K % 32 != 0, which they do not take: those sums
//     were the one-thread-per-output kernel's, in whole f32 products;
//   f16 weights: w as two pieces (exact), x as three (exact), the five
//     products above the f32 rounding of one product;
//   f32 weights: w and x as three pieces, six products.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "internal.hpp"

namespace spissa {

namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

constexpr int kTBK = 32;              // k tile
constexpr int kTRow = kTBK * 2;       // bytes of one bf16 LDS row: four 16-byte chunks
constexpr unsigned kOutside = 0x7ffffff0u;  // a buffer offset past every range: the load returns zeros

// Chunk swizzle of a 64-byte LDS row (any 8 aligned consecutive rows reading
// one chunk hit 8 distinct 16-byte groups modulo 128 bytes).
__device__ __forceinline__ int tile_swz(int row) { return ((row >> 1) ^ (row >> 2)) & 3; }

// (rne(a), rne(b)) as bf16 bits, a in the low half.
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

// The bf16 pieces of two f32 values, the first value's in the low halves.
template <int NP>
__device__ __forceinline__ void split2(float a, float b, unsigned (&p)[NP]) {
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    p[i] = pack_bf16(a, b);
    if (i + 1 < NP) {
      a -= __uint_as_float(p[i] << 16);
      b -= __uint_as_float(p[i] & 0xffff0000u);
    }
  }
}

// Per weight type: bf16 pieces of a weight, and weights per 16 bytes. An
// activation is NX pieces; the products of pieces i (activation) and j (weight)
// with i + j < NX are taken.
template <typename WT>
struct TileW;
template <>
struct TileW<__bf16> {
  static constexpr int NW = 1, EPC = 8;
};
template <>
struct TileW<_Float16> {
  static constexpr int NW = 2, EPC = 8;
};
template <>
struct TileW<float> {
  static constexpr int NW = 3, EPC = 4;
};

__device__ __forceinline__ u32x4 load16(__amdgpu_buffer_rsrc_t r, unsigned off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)off, 0, 0));
}

__device__ __forceinline__ void tile_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// f(u, s0) for u = 0 .. N-1, straight-line.
template <int N, int U = 0, typename F>
__device__ __forceinline__ void unrolled_steps(F &f, int s0) {
  if constexpr (U < N) {
    f(std::integral_constant<int, U>(), s0);
    unrolled_steps<N, U + 1>(f, s0);
  }
}
// The same while s0 + u < n. (Exits only: a branch that rejoins between the
// steps would make the compiler's waits cover the path that skipped them, and
// so leave one step of loads in flight instead of the ring's.)
template <int N, int U = 0, typename F>
__device__ __forceinline__ void remaining_steps(F &f, int s0, int n) {
  if constexpr (U < N) {
    if (s0 + U >= n) return;
    f(std::integral_constant<int, U>(), s0);
    remaining_steps<N, U + 1>(f, s0, n);
  }
}

// One output in the reference's order (ops.rs:94-103), as linear_generic_kernel forms it.
template <typename WT>
__device__ __forceinline__ float dot_in_order(const LinearArgs &a, int m, int n) {
#pragma clang fp contract(off)
  const WT *w = reinterpret_cast<const WT *>(a.w) + (long)n * a.K;
  const float *x = a.x + (long)m * a.K;
  float sum = a.bias ? a.bias[n] : 0.0f;
#pragma clang loop unroll(disable)
  for (int k = 0; k < a.K; ++k) {
    float wf;
    if constexpr (__is_same(WT, __bf16))
      wf = __uint_as_float((unsigned)__builtin_bit_cast(unsigned short, w[k]) << 16);
    else
      wf = (float)w[k];
    const float p = x[k] * wf;
    sum = sum + p;
  }
  return sum;
}

}  // namespace

// Workgroups of WM x WN waves, each (BM / WM) x (BN / WN) outputs in 32 x 32
// blocks, on one of `splits` ranges of K. Per 32-deep k tile t, in one step:
// the tile's two 16-deep MFMA steps, whose operands were read from LDS one
// step ahead; the reads of the operands that follow, tile t + 1's first
// included; the split of tile t + 2, from registers into the LDS buffer that
// tile t - 1 left (three buffers); and the loads of tile t + 2 + PD into the
// registers that freed (PD tiles in flight). Interleaved by
// sched_group_barrier, one barrier per step, which waits for LDS only.
// What bounds it: at one or two waves per SIMD, the issue of the splits and
// LDS reads beside the MFMAs (64 x 128 tiles of bf16 weights: 110
// instructions a step against eight MFMAs of 32 cycles).
// Packing the split activations with a launch of their own, in operand order,
// and loading them straight into registers took longer in all for bf16
// weights (1500 x 1536 x 1152: 17.2 us + 6.1 for the packing, against 18.9).
template <typename WT, int NX, int BM, int BN, int WM, int WN, int PD, int MINW>
__global__ __launch_bounds__(WM * WN * 64, MINW) void linear_tile_kernel(const LinearTileArgs t) {
  constexpr int NT = WM * WN * 64;
  constexpr int NW = TileW<WT>::NW, EPC = TileW<WT>::EPC;
  constexpr int TM = BM / WM, TN = BN / WN, BI = TM / 32, BJ = TN / 32;
  static_assert(BI * 32 * WM == BM && BJ * 32 * WN == BN, "32 x 32 blocks");
  constexpr int XL = BM * kTBK / 4 / NT;          // 16-byte activation loads per thread and k tile
  constexpr int CPR = kTBK / EPC;                 // 16-byte pieces of a weight row's k tile
  constexpr int WL = BN * CPR / NT;               // weight loads per thread and k tile
  static_assert(XL * NT * 4 == BM * kTBK && WL * NT == BN * CPR, "whole loads");
  static_assert(PD % 3 == 0, "the buffer of a step is its index modulo 3");
  __shared__ __attribute__((aligned(1024))) char x_lds0[NX][BM * kTRow], w_lds0[NW][BN * kTRow];
  __shared__ __attribute__((aligned(1024))) char x_lds1[NX][BM * kTRow], w_lds1[NW][BN * kTRow];
  __shared__ __attribute__((aligned(1024))) char x_lds2[NX][BM * kTRow], w_lds2[NW][BN * kTRow];

  // Workgroup -> (split, m tile, segment, n tile). Ids equal modulo 8 run on
  // one XCD: each takes a contiguous run of the tile order.
  int id = blockIdx.x;
  {
    const int g = gridDim.x, q = g >> 3, r = g & 7, xcd = id & 7;
    id = xcd * q + min(xcd, r) + (id >> 3);
  }
  const int tiles = t.tiles_m * t.tiles_n;
  const int split = id / tiles;
  id -= split * tiles;
  int tm, tn;
  if (t.m_fast) {
    tn = id / t.tiles_m;
    tm = id - tn * t.tiles_m;
  } else {
    tm = id / t.tiles_n;
    tn = id - tm * t.tiles_n;
  }
  int sg = 0;
  while (sg + 1 < t.nseg && tn >= t.seg_tiles[sg]) tn -= t.seg_tiles[sg++];
  const LinearArgs &a = t.seg[sg];
  const int K = a.K, m0 = tm * BM, n0 = tn * BN;
  const int k_begin = split * t.kps, k_end = min(K, k_begin + t.kps);
  const int nsteps = (k_end - k_begin + kTBK - 1) / kTBK;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wm = wave / WN, wn = wave % WN, lr = lane & 31, hl = lane >> 5;

  // Rows past M or N lie past the buffers' ends and load as zeros, as do the
  // columns past k_end (their offset is replaced).
  const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float *>(a.x) + (long)m0 * K, 0, min(BM, a.M - m0) * K * 4, 0x00027000);
  const __amdgpu_buffer_rsrc_t wr =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(reinterpret_cast<const char *>(a.w)) + (long)n0 * K * (long)sizeof(WT),
                                        0, min(BN, a.N - n0) * K * (int)sizeof(WT), 0x00027000);
  u32x4 xv[PD][XL], wv[PD][WL];
  auto load = [&](int step, u32x4 (&xs)[XL], u32x4 (&ws)[WL]) {
    const int k = k_begin + step * kTBK;
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int s = tid + NT * i, row = s >> 3, kk = k + 4 * (s & 7);
      xs[i] = load16(xr, kk < k_end ? (unsigned)(row * K + kk) * 4u : kOutside);
    }
#pragma unroll
    for (int i = 0; i < WL; ++i) {
      const int s = tid + NT * i, row = s / CPR, kk = k + EPC * (s % CPR);
      ws[i] = load16(wr, kk < k_end ? (unsigned)(row * K + kk) * (unsigned)sizeof(WT) : kOutside);
    }
  };
  auto store = [&](const u32x4 (&xs)[XL], const u32x4 (&ws)[WL], char (*xd)[BM * kTRow], char (*wd)[BN * kTRow]) {
#pragma unroll
    for (int i = 0; i < XL; ++i) {
      const int s = tid + NT * i, row = s >> 3, c = s & 7;
      unsigned p0[NX], p1[NX];
      split2<NX>(__uint_as_float(xs[i].x), __uint_as_float(xs[i].y), p0);
      split2<NX>(__uint_as_float(xs[i].z), __uint_as_float(xs[i].w), p1);
      const int off = row * kTRow + 16 * ((c >> 1) ^ tile_swz(row)) + 8 * (c & 1);
#pragma unroll
      for (int j = 0; j < NX; ++j) *reinterpret_cast<uint2 *>(xd[j] + off) = make_uint2(p0[j], p1[j]);
    }
#pragma unroll
    for (int i = 0; i < WL; ++i) {
      const int s = tid + NT * i, row = s / CPR, c = s % CPR;
      if constexpr (__is_same(WT, float)) {
        unsigned p0[NW], p1[NW];
        split2<NW>(__uint_as_float(ws[i].x), __uint_as_float(ws[i].y), p0);
        split2<NW>(__uint_as_float(ws[i].z), __uint_as_float(ws[i].w), p1);
        const int off = row * kTRow + 16 * ((c >> 1) ^ tile_swz(row)) + 8 * (c & 1);
#pragma unroll
        for (int j = 0; j < NW; ++j) *reinterpret_cast<uint2 *>(wd[j] + off) = make_uint2(p0[j], p1[j]);
      } else {
        const int off = row * kTRow + 16 * (c ^ tile_swz(row));
        if constexpr (__is_same(WT, _Float16)) {
          u32x4 o[NW];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const unsigned u = ws[i][e];
            unsigned p[NW];
            split2<NW>((float)__builtin_bit_cast(_Float16, (unsigned short)(u & 0xffffu)),
                       (float)__builtin_bit_cast(_Float16, (unsigned short)(u >> 16)), p);
#pragma unroll
            for (int j = 0; j < NW; ++j) o[j][e] = p[j];
          }
#pragma unroll
          for (int j = 0; j < NW; ++j) *reinterpret_cast<u32x4 *>(wd[j] + off) = o[j];
        } else {
          *reinterpret_cast<u32x4 *>(wd[0] + off) = ws[i];
        }
      }
    }
  };

  f32x16 acc[BI][BJ];
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  // Fragments of 16 k (k step S of a tile): row lr of a 32-row block, chunk 2 S + hl.
  const int xa = (wm * TM + lr) * kTRow, wa = (wn * TN + lr) * kTRow;  // (+32 rows leave tile_swz unchanged)
  const int ch0 = 16 * (hl ^ tile_swz(lr)), ch1 = 16 * ((2 + hl) ^ tile_swz(lr));
  struct Frags {
    bf16x8 x[NX][BI], w[NW][BJ];
  };
  auto read = [&](Frags &f, const char (*xs)[BM * kTRow], const char (*ws)[BN * kTRow], int ch) {
#pragma unroll
    for (int p = 0; p < NX; ++p)
#pragma unroll
      for (int b = 0; b < BI; ++b) f.x[p][b] = *reinterpret_cast<const bf16x8 *>(xs[p] + xa + b * 32 * kTRow + ch);
#pragma unroll
    for (int p = 0; p < NW; ++p)
#pragma unroll
      for (int b = 0; b < BJ; ++b) f.w[p][b] = *reinterpret_cast<const bf16x8 *>(ws[p] + wa + b * 32 * kTRow + ch);
  };
  auto multiply = [&](const Frags &f) {
#pragma unroll
    for (int px = 0; px < NX; ++px)
#pragma unroll
      for (int pw = 0; pw < NW; ++pw)
        if (px + pw < NX) {
#pragma unroll
          for (int i = 0; i < BI; ++i)
#pragma unroll
            for (int j = 0; j < BJ; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.x[px][i], f.w[pw][j], acc[i][j], 0, 0, 0);
        }
  };

  // Tiles 0 and 1 in LDS, tile 0's first fragments in registers, tiles 2 .. PD+1 in flight.
#pragma unroll
  for (int u = 0; u < PD; ++u) load(u, xv[u], wv[u]);
  store(xv[0], wv[0], x_lds0, w_lds0);
  load(PD, xv[0], wv[0]);
  store(xv[1], wv[1], x_lds1, w_lds1);
  load(PD + 1, xv[1], wv[1]);
  tile_barrier();
  Frags f0, f1;
  read(f0, x_lds0, w_lds0, ch0);
  constexpr int NP = NX * NW - (NW > 1 ? (NW == 2 ? 1 : 3) : 0);  // products per fragment pair
  constexpr int NM = NP * BI * BJ, NR = NX * BI + NW * BJ;
  constexpr int NDW = XL * NX + WL * NW;
  // One step on tile t (buffer t % 3): MFMAs of its two k steps next to the
  // reads of the fragments that follow, the split and store of tile t + 2
  // (whose buffer held tile t - 1) and the loads of tile t + 2 + PD.
  auto step = [&](auto u_, int s0) {
    constexpr int u = decltype(u_)::value, st = (u + 2) % PD;
    char(*const xc)[BM * kTRow] = u % 3 == 0 ? x_lds0 : u % 3 == 1 ? x_lds1 : x_lds2;
    char(*const wc)[BN * kTRow] = u % 3 == 0 ? w_lds0 : u % 3 == 1 ? w_lds1 : w_lds2;
    char(*const xn)[BM * kTRow] = u % 3 == 2 ? x_lds0 : u % 3 == 0 ? x_lds1 : x_lds2;
    char(*const wn_)[BN * kTRow] = u % 3 == 2 ? w_lds0 : u % 3 == 0 ? w_lds1 : w_lds2;
    char(*const xf)[BM * kTRow] = u % 3 == 1 ? x_lds0 : u % 3 == 2 ? x_lds1 : x_lds2;
    char(*const wf)[BN * kTRow] = u % 3 == 1 ? w_lds0 : u % 3 == 2 ? w_lds1 : w_lds2;
    read(f1, xc, wc, ch1);
    multiply(f0);
    store(xv[st], wv[st], xf, wf);
    load(s0 + u + 2 + PD, xv[st], wv[st]);
    read(f0, xn, wn_, ch0);
    multiply(f1);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int i = 0; i < NM; ++i) {
        constexpr int RP = (NR + NM - 1) / NM > 2 ? (NR + NM - 1) / NM : 2;
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                       // MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, RP, 0);                      // LDS reads
        __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);                       // VALU
        __builtin_amdgcn_sched_group_barrier(0x200, (NDW + NM - 1) / NM, 0);     // LDS writes
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);                       // loads
      }
    }
    tile_barrier();
  };
  int s0 = 0;
  for (; s0 + PD <= nsteps; s0 += PD) unrolled_steps<PD>(step, s0);
  remaining_steps<PD - 1>(step, s0, nsteps);

  // Accumulator layout: element e of lane l is row 8 (e / 4) + 4 hl + e % 4
  // (token), column lr (output) of its 32 x 32 block. Stores go through a
  // buffer that ends with row M - 1 (rows past it are dropped, columns past N
  // get an offset past its end), with no branch and no argument read between
  // them: a test per element had taken 10 us of a launch of 64 x 128 tiles.
  const bool part = t.splits > 1;
  const int M = a.M, N = a.N, pitch = part ? t.n_total : N;
  float *const obase = (part ? t.partial + (long)split * M * t.n_total + t.seg_off[sg] : a.out) + (long)m0 * pitch;
  const __amdgpu_buffer_rsrc_t ob =
      __builtin_amdgcn_make_buffer_rsrc(obase, 0, ((min(BM, M - m0) - 1) * pitch + N) * 4, 0x00027000);
  bool nan = false;
#pragma unroll
  for (int i = 0; i < BI; ++i)
#pragma unroll
    for (int j = 0; j < BJ; ++j) {
      const int n = n0 + wn * TN + 32 * j + lr;
      const float bn = a.bias && !part ? a.bias[min(n, N - 1)] : 0.0f;
      const unsigned o0 = n < N ? (unsigned)((wm * TM + 32 * i + 4 * hl) * pitch + n) * 4u : 0x80000000u;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float v = bn + acc[i][j][e];
        nan |= v != v;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), ob,
                                              (int)(o0 + (unsigned)((8 * (e >> 2) + (e & 3)) * pitch) * 4u), 0, 0);
      }
    }
  // Infinite or huge values split into pieces of both signs; such outputs (and
  // true NaNs) are formed again in the reference's order.
  if (t.in_order_nan && !part && nan) {
#pragma clang loop unroll(disable)
    for (int j = 0; j < BJ; ++j) {
      const int n = n0 + wn * TN + 32 * j + lr;
#pragma clang loop unroll(disable)
      for (int i = 0; i < BI * 16; ++i) {
        const int m = m0 + wm * TM + 4 * hl + 32 * (i >> 4) + 8 * ((i >> 2) & 3) + (i & 3);
        if (n < N && m < M) {
          const float v = a.out[(long)m * N + n];
          if (v != v) a.out[(long)m * N + n] = dot_in_order<WT>(a, m, n);
        }
      }
    }
  }
}

// out = bias + the splits' partial sums in split order, VEC columns per
// thread (4 when the segments and rows allow 16-byte accesses). Grid:
// (ceil(columns / (256 VEC)), M).
template <typename WT, int VEC>
__global__ __launch_bounds__(256) void linear_tile_reduce_kernel(const LinearTileArgs t) {
  typedef __attribute__((ext_vector_type(VEC))) float vec;
  const int c = (blockIdx.x * 256 + threadIdx.x) * VEC, m = blockIdx.y;
  if (c >= t.n_total) return;
  const long stride = (long)t.seg[0].M * t.n_total;
  const float *p = t.partial + (long)m * t.n_total + c;
  vec v = *reinterpret_cast<const vec *>(p);
  int s = 1;
  for (; s + 4 <= t.splits; s += 4) {
    vec q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = *reinterpret_cast<const vec *>(p + (s + i) * stride);
#pragma unroll
    for (int i = 0; i < 4; ++i) v += q[i];
  }
  for (; s < t.splits; ++s) v += *reinterpret_cast<const vec *>(p + s * stride);
  int sg = 0;
  while (sg + 1 < t.nseg && c >= t.seg_off[sg + 1]) ++sg;
  const LinearArgs &a = t.seg[sg];
  const int n = c - t.seg_off[sg];
#pragma unroll
  for (int i = 0; i < VEC; ++i) {
    float r = v[i] + (a.bias ? a.bias[n + i] : 0.0f);
    if (t.in_order_nan && r != r) r = dot_in_order<WT>(a, m, n + i);
    v[i] = r;
  }
  *reinterpret_cast<vec *>(a.out + (long)m * a.N + n) = v;
}

namespace {

// The tile shapes and what a k tile's step takes (us, bf16 weights): lat on a
// CU that holds one workgroup; share times the workgroups per CU when the CUs
// are full, a last round that is partly empty counting as `part` of one.
// Measured on 14 shapes from 64 x 1024 to 8192 x 5120 (within 10% of the times
// below for most); the other weight types take `slow` times as long.
struct TileShape {
  int bm, bn;
  float lat, share, part;
};
constexpr TileShape kTileShapes[] = {
    {32, 128, 0.19f, 0.24f, 0.7f},   // 1 x 4 waves
    {64, 128, 0.29f, 0.34f, 0.7f},   // 2 x 2 waves
    {128, 128, 0.41f, 0.56f, 0.8f},  // 4 x 2 waves
    {128, 256, 0.72f, 0.97f, 0.8f},  // 2 x 4 waves, bf16 weights (LDS)
};
constexpr int kMaxTileSplits = 16;

template <typename WT, int NX, int BM, int BN, int WM, int WN, int PD, int MINW>
hipError_t launch_tile(hipStream_t st, const LinearTileArgs &t) {
  const long grid = (long)t.tiles_m * t.tiles_n * t.splits;
  hipLaunchKernelGGL((linear_tile_kernel<WT, NX, BM, BN, WM, WN, PD, MINW>), dim3((unsigned)grid), dim3(WM * WN * 64), 0, st, t);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || t.splits == 1) return e;
  bool vec = t.n_total % 4 == 0;
  for (int i = 0; i < t.nseg; ++i)
    vec = vec && t.seg[i].N % 4 == 0 && (reinterpret_cast<uintptr_t>(t.seg[i].out) & 15) == 0;
  const int cols = vec ? 1024 : 256;
  const dim3 rg((unsigned)((t.n_total + cols - 1) / cols), (unsigned)t.seg[0].M);
  if (vec)
    hipLaunchKernelGGL((linear_tile_reduce_kernel<WT, 4>), rg, dim3(256), 0, st, t);
  else
    hipLaunchKernelGGL((linear_tile_reduce_kernel<WT, 1>), rg, dim3(256), 0, st, t);
  return hipGetLastError();
}

template <typename WT, int NX>
hipError_t launch_shape(hipStream_t st, const LinearTileArgs &t, int shape) {
  // two workgroups per CU where LDS holds them, six tiles in flight where the
  // registers do
  constexpr bool B = __is_same(WT, __bf16);
  switch (shape) {
    case 0: return launch_tile<WT, NX, 32, 128, 1, 4, B ? 6 : 3, B ? 2 : 1>(st, t);
    case 1: return launch_tile<WT, NX, 64, 128, 2, 2, 3, B ? 2 : 1>(st, t);
    case 2: return launch_tile<WT, NX, 128, 128, 4, 2, 3, 2>(st, t);
    case 3:
      if constexpr (B) return launch_tile<WT, NX, 128, 256, 2, 4, 3, 2>(st, t);
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}
}  // namespace

// (a plan has K splits only while they and the tiles are at most two
// workgroups per CU)
size_t linear_tile_partial_bytes(int cus) {
  long most = 0;
  for (const TileShape &s : kTileShapes) most = std::max<long>(most, (long)s.bm * s.bn);
  return 2 * (size_t)(cus > 0 ? cus : 256) * most * sizeof(float);
}

LinearTilePlan linear_tile_plan(int dtype, long M, const long *N, int nseg, long K, int cus) {
  const long c = cus > 0 ? cus : 256;
  // (three pieces of x instead of two: 1.2-1.3 times on seven shapes, 24 x 512 x 2040 to 4096 x 5120 x 3080)
  const double slow = dtype == SPISSA_DTYPE_BF16 ? (K % kTBK == 0 ? 1.0 : 1.25) : dtype == SPISSA_DTYPE_F16 ? 2.1 : 2.6;
  const long steps = (K + kTBK - 1) / kTBK;
  long n_total = 0;
  for (int i = 0; i < nseg; ++i) n_total += N[i];
  LinearTilePlan best{};
  for (int sh = 0; sh < 4; ++sh) {
    const TileShape &s = kTileShapes[sh];
    if (s.bn > 128 && dtype != SPISSA_DTYPE_BF16) continue;
    long tiles = 0;
    for (int i = 0; i < nseg; ++i) tiles += (N[i] + s.bn - 1) / s.bn;
    tiles *= (M + s.bm - 1) / s.bm;
    for (int sp = 1; sp <= kMaxTileSplits; ++sp) {
      const long tps = (steps + sp - 1) / sp;
      if (sp > 1 && (tps < 4 || (steps + tps - 1) / tps != sp || tiles * sp > 2 * c)) continue;
      const double rounds = (double)((tiles * sp + c - 1) / c), fill = (double)(tiles * sp) / c;
      const double part = s.bm == 64 && dtype != SPISSA_DTYPE_BF16 ? 0.8 : s.part;  // (LDS: one workgroup per CU)
      const double load = std::max(fill, part * rounds);
      // launch, prologue and stores; the steps; the second launch and the
      // partials' way through memory
      double us = 4.0 + 0.03 * (s.bm * s.bn / 1024) + slow * tps * std::max<double>(s.lat, load * s.share);
      if (sp > 1) us += 3.0 + 8.0 * sp * M * n_total / 3.5e6;
      if (best.us == 0.0 || us < best.us) best = LinearTilePlan{sh, sp, (int)tps, us, sp > 1 ? (size_t)sp * M * n_total * 4 : 0};
    }
  }
  return best;
}

void linear_tile_dims(const LinearTilePlan &plan, int *rows, int *columns) {
  *rows = kTileShapes[plan.shape].bm;
  *columns = kTileShapes[plan.shape].bn;
}

hipError_t launch_linear_tile(hipStream_t st, const LinearArgs *segs, int nseg, const LinearTilePlan &plan, float *partial) {
  if (nseg < 1 || nseg > kMaxLinearSegments || plan.shape < 0 || plan.shape > 3 || (plan.splits > 1 && !partial))
    return hipErrorInvalidValue;
  const TileShape &s = kTileShapes[plan.shape];
  LinearTileArgs t{};
  t.nseg = nseg;
  for (int i = 0; i < nseg; ++i) {
    t.seg[i] = segs[i];
    t.seg_off[i] = t.n_total;
    t.n_total += segs[i].N;
    t.seg_tiles[i] = (segs[i].N + s.bn - 1) / s.bn;
    t.tiles_n += t.seg_tiles[i];
  }
  const LinearArgs &a = segs[0];
  t.tiles_m = (a.M + s.bm - 1) / s.bm;
  if ((long)t.tiles_m * t.tiles_n * plan.splits > INT_MAX) return hipErrorInvalidValue;
  t.splits = plan.splits;
  t.kps = plan.tps * kTBK;
  t.partial = partial;
  // An XCD's run of tiles covers a band of rows and every column, or the other
  // way round: the operand read by all eight XCDs is the smaller one.
  const long es = a.dtype == SPISSA_DTYPE_F32 ? 4 : 2;
  t.m_fast = 4L * a.M < es * t.n_total;
  // what the generic kernel took before keeps its infinities
  t.in_order_nan = a.dtype != SPISSA_DTYPE_BF16 || a.K % kTBK != 0;
  switch (a.dtype) {
    case SPISSA_DTYPE_F32: return launch_shape<float, 3>(st, t, plan.shape);
    case SPISSA_DTYPE_F16: return launch_shape<_Float16, 3>(st, t, plan.shape);
    case SPISSA_DTYPE_BF16:
      return a.K % kTBK == 0 ? launch_shape<__bf16, 2>(st, t, plan.shape) : launch_shape<__bf16, 3>(st, t, plan.shape);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace spissa
