// f32 contraction on the bf16 matrix cores, for products whose operands carry more than bf16's
// 8 significant bits: every f32 operand is split exactly into three bf16 values (24 bits = 3 x 8),
//   v = h + m + l,   h = bf16(v), m = bf16(v - h), l = v - h - m
// (Henry, Tang and Heinecke, "Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", 2019),
// and the products of the parts are summed in one f32 accumulator by v_mfma_f32_16x16x32_bf16.
// A bf16 x and an integer weight code (|code| <= 255) are one part and exact.  Split x against one
// part takes 3 products per term, against three parts 6 (m*l, l*m and l*l, at most 2^-25 of the
// term each, are left out).  The bf16 MFMAs have 16 times the rate of v_mfma_f32_16x16x4_f32, so 3
// products have 5.3 times and 6 products 2.7 times the f32 matrix cores' peak.
// The split is exact for every f32: the parts hold 2^16 v, so that f32's smallest step, 2^-149, is
// bf16's, 2^-133 (the matrix cores keep subnormals); unlifted, operands below 2^-110 lose bits (9e-5 of
// a value at 1e-36).  x times its row's scale is lifted by 2^24: its bits below 2^-149 count, since a
// code of up to 8 bits comes after it.  The sums are brought back once.
//
// What bounds it: matrix-core and VALU issue together (an MFMA keeps the VALU from about 2.5 of its own
// issue slots; at four VALU instructions per MFMA, the conversions' share with 3 products, the
// two run 12 ns per MFMA and SIMD where the MFMA alone takes 8; counters: MFMA busy 42 %, VALU 39 %).
// Measured, f32 x [2048,4096] x Int4 [4096,11008], against an f32-MFMA kernel at 0.63 of the f32 peak:
// scales per row and 128 columns (3 products) 1868 -> 560 us, 0.99 PFLOP/s of products; per row and 64
// columns (6 products) 1868 -> 1069 us; with 100 rows 363 -> 68 us (K in 2 slices).  The error against
// 64 bits fell from 1.1e-6 to 5.8e-7 (four waves) and 1.1e-7 (eight): a step sums 32 terms where the
// f32 MFMA summed 4, and eight waves keep the sums in three levels.
//
// Tiling: a workgroup of 4 (or 8) waves owns a 128 x 128 output tile, 2 x 2 waves of 64 x 64 (4 x 2
// of 32 x 64), K in blocks of 32 (one MFMA step).  An operand's part lies in LDS as 128 rows of 32
// bf16 (64 bytes, four 16-byte chunks XOR-swizzled by (row >> 1) & 3: every operand read and every
// staging write covers all banks).  Block kb is multiplied while block kb + 1, in registers, is
// split into the other LDS buffer and block kb + 2 is requested.  K past the last whole block: that
// block starts 32 before K's end and the values the block before it holds are zeroed.  K below 32 (at
// least 8): one block, whose loads past K read values before it and are zeroed.
//
// Column n of the tile lies in LDS row (n & 3) * 32 + (n >> 2): MFMA column set c of wave half wn
// holds columns 64 wn + 4 cg + c, so a lane ends with four consecutive columns of each of its rows.
//
// Infinities, and finite operands, products or sums past the range of the parts, leave sums that are
// not finite (the parts of an infinity are inf, NaN, NaN; leading and lower products that overflow meet
// as inf - inf): a wave that ends with such sums forms those again by f32 FMAs in k order, each term
// with the weight factor as the reference rounds it, before the epilogue.  Rows with a NaN in x are
// left as they are.
#pragma once

#include <algorithm>
#include <cmath>

#include "device_common.h"
#include "mxrt_internal.h"

namespace mx {
namespace sg {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_t;
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2_t;
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_v __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_v __attribute__((ext_vector_type(2)));

constexpr int kBM = 128, kBN = 128, kBK = 32;
constexpr int kPlane = kBM * kBK * 2;  // LDS bytes of one part of an operand
constexpr size_t kCounterBytes = 64 * 1024;
constexpr int kPartBytes = kBM * kBN * 4;  // one partial tile
// Partial tiles of a split K: the most that the allocation-free entry point's static scratch holds
// (the split is the same for both entry points, so their results are the same bits).
constexpr int kMaxParts = (int)((MX_QDENSE_NOALLOC_SCRATCH_BYTES - kCounterBytes) / kPartBytes);

constexpr float kLift = 0x1p16f, kLiftRow = 0x1p24f;

struct Args {
  const void* x;      // [M, K] f32 or bf16
  const uint8_t* w;   // weight storage
  const void* scale;
  const void* zp;     // same layout as scale, or null
  const void* bias;   // [N] or null
  void* out;          // [M, N], x's dtype
  int M, K, N;
  int s_dt, zp_dt, b_dt, act;
  int B, kB;          // columns and rows of weights per scale (1 along the axis that is not blocked)
  int nb;             // scale row length: ceil(N / B)
  int64_t bpr;        // GGML: bytes per weight row
  // Work items: `whole` whole tiles (a multiple of 8), then `tail` items, the S slices of each of the
  // remaining tiles next to each other.
  int tiles_n, whole, tail, per_xcd;  // per_xcd: tail items per XCD
  int vec;            // out's rows take stores of 4 values
  int S, kpb;         // K slices of a tail tile, 32-row blocks per slice
  float* part;        // [tail tile][S] partial tiles (S > 1)
  uint32_t* ctr;      // [tail tile] arrivals, zero between launches
};

__device__ __forceinline__ f32x4_t mfma(const u32x4_v& a, const u32x4_v& b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// The aligned word holding element i of an f32 or bf16 array, and the shift that moves a bf16
// element to its high half (no branch on the dtype, and the load never leaves the element's word).
__device__ __forceinline__ void word(const void* p, int64_t i, bool bf, uint32_t& w, uint32_t& sh) {
  const uintptr_t ad = (uintptr_t)p + (uintptr_t)i * (bf ? 2 : 4);
  w = *(const uint32_t*)(ad & ~(uintptr_t)3);
  sh = bf && (ad & 2) == 0 ? 16u : 0u;
}
__device__ __forceinline__ float word_f32(uint32_t w, uint32_t sh, bool bf) {
  return __uint_as_float((w << sh) & (bf ? 0xFFFF0000u : ~0u));
}

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  const f32x2_t v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// The three bf16 parts of a pair of values, one packed word per part.
__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
  h = pack_bf16(a, b);
  const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xFFFF0000u);
  m = pack_bf16(ra, rb);
  l = pack_bf16(ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xFFFF0000u));
}

// LDS offset of 16-byte chunk `chunk` of LDS row p of a part.
__device__ __forceinline__ uint32_t chunk_at(int p, int chunk) {
  return (uint32_t)(p * 64 + ((chunk ^ ((p >> 1) & 3)) << 4));
}

// LDS row of column n of the tile, and back.
__device__ __forceinline__ int row_of_col(int n) { return (n & 3) * 32 + (n >> 2); }
__device__ __forceinline__ int col_of_row(int p) { return 4 * (p & 31) + (p >> 5); }

// Element i of an f32 or bf16 array as f32.
__device__ __forceinline__ float elem(const void* p, int64_t i, int dt) {
  return dt == MX_DTYPE_BFLOAT16 ? bf16_to_f32(((const uint16_t*)p)[i]) : ((const float*)p)[i];
}

// P: the operand policy.  P::kXbf bf16 x (else f32); P::kPA, P::kPB parts of x and of the weights;
// P::kLiftW whether the weights' parts are lifted (those of f32 weight factors of any size);
// P::kRow each x value multiplied by its row's scale of the tile's column block before the split
// (reference layout, one block per tile);
// P::kCol one scale per column, applied to a slice's sums; P::Regs, load, stage: a thread's weights of a
// block, their loads, and their parts into LDS (kTail: zeros past K); P::value: the f32 weight
// factor of one (k, n), its scale included; P::table_value: the 16 entries of the lookup table.
// NW: waves of the workgroup, 4 (2 x 2 waves of 64 x 64) or 8 (4 x 2 waves of 32 x 64).
// A block of K: its first row, how many of its rows the block before it holds (the last block of a K
// that is no multiple of 32), and its rows up to K's end (fewer than 32 where K is).
struct Block {
  int k, skip, end;
  __device__ __forceinline__ Block(int kb, int K) : k(max(0, min(kb * kBK, K - kBK))), skip(kb * kBK - k), end(K - k) {}
};

template <class P, int NW>
__global__ __launch_bounds__(64 * NW, 2) void split_gemm_kernel(Args a) {
  constexpr int PA = P::kPA, PB = P::kPB;
  constexpr int kThreads = 64 * NW, RB = 16 / NW;  // 16-row blocks per wave
  constexpr int kBufBytes = (PA + PB) * kPlane;
  constexpr int XR = 8 / NW;  // rows of x per thread and block
  static_assert(!P::kRow || (PA == 3 && PB == 1), "row scales: split x, exact weight codes");
  __shared__ __attribute__((aligned(16))) char sm[2][kBufBytes];
  __shared__ __attribute__((aligned(16))) float ring[P::kRow ? 2 : 1][kBK];  // scales of a block's rows
  __shared__ float table[16];
  __shared__ int last_slice;

  // Workgroups go round-robin over the 8 XCDs: each XCD takes a contiguous run of the whole tiles
  // (M-major: its tiles share x rows in its L2) and one of the tail items.
  const int bid = blockIdx.x, xcd = bid & 7;
  int tile, slice = 0, kpb = 1 << 26;
  const bool sliced = bid >= a.whole && a.S > 1;
  if (bid < a.whole) {
    tile = xcd * (a.whole >> 3) + (bid >> 3);
  } else {
    const int j = (bid - a.whole) >> 3, item = xcd * a.per_xcd + j;
    if (j >= a.per_xcd || item >= a.tail) return;
    tile = item / a.S;
    slice = item - tile * a.S;
    kpb = a.kpb;
    tile += a.whole;
  }
  const int m0 = (tile / a.tiles_n) * kBM, n0 = (tile % a.tiles_n) * kBN;
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1, cg = lane & 15, kq = lane >> 4;
  const int M = a.M, K = a.K, N = a.N;
  const int row0 = 16 * RB * wm;  // the wave's first row in the tile
  if (t < 16) table[t] = P::table_value(t);

  const int kb0 = slice * kpb, kb1 = min(kb0 + kpb, (K + kBK - 1) / kBK);

  // ---- x: thread t stages k chunk t & 3 (8 values) of rows t / 4 and, with 4 waves, t / 4 + 64.
  // Rows past M read row M - 1 (their outputs are not stored).
  const int xr = t >> 2, xc = t & 3;
  constexpr int kXe = P::kXbf ? 2 : 4;  // bytes of an element
  const char* xbase = (const char*)a.x + (int64_t)m0 * K * kXe;
  uint32_t xoff[XR];  // from the tile's first row (128 K elements stay below 2^31 bytes, checked by the host)
#pragma unroll
  for (int i = 0; i < XR; ++i) xoff[i] = ((uint32_t)min(xr + 64 * i, M - 1 - m0) * (uint32_t)K + (uint32_t)min(8 * xc, K - 8)) * kXe;
  struct XRegs {
    u32x4_v v[XR][P::kXbf ? 1 : 2];
  };
  auto load_x = [&](Block b, XRegs& R) __attribute__((always_inline)) {
    const char* base = xbase + (int64_t)b.k * kXe;
#pragma unroll
    for (int i = 0; i < XR; ++i) {
      R.v[i][0] = *(const u32x4_v*)(base + xoff[i]);
      if constexpr (!P::kXbf) R.v[i][1] = *(const u32x4_v*)(base + xoff[i] + 16);
    }
  };
  // With kTail, the values that the block before holds and those past K are zero (whole runs of 8 bf16
  // or 4 f32; the 4 before K where K is below 32 and no multiple of 8 came second).
  auto stage_x = [&](int slot, Block b, const XRegs& R, char* As, auto tail) __attribute__((always_inline)) {
    constexpr bool kTail = decltype(tail)::value;
    const bool lo = !kTail || (8 * xc >= b.skip && 8 * xc < b.end);
    const bool hi = !kTail || (P::kXbf ? lo : 8 * xc + 4 >= b.skip && 8 * xc + 4 < b.end);
#pragma unroll
    for (int i = 0; i < XR; ++i) {
      char* dst = As + chunk_at(xr + 64 * i, xc);
      if constexpr (PA == 1) {
        u32x4_v v = R.v[i][0];
        if (kTail && !lo) v = u32x4_v{0u, 0u, 0u, 0u};
        *(u32x4_v*)dst = v;
      } else {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          if constexpr (P::kXbf)
            v[e] = __uint_as_float(e & 1 ? R.v[i][0][e >> 1] & 0xFFFF0000u : R.v[i][0][e >> 1] << 16);
          else
            v[e] = __uint_as_float(R.v[i][e >> 2][e & 3]);
          if constexpr (kTail && !P::kXbf) {
            if (e < 4 && 8 * xc + 4 == b.end) v[e] = __uint_as_float(R.v[i][1][e & 3]);
          }
          if constexpr (kTail) v[e] = (e < 4 ? lo : hi) ? v[e] : 0.0f;
        }
        if constexpr (P::kRow) {
          const float* s = &ring[slot][8 * xc];
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = mul_rn(v[e], s[e]);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] *= kLift;
        }
        u32x4_v h, m, l;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          uint32_t hh, mm, ll;
          split2(v[2 * q], v[2 * q + 1], hh, mm, ll);
          h[q] = hh;
          m[q] = mm;
          l[q] = ll;
        }
        *(u32x4_v*)dst = h;
        *(u32x4_v*)(dst + kPlane) = m;
        *(u32x4_v*)(dst + 2 * kPlane) = l;
      }
    }
  };
  // Row scales of a block, its row t & 31 by every thread (the copies write the
  // same words), into their slot two blocks ahead of their use.
  uint32_t rs = 0, rssh = 0;
  const bool sbf = a.s_dt == MX_DTYPE_BFLOAT16;
  const int scol = P::kRow ? n0 / a.B : 0, srow = min(t & 31, K - 1);
  auto load_row_scale = [&](Block b) __attribute__((always_inline)) {
    if constexpr (P::kRow) {
      const int64_t i = (int64_t)(b.k + srow) * a.nb + scol;
      word(a.scale, i, sbf, rs, rssh);
    }
  };
  auto store_row_scale = [&](int slot) __attribute__((always_inline)) {
    if constexpr (P::kRow) ring[slot][t & 31] = word_f32(rs, rssh, sbf) * kLiftRow;
  };

  // Eight waves leave registers to round less: the products of leading parts and those of the others
  // have sums of their own (a step then rounds the large sums once instead of 3 or 6 times), and the
  // large sums go to a total every kFold blocks (chains of kFold and K / 32 kFold additions).
  constexpr bool kLow = NW == 8 && PA + PB > 2;
  constexpr int kFold = 8;
  f32x4_t acc[RB][4], low[RB][4], total[RB][4];
  auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[i][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
  clear();
  if constexpr (kLow) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) low[i][c] = total[i][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  // One block: small products first.
  auto compute = [&](const char* buf) __attribute__((always_inline)) {
    const char* As = buf;
    const char* Bs = buf + PA * kPlane;
    u32x4_v B[PB][4];
#pragma unroll
    for (int p = 0; p < PB; ++p)
#pragma unroll
      for (int c = 0; c < 4; ++c) B[p][c] = *(const u32x4_v*)(Bs + p * kPlane + chunk_at(c * 32 + 16 * wn + cg, kq));
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      u32x4_v A[PA];
#pragma unroll
      for (int p = 0; p < PA; ++p) A[p] = *(const u32x4_v*)(As + p * kPlane + chunk_at(row0 + 16 * rb + cg, kq));
#pragma unroll
      for (int order = PA + PB - 2; order >= 0; --order) {
        if (order > 2) continue;
#pragma unroll
        for (int pa = 0; pa < PA; ++pa) {
          const int pb = order - pa;
          if (pb < 0 || pb >= PB) continue;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            if (kLow && order > 0)
              low[rb][c] = mfma(A[pa], B[pb][c], low[rb][c]);
            else
              acc[rb][c] = mfma(A[pa], B[pb][c], acc[rb][c]);
          }
        }
      }
    }
  };

  using Whole = std::integral_constant<bool, false>;
  using Tail = std::integral_constant<bool, true>;
  P src(a, t, n0);
  XRegs X;
  typename P::Regs W;
  const int last = kb1 - 1;
  auto block = [&](int kb) { return Block(min(kb, last), K); };  // requests past the slice repeat its last block
  load_row_scale(block(kb0));
  load_x(block(kb0), X);
  src.load(a, block(kb0), W);
  store_row_scale(0);
  load_row_scale(block(kb0 + 1));
  __syncthreads();  // the table and block kb0's row scales are written
  store_row_scale(1);
  stage_x(0, block(kb0), X, sm[0], Tail{});
  src.stage(a, block(kb0), W, table, sm[0] + PA * kPlane, Tail{});
  load_x(block(kb0 + 1), X);
  src.load(a, block(kb0 + 1), W);
  load_row_scale(block(kb0 + 2));
  __syncthreads();
  // One basic block per step, so that the conversions run under the MFMAs.
  auto step = [&](int kb, auto tail) __attribute__((always_inline)) {
    const int cur = (kb - kb0) & 1;
    char* nxt = sm[cur ^ 1];
    compute(sm[cur]);
    stage_x(cur ^ 1, block(kb + 1), X, nxt, tail);
    src.stage(a, block(kb + 1), W, table, nxt + PA * kPlane, tail);
    load_x(block(kb + 2), X);
    src.load(a, block(kb + 2), W);
    store_row_scale(cur);
    load_row_scale(block(kb + 3));
    __syncthreads();
  };
  const int whole = kb1 * kBK > K ? last - 1 : last;  // steps that stage a whole block
  int kb = kb0;
#pragma unroll 1
  for (; kb < whole; ++kb) {
    step(kb, Whole{});
    if (kLow && (kb - kb0) % kFold == kFold - 1) {
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          total[i][c] += acc[i][c];
          acc[i][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
  if (kb < last) step(kb, Tail{});
  compute(sm[(last - kb0) & 1]);
  if constexpr (kLow) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[i][c] = total[i][c] + (acc[i][c] + low[i][c]);
  }
  constexpr float kBack = (PA == 3 ? 1 / (P::kRow ? kLiftRow : kLift) : 1.0f) * (P::kLiftW ? 1 / kLift : 1.0f);
  if constexpr (kBack != 1.0f) {
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[i][c] *= kBack;
  }

  const int ncol = n0 + 64 * wn + 4 * cg;  // this lane's four columns
  if constexpr (P::kCol) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float s = elem(a.scale, min(ncol + c, N - 1), a.s_dt);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[rb][c][r] = mul_rn(acc[rb][c][r], s);
    }
  }
  auto finite = [](float v) { return fabsf(v) < __builtin_inff(); };
  float probe = 0.0f;  // NaN after a sum that is not finite
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) probe = __builtin_fmaf(acc[rb][c][r], 0.0f, probe);
  uint64_t redo = 0;  // the wave's rows that hold such sums
  if (__any(probe != 0.0f)) {
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        bool bad = false;
#pragma unroll
        for (int c = 0; c < 4; ++c) bad |= !finite(acc[rb][c][r]);
        const uint64_t lanes = __ballot(bad);
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (lanes >> (16 * q) & 0xFFFFu) redo |= (uint64_t)1 << (16 * rb + 4 * q + r);
      }
  }
  // Row by row, a column per lane (0.7 ms a row of a tile at K = 4096, bound by the latency of the loads).
  const int kbeg = kb0 * kBK, kend = min(K, kb1 * kBK);
  for (; redo; redo &= redo - 1) {
    const int i = __builtin_ctzll(redo), m = m0 + row0 + i;
    if (m >= M) break;  // rows of padding, not stored
    auto xat = [&](int k) { return elem(a.x, (int64_t)m * K + k, P::kXbf ? MX_DTYPE_BFLOAT16 : MX_DTYPE_FLOAT32); };
    bool nan = false;  // a NaN in the row of x: the sums are NaN, as they should be
    for (int k = kbeg; k < kend && !nan; k += 256) {
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = xat(min(k + 64 * e + lane, kend - 1));
      nan = __any(v[0] != v[0] || v[1] != v[1] || v[2] != v[2] || v[3] != v[3]);
    }
    if (nan) continue;
    const int n = min(n0 + 64 * wn + lane, N - 1);
    float sum = 0.0f;
#pragma unroll 1
    for (int k = kbeg; k < kend; k += 4) {  // K is a multiple of 4
      float xv[4], wv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        xv[e] = xat(k + e);
        wv[e] = src.value(a, k + e, n, table);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) sum = __builtin_fmaf(xv[e], wv[e], sum);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float v = __shfl(sum, 4 * cg + c);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (i == 16 * rb + 4 * kq + r && !finite(acc[rb][c][r])) acc[rb][c][r] = v;
    }
  }

  if (sliced) {
    // Every slice stores its sums; the last to arrive at the tile adds them in slice order and goes
    // on to the epilogue.  Agent-scope coherent accesses (sc1): the slices may run on other XCDs.
    const __amdgpu_buffer_rsrc_t prs =
        __builtin_amdgcn_make_buffer_rsrc(a.part + (size_t)(tile - a.whole) * a.S * kBM * kBN, (short)0, a.S * kPartBytes, 0x00020000);
    constexpr int kSc1 = 16;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int c = 0; c < 4; ++c)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_v, acc[rb][c]), prs,
                                              (unsigned)(slice * kPartBytes + ((4 * rb + c) * kThreads + t) * 16), 0, kSc1);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    if (t == 0) {
      const uint32_t prev = __hip_atomic_fetch_add(&a.ctr[tile - a.whole], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (prev + 1u == (uint32_t)a.S) __hip_atomic_store(&a.ctr[tile - a.whole], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      last_slice = prev + 1u == (uint32_t)a.S;
    }
    __syncthreads();
    if (!last_slice) return;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int c = 0; c < 4; ++c) acc[rb][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int s = 0; s < a.S; ++s) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          acc[rb][c] += __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                        prs, (unsigned)(s * kPartBytes + ((4 * rb + c) * kThreads + t) * 16), 0, kSc1));
    }
  }

  // Epilogue: bias (added after the sum), the reference activation, x's dtype.  The
  // activation's code is there once: each half of the tile goes through LDS (free after the loop's
  // last barrier) to a rolled loop over four consecutive columns of a row.
  float bi[4] = {0.f, 0.f, 0.f, 0.f};
  if (a.bias && ncol < N) {
#pragma unroll
    for (int c = 0; c < 4; ++c) bi[c] = elem(a.bias, min(ncol + c, N - 1), a.b_dt);
  }
  auto store4 = [&](int m, int n, const float (&y)[4]) __attribute__((always_inline)) {
    const int64_t o = (int64_t)m * N + n;
    if (!a.vec) {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (n + c < N) store_f(a.out, o + c, P::kXbf ? MX_DTYPE_BFLOAT16 : MX_DTYPE_FLOAT32, y[c]);
    } else if constexpr (P::kXbf) {
      *(u32x2_v*)((uint16_t*)a.out + o) = u32x2_v{(uint32_t)f32_to_bf16(y[0]) | (uint32_t)f32_to_bf16(y[1]) << 16,
                                                  (uint32_t)f32_to_bf16(y[2]) | (uint32_t)f32_to_bf16(y[3]) << 16};
    } else {
      *(f32x4_t*)((float*)a.out + o) = f32x4_t{y[0], y[1], y[2], y[3]};
    }
  };
  auto finish = [&](float v, int c) __attribute__((always_inline)) { return a.bias ? add_rn(bi[c], v) : v; };
  if (a.act == MX_ACT_NONE) {
    if (ncol >= N) return;
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + row0 + 16 * rb + 4 * kq + r;
        float y[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) y[c] = finish(acc[rb][c][r], c);
        if (m < M) store4(m, ncol, y);
      }
    return;
  }
  constexpr int kCS = kBN * 4;  // LDS bytes per row of a half tile
  static_assert(64 * kCS <= 2 * kBufBytes, "half a tile fits the LDS buffers");
  char* Cs = sm[0];
#pragma unroll 1
  for (int half = 0; half < 2; ++half) {
    __syncthreads();
    if (row0 / 64 == half) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          *(f32x4_t*)(Cs + (row0 % 64 + 16 * rb + 4 * kq + r) * kCS + (64 * wn + 4 * cg) * 4) =
              f32x4_t{finish(acc[rb][0][r], 0), finish(acc[rb][1][r], 1), finish(acc[rb][2][r], 2), finish(acc[rb][3][r], 3)};
    }
    __syncthreads();
#pragma unroll 1
    for (int idx = t; idx < 64 * (kBN / 4); idx += kThreads) {
      const int row = idx >> 5, col = (idx & 31) * 4;
      const int m = m0 + 64 * half + row, n = n0 + col;
      if (m >= M || n >= N) continue;
      float* v = (float*)(Cs + row * kCS + col * 4);
#pragma unroll 1
      for (int c = 0; c < 4; ++c) v[c] = act_ref(v[c], a.act);
      const float y[4] = {v[0], v[1], v[2], v[3]};
      store4(m, n, y);
    }
  }
}

// Waves per workgroup, tail slices and grid of a problem (planned for 256 CUs whatever the device
// reports, so the summation order depends on the shape alone).
//   Below 256 tiles every tile is sliced along K, as many slices as fill the CUs at most.  A slice adds
//   0.6 us to the tile's sum at its end and a block takes 1.1 us with six products per term and 0.8
//   with three, so S = sqrt(1.8 or 1.3 blocks) is best: Q4_K rows, x [128,512] x 512 14.6 us in four
//   slices (19.2 in two, 14.1 in eight), [128,1024] x 1024 17.1 in eight (20.2 in four, 19.8 in 16),
//   [128,4096] x 1024 27.0 in 16 (29.8 in 26); DotGeneral [96,115004] x 100 101 us in 80 (155 in 255).
//   One workgroup per CU then has eight waves, two per SIMD: x f32 [100,4096] x Int4 [4096,11008] with
//   86 tiles in two slices 77 us with four waves, 68 us with eight.
//   Past that, forms whose operands have at most four parts in all run two workgroups of four waves
//   per CU (64 KB of LDS each; [2048,4096] x [4096,11008] 560 us, a third more with eight waves), the
//   others one of eight waves (96 KB).  Up to 64 rows of f32 x have eight waves too: the GEMV, which
//   would take them else, is 1.4e-7 to 3.2e-7 off 64 bits, four waves' single chain of sums 6.4e-7,
//   eight waves 0.7e-7 to 1.2e-7 ([48,4096] x Int4 [4096,32768] 124 us with four waves, 125 with
//   eight; x [4096,128256] 377 and 535; the GEMV 1005 at 32 rows there).
//   Tiles past the last whole round of resident workgroups are sliced if the slices fit one round:
//   258 tiles of GGML Q6_K rows (x [333,4096], N = 11008) took 357 us in two rounds, 212 us with the
//   last two tiles in slices.
inline int plan(mx_backend* b, Args& a, int64_t M, int parts, bool xbf, int* nw, int* grid) {
  const int64_t tiles_n = (a.N + kBN - 1) / kBN, tiles = ((M + kBM - 1) / kBM) * tiles_n;
  if (tiles >= (int64_t)1 << 28) return set_error(MX_ERR_INVALID, "FusedQuantizedDense: M=%lld too large", (long long)M);
  const int blocks = (a.K + kBK - 1) / kBK;
  *nw = parts > 4 || tiles < 256 || (M <= 64 && !xbf) ? 8 : 4;
  const int64_t round = *nw == 8 ? 256 : 512;
  a.whole = (int)(tiles / round * round);
  const int64_t tail = tiles - a.whole;
  int64_t S = 1;
  if (tail > 0) {
    const int64_t best = std::max<int64_t>(1, (int64_t)(sqrtf((parts > 4 ? 1.8f : 1.3f) * (float)blocks) + 0.5f));
    S = std::max<int64_t>(1, std::min<int64_t>((a.whole ? round : kMaxParts) / tail, best));
    if (a.whole && b->noalloc_active && tail * S > kMaxParts) S = std::max<int64_t>(1, kMaxParts / tail);
  }
  a.kpb = (int)((blocks + S - 1) / S);
  a.S = (blocks + a.kpb - 1) / a.kpb;
  a.tiles_n = (int)tiles_n;
  a.tail = (int)tail * a.S;
  a.per_xcd = (a.tail + 7) / 8;
  *grid = a.whole + 8 * a.per_xcd;
  a.vec = (uintptr_t)a.out % 16 == 0 && a.N % 4 == 0;
  a.part = nullptr;
  a.ctr = nullptr;
  if (a.S > 1) {
    void* scratch = nullptr;
    MX_TRY(ensure_scratch(b, kCounterBytes + (size_t)a.tail * kPartBytes, &scratch));
    a.ctr = (uint32_t*)scratch;
    a.part = (float*)((char*)scratch + kCounterBytes);
  }
  return MX_OK;
}

}  // namespace sg
}  // namespace mx
