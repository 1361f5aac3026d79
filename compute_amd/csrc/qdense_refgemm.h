// FusedQuantizedDense past the GEMV for the layouts the bf16 GEMM does not take: the reference's own
// scale layout [K, ceil(N/B)] (BlockAxis = 1), f32 x, zero points and NF4 (fused_ops.go:204-234;
// quantizeddense.go:586-650).  The contraction is split_gemm.h's: f32 operands in three exact bf16
// parts on the bf16 matrix cores.  No copy of the weight matrix is ever made.
//
// Three forms, by where the scale enters:
//   row      reference layout, one column block per 128-column tile (B % 128 == 0 or one block),
//            linear scheme, no zero points: x * s is formed and rounded once per (row, k) of the
//            tile, the codes stay exact; 3 products per term.  (With zero points the sums of x*s*w
//            and x*zp would cancel, codes near the zero point above all.)
//   column   one scale per output column, linear scheme, no zero points: the sums of x * w, scaled
//            once; 3 products (1 with bf16 x).
//   weight   everything else: the weight factor formed as the reference forms it (w*s, w*s + zp
//            with its two roundings, nf4[w]*s) and split; 6 products (3 with bf16 x).
// The reference rounds (x*w)*s per term and sums in k order; the results stay within the f32
// accumulation bound of its sum.  The bias is added after the sum (the reference starts from it),
// then the reference activation (act_ref) and the output dtype.
#pragma once

#include <algorithm>

#include "split_gemm.h"

namespace mx {
namespace {

using namespace sg;

enum RgForm { kRow, kColumn, kWeight };
// Where the weight form finds the scales (and zero points) of 4 consecutive columns of 4 rows.
// kRgCols holds one scale row where the others hold four: x [2048,4096] x [4096,4096], groups of 128 with
// zero points 546 -> 386 us (f32 x) and 348 -> 218 (bf16 x, whose four-wave kernel spilled with four).
enum RgScales {
  kRgCols = 0,  // [ceil(K/B), N], B % 4 == 0: one per column
  kRgBlk = 1,   // [K, ceil(N/B)], B % 4 == 0: one per row
  kRgAny = 2,   // [K, ceil(N/B)], any other B: one each
  kRgRows = 3   // [ceil(K/B), N], any other B: one each
};

// What the weight factor holds beside the code times the scale.
enum RgKind { kLinear = 0, kZeroPoint, kNf4 };

// Weights [K, N]: thread t converts CT = 16 / NW columns of rows 4 j .. 4 j + 3 of a block, with j's
// low bit in the thread's (so that lane pairs write whole 16-byte chunks): columns 4 cq + c0 ..
// 4 cq + c0 + CT - 1 of the tile.
template <int WDT, int FORM, int SM, int KIND, bool XBF, int NW>
struct RgSource {
  static constexpr bool kXbf = XBF;
  static constexpr bool kRow = FORM == RgForm::kRow, kCol = FORM == kColumn, kZp = KIND == kZeroPoint;
  static_assert(KIND == kLinear || FORM == kWeight, "zero points and NF4 are in the weight factor");
  static constexpr int kPA = XBF && FORM != RgForm::kRow ? 1 : 3;
  static constexpr int kPB = FORM == kWeight ? 3 : 1;
  static constexpr bool kLiftW = FORM == kWeight;
  static constexpr bool kI4 = WDT == MX_DTYPE_INT4 || WDT == MX_DTYPE_UINT4;
  static constexpr bool kSigned = WDT == MX_DTYPE_INT4 || WDT == MX_DTYPE_INT8;
  static constexpr int CT = 16 / NW;
  static constexpr int kScales = FORM != kWeight ? 1 : SM == kRgBlk ? 1 : CT;  // per scale row
  static constexpr int kSRows = SM == kRgCols ? 1 : 4;                         // scale rows of 4 rows
  static constexpr bool kAlongK = SM == kRgCols || SM == kRgRows;

  struct Regs {
    uint32_t w[4];
    uint32_t s[kSRows][kScales], z[kSRows][kScales];  // raw words (kRgCols with bf16: pairs)
    uint32_t ssh[kSRows][kScales], zsh[kSRows][kScales];
  };
  int cq, c0, j, ncl;
  uint32_t woff[4];  // from a block's first row
  static __device__ __forceinline__ float table_value(int i) { return kNF4Table[i]; }

  __device__ __forceinline__ RgSource(const Args& a, int t, int n0) {
    cq = (t >> 1) & 31;
    c0 = NW == 8 ? 2 * ((t >> 6) & 1) : 0;
    j = (t & 1) | (t >> (NW == 8 ? 7 : 6)) << 1;
    const int jl = min(j, a.K / 4 - 1);  // rows past K (below 32): K's last four
    // N % 16 == 0: the columns are all in range or all past N (then the first are read and the
    // outputs are not stored).
    ncl = n0 + 4 * cq < a.N ? n0 + 4 * cq + c0 : 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) woff[e] = ((uint32_t)(4 * jl + e) * (uint32_t)a.N + (uint32_t)ncl) / (kI4 ? 2 : 1);
  }
  // k / kB: the quotient's error, at most k 2^-23, is below the half that keeps it off the integers (K
  // is at most 2^22).
  static __device__ __forceinline__ int scale_row(const Args& a, int k) {
    return (int)(((float)k + 0.5f) * (1.0f / (float)a.kB));
  }
  // CT consecutive elements from i on: f32 CT words; bf16 CT / 2 words, repeated (one form for both).
  static __device__ __forceinline__ void words(const void* p, int64_t i, bool bf, uint32_t (&w)[kScales]) {
    const uint32_t* q = (const uint32_t*)((const char*)p + i * (bf ? 2 : 4));
#pragma unroll
    for (int c = 0; c < kScales; ++c) w[c] = q[bf ? c / 2 : c];
  }
  __device__ __forceinline__ void load(const Args& a, Block b, Regs& R) const {
    const char* base = (const char*)a.w + (int64_t)b.k * (kI4 ? a.N / 2 : a.N);
    const bool sbf = a.s_dt == MX_DTYPE_BFLOAT16, zbf = a.zp_dt == MX_DTYPE_BFLOAT16;
    if constexpr (FORM == kWeight && kAlongK) {
#pragma unroll
      for (int r = 0; r < kSRows; ++r) {
        const int64_t i = (int64_t)scale_row(a, min(b.k + 4 * j + r, a.K - 1)) * a.N + ncl;
        words(a.scale, i, sbf, R.s[r]);
        if constexpr (kZp) words(a.zp, i, zbf, R.z[r]);
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const char* p = base + woff[e];
      if constexpr (kI4 && CT == 2)
        R.w[e] = *(const uint8_t*)p;
      else if constexpr (kI4 || CT == 2)
        R.w[e] = *(const uint16_t*)p;
      else
        R.w[e] = *(const uint32_t*)p;
      if constexpr (FORM == kWeight && !kAlongK) {
        const int k = min(b.k + 4 * j + e, a.K - 1);
#pragma unroll
        for (int c = 0; c < kScales; ++c) {
          const int64_t i = (int64_t)k * a.nb + (ncl + c) / a.B;
          word(a.scale, i, sbf, R.s[e][c], R.ssh[e][c]);
          if constexpr (kZp) word(a.zp, i, zbf, R.z[e][c], R.zsh[e][c]);
        }
      }
    }
  }
  static __device__ __forceinline__ int code(uint32_t w, int c) {
    if constexpr (kI4)
      return kSigned ? __builtin_amdgcn_sbfe((int)w, 4 * c, 4) : (int)__builtin_amdgcn_ubfe(w, 4 * c, 4);
    else
      return kSigned ? (int)(int8_t)(w >> (8 * c)) : (int)(uint8_t)(w >> (8 * c));
  }
  static __device__ __forceinline__ float scale_of(const uint32_t (&s)[kScales], const uint32_t (&sh)[kScales], int c, bool bf) {
    if constexpr (kAlongK)
      return __uint_as_float(bf ? (c & 1 ? s[c % kScales] & 0xFFFF0000u : s[c % kScales] << 16) : s[c % kScales]);
    else
      return word_f32(s[c % kScales], sh[c % kScales], bf);
  }
  template <class TailT>
  __device__ __forceinline__ void stage(const Args& a, Block b, const Regs& R, const float* table, char* Bs, TailT) const {
    const bool sbf = a.s_dt == MX_DTYPE_BFLOAT16, zbf = a.zp_dt == MX_DTYPE_BFLOAT16;
#pragma unroll
    for (int c = 0; c < CT; ++c) {
      char* dst = Bs + chunk_at(row_of_col(4 * cq + c0 + c), j >> 1) + 8 * (j & 1);
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int q = code(R.w[e], c);
        if constexpr (FORM == kWeight) {
          const float wf = KIND == kNf4 ? table[(uint32_t)q & 15u] : (float)q;
          const int r = e % kSRows;
          v[e] = mul_rn(wf, scale_of(R.s[r], R.ssh[r], c, sbf) * kLift);
          if constexpr (kZp) v[e] = add_rn(v[e], scale_of(R.z[r], R.zsh[r], c, zbf) * kLift);
          if (TailT::value && (4 * j < b.skip || 4 * j >= b.end)) v[e] = 0.0f;  // x is zero there, but 0 * inf is not
        } else {
          v[e] = (float)q;
        }
      }
      if constexpr (FORM == kWeight) {
        uint32_t h0, m0, l0, h1, m1, l1;
        split2(v[0], v[1], h0, m0, l0);
        split2(v[2], v[3], h1, m1, l1);
        *(u32x2_v*)dst = u32x2_v{h0, h1};
        *(u32x2_v*)(dst + kPlane) = u32x2_v{m0, m1};
        *(u32x2_v*)(dst + 2 * kPlane) = u32x2_v{l0, l1};
      } else {
        // Codes have at most 8 significant bits: the high halves of their f32 values are exact.
        *(u32x2_v*)dst = u32x2_v{__builtin_amdgcn_perm(__float_as_uint(v[1]), __float_as_uint(v[0]), 0x07060302u),
                                 __builtin_amdgcn_perm(__float_as_uint(v[3]), __float_as_uint(v[2]), 0x07060302u)};
      }
    }
  }
  // The weight factor of (k, n) as the reference forms it.
  __device__ __forceinline__ float value(const Args& a, int k, int n, const float* table) const {
    const int q = decode_weight(a.w, (int64_t)k * a.N + n, WDT);
    const float wf = KIND == kNf4 ? table[(uint32_t)q & 15u] : (float)q;
    const int64_t i = (int64_t)(k / a.kB) * a.nb + n / a.B;
    const float ws = mul_rn(wf, elem(a.scale, i, a.s_dt));
    return kZp ? add_rn(ws, elem(a.zp, i, a.zp_dt)) : ws;
  }
};

template <int WDT, int FORM, int SM, int KIND, bool XBF>
int rg_launch(mx_backend* b, const char* name, Args& a) {
  using S8 = RgSource<WDT, FORM, SM, KIND, XBF, 8>;
  int nw = 0, grid = 0;
  MX_TRY(plan(b, a, a.M, S8::kPA + S8::kPB, XBF, &nw, &grid));
  return launch(b, name, [&] {
    if constexpr (S8::kPA + S8::kPB <= 4) {
      if (nw == 4) {
        dispatch(split_gemm_kernel<RgSource<WDT, FORM, SM, KIND, XBF, 4>, 4>, grid, 256, 0, b->stream, a);
        return;
      }
    }
    dispatch(split_gemm_kernel<S8, 8>, grid, 512, 0, b->stream, a);
  });
}

template <int WDT, int SM, int KIND, bool XBF>
int rg_forms(mx_backend* b, const char* name, const QDenseDesc& d, Args& a) {
  if constexpr (KIND == kLinear && SM == kRgCols) {
    if (d.block_size >= d.K) return rg_launch<WDT, kColumn, kRgCols, KIND, XBF>(b, name, a);
  }
  if constexpr (KIND == kLinear && SM == kRgBlk) {
    if (a.nb == 1 || a.B % kBN == 0) return rg_launch<WDT, RgForm::kRow, kRgBlk, KIND, XBF>(b, name, a);
  }
  return rg_launch<WDT, kWeight, SM, KIND, XBF>(b, name, a);
}

template <int WDT, int KIND, bool XBF>
int rg_scales(mx_backend* b, const char* name, const QDenseDesc& d, Args& a) {
  if (d.block_axis == 0 && a.kB % 4 != 0) return rg_forms<WDT, kRgRows, KIND, XBF>(b, name, d, a);
  if (d.block_axis == 0) return rg_forms<WDT, kRgCols, KIND, XBF>(b, name, d, a);
  if (a.B % 4 == 0 || a.nb == 1) return rg_forms<WDT, kRgBlk, KIND, XBF>(b, name, d, a);
  return rg_forms<WDT, kRgAny, KIND, XBF>(b, name, d, a);
}

template <int WDT, bool XBF>
int rg_dispatch(mx_backend* b, const char* name, const QDenseDesc& d, Args& a) {
  // NF4 codes are taken & 15: signed and unsigned storage are the same.
  if (d.scheme == MX_QUANT_NF4)
    return rg_scales<WDT == MX_DTYPE_INT8 ? MX_DTYPE_UINT8 : WDT == MX_DTYPE_INT4 ? MX_DTYPE_UINT4 : WDT, kNf4, XBF>(b, name, d, a);
  return d.zp ? rg_scales<WDT, kZeroPoint, XBF>(b, name, d, a) : rg_scales<WDT, kLinear, XBF>(b, name, d, a);
}

// All weight types and forms of one type of x.
template <bool XBF>
int rg_run(mx_backend* b, const char* name, const QDenseDesc& d, Args& a) {
  switch (d.w_dt) {
    case MX_DTYPE_INT8: return rg_dispatch<MX_DTYPE_INT8, XBF>(b, name, d, a);
    case MX_DTYPE_UINT8: return rg_dispatch<MX_DTYPE_UINT8, XBF>(b, name, d, a);
    case MX_DTYPE_INT4: return rg_dispatch<MX_DTYPE_INT4, XBF>(b, name, d, a);
    default: return rg_dispatch<MX_DTYPE_UINT4, XBF>(b, name, d, a);
  }
}

}  // namespace

// The kernels of bf16 x are compiled by themselves (qdense_refgemm_bf16.hip), beside those of f32 x.
int qdense_refgemm_run_bf16(mx_backend* b, const char* name, const QDenseDesc& d, sg::Args& a);

}  // namespace mx
