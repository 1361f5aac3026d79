// FusedQuantizedDense past the GEMV for the layouts the bf16 GEMM does not take: the reference's own
// scale layout [K, ceil(N/B)] (BlockAxis = 1), f32 x, zero points and NF4 (fused_ops.go:204-234;
// quantizeddense.go:586-650).  The contraction is split_gemm.h's: f32 operands in three exact bf16
// parts on the bf16 matrix cores.  No copy of the weight matrix is ever made.
//
// Three forms, by where the scale enters:
//   row      reference layout, one column block per 128-column tile (B % 128 == 0 or one block),
//            linear scheme: x * s is formed and rounded once per (row, k) of the tile, the codes
//            stay exact; 3 products per term.  Zero points add x . zp, summed in f32 beside it.
//   column   one scale per output column, linear scheme, no zero points: the sums of x * w, scaled
//            once; 3 products (1 with bf16 x).
//   weight   everything else: the weight factor formed as the reference forms it (w*s, w*s + zp
//            with its two roundings, nf4[w]*s) and split; 6 products (3 with bf16 x).
// The reference rounds (x*w)*s per term and sums in k order; the results stay within the f32
// accumulation bound of its sum.  The bias is added after the sum (the reference starts from it),
// then the reference activation (act_ref) and the output dtype.
#include <algorithm>

#include "split_gemm.h"

namespace mx {
namespace {

using namespace sg;

enum RgForm { kRow, kColumn, kWeight };
// Where the weight form finds the scales (and zero points) of 4 consecutive columns of row k.
enum RgScales {
  kRgCols = 0,  // one per column of a scale row: [ceil(K/B), N]
  kRgBlk = 1,   // [K, ceil(N/B)] with B % 4 == 0: one
  kRgAny = 2    // [K, ceil(N/B)], any B: one per column
};

// Weights [K, N]: thread t converts columns 4 cq .. 4 cq + 3 of rows 4 j .. 4 j + 3 of a block, with
// j's low bit in the thread's (so that lane pairs write whole 16-byte chunks).
template <int WDT, int FORM, int SM, bool XBF>
struct RgSource {
  static constexpr bool kXbf = XBF;
  static constexpr bool kRow = FORM == RgForm::kRow, kCol = FORM == kColumn;
  static constexpr int kPA = XBF && FORM != RgForm::kRow ? 1 : 3;
  static constexpr int kPB = FORM == kWeight ? 3 : 1;
  static constexpr bool kI4 = WDT == MX_DTYPE_INT4 || WDT == MX_DTYPE_UINT4;
  static constexpr bool kSigned = WDT == MX_DTYPE_INT4 || WDT == MX_DTYPE_INT8;
  static constexpr int kScales = FORM != kWeight ? 1 : SM == kRgBlk ? 1 : 4;  // per row

  struct Regs {
    uint32_t w[4];
    uint32_t s[4][kScales], z[4][kScales];  // raw words (kRgCols with bf16: two pairs)
    uint32_t ssh[4][kScales], zsh[4][kScales];
  };
  int cq, j, ncl;
  const char* wp;

  __device__ __forceinline__ RgSource(const Args& a, int t, int n0) {
    cq = (t >> 1) & 31;
    j = (t & 1) | (t >> 6) << 1;
    // N % 16 == 0: the 4 columns are all in range or all past N (then column 0 is read and the
    // outputs are not stored).
    ncl = n0 + 4 * cq < a.N ? n0 + 4 * cq : 0;
    wp = (const char*)a.w + (kI4 ? ncl / 2 : ncl);
  }
  // The aligned word holding element i of an f32 or bf16 array, and the shift that moves a bf16
  // element to its high half.
  static __device__ __forceinline__ void word(const void* p, int64_t i, bool bf, uint32_t& w, uint32_t& sh) {
    const uintptr_t ad = (uintptr_t)p + (uintptr_t)i * (bf ? 2 : 4);
    w = *(const uint32_t*)(ad & ~(uintptr_t)3);
    sh = bf && (ad & 2) == 0 ? 16u : 0u;
  }
  __device__ __forceinline__ void load(const Args& a, int kb, Regs& R) const {
    const int k0 = kb * kBK + 4 * j;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = min(k0 + e, a.K - 1);
      const char* p = wp + (int64_t)k * (kI4 ? a.N / 2 : a.N);
      if constexpr (kI4)
        R.w[e] = *(const uint16_t*)p;
      else
        R.w[e] = *(const uint32_t*)p;
      if constexpr (FORM == kWeight) {
        const bool sbf = a.s_dt == MX_DTYPE_BFLOAT16, zbf = a.zp_dt == MX_DTYPE_BFLOAT16;
        if constexpr (SM == kRgCols) {
          const int64_t i = (int64_t)(k / a.B) * a.N + ncl;
          // bf16: 8 bytes are the 4 scales; f32: 16 (two loads, so that the form is one).
          const char* sp = (const char*)a.scale + i * (sbf ? 2 : 4);
          const u32x2_v lo = *(const u32x2_v*)sp, hi = *(const u32x2_v*)(sp + (sbf ? 0 : 8));
          R.s[e][0] = lo[0], R.s[e][1] = lo[1], R.s[e][2] = hi[0], R.s[e][3] = hi[1];
          if (a.zp) {
            const char* zq = (const char*)a.zp + i * (zbf ? 2 : 4);
            const u32x2_v zl = *(const u32x2_v*)zq, zh = *(const u32x2_v*)(zq + (zbf ? 0 : 8));
            R.z[e][0] = zl[0], R.z[e][1] = zl[1], R.z[e][2] = zh[0], R.z[e][3] = zh[1];
          }
        } else {
#pragma unroll
          for (int c = 0; c < kScales; ++c) {
            const int64_t i = (int64_t)k * a.nb + (ncl + c) / a.B;
            word(a.scale, i, sbf, R.s[e][c], R.ssh[e][c]);
            if (a.zp) word(a.zp, i, zbf, R.z[e][c], R.zsh[e][c]);
          }
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
    if constexpr (SM == kRgCols)
      return bf ? __uint_as_float(c & 1 ? s[(c >> 1) % kScales] & 0xFFFF0000u : s[(c >> 1) % kScales] << 16)
                : __uint_as_float(s[c % kScales]);
    else
      return __uint_as_float((s[c % kScales] << sh[c % kScales]) & (bf ? 0xFFFF0000u : ~0u));
  }
  __device__ __forceinline__ void stage(const Args& a, int kb, const Regs& R, const float* table, char* Bs, int& odd) const {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      char* dst = Bs + chunk_at(c * 32 + cq, j >> 1) + 8 * (j & 1);
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int q = code(R.w[e], c);
        if constexpr (FORM == kWeight) {
          const bool sbf = a.s_dt == MX_DTYPE_BFLOAT16, zbf = a.zp_dt == MX_DTYPE_BFLOAT16;
          const float wf = a.nf4 ? table[(uint32_t)q & 15u] : (float)q;
          const float ws = mul_rn(wf, scale_of(R.s[e], R.ssh[e], c, sbf));
          v[e] = a.zp ? add_rn(ws, scale_of(R.z[e], R.zsh[e], c, zbf)) : ws;
          if (kb * kBK + 4 * j + e >= a.K) v[e] = 0.0f;  // x is zero there, but 0 * inf is not
        } else {
          v[e] = (float)q;
        }
      }
      if constexpr (FORM == kWeight) {
        if (fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))) > MX_SPLIT_MAX) odd = 1;
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
  // The weight factor of (k, n) as the reference forms it (column form: without its scale).
  __device__ __forceinline__ float value(const Args& a, int k, int n, const float* table) const {
    const int q = decode_weight(a.w, (int64_t)k * a.N + n, WDT);
    const float wf = a.nf4 ? table[(uint32_t)q & 15u] : (float)q;
    if constexpr (FORM == kColumn) return wf;
    const int64_t i = SM == kRgCols ? (int64_t)(k / a.B) * a.N + n : (int64_t)k * a.nb + n / a.B;
    const float ws = mul_rn(wf, elem(a.scale, i, a.s_dt));
    return a.zp ? add_rn(ws, elem(a.zp, i, a.zp_dt)) : ws;
  }
};

template <int WDT, bool XBF>
void rg_dispatch(const QDenseDesc& d, const Args& a, int grid, hipStream_t st) {
  const bool linear = d.scheme == MX_QUANT_LINEAR;
  if (d.block_axis == 0) {
    if (linear && !d.zp && d.block_size >= d.K)
      dispatch(split_gemm_kernel<RgSource<WDT, kColumn, kRgCols, XBF>>, grid, kThreads, 0, st, a);
    else
      dispatch(split_gemm_kernel<RgSource<WDT, kWeight, kRgCols, XBF>>, grid, kThreads, 0, st, a);
  } else if (linear && (a.nb == 1 || a.B % kBN == 0)) {
    dispatch(split_gemm_kernel<RgSource<WDT, RgForm::kRow, kRgBlk, XBF>>, grid, kThreads, 0, st, a);
  } else if (a.B % 4 == 0) {
    dispatch(split_gemm_kernel<RgSource<WDT, kWeight, kRgBlk, XBF>>, grid, kThreads, 0, st, a);
  } else {
    dispatch(split_gemm_kernel<RgSource<WDT, kWeight, kRgAny, XBF>>, grid, kThreads, 0, st, a);
  }
}

}  // namespace

bool qdense_refgemm_fits(const QDenseDesc& d) {
  auto aligned = [](const void* p, size_t al) { return ((uintptr_t)p % al) == 0; };
  const bool xbf = d.x_dt == MX_DTYPE_BFLOAT16;
  const bool packed = dtype_is_packed(d.w_dt);
  if (!(d.scheme == MX_QUANT_LINEAR || d.scheme == MX_QUANT_NF4)) return false;
  if (!(d.x_dt == MX_DTYPE_FLOAT32 || xbf) || d.M < 1 || d.K < 8 || d.N < 16 || d.N % 16 != 0) return false;
  if (d.K % (xbf ? 8 : 4) != 0 || !aligned(d.x, 16) || !aligned(d.w, packed ? 8 : 16)) return false;
  if (d.M >= (int64_t)1 << 30 || d.K >= (int64_t)1 << 30 || d.N >= (int64_t)1 << 30) return false;
  if (d.block_axis == 0) {
    // 4 consecutive scales of a row: vector loads.
    if (!aligned(d.scale, 16) || (d.zp && !aligned(d.zp, 16))) return false;
  }
  return true;
}

int qdense_refgemm_run(mx_backend* b, const QDenseDesc& d, const char* name) {
  Args a{};
  a.x = d.x;
  a.w = (const uint8_t*)d.w;
  a.scale = d.scale;
  a.zp = d.zp;
  a.bias = d.bias;
  a.out = d.out;
  a.M = (int)d.M;
  a.K = (int)d.K;
  a.N = (int)d.N;
  a.s_dt = d.s_dt;
  a.zp_dt = d.zp ? d.zp_dt : MX_DTYPE_FLOAT32;
  a.b_dt = d.b_dt;
  a.act = d.act;
  a.nf4 = d.scheme == MX_QUANT_NF4 ? 1 : 0;
  a.B = (int)std::min<int64_t>(d.block_size, d.block_axis == 0 ? d.K : d.N);
  a.nb = (int)((d.N + a.B - 1) / a.B);
  int grid = 0;
  MX_TRY(plan(b, a, d.M, &grid));
  const bool xbf = d.x_dt == MX_DTYPE_BFLOAT16;
  hipStream_t st = b->stream;
  return launch(b, name, [&] {
    auto go = [&](auto wdt) {
      constexpr int W = decltype(wdt)::value;
      xbf ? rg_dispatch<W, true>(d, a, grid, st) : rg_dispatch<W, false>(d, a, grid, st);
    };
    switch (d.w_dt) {
      case MX_DTYPE_INT8: go(std::integral_constant<int, MX_DTYPE_INT8>{}); break;
      case MX_DTYPE_UINT8: go(std::integral_constant<int, MX_DTYPE_UINT8>{}); break;
      case MX_DTYPE_INT4: go(std::integral_constant<int, MX_DTYPE_INT4>{}); break;
      default: go(std::integral_constant<int, MX_DTYPE_UINT4>{}); break;
    }
  });
}

}  // namespace mx
