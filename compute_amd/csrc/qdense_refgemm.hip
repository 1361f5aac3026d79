// FusedQuantizedDense by the split contraction (qdense_refgemm.h): what it takes, its arguments, and the
// kernels of f32 x.
#include "qdense_refgemm.h"

namespace mx {

bool qdense_refgemm_fits(const QDenseDesc& d) {
  auto aligned = [](const void* p, size_t al) { return ((uintptr_t)p % al) == 0; };
  const bool xbf = d.x_dt == MX_DTYPE_BFLOAT16;
  const bool packed = dtype_is_packed(d.w_dt);
  if (!(d.scheme == MX_QUANT_LINEAR || d.scheme == MX_QUANT_NF4)) return false;
  if (!(d.x_dt == MX_DTYPE_FLOAT32 || xbf) || d.M < 1 || d.K < 8 || d.N < 16 || d.N % 16 != 0) return false;
  if (d.K % (xbf ? 8 : 4) != 0 || !aligned(d.x, 16) || !aligned(d.w, packed ? 8 : 16)) return false;
  // A tile's rows of x and a block's rows of weights are addressed by 32-bit offsets; past these limits
  // the GEMV per four rows or the reference-order kernel runs.
  if (d.M >= (int64_t)1 << 30 || d.K > (int64_t)1 << 22 || d.N > (int64_t)1 << 26) return false;
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
  a.B = d.block_axis == 0 ? 1 : (int)std::min<int64_t>(d.block_size, d.N);
  a.kB = d.block_axis == 0 ? (int)std::min<int64_t>(d.block_size, d.K) : 1;
  a.nb = (int)((d.N + a.B - 1) / a.B);
  return d.x_dt == MX_DTYPE_BFLOAT16 ? qdense_refgemm_run_bf16(b, name, d, a) : rg_run<false>(b, name, d, a);
}

}  // namespace mx
