// FusedQuantizedDense by the split contraction (qdense_refgemm.h): the kernels of bf16 x.
#include "qdense_refgemm.h"

namespace mx {

int qdense_refgemm_run_bf16(mx_backend* b, const char* name, const QDenseDesc& d, sg::Args& a) {
  return rg_run<true>(b, name, d, a);
}

}  // namespace mx
