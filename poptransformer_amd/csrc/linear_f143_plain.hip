// Linear layers of F143 weights without the codes that the hardware's conversion does not know (PTA_W_F143_PLAIN), for linear.hip.
#include "common.h"
#include "formats.h"

int run_linear_f143_plain(GemmArgs& a, int total_nb, int swiglu, hipStream_t s, const char* name) {
  if (swiglu) return dispatch_gemv<FmtF143Plain, true>(a, total_nb, s, name);
  return dispatch_gemv<FmtF143Plain, false>(a, total_nb, s, name);
}
