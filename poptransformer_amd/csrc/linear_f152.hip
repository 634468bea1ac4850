// Linear layers of F152 weights, for linear.hip (a file of their own: they compile beside the others).
#include "common.h"
#include "formats.h"

int run_linear_f152(GemmArgs& a, int total_nb, int swiglu, hipStream_t s, const char* name) {
  if (swiglu) return dispatch_gemv<FmtF8<1>, true>(a, total_nb, s, name);
  return dispatch_gemv<FmtF8<1>, false>(a, total_nb, s, name);
}
