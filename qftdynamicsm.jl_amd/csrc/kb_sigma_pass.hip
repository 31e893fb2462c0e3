// kb_sigma_pass.hip -- the passes of one mode of the self-energy stage
// (KB_SIGMA_MODE) in one form (KB_SIGMA_FORM), kb_sigma_impl.h: compiled once
// for each pair.
#include "kb_sigma_impl.h"

namespace qftkb {

template <>
hipError_t sigma_form<KB_SIGMA_MODE, KB_SIGMA_FORM>(const SigmaArgs& a, int rows, int want, hipStream_t st) {
#if KB_SIGMA_COMPILED
  return launch_compiled_stage<KB_SIGMA_MODE, KB_SIGMA_FORM>(a, rows, st);
#else
  return launch_plan_stage<KB_SIGMA_MODE, KB_SIGMA_FORM>(a, rows, want, st);
#endif
}

template <>
hipError_t sigma_form_prepare<KB_SIGMA_MODE, KB_SIGMA_FORM>() {
#if KB_SIGMA_COMPILED
  return prepare_compiled_stage<KB_SIGMA_MODE, KB_SIGMA_FORM>();
#else
  return prepare_plan_stage<KB_SIGMA_MODE, KB_SIGMA_FORM>();
#endif
}

}  // namespace qftkb
