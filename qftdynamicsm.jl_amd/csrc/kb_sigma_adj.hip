// kb_sigma_adj.hip -- self-energy stage (kb_sigma_impl.h): the sunset's adjoint.
#include "kb_sigma_impl.h"

namespace qftkb {
KB_SIGMA_MODE(SG_SUNSET_ADJ)
}  // namespace qftkb
