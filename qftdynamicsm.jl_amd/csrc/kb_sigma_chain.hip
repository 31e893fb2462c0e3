// kb_sigma_chain.hip -- self-energy stage (kb_sigma_impl.h): the 1/N chain pass.
#include "kb_sigma_impl.h"

namespace qftkb {
KB_SIGMA_MODE(SG_CHAIN)
}  // namespace qftkb
