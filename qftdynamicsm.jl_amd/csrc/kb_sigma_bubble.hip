// kb_sigma_bubble.hip -- self-energy stage (kb_sigma_impl.h): the 1/N bubble pass.
#include "kb_sigma_impl.h"

namespace qftkb {
KB_SIGMA_MODE(SG_BUBBLE)
}  // namespace qftkb
