// kb_sigma_plain.hip -- self-energy stage (kb_sigma_impl.h): the sunset of a caller's lattices.
#include "kb_sigma_impl.h"

namespace qftkb {
KB_SIGMA_MODE(SG_PLAIN)
}  // namespace qftkb
