// The wavefront x passes of one group of line lengths.
#include "xpass_impl.hpp"

namespace coral {

XLENGTHS_B(XINSTANCE)

}  // namespace coral
