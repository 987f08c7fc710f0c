// The wavefront x passes of one group of line lengths.
#include "xpass_impl.hpp"

namespace coral {

XLENGTHS_C(XINSTANCE)

}  // namespace coral
