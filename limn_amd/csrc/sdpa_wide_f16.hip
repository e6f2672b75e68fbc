// Float32-arithmetic attention on matrix cores (sdpa_wide.h), f16 storage.

#include "sdpa_wide.h"

namespace limn {

int launch_wide_f16(SdpaPass pass, const SdpaArgs& a) { return launch_wide_type<F16>(pass, a); }

}  // namespace limn
