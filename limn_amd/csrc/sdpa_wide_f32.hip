// Float32-arithmetic attention on matrix cores (sdpa_wide.h), f32 storage.

#include "sdpa_wide.h"

namespace limn {

int launch_wide_f32(SdpaPass pass, const SdpaArgs& a) { return launch_wide_type<F32>(pass, a); }

}  // namespace limn
