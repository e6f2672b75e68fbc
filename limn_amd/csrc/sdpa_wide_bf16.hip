// Float32-arithmetic attention on matrix cores (sdpa_wide.h), bf16 storage.

#include "sdpa_wide.h"

namespace limn {

int launch_wide_bf16(SdpaPass pass, const SdpaArgs& a) { return launch_wide_type<BF16>(pass, a); }

}  // namespace limn
