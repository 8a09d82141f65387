// The fused update kernels for bfloat16 storage, instantiated apart from the other
// storage type's so that the two compile side by side.
#include "ndc_backend_hip.h"
#include "ndc_fused_api.h"

namespace ndc {
namespace fused {
NDC_FUSED_ENTRY_POINTS(template, bf16_t)
}  // namespace fused
}  // namespace ndc
