// One of the translation units of the library's gfx950 kernels (see kernels_mmf.hip).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gq_device.h"
#include "gq_params.h"

#define GQ_TEMPLATES_ONLY
#include "mmf.hip.inc"
#undef GQ_TEMPLATES_ONLY

#include "mmfw.hip.inc"
#include "mmfx.hip.inc"
