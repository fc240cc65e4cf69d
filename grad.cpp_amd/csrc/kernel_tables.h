// Which compiled variant of a persistent kernel serves a model shape; the variants
// themselves are instantiated in persist.hip and xcd.hip.
#pragma once

#include "checkpoint.h"
#include "kernels_persist.h"
#include "kernels_resident.h"
#include "kernels_xcd.h"

namespace gh {

using PersistKernel = void (*)(const PersistParams);
using XcdKernel = void (*)(const XcdParams);
using ResidentKernel = void (*)(const ResidentParams);

// The shapes the persistent kernel is built for (head size 64, d_model and FFN
// width multiples of 256); nullptr for anything else.
// row_lds: the sampler's working row fits in LDS.
// feed: the variant that reports its picks to the host and can be told to stop.
PersistKernel persist_kernel_for(const Shape& sh, bool row_lds, bool feed = false);

// The Llama block at d_model 768; nullptr for anything else.
XcdKernel xcd_kernel_for(const Shape& sh, bool row_lds, bool feed);

// All layers of a step of 2 to kResidentRows sequences whose attention is cut into `items` runs of
// positions; nullptr for what it is not built for.
ResidentKernel resident_kernel_for(const Shape& sh, int batch, int items);

#ifdef GH_PICK_TICKS
bool read_pick_ticks(unsigned long long (&t)[32]);
#endif

}  // namespace gh
