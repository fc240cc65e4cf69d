// The XCD-sharded persistent kernel's variants (see persist.hip).
#include "kernel_tables.h"

namespace gh {

XcdKernel xcd_kernel_for(const Shape& sh, bool row_lds, bool feed) {
    if (!sh.modern() || sh.head_size() != 64 || sh.d_model != 768) return nullptr;
    if (feed) return row_lds ? xcd_decode_kernel<3, true, true> : xcd_decode_kernel<3, false, true>;
    return row_lds ? xcd_decode_kernel<3, true, false> : xcd_decode_kernel<3, false, false>;
}

}  // namespace gh
