// The resident step kernel's variants (kernels_resident.h), in a translation unit of their own.
#include "kernel_tables.h"

namespace gh {

template <int KD, int KF, bool MODERN>
static ResidentKernel of_rows(int batch) {
    if (batch <= 4) return resident_layers_kernel<KD, KF, MODERN, 4>;
    if (batch <= 8) return resident_layers_kernel<KD, KF, MODERN, 8>;
    return batch <= kResidentRows ? resident_layers_kernel<KD, KF, MODERN, 16> : nullptr;
}

ResidentKernel resident_kernel_for(const Shape& sh, int batch) {
    if (sh.head_size() != 64 || batch < 2) return nullptr;
    if (sh.modern()) return sh.d_model == 768 && sh.d_ff() == 2048 ? of_rows<3, 8, true>(batch) : nullptr;
    if (sh.d_model == 512) return of_rows<2, 8, false>(batch);
    if (sh.d_model == 768) return of_rows<3, 12, false>(batch);
    return nullptr;
}

}  // namespace gh
