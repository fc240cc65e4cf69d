// The resident step kernel's variants (kernels_resident.h), in a translation unit of their own.
#include "kernel_tables.h"

namespace gh {

template <int KD, int KF, bool MODERN>
static ResidentKernel of_rows(int batch, bool rounds) {
    // (up to 4 sequences a second round begins beyond 5120 positions, where a step of 4 goes from 351 us to 467)
    if (batch <= 4) return rounds ? nullptr : resident_layers_kernel<KD, KF, MODERN, 4, false>;
    if (batch <= 8) return rounds ? resident_layers_kernel<KD, KF, MODERN, 8, true> : resident_layers_kernel<KD, KF, MODERN, 8, false>;
    if (batch > kResidentRows) return nullptr;
    return rounds ? resident_layers_kernel<KD, KF, MODERN, 16, true> : resident_layers_kernel<KD, KF, MODERN, 16, false>;
}

ResidentKernel resident_kernel_for(const Shape& sh, int batch, int items) {
    if (sh.head_size() != 64 || batch < 2 || items > kResidentItems) return nullptr;
    const bool rounds = items > 2 * kResidentGrid;
    if (sh.modern()) return sh.d_model == 768 && sh.d_ff() == 2048 ? of_rows<3, 8, true>(batch, rounds) : nullptr;
    if (sh.d_model == 512) return of_rows<2, 8, false>(batch, rounds);
    if (sh.d_model == 768) return of_rows<3, 12, false>(batch, rounds);
    return nullptr;
}

}  // namespace gh
