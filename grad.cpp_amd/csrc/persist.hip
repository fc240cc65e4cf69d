// The all-to-all persistent kernel's variants, in a translation unit of their own: they
// are most of the library's compile time and nothing else needs their code.
#include "kernel_tables.h"

namespace gh {

// row_lds: the sampler's working row fits in LDS.
template <bool ROW_LDS, bool FEED>
static PersistKernel persist_kernel_of(const Shape& sh) {
    if (sh.head_size() != 64) return nullptr;
    const int d = sh.d_model, F = sh.d_ff();
    if (sh.modern()) {
        if (d == 768 && F == 2048) return persist_decode_kernel<3, 8, true, ROW_LDS, FEED>;
        return nullptr;
    }
    if (d == 512) return persist_decode_kernel<2, 8, false, ROW_LDS, FEED>;
    if (d == 768) return persist_decode_kernel<3, 12, false, ROW_LDS, FEED>;
    if (d == 1024) return persist_decode_kernel<4, 16, false, ROW_LDS, FEED>;
    return nullptr;
}

PersistKernel persist_kernel_for(const Shape& sh, bool row_lds, bool feed) {
    if (feed) return row_lds ? persist_kernel_of<true, true>(sh) : persist_kernel_of<false, true>(sh);
    return row_lds ? persist_kernel_of<true, false>(sh) : persist_kernel_of<false, false>(sh);
}

#ifdef GH_PICK_TICKS
bool read_pick_ticks(unsigned long long (&t)[32]) {
    return hipMemcpyFromSymbol(t, HIP_SYMBOL(g_pick_ticks), sizeof(t)) == hipSuccess;
}
#endif

}  // namespace gh
