// pk_kern_foldx_c.hip -- row kernels of the two-pass form (pk_fold_dev.hpp), modes XM_BIGGS_Y, XM_BIGGS_UPDATE, XM_BIGGS_FINAL;
// the modes are split over several translation units so they compile in parallel.
#include "pk_fold.hpp"

namespace pk {
bool launch_foldx_c(unsigned nt, dim3 grid, size_t lds, hipStream_t s, const FoldX& f, int mode,
                    const FoldX* ch, const int64_t* starts, int n) {
    switch (mode) {
        case XM_BIGGS_Y:
            return launch_foldx_kernel(k_foldx<XM_BIGGS_Y>, nt, grid, lds, s, f, ch, starts, n);
        case XM_BIGGS_UPDATE:
            return launch_foldx_kernel(k_foldx<XM_BIGGS_UPDATE>, nt, grid, lds, s, f, ch, starts, n);
        case XM_BIGGS_FINAL:
            return launch_foldx_kernel(k_foldx<XM_BIGGS_FINAL>, nt, grid, lds, s, f, ch, starts, n);
        default: return false;
    }
}
}  // namespace pk
