// pk_kern_foldx_a.hip -- row kernels of the two-pass form (pk_fold_dev.hpp), modes XM_RATIO, XM_RATIO_U16, XM_OMW_FINAL;
// the modes are split over several translation units so they compile in parallel.
#include "pk_fold.hpp"

namespace pk {
bool launch_foldx_a(unsigned nt, dim3 grid, size_t lds, hipStream_t s, const FoldX& f, int mode,
                    const FoldX* ch, const int64_t* starts, int n) {
    switch (mode) {
        case XM_RATIO:
            return launch_foldx_kernel(k_foldx<XM_RATIO>, nt, grid, lds, s, f, ch, starts, n);
        case XM_RATIO_U16:
            return launch_foldx_kernel(k_foldx<XM_RATIO_U16>, nt, grid, lds, s, f, ch, starts, n);
        case XM_OMW_FINAL:
            return launch_foldx_kernel(k_foldx<XM_OMW_FINAL>, nt, grid, lds, s, f, ch, starts, n);
        default: return false;
    }
}
}  // namespace pk
