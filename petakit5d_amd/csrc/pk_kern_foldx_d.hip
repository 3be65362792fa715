// pk_kern_foldx_d.hip -- row kernels of the two-pass form (pk_fold_dev.hpp), modes XM_R2C, XM_PREP_U16, XM_PREP_F32;
// the modes are split over several translation units so they compile in parallel.
#include "pk_fold.hpp"

namespace pk {
bool launch_foldx_d(unsigned nt, dim3 grid, size_t lds, hipStream_t s, const FoldX& f, int mode,
                    const FoldX* ch, const int64_t* starts, int n) {
    switch (mode) {
        case XM_R2C:
            return launch_foldx_kernel(k_foldx<XM_R2C>, nt, grid, lds, s, f, ch, starts, n);
        case XM_PREP_U16:
            return launch_foldx_kernel(k_foldx<XM_PREP_U16>, nt, grid, lds, s, f, ch, starts, n);
        case XM_PREP_F32:
            return launch_foldx_kernel(k_foldx<XM_PREP_F32>, nt, grid, lds, s, f, ch, starts, n);
        default: return false;
    }
}
}  // namespace pk
