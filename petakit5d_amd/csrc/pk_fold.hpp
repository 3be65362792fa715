// pk_fold.hpp -- host-side plan and launchers of the two-pass form (pk_fold_dev.hpp).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pk_fold_dev.hpp"
#include "pk_launch.hpp"

namespace pk {

// Shapes of the two fold passes for one padded size.  x and c hold everything
// but the pointers of a call.
struct FoldPlan {
    bool on = false;
    int a = 0, m = 0, b = 1, T = 8;
    unsigned xnt = 0, cnt = 0;
    size_t xlds = 0, clds = 0;
    int64_t xblocks = 0;  // row-pass blocks
    int cblocks = 0;      // column-pass blocks
    uint64_t layout = 0;  // spectrum order: OTFs of different layouts are different entries
    FoldX x{};
    FoldC c{};
};

// Plan of size n1 x n2 x n3 (spectrum pitch hp); on = false where the form does
// not fit.
FoldPlan fold_plan(int64_t n1, int64_t n2, int64_t n3, int64_t hp);

// mode: an XM_* of a call's row passes; n = 0: the volume of f, else the chunks at ch
hipError_t launch_foldx(unsigned nt, dim3 grid, size_t lds, hipStream_t s, const FoldX& f, int mode,
                        const FoldX* ch, const int64_t* starts, int n);
// mode CM_FWD, CM_CONV or CM_CONVJ; n = 0: the volume of f, else the chunks at ch
hipError_t launch_foldc(unsigned nt, dim3 grid, size_t lds, hipStream_t s, const FoldC& f, int mode, const FoldC* ch,
                        const int64_t* starts, int n);

// The row kernels' launchers (pk_kern_foldx_*.hip); false: another file's mode.
bool launch_foldx_a(unsigned nt, dim3 grid, size_t lds, hipStream_t s, const FoldX& f, int mode,
                    const FoldX* ch, const int64_t* starts, int n);
bool launch_foldx_b(unsigned nt, dim3 grid, size_t lds, hipStream_t s, const FoldX& f, int mode,
                    const FoldX* ch, const int64_t* starts, int n);
bool launch_foldx_c(unsigned nt, dim3 grid, size_t lds, hipStream_t s, const FoldX& f, int mode,
                    const FoldX* ch, const int64_t* starts, int n);
bool launch_foldx_d(unsigned nt, dim3 grid, size_t lds, hipStream_t s, const FoldX& f, int mode,
                    const FoldX* ch, const int64_t* starts, int n);
template <class K>
inline bool launch_foldx_kernel(K kernel, unsigned nt, dim3 grid, size_t lds, hipStream_t s, const FoldX& f,
                                const FoldX* ch, const int64_t* starts, int n) {
    if (lds > 65536) allow_large_lds(kernel);
    hipLaunchKernelGGL(kernel, grid, dim3(nt), lds, s, f, ch, starts, n);
    return true;
}

}  // namespace pk
