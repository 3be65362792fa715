// pk_deskew.hip -- deskew of a deconvolved stage-scan volume
// (pointDetection/llsmtools/transforms/deskewFrame3D.m:26-70, called from
// microscopeDataProcessing/decon/RLdecon.m:448-449).
//
// The reference shears the volume with imwarp: output column c (1-based) of
// plane p takes the input at column x = c - xstep * p - xshift, same row, same
// plane, linearly interpolated, where dx = cos(angle) dz / xyPixelSize,
// (xstep, xshift) = (dx, -dx) or (-dx, dx + ceil((nz - 1) dx)) when reversed,
// the output is ceil((nz - 1) dx) + nx columns wide and 'Crop' trims
// floor(nx / 2) (when that width reaches 2 nx) or floor(ceil((nz - 1) dx) / 2)
// columns off each side.  imwarp pads the input with one column of the fill
// value (0) on each side, so positions in [0, 1) and (nx, nx + 1] blend the edge
// column with 0 and positions further out are 0.
//
// MATLAB volumes are column-major: a column (fixed x, z) is ny contiguous
// floats, and every value of an output column uses the same two input columns
// and weight.  A block takes eight neighbouring output columns: they read nine
// neighbouring input columns, each once.  Coalesced and HBM-bound (4 bytes read
// + 4 written per value).  512x512x256 at 31.5 degrees, dz 0.2: 0.139 ms; with a
// block per output column 0.172 ms (both columns of a blend read by every block:
// 512 instead of 268 MB past L2).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "pk_engine.hpp"

namespace pk {

struct Affine3 {
    double a[4][4];  // row-vector convention: [x y z 1] = [u v w 1] * a
};

struct DeskewGeom {
    int64_t nx_out;
    double xstep, xshift;
};

DeskewGeom deskew_geometry(const int64_t dims[3], double angle, double dz, double xy, bool reverse, bool crop) {
    const int64_t nx = dims[1], nz = dims[2];
    const double dx = std::cos(angle * M_PI / 180.0) * dz / xy;
    const double span = std::ceil((double)(nz - 1) * dx);
    DeskewGeom g;
    g.xstep = reverse ? -dx : dx;
    g.xshift = reverse ? dx + span : -dx;
    g.nx_out = (int64_t)span + nx;
    if (crop) {
        const int64_t cw = g.nx_out >= 2 * nx ? nx / 2 : (int64_t)std::floor(span / 2.0);
        g.xshift -= (double)cw;
        g.nx_out -= 2 * cw;
    }
    return g;
}

// VEC: ny % 4 == 0 and 16-byte aligned buffers, so every column is whole
// float4s (one 16-byte load per operand and one store per four values).
constexpr int kDeskewRun = 8;
template <bool VEC>
__global__ void __launch_bounds__(256) k_deskew(const float* __restrict__ vol, float* __restrict__ out, int64_t ny,
                                                int64_t nx, int64_t nx_out, double xstep, double xshift, uint32_t runs,
                                                uint32_t total, uint32_t per_xcd) {
    using V = std::conditional_t<VEC, float4, float>;
    // one block per run of kDeskewRun output columns of a plane; its threads
    // walk down the columns.  Blocks go round-robin to the 8 XCDs: each XCD
    // walks a contiguous range
    const uint32_t item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (item >= total) return;
    const int64_t p = item / runs, c0 = (int64_t)(item - (uint32_t)p * runs) * kDeskewRun;
    const int n = (int)(nx_out - c0 < kDeskewRun ? nx_out - c0 : kDeskewRun);
    const int64_t rows = VEC ? ny / 4 : ny;
    auto zero = [] {
        if constexpr (VEC) return make_float4(0.f, 0.f, 0.f, 0.f);
        else return 0.f;
    };
    auto blend = [](const V& a, const V& b, float f) {
        if constexpr (VEC)
            return make_float4(a.x + f * (b.x - a.x), a.y + f * (b.y - a.y), a.z + f * (b.z - a.z),
                               a.w + f * (b.w - a.w));
        else return a + f * (b - a);
    };
    // 1-based input column of every output column; outside [0, nx + 1]: 0s
    int64_t i0[kDeskewRun];
    float f[kDeskewRun];
    bool any = false, row = n == kDeskewRun;  // row: neighbours read neighbours
#pragma unroll
    for (int k = 0; k < kDeskewRun; ++k) {
        const double x = (double)(c0 + k + 1) - xstep * (double)(p + 1) - xshift;
        const bool in = k < n && x >= 0.0 && x <= (double)(nx + 1);
        const double x0 = std::floor(in ? x : -1.0);
        i0[k] = (int64_t)x0;  // 0 ... nx + 1, or -1
        f[k] = in ? (float)(x - x0) : 0.f;
        any |= in;
        row = row && in && (k == 0 || i0[k] == i0[k > 0 ? k - 1 : 0] + 1);
    }
    V* __restrict__ o = reinterpret_cast<V*>(out + (p * nx_out + c0) * ny);
    const V* __restrict__ src = reinterpret_cast<const V*>(vol + p * ny * nx);
    auto col = [&](int64_t i, int64_t r) { return i >= 1 && i <= nx ? src[(i - 1) * rows + r] : zero(); };
    for (int64_t r = threadIdx.x; r < rows; r += blockDim.x) {
        if (row) {
            V v[kDeskewRun + 1];
#pragma unroll
            for (int k = 0; k <= kDeskewRun; ++k) v[k] = col(i0[0] + k, r);
#pragma unroll
            for (int k = 0; k < kDeskewRun; ++k) o[k * rows + r] = blend(v[k], v[k + 1], f[k]);
        } else {
            for (int k = 0; k < n; ++k) {
                const double x = (double)(c0 + k + 1) - xstep * (double)(p + 1) - xshift;
                if (!any || !(x >= 0.0 && x <= (double)(nx + 1))) {
                    o[k * rows + r] = zero();
                    continue;
                }
                const double x0 = std::floor(x);
                const int64_t i = (int64_t)x0;
                o[k * rows + r] = blend(col(i, r), col(i + 1, r), (float)(x - x0));
            }
        }
    }
}

void launch_deskew(const float* vol, float* out, const int64_t dims[3], const DeskewGeom& g, hipStream_t s) {
    const int64_t cols = g.nx_out * dims[2];
    if (cols <= 0 || dims[0] <= 0) return;
    const bool vec = dims[0] % 4 == 0 && reinterpret_cast<uintptr_t>(vol) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(out) % 16 == 0;
    const int64_t per_col = vec ? dims[0] / 4 : dims[0];  // threads' work items per column
    const unsigned nt = per_col >= 256 ? 256u : (unsigned)((per_col + 63) / 64 * 64);
    // the dispatch's grid size counts work-items in 32 bits
    if (cols * (int64_t)nt > 0xFFFFFFFFll) fail(PK_ERR_UNSUPPORTED_SIZE, "deskewed volume has too many columns");
    const int64_t runs = (g.nx_out + kDeskewRun - 1) / kDeskewRun, total = runs * dims[2], per_xcd = (total + 7) / 8;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(per_xcd * 8)), dim3(nt), 0, s, vol, out, dims[0], dims[1], g.nx_out,
                           g.xstep, g.xshift, (uint32_t)runs, (uint32_t)total, (uint32_t)per_xcd);
    };
    if (vec) go(k_deskew<true>);
    else go(k_deskew<false>);
    PK_HIP(hipGetLastError());
}

}  // namespace pk

namespace pk {

// Affine resampling of a column-major volume, imwarp-style: output voxel
// (row r, column c, page p), 1-based world point (u, v, w) = (c, r, p), reads
// the input at [x y z 1] = [u v w 1] * inv_m (row-vector convention, x the
// column, y the row, z the page), trilinear over the input padded with one
// voxel of the fill value 0 on every side (rotateFrame3D.m:46-100 resamples
// through imwarp this way).  One block per output column; threads walk down it.
__global__ void __launch_bounds__(256) k_affine3d(const float* __restrict__ vol, float* __restrict__ out, int64_t ny,
                                                  int64_t nx, int64_t nz, int64_t oy, int64_t ox, Affine3 m) {
    const int64_t col = blockIdx.x;
    const int64_t c = col % ox, p = col / ox;
    const double u = (double)(c + 1), w = (double)(p + 1);
    const double bx = u * m.a[0][0] + w * m.a[2][0] + m.a[3][0];
    const double by = u * m.a[0][1] + w * m.a[2][1] + m.a[3][1];
    const double bz = u * m.a[0][2] + w * m.a[2][2] + m.a[3][2];
    float* __restrict__ o = out + col * oy;
    for (int64_t r = threadIdx.x; r < oy; r += blockDim.x) {
        const double v = (double)(r + 1);
        const double x = bx + v * m.a[1][0], y = by + v * m.a[1][1], z = bz + v * m.a[1][2];
        float val = 0.f;
        if (x > -1.0 && x < (double)(nx + 2) && y > -1.0 && y < (double)(ny + 2) && z > -1.0 && z < (double)(nz + 2)) {
            const double fx0 = std::floor(x), fy0 = std::floor(y), fz0 = std::floor(z);
            const int64_t ix = (int64_t)fx0, iy = (int64_t)fy0, iz = (int64_t)fz0;  // 1-based lower corner
            const float fx = (float)(x - fx0), fy = (float)(y - fy0), fz = (float)(z - fz0);
            float cval[2][2][2];
#pragma unroll
            for (int dz = 0; dz < 2; ++dz)
#pragma unroll
                for (int dx = 0; dx < 2; ++dx)
#pragma unroll
                    for (int dy = 0; dy < 2; ++dy) {
                        const int64_t jx = ix + dx, jy = iy + dy, jz = iz + dz;
                        const bool in = jx >= 1 && jx <= nx && jy >= 1 && jy <= ny && jz >= 1 && jz <= nz;
                        cval[dz][dx][dy] = in ? vol[(jy - 1) + ny * ((jx - 1) + nx * (jz - 1))] : 0.f;
                    }
            float pl[2];
#pragma unroll
            for (int dz = 0; dz < 2; ++dz) {
                const float a = cval[dz][0][0] + fy * (cval[dz][0][1] - cval[dz][0][0]);
                const float b = cval[dz][1][0] + fy * (cval[dz][1][1] - cval[dz][1][0]);
                pl[dz] = a + fx * (b - a);
            }
            val = pl[0] + fz * (pl[1] - pl[0]);
        }
        o[r] = val;
    }
}

// The same for a transform that keeps dim-1 rows where they are (rotation about
// y: y = v, and v moves neither x nor z): an output column is a fixed blend of
// four input columns, with the general kernel's arithmetic at fy = 0.  A
// wavefront takes 64 V values of kRowsRun neighbouring output columns of one
// page; the wavefronts of a block take neighbouring pages and blocks go to the
// XCDs in contiguous ranges, so that the input columns they share meet in L1
// and L2.  Bound by memory: 512x980x200 rotated by 31.5 degrees 0.180 ms (4.1
// TB/s past L2), with the general kernel 0.311 ms.  Stores past the caches make
// this kernel 0.190 ms and leave the input cached for its other reader, the column
// flags (0.045 instead of 0.076 ms).  Calls, stores past the caches / plain: one
// volume again and again 0.319 / 0.339 ms, six in turn 0.320 / 0.345, six with the
// result copied next 0.516 / 0.523, after 512 MB of other writes 0.366 / 0.361.
constexpr int kRowsRun = 8;
template <int V>
__global__ void __launch_bounds__(256) k_affine_rows(const float* __restrict__ vol, float* __restrict__ out, int64_t ny,
                                                     int64_t nx, int64_t nz, int64_t oy, int64_t ox, int64_t oz,
                                                     Affine3 m, int64_t chunks, int64_t runs, int64_t pages,
                                                     int64_t per_xcd) {
    for (int64_t b = blockIdx.x >> 3; b < per_xcd; b += gridDim.x >> 3) {
        const int64_t item = (int64_t)(blockIdx.x & 7) * per_xcd + b;
        if (item >= chunks * runs * pages) break;
        const int64_t q = item / chunks, run = q % runs;
        const int64_t p = q / runs * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        const int64_t r = ((item % chunks) * 64 + (threadIdx.x & 63)) * V;
        if (p >= oz || r >= oy) continue;
        const bool in_y = r < ny, more = r + V < ny;  // V = 4: oy = ny
        const int64_t c1 = run * kRowsRun + kRowsRun < ox ? run * kRowsRun + kRowsRun : ox;
        const double w = (double)(p + 1);
        for (int64_t c = run * kRowsRun; c < c1; ++c) {
            const double u = (double)(c + 1);
            const double x = u * m.a[0][0] + w * m.a[2][0] + m.a[3][0];
            const double z = u * m.a[0][2] + w * m.a[2][2] + m.a[3][2];
            float o[V] = {};
            if (in_y && x > -1.0 && x < (double)(nx + 2) && z > -1.0 && z < (double)(nz + 2)) {
                const double fx0 = std::floor(x), fz0 = std::floor(z);
                const int64_t ix = (int64_t)fx0, iz = (int64_t)fz0;  // 1-based lower corner
                const float fx = (float)(x - fx0), fz = (float)(z - fz0);
                float v[2][2][V + 1];  // the four columns, one row more than the outputs
#pragma unroll
                for (int dz = 0; dz < 2; ++dz)
#pragma unroll
                    for (int dx = 0; dx < 2; ++dx) {
                        const int64_t jx = ix + dx, jz = iz + dz;
                        const bool in = jx >= 1 && jx <= nx && jz >= 1 && jz <= nz;
                        const float* __restrict__ g = vol + (r + ny * ((jx - 1) + nx * (jz - 1)));
                        if constexpr (V == 4) {
                            const float4 t = in ? *reinterpret_cast<const float4*>(g) : make_float4(0.f, 0.f, 0.f, 0.f);
                            v[dz][dx][0] = t.x; v[dz][dx][1] = t.y; v[dz][dx][2] = t.z; v[dz][dx][3] = t.w;
                        } else {
                            v[dz][dx][0] = in ? *g : 0.f;
                        }
                        v[dz][dx][V] = in && more ? g[V] : 0.f;
                    }
#pragma unroll
                for (int e = 0; e < V; ++e) {
                    float pl[2];
#pragma unroll
                    for (int dz = 0; dz < 2; ++dz) {
                        // weight 0 for the next row: only its infinities and NaN count, as in the general kernel
                        const float a = v[dz][0][e] + 0.f * (v[dz][0][e + 1] - v[dz][0][e]);
                        const float d = v[dz][1][e] + 0.f * (v[dz][1][e + 1] - v[dz][1][e]);
                        pl[dz] = a + fx * (d - a);
                    }
                    o[e] = pl[0] + fz * (pl[1] - pl[0]);
                }
            }
            float* __restrict__ g = out + ((p * ox + c) * oy + r);
            typedef float nt_f4 __attribute__((ext_vector_type(4)));
            if constexpr (V == 4)  // past the caches, which keep the input's columns
                __builtin_nontemporal_store(nt_f4{o[0], o[1], o[2], o[3]}, reinterpret_cast<nt_f4*>(g));
            else *g = o[0];
        }
    }
}

// rotateFrame3D.m:46-66's extents without the projection leaving the device:
// flag of a column = max over dim 1 ~= 0 (a positive value or a NaN settles it;
// else true when no value is 0).  Bound by reading the columns that hold only
// zeros.  512x980x200: 0.045-0.076 ms (0.112 with one column a wavefront) and 0.009 ms for the
// extents; the maximum as a reduction of the library, its copy and the host's
// search were 0.6 ms.
// A wavefront follows kFlagCols columns at once, 64 V values of each a step.
constexpr int kFlagCols = 4;
template <int V>
__global__ void __launch_bounds__(256) k_column_flags(const float* __restrict__ vol, int64_t ny, int64_t cols,
                                                      uint8_t* __restrict__ flag) {
    const int ln = threadIdx.x & 63;
    const int64_t groups = (cols + kFlagCols - 1) / kFlagCols, step = (int64_t)gridDim.x * 4;
    for (int64_t g = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); g < groups; g += step) {
        const float* __restrict__ v = vol + g * kFlagCols * ny;
        bool settled[kFlagCols], zero[kFlagCols] = {};
#pragma unroll
        for (int c = 0; c < kFlagCols; ++c) settled[c] = g * kFlagCols + c >= cols;
        for (int64_t y = 0; y < ny; y += 64 * V) {
            const int64_t i = y + (int64_t)ln * V;
            float4 a[kFlagCols];
            bool left = false;
#pragma unroll
            for (int c = 0; c < kFlagCols; ++c) {
                a[c] = make_float4(-1.f, -1.f, -1.f, -1.f);  // neither positive nor 0
                if (settled[c]) continue;
                left = true;
                if (i < ny) {
                    if constexpr (V == 4) a[c] = *reinterpret_cast<const float4*>(v + c * ny + i);
                    else a[c].x = v[c * ny + i];
                }
            }
            if (!left) break;
#pragma unroll
            for (int c = 0; c < kFlagCols; ++c) {
                if (settled[c]) continue;
                const float4 t = a[c];
                zero[c] |= t.x == 0.f || t.y == 0.f || t.z == 0.f || t.w == 0.f;
                settled[c] = __ballot(!(t.x <= 0.f) || !(t.y <= 0.f) || !(t.z <= 0.f) || !(t.w <= 0.f)) != 0;
            }
        }
#pragma unroll
        for (int c = 0; c < kFlagCols; ++c) {
            const bool any_zero = __ballot(zero[c]) != 0;
            if (ln == 0 && g * kFlagCols + c < cols) flag[g * kFlagCols + c] = settled[c] || !any_zero;
        }
    }
}
// Per block: whether a flag changes between columns x and x + 1 of a page
// (diff(proj, 1, 2) ~= 0 at [z, x], 1-based), and over those the extremes of
// c = a x + b z zx and of cx = b x + (-a) z zx.  part: 5 doubles a block.
__global__ void __launch_bounds__(256) k_edge_extents(const uint8_t* __restrict__ flag, int64_t nx, int64_t nz,
                                                      double a, double b, double zx, double* __restrict__ part) {
#pragma clang fp contract(off)  // numpy's sums
    __shared__ double sh[4][5];
    double v[5] = {0.0, INFINITY, -INFINITY, INFINITY, -INFINITY};
    const int64_t n = nx * nz;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int64_t xi = i % nx;
        if (xi + 1 >= nx || flag[i] == flag[i + 1]) continue;
        const double x = (double)(xi + 1), z = (double)(i / nx + 1);
        const double c = a * x + b * z * zx, cx = b * x + (-a) * z * zx;
        v[0] = 1.0;
        v[1] = fmin(v[1], c);
        v[2] = fmax(v[2], c);
        v[3] = fmin(v[3], cx);
        v[4] = fmax(v[4], cx);
    }
    for (int k = 32; k > 0; k >>= 1) {
        v[0] = fmax(v[0], __shfl_xor(v[0], k, 64));
        v[1] = fmin(v[1], __shfl_xor(v[1], k, 64));
        v[2] = fmax(v[2], __shfl_xor(v[2], k, 64));
        v[3] = fmin(v[3], __shfl_xor(v[3], k, 64));
        v[4] = fmax(v[4], __shfl_xor(v[4], k, 64));
    }
    if ((threadIdx.x & 63) == 0)
        for (int k = 0; k < 5; ++k) sh[threadIdx.x >> 6][k] = v[k];
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < 4; ++w) {
            v[0] = fmax(v[0], sh[w][0]);
            v[1] = fmin(v[1], sh[w][1]);
            v[2] = fmax(v[2], sh[w][2]);
            v[3] = fmin(v[3], sh[w][3]);
            v[4] = fmax(v[4], sh[w][4]);
        }
        for (int k = 0; k < 5; ++k) part[5 * blockIdx.x + k] = v[k];
    }
}

void pk_ctx_impl::edge_extents(const float* vol, const int64_t dims[3], double a, double b, double zx, double out[5]) {
    const int64_t cols = dims[1] * dims[2];
    constexpr int kBlocks = 64;
    const size_t off = ((size_t)cols + 255) / 256 * 256;
    ensure(ws.dsr, off + sizeof(double) * 5 * kBlocks);
    uint8_t* flag = ws.dsr.as<uint8_t>();
    double* part = reinterpret_cast<double*>(ws.dsr.as<char>() + off);
    const int64_t groups = (cols + kFlagCols - 1) / kFlagCols;
    const dim3 grid((unsigned)std::min<int64_t>((groups + 3) / 4, 65536));
    if (dims[0] % 4 == 0 && reinterpret_cast<uintptr_t>(vol) % 16 == 0)
        hipLaunchKernelGGL(k_column_flags<4>, grid, dim3(256), 0, stream, vol, dims[0], cols, flag);
    else
        hipLaunchKernelGGL(k_column_flags<1>, grid, dim3(256), 0, stream, vol, dims[0], cols, flag);
    hipLaunchKernelGGL(k_edge_extents, dim3(kBlocks), dim3(256), 0, stream, flag, dims[1], dims[2], a, b, zx, part);
    PK_HIP(hipGetLastError());
    double h[5 * kBlocks];
    PK_HIP(hipMemcpyAsync(h, part, sizeof(h), hipMemcpyDeviceToHost, stream));
    PK_HIP(hipStreamSynchronize(stream));
    out[0] = 0.0;
    out[1] = out[3] = INFINITY;
    out[2] = out[4] = -INFINITY;
    for (int k = 0; k < kBlocks; ++k) {
        out[0] = std::max(out[0], h[5 * k]);
        out[1] = std::min(out[1], h[5 * k + 1]);
        out[2] = std::max(out[2], h[5 * k + 2]);
        out[3] = std::min(out[3], h[5 * k + 3]);
        out[4] = std::max(out[4], h[5 * k + 4]);
    }
}

void launch_affine3d(const float* vol, float* out, const int64_t dims[3], const int64_t odims[3], const Affine3& m,
                     hipStream_t s) {
    const int64_t cols = odims[1] * odims[2];
    if (cols <= 0 || odims[0] <= 0) return;
    const unsigned nt = odims[0] >= 256 ? 256u : (unsigned)((odims[0] + 63) / 64 * 64);
    if (cols * (int64_t)nt > 0xFFFFFFFFll) fail(PK_ERR_UNSUPPORTED_SIZE, "output volume has too many columns");
    // rows stay where they are: the four-column kernel.  Rotations about y come
    // out of the host's products and inverse with these entries exact
    if (m.a[0][1] == 0.0 && m.a[2][1] == 0.0 && m.a[3][1] == 0.0 && m.a[1][1] == 1.0 && m.a[1][0] == 0.0 &&
        m.a[1][2] == 0.0) {
        const bool vec = odims[0] == dims[0] && dims[0] % 4 == 0 &&
                         (reinterpret_cast<uintptr_t>(vol) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
        const int64_t per = 64 * (vec ? 4 : 1), chunks = (odims[0] + per - 1) / per;
        const int64_t runs = (odims[1] + kRowsRun - 1) / kRowsRun, pages = (odims[2] + 3) / 4;
        // (a launch counts work items in 32 bits; blocks beyond that loop)
        const int64_t per_xcd = (chunks * runs * pages + 7) / 8, blocks = std::min<int64_t>(per_xcd, 1 << 20) * 8;
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, s, vol, out, dims[0], dims[1], dims[2],
                               odims[0], odims[1], odims[2], m, chunks, runs, pages, per_xcd);
        };
        if (vec) launch(k_affine_rows<4>);
        else launch(k_affine_rows<1>);
        PK_HIP(hipGetLastError());
        return;
    }
    hipLaunchKernelGGL(k_affine3d, dim3((unsigned)cols), dim3(nt), 0, s, vol, out, dims[0], dims[1], dims[2], odims[0],
                       odims[1], m);
    PK_HIP(hipGetLastError());
}

// ---------------------------------------------------------------- cubic
// imwarp(..., 'cubic', 'FillValues', 0): the input padded with one voxel of
// the fill value 0 on every side, then cubic convolution (Keys, a = -0.5:
// the kernel that reproduces quadratics) over that padded grid, whose two
// missing neighbours past each end come from Keys' boundary rule
// f(-1) = 3 f(0) - 3 f(1) + f(2); a point outside the padded grid takes the
// fill value.  Per axis the (up to) four taps fold into weights on real
// samples: a tap on the zero pad drops out, the extrapolated tap below the
// grid (padded index -1, i.e. 1-based -1) adds -3 w to sample 1 and w to
// sample 2, and symmetrically at the top.
struct CubicTaps {
    int64_t idx[4];  // 0-based samples
    float w[4];
    int n;
};

__device__ __forceinline__ CubicTaps cubic_taps(double x, int64_t n) {
    // x: 1-based coordinate, within [0, n + 1]
    const double f0 = floor(x);
    const int64_t i = (int64_t)f0;
    const float t = (float)(x - f0);
    const float t2 = t * t, t3 = t2 * t;
    const float w[4] = {-0.5f * t3 + t2 - 0.5f * t, 1.5f * t3 - 2.5f * t2 + 1.f, -1.5f * t3 + 2.f * t2 + 0.5f * t,
                        0.5f * t3 - 0.5f * t2};
    CubicTaps c{};
    auto add = [&](int64_t j, float v) {  // j: 1-based real sample
        if (j < 1 || j > n) return;        // the zero pad
        for (int k = 0; k < c.n; ++k)
            if (c.idx[k] == j - 1) {
                c.w[k] += v;
                return;
            }
        c.idx[c.n] = j - 1;
        c.w[c.n] = v;
        ++c.n;
    };
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int64_t j = i - 1 + k;
        if (w[k] == 0.f) continue;  // also the taps past the extension at x = n + 1 exactly
        if (j == -1) {               // 3 f(0) - 3 f(1) + f(2), f(0) the pad
            add(1, -3.f * w[k]);
            add(2, w[k]);
        } else if (j == n + 2) {     // 3 f(n+1) - 3 f(n) + f(n-1), f(n+1) the pad
            add(n, -3.f * w[k]);
            add(n - 1, w[k]);
        } else {
            add(j, w[k]);
        }
    }
    return c;
}

__global__ void __launch_bounds__(256) k_affine3d_cubic(const float* __restrict__ vol, float* __restrict__ out,
                                                        int64_t ny, int64_t nx, int64_t nz, int64_t oy, int64_t ox,
                                                        Affine3 m) {
    const int64_t col = blockIdx.x;
    const int64_t c = col % ox, p = col / ox;
    const double u = (double)(c + 1), w = (double)(p + 1);
    const double bx = u * m.a[0][0] + w * m.a[2][0] + m.a[3][0];
    const double by = u * m.a[0][1] + w * m.a[2][1] + m.a[3][1];
    const double bz = u * m.a[0][2] + w * m.a[2][2] + m.a[3][2];
    float* __restrict__ o = out + col * oy;
    for (int64_t r = threadIdx.x; r < oy; r += blockDim.x) {
        const double v = (double)(r + 1);
        const double x = bx + v * m.a[1][0], y = by + v * m.a[1][1], z = bz + v * m.a[1][2];
        float val = 0.f;
        if (x >= 0.0 && x <= (double)(nx + 1) && y >= 0.0 && y <= (double)(ny + 1) && z >= 0.0 &&
            z <= (double)(nz + 1)) {
            const CubicTaps tx = cubic_taps(x, nx), ty = cubic_taps(y, ny), tz = cubic_taps(z, nz);
            for (int kz = 0; kz < tz.n; ++kz) {
                float sx = 0.f;
                for (int kx = 0; kx < tx.n; ++kx) {
                    const float* __restrict__ rowp = vol + ny * (tx.idx[kx] + nx * tz.idx[kz]);
                    float sy = 0.f;
                    for (int ky = 0; ky < ty.n; ++ky) sy += ty.w[ky] * rowp[ty.idx[ky]];
                    sx += tx.w[kx] * sy;
                }
                val += tz.w[kz] * sx;
            }
        }
        o[r] = val;
    }
}

void launch_affine3d_cubic(const float* vol, float* out, const int64_t dims[3], const int64_t odims[3],
                           const Affine3& m, hipStream_t s) {
    for (int d = 0; d < 3; ++d)
        if (dims[d] < 2) fail(PK_ERR_INVALID_ARG, "cubic interpolation needs at least 2 voxels along every axis");
    const int64_t cols = odims[1] * odims[2];
    if (cols <= 0 || odims[0] <= 0) return;
    const unsigned nt = odims[0] >= 256 ? 256u : (unsigned)((odims[0] + 63) / 64 * 64);
    if (cols * (int64_t)nt > 0xFFFFFFFFll) fail(PK_ERR_UNSUPPORTED_SIZE, "output volume has too many columns");
    hipLaunchKernelGGL(k_affine3d_cubic, dim3((unsigned)cols), dim3(nt), 0, s, vol, out, dims[0], dims[1], dims[2],
                       odims[0], odims[1], m);
    PK_HIP(hipGetLastError());
}

}  // namespace pk
