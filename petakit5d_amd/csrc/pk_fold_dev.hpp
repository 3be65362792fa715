// pk_fold_dev.hpp -- the two-pass form of an iteration's transforms.
//
// The three-pass form moves the spectrum through memory once per axis (row
// pass, dim-2 pass, dim-3 convolution, dim-2 pass).  Here the dim-2 transform
// is split between its neighbours, so that a half iteration is two passes:
//
//   fold row pass     [dim-2 inverse, outer steps] -> C2R -> real-space step
//                     -> R2C -> [dim-2 forward, outer steps]
//   fold column pass  [dim-2 forward, inner steps] -> dim-3 forward -> x OTF/N
//                     -> dim-3 inverse -> [dim-2 inverse, inner steps]
//
// n2 = a * m.  The strided transforms run in place by decimation in frequency:
// the step of radix R and sub-block length M takes the R elements M apart of
// every block of M R positions and leaves output q at offset q M, times
// W_{MR}^{j q} (j the offset inside the sub-block); the steps of sub-blocks
// down to m only mix the positions y0 + i m (i < a) of one y0, and the rest
// stay inside one run of m positions.  So the row pass holds the a rows
// y0 + i m of a plane (b neighbouring y0) and runs the first steps between
// its rows, and the column pass holds the m rows of one run, all planes and T
// adjacent columns, and runs the rest and the whole dim-3 transform.  The
// frequencies come out in digit-reversed order.  Nothing reorders them: the OTF
// is made by the same two passes, and the inverse runs the same steps
// backwards.  A last dim-3 step, the OTF product and the first inverse step
// share the same R positions, so they chain in registers; every other step is
// one in-place trip through LDS and one barrier.
//
// Bytes of a half iteration: 40S + the real operands instead of 72S (S
// half-spectrum points of 8 bytes).  Measured on one half iteration (strided
// passes and ratio, or column and row pass), three passes with measured launch
// shapes / two passes, ms: 64x64x32 0.019 / 0.020, 128x128x64 0.030 / 0.026,
// 256x256x128 0.079 / 0.068, 300x300x160 0.159 / 0.112, 270x360x180 0.194 /
// 0.136, 384x384x256 0.332 / 0.247, 512x512x256 0.520 / 0.507.  Calls against the
// three passes with built-in shapes: Biggs-10 at 270x360x180 5.72 -> 4.02 ms, 8
// chunks of up to 384x384x256 25.9 -> 20.7 ms, OMW-2 at 512x512x256 2.42 -> 2.31
// ms.  HBM bytes there: column pass 0.86 GB, ratio 0.70, 1.07 and 1.03 times the
// algorithmic ones.  Sizes whose three passes are faster keep them (default_fold,
// pk_engine.hip).
//
// What bounds it: the column pass moves 3.4-4.2 TB/s.  Where the tiles leave one
// block a CU (512x512x256: 140 and 147 KB) nothing hides a block's load and store
// phases: the ratio's row pass takes 0.26 ms for 0.14 ms of vector instructions
// (about 100 an element: two row transforms, two splits, four dim-2 steps) and
// 0.15 ms of bytes at the copy rate, one after the other.
#pragma once
#include "pk_fft_dev.hpp"

namespace pk {

constexpr int kFoldSteps = 6;

// In-place steps of one axis, in forward order.
struct FoldSteps {
    int n = 0;
    int R[kFoldSteps] = {};         // radix
    int M[kFoldSteps] = {};         // distance of a butterfly's elements (local positions)
    uint32_t magM[kFoldSteps] = {};  // u / M = umulhi(u, magM); 0: M = 1
    int tws[kFoldSteps] = {};       // W_{MR} = W_len^tws
    int U[kFoldSteps] = {};         // butterflies of the local positions
    uint32_t magU[kFoldSteps] = {};  // u / U
};

struct FoldX {
    XArgs a;
    const float2* tw;   // W_L^e
    const float2* twy;  // W_{n2}^e
    int m, lb;          // y0 stride between local rows; log2 of the y0 per block
    int G;              // rows of a block: a << lb
    uint32_t mag_nyb;   // blk / nyb
    int nyb;            // blocks per plane: m >> lb
    int blk0;           // first block: a launch over planes from z0 starts at z0 nyb
    int n2;
    int L, H1, HP;      // row transform length, half-spectrum columns, their pitch in memory
    int M1p;            // LDS row: position p at (p / M1) M1p + p mod M1 (M1p odd: no bank conflicts across q1)
    int LP;             // LDS row pitch: R1 M1p positions and the column X_L
    uint32_t mag_R1, mag_R2;   // digits of a column index
    int npair;                 // pair tasks: k = 0 ... L / 2
    uint32_t mag_chH, mag_remH, mag_chP, mag_remP;  // task / (columns per 64, columns left over)
    FoldSteps sx;       // steps along the row, forward order
    FoldSteps st;       // dim-2 steps; M, U count local rows (index i << lb | y0 offset)
};

struct FoldC {
    float2* data;
    const float2* otf;
    const float2* twy;   // W_{n2}^e
    const float2* twz;   // W_{n3}^e
    int64_t plane;       // float2 between planes: hp * n2
    int hp, h1, m, n3;
    int lT;              // log2 of the columns of a tile
    int zs;              // LDS float2 between planes
    int gx;              // tiles along a row
    uint32_t mag_gx;
    int tiles;           // gx * a
    int per_xcd;         // tiles per XCD (blocks b, b + 8, ... walk one XCD's range)
    uint32_t mag_mT;     // task / (m T)
    float scale;         // 1 / N, applied with the OTF product
    int nt_st;           // nontemporal stores (whole 128-byte segments)
    FoldSteps sy, sz;
};

// u / d for u d < 2^32: mag = floor(2^32 / d) + 1, 0 for d = 1.  Tasks and their
// divisors count parts of a tile, at most 20480 values of LDS; block indexes are
// checked where the plan is built.
__device__ __forceinline__ int fold_div(int u, uint32_t mag) { return mag ? (int)__umulhi((uint32_t)u, mag) : u; }

// The arguments of a block: a launch over many chunks reads its chunk's
// descriptor (n > 0), a single volume reads the kernel's own first argument.
// Both are constant-address-space reads (scalar loads).
template <class T>
__device__ __forceinline__ const T& fold_args(const T* ch, const int64_t* starts, int n, int& blk) {
    typedef const __attribute__((address_space(4))) T* cptr;
    cptr p = (cptr)__builtin_amdgcn_kernarg_segment_ptr();
    blk = (int)blockIdx.x;
    if (n > 0) {
        const int c = chunk_of(starts, n, blockIdx.x);
        blk = (int)((int64_t)blockIdx.x - starts[c]);
        p = (cptr)(uintptr_t)(ch + c);
    }
    return *(const T*)p;
}

// ------------------------------------------------------------------ row pass
// The block's tile in LDS: G rows of LP float2.  The row transform runs in place
// on the tile as well: the forward steps take natural positions to
// digit-reversed frequencies, so column k of the half spectrum sits at the
// position of its digits (fold_slot).  The first forward step and the last
// inverse step share their R1 elements M1 apart, so the real-space step runs
// between them in registers.  Rows are even: the transform runs over their L = n1 / 2 value pairs.  The split of a row (X_k and X_{L-k}
// from Z_k and Z_{L-k}) rides in the innermost dim-2 step, whose butterflies
// hold both columns.  Spectra are kept at twice their value (the split's
// factor 1/2 is left out and 1/4 goes to the OTF product: exact).

__device__ __forceinline__ int fold_slot(const FoldX& f, int k) {
    if (f.sx.n == 1) return k * f.M1p;
    const int t = fold_div(k, f.mag_R1), q1 = k - t * f.sx.R[0];
    if (f.sx.n == 2) return q1 * f.M1p + t;
    const int q3 = fold_div(t, f.mag_R2), q2 = t - q3 * f.sx.R[1];
    return q1 * f.M1p + q2 * f.sx.M[1] + q3;
}

// Twiddles W_L^(m j tws), m < R, of one butterfly (m j tws < L).  A product
// carries the rounding of its factors, and a power of one value m times that
// value's: with stage_twiddle's powers of W^1 the error of OMW-2 against 64 bits
// was up to 1.46 times the three passes' (64x64x32, 3.5e-7 against 2.4e-7).  Here
// a power is a table value, or W^1 or W^2 and one of the table's W^4, W^8, W^12 (the
// last one of R = 12 and 16 takes three factors); R <= 4 and R = 8 read all from the table: 0.56-1.07 times the three passes'
// error over 20 sizes, for up to 1.4 % of the time (8 chunks of up to 384x384x256,
// Biggs-10, 20.4 -> 20.7 ms).  All radices from the table: no closer, 2-4 % slower.
template <int R, bool INV>
__device__ __forceinline__ void fold_twiddle(float2 (&v)[R], const float2* __restrict__ tw, int j, int tws) {
    constexpr bool all = R <= 4 || R == 8;
    float2 w[R];
    const int d = j * tws;
    static_for<1, R>([&](auto mc) {
        constexpr int m = decltype(mc)::value;
        if constexpr (all || m == 1 || m % 4 == 0) w[m] = tw[m * d];
    });
    if constexpr (!all) {
        w[2] = cmul(w[1], w[1]);
        static_for<3, R>([&](auto mc) {
            constexpr int m = decltype(mc)::value;
            if constexpr (m % 4 == 3 && m + 1 < R) w[m] = cmulc(w[m + 1], w[1]);
            else if constexpr (m % 4 != 0) w[m] = cmul(w[m / 4 * 4], w[m % 4]);
        });
    }
    static_for<1, R>([&](auto mc) {
        constexpr int m = decltype(mc)::value;
        v[m] = INV ? cmulc(v[m], w[m]) : cmul(v[m], w[m]);
    });
}

// Radix-R butterfly of a dim-2 step with its twiddles W_{n2}^{m j tws}: table
// values where j is the same for the whole wavefront (scalar loads).
template <int R, bool INV, bool UNI>
__device__ __forceinline__ void foldx_dft(float2 (&v)[R], const float2* __restrict__ tw, int j, int tws, bool twid) {
    if constexpr (!INV) dft<R, false>(v);
    if (twid) {
        if constexpr (UNI) {
            static_for<1, R>([&](auto mc) {
                constexpr int m = decltype(mc)::value;
                const float2 w = tw[m * j * tws];
                v[m] = INV ? cmulc(v[m], w) : cmul(v[m], w);
            });
        } else {
            fold_twiddle<R, INV>(v, tw, j, tws);
        }
    }
    if constexpr (INV) dft<R, true>(v);
}

// Runs fn(u, item, uniform) over butterflies u < U and items < 64 ch + rem:
// whole groups of 64 items go to a wavefront with one u (scalar indices and
// twiddles), the rem items left over are dealt over all lanes.
template <class Fn>
__device__ __forceinline__ void foldx_tasks(int U, int items, uint32_t mag_ch, uint32_t mag_rem, Fn&& fn) {
    const int ch = items >> 6, rem = items & 63;
    if (ch > 0) {
        const int nw = (int)(blockDim.x >> 6), ln = (int)(threadIdx.x & 63);
        for (int unit = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); unit < U * ch; unit += nw) {
            const int u = fold_div(unit, mag_ch);
            fn(u, (unit - u * ch) * 64 + ln, std::true_type{});
        }
    }
    if (rem > 0) {
        for (int task = threadIdx.x; task < rem * U; task += (int)blockDim.x) {
            const int u = fold_div(task, mag_rem);
            fn(u, ch * 64 + (task - u * rem), std::false_type{});
        }
    }
}

// Where a butterfly u of dim-2 step s sits: first local row, twiddle position,
// float2 distance of its rows in LDS and in memory, first row in memory.
struct FoldXPos {
    int l0, j, ld;
    int64_t g0, gd;
    bool twid;
};
__device__ __forceinline__ FoldXPos foldx_pos(const FoldX& f, int s, int u, int y0) {
    const int M = f.st.M[s], bm = (1 << f.lb) - 1;
    const int be = fold_div(u, f.st.magM[s]), jb = u - be * M;
    FoldXPos p;
    p.l0 = be * (M * f.st.R[s]) + jb;
    p.j = (jb >> f.lb) * f.m + y0 + (jb & bm);
    p.ld = M * f.LP;
    // row of local row l: (l >> lb) m + (l & bm) + y0; M is a multiple of b
    p.g0 = (int64_t)((p.l0 >> f.lb) * f.m + (p.l0 & bm)) * f.HP;
    p.gd = (int64_t)((M >> f.lb) * f.m) * f.HP;
    p.twid = (M >> f.lb) * f.m > 1;  // sub-blocks of one position: every twiddle is 1
    return p;
}

// Outer dim-2 step: memory -> LDS (inverse) or LDS -> memory (forward), one column per task.
// The row pass stores its spectrum past the caches: the column pass reads it on
// other XCDs (OMW-2 512x512x256 2.35 -> 2.32 ms, 16 chunks of up to 384x384x256 8.42 ->
// 8.26; the real-space volumes stored that way cost Biggs-10 2.5 %).
template <int R, bool INV>
__device__ __forceinline__ void foldx_mem_r(const FoldX& f, int s, float2* lds, float2* __restrict__ sp0, int y0) {
    foldx_tasks(f.st.U[s], f.H1, f.mag_chH, f.mag_remH, [&](int u, int k, auto uni) {
        const FoldXPos p = foldx_pos(f, s, u, y0);
        float2* __restrict__ g = sp0 + (p.g0 + k);
        float2* q = lds + p.l0 * f.LP + (k == f.L ? f.LP - 1 : fold_slot(f, k));
        float2 v[R];
        static_for<0, R>([&](auto c) { v[decltype(c)::value] = INV ? g[decltype(c)::value * p.gd] : q[decltype(c)::value * p.ld]; });
        foldx_dft<R, INV, decltype(uni)::value>(v, f.twy, p.j, f.st.tws[s], p.twid);
        static_for<0, R>([&](auto c) {
            if constexpr (INV) q[decltype(c)::value * p.ld] = v[decltype(c)::value];
            else st_f2<true>(g + decltype(c)::value * p.gd, v[decltype(c)::value]);
        });
    });
}

// Innermost dim-2 step with the split of the row transform: both columns k and
// L - k of R rows.
// MEM: the spectrum side is memory (the only dim-2 step), else LDS in place.
template <int R, bool INV, bool MEM>
__device__ __forceinline__ void foldx_pair_r(const FoldX& f, int s, float2* lds, float2* __restrict__ sp0, int y0) {
    foldx_tasks(f.st.U[s], f.npair, f.mag_chP, f.mag_remP, [&](int u, int k, auto uni) {
        constexpr bool UNI = decltype(uni)::value;
        const FoldXPos p = foldx_pos(f, s, u, y0);
        const int tws = f.st.tws[s];
        float2* row = lds + p.l0 * f.LP;
        float2* q1 = row + fold_slot(f, k);
        // partner column: L - k; of column 0 the column L (spectrum side)
        float2* q2 = row + (k == 0 ? 0 : fold_slot(f, f.L - k));
        float2* q2s = k == 0 ? row + (f.LP - 1) : q2;
        float2* __restrict__ g = sp0 + p.g0;
        float2 v1[R], v2[R];
        if constexpr (INV) {
            static_for<0, R>([&](auto c) {
                constexpr int q = decltype(c)::value;
                v1[q] = MEM ? g[q * p.gd + k] : q1[q * p.ld];
                v2[q] = MEM ? g[q * p.gd + (f.L - k)] : q2s[q * p.ld];
            });
            foldx_dft<R, true, UNI>(v1, f.twy, p.j, tws, p.twid);
            foldx_dft<R, true, UNI>(v2, f.twy, p.j, tws, p.twid);
            const float2 w = f.a.rtw[k];
            static_for<0, R>([&](auto c) {
                constexpr int q = decltype(c)::value;
                // Z_k = (A + B) + i W^{-k} (A - B), A = X_k, B = X*_{L-k}; Z_{L-k} from the conjugates
                const float2 B = cconj(v2[q]);
                const float2 ev = cadd(v1[q], B), od = cmulc(csub(v1[q], B), w);
                q1[q * p.ld] = make_float2(ev.x - od.y, ev.y + od.x);
                if (k > 0) q2[q * p.ld] = make_float2(ev.x + od.y, od.x - ev.y);
            });
        } else {
            const float2 w = f.a.rtw[k];
            static_for<0, R>([&](auto c) {
                constexpr int q = decltype(c)::value;
                // 2 X_k = (A + B) - i W^k (A - B), A = Z_k, B = Z*_{L-k}; 2 X_{L-k} from the conjugates
                const float2 A = q1[q * p.ld], B = cconj(q2[q * p.ld]);
                const float2 sm = cadd(A, B), d = cmul(csub(A, B), w);
                v1[q] = make_float2(sm.x + d.y, sm.y - d.x);
                v2[q] = make_float2(sm.x - d.y, -sm.y - d.x);
            });
            foldx_dft<R, false, UNI>(v2, f.twy, p.j, tws, p.twid);
            foldx_dft<R, false, UNI>(v1, f.twy, p.j, tws, p.twid);
            static_for<0, R>([&](auto c) {
                constexpr int q = decltype(c)::value;
                if constexpr (MEM) {
                    st_f2<true>(g + (q * p.gd + k), v1[q]);
                    st_f2<true>(g + (q * p.gd + (f.L - k)), v2[q]);
                } else {
                    q1[q * p.ld] = v1[q];
                    q2s[q * p.ld] = v2[q];
                }
            });
        }
    });
}

template <bool INV>
__device__ __forceinline__ void foldx_mem(const FoldX& f, int s, float2* lds, float2* sp0, int y0) {
    switch (f.st.R[s]) {
        case 4: foldx_mem_r<4, INV>(f, s, lds, sp0, y0); break;
        case 5: foldx_mem_r<5, INV>(f, s, lds, sp0, y0); break;
        case 6: foldx_mem_r<6, INV>(f, s, lds, sp0, y0); break;
        case 8: foldx_mem_r<8, INV>(f, s, lds, sp0, y0); break;
        case 9: foldx_mem_r<9, INV>(f, s, lds, sp0, y0); break;
        case 10: foldx_mem_r<10, INV>(f, s, lds, sp0, y0); break;
        case 12: foldx_mem_r<12, INV>(f, s, lds, sp0, y0); break;
        case 15: foldx_mem_r<15, INV>(f, s, lds, sp0, y0); break;
        case 16: foldx_mem_r<16, INV>(f, s, lds, sp0, y0); break;
        default: break;
    }
}
template <bool INV, bool MEM>
__device__ __forceinline__ void foldx_pair(const FoldX& f, int s, float2* lds, float2* sp0, int y0) {
    switch (f.st.R[s]) {
        case 2: foldx_pair_r<2, INV, MEM>(f, s, lds, sp0, y0); break;
        case 3: foldx_pair_r<3, INV, MEM>(f, s, lds, sp0, y0); break;
        case 4: foldx_pair_r<4, INV, MEM>(f, s, lds, sp0, y0); break;
        case 5: foldx_pair_r<5, INV, MEM>(f, s, lds, sp0, y0); break;
        case 6: foldx_pair_r<6, INV, MEM>(f, s, lds, sp0, y0); break;
        case 8: foldx_pair_r<8, INV, MEM>(f, s, lds, sp0, y0); break;
        default: break;
    }
}

// Step s >= 1 along the rows, in place.
template <int R, bool INV>
__device__ __forceinline__ void foldx_row_r(const FoldX& f, int s, float2* lds) {
    const int M = f.sx.M[s], U = f.sx.U[s], tws = f.sx.tws[s], M1 = f.sx.M[0];
    for (int task = threadIdx.x; task < f.G * U; task += (int)blockDim.x) {
        const int lr = fold_div(task, f.sx.magU[s]), u = task - lr * U;
        const int be = fold_div(u, f.sx.magM[s]), j = u - be * M;
        const int pos = be * (M * R) + j;
        float2* q = lds + lr * f.LP + pos + fold_div(pos, f.sx.magM[0]) * (f.M1p - M1);
        float2 v[R];
        static_for<0, R>([&](auto c) { v[decltype(c)::value] = q[decltype(c)::value * M]; });
        if constexpr (INV) {
            if (M > 1) fold_twiddle<R, true>(v, f.tw, j, tws);
            dft<R, true>(v);
        } else {
            dft<R, false>(v);
            if (M > 1) fold_twiddle<R, false>(v, f.tw, j, tws);
        }
        static_for<0, R>([&](auto c) { q[decltype(c)::value * M] = v[decltype(c)::value]; });
    }
}
template <bool INV>
__device__ __forceinline__ void foldx_row(const FoldX& f, int s, float2* lds) {
    switch (f.sx.R[s]) {
        case 2: foldx_row_r<2, INV>(f, s, lds); break;
        case 3: foldx_row_r<3, INV>(f, s, lds); break;
        case 4: foldx_row_r<4, INV>(f, s, lds); break;
        case 5: foldx_row_r<5, INV>(f, s, lds); break;
        case 6: foldx_row_r<6, INV>(f, s, lds); break;
        case 8: foldx_row_r<8, INV>(f, s, lds); break;
        case 9: foldx_row_r<9, INV>(f, s, lds); break;
        case 10: foldx_row_r<10, INV>(f, s, lds); break;
        case 12: foldx_row_r<12, INV>(f, s, lds); break;
        case 15: foldx_row_r<15, INV>(f, s, lds); break;
        case 16: foldx_row_r<16, INV>(f, s, lds); break;
        default: break;
    }
    __syncthreads();
}

// The modes that have a spectrum to transform back, and to produce.
constexpr bool foldx_in(int m) { return m == XM_RATIO || m == XM_OMW_UPDATE || m == XM_BIGGS_UPDATE; }

// Real-space step: last inverse row step -> elementwise -> first forward row
// step.  Adds the step length's two sums to s_num, s_den (Biggs update).
template <int R, int MODE_>
__device__ __forceinline__ void foldx_mid_r(const FoldX& f, float2* lds, int y0, int z, bool out_spec, double& s_num,
                                            double& s_den) {
    constexpr int MODE = xm_base(MODE_);
    constexpr bool EPI = xm_final(MODE_), IN = foldx_in(MODE), U16OP = xm_u16(MODE_);
    const XArgs& a = f.a;
    const int M1 = f.sx.M[0], tws = f.sx.tws[0];
    const int bm = (1 << f.lb) - 1;
    float lam = 0.f;
    if constexpr (MODE == XM_BIGGS_Y) lam = *a.lambda;
    auto ldr = [&](const float* __restrict__ base, int64_t i) -> float2 {
        return reinterpret_cast<const float2*>(base)[i];
    };
    auto str = [&](float* __restrict__ base, int64_t i, float2 o) {
        reinterpret_cast<float2*>(base)[i] = o;
    };
    auto ld16 = [&](const uint16_t* __restrict__ base, int64_t i) -> uint32_t {
        return reinterpret_cast<const uint32_t*>(base)[i];
    };
    auto st16 = [&](uint16_t* __restrict__ base, int64_t i, float2 o) {
        reinterpret_cast<uint32_t*>(base)[i] = (uint32_t)o.x | ((uint32_t)o.y << 16);
    };
    auto cvt16 = [&](uint32_t w) { return make_float2((float)(w & 0xffffu), (float)(w >> 16)); };
    for (int task = threadIdx.x; task < f.G * M1; task += (int)blockDim.x) {
        const int lr = fold_div(task, f.sx.magM[0]), j = task - lr * M1;
        const int y = (lr >> f.lb) * f.m + (lr & bm) + y0;
        const int64_t row = (int64_t)y + (int64_t)f.n2 * z;
        const int64_t r2 = row * f.L + j;  // index of pair 0
        float2* q = lds + lr * f.LP + j;
        RawRow rr{0, false};
        if constexpr (MODE == XM_PREP_U16 || MODE == XM_PREP_F32) {
            if (a.s0) rr = RawRow{((int64_t)y + a.s1 * z) * a.s0, y < a.s1 && z < a.s2};
        }
        // real-space operands first: their latency overlaps the inverse step
        float2 opA[R], opB[R];
        uint32_t opW[R];
        static_for<0, R>([&](auto c) {
            constexpr int e = decltype(c)::value;
            const int64_t i = r2 + e * M1;
            const int x = j + e * M1;  // position in the row
            opA[e] = opB[e] = make_float2(0.f, 0.f);
            if constexpr (U16OP) opW[e] = ld16(a.I16, i);
            if constexpr (MODE == XM_R2C) opA[e] = ldr(a.src, i);
            if constexpr (MODE == XM_PREP_U16)
                opA[e] = a.s0 ? ld_raw_padded(a.raw16, a, rr, 2 * (int64_t)x, true)
                              : cvt16(ld16(a.raw16, i));
            if constexpr (MODE == XM_PREP_F32)
                opA[e] = a.s0 ? ld_raw_padded(a.rawf, a, rr, 2 * (int64_t)x, true)
                              : ldr(a.rawf, i);
            if constexpr (MODE == XM_RATIO && !U16OP) opA[e] = ldr(a.I, i);
            if constexpr (MODE == XM_OMW_UPDATE && !U16OP) opA[e] = ldr(a.Jin ? a.Jin : a.J, i);
            if constexpr (MODE == XM_BIGGS_Y) {
                opA[e] = ldr(a.J, i);
                opB[e] = ldr(a.J3, i);
            }
            if constexpr (MODE == XM_BIGGS_UPDATE) {
                opA[e] = ldr(a.Y, i);
                if (R <= 10 && !EPI && a.acc) opB[e] = ldr(a.J4, i);
            }
        });
        float2 v[R];
        if constexpr (IN) {
            static_for<0, R>([&](auto c) { v[decltype(c)::value] = q[decltype(c)::value * f.M1p]; });
            if (M1 > 1) fold_twiddle<R, true>(v, f.tw, j, tws);
            dft<R, true>(v);
        }
        EpiRow er{0, 0, false};
        if constexpr (EPI) {
            const EpiArgs& ep = a.ep;
            er.src = row * ep.n1;
            er.keep = y >= ep.b2 && y < ep.b2 + ep.o2 && z >= ep.b3 && z < ep.b3 + ep.o3;
            er.dst = (((int64_t)y - ep.b2) + ep.o2 * ((int64_t)z - ep.b3)) * ep.o1 - ep.b1;
        }
        static_for<0, R>([&](auto c) {
            constexpr int e = decltype(c)::value;
            const int64_t i = r2 + e * M1;
            const int x = j + e * M1;
            if constexpr (U16OP) opA[e] = cvt16(opW[e]);
            float2 o = x_elem<MODE>(v[e], opA[e], opB[e], a.bg, a.eps, lam);
            if constexpr (MODE == XM_PREP_U16 || MODE == XM_PREP_F32) {
                if (MODE == XM_PREP_U16 && a.I16) st16(a.I16, i, o);
                else str(a.I, i, o);
                if (a.J) str(a.J, i, o);
            } else if constexpr (MODE == XM_OMW_UPDATE) {
                if constexpr (EPI) {
                    if (er.keep) epi_put(a.ep, er, 2 * (int64_t)x, true, o);
                } else {
                    str(a.J, i, o);
                }
            } else if constexpr (MODE == XM_BIGGS_Y) {
                str(a.Y, i, o);
            } else if constexpr (MODE == XM_BIGGS_UPDATE) {
                const float2 yv = opA[e];
                if constexpr (EPI) {
                    if (er.keep) epi_put(a.ep, er, 2 * (int64_t)x, true, o);
                } else {
                    str(a.Jn, i, o);
                }
                const float2 d = make_float2(o.x - yv.x, o.y - yv.y);
                if (!EPI && a.acc) {
                    const float2 j4 = R <= 10 ? opB[e] : ldr(a.J4, i);  // larger radices: no registers to hold it earlier
                    s_num += (double)(d.x * j4.x);
                    s_den += (double)(j4.x * j4.x);
                    s_num += (double)(d.y * j4.y);
                    s_den += (double)(j4.y * j4.y);
                }
                if (!EPI && a.write_j4) str(a.J4, i, d);
            }
            v[e] = o;
        });
        if (out_spec) {
            dft<R, false>(v);
            if (M1 > 1) fold_twiddle<R, false>(v, f.tw, j, tws);
            static_for<0, R>([&](auto c) { q[decltype(c)::value * f.M1p] = v[decltype(c)::value]; });
        }
    }
}

template <int MODE_>
__device__ __forceinline__ void foldx_body(const FoldX& f, float2* lds, int blk) {
    constexpr int MODE = xm_base(MODE_);
    constexpr bool EPI = xm_final(MODE_);
    const XArgs& a = f.a;
    const int z = fold_div(blk, f.mag_nyb);
    const int y0 = (blk - z * f.nyb) << f.lb;
    float2* __restrict__ sp0 = a.spec + ((int64_t)z * f.n2 + y0) * f.HP;
    const int nc = f.st.n, nx = f.sx.n;
    if constexpr (foldx_in(MODE)) {  // dim-2 inverse steps and the row transform's inverse steps but the last
        if (nc == 1) {
            foldx_pair<true, true>(f, 0, lds, sp0, y0);
        } else {
            foldx_mem<true>(f, 1, lds, sp0, y0);
            __syncthreads();
            foldx_pair<true, false>(f, 0, lds, sp0, y0);
        }
        __syncthreads();
        for (int s = nx - 1; s >= 1; --s) foldx_row<true>(f, s, lds);
    }
    // the Biggs update and the fused last updates leave no spectrum
    bool out_spec = !EPI && MODE != XM_BIGGS_UPDATE;
    if constexpr (MODE == XM_OMW_UPDATE) out_spec = !EPI && a.r2c_out != 0;
    double s_num = 0.0, s_den = 0.0;
    switch (f.sx.R[0]) {
        case 2: foldx_mid_r<2, MODE_>(f, lds, y0, z, out_spec, s_num, s_den); break;
        case 3: foldx_mid_r<3, MODE_>(f, lds, y0, z, out_spec, s_num, s_den); break;
        case 4: foldx_mid_r<4, MODE_>(f, lds, y0, z, out_spec, s_num, s_den); break;
        case 5: foldx_mid_r<5, MODE_>(f, lds, y0, z, out_spec, s_num, s_den); break;
        case 6: foldx_mid_r<6, MODE_>(f, lds, y0, z, out_spec, s_num, s_den); break;
        case 8: foldx_mid_r<8, MODE_>(f, lds, y0, z, out_spec, s_num, s_den); break;
        case 9: foldx_mid_r<9, MODE_>(f, lds, y0, z, out_spec, s_num, s_den); break;
        case 10: foldx_mid_r<10, MODE_>(f, lds, y0, z, out_spec, s_num, s_den); break;
        case 12: foldx_mid_r<12, MODE_>(f, lds, y0, z, out_spec, s_num, s_den); break;
        case 15: foldx_mid_r<15, MODE_>(f, lds, y0, z, out_spec, s_num, s_den); break;
        case 16: foldx_mid_r<16, MODE_>(f, lds, y0, z, out_spec, s_num, s_den); break;
        default: break;
    }
    if constexpr (!EPI && MODE != XM_BIGGS_UPDATE) {
        if (out_spec) {
            __syncthreads();
            for (int s = 1; s < nx; ++s) foldx_row<false>(f, s, lds);
            if (nc == 1) {
                foldx_pair<false, true>(f, 0, lds, sp0, y0);
            } else {
                foldx_pair<false, false>(f, 0, lds, sp0, y0);
                __syncthreads();
                foldx_mem<false>(f, 1, lds, sp0, y0);
            }
        }
    }

    // block partial sums of the Biggs step length (fixed order: lanes, then wavefronts)
    if constexpr (MODE == XM_BIGGS_UPDATE && !EPI) {
        if (a.acc) {
            const int t = threadIdx.x, wv = t >> 6, nw = (int)(blockDim.x >> 6);
            for (int w = 32; w > 0; w >>= 1) {
                s_num += __shfl_xor(s_num, w, 64);
                s_den += __shfl_xor(s_den, w, 64);
            }
            __syncthreads();
            double* red = reinterpret_cast<double*>(lds);
            if ((t & 63) == 0) {
                red[2 * wv] = s_num;
                red[2 * wv + 1] = s_den;
            }
            __syncthreads();
            if (t == 0) {
                double n = 0.0, d = 0.0;
                for (int w = 0; w < nw; ++w) {
                    n += red[2 * w];
                    d += red[2 * w + 1];
                }
                a.partials[2 * blk] = n;
                a.partials[2 * blk + 1] = d;
            }
        }
    }
}

constexpr int kFoldXThreads = 1024;  // at most; 128 registers, four wavefronts per SIMD

template <int MODE>
__global__ void __launch_bounds__(kFoldXThreads) k_foldx(FoldX, const FoldX* ch, const int64_t* starts, int n) {
    extern __shared__ float2 lds[];
    int blk;
    const FoldX& f = fold_args(ch, starts, n, blk);
    foldx_body<MODE>(f, lds, blk + f.blk0);
}

// ------------------------------------------------------------------ column pass
enum FoldKind : int {
    FK_LOAD = 0,   // forward, memory -> LDS
    FK_FWD = 1,    // forward, LDS -> LDS
    FK_STORE = 2,  // forward, LDS -> memory
    FK_CONV = 3,   // last dim-3 forward step, x OTF, first inverse step: LDS -> LDS
    FK_CONVJ = 4,  // the same with the conjugate OTF
    FK_INV = 5,    // inverse, LDS -> LDS
    FK_OUT = 6,    // inverse, LDS -> memory
};

// One step of the tile [n3][m][T] in LDS (plane stride zs).  ZAX: along dim 3.
template <int R, int KIND, bool ZAX>
__device__ __forceinline__ void foldc_step_r(const FoldC& f, int s, float2* lds, float2* __restrict__ g0,
                                             const float2* __restrict__ h0, int kx0) {
    constexpr bool INV = KIND == FK_INV || KIND == FK_OUT;
    constexpr bool CONV = KIND == FK_CONV || KIND == FK_CONVJ;
    const FoldSteps& st = ZAX ? f.sz : f.sy;
    const int M = st.M[s], U = st.U[s], tws = st.tws[s];
    const uint32_t magM = st.magM[s];
    const float2* __restrict__ tw = ZAX ? f.twz : f.twy;
    const int lT = f.lT, T = 1 << lT, mT = f.m << lT;
    const int total = ZAX ? mT * U : f.n3 * (U << lT);
    const int nt = (int)blockDim.x;
    struct Task {
        int slot, sd, j;
        int64_t go, gd;
        bool ok;
    };
    auto decode = [&](int task) {
        Task k;
        int c, u, z = 0, i;
        if constexpr (ZAX) {
            u = fold_div(task, f.mag_mT);
            c = task - u * mT;
        } else {
            const int w = task >> lT;
            z = fold_div(w, st.magU[s]);
            u = w - z * U;
            c = task & (T - 1);
        }
        const int be = fold_div(u, magM);
        k.j = u - be * M;
        const int pos = be * (M * R) + k.j;
        if constexpr (ZAX) {
            k.slot = pos * f.zs + c;
            k.sd = M * f.zs;
            k.gd = (int64_t)M * f.plane;
            z = pos;
            i = c >> lT;
            c &= T - 1;
        } else {
            k.slot = z * f.zs + (pos << lT) + c;
            k.sd = M << lT;
            k.gd = (int64_t)M * f.hp;
            i = pos;
        }
        k.ok = kx0 + c < f.h1;
        k.go = (int64_t)z * f.plane + (int64_t)i * f.hp + c;
        return k;
    };
    auto load = [&](float2 (&v)[R], const Task& k) {
        static_for<0, R>([&](auto qc) {
            constexpr int q = decltype(qc)::value;
            if constexpr (KIND == FK_LOAD) v[q] = k.ok ? g0[k.go + q * k.gd] : make_float2(0.f, 0.f);
            else v[q] = lds[k.slot + q * k.sd];
        });
    };
    auto finish = [&](float2 (&v)[R], const Task& k) {
        if constexpr (CONV) {
            float2 h[R];
            static_for<0, R>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                h[q] = k.ok ? ld_f2<kNtOtfLd>(h0 + k.go + q * k.gd) : make_float2(0.f, 0.f);
            });
            dft<R, false>(v);
            static_for<0, R>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                const float2 hs = make_float2(h[q].x * f.scale, h[q].y * f.scale);
                v[q] = KIND == FK_CONVJ ? cmulc(v[q], hs) : cmul(v[q], hs);
            });
            dft<R, true>(v);
        } else if constexpr (INV) {
            if (M > 1) fold_twiddle<R, true>(v, tw, k.j, tws);
            dft<R, true>(v);
        } else {
            dft<R, false>(v);
            if (M > 1) fold_twiddle<R, false>(v, tw, k.j, tws);
        }
        if constexpr (KIND == FK_STORE || KIND == FK_OUT) {
            if (k.ok) {
                if (f.nt_st) {
                    static_for<0, R>([&](auto qc) {
                        constexpr int q = decltype(qc)::value;
                        st_f2<true>(g0 + k.go + q * k.gd, v[q]);
                    });
                } else {
                    static_for<0, R>([&](auto qc) {
                        constexpr int q = decltype(qc)::value;
                        st_f2<false>(g0 + k.go + q * k.gd, v[q]);
                    });
                }
            }
        } else {
            static_for<0, R>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                lds[k.slot + q * k.sd] = v[q];
            });
        }
    };
    int task = threadIdx.x;
    if constexpr (KIND == FK_LOAD && R <= 10) {
        // two butterflies in flight: the loads of both are issued before either is used
        for (; task + nt < total; task += 2 * nt) {
            const Task ka = decode(task), kb = decode(task + nt);
            float2 va[R], vb[R];
            load(va, ka);
            load(vb, kb);
            finish(va, ka);
            finish(vb, kb);
        }
    }
    for (; task < total; task += nt) {
        const Task k = decode(task);
        float2 v[R];
        load(v, k);
        finish(v, k);
    }
}
template <int KIND, bool ZAX>
__device__ __forceinline__ void foldc_step(const FoldC& f, int s, float2* lds, float2* g0, const float2* h0, int kx0) {
    switch ((ZAX ? f.sz : f.sy).R[s]) {
        case 2: foldc_step_r<2, KIND, ZAX>(f, s, lds, g0, h0, kx0); break;
        case 3: foldc_step_r<3, KIND, ZAX>(f, s, lds, g0, h0, kx0); break;
        case 4: foldc_step_r<4, KIND, ZAX>(f, s, lds, g0, h0, kx0); break;
        case 5: foldc_step_r<5, KIND, ZAX>(f, s, lds, g0, h0, kx0); break;
        case 6: foldc_step_r<6, KIND, ZAX>(f, s, lds, g0, h0, kx0); break;
        case 8: foldc_step_r<8, KIND, ZAX>(f, s, lds, g0, h0, kx0); break;
        case 9: foldc_step_r<9, KIND, ZAX>(f, s, lds, g0, h0, kx0); break;
        case 10: foldc_step_r<10, KIND, ZAX>(f, s, lds, g0, h0, kx0); break;
        case 12: foldc_step_r<12, KIND, ZAX>(f, s, lds, g0, h0, kx0); break;
        case 15: foldc_step_r<15, KIND, ZAX>(f, s, lds, g0, h0, kx0); break;
        case 16: foldc_step_r<16, KIND, ZAX>(f, s, lds, g0, h0, kx0); break;
        default: break;
    }
    if constexpr (KIND != FK_STORE && KIND != FK_OUT) __syncthreads();
}

// MODE: CM_FWD (the OTF's own transform), CM_CONV, CM_CONVJ.  The plan has at
// least two steps in all, the last of them along dim 3.
template <int MODE>
__device__ __forceinline__ void foldc_body(const FoldC& f, float2* lds, int blk) {
    // blocks go round-robin to the 8 XCDs: each XCD walks a contiguous range
    // of tiles, so tiles that share lines meet in one L2
    const int tile = (blk & 7) * f.per_xcd + (blk >> 3);
    if (tile >= f.tiles) return;
    const int sidx = fold_div(tile, f.mag_gx);
    const int kx0 = (tile - sidx * f.gx) << f.lT;
    float2* __restrict__ g0 = f.data + ((int64_t)sidx * f.m * f.hp + kx0);
    const float2* __restrict__ h0 = MODE == CM_FWD ? nullptr : f.otf + ((int64_t)sidx * f.m * f.hp + kx0);
    const int ny = f.sy.n, nz = f.sz.n;
    if (ny > 0) {
        foldc_step<FK_LOAD, false>(f, 0, lds, g0, h0, kx0);
        for (int s = 1; s < ny; ++s) foldc_step<FK_FWD, false>(f, s, lds, g0, h0, kx0);
    } else {
        foldc_step<FK_LOAD, true>(f, 0, lds, g0, h0, kx0);
    }
    for (int s = ny > 0 ? 0 : 1; s < nz - 1; ++s) foldc_step<FK_FWD, true>(f, s, lds, g0, h0, kx0);
    if constexpr (MODE == CM_FWD) {
        foldc_step<FK_STORE, true>(f, nz - 1, lds, g0, h0, kx0);
    } else {
        foldc_step<MODE == CM_CONVJ ? FK_CONVJ : FK_CONV, true>(f, nz - 1, lds, g0, h0, kx0);
        for (int s = nz - 2; s >= (ny > 0 ? 0 : 1); --s) foldc_step<FK_INV, true>(f, s, lds, g0, h0, kx0);
        if (ny > 0) {
            for (int s = ny - 1; s >= 1; --s) foldc_step<FK_INV, false>(f, s, lds, g0, h0, kx0);
            foldc_step<FK_OUT, false>(f, 0, lds, g0, h0, kx0);
        } else {
            foldc_step<FK_OUT, true>(f, 0, lds, g0, h0, kx0);
        }
    }
}

template <int MODE, int NT>
__global__ void __launch_bounds__(NT) k_foldc(FoldC, const FoldC* ch, const int64_t* starts, int n) {
    extern __shared__ float2 lds[];
    int blk;
    const FoldC& f = fold_args(ch, starts, n, blk);
    foldc_body<MODE>(f, lds, blk);
}

}  // namespace pk
