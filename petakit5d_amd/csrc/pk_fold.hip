// pk_fold.hip -- plans and column-pass launches of the two-pass form (pk_fold_dev.hpp).
#include "pk_fold.hpp"

#include <algorithm>
#include <array>
#include <cmath>
#include <map>
#include <mutex>
#include <vector>

namespace pk {
namespace {

uint32_t magic(int d) { return d > 1 ? (uint32_t)((1ull << 32) / (uint64_t)d + 1ull) : 0u; }

// Fewest factors of n among `radices` (largest first), the product in
// non-increasing order; false when n has other factors.
bool factor(int n, const std::vector<int>& radices, std::vector<int>& out) {
    out.clear();
    if (n == 1) return true;
    std::vector<int> best, cur;
    auto go = [&](auto&& self, int rem, size_t from) -> void {
        if (rem == 1) {
            // fewest steps, then the most even ones
            if (best.empty() || cur.size() < best.size() || (cur.size() == best.size() && cur.back() > best.back()))
                best = cur;
            return;
        }
        if (cur.size() >= (size_t)kFoldSteps) return;
        for (size_t i = from; i < radices.size(); ++i)
            if (rem % radices[i] == 0) {
                cur.push_back(radices[i]);
                self(self, rem / radices[i], i);
                cur.pop_back();
            }
    };
    go(go, n, 0);
    out = best;
    return !best.empty();
}
// radices of the outer dim-2 step next to memory and of the inner one that also splits the row transform
const int kMemRadices[] = {16, 15, 12, 10, 9, 8, 6, 5, 4};
const int kPairRadices[] = {8, 6, 5, 4, 3, 2};
const std::vector<int> kColRadices = {16, 15, 12, 10, 9, 8, 6, 5, 4, 3, 2};

// steps over `len` local positions of a transform of length `whole`; unit:
// local distance of neighbouring positions of the decimated sequence; before:
// product of the radices that came earlier
FoldSteps steps(const std::vector<int>& R, int len, int unit, int before) {
    FoldSteps st;
    st.n = (int)R.size();
    int rem = len, tws = before;
    for (int i = 0; i < st.n; ++i) {
        rem /= R[(size_t)i];
        st.R[i] = R[(size_t)i];
        st.M[i] = rem * unit;
        st.magM[i] = magic(st.M[i]);
        st.tws[i] = tws;
        st.U[i] = len * unit / R[(size_t)i];
        st.magU[i] = magic(st.U[i]);
        tws *= R[(size_t)i];
    }
    return st;
}

// Dim-2 steps between a block's a rows, forward order: the pair radix r0 and,
// when a has more factors, one memory radix.
bool row_steps(int a, int r0, std::vector<int>& out) {
    if (a % r0) return false;
    out = {r0};
    const int r = a / r0;
    if (r == 1) return true;
    out.push_back(r);
    return r >= 4 && std::find(std::begin(kMemRadices), std::end(kMemRadices), r) != std::end(kMemRadices);
}

bool build(FoldPlan& fp, int64_t n1, int64_t n2, int64_t n3, int64_t hp, int a, int b, int T, int r0) {
    // even rows only: an odd row's transform has no half-length form, and with
    // twice the LDS and arithmetic the three passes are faster (405x400x200
    // OMW-2: 1.64 ms against 1.74-2.10)
    if (n1 % 2) return false;
    const int L = (int)(n1 / 2);
    if (L < 4 || n2 % a || a < 2) return false;
    const int m = (int)n2 / a;
    if (m % b) return false;
    std::vector<int> rx, ry, rz, rl;
    if (!row_steps(a, r0, rx) || !factor(m, kColRadices, ry) || !factor((int)n3, kColRadices, rz) ||
        !factor(L, kColRadices, rl) || rl.size() > 3)
        return false;
    if (rz.empty() || (ry.empty() && rz.size() < 2)) return false;
    std::reverse(rl.begin(), rl.end());  // the smallest radix carries the real-space step and its operands
    fp = FoldPlan{};
    fp.a = a;
    fp.m = m;
    fp.b = b;
    fp.T = T;
    int lb = 0, lT = 0;
    while ((1 << lb) < b) ++lb;
    while ((1 << lT) < T) ++lT;
    const int G = a * b;
    const int M1 = L / rl[0], M1p = M1 | 1, LP = rl[0] * M1p + 1;
    fp.xlds = std::max<size_t>((size_t)G * LP * sizeof(float2), 2 * 16 * sizeof(double));
    // plane stride of the column tile: 64 bytes past a multiple of 256, so the
    // same column of neighbouring planes falls on other banks
    int zs = m * T;
    while (zs % 32 != 8) ++zs;
    fp.clds = (size_t)n3 * zs * sizeof(float2);
    if (fp.xlds > kMaxLds || fp.clds > kMaxLds) return false;
    FoldX& x = fp.x;
    x.m = m;
    x.lb = lb;
    x.G = G;
    x.nyb = m / b;
    x.mag_nyb = magic(x.nyb);
    x.n2 = (int)n2;
    x.L = L;
    x.H1 = (int)(n1 / 2 + 1);
    x.HP = (int)hp;
    x.M1p = M1p;
    x.LP = LP;
    x.mag_R1 = magic(rl[0]);
    x.mag_R2 = rl.size() > 1 ? magic(rl[1]) : 0;
    x.npair = L / 2 + 1;
    x.mag_chH = magic(x.H1 / 64);
    x.mag_remH = magic(x.H1 % 64);
    x.mag_chP = magic(x.npair / 64);
    x.mag_remP = magic(x.npair % 64);
    x.sx = steps(rl, L, 1, 1);
    x.st = steps(rx, a, b, 1);
    fp.xblocks = (int64_t)x.nyb * n3;
    FoldC& c = fp.c;
    c.plane = hp * n2;
    c.hp = (int)hp;
    c.h1 = (int)(n1 / 2 + 1);
    c.m = m;
    c.n3 = (int)n3;
    c.lT = lT;
    c.zs = zs;
    c.gx = (c.h1 + T - 1) / T;
    c.mag_gx = magic(c.gx);
    c.tiles = c.gx * a;
    c.per_xcd = (c.tiles + 7) / 8;
    c.mag_mT = magic(m * T);
    // 1 / N, and 1/4 for the doubled spectra (pk_fold_dev.hpp)
    c.scale = (float)(0.25 / ((double)n1 * (double)n2 * (double)n3));
    c.nt_st = T >= 16;
    c.sy = steps(ry, m, 1, a);
    c.sz = steps(rz, (int)n3, 1, 1);
    fp.cblocks = c.per_xcd * 8;
    // block indexes are split with 32-bit multiply-high divisions too (fold_div)
    if (fp.xblocks * x.nyb >= (1ll << 32) || (int64_t)c.tiles * c.gx >= (1ll << 32)) return false;
    uint64_t h = 1469598103934665603ull;
    auto mix = [&](int v) { h = (h ^ (uint64_t)(unsigned)v) * 1099511628211ull; };
    mix(a);
    for (int r : rx) mix(r);
    mix(-1);
    for (int r : ry) mix(r);
    mix(-2);
    for (int r : rz) mix(r);
    fp.layout = h | 1;
    fp.on = true;
    return true;
}

}  // namespace

namespace {
// Lower is better.  The terms are those that explained the measured times of
// every feasible shape (both passes, 17 sizes from 64x64x32 to 512x512x256 and
// 1024x256x64, 12 to 544 shapes each); with the weights fitted to them the
// chosen shape is 1.3 % slower than the fastest one on average, 7 % at worst.
// The last two terms come from batches of equal volumes, where idle threads and
// large blocks cost what they do not in one volume's launch.  They change 17 of 367
// sizes: batches gain 1.04-1.30 times (30 volumes of 480x72x60, Biggs-5: 0.88 -> 1.15
// times the three passes' speed; 15 of 256x256x64, OMW-2: 0.96 -> 1.03), single calls
// 1.005 times on average (0.95-1.05).  Batches of 256x128x64, 128x256x64, 256x256x32,
// 1024x64x32 and 128x128x64 stay below the three passes (0.86-0.96), their single
// calls above (1.06-1.38).
double fold_score(const FoldPlan& fp, int64_t n3) {
    // blocks a CU holds at once: LDS, and registers (16 wavefronts of the row
    // kernel, 20 of the column kernel)
    const int kx = std::max(1, std::min((int)(kMaxLds / fp.xlds), 1024 / (int)fp.xnt));
    const int kc = std::max(1, std::min((int)(kMaxLds / fp.clds), 1280 / (int)fp.cnt));
    // a last round of blocks that leaves CUs idle
    auto rounds = [](int64_t blocks, int64_t slots) {
        return std::log((double)((blocks + slots - 1) / slots * slots) / (double)blocks);
    };
    const double xw = (double)fp.x.G * fp.x.L / 16.0 / fp.xnt;              // radix-16 butterflies a thread, row pass
    const double cw = (double)n3 * fp.m * fp.T / 16.0 / fp.cnt;             // the same, column pass
    double s = 0.6 * rounds(fp.xblocks, 256 * kx) + 0.28 * rounds(fp.c.tiles, 256 * kc);
    s += 0.8 * (1.0 - std::min(1.0, kx * fp.xnt / 1024.0)) - 0.22 * std::log2(xw);   // a full CU, of few-thread blocks
    s += 10.0 * (1.0 - std::min(1.0, kc * fp.cnt / 1024.0)) + 0.09 * std::fabs(std::log2(cw));
    s += fp.T == 16 ? 0.0 : fp.T == 8 ? 0.02 : 10.0;                        // 32-byte row segments cost 20-40 %
    s += (fp.xlds > 81920 ? 0.17 : 0.0) + (fp.clds > 81920 ? 0.09 : 0.0);   // one block a CU: nothing hides its phases
    s += 0.02 * fp.x.st.n + 10.0 * fp.c.sy.n;
    s += 0.12 * std::fabs(std::log2(fp.x.st.R[0] / 6.0)) + (fp.x.st.R[1] > 10 ? 0.07 : 0.0);
    // a batch holds blocks enough for any shape: idle threads, and a large block where two smaller ones fit a CU
    s += 0.12 * std::max(0.0, std::log2(0.5 / xw)) + (fp.xnt == 1024 && fp.xlds <= 81920 ? 0.06 : 0.0);
    return s;
}

FoldPlan search(int64_t n1, int64_t n2, int64_t n3, int64_t hp) {
    FoldPlan best, fp;
    double score = 1e30;
    for (int a = 2; a <= n2; ++a) {
        if (n2 % a) continue;
        for (int r0 : kPairRadices)
            for (int b : {1, 2})
                for (int T : {16, 8, 4}) {
                    if (!build(fp, n1, n2, n3, hp, a, b, T, r0)) continue;
                    for (unsigned xnt : {128u, 256u, 512u, 1024u})
                        for (unsigned cnt : {256u, 512u, 1024u}) {
                            fp.xnt = xnt;
                            fp.cnt = cnt;
                            const double xw = (double)fp.x.G * fp.x.L / 16.0 / xnt, cw = (double)n3 * fp.m * T / 16.0 / cnt;
                            if (xw > 4.0 || xw < 0.2 || cw > 4.0 || cw < 0.45) continue;
                            const double sc = fold_score(fp, n3);
                            if (sc < score) {
                                score = sc;
                                best = fp;
                            }
                        }
                }
    }
    return best;
}
}  // namespace

FoldPlan fold_plan(int64_t n1, int64_t n2, int64_t n3, int64_t hp) {
    if (n1 % 2 || n1 > 2048 || n2 > 8192 || n3 > 8192) return FoldPlan{};
    // a plan is a function of the size and holds no pointer; the search takes
    // about a millisecond, so the last sizes' plans are kept
    static std::mutex mu;
    static std::map<std::array<int64_t, 3>, FoldPlan> memo;
    const std::array<int64_t, 3> key{n1, n2, n3};
    std::lock_guard<std::mutex> lk(mu);
    auto it = memo.find(key);
    if (it != memo.end()) return it->second;
    if (memo.size() >= 256) memo.clear();
    return memo.emplace(key, search(n1, n2, n3, hp)).first->second;
}

hipError_t launch_foldx(unsigned nt, dim3 grid, size_t lds, hipStream_t s, const FoldX& f, int mode,
                        const FoldX* ch, const int64_t* starts, int n) {
    if (launch_foldx_a(nt, grid, lds, s, f, mode, ch, starts, n) ||
        launch_foldx_b(nt, grid, lds, s, f, mode, ch, starts, n) ||
        launch_foldx_c(nt, grid, lds, s, f, mode, ch, starts, n) ||
        launch_foldx_d(nt, grid, lds, s, f, mode, ch, starts, n))
        return hipGetLastError();
    return hipErrorInvalidValue;
}

hipError_t launch_foldc(unsigned nt, dim3 grid, size_t lds, hipStream_t s, const FoldC& f, int mode, const FoldC* ch,
                        const int64_t* starts, int n) {
    auto go = [&](auto kernel) {
        if (lds > 65536) allow_large_lds(kernel);
        hipLaunchKernelGGL(kernel, grid, dim3(nt), lds, s, f, ch, starts, n);
    };
    auto modes = [&](auto ntc) {
        constexpr int NT = decltype(ntc)::value;
        switch (mode) {
            case CM_FWD: go(k_foldc<CM_FWD, NT>); break;
            case CM_CONV: go(k_foldc<CM_CONV, NT>); break;
            case CM_CONVJ: go(k_foldc<CM_CONVJ, NT>); break;
            default: return hipErrorInvalidValue;
        }
        return hipGetLastError();
    };
    switch (nt) {
        case 256: return modes(std::integral_constant<int, 256>{});
        case 512: return modes(std::integral_constant<int, 512>{});
        case 1024: return modes(std::integral_constant<int, 1024>{});
        default: return hipErrorInvalidValue;
    }
}

}  // namespace pk
