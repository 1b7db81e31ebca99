// FP64 covariance-tile generator for gfx950: Cmm (type 1), Cmaa (2), Ctm (3), Ctt (4).
//
// Arithmetic follows the reference element by element (common/kernels/matcov_kernels.cpp):
//   vk_series      macdo_x56      37-62     x^(5/6) K_{5/6}(x) by its 11-term series
//   vk_asymptote   asymp_macdo    64-89     3-term Hankel asymptote for x > 3*pi/2
//   vk_dphi        rodconan/DPHI_gb 91-140  von Karman phase structure function
//   slope_cov      cov_XX/YY/XY/YX_gb 146-193  4-point second differences
//   meas_kernel    compute_element_tiled_4 + matcov_kernel_4   205-400
//   truth_kernel   compute_element_ts_tile + matcov_ts_kernel_tile 422-515
// with the tile/storage rules of MOAO_COMMON::matcov_tile (common/compute/matcov.cpp:17-98).
//
// GPU design (not a translation of matcov_kernels_gpu.cu):
//  * one lane per element, a wave runs down 64 consecutive rows of one column, so the column's
//    u/v/noise reads are wave-uniform and the 64 FP64 stores are one contiguous 512-byte run
//    of the column-major tile;
//  * the per-element WFS/subaperture/axis decode (a linear scan over WFS in the reference) is
//    a host-built int32 table per row and per column;
//  * per-layer constants 2*pi/L0 and k1*L0^(5/3) are computed once on the host with the
//    reference's own expressions (identical bits), not per call of the structure function;
//  * type 1 skips workgroups whose tile lies wholly above the diagonal;
//  * sensors on one regular grid (find_lattices) have as many covariances as the grid has
//    differences: lattice_table evaluates those, lattice_fill (whole matrices) and meas_kernel
//    (tiles) read them;
//  * the other pairs of a whole Cmm or Ctm (the lapack path's call) run pair_kernel: one lane
//    per pair of subapertures computes the pair's xx, xy, yx and yy elements, sharing the structure
//    functions those four have in common, bit-identical to the element kernel.
// Contraction into FMA is disabled here so each product/sum rounds as in the reference; the
// only differences left are the last-ulp differences of the device pow/exp/sqrt.
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "common.hpp"
#include "profile.hpp"
#include "stages.hpp"

namespace moao {
namespace {

constexpr double kPi = 3.1415926535897932384626433;
constexpr double kXlim = 0.75 * 2 * kPi;
constexpr double kLambda2 = 0.00026942094446267851;
constexpr double kK1 = 0.1716613621245709486;
constexpr double kK2 = 1.00563491799858928388289314170833;
constexpr double kK3 = 1.25331413731550012081;
constexpr double kA1 = 0.22222222222222222222;
constexpr double kA2 = -0.08641975308641974829;
constexpr double kA3 = 0.08001828989483310284;

// Series coefficients of the reference (common/moao_defs.h:18-27): Gamma-function values.
#define MOAO_VK_GA                                                                          \
    {0, 12.067619015983075, 5.17183672113560444, 0.795667187867016068, 0.0628158306210802181,  \
     0.00301515986981185091, 9.72632216068338833e-05, 2.25320204494595251e-06,               \
     3.93000356676612095e-08, 5.34694362825451923e-10, 5.83302941264329804e-12}
#define MOAO_VK_GMA                                                                         \
    {-3.74878707653729304, -2.04479295083852408, -0.360845814853857083, -0.0313778969438136685, \
     -0.001622994669507603, -5.56455315259749673e-05, -1.35720808599938951e-06,              \
     -2.47515152461894642e-08, -3.50257291219662472e-10, -3.95770950530691961e-12,           \
     -3.65327031259100284e-14}
__constant__ double cGa[11] = MOAO_VK_GA;
__constant__ double cGma[11] = MOAO_VK_GMA;

// Table of the normalised structure function f(t), t = q^2, q = 2 pi r / L0 (the function the two
// branches below define): kSub intervals per octave of t from 2^kLo up to 2^kHi, a polynomial of
// degree 5 each, then one constant (f is kK2 to the last bit past q = 45).  The interval that holds
// the branches' border q = 3 pi / 2 is there twice, with the series and with the asymptote.
// An evaluation costs its LDS reads (16 bytes a lane each): 6 coefficients at 1/64 octave, three
// reads, against 8 at 1/32 octave, four reads; two workgroups' tables fit a CU's LDS.
constexpr int kSub = 64, kSubBits = 6, kLo = -10, kHi = 11;
constexpr int kCoef = 6;
constexpr int kTabN = (kHi - kLo) * kSub + 2;
constexpr double kTBorder = kXlim * kXlim;
// Arguments below the table, those within rounding of the border, infinities and NaN take the direct
// formulas: interval numbers below 0 and from kInfinite on (one unsigned comparison).
constexpr int kInfinite = (2047 - 1023 - kLo) << kSubBits;
constexpr double kTBand = 1e-9;

constexpr int kRows = 64;       // rows per workgroup (one wave tall)
constexpr int kWaves = 8;       // waves per workgroup; each takes MatcovArgs::cw columns

constexpr int kLattice = -1, kFree = -2;  // MatcovArgs::cls without a table

struct MatcovArgs {
    double* out;
    long lda;
    int nrows, ncols, xoffset, yoffset;
    int Nlayer, nlgs, Nx, type_mat;
    int cw;                 // columns per wave
    double lgs_cst;
    const int* rowtab;      // packed (pos << 9) | (wfs << 1) | xy
    const int* coltab;
    const double* u;        // [Nlayer*Nx]
    const double* v;
    const double* sspL;     // [Nw*Nlayer]
    const double* lk;       // [Nlayer] 2*pi/L0
    const double* amp;      // [Nlayer] k1*L0^(5/3)
    const double* ftab;     // [kTabN * kCoef] table of f
    const double* cn2;      // [Nlayer]
    const double* sspsz;    // [Nw] diam/Nssp
    const double* nNGS;     // [Nw-nlgs]
    const double* nxx;      // [Nx]
    const double* nyy;
    const double* nxy;
    const double* X;        // [Nx]
    const double* Y;
    int truth_base;         // Nsubap_t*(Nw-1), index of the truth sensor's first subap
    int truth_nsub;         // Nsubap of the truth sensor
    // lattices: packed integer place (iy << 16 | ix) of every subaperture on its sensor's grid and
    // the grid's origin on every layer; cls[m*Nw + n]: slot of the pair's covariance table (rows of
    // sensor m, columns of n), kLattice (same grid, no table) or kFree
    const int* lat;         // [Nx]
    const double* u0;       // [Nw*Nlayer]
    const double* v0;
    const int* cls;         // [Nw*Nw]
    const int* slots;       // sensor pairs (m << 8 | n) of the tables
    double* ptab;           // [slots][3][W*W]: xx, yy, xy by (dy + ext - 1)*W + dx + ext - 1
    int Nw, ext;            // ext: cells across the widest lattice; W = 2*ext - 1
    // pair kernel (whole matrices of types 1 and 3): one entry per subaperture of the row and
    // column sensors, {(pos << 9) | (wfs << 1), matrix index of its x slope}; the y slope sits
    // nsub[wfs] further
    const int2* rsub;
    const int2* csub;
    const int* nsub;        // [Nw]
    int nrsub, ncsub;
};

// cx = cbrt(x), shared with vk_asymptote: lanes of one wave often take both branches.
__device__ __forceinline__ double vk_series(double x, double cx) {
    // x^(5/3) as x * cbrt(x)^2: a cube root costs a fraction of a general pow
    const double x2a = x * cx * cx;
    const double x22 = x * x / 4.;
    double xn = 0.5;
    double s = cGma[0] * x2a;
    s *= xn;
    xn *= x22;
#pragma unroll
    for (int n = 1; n <= 10; n++) {
        s += (cGma[n] * x2a + cGa[n]) * xn;
        xn *= x22;
    }
    return s;
}

__device__ __forceinline__ double vk_asymptote(double x, double cx) {
    const double ix = 1. / x;
    return kK2 - kK3 * exp(-x) * cx * (1.0 + ix * (kA1 + ix * (kA2 + ix * kA3)));
}

__device__ __forceinline__ double vk_dphi(double x, double y, double lk, double amp) {
    const double r = sqrt(x * x + y * y);
    const double q = lk * r;
    const double cq = cbrt(q);
    double res = (q > kXlim) ? vk_asymptote(q, cq) : -vk_series(q, cq);
    res *= amp;
    return res;
}

// The same function from the table (in LDS): t's exponent and top mantissa bits give the interval,
// its other bits the place in it (exact).  About 20 VALU instructions and three 16-byte LDS reads
// where sqrt, cube root, both branches and exp take about 230.
//
// N of them at a time: without a branch between them their LDS reads and products overlap (one by
// one, each waited for its own reads).  The direct formulas stay out of line, so the kernels'
// code is short of the instruction cache.
__device__ __noinline__ double vk_direct(double x, double y, double lk, double amp) {
    return vk_dphi(x, y, lk, amp);
}

template <int N>
__device__ __forceinline__ void vk_table(const double* tab, const double (&x)[N],
                                         const double (&y)[N], double lk, double amp,
                                         double (&f)[N]) {
    bool direct[N], any = false;
    double t[N];
    int iv[N];
#pragma unroll
    for (int n = 0; n < N; ++n) {
        t[n] = fma(x[n], x[n], y[n] * y[n]) * (lk * lk);
        iv[n] = (int)((unsigned)__double2hiint(t[n]) >> (20 - kSubBits)) -
                ((1023 + kLo) << kSubBits);
        direct[n] = (unsigned)iv[n] >= (unsigned)kInfinite || fabs(t[n] - kTBorder) < kTBand;
        any = any || direct[n];
    }
#pragma unroll
    for (int n = 0; n < N; ++n) {
        const unsigned hi = (unsigned)__double2hiint(t[n]);
        const int k = max(min(iv[n] + (t[n] > kTBorder ? 1 : 0), kTabN - 1), 0);
        const double w = __hiloint2double((int)((hi & ((1u << (20 - kSubBits)) - 1)) | 0x3ff00000u),
                                          __double2loint(t[n]));
        const double z = w - (1.0 + 0.5 / kSub);
        // coefficients 2c, 2c + 1 of interval k at double2 c * kTabN + k: lanes in different
        // intervals read neighbouring 16-byte pieces, not one bank group apart
        const double2* c = (const double2*)tab + k;
        double v = 0.0;
#pragma unroll
        for (int q = kCoef / 2 - 1; q >= 0; --q) {
            const double2 p = c[q * kTabN];
            v = q == kCoef / 2 - 1 ? p.y : fma(v, z, p.y);
            v = fma(v, z, p.x);
        }
        f[n] = v * amp;
    }
    if (__builtin_expect(any, 0)) {
#pragma unroll
        for (int n = 0; n < N; ++n)
            if (direct[n]) f[n] = vk_direct(x[n], y[n], lk, amp);
    }
}

__device__ __forceinline__ void load_table(const double* src, double* tab) {
    for (int e = threadIdx.x; e < kTabN * kCoef / 2; e += kWaves * 64)
        ((double2*)tab)[e] = ((const double2*)src)[e];
    __syncthreads();
}

// -D(p0) + D(p1) + D(p2) - D(p3): the second difference that is a slope covariance.
__device__ __forceinline__ double second_difference(const double (&f)[4]) {
    return -f[0] + f[1] + f[2] - f[3];
}

// kind: 0 xx, 1 xy, 2 yx, 3 yy.  Equal sizes (s1 == s2): the first and last term of xx and yy are
// D(du, dv) both, with the same bits.
__device__ __forceinline__ double slope_cov(const double* tab, int kind, double du, double dv,
                                            double s1, double s2, double lk, double amp) {
    const double ac = s1 - s2, ad = s1 + s2, bc = -ad, bd = -ac;
    double x[4], y[4], f[4];
    if (kind == 0 || kind == 3) {
        const double o[4] = {ac, ad, bc, bd};
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            x[n] = kind == 0 ? du + o[n] : du;
            y[n] = kind == 0 ? dv : dv + o[n];
        }
    } else {
        const double ox[4] = {s1, s1, -s1, -s1}, oy[4] = {-s2, s2, -s2, s2};
        const double px[4] = {-s2, s2, -s2, s2}, py[4] = {s1, s1, -s1, -s1};
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            x[n] = du + (kind == 1 ? ox[n] : px[n]);
            y[n] = dv + (kind == 1 ? oy[n] : py[n]);
        }
    }
    vk_table<4>(tab, x, y, lk, amp, f);
    return second_difference(f);
}

// xx and yy, and xy, of sensors of one subaperture size s1 + s1 = ad: nine structure functions.
__device__ __forceinline__ void slope_cov_equal(const double* tab, double du, double dv, double s1,
                                                double lk, double amp, bool diag, double& sxx,
                                                double& syy, double& sxy) {
    const double ad = s1 + s1, bc = -ad;
    if (diag) {
        const double x[5] = {du, du + ad, du + bc, du, du}, y[5] = {dv, dv, dv, dv + ad, dv + bc};
        double f[5];
        vk_table<5>(tab, x, y, lk, amp, f);
        sxx = -f[0] + f[1] + f[2] - f[0];
        syy = -f[0] + f[3] + f[4] - f[0];
    }
    const double x[4] = {du + s1, du + s1, du - s1, du - s1};
    const double y[4] = {dv - s1, dv + s1, dv - s1, dv + s1};
    double f[4];
    vk_table<4>(tab, x, y, lk, amp, f);
    sxy = second_difference(f);
}

// Separation of subapertures p1 (sensor m) and p2 (sensor n) on layer l.  On a common lattice it
// is a function of the integer places' difference alone, so every pair of one difference has the
// same bits, whichever kernel computes it; else the difference of the positions.
__device__ __forceinline__ void lattice_separation(const MatcovArgs& a, int m, int n, int dx, int dy,
                                                   int l, double step, double& du, double& dv) {
    const int om = m * a.Nlayer + l, on = n * a.Nlayer + l;
    du = (a.u0[om] - a.u0[on]) + dx * step;
    dv = (a.v0[om] - a.v0[on]) + dy * step;
}
__device__ __forceinline__ int lat_dx(int a, int b) { return (a & 0xffff) - (b & 0xffff); }
__device__ __forceinline__ int lat_dy(int a, int b) { return (a >> 16) - (b >> 16); }
__device__ __forceinline__ void separation(const MatcovArgs& a, bool lattice, int m, int n, int p1,
                                           int p2, int l, double step, double& du, double& dv) {
    if (lattice) {
        lattice_separation(a, m, n, lat_dx(a.lat[p1], a.lat[p2]), lat_dy(a.lat[p1], a.lat[p2]), l,
                           step, du, dv);
        return;
    }
    const long o = (long)l * a.Nx;
    du = a.u[o + p1] - a.u[o + p2];
    dv = a.v[o + p1] - a.v[o + p2];
}

// Covariance tables of the sensor pairs on a common lattice (both sensors' subapertures on one
// grid with the same size on every layer: every LGS pair of one altitude, every NGS pair).  All
// subaperture pairs of one lattice difference have the same xx, yy and xy (= yx) covariance, and
// there are (2*ext - 1)^2 differences against Nsubap^2 pairs (79^2 against 1168^2 at 40 x 40): one
// lane per difference and layer evaluates it, lattice_fill and meas_kernel read it.  A
// workgroup takes 64 differences, its waves the layers in turn (the chain of layers one lane would
// walk was most of the time); the terms meet in LDS and are added in layer order, as an element
// on its own adds them.
__global__ void __launch_bounds__(kWaves * 64) lattice_table(MatcovArgs a) {
    __shared__ __attribute__((aligned(16))) double tab[kTabN * kCoef];
    __shared__ double term[kWaves][3][64];
    load_table(a.ftab, tab);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int W = 2 * a.ext - 1, e = blockIdx.x * 64 + lane, WW = W * W;
    const int pr = a.slots[blockIdx.y], m = pr >> 8, n = pr & 0xff;
    const int dx = e % W - (a.ext - 1), dy = e / W - (a.ext - 1);
    const double kk = kLambda2 / (a.sspsz[m] * a.sspsz[n]);
    double sum = 0.0;  // waves 0, 1, 2: xx, yy, xy
    for (int l0 = 0; l0 < a.Nlayer; l0 += kWaves) {
        const int l = l0 + wave;
        const double sz = l < a.Nlayer ? a.sspL[m * a.Nlayer + l] : 0.0;
        if (sz > 0) {
            double du, dv;
            lattice_separation(a, m, n, dx, dy, l, sz, du, dv);
            double sxx = 0.0, syy = 0.0, sxy = 0.0;
            slope_cov_equal(tab, du, dv, sz * 0.5, a.lk[l], a.amp[l], true, sxx, syy, sxy);
            term[wave][0][lane] = 0.5 * sxx * kk * a.cn2[l];
            term[wave][1][lane] = 0.5 * syy * kk * a.cn2[l];
            term[wave][2][lane] = 0.5 * sxy * kk * a.cn2[l];
        }
        __syncthreads();
        if (wave < 3)
            for (int k = 0; k < kWaves && l0 + k < a.Nlayer; ++k)
                if (a.sspL[m * a.Nlayer + l0 + k] > 0) sum += term[k][wave][lane];
        __syncthreads();
    }
    if (wave < 3 && e < WW) a.ptab[((long)blockIdx.y * 3 + wave) * WW + e] = sum;
}

// Whole Cmm or Ctm: the pairs that have a table.  Bound by its stores (8 B an element; the tables
// are read from L2).  Rows and columns as in pair_kernel, which takes the other pairs.
__global__ void __launch_bounds__(256) lattice_fill(MatcovArgs a, int cols_per_wave) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int rs = blockIdx.x * 64 + lane;
    const int cs0 = (blockIdx.y * 4 + wave) * cols_per_wave;
    if (rs >= a.nrsub) return;
    const int2 re = a.rsub[rs];
    const int m = (re.x >> 1) & 0xff, p1 = re.x >> 9, la = a.lat[p1];
    const int xr = re.y, yr = re.y + a.nsub[m];
    const int W = 2 * a.ext - 1, WW = W * W;
    for (int c = 0; c < cols_per_wave; ++c) {
        const int cs = cs0 + c;
        if (cs >= a.ncsub) break;
        const int2 ce = a.csub[cs];
        const int n = (ce.x >> 1) & 0xff, p2 = ce.x >> 9;
        const int xc = ce.y, yc = ce.y + a.nsub[n];
        const bool lo = a.type_mat == 1;
        const bool nxx = !lo || xr >= xc, nyy = !lo || yr >= yc;
        const bool nxy = !lo || xr >= yc, nyx = !lo || yr >= xc;
        const int slot = a.cls[m * a.Nw + n];
        if (!nyx || slot < 0) continue;
        const int lb = a.lat[p2];
        const double* t = a.ptab + (long)slot * 3 * WW + (lat_dy(la, lb) + a.ext - 1) * W +
                          lat_dx(la, lb) + a.ext - 1;
        double cxx = t[0], cyy = t[WW], cxy = t[2 * WW], cyx = cxy;
        if (m == n) {
            if (m < a.nlgs) {
                if (p1 == p2) {
                    cxx += a.nxx[p1];
                    cyy += a.nyy[p1];
                    cxy += a.nxy[p1];
                    cyx += a.nxy[p1];
                }
                cxx += a.lgs_cst;
                cyy += a.lgs_cst;
            } else if (p1 == p2) {
                cxx += a.nNGS[m - a.nlgs];
                cyy += a.nNGS[m - a.nlgs];
            }
        }
        double* ox = a.out + (long)xc * a.lda;
        double* oy = a.out + (long)yc * a.lda;
        if (nxx) ox[xr] = cxx;
        ox[yr] = cyx;
        if (nxy) oy[xr] = cxy;
        if (nyy) oy[yr] = cyy;
    }
}

// Whether a sensor of rows [m0, m1] and one of columns [n0, n1] have to be evaluated (no table).
__device__ __forceinline__ bool any_without_table(const MatcovArgs& a, int m0, int m1, int n0,
                                                  int n1) {
    bool any = false;
    for (int m = m0; m <= m1; ++m)
        for (int n = n0; n <= n1; ++n) any = any || a.cls[m * a.Nw + n] < 0;
    return any;
}

__global__ void __launch_bounds__(kWaves * 64) meas_kernel(MatcovArgs a) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int lx = blockIdx.x * kRows + lane;
    const int kCols = kWaves * a.cw, ly0 = blockIdx.y * kCols + wave * a.cw;
    if (a.type_mat == 1) {
        // whole workgroup above the diagonal: nothing to write
        const int last_row = a.xoffset + min(a.nrows - 1, (int)blockIdx.x * kRows + kRows - 1);
        if (last_row < a.yoffset + (int)blockIdx.y * kCols) return;
    }
    __shared__ __attribute__((aligned(16))) double tab[kTabN * kCoef];
    const int cl = min((int)blockIdx.y * kCols + kCols, a.ncols) - 1;
    const int rl = min((int)blockIdx.x * kRows + kRows, a.nrows) - 1;
    if (any_without_table(a, (a.rowtab[blockIdx.x * kRows] >> 1) & 0xff, (a.rowtab[rl] >> 1) & 0xff,
                          (a.coltab[blockIdx.y * kCols] >> 1) & 0xff, (a.coltab[cl] >> 1) & 0xff))
        load_table(a.ftab, tab);
    if (lx >= a.nrows) return;
    const int ri = a.rowtab[lx];
    const int m = (ri >> 1) & 0xff, xi = ri & 1, p1 = ri >> 9;
    const int gx = lx + a.xoffset;
    for (int c = 0; c < a.cw; ++c) {
        const int ly = ly0 + c;
        if (ly >= a.ncols) break;
        if (a.type_mat == 1 && ly + a.yoffset > gx) continue;
        const int ci = a.coltab[ly];
        const int n = (ci >> 1) & 0xff, xj = ci & 1, p2 = ci >> 9;
        const int kind = xi * 2 + xj;
        const int cls = a.cls[m * a.Nw + n];
        const double kk = kLambda2 / (a.sspsz[m] * a.sspsz[n]);
        double covar = 0.0;
        if (cls >= 0) {
            const int W = 2 * a.ext - 1, la = a.lat[p1], lb = a.lat[p2];
            covar = a.ptab[((long)cls * 3 + (kind == 0 ? 0 : kind == 3 ? 1 : 2)) * W * W +
                           (lat_dy(la, lb) + a.ext - 1) * W + lat_dx(la, lb) + a.ext - 1];
        } else {
            // on a common lattice yx is xy, as in the tables
            const int k = cls == kLattice && kind == 2 ? 1 : kind;
            for (int l = 0; l < a.Nlayer; ++l) {
                const double sml = a.sspL[m * a.Nlayer + l];
                const double snl = a.sspL[n * a.Nlayer + l];
                if ((sml > 0) && (snl > 0)) {
                    double du, dv;
                    separation(a, cls == kLattice, m, n, p1, p2, l, sml, du, dv);
                    covar += 0.5 * slope_cov(tab, k, du, dv, sml * 0.5, snl * 0.5, a.lk[l],
                                             a.amp[l]) * kk * a.cn2[l];
                }
            }
        }
        if (m == n) {
            if (m < a.nlgs) {
                if (p1 == p2) {
                    if (kind == 0) covar += a.nxx[p1];
                    else if (kind == 3) covar += a.nyy[p1];
                    else covar += a.nxy[p1];
                }
                if (kind == 0 || kind == 3) covar += a.lgs_cst;
            } else if (p1 == p2 && (kind == 0 || kind == 3)) {
                covar += a.nNGS[m - a.nlgs];
            }
        }
        a.out[(long)ly * a.lda + lx] = covar;
    }
}

// Whole Cmm (type 1) or Ctm (type 3): one lane per pair of subapertures computes the 2 x 2
// block xx, xy, yx, yy of that pair, so the four slope covariances share their structure
// functions.  Per layer, for equal subaperture sizes (every pair of sensors at one altitude),
// xx and yy share D(du, dv), and xy and yx use the same four corners (du +- s, dv +- s): 9
// evaluations instead of the 14 the four elements take one by one.  Every element keeps the
// element kernel's expression and order (same arguments, same sums, same layer order), so the
// result is bit-identical to it.  Lanes run down consecutive row subapertures: the x and y
// rows of a pair are two contiguous runs of each column.
__global__ void __launch_bounds__(kWaves * 64) pair_kernel(MatcovArgs a) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int rs = blockIdx.x * kRows + lane;
    const int kCols = kWaves * a.cw, cs0 = blockIdx.y * kCols + wave * a.cw;
    if (a.type_mat == 1) {
        // no pair of this workgroup has a row (its y slope's, the largest) at or below a column
        const int2 last = a.rsub[min((int)blockIdx.x * kRows + kRows, a.nrsub) - 1];
        if (last.y + a.nsub[(last.x >> 1) & 0xff] < a.csub[blockIdx.y * kCols].y) return;
    }
    {
        const int2 r0 = a.rsub[blockIdx.x * kRows];
        const int2 r1 = a.rsub[min((int)blockIdx.x * kRows + kRows, a.nrsub) - 1];
        const int2 c0 = a.csub[blockIdx.y * kCols];
        const int2 c1 = a.csub[min((int)blockIdx.y * kCols + kCols, a.ncsub) - 1];
        if (!any_without_table(a, (r0.x >> 1) & 0xff, (r1.x >> 1) & 0xff, (c0.x >> 1) & 0xff,
                               (c1.x >> 1) & 0xff))
            return;  // lattice_fill's
    }
    __shared__ __attribute__((aligned(16))) double tab[kTabN * kCoef];
    load_table(a.ftab, tab);
    if (rs >= a.nrsub) return;
    const int2 re = a.rsub[rs];
    const int m = (re.x >> 1) & 0xff, p1 = re.x >> 9;
    const int xr = re.y, yr = re.y + a.nsub[m];
    for (int c = 0; c < a.cw; ++c) {
        const int cs = cs0 + c;
        if (cs >= a.ncsub) break;
        const int2 ce = a.csub[cs];
        const int n = (ce.x >> 1) & 0xff, p2 = ce.x >> 9;
        const int xc = ce.y, yc = ce.y + a.nsub[n];
        // type 1 writes only row >= column: nothing of this pair when its largest row is above
        // its smallest column; in a sensor's diagonal block a pair may need only some of its
        // four elements, and only their structure functions are evaluated
        const bool lo = a.type_mat == 1;
        const bool nxx = !lo || xr >= xc, nyy = !lo || yr >= yc;
        const bool nxy = !lo || xr >= yc, nyx = !lo || yr >= xc;
        const int cls = a.cls[m * a.Nw + n];
        // yx has the largest row and the smallest column; pairs with a table are lattice_fill's
        if (!nyx || cls >= 0) continue;
        const double kk = kLambda2 / (a.sspsz[m] * a.sspsz[n]);
        double cxx = 0.0, cxy = 0.0, cyx = 0.0, cyy = 0.0;
        for (int l = 0; l < a.Nlayer; ++l) {
            const double sml = a.sspL[m * a.Nlayer + l];
            const double snl = a.sspL[n * a.Nlayer + l];
            if ((sml > 0) && (snl > 0)) {
                double du, dv;
                separation(a, cls == kLattice, m, n, p1, p2, l, sml, du, dv);
                const double s1 = sml * 0.5, s2 = snl * 0.5;
                const double lk = a.lk[l], amp = a.amp[l];
                double sxx = 0.0, syy = 0.0, sxy = 0.0, syx;
                if (s1 == s2) {
                    slope_cov_equal(tab, du, dv, s1, lk, amp, nxx || nyy, sxx, syy, sxy);
                    // the corners of yx are those of xy, added in another order (on a common
                    // lattice yx is xy, as in the tables): its own element's expression
                    syx = cls == kLattice ? sxy : slope_cov(tab, 2, du, dv, s1, s2, lk, amp);
                } else {
                    if (nxx) sxx = slope_cov(tab, 0, du, dv, s1, s2, lk, amp);
                    if (nyy) syy = slope_cov(tab, 3, du, dv, s1, s2, lk, amp);
                    if (nxy) sxy = slope_cov(tab, 1, du, dv, s1, s2, lk, amp);
                    syx = slope_cov(tab, 2, du, dv, s1, s2, lk, amp);
                }
                cxx += 0.5 * sxx * kk * a.cn2[l];
                cxy += 0.5 * sxy * kk * a.cn2[l];
                cyx += 0.5 * syx * kk * a.cn2[l];
                cyy += 0.5 * syy * kk * a.cn2[l];
            }
        }
        if (m == n) {
            if (m < a.nlgs) {
                if (p1 == p2) {
                    cxx += a.nxx[p1];
                    cyy += a.nyy[p1];
                    cxy += a.nxy[p1];
                    cyx += a.nxy[p1];
                }
                cxx += a.lgs_cst;
                cyy += a.lgs_cst;
            } else if (p1 == p2) {
                cxx += a.nNGS[m - a.nlgs];
                cyy += a.nNGS[m - a.nlgs];
            }
        }
        double* ox = a.out + (long)xc * a.lda;
        double* oy = a.out + (long)yc * a.lda;
        if (nxx) ox[xr] = cxx;
        ox[yr] = cyx;
        if (nxy) oy[xr] = cxy;
        if (nyy) oy[yr] = cyy;
    }
}

__global__ void __launch_bounds__(kWaves * 64) truth_kernel(MatcovArgs a) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int lx = blockIdx.x * kRows + lane;
    const int kCols = kWaves * a.cw, ly0 = blockIdx.y * kCols + wave * a.cw;
    __shared__ __attribute__((aligned(16))) double tab[kTabN * kCoef];
    load_table(a.ftab, tab);
    if (lx >= a.nrows) return;
    const int gx = lx + a.xoffset;
    const int ns = a.truth_nsub;
    const int i = gx < ns ? gx : gx - ns;
    const int xi = gx < ns ? 0 : 1;
    const double ss = a.sspsz[0];  // diam / Nssp of the truth sensor (set by the host)
    const double kk = kLambda2 / (ss * ss);
    const double s = ss * 0.5;
    for (int c = 0; c < a.cw; ++c) {
        const int ly = ly0 + c;
        if (ly >= a.ncols) break;
        const int gy = ly + a.yoffset;
        const int j = gy < ns ? gy : gy - ns;
        const int xj = gy < ns ? 0 : 1;
        const int kind = xi * 2 + xj;
        const double du = a.X[a.truth_base + i] - a.X[a.truth_base + j];
        const double dv = a.Y[a.truth_base + i] - a.Y[a.truth_base + j];
        double covar = 0.0;
        for (int l = 0; l < a.Nlayer; ++l) {
            if (ss > 0) covar += 0.5 * slope_cov(tab, kind, du, dv, s, s, a.lk[l], a.amp[l]) * kk * a.cn2[l];
        }
        a.out[(long)ly * a.lda + lx] = covar;
    }
}

// Packed decode of measurement index g for the non-truth sensors (type 1/2/3 columns, type 1/2
// rows): WFS found by the cumulative 2*Nsubap scan of compute_element_tiled_4, x slopes first.
inline int pack_meas(long g, const moao_tomo_view* t, const std::vector<long>& off) {
    int w = 0;
    while (w < t->Nw - 1 && g >= 2 * (off[w] + t->Nsubap[w])) ++w;
    long i = g - 2 * off[w];
    int xy = 0;
    if (i >= t->Nsubap[w]) { i -= t->Nsubap[w]; xy = 1; }
    return (int)(((off[w] + i) << 9) | (w << 1) | xy);
}

// Row decode of type 3 (and column decode of type 2): the truth sensor.
inline int pack_truth(long g, const moao_tomo_view* t, const std::vector<long>& off) {
    const int w = t->Nw - 1;
    long i = g;
    int xy = 0;
    if (i >= t->Nsubap[w]) { i -= t->Nsubap[w]; xy = 1; }
    return (int)(((off[w] + i) << 9) | (w << 1) | xy);
}

// Coefficients of the table of f: interpolation at the kCoef Chebyshev points of an interval, in
// extended precision, as a polynomial in z = mantissa - (1 + 1/(2 kSub)) of the interval's start.
std::vector<double> structure_table() {
    auto series = [](long double t) {
        const long double q53 = std::pow(t, 5.0L / 6.0L), x22 = t / 4;
        const double ga[11] = MOAO_VK_GA, gma[11] = MOAO_VK_GMA;
        long double xn = 0.5L, s = 0;
        for (int n = 0; n <= 10; ++n, xn *= x22) s += (gma[n] * q53 + ga[n]) * xn;
        return -s;
    };
    auto asymptote = [](long double t) {
        const long double x = std::sqrt(t), ix = 1 / x;
        return kK2 - kK3 * std::exp(-x) * std::cbrt(x) *
                         (1 + ix * (kA1 + ix * (kA2 + ix * (long double)kA3)));
    };
    std::vector<double> tab((size_t)kTabN * kCoef, 0.0);
    for (int k = 0; k + 1 < kTabN; ++k) {
        // intervals past the border's are one entry later (its second copy)
        const int border = (int)((std::floor(std::log2(kTBorder)) - kLo) * kSub +
                                 (kTBorder / std::exp2(std::floor(std::log2(kTBorder))) - 1) * kSub);
        const int iv = k <= border ? k : k - 1;
        const int e = kLo + iv / kSub;
        const long double mid = 1 + (iv % kSub) / (long double)kSub + 0.5L / kSub;
        long double z[kCoef], c[kCoef];
        for (int n = 0; n < kCoef; ++n) {
            z[n] = std::cos((2 * n + 1) * (long double)kPi / (2 * kCoef)) / (2 * kSub);
            const long double t = std::ldexp(mid + z[n], e);
            c[n] = k <= border ? series(t) : asymptote(t);
        }
        for (int o = 1; o < kCoef; ++o)  // Newton's divided differences
            for (int n = kCoef - 1; n >= o; --n) c[n] = (c[n] - c[n - 1]) / (z[n] - z[n - o]);
        long double p[kCoef] = {};       // ... multiplied out
        for (int n = kCoef - 1; n >= 0; --n) {
            for (int d = kCoef - 1; d >= 1; --d) p[d] = p[d - 1] - z[n] * p[d];
            p[0] = c[n] - z[n] * p[0];
        }
        for (int d = 0; d < kCoef; ++d) tab[2 * ((size_t)(d / 2) * kTabN + k) + d % 2] = (double)p[d];
    }
    tab[2 * (size_t)(kTabN - 1)] = kK2;
    return tab;
}

// The table on the device, made on the first use and kept for the life of the process (63 KiB).
int structure_table_dev(const double** out) {
    static std::mutex mu;
    static double* dev = nullptr;
    std::lock_guard<std::mutex> g(mu);
    if (!dev) {
        const std::vector<double> tab = structure_table();
        double* d = nullptr;
        MOAO_HIP_TRY(hipMalloc(reinterpret_cast<void**>(&d), sizeof(double) * tab.size()));
        if (hipMemcpy(d, tab.data(), sizeof(double) * tab.size(), hipMemcpyHostToDevice) !=
            hipSuccess) {
            (void)hipFree(d);
            set_error("matcov: table upload failed");
            return MOAO_ERR_HIP;
        }
        dev = d;
    }
    *out = dev;
    return MOAO_OK;
}

// Regular grids among the sensors' subapertures.
struct Lattices {
    std::vector<int> place;         // [Nx] iy << 16 | ix
    std::vector<double> u0, v0;     // [Nw*Nlayer] grid origin on each layer
    std::vector<char> ok;           // [Nw] the sensor is a grid on every layer it sees
    int ext = 1;                    // cells across the widest grid
    // Sensors m and n on one grid: the same subaperture size, on the ground and on every layer.
    bool same(const moao_tomo_view* t, int m, int n) const {
        if (!ok[m] || !ok[n] || t->Nssp[m] != t->Nssp[n]) return false;
        const int L = t->Nlayer;
        for (int l = 0; l < L; ++l)
            if (t->sspSizeL[m * L + l] != t->sspSizeL[n * L + l]) return false;
        return true;
    }
};

// A sensor is a grid when its unprojected positions are integer multiples of its subaperture size
// apart and its positions on every layer are origin + place * size on that layer to within 4 ulp of
// their magnitude (projection scales and shifts them; a rotated sensor fails).  The origin is the
// mean of what the subapertures give, so it is nearer the exact one than any single position.
Lattices find_lattices(const moao_tomo_view* t, const std::vector<long>& off,
                       const std::vector<char>& used, const std::vector<double>& pitch) {
    const int Nw = t->Nw, L = t->Nlayer;
    Lattices r;
    r.place.assign(t->Nx, 0);
    r.u0.assign((size_t)Nw * L, 0.0);
    r.v0.assign((size_t)Nw * L, 0.0);
    r.ok.assign(Nw, 0);
    std::vector<double> fx, fy;
    for (int w = 0; w < Nw; ++w) {
        const long N = t->Nsubap[w], o = off[w];
        if (!used[w] || N < 1 || !(pitch[w] > 0)) continue;
        const double* X = t->X + o;
        const double* Y = t->Y + o;
        const double x0 = *std::min_element(X, X + N), y0 = *std::min_element(Y, Y + N);
        fx.resize(N);
        fy.resize(N);
        double most = 0;
        bool ok = true;  // comparisons that a NaN fails
        for (long i = 0; i < N; ++i) {
            const double x = (X[i] - x0) / pitch[w], y = (Y[i] - y0) / pitch[w];
            fx[i] = std::floor(x + 0.5);
            fy[i] = std::floor(y + 0.5);
            ok = ok & (std::fabs(x - fx[i]) < 1e-6) & (std::fabs(y - fy[i]) < 1e-6);
            most = std::max(most, std::max(fx[i], fy[i]));
        }
        ok = ok && most < 1024;
        for (int l = 0; l < L && ok; ++l) {
            const double s = t->sspSizeL[w * L + l];
            if (!(s > 0)) continue;
            auto origin = [&](const double* u, const double* f, double& u0) {
                const double first = u[0] - f[0] * s;
                double sum = 0, lo = first, hi = first;  // sum: of the differences to the first
                for (long i = 0; i < N; ++i) {
                    const double d = u[i] - f[i] * s;
                    sum += d - first;
                    lo = std::min(lo, d);
                    hi = std::max(hi, d);
                }
                u0 = first + sum / N;
                const double tol = 4 * 0x1p-52 * (std::fabs(u0) + most * s);
                return hi - u0 <= tol && u0 - lo <= tol;  // false for a NaN
            };
            const long lo = (long)l * t->Nx + o;
            ok = origin(t->u + lo, fx.data(), r.u0[w * L + l]) &&
                 origin(t->v + lo, fy.data(), r.v0[w * L + l]);
        }
        if (!ok) continue;
        r.ok[w] = 1;
        r.ext = std::max(r.ext, (int)most + 1);
        for (long i = 0; i < N; ++i) r.place[o + i] = (int)fy[i] << 16 | (int)fx[i];
    }
    return r;
}

size_t align256(size_t b) { return (b + 255) & ~size_t(255); }

}  // namespace

int matcov_tile_launch(double* d_data, int nrows, int ncols, int xoffset, int yoffset, int lda,
                       const moao_tomo_view* t, int type_mat, hipStream_t stream, MatcovTables* tables) {
    if (type_mat < 1 || type_mat > 4) {
        set_error("matcov_tile: unrecognized type_mat " + std::to_string(type_mat));
        return MOAO_ERR_ARG;
    }
    if (!t || nrows < 0 || ncols < 0 || lda < std::max(1, nrows) || xoffset < 0 || yoffset < 0 ||
        t->Nw < 2 || t->Nw > 255 || t->Nlayer < 1 || t->Nx < 1 || t->Nx >= (1L << 22)) {
        set_error("matcov_tile: invalid arguments");
        return MOAO_ERR_ARG;
    }
    if (nrows == 0 || ncols == 0) return MOAO_OK;
    const int Nw = t->Nw, L = t->Nlayer;
    const long Nx = t->Nx;
    std::vector<long> off(Nw, 0);
    for (int w = 1; w < Nw; ++w) off[w] = off[w - 1] + t->Nsubap[w - 1];
    const long nmeas = 2 * (Nx - t->Nsubap[Nw - 1]);
    const long nts = 2 * t->Nsubap[Nw - 1];
    // Row/column ranges must stay inside the matrix the type describes.
    long row_lim = (type_mat == 3 || type_mat == 4) ? nts : nmeas;
    long col_lim = (type_mat == 2 || type_mat == 4) ? nts : nmeas;
    if ((long)xoffset + nrows > row_lim || (long)yoffset + ncols > col_lim) {
        set_error("matcov_tile: tile exceeds the matrix of this type");
        return MOAO_ERR_ARG;
    }
    if (type_mat == 2 || type_mat == 4) {
        for (int w = 0; w < Nw; ++w)
            if (t->Nsubap[w] != t->Nsubap[0]) {
                set_error("matcov_tile: types 2 and 4 assume equal Nsubap on every WFS");
                return MOAO_ERR_ARG;
            }
    }

    if (type_mat == 1 && xoffset + nrows - 1 < yoffset) {
        // wholly above the diagonal: nothing to write, no tables to build or upload (1,000 x 1,000 at
        // n = 18,688: 147 -> 1.6 us); as below, the call returns when the stream is idle
        MOAO_HIP_TRY(hipStreamSynchronize(stream));
        return MOAO_OK;
    }

    // Whole Cmm / Ctm: lattice_fill and pair_kernel (one lane per subaperture pair).
    const bool pairs = (type_mat == 1 || type_mat == 3) && xoffset == 0 && yoffset == 0 &&
                       nrows == row_lim && ncols == col_lim;
    std::vector<int> rowtab, coltab;
    if (!pairs && type_mat != 4) {
        rowtab.resize(nrows);
        coltab.resize(ncols);
        for (int r = 0; r < nrows; ++r)
            rowtab[r] = (type_mat == 3) ? pack_truth(r + xoffset, t, off)
                                        : pack_meas(r + xoffset, t, off);
        for (int c = 0; c < ncols; ++c)
            coltab[c] = (type_mat == 2) ? pack_truth(c + yoffset, t, off)
                                        : pack_meas(c + yoffset, t, off);
    }
    std::vector<int2> rsub, csub;
    std::vector<int> nsub(Nw);
    for (int w = 0; w < Nw; ++w) nsub[w] = (int)t->Nsubap[w];
    if (pairs) {
        csub.reserve(nmeas / 2);
        for (int w = 0; w < Nw - 1; ++w)
            for (long i = 0; i < t->Nsubap[w]; ++i)
                csub.push_back(make_int2((int)(((off[w] + i) << 9) | (w << 1)),
                                         (int)(2 * off[w] + i)));
        if (type_mat == 1) {
            rsub = csub;
        } else {
            const int w = Nw - 1;
            for (long i = 0; i < t->Nsubap[w]; ++i)
                rsub.push_back(make_int2((int)(((off[w] + i) << 9) | (w << 1)), (int)i));
        }
    }
    std::vector<double> lk(L), amp(L), sspsz(Nw);
    for (int l = 0; l < L; ++l) {
        const double L0 = t->L0[l];
        lk[l] = (2 * kPi / L0);
        amp[l] = kK1 * std::pow(L0, 5. / 3.0);
    }
    for (int w = 0; w < Nw; ++w) sspsz[w] = t->diam / t->Nssp[w];
    if (type_mat == 4) sspsz[0] = t->diam / t->Nssp[Nw - 1];
    const int nngs = Nw - t->nlgs;

    // Sensors of the rows and of the columns, their lattices and the pairs that share one.
    std::vector<int> cls, slots;
    Lattices lat;
    bool positions = false;  // some pair reads u, v
    if (type_mat != 4) {
        const int rm0 = pairs ? (rsub.front().x >> 1) & 0xff : (rowtab.front() >> 1) & 0xff;
        const int rm1 = pairs ? (rsub.back().x >> 1) & 0xff : (rowtab.back() >> 1) & 0xff;
        const int cn0 = pairs ? (csub.front().x >> 1) & 0xff : (coltab.front() >> 1) & 0xff;
        const int cn1 = pairs ? (csub.back().x >> 1) & 0xff : (coltab.back() >> 1) & 0xff;
        std::vector<char> used(Nw, 0);
        for (int w = rm0; w <= rm1; ++w) used[w] = 1;
        for (int w = cn0; w <= cn1; ++w) used[w] = 1;
        lat = find_lattices(t, off, used, sspsz);
        cls.assign((size_t)Nw * Nw, kFree);
        for (int m = rm0; m <= rm1; ++m)
            for (int n = cn0; n <= cn1; ++n) {
                if (type_mat == 1 && n > m) continue;  // above the diagonal
                if (lat.same(t, m, n)) {
                    cls[m * Nw + n] = kLattice;
                    slots.push_back(m << 8 | n);
                } else {
                    positions = true;
                }
            }
        // A table entry takes 9 structure functions a layer, an element on its own 3 or 4: tables
        // where they are the smaller work (a tile of a few hundred elements is not), 256 MiB at most
        // or what the caller has room for.
        const double W = 2.0 * lat.ext - 1;
        const double room = tables && tables->space ? tables->space_bytes : 256 << 20;
        if (slots.size() * W * W * 9 < 3.5 * nrows * ncols && slots.size() * W * W * 24 <= room) {
            for (size_t k = 0; k < slots.size(); ++k)
                cls[(slots[k] >> 8) * Nw + (slots[k] & 0xff)] = (int)k;
        } else {
            slots.clear();
        }
    }

    // One contiguous upload of every vector the kernels read.
    struct Piece { const void* src; size_t bytes; size_t off; };
    std::vector<Piece> pieces;
    size_t total = 0;
    auto add = [&](const void* src, size_t bytes) {
        pieces.push_back({src, bytes, total});
        total += align256(bytes);
        return pieces.size() - 1;
    };
    const bool noise = type_mat == 1;  // only its sensors meet themselves
    const size_t iRow = add(rowtab.data(), sizeof(int) * rowtab.size());
    const size_t iCol = add(coltab.data(), sizeof(int) * coltab.size());
    const size_t iU = add(t->u, positions ? sizeof(double) * L * Nx : 0);
    const size_t iV = add(t->v, positions ? sizeof(double) * L * Nx : 0);
    const size_t iS = add(t->sspSizeL, sizeof(double) * Nw * L);
    const size_t iLk = add(lk.data(), sizeof(double) * L);
    const size_t iAmp = add(amp.data(), sizeof(double) * L);
    const size_t iCn2 = add(t->cn2, sizeof(double) * L);
    const size_t iSz = add(sspsz.data(), sizeof(double) * Nw);
    const size_t iNg = add(t->noiseNGS, noise ? sizeof(double) * nngs : 0);
    const size_t iXX = add(t->noiseLGSxx, noise ? sizeof(double) * Nx : 0);
    const size_t iYY = add(t->noiseLGSyy, noise ? sizeof(double) * Nx : 0);
    const size_t iXY = add(t->noiseLGSxy, noise ? sizeof(double) * Nx : 0);
    const size_t iX = add(t->X, type_mat == 4 ? sizeof(double) * Nx : 0);
    const size_t iY = add(t->Y, type_mat == 4 ? sizeof(double) * Nx : 0);
    const size_t iRs = add(rsub.data(), sizeof(int2) * rsub.size());
    const size_t iCs = add(csub.data(), sizeof(int2) * csub.size());
    const size_t iNs = add(nsub.data(), sizeof(int) * Nw);
    const size_t iLat = add(lat.place.data(), sizeof(int) * lat.place.size());
    const size_t iU0 = add(lat.u0.data(), sizeof(double) * lat.u0.size());
    const size_t iV0 = add(lat.v0.data(), sizeof(double) * lat.v0.size());
    const size_t iCls = add(cls.data(), sizeof(int) * cls.size());
    const size_t iSl = add(slots.data(), sizeof(int) * slots.size());

    MatcovArgs a;
    // Columns per wave of the evaluating kernels: as many as leave two workgroups per CU, at
    // most 8 (a workgroup's first work is its copy of the structure function's table).
    const long rblocks = pairs ? (rsub.size() + kRows - 1) / kRows : (nrows + kRows - 1) / kRows;
    const long ccount = pairs ? (long)csub.size() : ncols;
    auto cblocks = [&](int cw) { return (ccount + kWaves * cw - 1) / (kWaves * cw); };
    int cw = 8;
    while (cw > 1 && rblocks * cblocks(cw) < 512) cw /= 2;
    a.cw = cw;
    const dim3 grid((unsigned)rblocks, (unsigned)cblocks(cw));
    if (grid.y > 65535) {
        set_error("matcov_tile: too many columns for one launch");
        return MOAO_ERR_ARG;
    }
    if (int rc = structure_table_dev(&a.ftab)) return rc;

    // Tables of the library context are shared by every caller: hold the lock until the kernels
    // that read them have run.  A caller-owned buffer (one per serving slot) needs no lock.
    std::unique_lock<std::mutex> g;
    if (!tables) {
        g = std::unique_lock<std::mutex>(ctx().mu);
        tables = &ctx().matcov_tables;
    }
    const size_t W = 2 * (size_t)lat.ext - 1;
    if (int rc = tables->ensure(total, slots.size() * 3 * W * W * sizeof(double))) return rc;
    unsigned char* d = tables->dev.as<unsigned char>();
    // Staged in pinned memory (the copy is one DMA).  Every way out of here waits for the stream, so
    // the next call may rewrite the tables.
    struct Drain {
        hipStream_t s;
        ~Drain() { (void)hipStreamSynchronize(s); }
    } drain{stream};
    for (auto& p : pieces)
        if (p.src && p.bytes) std::memcpy(tables->host + p.off, p.src, p.bytes);
    MOAO_HIP_TRY(hipMemcpyAsync(d, tables->host, total, hipMemcpyHostToDevice, stream));

    a.out = d_data;
    a.lda = lda;
    a.nrows = nrows;
    a.ncols = ncols;
    a.xoffset = xoffset;
    a.yoffset = yoffset;
    a.Nlayer = L;
    a.nlgs = t->nlgs;
    a.Nx = (int)Nx;
    a.type_mat = type_mat;
    a.lgs_cst = t->lgs_cst;
    auto P = [&](size_t i) { return (const void*)(d + pieces[i].off); };
    a.rowtab = (const int*)P(iRow);
    a.coltab = (const int*)P(iCol);
    a.u = (const double*)P(iU);
    a.v = (const double*)P(iV);
    a.sspL = (const double*)P(iS);
    a.lk = (const double*)P(iLk);
    a.amp = (const double*)P(iAmp);
    a.cn2 = (const double*)P(iCn2);
    a.sspsz = (const double*)P(iSz);
    a.nNGS = (const double*)P(iNg);
    a.nxx = (const double*)P(iXX);
    a.nyy = (const double*)P(iYY);
    a.nxy = (const double*)P(iXY);
    a.X = (const double*)P(iX);
    a.Y = (const double*)P(iY);
    a.truth_nsub = (int)t->Nsubap[Nw - 1];
    a.truth_base = (int)(t->Nsubap[Nw - 1] * (Nw - 1));
    a.rsub = (const int2*)P(iRs);
    a.csub = (const int2*)P(iCs);
    a.nsub = (const int*)P(iNs);
    a.nrsub = (int)rsub.size();
    a.ncsub = (int)csub.size();
    a.lat = (const int*)P(iLat);
    a.u0 = (const double*)P(iU0);
    a.v0 = (const double*)P(iV0);
    a.cls = (const int*)P(iCls);
    a.slots = (const int*)P(iSl);
    a.ptab = (double*)(tables->space ? tables->space : d + tables->upload);
    a.Nw = Nw;
    a.ext = lat.ext;

    {
        // work = elements written (bytes = 8 x elements)
        double elems = (double)nrows * ncols;
        if (type_mat == 1 && profiling()) {
            elems = 0;
            for (int c = 0; c < ncols; ++c)
                elems += std::max(0, std::min(nrows, xoffset + nrows - (yoffset + c)));
        }
        ProfScope ps(kProfMatcov, elems, stream);
        if (!slots.empty()) {
            const dim3 tg((unsigned)((W * W + 63) / 64), (unsigned)slots.size());
            hipLaunchKernelGGL(lattice_table, tg, dim3(kWaves * 64), 0, stream, a);
        }
        if (pairs) {
            if (!slots.empty()) {
                // columns per wave: few enough that the launch fills the chip
                const long rb = (a.nrsub + 63) / 64;
                int cw = 8;
                while (cw > 1 && rb * ((a.ncsub + 4 * cw - 1) / (4 * cw)) < 1024) cw /= 2;
                hipLaunchKernelGGL(lattice_fill,
                                   dim3((unsigned)rb, (unsigned)((a.ncsub + 4 * cw - 1) / (4 * cw))),
                                   dim3(256), 0, stream, a, cw);
            }
            if (positions || slots.empty()) {
                hipLaunchKernelGGL(pair_kernel, grid, dim3(kWaves * 64), 0, stream, a);
            }
        } else if (type_mat == 4)
            hipLaunchKernelGGL(truth_kernel, grid, dim3(kWaves * 64), 0, stream, a);
        else
            hipLaunchKernelGGL(meas_kernel, grid, dim3(kWaves * 64), 0, stream, a);
    }
    MOAO_HIP_TRY(hipGetLastError());
    MOAO_HIP_TRY(hipStreamSynchronize(stream));
    return MOAO_OK;
}

}  // namespace moao

extern "C" {

int moao_hip_matcov_tile_dev(double* d_data, int nrows, int ncols, int xoffset, int yoffset,
                             int lda, const moao_tomo_view* tomo, int type_mat, void* stream) {
    if (int rc = moao::ensure_init()) return rc;
    return moao::matcov_tile_launch(d_data, nrows, ncols, xoffset, yoffset, lda, tomo, type_mat,
                                    moao::pick_stream(stream), nullptr);
}

int moao_hip_matcov_tile(double* data, int nrows, int ncols, int xoffset, int yoffset, int lda,
                         const moao_tomo_view* tomo, int type_mat) {
    if (int rc = moao::ensure_init()) return rc;
    if (!data || nrows < 0 || ncols < 0 || lda < std::max(1, nrows)) {
        moao::set_error("matcov_tile: invalid host buffer");
        return MOAO_ERR_ARG;
    }
    if (nrows == 0 || ncols == 0) return MOAO_OK;
    moao::Context& c = moao::ctx();
    hipStream_t s = c.stream;
    const size_t span = ((size_t)(ncols - 1) * lda + nrows) * sizeof(double);
    std::lock_guard<std::mutex> g(c.mu);
    if (int rc = c.host_stage.ensure(span)) return rc;
    double* d = c.host_stage.as<double>();
    // Type 1 leaves the strictly-upper part untouched and lda may leave gaps between columns:
    // start from the caller's contents so the copy back preserves them.
    if (type_mat == 1 || lda != nrows)
        MOAO_HIP_TRY(hipMemcpyAsync(d, data, span, hipMemcpyHostToDevice, s));
    // c.mu is held: hand the context's table buffer over explicitly
    int rc = moao::matcov_tile_launch(d, nrows, ncols, xoffset, yoffset, lda, tomo, type_mat, s,
                                      &c.matcov_tables);
    if (rc) return rc;
    MOAO_HIP_TRY(hipMemcpyAsync(data, d, span, hipMemcpyDeviceToHost, s));
    MOAO_HIP_TRY(hipStreamSynchronize(s));
    return MOAO_OK;
}

}  // extern "C"
