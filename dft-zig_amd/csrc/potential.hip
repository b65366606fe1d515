// Device-resident SCF grid state: density, Hartree + LDA-PZ or PBE potential, energies and
// potential mixing (linear, then Pulay/DIIS), so an SCF iteration keeps rho(r) and V(r) in HBM.
//
// Follows (paths relative to the dft-zig source tree):
//   Hartree V_H(G) = 8 pi rho(G) / G^2, G = 0 dropped              src/features/scf/potential.zig:34-44
//   LDA-PZ energy density and potential (Ry)                       src/features/xc/xc.zig:195-210, 344-384
//   PBE (Ry): exchange, correlation H(t^2, A) on PW92               src/features/xc/xc.zig:213-342
//   GGA fields: grad n = IFFT(i G n(G)), b = df/d|grad n|^2 grad n,
//   v_xc = df/dn - 2 div b, div by i G . b(G), real parts kept     src/features/scf/xc_fields.zig:87-140, 306-375
//   local_r = V_ion + V_Hxc on the FFT-order grid                   src/features/scf/potential.zig:320-334
//   linear potential mixing V <- V + beta (V_out - V)              src/features/scf/mixing.zig:10-18
//   Pulay on (V_in, R = V_out - V_in), history h, from iteration s  src/features/scf/mixing.zig:183-234,
//                                                                   src/features/scf/scf.zig:147-188
//   RMS density change                                              src/features/scf/util.zig:17-24
// The Pulay overlaps are taken in real space divided by N (the reference's G-space norm by
// Parseval) and the small system is scaled by its largest diagonal before elimination; a
// singular system keeps only the newest pair and takes a linear step (the reference would
// average the whole history).
#include <algorithm>
#include <cmath>
#include <type_traits>
#include <vector>

#include "fft_lds.h"
#include "potential.h"

namespace dzhip {

namespace {

constexpr int kRedThreads = 256;

// |G|^2 on the FFT-order grid (index x + nx (y + ny z), wrapped frequencies; b rows = b1, b2, b3), and
// the Hartree kernel 8 pi / G^2 (0 at G = 0), the mean of its values at an index and at the mirrored
// one (they differ at an even axis' Nyquist frequencies when the cell is not orthogonal).
__device__ __forceinline__ double hartree_factor(double g2) { return g2 > 1e-12 ? 8.0 * M_PI / g2 : 0.0; }
__global__ void k_g2(double* __restrict__ g2, double* __restrict__ kern, int nx, int ny, int nz, double3 b1, double3 b2,
                     double3 b3) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t n = (size_t)nx * ny * nz;
    if (i >= n) return;
    const int x = (int)(i % nx), y = (int)((i / nx) % ny), z = (int)(i / ((size_t)nx * ny));
    auto norm2 = [&](int ix, int iy, int iz) {
        const int fx = ix <= (nx - 1) / 2 ? ix : ix - nx;
        const int fy = iy <= (ny - 1) / 2 ? iy : iy - ny;
        const int fz = iz <= (nz - 1) / 2 ? iz : iz - nz;
        const double gx = fx * b1.x + fy * b2.x + fz * b3.x;
        const double gy = fx * b1.y + fy * b2.y + fz * b3.y;
        const double gz = fx * b1.z + fy * b2.z + fz * b3.z;
        return gx * gx + gy * gy + gz * gz;
    };
    const double g = norm2(x, y, z);
    g2[i] = g;
    kern[i] = 0.5 * (hartree_factor(g) +
                     hartree_factor(norm2(x ? nx - x : 0, y ? ny - y : 0, z ? nz - z : 0)));
}

__global__ void k_real_to_complex(const double* __restrict__ in, double2* __restrict__ out, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = make_double2(in[i], 0.0);
}

__device__ inline void lda_pz(double n, double* f, double* v) {
    if (!(n > 1e-12)) {
        *f = 0.0;
        *v = 0.0;
        return;
    }
    const double cbrt_n = cbrt(n);
    const double cx = -0.75 * cbrt(3.0 / M_PI);
    const double rs = cbrt(3.0 / (4.0 * M_PI * n));
    double ec, vc;
    if (rs < 1.0) {
        const double ln = log(rs);
        ec = 0.0311 * ln - 0.048 + 0.0020 * rs * ln - 0.0116 * rs;
        vc = ec - (rs / 3.0) * (0.0311 / rs + 0.0020 * ln + 0.0020 - 0.0116);
    } else {
        const double sq = sqrt(rs);
        const double den = 1.0 + 1.0529 * sq + 0.3334 * rs;
        ec = -0.1423 / den;
        vc = ec - (rs / 3.0) * (0.1423 * (0.5 * 1.0529 / sq + 0.3334) / (den * den));
    }
    *f = 2.0 * n * (cx * cbrt_n + ec);
    *v = 2.0 * (4.0 / 3.0 * cx * cbrt_n + vc);
}

// PW92 unpolarised correlation (Ha): eps, d eps / d rs, v_c = eps - rs/3 d eps/d rs.
__device__ inline void pw92(double rs, double* eps, double* deps, double* vc) {
    constexpr double a = 0.031091, a1 = 0.21370, b1 = 7.5957, b2 = 3.5876, b3 = 1.6382, b4 = 0.49294;
    const double sr = sqrt(rs);
    const double f = b1 * sr + b2 * rs + b3 * rs * sr + b4 * rs * rs;
    const double g = 1.0 + 1.0 / (2.0 * a * f);
    const double lg = log(g);
    const double df = 0.5 * b1 / sr + b2 + 1.5 * b3 * sr + 2.0 * b4 * rs;
    const double dlg = -(1.0 / (2.0 * a * f * f * g)) * df;
    *eps = -2.0 * a * (1.0 + a1 * rs) * lg;
    *deps = -2.0 * a * (a1 * lg + (1.0 + a1 * rs) * dlg);
    *vc = *eps - (rs / 3.0) * *deps;
}

// PBE at density n and g2 = |grad n|^2: f, df/dn, df/dg2 (Ry); zero below n = 1e-12.
__device__ inline void pbe(double n, double g2, double* f, double* fn, double* fg) {
    if (!(n > 1e-12)) {
        *f = *fn = *fg = 0.0;
        return;
    }
    // Exchange: F_x = 1 + kappa - kappa / (1 + mu s^2 / kappa).
    constexpr double mu = 0.2195149727645171, kappa = 0.804;
    const double cx = -0.75 * cbrt(3.0 / M_PI);
    const double n13 = cbrt(n);
    const double ex0 = n * cx * n13;
    const double kf = cbrt(3.0 * M_PI * M_PI * n);
    const double den_x = 4.0 * kf * kf * n * n;
    const double s2 = g2 > 0.0 ? g2 / den_x : 0.0;
    const double t = 1.0 + mu * s2 / kappa;
    const double fx = 1.0 + kappa - kappa / t;
    const double dfx = mu / (t * t);
    const double fx_n = 4.0 / 3.0 * cx * n13 * fx + ex0 * dfx * (-8.0 / 3.0 * s2 / n);
    const double fx_g = ex0 * dfx / den_x;
    // Correlation: H = gamma ln(1 + (beta/gamma) t^2 (1 + A t^2) / (1 + A t^2 + A^2 t^4)).
    constexpr double beta = 0.06672455060314922, gamma = 0.031090690869654895, bg = beta / gamma;
    const double rs = cbrt(3.0 / (4.0 * M_PI * n));
    double ec, deps, vc;
    pw92(rs, &ec, &deps, &vc);
    const double deps_dn = deps * (-rs / (3.0 * n));
    const double den_c = 4.0 * (4.0 * kf / M_PI) * n * n;
    const double t2 = g2 > 0.0 ? g2 / den_c : 0.0;
    const double x = bg * t2;
    const double u = exp(-ec / gamma);
    const double um = u - 1.0;
    const bool big = fabs(um) > 1e-12;
    const double A = big ? bg / um : 0.0;
    const double y = A * t2;
    const double d2 = 1.0 + y + y * y;
    const double q = (1.0 + y) / d2;
    const double arg = 1.0 + x * q;
    const bool pos = arg > 0.0;
    const double H = pos ? gamma * log(arg) : 0.0;
    const double dq = -A * y * (2.0 + y) / (d2 * d2);
    const double dH_dt2 = pos ? gamma * (bg * q + x * dq) / arg : 0.0;
    const double dH_dA = pos ? -gamma * x * t2 * y * (2.0 + y) / (arg * d2 * d2) : 0.0;
    const double dA_dn = big ? bg * u / (gamma * um * um) * deps_dn : 0.0;
    const double dH_dn = dH_dt2 * (-7.0 / 3.0 * t2 / n) + dH_dA * dA_dn;
    *f = 2.0 * (ex0 * fx + n * (ec + H));
    *fn = 2.0 * (fx_n + vc + H + n * dH_dn);
    *fg = 2.0 * (fx_g + n * dH_dt2 / den_c);
}

// ----------------------------------------------------------------- V_H + V_xc on the grid
// The density's transforms with everything point-wise folded into their passes.  An xy-pass holds one
// plane of k_z in LDS, transforms forward, multiplies in G space and transforms back; a z-pass holds a
// few columns of one y, back to r space, evaluates the functional and transforms forward (the columns
// are many workgroups, and the functional is what costs there).  Real fields share complex transforms
// in pairs: with i G_c taken as zero at an even axis' Nyquist frequency (whose term is imaginary in r
// space, where the real part is kept) the derivative of a real field is real, so
//   d_x n + i d_y n = IFFT[(-G_y + i G_x) n(G)],   d_z n = IFFT[i G_z n(G)],   V_H = IFFT[K n(G)],
//   div b = Re IFFT[(G_y + i G_x) FFT(b_x + i b_y) + i G_z FFT(b_z)],
// K the Hartree kernel 8 pi / G^2 (the mean over +G and -G, which is what the real part sees).  V_H is no
// field's partner: a transform rounds by the larger of a pair, and V_H would take d_z n's rounding times
// 8 pi / G_min^2 (1e-13 Ry at 60 bohr, 4e-15 alone).  PBE: five launches and seven transforms where there
// were some forty and ten, which launches bounded: 248 -> 103 us at 30 x 30 x 30 (101 with V_H as d_z n's
// partner).  There the xy-passes take 19 and 16 us, on 30 CUs (barriers of their short lines bound them),
// k_xc_z 10, k_rho_z 7, k_div_z 5, the rest launch gaps and the copies around them.  LDA: three launches.
struct GridAxes {
    FftAxis ax, ay, az;
    const double2* tw;
    const int* perm;
    double3 b1, b2, b3;
};

// Frequency of index i on an axis of n points, zero at an even axis' Nyquist index (derivatives).
__device__ __forceinline__ double deriv_freq(int i, int n) {
    return 2 * i == n ? 0.0 : (double)(i <= (n - 1) / 2 ? i : i - n);
}
__device__ __forceinline__ double3 deriv_g(int x, int y, int z, const GridAxes& g) {
    const double fx = deriv_freq(x, g.ax.n), fy = deriv_freq(y, g.ay.n), fz = deriv_freq(z, g.az.n);
    return make_double3(fx * g.b1.x + fy * g.b2.x + fz * g.b3.x, fx * g.b1.y + fy * g.b2.y + fz * g.b3.y,
                        fx * g.b1.z + fy * g.b2.z + fz * g.b3.z);
}

// xy-pass, out and back.  HARTREE: w1 = K w1.  GRADIENT: w1 = (-G_y + i G_x) w1, w2 = i G_z w1 and w3 =
// K w1.  DIVERGENCE: w1 = (G_y + i G_x) w1 + i G_z w2.  All times 1/N.  KP: points per thread.  F: planes
// in LDS; the fields that go the same way lie side by side there, rows interleaved, and share a
// transform's barriers (F = 3 and 2), or take turns where so many planes do not fit (1).
enum { kHartree = 0, kGradient = 1, kDivergence = 2 };
constexpr int gridxy_fields(int kind) { return kind == kGradient ? 3 : kind == kDivergence ? 2 : 1; }
template <int KIND, int KP, int F>
__global__ __launch_bounds__(512) void k_gridxy(double2* __restrict__ w1, double2* __restrict__ w2, double2* __restrict__ w3,
                                                const double* __restrict__ kern, double scale, GridAxes g) {
    extern __shared__ double2 lds[];
    const int nx = g.ax.n, ny = g.ay.n, half = nx + 1, pitch = F * half, tid = threadIdx.x, nthr = blockDim.x, np = nx * ny;
    double2 *twx = lds + pitch * ny, *twy = twx + nx;
    load_twiddles(twx, g.tw + g.ax.tw_off, nx, tid, nthr);
    load_twiddles(twy, g.tw + g.ay.tw_off, ny, tid, nthr);
    const size_t off = (size_t)blockIdx.x * np;
    const int *px = g.perm + g.ax.perm_off, *py = g.perm + g.ay.perm_off;
    const unsigned mx = div_magic(nx);
    // Natural order in, digit-reversed out; fields: planes in use (one or F).
    auto lines = [&](auto sign, int fields) {
        constexpr int S = decltype(sign)::value;
        lds_fft_lines<double, double2, false, S>(lds, g.ax, twx, LineSet{fields == F ? F * ny : ny, 1, fields == F ? half : pitch, nullptr},
                                                 tid, nthr);
        lds_fft_lines<double, double2, false, S>(lds, g.ay, twy, LineSet{fields > 1 ? pitch : nx, pitch, 1, nullptr}, tid, nthr);
    };
    const std::integral_constant<int, -1> fwd;
    const std::integral_constant<int, 1> inv;
    auto load = [&](const double2* src, int shift) {
        for (int i = tid; i < np; i += nthr) {
            const int y = fdiv(i, nx, mx);
            lds[i - y * nx + pitch * y + shift] = src[off + i];
        }
    };
    auto store = [&](double2* dst, int shift) {
        for (int i = tid; i < np; i += nthr) {
            const int y = fdiv(i, nx, mx);
            dst[off + i] = lds[px[i - y * nx] + pitch * py[y] + shift];
        }
    };
    double2 v[KP];  // this thread's points: spectrum of w1 (divergence: the sum's)
    load(w1, 0);
    if constexpr (KIND == kDivergence && F == 2) load(w2, half);
    __syncthreads();
    lines(fwd, KIND == kDivergence ? F : 1);
    auto take = [&]() {
#pragma unroll
        for (int k = 0; k < KP; ++k) {
            const int i = tid + k * nthr, y = fdiv(i, nx, mx);
            if (i < np) v[k] = lds[px[i - y * nx] + pitch * py[y]];
        }
        __syncthreads();
    };
    if constexpr (KIND != kDivergence || F == 1) take();
    if constexpr (KIND == kDivergence) {
        if constexpr (F == 1) {
            load(w2, 0);
            __syncthreads();
            lines(fwd, 1);
        }
#pragma unroll
        for (int k = 0; k < KP; ++k) {
            const int i = tid + k * nthr;
            if (i >= np) continue;
            const int y = fdiv(i, nx, mx), x = i - y * nx;
            const double2* l = lds + px[x] + pitch * py[y];
            const double3 q = deriv_g(x, y, blockIdx.x, g);
            const double2 p = F == 2 ? l[0] : v[k], r = F == 2 ? l[half] : l[0];
            const double2 a = make_double2(p.x * scale, p.y * scale), b = make_double2(r.x * scale, r.y * scale);
            v[k] = make_double2(q.y * a.x - q.x * a.y - q.z * b.y, q.x * a.x + q.y * a.y + q.z * b.x);
        }
        __syncthreads();
    }
    // Field f of the point's spectrum at its place in plane t.
    auto put = [&](int f, int t) {
#pragma unroll
        for (int k = 0; k < KP; ++k) {
            const int i = tid + k * nthr;
            if (i >= np) continue;
            const int y = fdiv(i, nx, mx), x = i - y * nx;
            double2 u = v[k];
            if (KIND == kHartree || (KIND == kGradient && f == 2)) {
                const double h = kern[off + i] * scale;
                u = make_double2(h * u.x, h * u.y);
            } else if constexpr (KIND == kGradient) {
                const double3 q = deriv_g(x, y, blockIdx.x, g);
                u = make_double2(u.x * scale, u.y * scale);
                u = f == 0 ? make_double2(-q.y * u.x - q.x * u.y, q.x * u.x - q.y * u.y) : make_double2(-q.z * u.y, q.z * u.x);
            }
            lds[x + pitch * y + half * t] = u;
        }
    };
    if constexpr (KIND == kGradient) {
        double2* const dst[3] = {w1, w2, w3};
        if constexpr (F == 3) {
#pragma unroll
            for (int f = 0; f < 3; ++f) put(f, f);
            __syncthreads();
            lines(inv, 3);
#pragma unroll
            for (int f = 0; f < 3; ++f) store(dst[f], f * half);
        } else {
#pragma unroll
            for (int f = 0; f < 3; ++f) {
                put(f, 0);
                __syncthreads();
                lines(inv, 1);
                store(dst[f], 0);
                __syncthreads();
            }
        }
    } else {
        put(0, 0);
        __syncthreads();
        lines(inv, 1);
        store(w1, 0);
    }
}

// Columns of one z-pass workgroup (one y): kZCols of each field, side by side.  At the longest axis (256)
// the tile of the GGA's three fields is 104 KiB.
constexpr int kZCols = 8, kZThreads = 256, kZPitch = 2 * kZCols + 1, kZPitchGga = 3 * kZCols + 1;
struct ZCols {
    int nx, y, x0, cols, cnt, ny;
    __device__ __forceinline__ ZCols(const GridAxes& g)
        : nx(g.ax.n), y(blockIdx.y), x0(blockIdx.x * kZCols), cols(min(kZCols, g.ax.n - (int)blockIdx.x * kZCols)),
          cnt(kZCols * g.az.n), ny(g.ay.n) {}
    __device__ __forceinline__ bool in(int i) const { return i % kZCols < cols; }
    __device__ __forceinline__ size_t at(int i) const {
        return (size_t)(x0 + i % kZCols) + (size_t)nx * (y + (size_t)ny * (i / kZCols));
    }
};

// z-pass of the density, forward: w = FFT_z(rho).
__global__ __launch_bounds__(kZThreads) void k_rho_z(const double* __restrict__ rho, double2* __restrict__ w, GridAxes g) {
    extern __shared__ double2 lds[];
    const ZCols c(g);
    const int nz = g.az.n, tid = threadIdx.x;
    const int* pz = g.perm + g.az.perm_off;
    double2* tw = lds + kZPitch * nz;
    load_twiddles(tw, g.tw + g.az.tw_off, nz, tid, kZThreads);
    for (int i = tid; i < c.cnt; i += kZThreads)
        lds[i % kZCols + kZPitch * (i / kZCols)] = make_double2(c.in(i) ? rho[c.at(i)] : 0.0, 0.0);
    __syncthreads();
    lds_fft_lines<double, double2, false, -1>(lds, g.az, tw, LineSet{kZCols, kZPitch, 1, nullptr}, tid, kZThreads);
    for (int i = tid; i < c.cnt; i += kZThreads)
        if (c.in(i)) w[c.at(i)] = lds[i % kZCols + kZPitch * pz[i / kZCols]];
}

// z-pass in r space: V_H (GGA: in w3, the gradient in w1 and w2), the functional at every point, the
// workgroup's sums [V_H rho, f_xc, v_in rho, (rho - rho_in)^2], and, GGA, b's z-transforms back into w1
// and w2.  vout = V_H + df/dn (LDA: V_H + v_xc).
template <bool GGA>
__global__ __launch_bounds__(kZThreads) void k_xc_z(double2* __restrict__ w1, double2* __restrict__ w2,
                                                    const double2* __restrict__ w3,
                                                    const double* __restrict__ rho, const double* __restrict__ rho_in,
                                                    const double* __restrict__ vin, double* __restrict__ vout,
                                                    double* __restrict__ part, GridAxes g) {
    extern __shared__ double2 lds[];
    __shared__ double red[4][kZThreads / 64];
    constexpr int P = GGA ? kZPitchGga : kZPitch;
    const ZCols c(g);
    const int nz = g.az.n, tid = threadIdx.x;
    const int* pz = g.perm + g.az.perm_off;
    double2* tw = lds + P * nz;
    load_twiddles(tw, g.tw + g.az.tw_off, nz, tid, kZThreads);
    for (int i = tid; i < c.cnt; i += kZThreads) {
        double2* l = lds + i % kZCols + P * pz[i / kZCols];
        const bool in = c.in(i);
        l[0] = in ? w1[c.at(i)] : make_double2(0.0, 0.0);
        if constexpr (GGA) {
            l[kZCols] = in ? w2[c.at(i)] : make_double2(0.0, 0.0);
            l[2 * kZCols] = in ? w3[c.at(i)] : make_double2(0.0, 0.0);
        }
    }
    __syncthreads();
    lds_fft_lines<double, double2, true, 1>(lds, g.az, tw, LineSet{GGA ? 3 * kZCols : kZCols, P, 1, nullptr}, tid,
                                            kZThreads);
    double sums[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
    for (int i = tid; i < c.cnt; i += kZThreads) {
        if (!c.in(i)) continue;
        double2* l = lds + i % kZCols + P * (i / kZCols);
        const size_t at = c.at(i);
        const double r = rho[at];
        double f, v, h;
        if constexpr (GGA) {
            const double gx = l[0].x, gy = l[0].y, gz = l[kZCols].x;
            double fg;
            h = l[2 * kZCols].x;
            pbe(r, gx * gx + gy * gy + gz * gz, &f, &v, &fg);
            l[0] = make_double2(fg * gx, fg * gy);
            l[kZCols] = make_double2(fg * gz, 0.0);
        } else {
            h = l[0].x;
            lda_pz(r, &f, &v);
        }
        vout[at] = h + v;
        const double d = r - rho_in[at];
        sums[0] += h * r;
        sums[1] += f;
        sums[2] += vin[at] * r;
        sums[3] += d * d;
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) sums[k] += __shfl_xor(sums[k], o, 64);
        if ((tid & 63) == 0) red[k][tid >> 6] = sums[k];
    }
    __syncthreads();
    if (tid < 4) {
        double s = 0.0;
        for (int q = 0; q < kZThreads / 64; ++q) s += red[tid][q];
        part[4 * (blockIdx.x + gridDim.x * blockIdx.y) + tid] = s;
    }
    if constexpr (GGA) {
        lds_fft_lines<double, double2, false, -1>(lds, g.az, tw, LineSet{2 * kZCols, P, 1, nullptr}, tid, kZThreads);
        for (int i = tid; i < c.cnt; i += kZThreads) {
            if (!c.in(i)) continue;
            const double2* l = lds + i % kZCols + P * pz[i / kZCols];
            w1[c.at(i)] = l[0];
            w2[c.at(i)] = l[kZCols];
        }
    }
}

// z-pass of the divergence: vout -= 2 Re(div b).
__global__ __launch_bounds__(kZThreads) void k_div_z(const double2* __restrict__ w, double* __restrict__ vout, GridAxes g) {
    extern __shared__ double2 lds[];
    const ZCols c(g);
    const int nz = g.az.n, tid = threadIdx.x;
    const int* pz = g.perm + g.az.perm_off;
    double2* tw = lds + kZPitch * nz;
    load_twiddles(tw, g.tw + g.az.tw_off, nz, tid, kZThreads);
    for (int i = tid; i < c.cnt; i += kZThreads)
        lds[i % kZCols + kZPitch * pz[i / kZCols]] = c.in(i) ? w[c.at(i)] : make_double2(0.0, 0.0);
    __syncthreads();
    lds_fft_lines<double, double2, true, 1>(lds, g.az, tw, LineSet{kZCols, kZPitch, 1, nullptr}, tid, kZThreads);
    for (int i = tid; i < c.cnt; i += kZThreads)
        if (c.in(i)) vout[c.at(i)] -= 2.0 * lds[i % kZCols + kZPitch * (i / kZCols)].x;
}

// part[b] = sum over block b of a[i] * c[i] (fixed order, reduced on the host).
__global__ void k_dot(const double* __restrict__ a, const double* __restrict__ c, double* __restrict__ part,
                      size_t n) {
    __shared__ double red[kRedThreads];
    double s = 0.0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        s += a[i] * c[i];
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

__global__ void k_fill(double* __restrict__ a, double v, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) a[i] = v;
}

// out = a + s b (out may alias a)
__global__ void k_axpy_to(const double* a, const double* __restrict__ b, double s, double* out, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = a[i] + s * b[i];
}

// r = vout - vin
__global__ void k_sub(const double* __restrict__ a, const double* __restrict__ b, double* __restrict__ out, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = a[i] - b[i];
}

// w(G) *= P(G), P = (l^2 G^2 + 1/eps) / (l^2 G^2 + 1), P(0) = 1/eps (mixing.zig:309-338); the
// forward transform is unnormalised and the inverse carries the 1/N, so only P is applied.
__global__ void k_dielectric(double2* __restrict__ w, const double* __restrict__ g2, double inv_eps, double l2,
                             size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double g = g2[i];
    const double x = l2 * g;
    const double p = g < 1e-12 ? inv_eps : (x + inv_eps) / (x + 1.0);
    w[i] = make_double2(w[i].x * p, w[i].y * p);
}

// out = Re(w)
__global__ void k_real_part(const double2* __restrict__ w, double* __restrict__ out, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = w[i].x;
}

// v = sum_j c_j (hv[slot_j] + beta hr[slot_j])
__global__ void k_pulay_combine(const double* __restrict__ hv, const double* __restrict__ hr, const int* __restrict__ slot,
                                const double* __restrict__ c, int m, double beta, double* __restrict__ v, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double acc = 0.0;
    for (int j = 0; j < m; ++j) {
        const size_t o = (size_t)slot[j] * n + i;
        acc += c[j] * (hv[o] + beta * hr[o]);
    }
    v[i] = acc;
}

unsigned grid_blocks(size_t n) { return (unsigned)((n + 255) / 256); }
constexpr int kRedBlocks = 512;

}  // namespace

double ScfGrid::reduce(const double* part_dev, int nblocks, int stride, int comp) {
    std::vector<double> h((size_t)nblocks * stride);
    DZ_HIP(hipMemcpyAsync(h.data(), part_dev, h.size() * sizeof(double), hipMemcpyDeviceToHost, stream()));
    DZ_HIP(hipStreamSynchronize(stream()));
    double s = 0.0;
    for (int i = 0; i < nblocks; ++i) s += h[(size_t)i * stride + comp];
    return s;
}

double ScfGrid::dot(const double* a, const double* c) {
    part.ensure(kRedBlocks * sizeof(double));
    hipLaunchKernelGGL(k_dot, dim3(kRedBlocks), dim3(kRedThreads), 0, stream(), a, c, part.as<double>(), n);
    DZ_HIP(hipGetLastError());
    return reduce(part.as<double>(), kRedBlocks, 1, 0);
}

namespace {
// Threads and points per thread of an xy-pass by the plane's points (one tile in LDS: at most 10,240; two:
// 5,120; three: 3,413, and always up to 1,024).
template <int KIND>
void launch_gridxy(int nx, int ny, int nz, hipStream_t s, double2* w1, double2* w2, double2* w3, const double* kern,
                   double scale, const GridAxes& g) {
    constexpr int F = gridxy_fields(KIND);
    const int np = nx * ny;
    size_t lds = fft_xy_lds_bytes(nx, ny, sizeof(double2));
    const size_t all = lds + (size_t)(F - 1) * (nx + 1) * ny * sizeof(double2);
    const bool together = F > 1 && all <= kMaxLdsBytes;
    if (together) lds = all;
    auto* fn = np <= 1024   ? k_gridxy<KIND, 4, F>
               : together   ? k_gridxy<KIND, F == 3 ? 8 : 12, F>
               : np <= 6144 ? k_gridxy<KIND, 12, 1>
                            : k_gridxy<KIND, 20, 1>;
    set_max_dynamic_lds((const void*)fn, lds);
    hipLaunchKernelGGL(fn, dim3((unsigned)nz), dim3(np <= 1024 ? 256 : 512), lds, s, w1, w2, w3, kern, scale, g);
    DZ_HIP(hipGetLastError());
}
}  // namespace

void ScfGrid::hxc(const double* rho, const double* rho_ref, const double* vin, double* vout, double* out) {
    hipStream_t s = stream();
    const bool gga = xc == DZHIP_XC_PBE;
    const GridAxes g{tab.ax[0], tab.ax[1], tab.ax[2], tab.tw64, tab.perm, recip_rows[0], recip_rows[1], recip_rows[2]};
    // The tiles of the plan's own passes bound the grids taken.
    DZ_REQUIRE(fft_xy_lds_bytes(nx, ny, sizeof(double2)) <= kMaxLdsBytes &&
                   fft_z_lds_bytes(nx, nz, sizeof(double2)) <= kMaxLdsBytes,
               DZHIP_ERR_HIP, "SCF grid: plane too large for the FFT kernels' LDS");
    double2 *w1 = work.as<double2>(), *w2 = work2.as<double2>(), *w3 = work3.as<double2>();
    double *kern = hartree.as<double>(), *sums = part.as<double>();
    const double scale = 1.0 / (double)n;
    const dim3 gz((unsigned)((nx + kZCols - 1) / kZCols), (unsigned)ny);
    const size_t ldsz = (size_t)(kZPitch + 1) * nz * sizeof(double2);
    set_max_dynamic_lds((const void*)k_rho_z, ldsz);
    hipLaunchKernelGGL(k_rho_z, gz, dim3(kZThreads), ldsz, s, rho, w1, g);
    DZ_HIP(hipGetLastError());
    if (gga) {
        launch_gridxy<kGradient>(nx, ny, nz, s, w1, w2, w3, kern, scale, g);
        const size_t ldsg = (size_t)(kZPitchGga + 1) * nz * sizeof(double2);
        set_max_dynamic_lds((const void*)k_xc_z<true>, ldsg);
        hipLaunchKernelGGL(k_xc_z<true>, gz, dim3(kZThreads), ldsg, s, w1, w2, w3, rho, rho_ref, vin, vout, sums, g);
        DZ_HIP(hipGetLastError());
        launch_gridxy<kDivergence>(nx, ny, nz, s, w1, w2, w3, kern, scale, g);
        set_max_dynamic_lds((const void*)k_div_z, ldsz);
        hipLaunchKernelGGL(k_div_z, gz, dim3(kZThreads), ldsz, s, w1, vout, g);
        DZ_HIP(hipGetLastError());
    } else {
        launch_gridxy<kHartree>(nx, ny, nz, s, w1, w2, w3, kern, scale, g);
        set_max_dynamic_lds((const void*)k_xc_z<false>, ldsz);
        hipLaunchKernelGGL(k_xc_z<false>, gz, dim3(kZThreads), ldsz, s, w1, w2, w3, rho, rho_ref, vin, vout, sums, g);
        DZ_HIP(hipGetLastError());
    }
    if (!out) return;
    const size_t nparts = (size_t)gz.x * gz.y;
    std::vector<double> h(nparts * 4);
    DZ_HIP(hipMemcpyAsync(h.data(), part.ptr, h.size() * sizeof(double), hipMemcpyDeviceToHost, s));
    DZ_HIP(hipStreamSynchronize(s));
    double t[4] = {0, 0, 0, 0};
    for (size_t i = 0; i < nparts; ++i)
        for (int c = 0; c < 4; ++c) t[c] += h[4 * i + c];
    const double dv = volume / (double)n;
    out[0] = 0.5 * t[0] * dv;
    out[1] = t[1] * dv;
    out[2] = t[2] * dv;
    out[3] = std::sqrt(t[3] / (double)n);
}

ScfGrid* scf_grid_create(Context* ctx, int nx, int ny, int nz, const double* recip, double volume, int history) {
    auto* g = new ScfGrid();
    try {
        g->ctx = ctx;
        g->nx = nx;
        g->ny = ny;
        g->nz = nz;
        g->n = (size_t)nx * ny * nz;
        g->volume = volume;
        g->hist_cap = history;
        for (int r = 0; r < 3; ++r) g->recip_rows[r] = make_double3(recip[3 * r], recip[3 * r + 1], recip[3 * r + 2]);
        g->tab.build(nx, ny, nz);
        const size_t n = g->n;
        g->g2.ensure(n * sizeof(double));
        g->hartree.ensure(n * sizeof(double));
        g->work.ensure(n * sizeof(double2));
        g->part.ensure(4 * std::max<size_t>((size_t)ny * ((nx + kZCols - 1) / kZCols), kRedBlocks) * sizeof(double));
        DevBuf* bufs[] = {&g->rho_in, &g->rho_out, &g->v_in, &g->v_out, &g->v_ion, &g->local};
        for (DevBuf* b : bufs) b->ensure(n * sizeof(double));
        if (history > 0) {
            g->hv.ensure((size_t)history * n * sizeof(double));
            g->hr.ensure((size_t)history * n * sizeof(double));
            g->slots.ensure(history * sizeof(int));
            g->coef.ensure(history * sizeof(double));
        }
        g->b.assign(std::max(history, 1), std::vector<double>(std::max(history, 1), 0.0));
        hipStream_t s = g->stream();
        hipLaunchKernelGGL(k_g2, dim3(grid_blocks(n)), dim3(256), 0, s, g->g2.as<double>(), g->hartree.as<double>(), nx, ny, nz,
                           make_double3(recip[0], recip[1], recip[2]), make_double3(recip[3], recip[4], recip[5]),
                           make_double3(recip[6], recip[7], recip[8]));
        DZ_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_fill, dim3(grid_blocks(n)), dim3(256), 0, s, g->v_ion.as<double>(), 0.0, n);
        DZ_HIP(hipGetLastError());
        DZ_HIP(hipStreamSynchronize(s));
    } catch (...) {
        scf_grid_destroy(g);
        throw;
    }
    return g;
}

void scf_grid_destroy(ScfGrid* g) {
    if (!g) return;
    DevBuf* bufs[] = {&g->g2, &g->work, &g->rho_in, &g->rho_out, &g->v_in, &g->v_out, &g->v_ion, &g->local,
                      &g->part, &g->hv, &g->hr, &g->slots, &g->coef, &g->work2, &g->work3, &g->hartree};
    for (DevBuf* b : bufs) b->release();
    g->tab.release();
    delete g;
}

void scf_grid_init(ScfGrid& g, double nelec, const double* rho_host) {
    hipStream_t s = g.stream();
    if (rho_host) {
        DZ_HIP(hipMemcpyAsync(g.rho_in.ptr, rho_host, g.n * sizeof(double), hipMemcpyHostToDevice, s));
    } else {
        hipLaunchKernelGGL(k_fill, dim3(grid_blocks(g.n)), dim3(256), 0, s, g.rho_in.as<double>(), nelec / g.volume, g.n);
        DZ_HIP(hipGetLastError());
    }
    // v_in = V_Hxc[rho_in]; the reference arguments for rho_ref/vin only feed the sums, not read here.
    g.hxc(g.rho_in.as<double>(), g.rho_in.as<double>(), g.rho_in.as<double>(), g.v_in.as<double>(), nullptr);
    g.order.clear();
    hipLaunchKernelGGL(k_fill, dim3(grid_blocks(g.n)), dim3(256), 0, s, g.rho_out.as<double>(), 0.0, g.n);
    DZ_HIP(hipGetLastError());
    DZ_HIP(hipStreamSynchronize(s));
}

void scf_grid_add(ScfGrid& g, const double* rho_k) {
    hipLaunchKernelGGL(k_axpy_to, dim3(grid_blocks(g.n)), dim3(256), 0, g.stream(), g.rho_out.as<double>(), rho_k, 1.0,
                       g.rho_out.as<double>(), g.n);
    DZ_HIP(hipGetLastError());
}

void scf_grid_local(ScfGrid& g) {
    hipLaunchKernelGGL(k_axpy_to, dim3(grid_blocks(g.n)), dim3(256), 0, g.stream(), g.v_ion.as<double>(),
                       g.v_in.as<double>(), 1.0, g.local.as<double>(), g.n);
    DZ_HIP(hipGetLastError());
}

// After the k-point densities are in rho_out: V_out, energies, drho; rho_in <- rho_out, rho_out <- 0.
void scf_grid_hxc(ScfGrid& g, double out[4]) {
    g.hxc(g.rho_out.as<double>(), g.rho_in.as<double>(), g.v_in.as<double>(), g.v_out.as<double>(), out);
    hipStream_t s = g.stream();
    DZ_HIP(hipMemcpyAsync(g.rho_in.ptr, g.rho_out.ptr, g.n * sizeof(double), hipMemcpyDeviceToDevice, s));
    hipLaunchKernelGGL(k_fill, dim3(grid_blocks(g.n)), dim3(256), 0, s, g.rho_out.as<double>(), 0.0, g.n);
    DZ_HIP(hipGetLastError());
}

void scf_grid_mix(ScfGrid& g, double beta, int pulay) {
    hipStream_t s = g.stream();
    const size_t n = g.n;
    if (!pulay || g.hist_cap <= 0) {
        // v_in += beta (v_out - v_in)
        hipLaunchKernelGGL(k_sub, dim3(grid_blocks(n)), dim3(256), 0, s, g.v_out.as<double>(), g.v_in.as<double>(),
                           g.work.as<double>(), n);
        DZ_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_axpy_to, dim3(grid_blocks(n)), dim3(256), 0, s, g.v_in.as<double>(), g.work.as<double>(),
                           beta, g.v_in.as<double>(), n);
        DZ_HIP(hipGetLastError());
        return;
    }
    // Append (v_in, R) into a free or the oldest slot.
    int slot;
    if ((int)g.order.size() < g.hist_cap) {
        slot = (int)g.order.size();
    } else {
        slot = g.order.front();
        g.order.erase(g.order.begin());
    }
    g.order.push_back(slot);
    double* hv = g.hv.as<double>() + (size_t)slot * n;
    double* hr = g.hr.as<double>() + (size_t)slot * n;
    DZ_HIP(hipMemcpyAsync(hv, g.v_in.ptr, n * sizeof(double), hipMemcpyDeviceToDevice, s));
    hipLaunchKernelGGL(k_sub, dim3(grid_blocks(n)), dim3(256), 0, s, g.v_out.as<double>(), g.v_in.as<double>(), hr, n);
    DZ_HIP(hipGetLastError());
    if (g.diemac > 1.0) {
        // R <- P R through the FFT (scf.zig:164-178 applies it in G space before the Pulay step).
        hipLaunchKernelGGL(k_real_to_complex, dim3(grid_blocks(n)), dim3(256), 0, s, hr, g.work.as<double2>(), n);
        DZ_HIP(hipGetLastError());
        fft3d_device<double>(g.work.as<double2>(), g.tab, false, s);
        hipLaunchKernelGGL(k_dielectric, dim3(grid_blocks(n)), dim3(256), 0, s, g.work.as<double2>(), g.g2.as<double>(),
                           1.0 / g.diemac, g.dielng * g.dielng, n);
        DZ_HIP(hipGetLastError());
        fft3d_device<double>(g.work.as<double2>(), g.tab, true, s);
        hipLaunchKernelGGL(k_real_part, dim3(grid_blocks(n)), dim3(256), 0, s, g.work.as<double2>(), hr, n);
        DZ_HIP(hipGetLastError());
    }
    for (int j : g.order) {
        const double d = g.dot(hr, g.hr.as<double>() + (size_t)j * n) / (double)n;
        g.b[slot][j] = d;
        g.b[j][slot] = d;
    }
    const int m = (int)g.order.size();
    auto linear = [&]() {
        hipLaunchKernelGGL(k_axpy_to, dim3(grid_blocks(n)), dim3(256), 0, s, g.v_in.as<double>(), hr, beta,
                           g.v_in.as<double>(), n);
        DZ_HIP(hipGetLastError());
    };
    if (m < 2) {
        linear();
        return;
    }
    // [B -1; -1 0] c = [0; -1], B scaled by its largest diagonal; partial-pivot elimination.
    const int sz = m + 1;
    std::vector<double> a((size_t)sz * sz, 0.0), rhs(sz, 0.0);
    double dmax = 0.0;
    for (int i = 0; i < m; ++i) dmax = std::max(dmax, g.b[g.order[i]][g.order[i]]);
    dmax = std::max(dmax, 1e-300);
    for (int i = 0; i < m; ++i) {
        for (int j = 0; j < m; ++j) a[(size_t)i * sz + j] = g.b[g.order[i]][g.order[j]] / dmax;
        a[(size_t)i * sz + m] = -1.0;
        a[(size_t)m * sz + i] = -1.0;
    }
    rhs[m] = -1.0;
    bool singular = false;
    for (int col = 0; col < sz && !singular; ++col) {
        int p = col;
        for (int r = col + 1; r < sz; ++r)
            if (std::fabs(a[(size_t)r * sz + col]) > std::fabs(a[(size_t)p * sz + col])) p = r;
        if (p != col) {
            for (int j = 0; j < sz; ++j) std::swap(a[(size_t)col * sz + j], a[(size_t)p * sz + j]);
            std::swap(rhs[col], rhs[p]);
        }
        const double piv = a[(size_t)col * sz + col];
        if (std::fabs(piv) < 1e-12) {
            singular = true;
            break;
        }
        for (int r = col + 1; r < sz; ++r) {
            const double f = a[(size_t)r * sz + col] / piv;
            for (int j = col; j < sz; ++j) a[(size_t)r * sz + j] -= f * a[(size_t)col * sz + j];
            rhs[r] -= f * rhs[col];
        }
    }
    if (singular) {
        g.order.assign(1, slot);
        linear();
        return;
    }
    std::vector<double> x(sz, 0.0);
    for (int i = sz - 1; i >= 0; --i) {
        double acc = rhs[i];
        for (int j = i + 1; j < sz; ++j) acc -= a[(size_t)i * sz + j] * x[j];
        x[i] = acc / a[(size_t)i * sz + i];
    }
    DZ_HIP(hipMemcpyAsync(g.slots.ptr, g.order.data(), m * sizeof(int), hipMemcpyHostToDevice, s));
    DZ_HIP(hipMemcpyAsync(g.coef.ptr, x.data(), m * sizeof(double), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_pulay_combine, dim3(grid_blocks(n)), dim3(256), 0, s, g.hv.as<double>(), g.hr.as<double>(),
                       g.slots.as<int>(), g.coef.as<double>(), m, beta, g.v_in.as<double>(), n);
    DZ_HIP(hipGetLastError());
    DZ_HIP(hipStreamSynchronize(s));  // slots/coef are host vectors
}

void scf_grid_set_xc(ScfGrid& g, int functional) {
    if (functional == DZHIP_XC_PBE) {
        g.work2.ensure(g.n * sizeof(double2));
        g.work3.ensure(g.n * sizeof(double2));
    }
    g.xc = functional;
}

}  // namespace dzhip
