// Lowest eigenpairs of a dense Hermitian matrix on the device (the Rayleigh-Ritz step of the
// block Davidson and CG solvers; src/features/linalg/lobpcg/common.zig:440-537 calls LAPACK
// zheev there).  Own design for one GPU; see heev.h for the four stages.
#include "heev.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <condition_variable>
#include <cstdlib>
#include <mutex>

#include "trd_shape.h"

namespace dzhip {

namespace {

constexpr unsigned kSpinLimit = 1u << 22;  // polls of one exchange (under a microsecond each) before giving up
// The same for a tridiagonalisation admitted by the gate: its grid may find the device short
// of CUs for a long time while other streams' kernels keep taking them, and it is then repeated as
// a cooperative launch (heev_lowest_shared).  Si-64 concurrent-k SCF, mixed arm to 1e-6 Ha: 5.7 s and no
// repeat at 2^16 polls and at 2^19; 5.7 s with cooperative launches only.
constexpr unsigned kSpinLimitShared = 1u << 19;

// One DPP row rotation of a double (both halves moved by the same row_ror:N control).
template <int CTRL>
__device__ __forceinline__ double dpp_rot(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, false);
    return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double read_lane(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}

// Exchange between the lane rows (16 lanes) of a wavefront and add: ROWS = 1 pairs rows 0-1 and 2-3,
// ROWS = 2 the halves.  Both lanes of a pair add the same two values in the same order.
template <int ROWS>
__device__ __forceinline__ double swap_add(double v) {
    const unsigned lo = (unsigned)__double2loint(v), hi = (unsigned)__double2hiint(v);
    if constexpr (ROWS == 1) {
        const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
        return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
    } else {
        const auto l = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
        return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
    }
}

// Sum over the 64 lanes of a wavefront (all lanes active), the same value in every lane: rotations
// by 8, 4, 2, 1 within each 16-lane row leave every lane of the row holding the row's sum (the same
// pairs added in every lane, so bitwise equal), then the rows are swapped and added pairwise.  No
// LDS traffic (a __shfl_xor butterfly is six ds_bpermute round trips) and no scalar registers.
__device__ __forceinline__ double wave_sum(double v) {
    v += dpp_rot<0x128>(v);  // row_ror:8
    v += dpp_rot<0x124>(v);  // row_ror:4
    v += dpp_rot<0x122>(v);  // row_ror:2
    v += dpp_rot<0x121>(v);  // row_ror:1
    return swap_add<2>(swap_add<1>(v));
}

// 1 / sqrt(s) and 1 / s from the hardware's estimates (relative error e about 1e-8) by one
// third-order Newton step, 1 - e expanded to e^2: a few dependent operations on the chain of every
// reflector, where the IEEE square root and divisions are some sixty.
__device__ __forceinline__ double rsqrt3(double s) {
    const double r = __builtin_amdgcn_rsq(s);
    const double e = fma(-(s * r), r, 1.0);
    return fma(r * e, fma(0.375, e, 0.5), r);
}
__device__ __forceinline__ double recip3(double s) {
    const double r = __builtin_amdgcn_rcp(s);
    const double e = fma(-s, r, 1.0);
    return fma(r, fma(e, e, e), r);
}

// The workgroups of the tridiagonalisation exchange two vectors per reflector (p_j and column j+1)
// through a buffer that is written once per call: every entry starts as kUnset, a signalling NaN
// that no arithmetic result can be (published values are canonicalised, which quiets NaNs), and a
// reader polls the entry itself until it is set.  One trip through memory per reflector, where a
// barrier costs three (wait for the stores, flag, then the values): 2.3 us against about 1 us.
// Stores and polls are relaxed agent-scope atomics, which write through the XCD's L2 and do not hit
// a stale copy there; each 8-byte entry carries its own arrival, so no ordering between entries is
// assumed.
constexpr unsigned long long kUnset = 0x7FF4DEADBEEF5A5Aull;

__device__ __forceinline__ void publish(double* p, double v) {
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(p),
                       (unsigned long long)__double_as_longlong(__builtin_canonicalize(v)), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long peek(const double* p) {
    return __hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED,
                             __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ double2 cm(double2 a, double2 b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
// conj(a) * b
__device__ __forceinline__ double2 cjm(double2 a, double2 b) {
    return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x);
}

struct TrdArgs {
    const double2* A;
    int lda, m;
    double2* vh;   // m x m: column j holds reflector v_j in rows j+1..m-1 (v_j[j+1] = 1), zeros above
    double2* tau;  // m
    double* d;     // m
    double* e;     // m - 1
    double* pub;   // m rows of 2 m doubles (several workgroups only): see trd_p, trd_n
    int* err;
    unsigned spin_limit;  // polls of one exchange before giving up
};

// Where step j's vectors lie in pub, real parts then (m doubles on) imaginary parts: p_j[r], r > j,
// in the upper part of row j and column j+1's rows r > j in the part of row m-1-j that p_{m-1-j}
// leaves free (0 <= r-j-1 <= m-2-j, and p_{m-1-j} starts at m-j).
__device__ __forceinline__ double* trd_p(double* pub, int m, int j, int r) { return pub + (size_t)j * 2 * m + r; }
__device__ __forceinline__ double* trd_n(double* pub, int m, int j, int r) {
    return pub + (size_t)(m - 1 - j) * 2 * m + (r - j - 1);
}

// Householder tridiagonalisation A = Q T Q^H, Q = H_0 ... H_{m-2}, H_j = I - tau_j v_j v_j^H, with
// zhetd2's reflectors (zlarfg: H_j^H x = beta e_1, beta real).  Every wavefront owns CW trailing
// columns for the whole reduction, in registers: lane l holds rows l + 64 q (q < NQ) of them and of
// every vector, so all products are lane-local and every sum is one wavefront's, and the wavefronts
// form v_j and w_j redundantly instead of exchanging them.  Step j:
//   A. receive p_{j-1} and column j (each wavefront polls a share of the rows into LDS; one
//      workgroup barrier);
//   B. w_{j-1} = p_{j-1} - (tau_{j-1} / 2) (p_{j-1}^H v_{j-1}) v_{j-1}; column j minus
//      v_{j-1} conj(w_{j-1}[j]) + w_{j-1} gives d_j and y; own columns i > j minus
//      v_{j-1} conj(w_{j-1}[i]) + w_{j-1} conj(v_{j-1}[i]) (the owner of column j+1 publishes it);
//   C. one reduction of |y|^2 and of the own columns' products with y gives tau_j, beta_j and
//      p_j[i] = tau_j a_i^H v_j (A Hermitian; v_j is y scaled below row j+1, where it is one), published;
//   D. while that travels: v_j, and the rows of v_j and of the own columns that step j+1 needs as
//      scalars (through LDS, like every other scalar row).
// The chain of a step is one memory trip, two wavefront sums and a square root with two divisions.
// The steps of one 64-row chunk are a loop of their own with the chunks above it left out at
// compile time: skipping them by branches kept every chunk's LDS reads from overlapping (0.36 us a
// chunk and step).  A workgroup whose columns are all reduced leaves.
template <int NQ, int CW>
struct Trd {
    static constexpr int NW = kTrdWaves, NT = 64 * NW, M64 = 64 * NQ, KR = NQ * 64 / NT + (NQ * 64 % NT != 0);
    const TrdArgs& a;
    double2* lds;  // two steps' [p | column j], M64 rows each
    double2* s_x;  // two steps' [NW * CW own columns' next row | v's next row]
    int* s_bad;    // two steps' flag: the exchange gave up
    int m, t, lane, wv, last_col;
    bool scribe;  // the wavefront that owns the last column writes T and the reflectors
    int ic[CW];
    double2 x[CW][NQ], y[NQ], v[NQ], w[NQ];
    double2 alpha, tau, vn;                // column j's row j+1, tau_j, v_{j-1}[j+1]
    double2 vi[CW], wi[CW], yi[CW], xo[CW];  // rows i of v, w and y; own columns' row j+1

    __device__ __forceinline__ double2 elem(int r, int i) const {
        // Only the lower triangle of A is read (the upper one is its mirror; the diagonal is real),
        // as LAPACK's zheev with uplo = 'L'.  Zero outside the matrix.
        if (r >= m || i >= m) return make_double2(0.0, 0.0);
        const double2 u = r >= i ? a.A[(size_t)i * a.lda + r] : a.A[(size_t)r * a.lda + i];
        return make_double2(u.x, r == i ? 0.0 : (r > i ? u.y : -u.y));
    }

    // C and D of step j, whose rows j+1.. lie in chunks QB and up.
    template <int QB>
    __device__ __forceinline__ void reflect(int j) {
#pragma unroll
        for (int c = 0; c < CW; ++c)
            if (ic[c] == j + 1) {
#pragma unroll
                for (int q = QB; q < NQ; ++q) {
                    const int r = lane + 64 * q;
                    if (r <= j || r >= m) continue;
                    double* pn = trd_n(a.pub, m, j, r);
                    publish(pn, x[c][q].x);
                    publish(pn + m, x[c][q].y);
                }
            }
        double sums[1 + 2 * CW];
#pragma unroll
        for (int c = 0; c < 1 + 2 * CW; ++c) sums[c] = 0.0;
#pragma unroll
        for (int q = QB; q < NQ; ++q) {
            sums[0] += y[q].x * y[q].x + y[q].y * y[q].y;
#pragma unroll
            for (int c = 0; c < CW; ++c) {
                const double2 u = cjm(x[c][q], y[q]);
                sums[1 + 2 * c] += u.x;
                sums[2 + 2 * c] += u.y;
            }
        }
#pragma unroll
        for (int c = 0; c < 1 + 2 * CW; ++c) sums[c] = wave_sum(sums[c]);
        const double xn2 = sums[0];
        double beta;
        double2 scale;
        if (fma(alpha.y, alpha.y, xn2) == 0.0) {  // reduced already, or but for entries below 1e-162
            tau = make_double2(0.0, 0.0);
            beta = alpha.x;
            scale = make_double2(0.0, 0.0);
        } else {
            const double n2 = alpha.x * alpha.x + alpha.y * alpha.y + xn2;
            const double ir = rsqrt3(n2), nrm = n2 * ir;
            const double ib = alpha.x >= 0.0 ? -ir : ir;
            beta = alpha.x >= 0.0 ? -nrm : nrm;
            tau = make_double2((beta - alpha.x) * ib, -alpha.y * ib);
            const double2 den = make_double2(alpha.x - beta, alpha.y);
            const double dd = den.x * den.x + den.y * den.y;
            // The reciprocal of the mantissa, its exponent with the numerator: 1 / dd itself leaves the range
            // below a norm of 1e-154.
            const int ex = -__builtin_amdgcn_frexp_exp(dd);
            const double id = recip3(__builtin_amdgcn_frexp_mant(dd));
            scale = make_double2(__builtin_amdgcn_ldexp(den.x, ex) * id, -__builtin_amdgcn_ldexp(den.y, ex) * id);
        }
#pragma unroll
        for (int c = 0; c < CW; ++c) {
            if (ic[c] <= j || ic[c] >= m) continue;
            const double2 s = cm(scale, make_double2(sums[1 + 2 * c], sums[2 + 2 * c]));
            const double2 p = cm(tau, make_double2(xo[c].x + s.x, s.y - xo[c].y));
            if (lane == 0) {
                double* pp = trd_p(a.pub, m, j, ic[c]);
                publish(pp, p.x);
                publish(pp + m, p.y);
            }
        }
        double2* sx = s_x + (j & 1) * (NW * CW + 1);
#pragma unroll
        for (int q = QB; q < NQ; ++q) {
            v[q] = cm(y[q], scale);
            if (q <= QB + 1) {
                const int r = lane + 64 * q;
                if (r == j + 1) v[q] = make_double2(1.0, 0.0);
                if (r == j + 2) {
                    if (wv == 0) sx[NW * CW] = v[q];
#pragma unroll
                    for (int c = 0; c < CW; ++c) sx[wv * CW + c] = x[c][q];
                }
            }
        }
#pragma unroll
        for (int c = 0; c < CW; ++c) vi[c] = ic[c] == j + 1 ? make_double2(1.0, 0.0) : cm(yi[c], scale);
        if (scribe) {
#pragma unroll
            for (int q = QB; q < NQ; ++q) {
                const int r = lane + 64 * q;
                if (r > j && r < m) a.vh[(size_t)j * m + r] = v[q];
            }
            if (lane == 0) {
                a.e[j] = beta;
                a.tau[j] = tau;
            }
        }
    }

    // A and B of step j (rows j.. in chunks QB and up); false when the exchange gave up.
    template <int QB>
    __device__ __forceinline__ bool advance(int j) {
        double2* sp = lds + (j & 1) * 2 * M64;
        double2* sn = sp + M64;
        unsigned long long in[KR][4];
        unsigned spins = 0;
        while (true) {
            bool set = true;
#pragma unroll
            for (int k = 0; k < KR; ++k) {
                const int r = t + k * NT;
                if (r >= j && r < m) {
                    const double* pp = trd_p(a.pub, m, j - 1, r);
                    const double* pn = trd_n(a.pub, m, j - 1, r);
                    in[k][0] = peek(pp);
                    in[k][1] = peek(pp + m);
                    in[k][2] = peek(pn);
                    in[k][3] = peek(pn + m);
                }
            }
#pragma unroll
            for (int k = 0; k < KR; ++k) {
                const int r = t + k * NT;
                if (r >= j && r < m)
                    set = set && in[k][0] != kUnset && in[k][1] != kUnset && in[k][2] != kUnset && in[k][3] != kUnset;
            }
            if (__all(set)) break;
            ++spins;
            const bool stop = (spins & 255u) == 0 &&
                              __hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
            if (spins > a.spin_limit || __any(stop)) {
                if (lane == 0) {
                    __hip_atomic_store(a.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    s_bad[j & 1] = 1;
                }
                break;
            }
        }
#pragma unroll
        for (int k = 0; k < KR; ++k) {
            const int r = t + k * NT;
            if (r >= j && r < m) {
                sp[r] = make_double2(__longlong_as_double((long long)in[k][0]), __longlong_as_double((long long)in[k][1]));
                sn[r] = make_double2(__longlong_as_double((long long)in[k][2]), __longlong_as_double((long long)in[k][3]));
            }
        }
        __syncthreads();
        if (s_bad[j & 1]) return false;  // by step parity: a faster wavefront may already give up in the next one
        // Rows below j of sp and sn are an earlier step's (finite) and meet v = 0 there; rows from m
        // on are zero.
        const double2* sx = s_x + ((j - 1) & 1) * (NW * CW + 1);
#pragma unroll
        for (int q = QB; q < NQ; ++q) w[q] = sp[lane + 64 * q];
        const int j1 = min(j + 1, M64 - 1);
        const double2 pj = sp[j], pj1 = sp[j1];
        vn = sx[NW * CW];
        double2 pi[CW];
#pragma unroll
        for (int c = 0; c < CW; ++c) {
            pi[c] = sp[min(ic[c], M64 - 1)];
            yi[c] = sn[min(ic[c], M64 - 1)];
            xo[c] = sx[wv * CW + c];
        }
        const double2 nj = sn[j], nj1 = sn[j1];
#pragma unroll
        for (int q = QB; q < NQ; ++q) y[q] = sn[lane + 64 * q];
        double2 dot = make_double2(0.0, 0.0);
#pragma unroll
        for (int q = QB; q < NQ; ++q) {
            const double2 u = cjm(w[q], v[q]);
            dot.x += u.x;
            dot.y += u.y;
        }
        dot.x = wave_sum(dot.x);
        dot.y = wave_sum(dot.y);
        const double2 al = cm(make_double2(-0.5 * tau.x, -0.5 * tau.y), dot);
        const double2 wj = make_double2(pj.x + al.x, pj.y + al.y);  // v_{j-1}[j] = 1
        const double2 aln = cm(al, vn), wn = make_double2(pj1.x + aln.x, pj1.y + aln.y);
        const double2 ua = cjm(wj, vn);
        alpha = make_double2(nj1.x - ua.x - wn.x, nj1.y - ua.y - wn.y);
        if (scribe && lane == 0) a.d[j] = nj.x - 2.0 * wj.x;
#pragma unroll
        for (int c = 0; c < CW; ++c) {
            const double2 u = cm(al, vi[c]);
            wi[c] = make_double2(pi[c].x + u.x, pi[c].y + u.y);
            const double2 uy = cjm(wj, vi[c]);
            yi[c] = make_double2(yi[c].x - uy.x - wi[c].x, yi[c].y - uy.y - wi[c].y);
            const double2 u1 = cjm(wi[c], vn), u2 = cjm(vi[c], wn);
            xo[c] = make_double2(xo[c].x - u1.x - u2.x, xo[c].y - u1.y - u2.y);
        }
#pragma unroll
        for (int q = QB; q < NQ; ++q) {
            const double2 u = cm(al, v[q]);
            w[q] = make_double2(w[q].x + u.x, w[q].y + u.y);
            const double2 u0 = cjm(wj, v[q]);
            y[q] = make_double2(y[q].x - u0.x - w[q].x, y[q].y - u0.y - w[q].y);
            if (q <= QB + 1 && lane + 64 * q < j + 2) y[q] = make_double2(0.0, 0.0);
#pragma unroll
            for (int c = 0; c < CW; ++c) {
                const double2 u1 = cjm(wi[c], v[q]), u2 = cjm(vi[c], w[q]);
                x[c][q].x -= u1.x + u2.x;
                x[c][q].y -= u1.y + u2.y;
            }
        }
        return true;
    }

    // Steps whose reflector starts in chunk QB, then the next chunks'.
    template <int QB>
    __device__ __forceinline__ void run() {
        if constexpr (QB < NQ) {
            const int end = min(64 * (QB + 1), m - 1);
            for (int j = 64 * QB; j < end; ++j) {
                reflect<QB>(j);
                if (last_col <= j + 1 && last_col != m - 1) return;
                if (!advance<QB>(j + 1)) return;
            }
            run<QB + 1>();
        }
    }
};

template <int NQ, int CW>
__global__ __launch_bounds__(64 * kTrdWaves, 1) void k_hetrd(TrdArgs a) {
    extern __shared__ double2 lds[];
    __shared__ double2 s_x[2 * (kTrdWaves * CW + 1)];
    __shared__ int s_bad[2];
    using K = Trd<NQ, CW>;
    const int t = (int)threadIdx.x, g = (int)blockIdx.x, m = a.m;
    K k{a, lds, s_x, s_bad, m, t, t & 63, __builtin_amdgcn_readfirstlane(t >> 6)};
    k.last_col = min(m, (g + 1) * K::NW * CW) - 1;
    k.scribe = false;
    for (int i = t; i < 4 * K::M64; i += K::NT) lds[i] = make_double2(0.0, 0.0);
    if (t < 2 * (K::NW * CW + 1)) s_x[t] = make_double2(0.0, 0.0);
    if (t < 2) s_bad[t] = 0;
#pragma unroll
    for (int c = 0; c < CW; ++c) {
        const int i = k.ic[c] = (g * K::NW + k.wv) * CW + c;
        k.scribe = k.scribe || i == m - 1;
#pragma unroll
        for (int q = 0; q < NQ; ++q) k.x[c][q] = k.elem(k.lane + 64 * q, i);
        k.xo[c] = k.elem(1, i);
        k.yi[c] = k.elem(i, 0);
        k.vi[c] = make_double2(0.0, 0.0);
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int r = k.lane + 64 * q;
        k.y[q] = r >= 2 ? k.elem(r, 0) : make_double2(0.0, 0.0);
        k.v[q] = make_double2(0.0, 0.0);
    }
    k.alpha = k.elem(1, 0);
    k.tau = k.vn = make_double2(0.0, 0.0);
    if (k.scribe && k.lane == 0) a.d[0] = a.A[0].x;
    __syncthreads();
    k.template run<0>();
}

// The exchange buffer's entries unset, the reflectors' rows (of which the tridiagonalisation writes
// those from v_j[j+1] on) zero, the error flag cleared.
__global__ __launch_bounds__(256) void k_trd_init(ulonglong2* pub, double2* vh, size_t n, int* err) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i == 0) *err = 0;
    if (i < n) {
        pub[i] = make_ulonglong2(kUnset, kUnset);
        vh[i] = make_double2(0.0, 0.0);
    }
}

// Number of eigenvalues of T below x from a factorisation twisted at row h = (m - 1) / 2: pivots
// q_i = d_i - x - e_{i-1}^2 / q_{i-1} down from the top, r_i = d_i - x - e_i^2 / r_{i+1} up from the
// bottom, and g = d_h - x - e_{h-1}^2 / q_{h-1} - e_h^2 / r_{h+1}; by Sylvester's law of inertia as
// many eigenvalues lie below x as pivots are negative.  The two recurrences are independent, so the
// chain is half as long as one recurrence over all rows.  de: (d_i, e_i^2), e_{m-1} = 0.  Quotients
// come from the hardware's reciprocal with one third-order Newton step and no test for small
// pivots; one (tiny or zero) that overflows turns its recurrence into NaN within a step, and those
// kSturmBlock rows are done again with divisions and pivots raised to pivmin (LAPACK dlaebz's rule).
constexpr int kSturmBlock = 8;
struct SturmState {
    double f, b;  // e^2 / q and e^2 / r to subtract from the next rows
    int cnt;
};
template <bool SAFE>
__device__ __forceinline__ void sturm_step(double pivot_in, double e2, double pivmin, double* out, int* cnt) {
    double q = pivot_in;
    if (SAFE) {
        if (fabs(q) < pivmin) q = -pivmin;
        *out = e2 / q;
    } else {
        const double r = __builtin_amdgcn_rcp(q), t = e2 * r, e = fma(-q, r, 1.0);
        *out = fma(t, fma(e, e, e), t);
    }
    *cnt += (int)((unsigned)__double2hiint(q) >> 31);
}
template <bool SAFE>
__device__ __forceinline__ void sturm_rows(const double2* de, int m, int s, double x, double pivmin, SturmState& st) {
    const double2 a = de[s], c = de[m - 1 - s];
    sturm_step<SAFE>(a.x - x - st.f, a.y, pivmin, &st.f, &st.cnt);
    sturm_step<SAFE>(c.x - x - st.b, de[m - 2 - s].y, pivmin, &st.b, &st.cnt);
}
__device__ __forceinline__ int sturm_count(const double2* de, int m, double x, double pivmin) {
    const int h = (m - 1) / 2;
    SturmState st{0.0, 0.0, 0};
    for (int s = 0; s < h; s += kSturmBlock) {
        const SturmState st0 = st;
        const int n = min(kSturmBlock, h - s);
        if (n == kSturmBlock) {
#pragma unroll
            for (int k = 0; k < kSturmBlock; ++k) sturm_rows<false>(de, m, s + k, x, pivmin, st);
        } else {
            for (int k = 0; k < n; ++k) sturm_rows<false>(de, m, s + k, x, pivmin, st);
        }
        if (__any(st.f != st.f || st.b != st.b)) {
            st = st0;
            for (int k = 0; k < n; ++k) sturm_rows<true>(de, m, s + k, x, pivmin, st);
        }
    }
    if (m - 1 - h > h) sturm_step<true>(de[h + 1].x - x - st.b, de[h].y, pivmin, &st.b, &st.cnt);
    double unused;
    sturm_step<true>(de[h].x - x - st.f - st.b, 0.0, pivmin, &unused, &st.cnt);
    return st.cnt;
}

// Eigenvalue blockIdx.x (ascending) of T by multisection: each round the workgroup's 256 lanes count
// at 256 interior points of [lo, hi] and keep the sub-interval that holds the eigenvalue; seven
// rounds reach the last bits, where 64 points took nine.  The FP64 issue rate bounds it, one
// wavefront per SIMD (the registers of compact_reflectors, which shares the launch).  Also writes the
// Gershgorin scale of T to scal[0] (block 0).  nev = 160, one wavefront per eigenvalue, one recurrence and
// divisions before: m = 164 / 648 113 -> 65 us, 418 -> 228 us, the reflectors' compact form (11 and 30 us
// before) included.  More eigenvalues than CUs take turns; whole calls for all of them: m = 648 7,276 ->
// 3,596 us, m = 1,000 14,219 -> 8,971 us.
__device__ __forceinline__ void stebz(const double* __restrict__ d_in, const double* __restrict__ e_in, int m,
                                      double* __restrict__ w, double* __restrict__ scal, const int* __restrict__ err,
                                      double2* de) {
    __shared__ double red[4 * 3];
    __shared__ int s_low[2][4];
    const int t = (int)threadIdx.x, idx = (int)blockIdx.x;
    double lo_l = 1e300, hi_l = -1e300, e2max = 0.0;
    for (int k = t; k < m; k += 256) {
        const double dk = d_in[k];
        const double el = k > 0 ? fabs(e_in[k - 1]) : 0.0;
        const double er = k + 1 < m ? fabs(e_in[k]) : 0.0;
        de[k] = make_double2(dk, er * er);
        lo_l = fmin(lo_l, dk - el - er);
        hi_l = fmax(hi_l, dk + el + er);
        e2max = fmax(e2max, er * er);
    }
    // Block min / max / max via negation into a sum-free reduction.
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        lo_l = fmin(lo_l, __shfl_xor(lo_l, o, 64));
        hi_l = fmax(hi_l, __shfl_xor(hi_l, o, 64));
        e2max = fmax(e2max, __shfl_xor(e2max, o, 64));
    }
    if ((t & 63) == 0) {
        red[(t >> 6) * 3] = lo_l;
        red[(t >> 6) * 3 + 1] = hi_l;
        red[(t >> 6) * 3 + 2] = e2max;
    }
    __syncthreads();
    double gl = red[0], gu = red[1], em = red[2];
    for (int i = 1; i < 4; ++i) {
        gl = fmin(gl, red[i * 3]);
        gu = fmax(gu, red[i * 3 + 1]);
        em = fmax(em, red[i * 3 + 2]);
    }
    const double bnorm = fmax(fabs(gl), fabs(gu));
    const double pivmin = 2.2250738585072014e-308 * fmax(1.0, em) / 2.220446049250313e-16;
    // Widen so that the ends are strictly outside the spectrum.
    const double wid = 2.220446049250313e-16 * 4.0 * bnorm + 2.0 * pivmin + 1e-300;
    gl -= wid + 1e-14 * (gu - gl);
    gu += wid + 1e-14 * (gu - gl);
    if (idx == 0 && t == 0) scal[0] = bnorm;
    // A tridiagonalisation whose exchange did not complete leaves NaN eigenvalues (the signal
    // a caller without a synchronising check sees).
    if (*err != 0) {
        if (t == 0) w[idx] = __builtin_nan("");
        return;
    }
    constexpr double kParts = 257.0;
    double lo = gl, hi = gu;
    for (int round = 0; round < 14; ++round) {
        const double width = hi - lo;
        if (!(width > 2.0 * 2.220446049250313e-16 * fmax(fabs(lo), fabs(hi)) + 2.0 * pivmin)) break;
        const int cnt = sturm_count(de, m, lo + width * (double)(t + 1) / kParts, pivmin);
        // Highest point that still has the eigenvalue at or above it; -1 if none.
        const unsigned long long below = __ballot(cnt <= idx);
        if ((t & 63) == 0) s_low[round & 1][t >> 6] = below ? (t | (63 - __builtin_clzll(below))) : -1;
        __syncthreads();
        int L = -1;
#pragma unroll
        for (int q = 0; q < 4; ++q) L = max(L, s_low[round & 1][q]);
        double nlo = lo, nhi = hi;
        if (L < 0) {
            nhi = lo + width * 1.0 / kParts;
        } else {
            nlo = lo + width * (double)(L + 1) / kParts;
            if (L < 255) nhi = lo + width * (double)(L + 2) / kParts;
        }
        lo = nlo;
        hi = nhi;
    }
    if (t == 0) w[idx] = 0.5 * (lo + hi);
}

// The reflectors of A = Q T Q^H in compact form, blocks of kWyNb of them: H_k0 ... H_k1 = I - V T V^H
// with T upper triangular (T[j][j] = tau_j, T[0:j, j] = -tau_j T[0:j, 0:j] V[:, 0:j]^H v_j), and
// W = V T, so that a block acts on a vector as y - W (V^H y).  One workgroup per two blocks: the
// Gram products V^H V on the matrix cores (FP64 16x16x4; both operands are the same registers, lane
// l holding row l / 16 of a group of four of reflector l % 16), the two triangles by one lane per
// row, W by one thread per row.  w: column k0 + j holds W_j, its rows up to
// k0 zero like V's.
constexpr int kWyNb = 8;
typedef double wy_v4d __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void compact_reflectors(const double2* __restrict__ vh, const double2* __restrict__ tau, int m,
                                                   double2* __restrict__ w, int group, double2* lds) {
    auto gs = reinterpret_cast<double2(*)[16][17]>(lds);  // each wavefront's share of V^H V, then their sum in gs[0]
    __shared__ double2 ts[2][kWyNb][kWyNb];
    const int t = (int)threadIdx.x, wv = t >> 6, lane = t & 63, l16 = lane & 15, l4 = lane >> 4;
    const int k0 = group * 2 * kWyNb, nref = m - 1;
    // Row 0 of every reflector and the column past the last one are zero.
    const double2* vcol = vh + (size_t)min(k0 + l16, nref) * m;
    wy_v4d re = {0, 0, 0, 0}, im = {0, 0, 0, 0};
#pragma unroll 8
    for (int r0 = k0 + 1 + 4 * wv; r0 < m; r0 += 16) {
        const double2 v = vcol[r0 + l4 < m ? r0 + l4 : 0];
        re = __builtin_amdgcn_mfma_f64_16x16x4f64(v.x, v.x, re, 0, 0, 0);
        im = __builtin_amdgcn_mfma_f64_16x16x4f64(v.x, v.y, im, 0, 0, 0);
        re = __builtin_amdgcn_mfma_f64_16x16x4f64(v.y, v.y, re, 0, 0, 0);
        im = __builtin_amdgcn_mfma_f64_16x16x4f64(-v.y, v.x, im, 0, 0, 0);
    }
    // D slot r: row l / 16 + 4 r, column l % 16.
#pragma unroll
    for (int r = 0; r < 4; ++r) gs[wv][l4 + 4 * r][l16] = make_double2(re[r], im[r]);
    __syncthreads();
    {
        const int i = t >> 4, j = t & 15;
        double2 g = gs[0][i][j];
#pragma unroll
        for (int q = 1; q < 4; ++q) {
            g.x += gs[q][i][j].x;
            g.y += gs[q][i][j].y;
        }
        __syncthreads();
        gs[0][i][j] = g;
    }
    __syncthreads();
    if (t < 2 * kWyNb) {
        const int h = t / kWyNb, a = t % kWyNb;  // row a of block h
        double2 row[kWyNb];
#pragma unroll
        for (int j = 0; j < kWyNb; ++j) {
            const int kj = k0 + h * kWyNb + j;
            const double2 tj = kj < nref ? tau[kj] : make_double2(0.0, 0.0);
            double2 s = make_double2(0.0, 0.0);
#pragma unroll
            for (int b = 0; b < j; ++b) {
                const double2 u = cm(row[b], gs[0][h * kWyNb + b][h * kWyNb + j]);
                s.x += u.x;
                s.y += u.y;
            }
            const double2 u = cm(tj, s);
            row[j] = a == j ? tj : (a < j ? make_double2(-u.x, -u.y) : make_double2(0.0, 0.0));
            ts[h][a][j] = row[j];
        }
    }
    __syncthreads();
    for (int r = t; r < m; r += 256) {
        double2 v[2 * kWyNb];
#pragma unroll
        for (int i = 0; i < 2 * kWyNb; ++i) v[i] = vh[(size_t)min(k0 + i, nref) * m + r];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < kWyNb; ++j) {
                double2 s = make_double2(0.0, 0.0);
#pragma unroll
                for (int i = 0; i <= j; ++i) {
                    const double2 u = cm(v[h * kWyNb + i], ts[h][i][j]);
                    s.x += u.x;
                    s.y += u.y;
                }
                const int k = k0 + h * kWyNb + j;
                if (k < m) w[(size_t)k * m + r] = s;
            }
    }
}

// The eigenvalues of T (blocks 0..nev-1) and, beside them because neither needs the other, the
// compact form of the reflectors (the blocks after them).
__global__ __launch_bounds__(256) void k_stebz(const double* __restrict__ d_in, const double* __restrict__ e_in, int m,
                                               int nev, double* __restrict__ w, double* __restrict__ scal,
                                               const int* __restrict__ err, const double2* __restrict__ vh,
                                               const double2* __restrict__ tau, double2* __restrict__ wy) {
    extern __shared__ double2 sh2[];
    if ((int)blockIdx.x < nev) stebz(d_in, e_in, m, w, scal, err, sh2);
    else compact_reflectors(vh, tau, m, wy, (int)blockIdx.x - nev, sh2);
}
constexpr int kWyLds = 4 * 16 * 17 * (int)sizeof(double2);

// Eigenvalues closer than this (consecutive gaps, relative to the Gershgorin scale) form a cluster
// whose inverse-iteration vectors are orthonormalised together.
__device__ __forceinline__ double cluster_tol(double bnorm) { return 1e-12 * fmax(bnorm, 1.0); }

// Eigenvector of T for eigenvalue k by inverse iteration, one wavefront per eigenvalue (all
// independent).  T - lambda I = P L U with partial pivoting (dlagtf's factorisation, U with two
// superdiagonals; pivots below eps |T| are raised to that size), then three solves from a seeded
// start, each followed by scaling and normalisation.  T, the factors and the iterate live in LDS.
// The recurrences are serial and set the time.  Every lane runs them (reads are broadcasts): the
// rows of the next kSteinBlock steps are loaded while the current ones are computed, a pivot costs
// one reciprocal for its multiplier and its inverse, exchanges are selects (`divergent` hides from
// the compiler that all lanes agree, which would make each a branch on a vector compare), and T is
// padded with decoupled rows (lambda + 1, 0) to whole blocks.  Rows on one lane with an LDS wait and
// divisions a step before: nev = 160, m = 164 / 648 99 -> 53 us, 372 -> 190 us.
constexpr int kSteinBlock = 8;
__host__ __device__ constexpr int stein_rows(int m) { return (m + kSteinBlock - 1) / kSteinBlock * kSteinBlock; }
__device__ __forceinline__ double divergent(double v) {
    asm volatile("" : "+v"(v));
    return v;
}
struct Stein {
    int m, mp;     // rows; rows computed
    double2* de;   // d, e
    double2* lp;   // multiplier, 1 where rows r and r + 1 are exchanged
    double2* uu;   // 1 / U[r][r], U[r][r + 1]
    double* u2;    // U[r][r + 2]
    double* x;
    int ma;        // rows the loads ahead may touch

    __device__ __forceinline__ Stein(double* sh, int rows) : m(rows), mp(stein_rows(rows)) {
        ma = mp + kSteinBlock;
        de = reinterpret_cast<double2*>(sh);
        lp = de + ma;
        uu = lp + ma;
        u2 = reinterpret_cast<double*>(uu + ma);
        x = u2 + ma;
    }
    __device__ __forceinline__ void load(const double* __restrict__ d_in, const double* __restrict__ e_in, double lam, int r) const {
        de[r] = make_double2(r < m ? d_in[r] : lam + 1.0, r + 1 < m ? e_in[r] : 0.0);
    }
    // T - lam = P L U, pivots raised to pert.
    __device__ __forceinline__ void factor(double lam, double pert) const {
        constexpr int NB = kSteinBlock;
        // Row r: (ca, cb); row r + 1 starts with c = e_r.
        double ca = divergent(de[0].x - lam), cb = divergent(de[0].y), c = cb;
        double2 nx[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) nx[i] = de[1 + i];
        for (int r0 = 0; r0 < mp; r0 += NB) {
            double2 cur[NB];
#pragma unroll
            for (int i = 0; i < NB; ++i) cur[i] = nx[i];
            const int ahead = min(r0 + NB, mp - 1);
#pragma unroll
            for (int i = 0; i < NB; ++i) nx[i] = de[ahead + 1 + i];
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const double na = cur[i].x - lam, nb = cur[i].y;
                const bool keep = fabs(ca) >= fabs(c);
                const double p = keep ? ca : c;
                const double inv = recip3(copysign(fmax(fabs(p), pert), p));
                const double l = (keep ? c : ca) * inv;
                const double top = keep ? cb : na, low = keep ? na : cb;
                lp[r0 + i] = make_double2(l, keep ? 0.0 : 1.0);
                uu[r0 + i] = make_double2(inv, top);
                u2[r0 + i] = keep ? 0.0 : nb;
                ca = low - l * top;
                cb = keep ? nb : -l * nb;
                c = nb;
            }
        }
    }
    // x <- (T - lam)^-1 x.
    __device__ __forceinline__ void solve() const {
        constexpr int NB = kSteinBlock;
        // P L y = x, in place.
        double xr = divergent(x[0]);
        double2 nl[NB];
        double nx[NB];
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            nl[i] = lp[i];
            nx[i] = x[1 + i];
        }
        for (int r0 = 0; r0 < mp; r0 += NB) {
            double2 l[NB];
            double xi[NB];
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                l[i] = nl[i];
                xi[i] = nx[i];
            }
            const int ahead = min(r0 + NB, mp - 1);
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                nl[i] = lp[ahead + i];
                nx[i] = x[ahead + 1 + i];
            }
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const bool swap = divergent(l[i].y) != 0.0;
                const double a = swap ? xi[i] : xr, b = swap ? xr : xi[i];
                x[r0 + i] = a;
                xr = b - l[i].x * a;
            }
        }
        // U z = y, in place, from the last row.
        double z0 = 0.0, z1 = 0.0;
        double2 nu[NB];
        double n2[NB];
        auto ahead = [&](int top) {
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                nu[i] = uu[top - i];
                n2[i] = u2[top - i];
                nx[i] = x[top - i];
            }
        };
        ahead(mp - 1);
        for (int r0 = mp - 1; r0 >= 0; r0 -= NB) {
            double2 u[NB];
            double v2[NB], xi[NB];
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                u[i] = nu[i];
                v2[i] = n2[i];
                xi[i] = nx[i];
            }
            ahead(max(r0 - NB, NB - 1));
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const double z = (xi[i] - v2[i] * z1 - u[i].y * z0) * u[i].x;
                x[r0 - i] = z;
                z1 = z0;
                z0 = z;
            }
        }
    }
    // x / |x| (one wavefront): scaled by the largest entry first (a solve amplifies by up to 1 / pert).
    __device__ __forceinline__ void normalise(int lane) const {
        double mx = 0.0;
        for (int r = lane; r < m; r += 64) mx = fmax(mx, fabs(x[r]));
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o, 64));
        const double inv_mx = mx > 0.0 ? 1.0 / mx : 1.0;
        double s2 = 0.0;
        for (int r = lane; r < m; r += 64) {
            const double v = x[r] * inv_mx;
            s2 += v * v;
        }
        s2 = wave_sum(s2);
        const double sc = inv_mx / sqrt(fmax(s2, 1e-300));
        for (int r = lane; r < m; r += 64) x[r] *= sc;
    }
};
__device__ __forceinline__ double stein_pert(double bnorm) { return 2.220446049250313e-16 * fmax(bnorm, 1e-300) + 1e-300; }

__global__ __launch_bounds__(64) void k_stein(const double* __restrict__ d_in, const double* __restrict__ e_in, int m,
                                              int nev, const double* __restrict__ w, const double* __restrict__ scal,
                                              double* __restrict__ Z, int ldz) {
    extern __shared__ double sh[];
    const int k = (int)blockIdx.x, lane = (int)threadIdx.x;
    if (k >= nev) return;
    const Stein t(sh, m);
    const double lam = w[k];
    for (int r = lane; r < t.ma; r += 64) {
        t.load(d_in, e_in, lam, r);
        // Seeded start (splitmix64 of eigenvalue and row).
        unsigned long long h = 0x9E3779B97F4A7C15ull * (unsigned long long)(k + 1) + (unsigned long long)r;
        h = (h ^ (h >> 30)) * 0xBF58476D1CE4E5B9ull;
        h = (h ^ (h >> 27)) * 0x94D049BB133111EBull;
        h ^= h >> 31;
        t.x[r] = r < m ? (double)(h >> 11) * (1.0 / 9007199254740992.0) - 0.5 : 0.0;
    }
    __syncthreads();
    t.factor(lam, stein_pert(scal[0]));
    __syncthreads();
    for (int it = 0; it < 3; ++it) {
        t.solve();
        __syncthreads();
        t.normalise(lane);
        __syncthreads();
    }
    for (int r = lane; r < m; r += 64) Z[(size_t)k * ldz + r] = t.x[r];
}

// Members of each cluster (consecutive eigenvalues closer than cluster_tol), in order, made
// orthonormal against the cluster's earlier members by two passes of classical Gram-Schmidt (one
// workgroup per cluster; the first member leads).  Inverse iteration gives each member a vector in
// the cluster's invariant subspace, so the orthonormal result spans the same subspace.  Where the members
// of a split T (equal blocks) came out nearly parallel, what a projection leaves has lost as many digits as
// it is short; below kSteinLeft of the vector another solve (by wavefront 0) brings them back, with the
// earlier members out of its start.
constexpr double kSteinLeft = 0.05;
__global__ __launch_bounds__(256) void k_stein_cluster(const double* __restrict__ d_in, const double* __restrict__ e_in,
                                                       const double* __restrict__ w, const double* __restrict__ scal,
                                                       int nev, int m, double* __restrict__ Z, int ldz) {
    extern __shared__ double sh[];
    __shared__ double dots[kHeevMaxM];
    __shared__ double red[4];
    const int i = (int)blockIdx.x;
    if (i >= nev) return;
    const double tau_c = cluster_tol(scal[0]);
    if (i > 0 && w[i] - w[i - 1] <= tau_c) return;
    int last = i;
    while (last + 1 < nev && w[last + 1] - w[last] <= tau_c) ++last;
    if (last == i) return;
    const Stein s(sh, m);
    const int t = (int)threadIdx.x, wv = t >> 6, lane = t & 63;
    for (int k = i + 1; k <= last; ++k) {
        double* x = Z + (size_t)k * ldz;
        for (int attempt = 0;; ++attempt) {
            for (int pass = 0; pass < 2; ++pass) {
                for (int p = i + wv; p < k; p += 4) {
                    const double* zp = Z + (size_t)p * ldz;
                    double sdot = 0.0;
                    for (int r = lane; r < m; r += 64) sdot += zp[r] * x[r];
                    sdot = wave_sum(sdot);
                    if (lane == 0) dots[p - i] = sdot;
                }
                __syncthreads();
                for (int r = t; r < m; r += 256) {
                    double acc = x[r];
                    for (int p = i; p < k; ++p) acc -= dots[p - i] * Z[(size_t)p * ldz + r];
                    x[r] = acc;
                }
                __syncthreads();
            }
            double s2 = 0.0;
            for (int r = t; r < m; r += 256) s2 += x[r] * x[r];
            s2 = wave_sum(s2);
            if (lane == 0) red[wv] = s2;
            __syncthreads();
            const double nrm = sqrt(red[0] + red[1] + red[2] + red[3]);
            const double inv = nrm > 0.0 ? 1.0 / nrm : 0.0;
            for (int r = t; r < m; r += 256) x[r] *= inv;
            __syncthreads();
            if (nrm >= kSteinLeft || attempt == 2) break;
            const double lam = w[k];
            for (int r = t; r < s.ma; r += 256) {
                s.load(d_in, e_in, lam, r);
                s.x[r] = r < m ? x[r] : 0.0;
            }
            __syncthreads();
            if (wv == 0) {
                s.factor(lam, stein_pert(scal[0]));
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                s.solve();
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                s.normalise(lane);
            }
            __syncthreads();
            for (int r = t; r < m; r += 256) x[r] = s.x[r];
            __syncthreads();
        }
    }
}

// C[0:n, 0:n] = Z^T Z (Z: m x n, leading dimension ldz) and Out = Z (1.5 I - 0.5 C), one Newton-Schulz
// step towards orthonormal columns: 16 x 16 tiles on the matrix cores, the sum in chunks of 16 dealt to
// the workgroup's four wavefronts (few tiles, so latency bounds them) and added in LDS.  The sum's
// order within a chunk is free, so a lane takes four consecutive elements.  Both products, two steps:
// m = 164 67 -> 20 us, m = 648 114 -> 29 us (one thread a result before).

// Sum of the four wavefronts' accumulators, in wavefront 0.
__device__ __forceinline__ wy_v4d tile_sum(wy_v4d acc, double (&red)[3][4][64], int wave, int lane) {
    if (wave > 0)
#pragma unroll
        for (int t = 0; t < 4; ++t) red[wave - 1][t][lane] = acc[t];
    __syncthreads();
    if (wave == 0)
#pragma unroll
        for (int t = 0; t < 4; ++t) acc[t] += red[0][t][lane] + red[1][t][lane] + red[2][t][lane];
    return acc;
}

__global__ __launch_bounds__(256) void k_gram_real(const double* __restrict__ Z, int ldz, int m, int n,
                                                   double* __restrict__ C) {
    __shared__ double red[3][4][64];
    const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63, l16 = lane & 15, l4 = lane >> 4;
    const int i0 = (int)blockIdx.x * 16, j0 = (int)blockIdx.y * 16;
    const double *a = Z + (size_t)min(i0 + l16, n - 1) * ldz, *b = Z + (size_t)min(j0 + l16, n - 1) * ldz;
    wy_v4d acc{0, 0, 0, 0};
    int r0 = 16 * wave;
#pragma unroll 4
    for (; r0 + 16 <= m; r0 += 64)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int r = r0 + 4 * l4 + t;
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[r], b[r], acc, 0, 0, 0);
        }
    if (r0 < m)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int r = r0 + 4 * l4 + t, rc = min(r, m - 1);
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(r < m ? a[rc] : 0.0, b[rc], acc, 0, 0, 0);
        }
    acc = tile_sum(acc, red, wave, lane);
    if (wave == 0 && j0 + l16 < n)
#pragma unroll
        for (int t = 0; t < 4; ++t)
            if (i0 + l4 + 4 * t < n) C[(size_t)(i0 + l4 + 4 * t) * n + j0 + l16] = acc[t];  // C is symmetric
}

__global__ __launch_bounds__(256) void k_ns_update(const double* __restrict__ Z, int ldz, int m, int n,
                                                   const double* __restrict__ C, double* __restrict__ out) {
    __shared__ double red[3][4][64];
    const int wave = (int)threadIdx.x >> 6, lane = (int)threadIdx.x & 63, l16 = lane & 15, l4 = lane >> 4;
    const int r = (int)blockIdx.x * 16 + l16, j0 = (int)blockIdx.y * 16;
    const double *c = C + (size_t)min(j0 + l16, n - 1) * n, *z = Z + min(r, m - 1);
    wy_v4d acc{0, 0, 0, 0};
    int k0 = 16 * wave;
#pragma unroll 2
    for (; k0 + 16 <= n; k0 += 64)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int k = k0 + 4 * l4 + t;
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(c[k], z[(size_t)k * ldz], acc, 0, 0, 0);
        }
    if (k0 < n)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int k = k0 + 4 * l4 + t, kc = min(k, n - 1);
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(k < n ? c[kc] : 0.0, z[(size_t)kc * ldz], acc, 0, 0, 0);
        }
    acc = tile_sum(acc, red, wave, lane);
    if (wave == 0 && r < m)
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int j = j0 + l4 + 4 * t;
            if (j < n) out[(size_t)j * ldz + r] = 1.5 * Z[(size_t)j * ldz + r] - 0.5 * acc[t];
        }
}

// Two values' lane exchange and sum (see swap_add): the first value's pairs land in the even lane
// rows (the lower half), the second's in the odd ones (the upper half).
template <int ROWS>
__device__ __forceinline__ double swap_add2(double a, double b) {
    const unsigned al = (unsigned)__double2loint(a), ah = (unsigned)__double2hiint(a);
    const unsigned bl = (unsigned)__double2loint(b), bh = (unsigned)__double2hiint(b);
    if constexpr (ROWS == 1) {
        const auto l = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
        const auto h = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
        return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
    } else {
        const auto l = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
        const auto h = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
        return __hiloint2double((int)h[0], (int)l[0]) + __hiloint2double((int)h[1], (int)l[1]);
    }
}

// Y[:, col] = Q Z[:, col] = H_0 (H_1 (... H_{m-2} Z[:, col])), one workgroup per column, one block of
// reflectors after another from the last: u = V^H y, y -= W u.  Thread t holds one row of each row
// group of y; V and W of the next two blocks are in flight while one is applied (all workgroups read
// a block at about the same time, so its first reader on an XCD waits for memory).  The chain is one workgroup sum per kWyNb reflectors, where one reflector at a time (a
// wavefront per column) took a wavefront sum each; V and W (16 m^2 bytes between them) stream through
// every CU from L2, which sets the floor (m = 648: 45 us).  nev = 160, m = 164 / 648:
// 109 -> 26 us and 918 -> 157 us (and the compact form, 11 and 30 us alone, beside the eigenvalues).
template <int NQ, int NW>
struct ApplyQ {
    static constexpr int GR = 64 * NW;  // rows of one group (one per thread)
    const double2 *vh, *w;
    int m;
    double (*red)[2 * kWyNb][NW];  // [block parity][reflector, real and imaginary][wavefront]
    int wv, lane;
    int row[NQ];  // rows from m on read row 0, which is zero in V and W
    double2 y[NQ];
    double2 va[kWyNb][NQ], wa[kWyNb][NQ], vb[kWyNb][NQ], wb[kWyNb][NQ];

    // Rows of groups Q0 and up of the block from k0 (columns past the last reflector's are zero).
    template <int Q0, int Q1>
    __device__ __forceinline__ void fetch(const double2* src, double2 (&dst)[kWyNb][NQ], int k0) {
#pragma unroll
        for (int i = 0; i < kWyNb; ++i) {
            const double2* c = src + (size_t)min(k0 + i, m - 1) * m;
#pragma unroll
            for (int q = Q0; q < Q1; ++q) dst[i][q] = c[row[q]];
        }
    }

    template <int Q0, int Q1>
    __device__ __forceinline__ void load(int kb) {
        fetch<Q0, Q1>(vh, va, kb + kWyNb);
        fetch<Q0, Q1>(w, wa, kb + kWyNb);
        fetch<Q0, Q1>(vh, vb, kb);
        fetch<Q0, Q1>(w, wb, kb);
    }

    // One block from its registers, which the block `next` takes over as they fall free.
    template <int QB>
    __device__ __forceinline__ void block(double2 (&v)[kWyNb][NQ], double2 (&u)[kWyNb][NQ], int par, int next) {
        double acc[2 * kWyNb];
#pragma unroll
        for (int i = 0; i < kWyNb; ++i) {
            acc[2 * i] = acc[2 * i + 1] = 0.0;
#pragma unroll
            for (int q = QB; q < NQ; ++q) {
                const double2 p = cjm(v[i][q], y[q]);
                acc[2 * i] += p.x;
                acc[2 * i + 1] += p.y;
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // the loads below go into registers just read
        fetch<QB, NQ>(vh, v, next);
        __builtin_amdgcn_sched_barrier(0);
        // Sixteen sums at once: halves, then lane rows, hold different values; register i's lane
        // rows 0..3 end with values 4 i + 0, 2, 1, 3.
#pragma unroll
        for (int i = 0; i < kWyNb; ++i) acc[i] = swap_add2<2>(acc[2 * i], acc[2 * i + 1]);
#pragma unroll
        for (int i = 0; i < kWyNb / 2; ++i) {
            double s = swap_add2<1>(acc[2 * i], acc[2 * i + 1]);
            s += dpp_rot<0x128>(s);
            s += dpp_rot<0x124>(s);
            s += dpp_rot<0x122>(s);
            s += dpp_rot<0x121>(s);
            acc[i] = s;
        }
        const int lr = lane >> 4, first = lr == 1 ? 2 : lr == 2 ? 1 : lr;
        if ((lane & 15) == 0) {
#pragma unroll
            for (int i = 0; i < kWyNb / 2; ++i) red[par][4 * i + first][wv] = acc[i];
        }
        __syncthreads();
        // Lane l adds the wavefronts' shares of value l; every lane then takes them from there.
        double c = red[par][lane & (2 * kWyNb - 1)][0];
#pragma unroll
        for (int q = 1; q < NW; ++q) c += red[par][lane & (2 * kWyNb - 1)][q];
#pragma unroll
        for (int i = 0; i < kWyNb; ++i) {
            const double2 ci = make_double2(read_lane(c, 2 * i), read_lane(c, 2 * i + 1));
#pragma unroll
            for (int q = QB; q < NQ; ++q) {
                const double2 d = cm(u[i][q], ci);
                y[q].x -= d.x;
                y[q].y -= d.y;
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch<QB, NQ>(w, u, next);
        __builtin_amdgcn_sched_barrier(0);
    }

    // Pairs of blocks that start in row group QB, from the last; then the groups above it.
    template <int QB>
    __device__ __forceinline__ void run(int last) {
        constexpr int PB = 2 * kWyNb;
        int kb = min(last, GR * QB + GR - PB);
        if (kb >= GR * QB) {
            // Group QB joins here: its rows of the pair already in flight.
            if (kb == last) load<QB, NQ>(kb);
            else load<QB, QB + 1>(kb);
            for (; kb >= GR * QB; kb -= PB) {
                const int next = max(kb - PB, 0);  // past the last pair: loaded, not used
                block<QB>(va, wa, 1, next + kWyNb);
                block<QB>(vb, wb, 0, next);
            }
        }
        if constexpr (QB > 0) run<QB - 1>(last);
    }
};

template <int NQ, int NW>
__global__ __launch_bounds__(64 * NW, 1) void k_apply_q(const double2* __restrict__ vh, const double2* __restrict__ w,
                                                        int m, const double* __restrict__ Z, int ldz,
                                                        double2* __restrict__ Y, int ldy) {
    __shared__ __align__(16) double red[2][2 * kWyNb][NW];
    const int t = (int)threadIdx.x, col = (int)blockIdx.x;
    ApplyQ<NQ, NW> k{vh, w, m, red, t >> 6, t & 63};
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int r = t + 64 * NW * q;
        k.row[q] = r < m ? r : 0;
        k.y[q] = make_double2(r < m ? Z[(size_t)col * ldz + r] : 0.0, 0.0);
#pragma unroll
        for (int i = 0; i < kWyNb; ++i) k.va[i][q] = k.wa[i][q] = k.vb[i][q] = k.wb[i][q] = make_double2(0.0, 0.0);
    }
    if (m > 1) k.template run<NQ - 1>((m - 2) / (2 * kWyNb) * 2 * kWyNb);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int r = t + 64 * NW * q;
        if (r < m) Y[(size_t)col * ldy + r] = k.y[q];
    }
}

// The instance and its wavefronts.  Above 768 rows two blocks' V and W take all registers of eight
// wavefronts, which spill 94 of them; four wavefronts would hold twice as much each.  Whole calls there
// against one wavefront per eigenvector and one reflector at a time: m = 1,000, 160 vectors 11,829 -> 5,914
// us, all 14,219 -> 8,971 us.
const void* apply_q_kernel(int m, int* waves) {
    *waves = m <= 768 ? 4 : 8;
    if (m <= 256) return (const void*)k_apply_q<1, 4>;
    if (m <= 512) return (const void*)k_apply_q<2, 4>;
    if (m <= 768) return (const void*)k_apply_q<3, 4>;
    return (const void*)k_apply_q<2, 8>;
}

size_t stein_lds_bytes(int m) { return (size_t)8 * (stein_rows(m) + kSteinBlock) * sizeof(double); }

// One instance of the tridiagonalisation: m <= 64 nq rows, cw columns per wavefront.
struct TrdKernel {
    int nq, cw;
    const void* fn;
    size_t lds() const { return (size_t)4 * 64 * nq * sizeof(double2); }
};
#define DZ_TRD_ENTRY(NQ, CW) {NQ, CW, (const void*)k_hetrd<NQ, CW>},
const TrdKernel kTrdKernels[] = {DZ_TRD_INSTANCES(DZ_TRD_ENTRY)};
#undef DZ_TRD_ENTRY

// Co-resident workgroups per device for the tridiagonalisation (one per CU at its LDS size),
// queried once per device.
struct CoopInfo {
    int groups = 0;
    int cols_per_group = 0;
};
std::mutex g_coop_mu;
CoopInfo g_coop[64];

CoopInfo coop_info(int dev) {
    DZ_REQUIRE(dev >= 0 && dev < 64, DZHIP_ERR_ARG, "device index out of range");
    std::lock_guard<std::mutex> lk(g_coop_mu);
    CoopInfo& c = g_coop[dev];
    if (c.groups == 0) {
        int cus = 0, coop = 0;
        DZ_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        DZ_HIP(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev));
        DZ_REQUIRE(coop != 0, DZHIP_ERR_HIP, "device does not support cooperative launches");
        for (const TrdKernel& k : kTrdKernels) set_max_dynamic_lds(k.fn, k.lds());
        set_max_dynamic_lds((const void*)k_stein, stein_lds_bytes(kHeevMaxM));
        set_max_dynamic_lds((const void*)k_stein_cluster, stein_lds_bytes(kHeevMaxM));
        // Launch-shape override: at least so many trailing columns per workgroup (4, 8 or 16).
        if (const char* env = std::getenv("DZHIP_HEEV_COLS")) c.cols_per_group = std::max(0, std::atoi(env));
        c.groups = cus;
    }
    return c;
}

// Launch shape of the tridiagonalisation: the instance and its G workgroups (trd_pick).  On 256 CUs every
// size takes one column per wavefront; whole eigensolver calls with one / two of them, us: m = 164
// 577 / 626, 328 1,420 / 1,547, 648 (300 vectors) 3,152 / 3,718.  This kernel alone at one: 1,024 -> 400 us
// at m = 164 and 4,887 -> 2,150 us at m = 648 (6.2 -> 2.4 and 7.5 -> 3.3 us a reflector) against columns in
// LDS shared by four wavefronts with block sums and a grid barrier.
TrdKernel trd_shape(int m, int* G_out) {
    int dev = 0;
    DZ_HIP(hipGetDevice(&dev));
    const CoopInfo ci = coop_info(dev);
    const TrdPick p = trd_pick(m, ci.groups, ci.cols_per_group);
    const TrdKernel* k = nullptr;
    for (const TrdKernel& c : kTrdKernels)
        if (c.nq == p.nq && c.cw == p.cw) k = &c;
    DZ_REQUIRE(k, DZHIP_ERR_ARG, "Hermitian eigensolver: matrix too large for the tridiagonalisation");
    // Every workgroup must be co-resident.
    int per_cu = 0;
    DZ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k->fn, 64 * kTrdWaves, k->lds()));
    DZ_REQUIRE(per_cu >= 1, DZHIP_ERR_HIP, "Hermitian eigensolver: grid does not fit on the device");
    *G_out = p.groups;
    return *k;
}

// Device buffers of one eigensolver call (from a HeevWork, or carved from the static scratch array).
struct HeevBufs {
    double2 *vh, *tau;
    double *pub;  // 2 m^2: the tridiagonalisation's exchange
    double *d, *e, *z, *zt, *gram;
    int* err;
};

// The tridiagonalisation gate of each device (see TrdAdmission): CUs per XCD taken by admitted
// grids, out of cap.
constexpr int kXcds = 8;
struct TrdGate {
    std::mutex mu;
    std::condition_variable cv;
    int used = 0, cap = 0;
};
TrdGate g_trd_gate[64];

int trd_units(int G) { return (G + kXcds - 1) / kXcds; }

void trd_gate_acquire(int dev, int units) {
    TrdGate& gt = g_trd_gate[dev];
    std::unique_lock<std::mutex> lk(gt.mu);
    if (gt.cap == 0) {
        int cus = 0;
        DZ_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        gt.cap = std::max(1, cus / kXcds);
    }
    DZ_REQUIRE(units >= 1 && units <= gt.cap, DZHIP_ERR_HIP, "Hermitian eigensolver: grid does not fit on the device");
    gt.cv.wait(lk, [&] { return gt.used + units <= gt.cap; });
    gt.used += units;
}

void trd_gate_release(int dev, int units) {
    TrdGate& gt = g_trd_gate[dev];
    {
        std::lock_guard<std::mutex> lk(gt.mu);
        gt.used -= units;
    }
    gt.cv.notify_all();
}

// Ordinary rather than cooperative launches of the gated tridiagonalisation; DZHIP_HEEV_COOP=1
// forces the cooperative launch everywhere (for comparisons).
bool trd_gated_enabled() {
    static const bool on = [] {
        const char* env = std::getenv("DZHIP_HEEV_COOP");
        return !(env && std::atoi(env) != 0);
    }();
    return on;
}

// Spin limit of admitted launches; DZHIP_HEEV_SHARED_SPIN overrides it (a test sets 1 so that the
// exchange gives up at once and the cooperative repeat runs).
unsigned shared_spin_limit() {
    static const unsigned v = [] {
        const char* env = std::getenv("DZHIP_HEEV_SHARED_SPIN");
        return env ? (unsigned)std::max(1, std::atoi(env)) : kSpinLimitShared;
    }();
    return v;
}

void run_tridiag(const HeevBufs& b, const TrdKernel& k, int G, const double2* A, int lda, int m, hipStream_t s,
                 bool cooperative = true) {
    // The exchange's entries unset, the reflectors zero and the error flag cleared by a kernel (not a memset node) on the
    // same stream.
    const size_t npub = (size_t)m * m;
    hipLaunchKernelGGL(k_trd_init, dim3((unsigned)((npub + 255) / 256)), dim3(256), 0, s,
                       reinterpret_cast<ulonglong2*>(b.pub), b.vh, npub, b.err);
    DZ_HIP(hipGetLastError());
    TrdArgs args{A, lda, m, b.vh, b.tau, b.d, b.e, b.pub, b.err, cooperative ? kSpinLimit : shared_spin_limit()};
    void* kargs[] = {&args};
    if (cooperative && G > 1) {
        DZ_HIP(hipLaunchCooperativeKernel(k.fn, dim3((unsigned)G), dim3(64u * kTrdWaves), kargs, (unsigned)k.lds(), s));
    } else {
        DZ_HIP(hipLaunchKernel(k.fn, dim3((unsigned)G), dim3(64u * kTrdWaves), kargs, k.lds(), s));
    }
}

void run_eig(const HeevBufs& b, int m, int nev, double* w_dev, double2* Y, int ldy, hipStream_t s) {
    double* scal = b.gram + (size_t)nev * nev;
    // W takes the exchange buffer, which the tridiagonalisation has done with.
    double2* wy = reinterpret_cast<double2*>(b.pub);
    const int groups = (m - 1 + 2 * kWyNb - 1) / (2 * kWyNb);
    hipLaunchKernelGGL(k_stebz, dim3((unsigned)(nev + groups)), dim3(256), std::max(m * (int)sizeof(double2), kWyLds), s,
                       b.d, b.e, m, nev, w_dev, scal, b.err, b.vh, b.tau, wy);
    DZ_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_stein, dim3((unsigned)nev), dim3(64), stein_lds_bytes(m), s, b.d, b.e, m, nev, w_dev, scal,
                       b.z, m);
    DZ_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_stein_cluster, dim3((unsigned)nev), dim3(256), stein_lds_bytes(m), s, b.d, b.e, w_dev, scal, nev, m,
                       b.z, m);
    DZ_HIP(hipGetLastError());
    double* zc = b.z;
    double* zn = b.zt;
    for (int it = 0; it < 2; ++it) {
        hipLaunchKernelGGL(k_gram_real, dim3((unsigned)((nev + 15) / 16), (unsigned)((nev + 15) / 16)), dim3(256), 0, s,
                           zc, m, m, nev, b.gram);
        DZ_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_ns_update, dim3((unsigned)((m + 15) / 16), (unsigned)((nev + 15) / 16)), dim3(256), 0, s, zc, m, m,
                           nev, b.gram, zn);
        DZ_HIP(hipGetLastError());
        std::swap(zc, zn);
    }
    {
        const double2* vh = b.vh;
        const double2* w = wy;
        const double* zcc = zc;
        int mm = m, ldz = m, ldyy = ldy, waves = 4;
        const void* fn = apply_q_kernel(m, &waves);
        void* kargs[] = {&vh, &w, &mm, &zcc, &ldz, &Y, &ldyy};
        DZ_HIP(hipLaunchKernel(fn, dim3((unsigned)nev), dim3(64u * waves), kargs, 0, s));
    }
    DZ_HIP(hipGetLastError());
}

HeevBufs work_bufs(HeevWork& w, int m, int nev) {
    w.vh.ensure((size_t)m * m * sizeof(double2));
    w.tau.ensure((size_t)m * sizeof(double2));
    w.d.ensure((size_t)m * sizeof(double));
    w.e.ensure((size_t)m * sizeof(double));
    w.pub.ensure((size_t)m * m * sizeof(double2));
    w.err.ensure(64);
    if (nev > 0) {
        w.z.ensure((size_t)m * nev * sizeof(double));
        w.zt.ensure((size_t)m * nev * sizeof(double));
        w.gram.ensure((size_t)nev * nev * sizeof(double) + 64);
    }
    return HeevBufs{w.vh.as<double2>(), w.tau.as<double2>(), w.pub.as<double>(), w.d.as<double>(),   w.e.as<double>(),
                    w.z.as<double>(),   w.zt.as<double>(),   w.gram.as<double>(), w.err.as<int>()};
}

// ----------------------------------------------------------------- allocation-free variant
// A file-scope device array holds every buffer of an eigensolver call of m <= kHeevNoAllocMaxM, for
// callers that cannot allocate.  Its device address is taken once per device at set-up
// (heev_scratch_init, from dzhip_ctx_create with the device current) and only that address is used
// on the host.  Calls that overlap on one device share the array and race.
constexpr size_t kHeevNoAllocBytes = 6u << 20;
static __device__ __align__(256) unsigned char scratch[kHeevNoAllocBytes];
std::mutex g_scratch_mu;
void* g_scratch_ptr[64] = {};

size_t carve(size_t& off, size_t bytes) {
    const size_t at = off;
    off = round_up(off + bytes, 256);
    return at;
}

// Offsets of the buffers in the scratch for (m, nev); returns the bytes needed.
size_t scratch_layout(int m, int nev, size_t out[9]) {
    size_t off = 0;
    out[0] = carve(off, (size_t)m * m * sizeof(double2));       // vh
    out[1] = carve(off, (size_t)m * sizeof(double2));           // tau
    out[2] = carve(off, (size_t)m * m * sizeof(double2));       // pub
    out[3] = carve(off, (size_t)m * sizeof(double));            // d
    out[4] = carve(off, (size_t)m * sizeof(double));            // e
    out[5] = carve(off, (size_t)m * nev * sizeof(double));      // z
    out[6] = carve(off, (size_t)m * nev * sizeof(double));      // zt
    out[7] = carve(off, (size_t)nev * nev * sizeof(double) + 64);  // gram + scale
    out[8] = carve(off, 64);                                    // error flag
    return off;
}

}  // namespace

void heev_scratch_init(int device) {
    DZ_REQUIRE(device >= 0 && device < 64, DZHIP_ERR_ARG, "device index out of range");
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[device]) return;
    void* ptr = nullptr;
    DZ_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    DZ_REQUIRE(ptr != nullptr, DZHIP_ERR_HIP, "no device address for the eigensolver scratch");
    g_scratch_ptr[device] = ptr;
}

void heev_lowest_noalloc(int device, const double2* A, int lda, int m, int nev, double* w_dev, double2* Y, int ldy,
                         hipStream_t s) {
    DZ_REQUIRE(m >= 1 && m <= kHeevNoAllocMaxM && nev >= 1 && nev <= m && lda >= m && ldy >= m, DZHIP_ERR_ARG,
               "allocation-free Hermitian eigensolver: need 1 <= nev <= m <= 256 (its scratch is 6 MiB) and "
               "leading dimensions >= m");
    void* base = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        base = device >= 0 && device < 64 ? g_scratch_ptr[device] : nullptr;
    }
    DZ_REQUIRE(base, DZHIP_ERR_STATE, "eigensolver scratch not set up on this device (dzhip_ctx_create)");
    int G = 1;
    const TrdKernel k = trd_shape(m, &G);
    size_t off[9];
    const size_t need = scratch_layout(m, nev, off);
    DZ_REQUIRE(need <= kHeevNoAllocBytes, DZHIP_ERR_ARG, "allocation-free Hermitian eigensolver: scratch too small");
    unsigned char* p = static_cast<unsigned char*>(base);
    const HeevBufs b{reinterpret_cast<double2*>(p + off[0]), reinterpret_cast<double2*>(p + off[1]),
                     reinterpret_cast<double*>(p + off[2]),  reinterpret_cast<double*>(p + off[3]),
                     reinterpret_cast<double*>(p + off[4]),  reinterpret_cast<double*>(p + off[5]),
                     reinterpret_cast<double*>(p + off[6]),  reinterpret_cast<double*>(p + off[7]),
                     reinterpret_cast<int*>(p + off[8])};
    run_tridiag(b, k, G, A, lda, m, s);
    run_eig(b, m, nev, w_dev, Y, ldy, s);
}

void HeevWork::release() {
    DevBuf* bufs[] = {&vh, &tau, &d, &e, &pub, &err, &z, &zt, &gram};
    for (DevBuf* b : bufs) b->release();
    if (flag) (void)hipHostFree(flag);
    flag = nullptr;
}

void heev_tridiag_only(HeevWork& w, const double2* A, int lda, int m, hipStream_t s) {
    DZ_REQUIRE(m >= 1 && m <= kHeevMaxM && lda >= m, DZHIP_ERR_ARG, "Hermitian eigensolver: bad size");
    int G = 1;
    const TrdKernel k = trd_shape(m, &G);
    run_tridiag(work_bufs(w, m, 0), k, G, A, lda, m, s);
}

TrdAdmission::~TrdAdmission() {
    if (units <= 0) return;
    (void)hipStreamSynchronize(stream);
    trd_gate_release(device, units);
}

void heev_lowest(HeevWork& w, const double2* A, int lda, int m, int nev, double* w_dev, double2* Y, int ldy,
                 hipStream_t s, TrdAdmission* adm) {
    DZ_REQUIRE(m >= 1 && m <= kHeevMaxM && nev >= 1 && nev <= m && lda >= m && ldy >= m, DZHIP_ERR_ARG,
               "Hermitian eigensolver: need 1 <= nev <= m <= 1024 and leading dimensions >= m");
    int G = 1;
    const TrdKernel k = trd_shape(m, &G);
    const HeevBufs b = work_bufs(w, m, nev);
    if (adm && trd_gated_enabled()) {
        DZ_REQUIRE(adm->units == 0, DZHIP_ERR_STATE, "Hermitian eigensolver: admission already held");
        int dev = 0;
        DZ_HIP(hipGetDevice(&dev));
        DZ_REQUIRE(dev >= 0 && dev < 64, DZHIP_ERR_ARG, "device index out of range");
        const int units = trd_units(G);
        trd_gate_acquire(dev, units);
        adm->device = dev;
        adm->units = units;
        adm->stream = s;
        run_tridiag(b, k, G, A, lda, m, s, false);
    } else {
        run_tridiag(b, k, G, A, lda, m, s);
    }
    run_eig(b, m, nev, w_dev, Y, ldy, s);
}

std::atomic<unsigned long long> g_trd_retries{0};

void heev_lowest_shared(HeevWork& w, const double2* A, int lda, int m, int nev, double* w_dev, double2* Y, int ldy,
                        hipStream_t s) {
    {
        TrdAdmission adm;
        heev_lowest(w, A, lda, m, nev, w_dev, Y, ldy, s, &adm);
        if (heev_error_flag(w, s) == 0) return;  // synchronises s
    }
    // The admitted grid gave up waiting for its workgroups (A is unchanged): cooperative launch.
    g_trd_retries.fetch_add(1, std::memory_order_relaxed);
    heev_lowest(w, A, lda, m, nev, w_dev, Y, ldy, s);
    DZ_REQUIRE(heev_error_flag(w, s) == 0, DZHIP_ERR_HIP,
               "Hermitian eigensolver: tridiagonalisation barrier did not complete");
}

unsigned long long heev_shared_retries() { return g_trd_retries.load(std::memory_order_relaxed); }

int heev_error_flag(HeevWork& w, hipStream_t s) {
    if (!w.err.ptr) return 0;
    if (!w.flag) DZ_HIP(hipHostMalloc(reinterpret_cast<void**>(&w.flag), sizeof(int), hipHostMallocDefault));
    DZ_HIP(hipMemcpyAsync(w.flag, w.err.ptr, sizeof(int), hipMemcpyDeviceToHost, s));
    DZ_HIP(hipStreamSynchronize(s));
    return *w.flag;
}

}  // namespace dzhip
