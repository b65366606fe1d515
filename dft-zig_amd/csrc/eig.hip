// Device-resident block eigensolver for H x = lambda x (S = I) on one k-point.
//
// Follows the reference's block-Davidson ("LOBPCG" there,
// src/features/linalg/lobpcg/serial.zig:55-307) in its outer semantics: subspace grows from
// block = nbands + 4 by appending preconditioned residuals of the unconverged bands, up to
// max_subspace = min(n, 4 nbands + 8); converged when max_b ||H x_b - lambda_b x_b||_2 < tol
// or when no vector can be added; kinetic-shift preconditioner r / (diag - lambda) with
// |denominator| clamped at 1e-8 (common.zig:214-226); random start from the reference LCG
// (common.zig:287-319, seed 0x6f3d3cbe).  The block operations are re-designed for the GPU:
//   * new vectors are orthogonalised against the basis with two passes of block classical
//     Gram-Schmidt (GEMMs) and orthonormalised with Cholesky QR (in place of one-vector MGS);
//   * the projected matrix T = V^H H V is extended by the new columns only;
//   * Rayleigh-Ritz takes the lowest nbands eigenpairs of T with the library's own device
//     Hermitian eigensolver (heev.hip: one-launch tridiagonalisation, multisection, inverse
//     iteration), rocSOLVER zheevd only for subspaces above 1024;
//   * a full subspace restarts from [Ritz vectors, new block], reusing H x = W c (no H applies
//     are discarded).
// All subspace algebra is FP64.  In mixed mode the H apply runs in FP32 until the largest
// residual falls below `mixed_switch_tol`, then the basis restarts from the Ritz vectors with an
// FP64 apply, so the final eigenpairs are those of the FP64 operator.
#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <vector>

#include "ham.h"
#include "heev.h"
#include "herm3.h"

namespace dzhip {

#define DZ_BLAS(call)                                                                           \
    do {                                                                                        \
        rocblas_status st_ = (call);                                                            \
        if (st_ != rocblas_status_success)                                                      \
            throw Error{DZHIP_ERR_HIP, std::string(#call) + ": " + rocblas_status_to_string(st_)}; \
    } while (0)

using zc = rocblas_double_complex;

// ----------------------------------------------------------------- kernels
__global__ void k_col_norm2(const double2* __restrict__ v, size_t ld, int n, double* __restrict__ out) {
    __shared__ double red[256];
    const double2* c = v + (size_t)blockIdx.x * ld;
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += c[i].x * c[i].x + c[i].y * c[i].y;
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}

// R[:, b] = HX[:, b] - lambda_b X[:, b]
__global__ void k_residual(const double2* __restrict__ hx, const double2* __restrict__ x,
                           const double* __restrict__ lam, double2* __restrict__ r, size_t ld, int n) {
    const int b = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t o = (size_t)b * ld + i;
    const double l = lam[b];
    r[o] = make_double2(hx[o].x - l * x[o].x, hx[o].y - l * x[o].y);
}

// Q[:, j] = P(R[:, sel_j]): kinetic shift r / (diag - lambda) with the reference's 1e-8 clamp,
// or Teter-Payne-Allan K(x) r with x = diag / ekin_b (ekin = <x_b|T|x_b>).
__global__ void k_precondition(const double2* __restrict__ r, const int* __restrict__ sel,
                               const double* __restrict__ lam, const double* __restrict__ ekin,
                               const double* __restrict__ diag, double2* __restrict__ q, size_t ld,
                               int n, int mode) {
    const int j = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int b = sel[j];
    const double2 v = r[(size_t)b * ld + i];
    const double f = mode == 0 ? precond_kinetic_shift(diag[i], lam[b]) : precond_tpa(diag[i], ekin[b]);
    q[(size_t)j * ld + i] = make_double2(v.x * f, v.y * f);
}

// ----------------------------------------------------------------- basis products
// The solver's tall-skinny products (n = n_pw rows, up to a few hundred columns), where the library
// GEMM runs at a few TF/s.  A tile is WX wavefronts of 16 columns of A (Gram) or 16 rows (basis times
// coefficients) by JB blocks of 16 columns of the other side, the same for each, on the FP64 matrix
// cores (16x16x4) with each complex product as three real ones.  K runs in stages of 8 through two
// LDS buffers: the next stage's loads are in flight (unmasked, from clamped addresses; what lies
// beyond the end is zeroed on its way to LDS) while one is multiplied, with one barrier a stage, and
// two workgroups share a CU.  The matrix cores' rate bounds the large shapes, latency the small
// ones.  Before: 64 x 64 tiles whose loads were masked, and so waited for, ahead of the products.  Gram /
// basis products of a Si-64 solve (n = 23,984, medians over m = 164..648) 173 / 376 -> 147 / 219 us, of a
// Si-8 solve (n = 1,637, 20 bands) 23 / 13 -> 5 / 8 us.
typedef double v4d_t __attribute__((ext_vector_type(4)));
constexpr int kBpK = 8, kBpPitch = kBpK + 1, kBpMaxBlocks = 6;

// Column blocks of one tile and the tiles of N columns.
static void bp_tiles(int N, int* jb, int* tiles) {
    const int nbk = (N + 15) / 16;
    *tiles = (nbk + kBpMaxBlocks - 1) / kBpMaxBlocks;
    *jb = (nbk + *tiles - 1) / *tiles;
}

// partial[ks][j][i] = sum over K-chunk ks of conj(A[k][i]) B[k][j]; k_gram_reduce adds the chunks.
template <int WX, int JB>
__global__ __launch_bounds__(64 * WX, 2) void k_gram_cn(const double2* __restrict__ A, int lda, int M,
                                                        const double2* __restrict__ B, int ldb, int N, int K, int kchunk,
                                                        int mtiles, double2* __restrict__ partial) {
    constexpr int NT = 64 * WX, AR = 16 * WX, BR = 16 * JB;
    constexpr int AP = (AR * kBpK + NT - 1) / NT, BP = (BR * kBpK + NT - 1) / NT;
    __shared__ double2 lds[2][(AR + BR) * kBpPitch];
    const int mt = blockIdx.x % mtiles, ks = blockIdx.x / mtiles;
    const int i_base = mt * AR, j_base = blockIdx.y * BR;
    const int k0 = ks * kchunk, k1 = min(K, k0 + kchunk);
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int l16 = lane & 15, l4 = lane >> 4;
    double2 ar[AP], br[BP];
    auto fetch = [&](int kt) {
#pragma unroll
        for (int q = 0; q < AP; ++q) {
            const int e = tid + q * NT;
            ar[q] = A[(size_t)min(i_base + e / kBpK, M - 1) * lda + min(kt + e % kBpK, k1 - 1)];
        }
#pragma unroll
        for (int q = 0; q < BP; ++q) {
            const int e = tid + q * NT;
            br[q] = B[(size_t)min(j_base + e / kBpK, N - 1) * ldb + min(kt + e % kBpK, k1 - 1)];
        }
    };
    auto stash = [&](double2* st, int kt) {
        const bool tail = kt + kBpK > k1;
#pragma unroll
        for (int q = 0; q < AP; ++q) {
            const int e = tid + q * NT;
            if (tail && kt + e % kBpK >= k1) ar[q] = make_double2(0.0, 0.0);
            if (e < AR * kBpK) st[(e / kBpK) * kBpPitch + e % kBpK] = ar[q];
        }
#pragma unroll
        for (int q = 0; q < BP; ++q) {
            const int e = tid + q * NT;
            if (tail && kt + e % kBpK >= k1) br[q] = make_double2(0.0, 0.0);
            if (e < BR * kBpK) st[(AR + e / kBpK) * kBpPitch + e % kBpK] = br[q];
        }
    };
    // conj(a) b = (ar br + ai bi) + i (ar bi - ai br) by three real MFMAs (Gauss):
    // p1 = sum ar br, p2 = sum ai bi, p3 = sum (ar - ai)(br + bi); Re = p1 + p2, Im = p3 - p1 + p2.
    v4d_t p1[JB], p2[JB], p3[JB];
#pragma unroll
    for (int y = 0; y < JB; ++y) p1[y] = p2[y] = p3[y] = v4d_t{0, 0, 0, 0};
    fetch(k0);
    stash(lds[0], k0);
    __syncthreads();
    int buf = 0;
    for (int kt = k0; kt < k1; kt += kBpK, buf ^= 1) {
        const bool more = kt + kBpK < k1;
        if (more) fetch(kt + kBpK);
        __builtin_amdgcn_sched_barrier(0);  // the loads go out first
        const double2* as = lds[buf] + (wave * 16 + l16) * kBpPitch + l4;
        const double2* bs = lds[buf] + (AR + l16) * kBpPitch + l4;
#pragma unroll
        for (int kk = 0; kk < kBpK; kk += 4) {
            const double2 a = as[kk];
            const double adif = a.x - a.y;
#pragma unroll
            for (int y = 0; y < JB; ++y) {
                const double2 b = bs[y * 16 * kBpPitch + kk];
                p1[y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, p1[y], 0, 0, 0);
                p2[y] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.y, p2[y], 0, 0, 0);
                p3[y] = __builtin_amdgcn_mfma_f64_16x16x4f64(adif, b.x + b.y, p3[y], 0, 0, 0);
            }
        }
        // The other buffer was last read before the barrier that ended the previous stage.
        if (more) stash(lds[buf ^ 1], kt + kBpK);
        __syncthreads();
    }
    // D slot r of a 16x16 block: row (l/16) + 4 r, column l % 16.
#pragma unroll
    for (int y = 0; y < JB; ++y)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = i_base + wave * 16 + l4 + 4 * r;
            const int j = j_base + y * 16 + l16;
            const double a1 = p1[y][r], a2 = p2[y][r];
            if (i < M && j < N) partial[((size_t)ks * N + j) * M + i] = make_double2(a1 + a2, p3[y][r] - a1 + a2);
        }
}

// C[:, 0:N] = alpha A[:, 0:K] B[0:K, 0:N] + beta C, alpha and beta real: A is n x K (leading
// dimension lda), B is K x N (ldb), C is n x N (ldc), all column-major.  The MFMA computes
// C^T = B^T A^T so that a wavefront's accumulator slots hold 16 consecutive rows of a column of C
// (coalesced loads of the old C and stores).
template <int WX, int JB>
__global__ __launch_bounds__(64 * WX, 2) void k_gemm_nn(const double2* __restrict__ A, int lda,
                                                        const double2* __restrict__ B, int ldb, double2* __restrict__ C,
                                                        int ldc, int n, int K, int N, double alpha, double beta) {
    constexpr int NT = 64 * WX, RA = 16 * WX, RP = RA + 1, CB = 16 * JB;
    constexpr int AP = (RA * kBpK + NT - 1) / NT, BP = (CB * kBpK + NT - 1) / NT;
    __shared__ double2 la[2][kBpK * RP];        // [k][row]
    __shared__ double2 lb[2][CB * kBpPitch];    // [column][k]
    const int r_base = blockIdx.x * RA, c_base = blockIdx.y * CB;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int l16 = lane & 15, l4 = lane >> 4;
    double2 ar[AP], br[BP];
    auto fetch = [&](int kt) {
#pragma unroll
        for (int q = 0; q < AP; ++q) {  // consecutive threads read consecutive rows of one column
            const int e = tid + q * NT;
            ar[q] = A[(size_t)min(kt + e / RA, K - 1) * lda + min(r_base + e % RA, n - 1)];
        }
#pragma unroll
        for (int q = 0; q < BP; ++q) {
            const int e = tid + q * NT;
            br[q] = B[(size_t)min(c_base + e / kBpK, N - 1) * ldb + min(kt + e % kBpK, K - 1)];
        }
    };
    auto stash = [&](int st, int kt) {
        const bool tail = kt + kBpK > K;
#pragma unroll
        for (int q = 0; q < AP; ++q) {
            const int e = tid + q * NT;
            if (tail && kt + e / RA >= K) ar[q] = make_double2(0.0, 0.0);
            if (e < RA * kBpK) la[st][(e / RA) * RP + e % RA] = ar[q];
        }
#pragma unroll
        for (int q = 0; q < BP; ++q) {
            const int e = tid + q * NT;
            if (tail && kt + e % kBpK >= K) br[q] = make_double2(0.0, 0.0);
            if (e < CB * kBpK) lb[st][(e / kBpK) * kBpPitch + e % kBpK] = br[q];
        }
    };
    // b a = (br ar - bi ai) + i (br ai + bi ar): p1 = sum br ar, p2 = sum bi ai,
    // p3 = sum (br + bi)(ar + ai); Re = p1 - p2, Im = p3 - p1 - p2.
    v4d_t p1[JB], p2[JB], p3[JB];
#pragma unroll
    for (int x = 0; x < JB; ++x) p1[x] = p2[x] = p3[x] = v4d_t{0, 0, 0, 0};
    fetch(0);
    stash(0, 0);
    __syncthreads();
    int buf = 0;
    for (int kt = 0; kt < K; kt += kBpK, buf ^= 1) {
        const bool more = kt + kBpK < K;
        if (more) fetch(kt + kBpK);
        __builtin_amdgcn_sched_barrier(0);  // the loads go out first
        const double2* as = la[buf] + l4 * RP + wave * 16 + l16;
        const double2* bs = lb[buf] + l16 * kBpPitch + l4;
#pragma unroll
        for (int kk = 0; kk < kBpK; kk += 4) {
            const double2 a = as[kk * RP];
            const double asum = a.x + a.y;
            // Operand 0 (MFMA rows): columns of C; operand 1 (MFMA columns): rows of C.
#pragma unroll
            for (int x = 0; x < JB; ++x) {
                const double2 b = bs[x * 16 * kBpPitch + kk];
                p1[x] = __builtin_amdgcn_mfma_f64_16x16x4f64(b.x, a.x, p1[x], 0, 0, 0);
                p2[x] = __builtin_amdgcn_mfma_f64_16x16x4f64(b.y, a.y, p2[x], 0, 0, 0);
                p3[x] = __builtin_amdgcn_mfma_f64_16x16x4f64(b.x + b.y, asum, p3[x], 0, 0, 0);
            }
        }
        // The other buffer was last read before the barrier that ended the previous stage.
        if (more) stash(buf ^ 1, kt + kBpK);
        __syncthreads();
    }
    // Slot r of a 16x16 block: MFMA row (l/16) + 4 r = column of C, MFMA column l % 16 = row of C.
#pragma unroll
    for (int x = 0; x < JB; ++x)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int col = c_base + x * 16 + l4 + 4 * r;
            const int row = r_base + wave * 16 + l16;
            if (col < N && row < n) {
                const double a1 = p1[x][r], a2 = p2[x][r];
                double2 v = make_double2(alpha * (a1 - a2), alpha * (p3[x][r] - a1 - a2));
                double2* cp = C + (size_t)col * ldc + row;
                if (beta != 0.0) {
                    const double2 o = *cp;
                    v.x += beta * o.x;
                    v.y += beta * o.y;
                }
                *cp = v;
            }
        }
}

using GramFn = void (*)(const double2*, int, int, const double2*, int, int, int, int, int, double2*);
using GemmFn = void (*)(const double2*, int, const double2*, int, double2*, int, int, int, int, double, double);
template <int WX>
static GramFn gram_fn(int jb) {
    static const GramFn f[kBpMaxBlocks] = {k_gram_cn<WX, 1>, k_gram_cn<WX, 2>, k_gram_cn<WX, 3>,
                                           k_gram_cn<WX, 4>, k_gram_cn<WX, 5>, k_gram_cn<WX, 6>};
    return f[jb - 1];
}
template <int WX>
static GemmFn gemm_fn(int jb) {
    static const GemmFn f[kBpMaxBlocks] = {k_gemm_nn<WX, 1>, k_gemm_nn<WX, 2>, k_gemm_nn<WX, 3>,
                                           k_gemm_nn<WX, 4>, k_gemm_nn<WX, 5>, k_gemm_nn<WX, 6>};
    return f[jb - 1];
}

// C[j * ldc + i] = sum_ks partial[ks][j][i]
__global__ void k_gram_reduce(const double2* __restrict__ partial, int nks, int M, int N, double2* __restrict__ C,
                              int ldc) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int j = blockIdx.y;
    if (i >= M) return;
    double re = 0.0, im = 0.0;
#pragma unroll 8
    for (int ks = 0; ks < nks; ++ks) {
        const double2 v = partial[((size_t)ks * N + j) * M + i];
        re += v.x;
        im += v.y;
    }
    C[(size_t)j * ldc + i] = make_double2(re, im);
}

// p = r / (diag - lambda) with the 1e-8 clamp (single vector, CG).
__global__ void k_precondition_one(const double2* __restrict__ r, const double* __restrict__ diag, double lam,
                                   double2* __restrict__ p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double f = precond_kinetic_shift(diag[i], lam);
    p[i] = make_double2(r[i].x * f, r[i].y * f);
}

// out = c0 a + c1 b (+ c2 c), complex coefficients (CG Ritz update of psi and H psi).
__global__ void k_combine3(const double2* __restrict__ a, const double2* __restrict__ b,
                           const double2* __restrict__ c, double2 c0, double2 c1, double2 c2, int use_c,
                           double2* __restrict__ out, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double2 x = a[i], y = b[i];
    double re = c0.x * x.x - c0.y * x.y + c1.x * y.x - c1.y * y.y;
    double im = c0.x * x.y + c0.y * x.x + c1.x * y.y + c1.y * y.x;
    if (use_c) {
        const double2 z = c[i];
        re += c2.x * z.x - c2.y * z.y;
        im += c2.x * z.y + c2.y * z.x;
    }
    out[i] = make_double2(re, im);
}

// <x_b|T|x_b> = sum_G |k+G|^2 |x_bG|^2 (one workgroup per band)
__global__ void k_kinetic_energy(const double2* __restrict__ x, const double* __restrict__ diag, size_t ld,
                                 int n, double* __restrict__ out) {
    __shared__ double red[256];
    const double2* c = x + (size_t)blockIdx.x * ld;
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += blockDim.x) s += diag[i] * (c[i].x * c[i].x + c[i].y * c[i].y);
    red[threadIdx.x] = s;
    __syncthreads();
    for (int w = blockDim.x / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = red[0];
}

// dst[:, j] = src[:, idx_j] * scale_j
__global__ void k_gather_cols(const double2* __restrict__ src, const int* __restrict__ idx,
                              const double* __restrict__ scale, double2* __restrict__ dst, size_t ld, int n) {
    const int j = blockIdx.y;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double s = scale[j];
    const double2 v = src[(size_t)idx[j] * ld + i];
    dst[(size_t)j * ld + i] = make_double2(v.x * s, v.y * s);
}

// New directions to keep: idx[0:k] (ascending), the columns whose norm after projection (n2, squared)
// exceeds 1e-8 of the one before (n2_0), scl their 1 / norm; *kept = k.  One workgroup.  On the device
// because only the count is needed by the host: two readbacks, two uploads and a wait fewer per block.
__global__ __launch_bounds__(256) void k_keep_cols(const double* __restrict__ n2_0, const double* __restrict__ n2, int a,
                                                   int* __restrict__ idx, double* __restrict__ scl, int* __restrict__ kept) {
    __shared__ int cnt[4];
    const int tid = (int)threadIdx.x, wave = tid >> 6, lane = tid & 63;
    int k = 0;
    for (int b = 0; b < a; b += 256) {
        const int j = b + tid;
        const double before = j < a ? sqrt(n2_0[j]) : 0.0, norm = j < a ? sqrt(n2[j]) : 0.0;
        const bool keep = before > 0.0 && norm > 1e-8 * before;
        const unsigned long long mask = __ballot(keep);
        if (lane == 0) cnt[wave] = __popcll(mask);
        __syncthreads();
        int at = k + __popcll(mask & ((1ull << lane) - 1));
        for (int q = 0; q < 4; ++q) {
            if (q < wave) at += cnt[q];
            k += cnt[q];
        }
        if (keep) {
            idx[at] = j;
            scl[at] = 1.0 / norm;
        }
        __syncthreads();
    }
    if (tid == 0) *kept = k;
}

// Q[:, j] *= scale[j]
__global__ void k_scale_cols(double2* __restrict__ q, const double* __restrict__ scale, size_t ld, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double2* p = q + (size_t)blockIdx.y * ld + i;
    const double f = scale[blockIdx.y];
    *p = make_double2(p->x * f, p->y * f);
}

// T[m0 + i, j] = conj(T[j, m0 + i]) for j < m0 (mirror of the new columns), and the new
// a x a diagonal block made Hermitian with a real diagonal (common.zig:247-258).
__global__ void k_mirror_new(double2* __restrict__ t, int ld, int m0, int a) {
    const int i = blockIdx.y;  // new column index 0..a-1
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= m0 + a) return;
    const int c = m0 + i;
    if (j < m0) {
        const double2 v = t[(size_t)c * ld + j];
        t[(size_t)j * ld + c] = make_double2(v.x, -v.y);
    } else {
        const int jj = j - m0;
        if (jj > i) return;
        const double2 u = t[(size_t)c * ld + j];  // T[j][c]
        const double2 w = t[(size_t)j * ld + c];  // T[c][j]
        if (jj == i) {
            t[(size_t)c * ld + j] = make_double2(u.x, 0.0);
        } else {
            const double re = 0.5 * (u.x + w.x), im = 0.5 * (u.y - w.y);
            t[(size_t)c * ld + j] = make_double2(re, im);
            t[(size_t)j * ld + c] = make_double2(re, -im);
        }
    }
}

// ----------------------------------------------------------------- solver
struct EigWork {
    rocblas_handle blas = nullptr;
    hipStream_t stream = nullptr;
    size_t n = 0;
    int max_sub = 0, nb = 0;
    DevBuf V, W, X, HX, R, Q, HQ, T, Tw, S, G, evals, ework, info, norms, norms0, ekin, diag, sel, scl, idx;
    DevBuf x32, y32;
    uint64_t x_cols = 0;  // columns of X holding the last solve's Ritz vectors (0: none)
    bool x_converged = false;
    // Learned preconditioner: residual norms of the current iteration; training snapshots
    // (Ritz vectors, residuals, Ritz values, residual norms, <T> per band) of the last solve.
    DevBuf rnorm, snapX, snapR, snapLam, snapRn, snapEk, bandsum, samples, gram_part;
    int snaps = 0, snap_nb = 0;
    // Section timing: events recorded on the stream at section starts (pooled).
    std::vector<hipEvent_t> ev_pool;
    std::vector<int> ev_tag;
    size_t ev_used = 0;
    HeevWork heev;  // dense Hermitian eigensolver workspace (subspace problems)
    // What the host reads back in every iteration, in pinned memory that the kernels write (valid once
    // the stream is synchronised): column norms, Ritz values, and verdicts (the Cholesky
    // factorisation's two, the columns kept).  A copy after the kernel takes 3 us and a launch.
    double *host_norms = nullptr, *host_evals = nullptr;
    int* host_info = nullptr;
    size_t host_cap = 0;
    void ensure_host(size_t cols) {
        if (cols <= host_cap) return;
        release_host();
        void* p = nullptr;
        DZ_HIP(hipHostMalloc(&p, 2 * cols * sizeof(double) + 64, hipHostMallocDefault));
        host_norms = static_cast<double*>(p);
        host_evals = host_norms + cols;
        host_info = reinterpret_cast<int*>(host_evals + cols);
        host_cap = cols;
    }
    void release_host() {
        if (host_norms) (void)hipHostFree(host_norms);
        host_norms = nullptr;
        host_cap = 0;
    }
    ~EigWork() {
        release_host();
        heev.release();
        for (hipEvent_t e : ev_pool) (void)hipEventDestroy(e);
        if (blas) rocblas_destroy_handle(blas);
        DevBuf* bufs[] = {&V, &W, &X, &HX, &R, &Q, &HQ, &T, &Tw, &S, &G, &evals, &ework, &info,
                          &norms, &norms0, &ekin, &diag, &sel, &scl, &idx, &x32, &y32, &rnorm,
                          &snapX, &snapR, &snapLam, &snapRn, &snapEk, &bandsum, &samples, &gram_part};
        for (DevBuf* b : bufs) b->release();
    }
};

// Sections of a solve timed with events: a mark starts a section and ends the previous one.
enum EigSection { SEC_RR = 0, SEC_RITZ, SEC_PRECOND, SEC_ORTHO, SEC_APPLY, SEC_EXTEND, SEC_COUNT, SEC_END = SEC_COUNT };

static void mark(EigWork& w, hipStream_t s, int tag) {
    if (w.ev_used == w.ev_pool.size()) {
        hipEvent_t e;
        DZ_HIP(hipEventCreate(&e));
        w.ev_pool.push_back(e);
        w.ev_tag.push_back(0);
    }
    DZ_HIP(hipEventRecord(w.ev_pool[w.ev_used], s));
    w.ev_tag[w.ev_used++] = tag;
}

static void section_times(EigWork& w, double* out) {
    for (int i = 0; i < SEC_COUNT; ++i) out[i] = 0.0;
    if (w.ev_used < 2) {
        w.ev_used = 0;
        return;
    }
    DZ_HIP(hipEventSynchronize(w.ev_pool[w.ev_used - 1]));
    for (size_t i = 0; i + 1 < w.ev_used; ++i) {
        float ms = 0.f;
        DZ_HIP(hipEventElapsedTime(&ms, w.ev_pool[i], w.ev_pool[i + 1]));
        if (w.ev_tag[i] < SEC_COUNT) out[w.ev_tag[i]] += ms;
    }
    w.ev_used = 0;
}

// Upper Cholesky factorisation S = R^H R of a Hermitian k x k matrix (column-major, leading dimension
// ld; the upper triangle of S is read, A gets R and zeros below it), k <= kPotrfMax, one workgroup,
// right-looking in blocks of kPotrfNb rows:
//   1. the block's rows, one column of them per thread in registers: a step posts row j of the diagonal
//      block in LDS and every column, in the diagonal block or right of it, eliminates with it (one
//      barrier a step; the next step's row is posted before the rest of the update);
//   2. the trailing upper triangle minus the Gram products of those rows (in LDS) on the matrix cores,
//      16 x 16 tiles per wavefront; the next block's rows stay in LDS.
// info[0] = 0, or j + 1 for the first pivot j that is not positive (the factorisation stops there), as
// LAPACK's zpotrf reports it.  info[1] = 1 when it succeeded and every pivot keeps at least 1e-7 of its
// column's norm (R_jj > 1e-7 sqrt(S_jj)).
// The steps' chain bounds it (k of them: an LDS round trip, a reciprocal square root, a barrier).
// k = 24: 13 us, k = 164: 106 us (26 and 261 with wavefront 0 alone on the diagonal block by lane
// shuffles, substitution as a second phase and 4 x 4 tiles a thread with uncoalesced updates, a copy
// of S before and a check kernel after not counted).
constexpr int kPotrfMax = 256;
constexpr int kPotrfNb = 16;
constexpr int kPanelPitch = kPotrfNb + 1;
static __host__ __device__ int potrf_row_pitch(int k) { return (k > kPotrfNb ? (k - 1) / 16 * 16 : 0) + 1; }
static size_t potrf_lds_bytes(int k) {
    return ((size_t)kPotrfNb * potrf_row_pitch(k) + (size_t)kPanelPitch * k) * sizeof(double2);
}
// 1 / sqrt(d): the hardware's estimate (relative error about 1e-8) and one third-order Newton step.
static __device__ __forceinline__ double rsqrt_newton(double d) {
    const double r = __builtin_amdgcn_rsq(d);
    const double e = fma(-(d * r), r, 1.0);
    return fma(r * e, fma(0.375, e, 0.5), r);
}
__global__ __launch_bounds__(512) void k_potrf_upper(const double2* S, double2* A, int ld, int k,
                                                     int* __restrict__ info) {
    extern __shared__ double2 lds[];
    __shared__ double2 urow[2][kPotrfNb];  // row j of the diagonal block before its scaling
    __shared__ int s_fail, s_bad;
    const int tid = (int)threadIdx.x, nthr = (int)blockDim.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, l4 = lane >> 4;
    const int P = potrf_row_pitch(k);
    double2* rows = lds;                   // R right of the diagonal block [row][column - c0], pitch P
    double2* panel = lds + kPotrfNb * P;   // the next block's rows before elimination [column - jb][row]
    if (tid == 0) s_fail = s_bad = 0;
    for (int e = tid; e < kPotrfNb * k; e += nthr) {
        const int i = e & 15, c = e >> 4;
        panel[c * kPanelPitch + i] = i < k ? S[(size_t)c * ld + i] : double2{0.0, 0.0};
    }
    __syncthreads();
    int failed = 0;
    for (int jb = 0; jb < k; jb += kPotrfNb) {
        const int w = k - jb, nb = min(kPotrfNb, w), c0 = jb + nb, m = w - nb, mt = (m + 15) / 16;
        const bool active = (tid & ~63) < w;  // the wavefront has columns
        double2 col[kPotrfNb];                // A[jb + i][jb + tid]
        double rjj = 0.0, gjj = 0.0;
        int fail = 0;
        if (active) {
#pragma unroll
            for (int i = 0; i < kPotrfNb; ++i)
                col[i] = tid < w && i < nb ? panel[tid * kPanelPitch + i] : double2{0.0, 0.0};
            if (tid < nb) {
                urow[0][tid] = col[0];
                gjj = S[(size_t)(jb + tid) * (ld + 1)].x;
            }
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kPotrfNb; ++j) {
            if (j < nb) {
                if (active) {
                    const double2* u = urow[j & 1];
                    const double d = u[j].x, rs = rsqrt_newton(d);
                    fail = fail == 0 && !(d > 0.0) ? jb + j + 1 : fail;
                    double2 t{col[j].x * rs, col[j].y * rs};  // R[j][c]
                    if (tid == j) {
                        t = double2{d * rs, 0.0};
                        rjj = t.x;
                    }
                    col[j] = t;
                    const double2 v{t.x * rs, t.y * rs};
                    // A[i][c] -= conj(R[j][i]) R[j][c], R[j][i] = u[i] rs
#pragma unroll
                    for (int i = j + 1; i < kPotrfNb; ++i) {
                        col[i].x -= u[i].x * v.x + u[i].y * v.y;
                        col[i].y -= u[i].x * v.y - u[i].y * v.x;
                        if (i == j + 1 && tid < kPotrfNb) urow[(j + 1) & 1][tid] = col[i];
                    }
                }
                __syncthreads();
            }
        }
        if (active) {
            if (tid < nb) {
                if (!(rjj > 1e-7 * sqrt(fmax(gjj, 0.0)))) s_bad = 1;
#pragma unroll
                for (int i = 0; i < kPotrfNb; ++i)
                    if (i < nb) A[(size_t)(jb + tid) * ld + jb + i] = i <= tid ? col[i] : double2{0.0, 0.0};
            } else if (tid >= kPotrfNb && tid < kPotrfNb * (1 + mt)) {  // zeros up to the last tile's edge
#pragma unroll
                for (int i = 0; i < kPotrfNb; ++i) rows[i * P + tid - kPotrfNb] = col[i];
            }
            if (tid == 0) s_fail = fail;
        }
        __syncthreads();
        failed = s_fail;
        if (failed || m <= 0) break;
        for (int e = tid; e < kPotrfNb * m; e += nthr) {
            const int i = e & 15, c = e >> 4;
            A[(size_t)(c0 + c) * ld + jb + i] = rows[i * P + c];
        }
        for (int c = wave; c < kPotrfNb; c += nthr >> 6)
            for (int i = lane; i < m; i += 64) A[(size_t)(jb + c) * ld + c0 + i] = double2{0.0, 0.0};
        // Trailing upper triangle: A[i][c] -= sum_t conj(R[t][i]) R[t][c]; MFMA rows are columns c, MFMA
        // columns rows i, so that a load or store takes 16 consecutive rows.
        const double2* src = jb == 0 ? S : A;
        for (int e = wave; e < mt * (mt + 1) / 2; e += nthr >> 6) {
            int tc = 0, ti = e;  // tile column tc, row ti <= tc
            while (ti > tc) ti -= ++tc;
            const int i = 16 * ti + l16;
            double2 o[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int c = 16 * tc + l4 + 4 * r;
                o[r] = src[(size_t)(c0 + min(c, m - 1)) * ld + c0 + min(i, m - 1)];
            }
            v4d_t re{0, 0, 0, 0}, im{0, 0, 0, 0};
#pragma unroll
            for (int t = 0; t < kPotrfNb; t += 4) {
                const double2 a = rows[(t + l4) * P + 16 * tc + l16], b = rows[(t + l4) * P + 16 * ti + l16];
                re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, re, 0, 0, 0);
                im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.x, im, 0, 0, 0);
                re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.y, re, 0, 0, 0);
                im = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.x, b.y, im, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int c = 16 * tc + l4 + 4 * r;
                const double2 v{o[r].x - re[r], o[r].y - im[r]};
                if (c >= m) continue;
                if (ti == 0)
                    panel[c * kPanelPitch + l16] = v;
                else if (i <= c)
                    A[(size_t)(c0 + c) * ld + c0 + i] = v;
            }
        }
        __syncthreads();
    }
    if (tid == 0) {
        info[0] = failed;
        info[1] = failed == 0 && s_bad == 0 ? 1 : 0;
    }
}

// Q <- Q R^{-1} in place, Q n x k and R upper triangular (its upper triangle is read; column-major,
// leading dimensions ldq, ldr).  A wavefront takes 16 rows through the 16-column blocks from left to
// right: the products with the finished blocks on the matrix cores, then substitution with the diagonal
// block (in LDS).  MFMA rows are columns of Q and MFMA columns its rows, so that the result's register
// layout (row l % 16, columns l / 16 + 4 r) is the next products' operand layout and a finished block is
// read back by the lane that wrote it: no exchange but the substitution's row broadcasts.  One
// wavefront a workgroup while there are fewer of them than SIMDs, four (sharing R in L1) beyond.
// The chain bounds it: n = 1,637, k = 24: 7.8 us (rocBLAS' trsm 13.9); n = 20,000, k = 164: 102 us (147
// in several launches; 55 at the matrix cores' rate).
template <int NW>
__global__ __launch_bounds__(64 * NW) void k_trsm_right(double2* Q, size_t ldq, int n, int k, const double2* __restrict__ R,
                                                        int ldr) {
    __shared__ double2 diag[2][16][16];  // the diagonal block above its diagonal, zeros elsewhere [row][column]
    __shared__ double inv[2][16];
    const int tid = (int)threadIdx.x, lane = tid & 63, l16 = lane & 15, l4 = lane >> 4;
    const int row = ((int)blockIdx.x * NW + (tid >> 6)) * 16 + l16;
    double2* qrow = Q + min(row, n - 1);
    constexpr int ND = 4 / NW;  // elements of the diagonal block per thread
    double2 dn[ND], qn[4];      // the next block's, loaded before this one's substitution
    auto fetch_block = [&](int c0) {
        c0 = min(c0, (k - 1) / 16 * 16);
#pragma unroll
        for (int q = 0; q < ND; ++q) {
            const int e = tid + q * 64 * NW;
            dn[q] = R[(size_t)min(c0 + (e >> 4), k - 1) * ldr + min(c0 + (e & 15), k - 1)];
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) qn[r] = qrow[(size_t)min(c0 + l4 + 4 * r, k - 1) * ldq];
    };
    fetch_block(0);
    int buf = 0;
    for (int c0 = 0; c0 < k; c0 += 16, buf ^= 1) {
        const int nb = min(16, k - c0);
#pragma unroll
        for (int q = 0; q < ND; ++q) {
            const int e = tid + q * 64 * NW, i = e & 15, c = e >> 4;
            if (i == c) inv[buf][c] = c < nb ? 1.0 / dn[q].x : 1.0;
            diag[buf][i][c] = i < c && c < nb ? dn[q] : double2{0.0, 0.0};
        }
        v4d_t re, im;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            re[r] = qn[r].x;
            im[r] = qn[r].y;
        }
        // Q[:, block] -= Y[:, p] R[p, block]
        const double2* rc = R + (size_t)min(c0 + l16, k - 1) * ldr + l4;
        double2 a[4], y[4];
        auto fetch = [&](int p, double2 (&av)[4], double2 (&yv)[4]) {
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                av[t] = rc[p + 4 * t];
                yv[t] = qrow[(size_t)(p + l4 + 4 * t) * ldq];
            }
        };
        if (c0 > 0) fetch(0, a, y);
        for (int p = 0; p < c0; p += 16) {
            double2 an[4], yn[4];
            fetch(min(p + 16, c0 - 16), an, yn);
            __builtin_amdgcn_sched_barrier(0);  // the loads go out first
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                re = __builtin_amdgcn_mfma_f64_16x16x4f64(-a[t].x, y[t].x, re, 0, 0, 0);
                im = __builtin_amdgcn_mfma_f64_16x16x4f64(-a[t].x, y[t].y, im, 0, 0, 0);
                re = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t].y, y[t].y, re, 0, 0, 0);
                im = __builtin_amdgcn_mfma_f64_16x16x4f64(-a[t].y, y[t].x, im, 0, 0, 0);
            }
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                a[t] = an[t];
                y[t] = yn[t];
            }
        }
        __syncthreads();  // diag; the other buffer was read before the previous one
        fetch_block(c0 + 16);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 16; ++j) {
            const int src = 16 * (j & 3) + l16;
            const double f = inv[buf][j];
            const double yx = __shfl(re[j >> 2], src) * f, yy = __shfl(im[j >> 2], src) * f;
            if (l4 == (j & 3)) {
                re[j >> 2] = yx;
                im[j >> 2] = yy;
            }
#pragma unroll
            for (int r = j >> 2; r < 4; ++r) {
                const double2 d = diag[buf][j][l4 + 4 * r];
                re[r] -= yx * d.x - yy * d.y;
                im[r] -= yx * d.y + yy * d.x;
            }
        }
        if (row < n) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (l4 + 4 * r < nb) qrow[(size_t)(c0 + l4 + 4 * r) * ldq] = double2{re[r], im[r]};
        }
    }
}

// The verdicts of k_potrf_upper (out[0:2]) on another factorisation: its info, and ok = 1 when info is 0
// and every pivot keeps at least 1e-7 of its column's norm (the diagonal of G from its copy gcopy, R in
// r, both k x k with leading dimension k).  One workgroup.
__global__ __launch_bounds__(256) void k_chol_check(const double2* __restrict__ gcopy, const double2* __restrict__ r,
                                                    int k, const rocblas_int* __restrict__ info, int* __restrict__ out) {
    int bad = 0;
    for (int j = (int)threadIdx.x; j < k; j += 256) {
        const double g = gcopy[(size_t)j * (k + 1)].x, rj = r[(size_t)j * (k + 1)].x;
        if (!(rj > 1e-7 * sqrt(fmax(g, 0.0)))) bad = 1;
    }
    bad = __syncthreads_or(bad);
    if (threadIdx.x == 0) {
        out[0] = *info;
        out[1] = (*info == 0 && !bad) ? 1 : 0;
    }
}

// Lowest nev eigenpairs of the Hermitian m x m matrix A (lower triangle, leading dimension lda): vectors into
// Y (leading dimension ldy), values, ascending, into w.evals and, once s is synchronised, w.host_evals.  The
// library's device eigensolver up to m = kHeevMaxM; rocSOLVER zheevd beyond (it overwrites a copy of A in Y,
// which must then hold m columns).
static void subspace_eigh(EigWork& w, const double2* A, int lda, int m, int nev, double2* Y, int ldy, hipStream_t s) {
    if (m <= kHeevMaxM) {
        heev_lowest_shared(w.heev, A, lda, m, nev, w.evals.as<double>(), Y, ldy, s);
        DZ_HIP(hipMemcpyAsync(w.host_evals, w.evals.ptr, nev * sizeof(double), hipMemcpyDeviceToHost, s));
        return;
    }
    DZ_HIP(hipMemcpy2DAsync(Y, (size_t)ldy * sizeof(double2), A, (size_t)lda * sizeof(double2),
                            (size_t)m * sizeof(double2), m, hipMemcpyDeviceToDevice, s));
    DZ_BLAS(rocsolver_zheevd(w.blas, rocblas_evect_original, rocblas_fill_lower, m, reinterpret_cast<zc*>(Y), ldy,
                             w.evals.as<double>(), w.ework.as<double>(), w.info.as<rocblas_int>()));
    rocblas_int info = 0;
    DZ_HIP(hipMemcpyAsync(w.host_evals, w.evals.ptr, nev * sizeof(double), hipMemcpyDeviceToHost, s));
    DZ_HIP(hipMemcpyAsync(&info, w.info.ptr, sizeof(info), hipMemcpyDeviceToHost, s));
    DZ_HIP(hipStreamSynchronize(s));
    DZ_REQUIRE(info == 0, DZHIP_ERR_HIP, "zheevd did not converge");
}

static void eig_work_release(Ham& h) {
    delete static_cast<EigWork*>(h.eig_work);
    h.eig_work = nullptr;
}

struct Solver {
    Ham& h;
    EigWork& w;
    const dzhip_eig_opts& o;
    hipStream_t s;
    size_t n;
    int nb, max_sub;
    bool fp64_apply;
    dzhip_eig_stats st{};
    unsigned long long seed;

    double2* V() { return w.V.as<double2>(); }
    double2* W() { return w.W.as<double2>(); }
    double2* T() { return w.T.as<double2>(); }

    dim3 cols_grid(int cols) const { return dim3((unsigned)((n + 255) / 256), (unsigned)cols); }

    // W_out[:, 0:cols] = H V_in[:, 0:cols] in the current apply precision.
    void apply(const double2* vin, double2* wout, int cols) {
        if (cols <= 0) return;
        if (fp64_apply) {
            ham_apply_dev<double>(h, vin, wout, cols, true, true);
            st.fp64_applies += cols;
        } else {
            const size_t cnt = n * cols;
            w.x32.ensure(cnt * sizeof(float2));
            w.y32.ensure(cnt * sizeof(float2));
            convert_to_float(vin, w.x32.as<float2>(), cnt, s);
            ham_apply_dev<float>(h, w.x32.ptr, w.y32.ptr, cols, true, true);
            convert_to_double(w.y32.as<float2>(), wout, cnt, s);
            st.fp32_applies += cols;
        }
        st.apply_calls += cols;
    }

    // C[0:M, 0:N] (ld ldc) = A[:, 0:M]^H B[:, 0:N], columns of length n with leading dimension n.
    void gram(const double2* A, int M, const double2* B, int N, double2* C, int ldc) {
        if (M <= 0 || N <= 0) return;
        const int K = (int)n;
        // Two wavefronts a tile up to 96 columns of A (more, smaller workgroups where there are few),
        // four beyond; K-chunks so that the tiles fill two workgroups (four small ones) per CU.
        const int wx = M <= 96 ? 2 : 4;
        int jb = 1, ntiles = 1;
        bp_tiles(N, &jb, &ntiles);
        const int mtiles = (M + 16 * wx - 1) / (16 * wx);
        const int want = std::max(1, (wx == 4 ? 512 : 1024) / (mtiles * ntiles));
        int kchunk = (K + want - 1) / want;
        kchunk = std::max(kBpK * 4, (kchunk + kBpK - 1) / kBpK * kBpK);
        const int nks = (K + kchunk - 1) / kchunk;
        w.gram_part.ensure((size_t)nks * M * N * sizeof(double2));
        hipLaunchKernelGGL((wx == 4 ? gram_fn<4>(jb) : gram_fn<2>(jb)), dim3((unsigned)(mtiles * nks), (unsigned)ntiles),
                           dim3(64u * wx), 0, s, A, K, M, B, K, N, K, kchunk, mtiles, w.gram_part.as<double2>());
        DZ_HIP(hipGetLastError());
        hipLaunchKernelGGL(k_gram_reduce, dim3((unsigned)((M + 255) / 256), (unsigned)N), dim3(256), 0, s,
                           w.gram_part.as<double2>(), nks, M, N, C, ldc);
        DZ_HIP(hipGetLastError());
    }

    // C[:, 0:nn] = alpha A[:, 0:k] B[0:k, 0:nn] + beta C (m rows): basis times coefficients.
    void gemm(int m, int nn, int k, double alpha, const double2* A, int lda, const double2* B, int ldb, double beta,
              double2* C, int ldc) {
        if (m <= 0 || nn <= 0) return;
        DZ_REQUIRE(k > 0, DZHIP_ERR_STATE, "basis product over no columns");
        int jb = 1, ntiles = 1;
        bp_tiles(nn, &jb, &ntiles);
        const int wx = m <= 8192 ? 2 : 4;  // 32-row tiles where 64-row ones would not fill the CUs
        hipLaunchKernelGGL((wx == 4 ? gemm_fn<4>(jb) : gemm_fn<2>(jb)),
                           dim3((unsigned)((m + 16 * wx - 1) / (16 * wx)), (unsigned)ntiles), dim3(64u * wx), 0, s, A, lda, B,
                           ldb, C, ldc, m, k, nn, alpha, beta);
        DZ_HIP(hipGetLastError());
    }

    // Squared column norms into out (device or pinned memory).
    void col_norms2(const double2* v, int cols, double* out) {
        if (cols == 0) return;
        hipLaunchKernelGGL(k_col_norm2, dim3(cols), dim3(256), 0, s, v, n, (int)n, out);
        DZ_HIP(hipGetLastError());
    }

    // Orthogonalise Q[:, 0:a] against V[:, 0:m] (two block CGS passes) and orthonormalise it
    // with Cholesky QR.  A column is dropped when projection leaves less than 1e-8 of its norm
    // (the reference's MGS threshold, common.zig:263-284, applied relative to the direction's
    // own norm so that tolerances below 1e-8 Ry remain reachable).  Returns the number of
    // columns kept (compacted to the front).
    int orthonormalize_new(double2* Q, int a, int m) {
        const int ldn = (int)n;
        if (a <= 0) return 0;
        col_norms2(Q, a, w.norms0.as<double>());
        for (int pass = 0; pass < 2 && m > 0; ++pass) {
            // S = V^H Q ; Q -= V S
            gram(V(), m, Q, a, w.S.as<double2>(), max_sub);
            gemm(ldn, a, m, -1.0, V(), ldn, w.S.as<double2>(), max_sub, 1.0, Q, ldn);
        }
        col_norms2(Q, a, w.norms.as<double>());
        hipLaunchKernelGGL(k_keep_cols, dim3(1), dim3(256), 0, s, w.norms0.as<double>(), w.norms.as<double>(), a,
                           w.idx.as<int>(), w.scl.as<double>(), w.host_info + 2);
        DZ_HIP(hipGetLastError());
        DZ_HIP(hipStreamSynchronize(s));
        const int k = w.host_info[2];
        if (k == 0) return 0;
        // Normalise, compacted through HQ (scratch) where a column was dropped.
        if (k == a) {
            hipLaunchKernelGGL(k_scale_cols, cols_grid(k), dim3(256), 0, s, Q, w.scl.as<double>(), n, (int)n);
            DZ_HIP(hipGetLastError());
        } else {
            hipLaunchKernelGGL(k_gather_cols, cols_grid(k), dim3(256), 0, s, Q, w.idx.as<int>(), w.scl.as<double>(),
                               w.HQ.as<double2>(), n, (int)n);
            DZ_HIP(hipGetLastError());
            DZ_HIP(hipMemcpyAsync(Q, w.HQ.ptr, n * k * sizeof(double2), hipMemcpyDeviceToDevice, s));
        }
        int kk = k;
        for (int pass = 0; pass < 2 && kk > 0; ++pass) kk = ortho_block(Q, kk);
        return kk;
    }

    // S = R^H R for the k x k Gram matrix in S (left as it is, leading dimension k), R -> G; the verdicts
    // in w.host_info[0:2] as k_potrf_upper leaves them: the library's one-workgroup factorisation up to
    // kPotrfMax, rocSOLVER's zpotrf beyond.
    void potrf_upper(int k) {
        static_assert(sizeof(rocblas_int) == sizeof(int), "info is read as int");
        double2 *S = w.S.as<double2>(), *G = w.G.as<double2>();
        if (k <= kPotrfMax) {
            const size_t lds = potrf_lds_bytes(k);
            set_max_dynamic_lds((const void*)k_potrf_upper, lds);
            // More than 96 columns: enough tiles for eight wavefronts.
            hipLaunchKernelGGL(k_potrf_upper, dim3(1), dim3(k > 96 ? 512 : 256), lds, s, S, G, k, k,
                               w.host_info);
        } else {
            DZ_HIP(hipMemcpyAsync(G, S, (size_t)k * k * sizeof(double2), hipMemcpyDeviceToDevice, s));
            DZ_BLAS(rocsolver_zpotrf(w.blas, rocblas_fill_upper, k, reinterpret_cast<zc*>(G), k,
                                     w.info.as<rocblas_int>()));
            hipLaunchKernelGGL(k_chol_check, dim3(1), dim3(256), 0, s, S, G, k, w.info.as<rocblas_int>(), w.host_info);
        }
        DZ_HIP(hipGetLastError());
    }

    // Q[:, 0:k] <- Q R^{-1}, R the upper triangle of G (leading dimension k).
    void trsm(double2* Q, int k) {
        const unsigned tiles = (unsigned)((n + 15) / 16);
        if (tiles < 1024)
            hipLaunchKernelGGL(k_trsm_right<1>, dim3(tiles), dim3(64), 0, s, Q, n, (int)n, k, w.G.as<double2>(), k);
        else
            hipLaunchKernelGGL(k_trsm_right<4>, dim3((tiles + 3) / 4), dim3(256), 0, s, Q, n, (int)n, k, w.G.as<double2>(), k);
        DZ_HIP(hipGetLastError());
    }

    // Orthonormalise Q[:, 0:k] in place: Cholesky QR, or, when the Gram matrix is not
    // numerically positive definite, its eigen-decomposition G = U L U^H with the directions of
    // L < 1e-12 max(L) dropped and Q <- Q U L^{-1/2} (compacted to the front).  Returns the
    // number of columns kept.  Cholesky counts as failed also when a pivot keeps less than 1e-7 of
    // its column's norm (R_jj < 1e-7 sqrt(G_jj)): such a column is numerically dependent on the
    // ones before it, and dividing by its pivot would turn rounding noise into a basis vector.
    int ortho_block(double2* Q, int k) {
        const int ldn = (int)n;
        gram(Q, k, Q, k, w.S.as<double2>(), k);
        potrf_upper(k);
        DZ_HIP(hipStreamSynchronize(s));
        if (w.host_info[1]) {
            trsm(Q, k);
            return k;
        }
        st.ortho_fallbacks++;
        // Eigen-decomposition of the Gram matrix (S, lower triangle) into G.
        subspace_eigh(w, w.S.as<double2>(), k, k, k, w.G.as<double2>(), k, s);
        DZ_HIP(hipStreamSynchronize(s));
        const double* lam = w.host_evals;
        const double thr = 1e-12 * std::max(lam[k - 1], 0.0);
        int first = 0;
        while (first < k && !(lam[first] > thr)) ++first;
        const int kk = k - first;
        if (kk == 0) return 0;
        gemm(ldn, kk, k, 1.0, Q, ldn, w.G.as<double2>() + (size_t)first * k, k, 0.0, w.HQ.as<double2>(), ldn);
        std::vector<int> idx(kk);
        std::vector<double> scl(kk);
        for (int j = 0; j < kk; ++j) {
            idx[j] = j;
            scl[j] = 1.0 / std::sqrt(lam[first + j]);
        }
        DZ_HIP(hipMemcpyAsync(w.idx.ptr, idx.data(), kk * sizeof(int), hipMemcpyHostToDevice, s));
        DZ_HIP(hipMemcpyAsync(w.scl.ptr, scl.data(), kk * sizeof(double), hipMemcpyHostToDevice, s));
        hipLaunchKernelGGL(k_gather_cols, cols_grid(kk), dim3(256), 0, s, w.HQ.as<double2>(), w.idx.as<int>(),
                           w.scl.as<double>(), Q, n, (int)n);
        DZ_HIP(hipGetLastError());
        DZ_HIP(hipStreamSynchronize(s));  // idx / scl are host vectors
        return kk;
    }

    // Q <- Q R^{-1} with G = Q^H Q = R^H R.  Throws if G is not positive definite.
    void cholqr(double2* Q, int k) {
        gram(Q, k, Q, k, w.S.as<double2>(), k);
        potrf_upper(k);
        DZ_HIP(hipStreamSynchronize(s));
        DZ_REQUIRE(w.host_info[0] == 0, DZHIP_ERR_HIP, "Cholesky QR: Gram matrix not positive definite");
        trsm(Q, k);
    }

    // T[0:m+a, m:m+a] = V[:, 0:m+a]^H W[:, m:m+a], mirrored into the rows.
    void extend_T(int m, int a) {
        gram(V(), m + a, W() + (size_t)m * n, a, T() + (size_t)m * max_sub, max_sub);
        hipLaunchKernelGGL(k_mirror_new, dim3((unsigned)((m + a + 255) / 256), (unsigned)a), dim3(256), 0, s, T(),
                           max_sub, m, a);
        DZ_HIP(hipGetLastError());
    }

    // Orthonormal start block, its H image and T.  Columns [0, cols) come from the host start
    // vectors or, with reuse, from the previous solve's Ritz vectors still in X; the rest are
    // unit vectors at the smallest diag entries or LCG values (common.zig:287-319), with the
    // generator advanced past the columns that were supplied.  A start block that is not of full
    // rank (duplicated or dependent columns) keeps its independent directions and is completed
    // with fresh LCG vectors orthogonalised against them, up to three rounds, as
    // orthonormalize_all replaces dependent columns (common.zig:298-312).
    void start(int m, const double* init, uint64_t init_cols, bool reuse, const double* diag_host) {
        size_t cols = 0;
        if (init && init_cols > 0) cols = std::min<uint64_t>(init_cols, (uint64_t)m);
        else if (reuse) cols = std::min<uint64_t>(w.x_cols, (uint64_t)m);
        const size_t rest = (size_t)m - cols;
        const unsigned long long A = 6364136223846793005ULL, C = 1ULL;
        // x_{k+j} = Aj x_k + Cj: affine map of j steps by repeated squaring.
        unsigned long long aj = 1, cj = 0, ap = A, cp = C;
        for (unsigned long long j = 2ULL * n * cols; j; j >>= 1) {
            if (j & 1) {
                aj = ap * aj;
                cj = ap * cj + cp;
            }
            cp = ap * cp + cp;
            ap = ap * ap;
        }
        unsigned long long x = aj * seed + cj;
        auto next = [&]() {
            x = x * A + C;
            return (double)(x >> 11) / 9007199254740992.0;
        };
        auto lcg_block = [&](std::vector<double2>& v, size_t ncol) {
            v.resize(n * ncol);
            for (size_t c = 0; c < ncol; ++c)
                for (size_t i = 0; i < n; ++i) {
                    const double re = next() - 0.5;
                    const double im = next() - 0.5;
                    v[c * n + i] = make_double2(re, im);
                }
        };
        std::vector<double2> v;
        if (o.init_diagonal) {
            std::vector<size_t> order(n);
            for (size_t i = 0; i < n; ++i) order[i] = i;
            std::stable_sort(order.begin(), order.end(),
                             [&](size_t a, size_t b) { return diag_host[a] < diag_host[b]; });
            v.assign(n * rest, make_double2(0.0, 0.0));
            for (size_t c = 0; c < rest; ++c) v[c * n + order[cols + c]] = make_double2(1.0, 0.0);
        } else {
            lcg_block(v, rest);
        }
        if (init && init_cols > 0)
            DZ_HIP(hipMemcpyAsync(V(), init, cols * n * sizeof(double2), hipMemcpyHostToDevice, s));
        else if (cols > 0)
            DZ_HIP(hipMemcpyAsync(V(), w.X.ptr, cols * n * sizeof(double2), hipMemcpyDeviceToDevice, s));
        if (rest > 0)
            DZ_HIP(hipMemcpyAsync(V() + cols * n, v.data(), v.size() * sizeof(double2), hipMemcpyHostToDevice, s));
        DZ_HIP(hipStreamSynchronize(s));
        int k = ortho_block(V(), m);
        if (k > 0) k = ortho_block(V(), k);
        for (int round = 0; round < 3 && k < m; ++round) {
            const int need = m - k;
            lcg_block(v, (size_t)need);
            DZ_HIP(hipMemcpyAsync(w.Q.ptr, v.data(), v.size() * sizeof(double2), hipMemcpyHostToDevice, s));
            const int got = orthonormalize_new(w.Q.as<double2>(), need, k);
            if (got > 0)
                DZ_HIP(hipMemcpyAsync(V() + (size_t)k * n, w.Q.ptr, (size_t)got * n * sizeof(double2),
                                      hipMemcpyDeviceToDevice, s));
            DZ_HIP(hipStreamSynchronize(s));  // v is refilled next round
            k += got;
        }
        DZ_REQUIRE(k == m, DZHIP_ERR_STATE, "start block: no orthonormal basis of the requested size");
        apply(V(), W(), m);
        extend_T(0, m);
    }

    // Lowest nb eigenpairs of T[0:m, 0:m] (m >= nb); eigenvectors land in Tw, eigenvalues in w.evals and
    // w.host_evals.
    void rayleigh_ritz(int m) {
        subspace_eigh(w, T(), max_sub, m, std::min(m, nb), w.Tw.as<double2>(), max_sub, s);
    }

    void ritz(int m) {
        const int ldn = (int)n;
        gemm(ldn, nb, m, 1.0, V(), ldn, w.Tw.as<double2>(), max_sub, 0.0, w.X.as<double2>(), ldn);
        gemm(ldn, nb, m, 1.0, W(), ldn, w.Tw.as<double2>(), max_sub, 0.0, w.HX.as<double2>(), ldn);
    }

    // Basis <- [X, Qnew] (already orthonormal), W <- [HX, HQnew], T rebuilt.
    void restart_with(int a) {
        DZ_HIP(hipMemcpyAsync(V(), w.X.ptr, n * nb * sizeof(double2), hipMemcpyDeviceToDevice, s));
        DZ_HIP(hipMemcpyAsync(W(), w.HX.ptr, n * nb * sizeof(double2), hipMemcpyDeviceToDevice, s));
        if (a > 0) {
            DZ_HIP(hipMemcpyAsync(V() + (size_t)nb * n, w.Q.ptr, n * a * sizeof(double2), hipMemcpyDeviceToDevice, s));
            DZ_HIP(hipMemcpyAsync(W() + (size_t)nb * n, w.HQ.ptr, n * a * sizeof(double2), hipMemcpyDeviceToDevice, s));
        }
        extend_T(0, nb + a);
    }
};

static void ensure_work(Ham& h, int max_sub, int nb) {
    auto* w = static_cast<EigWork*>(h.eig_work);
    if (!w) {
        w = new EigWork();
        h.eig_work = w;
        if (rocblas_create_handle(&w->blas) != rocblas_status_success) {
            w->blas = nullptr;
            throw Error{DZHIP_ERR_HIP, "rocblas_create_handle failed"};
        }
    }
    DZ_BLAS(rocblas_set_stream(w->blas, h.stream()));
    w->stream = h.stream();
    const size_t n = h.npw;
    const size_t c = sizeof(double2);
    if (w->X.bytes < n * nb * c) w->x_cols = 0;  // X is reallocated below
    w->V.ensure(n * max_sub * c);
    w->W.ensure(n * max_sub * c);
    w->ensure_host((size_t)max_sub);
    w->X.ensure(n * nb * c);
    w->HX.ensure(n * nb * c);
    w->R.ensure(n * nb * c);
    w->Q.ensure(n * max_sub * c);
    w->HQ.ensure(n * max_sub * c);
    w->T.ensure((size_t)max_sub * max_sub * c);
    w->Tw.ensure((size_t)max_sub * max_sub * c);
    w->S.ensure((size_t)max_sub * max_sub * c);
    w->G.ensure((size_t)max_sub * max_sub * c);
    w->evals.ensure(max_sub * sizeof(double));
    w->ework.ensure(max_sub * sizeof(double));
    w->info.ensure(64);
    w->norms.ensure(max_sub * sizeof(double));
    w->norms0.ensure(max_sub * sizeof(double));
    w->ekin.ensure(max_sub * sizeof(double));
    w->diag.ensure(n * sizeof(double));
    w->sel.ensure(max_sub * sizeof(int));
    w->scl.ensure(max_sub * sizeof(double));
    w->idx.ensure(max_sub * sizeof(int));
    w->rnorm.ensure(max_sub * sizeof(double));
}

void eig_solve(Ham& h, const double* diag, uint64_t nbands, const dzhip_eig_opts& o, const double* init,
               uint64_t init_cols, double* values, double* vectors, dzhip_eig_stats* stats_out) {
    const size_t n = h.npw;
    DZ_REQUIRE(nbands > 0 && nbands <= n, DZHIP_ERR_ARG, "nbands must be in 1..n");
    DZ_REQUIRE(o.precision == DZHIP_FP64 || o.precision == DZHIP_FP32, DZHIP_ERR_ARG, "bad precision");
    DZ_REQUIRE(o.preconditioner >= DZHIP_PRECOND_KINETIC && o.preconditioner <= DZHIP_PRECOND_MLP, DZHIP_ERR_ARG,
               "bad preconditioner");
    DZ_REQUIRE(o.preconditioner != DZHIP_PRECOND_MLP || h.has_mlp, DZHIP_ERR_STATE,
               "DZHIP_PRECOND_MLP without a model (dzhip_ham_set_precond_model)");
    const int nb = (int)nbands;
    const int max_sub = (int)(o.max_subspace == 0 ? std::min<uint64_t>(n, 4 * nbands + 8)
                                                   : std::min<uint64_t>(n, std::max<uint64_t>(o.max_subspace, nbands)));
    const int block = (int)(o.block_size == 0 ? std::min<uint64_t>(max_sub, nbands + 4)
                                              : std::min<uint64_t>(max_sub, std::max<uint64_t>(o.block_size, nbands)));
    ensure_work(h, max_sub, nb);
    EigWork& w = *static_cast<EigWork*>(h.eig_work);
    Solver S{h, w, o, h.stream(), n, nb, max_sub, o.precision == DZHIP_FP64, {}, o.seed ? o.seed : 0x6f3d3cbeULL};
    hipStream_t s = S.s;
    DZ_HIP(hipMemcpyAsync(w.diag.ptr, diag, n * sizeof(double), hipMemcpyHostToDevice, s));
    const double switch_tol = o.mixed_switch_tol > 0 ? o.mixed_switch_tol : 1e-5;

    int m = block;
    // Leave the FP32 apply: restart from the Ritz vectors with an FP64 image.
    auto switch_to_fp64 = [&](uint64_t it) {
        S.fp64_apply = true;
        S.st.precision_switch_iter = it + 1;
        DZ_HIP(hipMemcpyAsync(S.V(), w.X.ptr, n * nb * sizeof(double2), hipMemcpyDeviceToDevice, s));
        S.cholqr(S.V(), nb);
        S.apply(S.V(), S.W(), nb);
        S.extend_T(0, nb);
        m = nb;
    };
    const bool reuse = o.reuse_vectors != 0 && !(init && init_cols > 0) && w.x_cols > 0;
    S.start(m, init, init_cols, reuse, diag);
    w.x_cols = 0;
    w.x_converged = false;
    const int nsnap = (int)std::min<uint64_t>(o.collect_snapshots, 64);
    if (nsnap > 0) {
        const size_t blk = n * nb * sizeof(double2);
        w.snapX.ensure(nsnap * blk);
        w.snapR.ensure(nsnap * blk);
        w.snapLam.ensure(nsnap * nb * sizeof(double));
        w.snapRn.ensure(nsnap * nb * sizeof(double));
        w.snapEk.ensure(nsnap * nb * sizeof(double));
    }
    w.snaps = 0;
    w.snap_nb = nb;
    int precond = o.preconditioner;
    // A learned model that fell back in two solves in a row on this context sits out the next
    // kMlpRest solves (the base preconditioner runs; precond_fallback reports iteration 1).
    constexpr int kMlpRest = 8;
    constexpr size_t kCurveMax = 64;  // iterations of the base preconditioner's progress record
    if (precond == DZHIP_PRECOND_MLP && h.mlp_rest > 0) {
        h.mlp_rest--;
        precond = h.mlp_base;
        S.st.precond_fallback = 1;
    }
    const bool mlp_ran = precond == DZHIP_PRECOND_MLP;
    std::vector<double> res_hist;
    const int nconv = (o.nconv == 0 || o.nconv > (uint64_t)nb) ? nb : (int)o.nconv;
    std::vector<double> lam(nb), best(nb), rn(nb);
    bool have_best = false;
    uint64_t iter = 0;
    w.ev_used = 0;
    for (; iter < o.max_iter; ++iter) {
        mark(w, s, SEC_RR);
        S.rayleigh_ritz(m);
        mark(w, s, SEC_RITZ);
        S.ritz(m);
        hipLaunchKernelGGL(k_residual, S.cols_grid(nb), dim3(256), 0, s, w.HX.as<double2>(), w.X.as<double2>(),
                           w.evals.as<double>(), w.R.as<double2>(), n, (int)n);
        DZ_HIP(hipGetLastError());
        S.col_norms2(w.R.as<double2>(), nb, w.host_norms);
        DZ_HIP(hipStreamSynchronize(s));
        lam.assign(w.host_evals, w.host_evals + nb);
        best = lam;
        have_best = true;
        for (int b = 0; b < nb; ++b) rn[b] = std::sqrt(w.host_norms[b]);
        // Convergence is judged on the first nconv bands (all by default); the others are a buffer.
        const double max_res = *std::max_element(rn.begin(), rn.begin() + nconv);
        S.st.max_residual = max_res;
        if (iter == 0) S.st.initial_residual = max_res;
        {
            // Convergence progress: mean over the bands that must converge of log10 max(r_b, tol).
            double sl = 0.0;
            for (int b = 0; b < nconv; ++b) sl += std::log10(std::max(rn[b], std::max(o.tol, 1e-300)));
            res_hist.push_back(sl / nconv);
        }
        if (w.snaps < nsnap && S.fp64_apply) {
            const size_t blk = n * nb;
            double2* sx = w.snapX.as<double2>() + w.snaps * blk;
            double2* sr = w.snapR.as<double2>() + w.snaps * blk;
            DZ_HIP(hipMemcpyAsync(sx, w.X.ptr, blk * sizeof(double2), hipMemcpyDeviceToDevice, s));
            DZ_HIP(hipMemcpyAsync(sr, w.R.ptr, blk * sizeof(double2), hipMemcpyDeviceToDevice, s));
            DZ_HIP(hipMemcpyAsync(w.snapLam.as<double>() + w.snaps * nb, lam.data(), nb * sizeof(double),
                                  hipMemcpyHostToDevice, s));
            DZ_HIP(hipMemcpyAsync(w.snapRn.as<double>() + w.snaps * nb, rn.data(), nb * sizeof(double),
                                  hipMemcpyHostToDevice, s));
            hipLaunchKernelGGL(k_kinetic_energy, dim3(nb), dim3(256), 0, s, w.X.as<double2>(), w.diag.as<double>(), n,
                               (int)n, w.snapEk.as<double>() + w.snaps * nb);
            DZ_HIP(hipGetLastError());
            DZ_HIP(hipStreamSynchronize(s));  // lam / rn are host vectors rebuilt next iteration
            w.snaps++;
        }
        // Learned preconditioner: fall back to its base preconditioner for the rest of the solve
        // when, from the fourth iteration on, the progress so far (drop of the mean log residual
        // since the first iteration) trails the base's mean progress at the same iteration on
        // this context by more than 0.25 decades, or (no base record for this iteration yet)
        // when the last three iterations gained less than 0.05 decades per iteration.
        if (precond == DZHIP_PRECOND_MLP && res_hist.size() > 3) {
            const size_t i = res_hist.size() - 1;
            const auto& curve = h.precond_curve[h.mlp_base == DZHIP_PRECOND_TPA ? 1 : 0];
            const double drop = res_hist.front() - res_hist.back();
            const bool behind = i < curve.size() ? drop < curve[i] - 0.25
                                                 : (res_hist[i - 3] - res_hist[i]) / 3.0 < 0.05;
            if (behind) {
                precond = h.mlp_base;
                S.st.precond_fallback = iter + 1;
            }
        }
        // FP32 apply: a tolerance looser than the switch threshold is met in FP32; tighter
        // tolerances switch the apply to FP64 once the residual is below the threshold.
        if (max_res < o.tol && (S.fp64_apply || o.tol >= switch_tol)) {
            S.st.converged = 1;
            break;
        }
        if (!S.fp64_apply && max_res < switch_tol) {
            switch_to_fp64(iter);
            continue;
        }
        // New directions for the unconverged bands, in band order (serial.zig:249-261).
        const int room = std::min(nb, max_sub - nb);
        std::vector<int> sel;
        for (int b = 0; b < nb && (int)sel.size() < room; ++b)
            if (rn[b] >= o.tol) sel.push_back(b);
        int a = 0;
        // The new block is built at its place in the basis, its H image in W, where they fit; before a
        // restart in Q and HQ.
        const bool in_place = m + (int)sel.size() <= max_sub;
        double2 *qn = in_place ? S.V() + (size_t)m * n : w.Q.as<double2>(), *hqn = in_place ? S.W() + (size_t)m * n : w.HQ.as<double2>();
        if (!sel.empty()) {
            mark(w, s, SEC_PRECOND);
            DZ_HIP(hipMemcpyAsync(w.sel.ptr, sel.data(), sel.size() * sizeof(int), hipMemcpyHostToDevice, s));
            if (precond != DZHIP_PRECOND_KINETIC) {
                hipLaunchKernelGGL(k_kinetic_energy, dim3(nb), dim3(256), 0, s, w.X.as<double2>(), w.diag.as<double>(),
                                   n, (int)n, w.ekin.as<double>());
                DZ_HIP(hipGetLastError());
            }
            if (precond == DZHIP_PRECOND_MLP) {
                DZ_HIP(hipMemcpyAsync(w.rnorm.ptr, rn.data(), nb * sizeof(double), hipMemcpyHostToDevice, s));
                precondition_mlp(w.R.as<double2>(), w.sel.as<int>(), (int)sel.size(), w.evals.as<double>(),
                                 w.ekin.as<double>(), w.rnorm.as<double>(), w.diag.as<double>(), h.mlp_params.as<float>(),
                                 h.mlp_energy_scale, h.mlp_base, qn, n, (int)n, s);
            } else {
                hipLaunchKernelGGL(k_precondition, S.cols_grid((int)sel.size()), dim3(256), 0, s, w.R.as<double2>(),
                                   w.sel.as<int>(), w.evals.as<double>(), w.ekin.as<double>(), w.diag.as<double>(),
                                   qn, n, (int)n, precond == DZHIP_PRECOND_TPA ? 1 : 0);
                DZ_HIP(hipGetLastError());
            }
            mark(w, s, SEC_ORTHO);
            a = S.orthonormalize_new(qn, (int)sel.size(), m);
        }
        if (a == 0) {
            // Nothing could be added: every residual is individually below tol
            // (serial.zig:262-273) or the new directions lie in the basis.
            if (!S.fp64_apply && o.tol < switch_tol) {
                switch_to_fp64(iter);
                continue;
            }
            S.st.converged = max_res < o.tol ? 1 : 0;
            break;
        }
        mark(w, s, SEC_APPLY);
        S.apply(qn, hqn, a);
        mark(w, s, SEC_EXTEND);
        if (m + a > max_sub) {
            // Thick restart from [Ritz vectors, new block]; their H images are W c and H Q.
            S.restart_with(a);
            m = nb + a;
            S.st.restarts++;
            continue;
        }
        if (!in_place) {
            DZ_HIP(hipMemcpyAsync(S.V() + (size_t)m * n, w.Q.ptr, n * a * sizeof(double2), hipMemcpyDeviceToDevice, s));
            DZ_HIP(hipMemcpyAsync(S.W() + (size_t)m * n, w.HQ.ptr, n * a * sizeof(double2), hipMemcpyDeviceToDevice, s));
        }
        S.extend_T(m, a);
        m += a;
    }
    mark(w, s, SEC_END);
    S.st.iterations = iter;
    if (mlp_ran) {
        h.mlp_fail_streak = S.st.precond_fallback > 0 ? h.mlp_fail_streak + 1 : 0;
        if (h.mlp_fail_streak >= 2) {
            h.mlp_rest = kMlpRest;
            h.mlp_fail_streak = 0;
        }
    }
    // Mean progress per iteration index of kinetic-shift and TPA solves on this context (drop of
    // the mean log residual since the first iteration), the yardstick of the learned
    // preconditioner's fallback.  A converged solve's last value stands for the iterations it
    // did not need.
    if ((o.preconditioner == DZHIP_PRECOND_KINETIC || o.preconditioner == DZHIP_PRECOND_TPA) &&
        res_hist.size() >= 2) {
        const int c = o.preconditioner == DZHIP_PRECOND_TPA ? 1 : 0;
        auto& curve = h.precond_curve[c];
        auto& cnt = h.precond_curve_n[c];
        const size_t len = std::max(curve.size(), S.st.converged ? (size_t)kCurveMax : res_hist.size());
        const size_t keep = std::min(len, (size_t)kCurveMax);
        curve.resize(keep, 0.0);
        cnt.resize(keep, 0);
        for (size_t i = 0; i < keep; ++i) {
            if (i >= res_hist.size() && !S.st.converged) break;
            const double d = res_hist.front() - res_hist[std::min(i, res_hist.size() - 1)];
            cnt[i]++;
            curve[i] += (d - curve[i]) / cnt[i];
        }
    }
    if (have_best) {
        std::memcpy(values, best.data(), nb * sizeof(double));
        w.x_cols = nb;
        w.x_converged = S.st.converged != 0;
    }
    if (vectors) DZ_HIP(hipMemcpyAsync(vectors, w.X.ptr, n * nb * sizeof(double2), hipMemcpyDeviceToHost, s));
    DZ_HIP(hipStreamSynchronize(s));
    double sec[SEC_COUNT];
    section_times(w, sec);
    S.st.t_rr_ms = sec[SEC_RR];
    S.st.t_ritz_ms = sec[SEC_RITZ];
    S.st.t_precond_ms = sec[SEC_PRECOND];
    S.st.t_ortho_ms = sec[SEC_ORTHO];
    S.st.t_apply_ms = sec[SEC_APPLY];
    S.st.t_extend_ms = sec[SEC_EXTEND];
    if (stats_out) *stats_out = S.st;
}

// ----------------------------------------------------------------- band-by-band CG
namespace {

struct CgRun {
    Ham& h;
    EigWork& w;
    hipStream_t s;
    size_t n;
    int ldn;
    dzhip_eig_stats& st;

    dim3 grid1() const { return dim3((unsigned)((n + 255) / 256)); }
    cplx dot(const double2* a, const double2* b) {  // <a|b>
        zc r;
        DZ_BLAS(rocblas_zdotc(w.blas, ldn, reinterpret_cast<const zc*>(a), 1, reinterpret_cast<const zc*>(b), 1, &r));
        return cplx(r.real(), r.imag());
    }
    double nrm(const double2* a) {
        double r = 0.0;
        DZ_BLAS(rocblas_dznrm2(w.blas, ldn, reinterpret_cast<const zc*>(a), 1, &r));
        return r;
    }
    void axpy(cplx alpha, const double2* x, double2* y) {
        const zc al(alpha.real(), alpha.imag());
        DZ_BLAS(rocblas_zaxpy(w.blas, ldn, &al, reinterpret_cast<const zc*>(x), 1, reinterpret_cast<zc*>(y), 1));
    }
    void scal(double a, double2* x) {
        DZ_BLAS(rocblas_zdscal(w.blas, ldn, &a, reinterpret_cast<zc*>(x), 1));
    }
    void copy(double2* dst, const double2* src) {
        DZ_HIP(hipMemcpyAsync(dst, src, n * sizeof(double2), hipMemcpyDeviceToDevice, s));
    }
    void apply(const double2* x, double2* y) {
        ham_apply_dev<double>(h, x, y, 1, true, true);
        st.apply_calls++;
        st.fp64_applies++;
    }
    // v -= sum_{j<m} <V_j|v> V_j, one column at a time in order (modified Gram-Schmidt).
    void orth(double2* v, const double2* V, int m) {
        for (int j = 0; j < m; ++j) axpy(-dot(V + (size_t)j * n, v), V + (size_t)j * n, v);
    }
    void combine(const double2* a, const double2* b, const double2* c, cplx c0, cplx c1, cplx c2, bool use_c,
                 double2* out) {
        hipLaunchKernelGGL(k_combine3, grid1(), dim3(256), 0, s, a, b, c, make_double2(c0.real(), c0.imag()),
                           make_double2(c1.real(), c1.imag()), make_double2(c2.real(), c2.imag()), use_c ? 1 : 0, out,
                           (int)n);
        DZ_HIP(hipGetLastError());
    }
};

}  // namespace

void cg_solve(Ham& h, const double* diag, uint64_t nbands, const dzhip_eig_opts& o, const double* init,
              uint64_t init_cols, double* values, double* vectors, dzhip_eig_stats* stats_out) {
    const size_t n = h.npw;
    DZ_REQUIRE(nbands > 0 && nbands <= n, DZHIP_ERR_ARG, "nbands must be in 1..n");
    const int nb = (int)nbands;
    const uint64_t max_iter = o.max_iter ? o.max_iter : 20;
    const double tol = o.tol > 0.0 ? o.tol : 1e-6;
    ensure_work(h, nb, nb);
    EigWork& w = *static_cast<EigWork*>(h.eig_work);
    // Work vectors: psi block in V, H psi in W[:,0], r/p/d/Hd/psi_old/Hpsi_old/psi_prev/Hpsi_prev
    // in Q columns 0..7 (Q holds n x max_sub >= n x 8 when nb >= 8; else grow it).
    w.Q.ensure(n * std::max(nb, 8) * sizeof(double2));
    w.W.ensure(n * std::max(nb, 8) * sizeof(double2));
    dzhip_eig_stats st{};
    hipStream_t s = h.stream();
    CgRun R{h, w, s, n, (int)n, st};
    DZ_BLAS(rocblas_set_pointer_mode(w.blas, rocblas_pointer_mode_host));
    DZ_HIP(hipMemcpyAsync(w.diag.ptr, diag, n * sizeof(double), hipMemcpyHostToDevice, s));

    // Start: copied vectors, reused device vectors, or the LCG; orthonormalised (MGS).
    double2* V = w.V.as<double2>();
    {
        const bool reuse = o.reuse_vectors != 0 && !(init && init_cols > 0) && w.x_cols > 0;
        size_t cols = 0;
        if (init && init_cols > 0) cols = std::min<uint64_t>(init_cols, nbands);
        else if (reuse) cols = std::min<uint64_t>(w.x_cols, nbands);
        std::vector<double2> v(n * (nb - cols));
        unsigned long long x = o.seed ? o.seed : 0x6f3d3cbeULL;
        for (size_t i = 0; i < v.size(); ++i) {
            auto nxt = [&]() {
                x = x * 6364136223846793005ULL + 1ULL;
                return (double)(x >> 11) / 9007199254740992.0;
            };
            const double re = nxt() - 0.5;
            const double im = nxt() - 0.5;
            v[i] = make_double2(re, im);
        }
        if (init && init_cols > 0) DZ_HIP(hipMemcpyAsync(V, init, cols * n * sizeof(double2), hipMemcpyHostToDevice, s));
        else if (cols > 0) DZ_HIP(hipMemcpyAsync(V, w.X.ptr, cols * n * sizeof(double2), hipMemcpyDeviceToDevice, s));
        if (!v.empty())
            DZ_HIP(hipMemcpyAsync(V + cols * n, v.data(), v.size() * sizeof(double2), hipMemcpyHostToDevice, s));
        DZ_HIP(hipStreamSynchronize(s));
        for (int b = 0; b < nb; ++b) {
            double2* vb = V + (size_t)b * n;
            R.orth(vb, V, b);
            const double nv = R.nrm(vb);
            DZ_REQUIRE(nv > 1e-8, DZHIP_ERR_ARG, "start vectors are linearly dependent");
            R.scal(1.0 / nv, vb);
        }
    }
    w.x_cols = 0;
    w.x_converged = false;
    double2* Q = w.Q.as<double2>();
    double2 *hpsi = w.W.as<double2>(), *r = Q, *p = Q + n, *d = Q + 2 * n, *hd = Q + 3 * n, *pold = Q + 4 * n,
            *hpold = Q + 5 * n, *pp = Q + 6 * n, *hpp = Q + 7 * n;
    std::vector<double> vals(nb);
    bool all_conv = true;
    for (int b = 0; b < nb; ++b) {
        double2* psi = V + (size_t)b * n;
        if (b > 0) {
            R.orth(psi, V, b);
            R.scal(1.0 / R.nrm(psi), psi);
        }
        R.apply(psi, hpsi);
        double lam = R.dot(psi, hpsi).real();
        double prev_zr = 0.0;
        bool has_prev = false, conv = false;
        for (uint64_t it = 0; it < max_iter; ++it) {
            st.iterations++;
            R.copy(r, hpsi);
            R.axpy(cplx(-lam, 0.0), psi, r);
            R.orth(r, V, b);
            if (R.nrm(r) < tol) {
                conv = true;
                break;
            }
            hipLaunchKernelGGL(k_precondition_one, R.grid1(), dim3(256), 0, s, r, w.diag.as<double>(), lam, p, (int)n);
            DZ_HIP(hipGetLastError());
            R.orth(p, V, b + 1);
            const double zr = R.dot(p, r).real();
            if (has_prev && prev_zr > 1e-30) {
                R.scal(std::max(0.0, zr / prev_zr), d);
                R.axpy(cplx(1.0, 0.0), p, d);
            } else {
                R.copy(d, p);
            }
            prev_zr = zr;
            R.orth(d, V, b + 1);
            const double dn = R.nrm(d);
            if (dn < 1e-14) break;
            R.scal(1.0 / dn, d);
            R.apply(d, hd);
            // Three-term Rayleigh-Ritz on {psi, d, psi_prev} when the previous psi adds a direction.
            bool three = false;
            double lam_new = lam;
            cplx c0, c1, c2;
            if (has_prev) {
                R.copy(pp, pold);
                R.copy(hpp, hpold);
                const cplx ov = R.dot(psi, pp);
                R.axpy(-ov, psi, pp);
                R.axpy(-ov, hpsi, hpp);
                const cplx ovd = R.dot(d, pp);
                R.axpy(-ovd, d, pp);
                R.axpy(-ovd, hd, hpp);
                const double pn = R.nrm(pp);
                if (pn > 1e-6) {
                    R.scal(1.0 / pn, pp);
                    R.scal(1.0 / pn, hpp);
                    const double a22 = R.dot(d, hd).real(), a33 = R.dot(pp, hpp).real();
                    const cplx a12 = R.dot(psi, hd), a13 = R.dot(psi, hpp), a23 = R.dot(d, hpp);
                    const cplx m3[9] = {lam, a12, a13, std::conj(a12), a22, a23, std::conj(a13), std::conj(a23), a33};
                    cplx vec[3];
                    herm3_lowest(m3, &lam_new, vec);
                    // Phase convention: the psi coefficient real and non-negative.
                    if (std::abs(vec[0]) > 0.0) {
                        const cplx ph = std::abs(vec[0]) / vec[0];
                        for (auto& c : vec) c *= ph;
                    }
                    c0 = vec[0];
                    c1 = vec[1];
                    c2 = vec[2];
                    three = true;
                }
            }
            if (!three) {
                const double a11 = lam, a22 = R.dot(d, hd).real();
                const cplx a12 = R.dot(psi, hd);
                const double avg = 0.5 * (a11 + a22), diff = 0.5 * (a11 - a22), off = std::norm(a12);
                lam_new = avg - std::sqrt(diff * diff + off);
                if (off > 1e-30) {
                    c0 = -a12;
                    c1 = cplx(a11 - lam_new, 0.0);
                } else if (a11 <= a22) {
                    c0 = 1.0;
                    c1 = 0.0;
                } else {
                    c0 = 0.0;
                    c1 = 1.0;
                }
                const double cn = std::sqrt(std::norm(c0) + std::norm(c1));
                if (cn > 1e-30) {
                    c0 /= cn;
                    c1 /= cn;
                }
                c2 = 0.0;
            }
            R.copy(pold, psi);
            R.copy(hpold, hpsi);
            has_prev = true;
            R.combine(pold, d, pp, c0, c1, c2, three, psi);
            R.combine(hpold, hd, hpp, c0, c1, c2, three, hpsi);
            const double pn2 = R.nrm(psi);
            if (pn2 > 1e-14) {
                R.scal(1.0 / pn2, psi);
                R.scal(1.0 / pn2, hpsi);
            }
            const double change = std::fabs(lam_new - lam);
            lam = lam_new;
            if (change < tol) {
                conv = true;
                break;
            }
        }
        vals[b] = lam;
        all_conv = all_conv && conv;
        if (b > 0) {
            R.orth(psi, V, b);
            R.scal(1.0 / R.nrm(psi), psi);
        }
    }
    // Final subspace rotation: T = V^H H V, eigen-decomposition, X = V C (cg.zig:450-482).
    double2* HV = w.HX.as<double2>();
    ham_apply_dev<double>(h, V, HV, nb, true, true);
    st.apply_calls += nb;
    st.fp64_applies += nb;
    const zc one(1.0, 0.0), zero(0.0, 0.0);
    DZ_BLAS(rocblas_zgemm(w.blas, rocblas_operation_conjugate_transpose, rocblas_operation_none, nb, nb, (int)n, &one,
                          reinterpret_cast<const zc*>(V), (int)n, reinterpret_cast<const zc*>(HV), (int)n, &zero,
                          w.Tw.as<zc>(), nb));
    // Eigenvectors of T (in Tw) into S (nb x nb).
    subspace_eigh(w, w.Tw.as<double2>(), nb, nb, nb, w.S.as<double2>(), nb, s);
    DZ_HIP(hipStreamSynchronize(s));
    const std::vector<double> ev(w.host_evals, w.host_evals + nb);
    DZ_BLAS(rocblas_zgemm(w.blas, rocblas_operation_none, rocblas_operation_none, (int)n, nb, nb, &one,
                          reinterpret_cast<const zc*>(V), (int)n, w.S.as<zc>(), nb, &zero, w.X.as<zc>(), (int)n));
    std::copy(ev.begin(), ev.end(), values);
    if (vectors) DZ_HIP(hipMemcpyAsync(vectors, w.X.ptr, n * nb * sizeof(double2), hipMemcpyDeviceToHost, s));
    DZ_HIP(hipStreamSynchronize(s));
    w.x_cols = nb;
    w.x_converged = all_conv;
    st.converged = all_conv ? 1 : 0;
    if (stats_out) *stats_out = st;
}

void eig_release(Ham& h) { eig_work_release(h); }

size_t eig_training_samples(Ham& h, double energy_scale, int base, int stride, float* out_host, size_t cap) {
    auto* w = static_cast<EigWork*>(h.eig_work);
    DZ_REQUIRE(w && w->snaps > 0, DZHIP_ERR_STATE, "no training snapshots (solve with collect_snapshots > 0)");
    DZ_REQUIRE(w->x_converged && w->x_cols == (uint64_t)w->snap_nb, DZHIP_ERR_STATE,
               "the recording solve did not converge");
    DZ_REQUIRE(stride >= 1 && energy_scale > 0.0, DZHIP_ERR_ARG, "stride >= 1 and energy_scale > 0");
    DZ_REQUIRE(base == DZHIP_PRECOND_KINETIC || base == DZHIP_PRECOND_TPA, DZHIP_ERR_ARG,
               "base must be DZHIP_PRECOND_KINETIC or DZHIP_PRECOND_TPA");
    hipStream_t s = h.stream();
    DZ_BLAS(rocblas_set_stream(w->blas, s));
    const int nb = w->snap_nb;
    const size_t n = h.npw, blk = n * nb;
    const int per_col = (int)((n + stride - 1) / stride);
    const size_t total = std::min<size_t>(cap, (size_t)w->snaps * nb * per_col);
    if (total == 0) return 0;
    w->samples.ensure(6 * total * sizeof(float));
    w->bandsum.ensure(3 * nb * sizeof(double));
    w->Q.ensure(blk * sizeof(double2));
    w->G.ensure((size_t)nb * nb * sizeof(double2));
    const zc one(1.0, 0.0), zero(0.0, 0.0), mone(-1.0, 0.0);
    size_t done = 0;
    for (int i = 0; i < w->snaps && done < total; ++i) {
        const double2* xi = w->snapX.as<double2>() + i * blk;
        // C = X^H x_i, E = X C - x_i (the part of x_i outside the converged subspace, negated).
        DZ_BLAS(rocblas_zgemm(w->blas, rocblas_operation_conjugate_transpose, rocblas_operation_none, nb, nb, (int)n,
                              &one, reinterpret_cast<const zc*>(w->X.ptr), (int)n, reinterpret_cast<const zc*>(xi),
                              (int)n, &zero, w->G.as<zc>(), nb));
        DZ_HIP(hipMemcpyAsync(w->Q.ptr, xi, blk * sizeof(double2), hipMemcpyDeviceToDevice, s));
        DZ_BLAS(rocblas_zgemm(w->blas, rocblas_operation_none, rocblas_operation_none, (int)n, nb, nb, &one,
                              reinterpret_cast<const zc*>(w->X.ptr), (int)n, w->G.as<zc>(), nb, &mone,
                              w->Q.as<zc>(), (int)n));
        done += mlp_write_samples(w->Q.as<double2>(), w->snapR.as<double2>() + i * blk, w->snapLam.as<double>() + i * nb,
                                  w->snapEk.as<double>() + i * nb, w->snapRn.as<double>() + i * nb,
                                  w->diag.as<double>(), n, (int)n, nb, stride, energy_scale, base, w->bandsum.as<double>(),
                                  w->samples.as<float>(), total, done, s);
    }
    for (int f = 0; f < 6; ++f)
        DZ_HIP(hipMemcpyAsync(out_host + (size_t)f * cap, w->samples.as<float>() + (size_t)f * total,
                              done * sizeof(float), hipMemcpyDeviceToHost, s));
    DZ_HIP(hipStreamSynchronize(s));
    return done;
}

const double2* eig_solution(const Ham& h, uint64_t* cols) {
    const auto* w = static_cast<const EigWork*>(h.eig_work);
    *cols = w ? w->x_cols : 0;
    return (w && w->x_cols > 0) ? w->X.as<double2>() : nullptr;
}

}  // namespace dzhip
