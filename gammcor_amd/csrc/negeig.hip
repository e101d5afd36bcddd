// Eigenpairs below zero of symmetric FP64 matrices by block Krylov (Lanczos)
// iteration, and the Cholesky factor of |A| = A - 2 sum_{l < 0} l x x^T.
//
// The ERPA needs a factor of |A+| and A+ has few eigenvalues below zero (1 to
// 21 of 410 to 4524), at the lower end of its spectrum, where a Krylov space
// converges first: about 52 blocks of 16 vectors to a residual at rounding
// level (numpy, A+ of orders 410 to 2664), each one pass over A.  A full
// eigensolve reads A's trailing matrix once per column instead.
//
// Per block: W = A Q (HBM: A once), W orthogonalised against the basis V
// twice (V twice each time), and its Gram matrix factored (CholeskyQR, after
// each orthogonalisation).  A Rayleigh-Ritz problem H = V^T A V then gives
// the pairs, whose residuals are formed and checked.  No pair is missed
// unseen: |A| with one left out has a negative eigenvalue and its Cholesky
// factorisation fails.
#include <algorithm>
#include <cmath>
#include <vector>

#include "chol.hpp"
#include "gemm.hpp"
#include "negeig.hpp"
#include "prof.hpp"
#include "wave_ops.hpp"

namespace gmc {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));
constexpr int KB = 16;                 // block width: one MFMA tile
constexpr int KM_FIRST = 832, KM_MAX = 1536;   // basis sizes of the first Ritz pairs and at most
constexpr int SK_ROWS = 32, SK_WAVES = 8;

// Out = Mat Q (sub = 0, and a copy into Out2), or Out -= Mat Q: Mat n x K
// (column-major, ld n), Qt = Q row-major (K x 16), Out n x 16 (ld n).  A
// workgroup forms 32 rows; its waves split K and add up through LDS in a
// fixed order.  Bound by reading Mat once: an MFMA takes 16 rows x 4 columns
// of it straight from memory (128-byte segments), U steps in flight.
__global__ __launch_bounds__(64 * SK_WAVES) void skinny_kernel(const double* Mat, int64_t sm, int n, int K,
                                                               const double* Qt, int64_t sq, double* Out, int64_t so,
                                                               double* Out2, int64_t so2, int sub)
{
    __shared__ double red[SK_WAVES][2][4][64];
    const int b = blockIdx.y, r0 = blockIdx.x * SK_ROWS, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const double* M = Mat + (size_t)b * sm;
    const double* Q = Qt + (size_t)b * sq;
    const int row = lane & 15, kk = lane >> 4;
    const bool in0 = r0 + row < n, in1 = r0 + 16 + row < n;
    const double* m0 = M + (in0 ? r0 + row : 0);
    const double* m1 = M + (in1 ? r0 + 16 + row : 0);
    v4d acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};
    constexpr int U = 8;
    const int per = ((K + 4 * U - 1) / (4 * U) + SK_WAVES - 1) / SK_WAVES * 4 * U;
    const int kend = min(K, (wave + 1) * per);
    for (int k0 = wave * per; k0 < kend; k0 += 4 * U) {
        double a0[U], a1[U], q[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int k = k0 + 4 * u + kk;
            const bool ok = k < kend;
            const size_t o = ok ? (size_t)k * n : 0;
            a0[u] = ok && in0 ? m0[o] : 0.0;
            a1[u] = ok && in1 ? m1[o] : 0.0;
            q[u] = ok ? Q[k * KB + row] : 0.0;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            // (formed transposed: the registers hold 16 rows of one column)
            acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(q[u], a0[u], acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(q[u], a1[u], acc1, 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
        red[wave][0][r][lane] = acc0[r];
        red[wave][1][r][lane] = acc1[r];
    }
    __syncthreads();
    // 512 outputs, one per thread: tile t, register r, lane l
    const int t = threadIdx.x >> 8, r = (threadIdx.x >> 6) & 3;
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < SK_WAVES; w++) s += red[w][t][r][lane];
    const int orow = r0 + 16 * t + row, col = kk + 4 * r;
    if (orow < n) {
        double* o = Out + (size_t)b * so + orow + (size_t)col * n;
        if (sub) s = *o - s;
        *o = s;
        if (Out2) Out2[(size_t)b * so2 + orow + (size_t)col * n] = s;
    }
}

// Ct = V^T W (row-major, m x 16): a workgroup forms 16 rows, its waves split
// the n rows of V and W and add up through LDS in a fixed order.
__global__ __launch_bounds__(64 * SK_WAVES) void vtw_kernel(const double* V, int64_t sv, int n, const double* W,
                                                            int64_t sw, double* Ct, int64_t sc)
{
    __shared__ double red[SK_WAVES][4][64];
    const int b = blockIdx.y, v0 = blockIdx.x * KB, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = lane & 15, g = lane >> 4;
    const double* v = V + (size_t)b * sv + (size_t)(v0 + c) * n;
    const double* w = W + (size_t)b * sw + (size_t)c * n;
    v4d acc = {0, 0, 0, 0};
    constexpr int U = 4;   // chunks of 16 rows in flight
    for (int k0 = wave * 16 * U; k0 < n; k0 += SK_WAVES * 16 * U) {
        double x[U][4], y[U][4];
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int k = k0 + 16 * u + 4 * g + e;
                x[u][e] = k < n ? v[k] : 0.0;
                y[u][e] = k < n ? w[k] : 0.0;
            }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[u][e], y[u][e], acc, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) red[wave][r][lane] = acc[r];
    __syncthreads();
    if (threadIdx.x < 256) {
        const int r = threadIdx.x >> 6;
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < SK_WAVES; q++) s += red[q][r][lane];
        Ct[(size_t)b * sc + (size_t)(v0 + g + 4 * r) * KB + c] = s;
    }
}

// W (n x 16) -> W R^-1, W^T W = R^T R: into Vd (column-major, ld n) and Qt
// (row-major).  One workgroup per problem.  A pivot at rounding level of the
// block's largest column marks the problem in bad.
__global__ __launch_bounds__(1024) void cholqr_kernel(const double* W, int64_t sw, int n, double* Vd, int64_t sv,
                                                      double* Qt, int64_t sq, int* bad)
{
    __shared__ double red[16][4][64];
    __shared__ double G[KB][KB + 1], Ti[KB][KB + 1];
    const int b = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = lane & 15, g = lane >> 4;
    const double* w = W + (size_t)b * sw;
    {
        v4d acc = {0, 0, 0, 0};
        for (int k0 = wave * 32; k0 < n; k0 += 16 * 32) {
            double x[8];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const int k = k0 + 16 * (e >> 2) + 4 * g + (e & 3);
                x[e] = k < n ? w[k + (size_t)c * n] : 0.0;
            }
#pragma unroll
            for (int e = 0; e < 8; e++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(x[e], x[e], acc, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) red[wave][r][lane] = acc[r];
    }
    __syncthreads();
    if (threadIdx.x < 256) {
        const int r = threadIdx.x >> 6;
        double s = 0.0;
#pragma unroll
        for (int q = 0; q < 16; q++) s += red[q][r][lane];
        G[g + 4 * r][c] = s;
    }
    __syncthreads();
    if (wave == 0) {
        // R (upper) column by column from G, lanes over its columns; then Ti =
        // R^-1 by back substitution
        double top = 0.0;
        for (int i = 0; i < KB; i++) top = fmax(top, G[i][i]);
        bool fail = false;
        for (int i = 0; i < KB; i++) {
            double d = G[i][i];
            if (!(d > 1e-28 * top)) {
                fail = true;
                d = 1.0;
            }
            const double rd = sqrt(d);
            const double rij = lane < KB && lane >= i ? G[i][lane] / rd : 0.0;
            __builtin_amdgcn_wave_barrier();
            if (lane < KB && lane >= i) G[i][lane] = lane == i ? rd : rij;
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (lane < KB && lane > i)
                for (int k = i + 1; k <= lane; k++) G[k][lane] -= G[i][k] * G[i][lane];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        if (lane < KB) {
            for (int i = KB - 1; i >= 0; i--) {
                double s = i == lane ? 1.0 : 0.0;
                for (int k = i + 1; k <= lane; k++) s -= G[i][k] * Ti[k][lane];
                Ti[i][lane] = i <= lane ? s / G[i][i] : 0.0;
            }
        }
        if (fail && lane == 0) bad[b] = 1;
    }
    __syncthreads();
    double tk[4];
#pragma unroll
    for (int e = 0; e < 4; e++) tk[e] = Ti[4 * e + g][c];   // T(k = 4e + g, column c)
    double* vd = Vd + (size_t)b * sv;
    double* qt = Qt ? Qt + (size_t)b * sq : nullptr;
    for (int r0 = wave * 16; r0 < n; r0 += 16 * 16) {
        double x[4];
#pragma unroll
        for (int e = 0; e < 4; e++) x[e] = r0 + c < n ? w[r0 + c + (size_t)(4 * e + g) * n] : 0.0;
        v4d acc = {0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < 4; e++) acc = __builtin_amdgcn_mfma_f64_16x16x4f64(tk[e], x[e], acc, 0, 0, 0);
        if (r0 + c < n) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int col = g + 4 * r;
                vd[r0 + c + (size_t)col * n] = acc[r];
                if (qt) qt[(size_t)(r0 + c) * KB + col] = acc[r];
            }
        }
    }
}

// A fixed pseudo-random start block, the same for every problem.
__global__ void start_block_kernel(double* W, int64_t sw, int n)
{
    const int b = blockIdx.y;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n * KB; i += gridDim.x * blockDim.x) {
        unsigned long long x = (unsigned long long)i * 0x9e3779b97f4a7c15ull + 0x243f6a8885a308d3ull;
        x = (x ^ (x >> 30)) * 0xbf58476d1ce4e5b9ull;
        x = (x ^ (x >> 27)) * 0x94d049bb133111ebull;
        x ^= x >> 31;
        W[(size_t)b * sw + i] = (double)(long long)x * 0x1p-63;
    }
}

// ||A x_j - theta_j x_j|| of column j of problem b, one workgroup each.
__global__ __launch_bounds__(256) void ritz_resid_kernel(const double* X, const double* AX, int64_t sx,
                                                         const double* theta, int m, int n, int K, double* res)
{
    __shared__ double red[4];
    const int j = blockIdx.x, b = blockIdx.y;
    const double t = theta[(size_t)b * m + j];
    const size_t o = (size_t)b * sx + (size_t)j * n;
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) {
        const double r = AX[o + i] - t * X[o + i];
        s += r * r;
    }
    s = wave_total(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) res[(size_t)b * K + j] = sqrt(red[0] + red[1] + red[2] + red[3]);
}

// T = X diag(-2 min(theta, 0)) over K columns.
__global__ void reflect_cols_kernel(const double* X, int64_t sx, const double* theta, int m, int n, double* T)
{
    const int j = blockIdx.y, b = blockIdx.z, i = blockIdx.x * blockDim.x + threadIdx.x;
    const double t = theta[(size_t)b * m + j], d = t < 0.0 ? -2.0 * t : 0.0;
    const size_t o = (size_t)b * sx + (size_t)j * n + i;
    if (i < n) T[o] = d * X[o];
}

__global__ void set_ints_kernel(int* x, int n, int v)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = v;
}

int basis_max(int n) { return std::min(KM_MAX, (int)(n * 0.45) / KB * KB); }

}  // namespace

size_t negeig_bytes(int n, int B)
{
    const size_t mm = KM_MAX, b = B;
    return carve_bytes({b * n * KB * 8, b * n * KB * 8, b * mm * KB * 8, b * mm * 8, b * mm * 8, b * 4, b * 4,
                        potrf_work_bytes(n, B)});
}

int abs_factor(hipStream_t s, int n, int B, double* A, double* t0, double* t1, void* scratch, size_t scratch_bytes,
               int* nneg, const EigSolveAt& eig, void* ws, size_t ws_bytes, bool stats, bool* ok)
{
    *ok = false;
    const int mmax = basis_max(n);
    const int64_t nn = (int64_t)n * n;
    if (mmax < KM_FIRST) return 0;
    Arena ar{static_cast<char*>(scratch), scratch_bytes};
    double* W = ar.take<double>((size_t)B * n * KB);
    double* Qt = ar.take<double>((size_t)B * n * KB);
    double* Ct = ar.take<double>((size_t)B * KM_MAX * KB);
    double* theta = ar.take<double>((size_t)B * KM_MAX);
    double* res = ar.take<double>((size_t)B * KM_MAX);
    int* bad = ar.take<int>(B);
    int* info = ar.take<int>(B);
    char* pwork = ar.take<char>(potrf_work_bytes(n, B));
    GMC_CHECK(ar.fits(), "negative eigenpairs: scratch layout overflow");
    // t0: the basis V; t1: A V, then X and A X beside it
    double *V = t0, *AV = t1, *X = t1 + (int64_t)n * mmax;
    const int64_t sw = (int64_t)n * KB, sc = (int64_t)KM_MAX * KB;
    const dim3 gsk((n + SK_ROWS - 1) / SK_ROWS, B), bsk(64 * SK_WAVES);
    ProfScope ps_all(s, "abs_factor", 0.0);
    hipLaunchKernelGGL(set_ints_kernel, dim3((B + 255) / 256), dim3(256), 0, s, bad, B, 0);
    hipLaunchKernelGGL(start_block_kernel, dim3(64, B), dim3(256), 0, s, W, sw, n);
    hipLaunchKernelGGL(cholqr_kernel, dim3(B), dim3(1024), 0, s, W, sw, n, W, sw, nullptr, 0, bad);
    hipLaunchKernelGGL(cholqr_kernel, dim3(B), dim3(1024), 0, s, W, sw, n, V, nn, Qt, sw, bad);
    GMC_HIP(hipGetLastError());
    int m = KB;   // columns of V
    std::vector<double> th, rs;
    std::vector<int> hb(B);
    int K = 0;
    constexpr double tol = 256 * 2.220446049250313e-16;   // (the residual's rounding floor is a few eps of the norm)
    // W orthogonalised against V: the next block of V, and into Qt
    auto next_block = [&]() -> int {
        for (int pass = 0; pass < 2; pass++) {
            hipLaunchKernelGGL(vtw_kernel, dim3(m / KB, B), bsk, 0, s, V, nn, n, W, sw, Ct, sc);
            hipLaunchKernelGGL(skinny_kernel, gsk, bsk, 0, s, V, nn, n, m, Ct, sc, W, sw, nullptr, 0, 1);
            if (pass == 0)
                hipLaunchKernelGGL(cholqr_kernel, dim3(B), dim3(1024), 0, s, W, sw, n, W, sw, nullptr, 0, bad);
            else
                hipLaunchKernelGGL(cholqr_kernel, dim3(B), dim3(1024), 0, s, W, sw, n, V + (int64_t)m * n, nn, Qt, sw,
                                   bad);
        }
        GMC_HIP(hipGetLastError());
        m += KB;
        return 0;
    };
    auto breakdown = [&](bool* any) -> int {
        GMC_HIP(hipMemcpyAsync(hb.data(), bad, B * sizeof(int), hipMemcpyDeviceToHost, s));
        GMC_HIP(hipStreamSynchronize(s));
        *any = false;
        for (int v : hb) *any = *any || v != 0;
        return 0;
    };
    // the caller's eigensolve, and why
    auto give_up = [&](const char* why) {
        if (stats) fprintf(stderr, "[gmc] abs_factor: %s in a basis of %d, the eigensolve takes over\n", why, m);
        return 0;
    };
    for (int goal = KM_FIRST;;) {
        ProfScope ps(s, "abs_factor_krylov", 0.0);
        for (;;) {
            // A times the newest block; W starts as that
            hipLaunchKernelGGL(skinny_kernel, gsk, bsk, 0, s, A, nn, n, n, Qt, sw, AV + (int64_t)(m - KB) * n, nn, W, sw,
                               0);
            GMC_HIP(hipGetLastError());
            if (m == goal) break;
            GMC_TRY(next_block());
            // an exhausted space is noticed here, not after the Ritz problem (at few
            // sizes: a wait leaves the GPU idle for 40 us)
            if (m == 8 * KB || m == 16 * KB || m == 32 * KB) {
                bool any;
                GMC_TRY(breakdown(&any));
                if (any) return give_up("breakdown");
            }
        }
        ps.close();
        // Rayleigh-Ritz: H = V^T (A V)
        ProfScope ps2(s, "abs_factor_ritz", 0.0);
        const int64_t mm = (int64_t)m * m;
        const size_t hbytes = align_up((size_t)B * mm * 8);
        GMC_CHECK(ws_bytes > hbytes, "Ritz problem: workspace");
        double* H = static_cast<double*>(ws);   // its eigenvectors after eig
        GemmShape gh{m, m, n, true, false, n, n, m, nn, nn, mm, B, 0};
        GMC_TRY(gemm_big<double>(s, gh, 1.0, V, AV, 0.0, H));
        GMC_TRY(eig(H, theta, m, B, static_cast<char*>(ws) + hbytes, ws_bytes - hbytes));
        th.resize((size_t)B * m);
        GMC_HIP(hipMemcpyAsync(th.data(), theta, th.size() * 8, hipMemcpyDeviceToHost, s));
        K = 0;
        std::vector<int> nb(B, 0);
        bool broken;
        GMC_TRY(breakdown(&broken));
        for (int b = 0; b < B; b++) {
            while (nb[b] < m && th[(size_t)b * m + nb[b]] < 0.0) nb[b]++;
            K = std::max(K, nb[b]);
            broken = broken || !std::isfinite(th[(size_t)b * m]) || !std::isfinite(th[(size_t)b * m + m - 1]);
        }
        K = (K + 1) / 2 * 2;
        if (broken) return give_up("breakdown");
        if (K > m / 4) return give_up("too many pairs below zero");
        double worst = 0.0;
        if (K > 0) {
            // Ritz vectors and their residuals
            GemmShape gx{n, K, m, false, false, n, m, n, nn, mm, nn, B, 0};
            GMC_TRY(gemm_big<double>(s, gx, 1.0, V, H, 0.0, X));
            GMC_TRY(gemm_big<double>(s, gx, 1.0, AV, H, 0.0, X + (int64_t)n * K));
            hipLaunchKernelGGL(ritz_resid_kernel, dim3(K, B), dim3(256), 0, s, X, X + (int64_t)n * K, nn, theta, m, n, K,
                               res);
            GMC_HIP(hipGetLastError());
            rs.resize((size_t)B * K);
            GMC_HIP(hipMemcpyAsync(rs.data(), res, rs.size() * 8, hipMemcpyDeviceToHost, s));
            GMC_HIP(hipStreamSynchronize(s));
            for (int b = 0; b < B; b++) {
                const double norm = std::max(std::fabs(th[(size_t)b * m]), std::fabs(th[(size_t)b * m + m - 1]));
                for (int j = 0; j < nb[b]; j++) {
                    const double r = rs[(size_t)b * K + j] / norm;
                    if (!std::isfinite(r)) return give_up("a residual that is not finite");
                    worst = std::max(worst, r);
                }
            }
        }
        if (stats)
            fprintf(stderr, "[gmc] Cholesky route: restricted step on a basis of %d, %d pairs below zero, residual %.2e\n", m, K,
                    worst);
        if (worst <= tol) {
            GMC_HIP(hipMemcpyAsync(nneg, nb.data(), B * sizeof(int), hipMemcpyHostToDevice, s));
            GMC_HIP(hipStreamSynchronize(s));   // (nb leaves the scope)
            break;
        }
        // a block gains a factor of 2.1 to 2.5 (orders 2236 to 2444, 11 to 40 pairs):
        // no further where even e each would not do
        const double gap = std::log(worst / tol);
        if (m + KB * (int)std::ceil(gap) > mmax) return give_up("no convergence");
        goal = std::min(mmax, m + KB * std::max(4, std::min(24, (int)std::ceil(gap / 0.8) + 1)));
        // the basis grows on: the newest block's A Q was formed, its successor was not
        GMC_TRY(next_block());
    }
    if (K > 0) {
        // |A| on the lower triangle
        double* T = X + (int64_t)n * K;
        hipLaunchKernelGGL(reflect_cols_kernel, dim3((n + 255) / 256, K, B), dim3(256), 0, s, X, nn, theta, m, n, T);
        GemmShape gr{n, n, K, false, true, n, n, n, nn, nn, nn, B, 1};
        GMC_TRY(gemm<double>(s, gr, 1.0, T, X, 1.0, A));
        GMC_HIP(hipGetLastError());
    }
    GMC_TRY(potrf_batched(s, n, B, A, pwork, info));
    GMC_HIP(hipMemcpyAsync(hb.data(), info, B * sizeof(int), hipMemcpyDeviceToHost, s));
    GMC_HIP(hipStreamSynchronize(s));
    int failed = 0;
    for (int v : hb) failed += v != 0;
    if (failed) {
        if (stats) fprintf(stderr, "[gmc] Cholesky route: %d of %d factorisations failed\n", failed, B);
        return give_up("a pivot of |A| not above zero");
    }
    if (stats) fprintf(stderr, "[gmc] abs_factor: |A| factored\n");
    *ok = true;
    return 0;
}

}  // namespace gmc
