// 4-index AO -> NO transformation of 8-fold packed integrals (the work of
// TwoNO1, misc.f:166-317):
//   (ab|cd) = sum U[a,m] U[b,n] U[c,l] U[d,s] (mn|ls),   U = URe(NO, AO)
//
// Pipeline on one GPU, T = N(N+1)/2 pair index, everything int64-addressed:
//   1. expand     packed lower triangle (NInte2) -> dense symmetric V (T x T)
//   2. half       for every column kl of V: Z = U * unpack(V[:,kl]) * U^T,
//                 the b<=a half of Z into column kl of H (T x T)
//   3. transpose  H -> V
//   4. half       for every column ab of V: Z = U * unpack(V[:,ab]) * U^T,
//                 the pairs cd <= ab straight into row ab of the packed
//                 output, which is the input array (in place).
// A half transform is one launch: see half_transform_kernel.
#include "common.hpp"
#include "gemm_tile.hpp"
#include "transform.hpp"
#include "prof.hpp"

namespace gmc {

// ---------------------------------------------------------------- expand
// Tile (rb, cb) with rb >= cb of the T x T pair matrix.  Packed row r holds
// V[r, 0..r] contiguously.
__global__ __launch_bounds__(256) void expand_kernel(const double* __restrict__ packed, double* __restrict__ V,
                                                       int64_t T)
{
    __shared__ double tile[64][65];
    const int64_t nbt = (T + 63) / 64;
    // blockIdx.x enumerates lower-triangular tiles
    int64_t t = blockIdx.x;
    int64_t rb = (int64_t)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while ((rb + 1) * (rb + 2) / 2 <= t) rb++;
    while (rb * (rb + 1) / 2 > t) rb--;
    int64_t cb = t - rb * (rb + 1) / 2;
    if (rb >= nbt) return;
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int64_t r0 = rb * 64, c0 = cb * 64;
    for (int y = ty; y < 64; y += 4) {
        int64_t r = r0 + y, c = c0 + tx;
        double v = 0.0;
        if (r < T && c <= r) v = packed[r * (r + 1) / 2 + c];
        tile[y][tx] = v;
    }
    __syncthreads();
    // V[c + r*T] (column r, rows c) from tile row y
    for (int y = ty; y < 64; y += 4) {
        int64_t r = r0 + y, c = c0 + tx;
        if (r < T && c <= r) V[c + r * T] = tile[y][tx];
    }
    // V[r + c*T] (column c, rows r) from tile column
    for (int y = ty; y < 64; y += 4) {
        int64_t c = c0 + y, r = r0 + tx;
        if (r < T && c <= r) V[r + c * T] = tile[tx][y];
    }
}

// ---------------------------------------------------------------- transpose
__global__ __launch_bounds__(256) void transpose_kernel(const double* __restrict__ A, double* __restrict__ B,
                                                          int64_t T)
{
    __shared__ double tile[64][65];
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int64_t r0 = (int64_t)blockIdx.x * 64, c0 = (int64_t)blockIdx.y * 64;
    for (int y = ty; y < 64; y += 4) {
        int64_t r = r0 + tx, c = c0 + y;
        tile[y][tx] = (r < T && c < T) ? A[r + c * T] : 0.0;
    }
    __syncthreads();
    for (int y = ty; y < 64; y += 4) {
        int64_t c = c0 + tx, r = r0 + y;
        if (r < T && c < T) B[c + r * T] = tile[tx][y];
    }
}

// ---------------------------------------------------------------- half transform
int transform_plan(int N, TransformPlan* p)
{
    p->N = N;
    p->T = (int64_t)N * (N + 1) / 2;
    p->scratch_bytes = 2 * align_up((size_t)p->T * p->T * sizeof(double));
    return 0;
}

constexpr int HT_ROWS = 32;   // rows of U (and of Z) per workgroup
constexpr int HT_NG = 2;      // column blocks of Z a wave forms together, at most

// A double at a byte offset of a buffer; past its end it is zero, which is what
// the padding of N to blocks of 16 needs.
__device__ inline double buf1(__amdgpu_buffer_rsrc_t r, int o)
{
    return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0));
}

// NR blocks of 16 rows of Z = Y U^T, Y rows in LDS from row y0 on (see below),
// for NG column blocks b0, b0 + ST, ..., the pairs b <= a stored.
template <int ST, int NR, int NG, class Store>
__device__ inline void half_z_blocks(const double* Yl, __amdgpu_buffer_rsrc_t U, int N, int nsl, int y0, int b0, int lane,
                                     const Store& store)
{
    const int jl = lane & 15, kg = lane >> 4;
    v4d acc[NR][NG];
#pragma unroll
    for (int r = 0; r < NR; r++)
#pragma unroll
        for (int i = 0; i < NG; i++) acc[r][i] = v4d{0, 0, 0, 0};
    const int uv = 8 * (16 * b0 + jl + kg * N), kstep = 4 * 8 * N;
    // (k = 16 ks + 4 s + kg; an odd kg is an odd k)
    const double* yl = Yl + kg * HT_ROWS + ((y0 + jl) ^ ((kg & 1) << 4));
    const int y1 = (kg & 1) ? -16 : 16;   // the second block of rows
    double ya[NR][4], yb[NR][4], ua[NG][4], ubf[NG][4];
    auto load = [&](int ks, double (&y)[NR][4], double (&u)[NG][4]) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
#pragma unroll
            for (int r = 0; r < NR; r++) y[r][s] = yl[(16 * ks + 4 * s) * HT_ROWS + (r ? y1 : 0)];
#pragma unroll
            for (int i = 0; i < NG; i++) u[i][s] = buf1(U, uv + (4 * ks + s) * kstep + 128 * ST * i);
        }
    };
    auto mul = [&](const double (&y)[NR][4], const double (&u)[NG][4]) {
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < NG; i++)
#pragma unroll
                for (int r = 0; r < NR; r++)
                    acc[r][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[r][s], u[i][s], acc[r][i], 0, 0, 0);
    };
    load(0, ya, ua);
    for (int ks = 0; ks < nsl; ks += 2) {
        if (ks + 1 < nsl) load(ks + 1, yb, ubf);
        mul(ya, ua);
        if (ks + 1 < nsl) {
            if (ks + 2 < nsl) load(ks + 2, ya, ua);
            mul(yb, ubf);
        }
    }
#pragma unroll
    for (int r = 0; r < NR; r++)
#pragma unroll
        for (int i = 0; i < NG; i++) store(r, 16 * (b0 + ST * i) + jl, acc[r][i]);
}
// The same for the first min(left, NG) of the blocks.
template <int ST, int NR, int NG, class Store>
__device__ inline void half_z_some(int left, const double* Yl, __amdgpu_buffer_rsrc_t U, int N, int nsl, int y0, int b0,
                                   int lane, const Store& store)
{
    if constexpr (NG > 1)
        if (left < NG) return half_z_some<ST, NR, NG - 1>(left, Yl, U, N, nsl, y0, b0, lane, store);
    half_z_blocks<ST, NR, NG>(Yl, U, N, nsl, y0, b0, lane, store);
}

// NR blocks of 16 rows of Y = U M from row block rb on, for NB column blocks g,
// g + ST, ..., into LDS rows from y0 on: M the symmetric matrix packed in col.
template <int ST, int NR, int NB>
__device__ inline void half_y_blocks(__amdgpu_buffer_rsrc_t col, __amdgpu_buffer_rsrc_t U, int N, int nsl, int rb, int y0,
                                     int g, int lane, double* Yl)
{
    const int jl = lane & 15, kg = lane >> 4;
    v4d acc[NR][NB];
    int jt[NB], j8[NB];   // packed row of column j and k = kg in it, column j: bytes
#pragma unroll
    for (int i = 0; i < NB; i++) {
        const int j = 16 * (g + ST * i) + jl;
        jt[i] = 8 * (j * (j + 1) / 2 + kg);
        j8[i] = 8 * j;
#pragma unroll
        for (int r = 0; r < NR; r++) acc[r][i] = v4d{0, 0, 0, 0};
    }
    const int uv = 8 * (16 * rb + jl + kg * N), kstep = 4 * 8 * N;
    double ua[NR][4], ubf[NR][4], ma[NB][4], mb[NB][4];
    // (every path has the same loads, so that a wait for one slab's never
    // reaches into the next one's)
    auto load = [&](int ks, double (&u)[NR][4], double (&m)[NB][4]) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
            const int k = 16 * ks + 4 * s + kg, kt = 8 * (k * (k + 1) / 2), k8 = 8 * k;
#pragma unroll
            for (int r = 0; r < NR; r++) u[r][s] = buf1(U, uv + (4 * ks + s) * kstep + 128 * r);
#pragma unroll
            for (int i = 0; i < NB; i++)
                m[i][s] = buf1(col, k8 >= j8[i] ? kt + j8[i] : jt[i] + 128 * ks + 32 * s);
        }
    };
    // (formed transposed: the registers hold 16 rows a of one column)
    auto mul = [&](const double (&u)[NR][4], const double (&m)[NB][4]) {
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int i = 0; i < NB; i++)
#pragma unroll
                for (int r = 0; r < NR; r++)
                    acc[r][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(m[i][s], u[r][s], acc[r][i], 0, 0, 0);
    };
    load(0, ua, ma);
    for (int ks = 0; ks < nsl; ks += 2) {
        if (ks + 1 < nsl) load(ks + 1, ubf, mb);
        mul(ua, ma);
        if (ks + 1 < nsl) {
            if (ks + 2 < nsl) load(ks + 2, ua, ma);
            mul(ubf, mb);
        }
    }
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int k = 16 * (g + ST * i) + kg + 4 * q;
#pragma unroll
            for (int r = 0; r < NR; r++) Yl[k * HT_ROWS + ((y0 + 16 * r + jl) ^ ((k & 1) << 4))] = acc[r][i][q];
        }
}
// The same for the first min(left, NB) of the blocks.
template <int ST, int NR, int NB>
__device__ inline void half_y_some(int left, __amdgpu_buffer_rsrc_t col, __amdgpu_buffer_rsrc_t U, int N, int nsl, int rb,
                                   int y0, int g, int lane, double* Yl)
{
    if constexpr (NB > 1)
        if (left < NB) return half_y_some<ST, NR, NB - 1>(left, col, U, N, nsl, rb, y0, g, lane, Yl);
    half_y_blocks<ST, NR, NB>(col, U, N, nsl, rb, y0, g, lane, Yl);
}

// Z = U M U^T of one column c of S, M its unpacked symmetric matrix, for 32
// rows of Z: Y = U M (32 x N) stays in LDS, then the b <= a half of Y U^T goes
// straight to its packed place: column c of H (mode 0), or the pairs <= c of
// row c of the packed result (mode 1; rows past c's own a are not formed).
//
// Bound by the FP64 matrix rate, then by the L1's: an MFMA takes 64 cycles, so
// its operands come from L2 without a detour through LDS, 16 values of k
// ahead, but at 64 bytes a cycle a wave has to use them for two blocks of rows
// where there are enough column blocks to go round: ST = 4, a wave has all 32
// rows and every fourth block of 16 columns, starting at another one from
// panel to panel.  ST = 2, small N: 16 rows and every second block.  Lane l
// supplies k = l / 16 + 4 s: four consecutive packed elements where the column
// index j is the larger, one row's 16 columns where k is.  Y lies k-major, rows
// xor 16 (k & 1): conflict-free both ways.  The panels of a column run on one
// XCD, whose L2 then reads it once.
// NB = 2 column blocks at a time leave registers for three workgroups per compute
// unit (LDS for three up to N = 208, for two above), whose waits then overlap: whole
// transform at N = 200 21.5 ms against
// 26.2 with NB = 4 and two workgroups, and against 47.6 as gather, two library
// products per column and scatter (37 TFLOP/s of a product twice this work; N =
// 48 0.153 -> 0.083 ms, 160 about 18 -> 7.1).
template <int ST, int NB>
__global__ __launch_bounds__(256, 3) void half_transform_kernel(const double* __restrict__ S, int64_t T, int N, int np,
                                                                const double* __restrict__ U, int mode,
                                                                double* __restrict__ out)
{
    extern __shared__ double Yl[];
    constexpr int NR = ST / 2;   // blocks of rows of a wave, at most
    const int y = blockIdx.x >> 3, panel = y % np;
    const int64_t c = (int64_t)(y / np) * 8 + (blockIdx.x & 7);
    if (c >= T) return;
    int amax = N - 1;
    if (mode == 1) {
        amax = (int)((sqrt(8.0 * (double)c + 1.0) - 1.0) * 0.5);
        while ((int64_t)(amax + 1) * (amax + 2) / 2 <= c) amax++;
        while ((int64_t)amax * (amax + 1) / 2 > c) amax--;
    }
    if (HT_ROWS * panel > amax) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int rb = 2 * panel + (ST == 2 ? wave & 1 : 0), y0 = 16 * (rb - 2 * panel);
    const int first = ST == 2 ? wave >> 1 : (wave + panel) & 3, kg = lane >> 4;
    const int nsl = (N + 15) / 16;   // blocks of 16
    // blocks of rows of this wave: NR, or the one (or none) that is left
    const int nr = min(NR, amax / 16 + 1 - rb);
    const __amdgpu_buffer_rsrc_t ub = __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(U), 0, 8 * N * N, 0x20000);
    const __amdgpu_buffer_rsrc_t cb =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(S + c * T), 0, 8 * (int)T, 0x20000);
    if (nr > 0)
        for (int g = first; g < nsl; g += ST * NB) {
            const int left = (nsl - 1 - g) / ST + 1;
            if (nr == NR) half_y_some<ST, NR, NB>(left, cb, ub, N, nsl, rb, y0, g, lane, Yl);
            else half_y_some<ST, 1, NB>(left, cb, ub, N, nsl, rb, y0, g, lane, Yl);
        }
    __syncthreads();
    if (nr <= 0) return;
    double* dst = mode == 0 ? out + c * T : out + c * (c + 1) / 2;
    const int last = mode == 0 ? (int)T - 1 : (int)c;
    auto store = [&](int r, int b, const v4d& z) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int a = 16 * (rb + r) + kg + 4 * q;
            const int pr = a * (a + 1) / 2 + b;
            if (a < N && b <= a && pr <= last) dst[pr] = z[q];
        }
    };
    const int rl = rb + nr - 1;
    for (int b0 = first; b0 <= rl; b0 += ST * HT_NG) {
        const int left = (rl - b0) / ST + 1;
        if (nr == NR) half_z_some<ST, NR, HT_NG>(left, Yl, ub, N, nsl, y0, b0, lane, store);
        else half_z_some<ST, 1, HT_NG>(left, Yl, ub, N, nsl, y0, b0, lane, store);
    }
}

static int half_transform(hipStream_t s, const TransformPlan& p, const double* S, const double* U, double* out, int mode)
{
    const int N = p.N, nsl = (N + 15) / 16, np = (N + HT_ROWS - 1) / HT_ROWS;
    const size_t lds = (size_t)nsl * 16 * HT_ROWS * sizeof(double);
    GMC_CHECK(lds <= 160 * 1024, "transform: N=%d needs %zu bytes of LDS per workgroup", N, lds);
    const int64_t wgs = (p.T + 7) / 8 * 8 * np;
    GMC_CHECK(wgs < (1LL << 31), "transform: %lld workgroups", (long long)wgs);
    // up to 64 orbitals (four blocks) a wave of 32 rows would leave others idle
    // (both ways, ms: N = 64 0.156 / 0.156, 80 0.355 / 0.333, 128 3.27 / 2.74)
    const int st = nsl <= 4 ? 2 : 4;
    using K = void (*)(const double*, int64_t, int, int, const double*, int, double*);
    const K k = nsl <= st ? (st == 2 ? (K)half_transform_kernel<2, 1> : (K)half_transform_kernel<4, 1>)
                          : (st == 2 ? (K)half_transform_kernel<2, 2> : (K)half_transform_kernel<4, 2>);
    hipStreamCaptureStatus cst = hipStreamCaptureStatusNone;
    GMC_HIP(hipStreamIsCapturing(s, &cst));
    if (lds > 64 * 1024 && cst == hipStreamCaptureStatusNone)
        GMC_HIP(hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(k, dim3((unsigned)wgs), dim3(256), lds, s, S, p.T, N, np, U, mode, out);
    GMC_HIP(hipGetLastError());
    return 0;
}

int twono1_device(hipStream_t s, const TransformPlan& p, double* tno, const double* U, void* scratch)
{
    double* V = static_cast<double*>(scratch);
    double* H = reinterpret_cast<double*>(static_cast<char*>(scratch) + align_up((size_t)p.T * p.T * sizeof(double)));
    ProfScope ps(s, "twono1", 8.0 * (double)p.N * p.N * p.N * (double)p.T);
    const int64_t nbt = (p.T + 63) / 64;
    hipLaunchKernelGGL(expand_kernel, dim3((unsigned)(nbt * (nbt + 1) / 2)), dim3(256), 0, s, tno, V, p.T);
    GMC_HIP(hipGetLastError());
    GMC_TRY(half_transform(s, p, V, U, H, 0));
    hipLaunchKernelGGL(transpose_kernel, dim3((unsigned)nbt, (unsigned)nbt), dim3(256), 0, s, H, V, p.T);
    GMC_HIP(hipGetLastError());
    GMC_TRY(half_transform(s, p, V, U, tno, 1));
    return 0;
}

}  // namespace gmc
