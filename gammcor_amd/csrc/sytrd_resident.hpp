// Tridiagonalisation of trailing problems that fit in the register files of
// the GPU: one persistent launch holds the whole matrix in registers and
// applies every rank-2 update at once (no panels, no trailing products).
// Workgroup gi of a problem keeps the rows gi, gi + G, ... (at most R of
// them), thread t their columns t, t + blockDim, ... (at most C), both
// triangles.
//
// What bounds it is the latency of one exchange per column, so there is only
// one: each workgroup publishes, for its own rows r, w_r = tau (A v)_r and
// a_r = A(r, j+1), and every workgroup forms a2, w' = w + a2 v, column j+1 of
// the updated matrix and its reflector redundantly from them, then updates
// and multiplies its own rows.  (The panel kernel's lower-triangle SYMV
// needs two exchanges: its scatter sums must be collected before w exists.)
// A value travels in 8-byte words of 32 data bits and the column's epoch,
// stored and polled as relaxed agent-scope atomics: no flag, no fence and no
// cache-wide write-back, the words themselves say when they are there.  Two
// buffers suffice: a workgroup publishes epoch e + 2 only after it has read
// every row's e + 1, which each owner publishes after it has read e; a
// workgroup whose rows are all done has nothing left to read and leaves.
//
// Every sum is formed in a fixed order, so the result does not depend on
// timing (it serves the deterministic mode as it is).
//
// Measured, tridiagonalisation alone, panels and trailing updates -> here:
//   order x problems    410 x 8        1281 x 1        2048 x 1        1024 x 8
//   FP64             6.7 -> 1.4 ms  23.5 -> 5.3 ms  39.3 -> 9.2 ms  20.7 -> 4.8 ms
//   FP32             7.0 -> 1.1 ms  25.7 -> 4.4 ms  45.9 -> 7.2 ms  22.2 -> 3.5 ms
// 3.3 us per column at order 410, about half of it the exchange; the FP64
// update and product of R C elements per thread are most of the rest at 2048.
//
// Included by eigen.hip only, inside its namespace.
#pragma once

constexpr int RES_THREADS = 512, RES_WAVES = RES_THREADS / 64;
constexpr int RES_CH = 16;   // own rows whose products are reduced together
constexpr int RES_WAIT = 14;   // pause before a column's first poll, in units of 64 clocks

template <class T>
struct ResArgs {
    T *A, *d, *e, *tau;
    unsigned long long* ring;   // per problem 2 buffers x m rows x res_words, zero on entry
    int* err;
    int n, j0, G;               // order (ld and stride of A, d, e, tau), first column, workgroups per problem
};

// Words of one row's (w, a).
template <class T>
constexpr int res_words() { return 2 * (int)(sizeof(T) / 4); }

// Half h of a row's packet (0: w, 1: a).
__device__ inline void res_put(unsigned long long* q, int h, float x, unsigned ep)
{
    const unsigned long long t = (unsigned long long)ep << 32;
    __hip_atomic_store(q + h, t | __float_as_uint(x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void res_put(unsigned long long* q, int h, double x, unsigned ep)
{
    const unsigned long long t = (unsigned long long)ep << 32, b = (unsigned long long)__double_as_longlong(x);
    __hip_atomic_store(q + 2 * h, t | (b & 0xffffffffull), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(q + 2 * h + 1, t | (b >> 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ inline void res_unpack(const unsigned long long (&x)[2], float& w, float& a)
{
    w = __uint_as_float((unsigned)x[0]);
    a = __uint_as_float((unsigned)x[1]);
}
__device__ inline void res_unpack(const unsigned long long (&x)[4], double& w, double& a)
{
    w = __longlong_as_double((long long)((x[1] << 32) | (x[0] & 0xffffffffull)));
    a = __longlong_as_double((long long)((x[3] << 32) | (x[2] & 0xffffffffull)));
}
// Dynamic LDS of the kernel for a trailing order m.
template <class T>
constexpr size_t res_lds(int m, int R) { return ((size_t)m + 2 * RES_WAVES + 4 + 2 * R + (size_t)RES_WAVES * R) * sizeof(T); }

template <class T, int R, int C>
__global__ __launch_bounds__(RES_THREADS) void sytrd_resident_kernel(ResArgs<T> g)
{
    constexpr int NW = res_words<T>();
    constexpr int CH = R < RES_CH ? R : RES_CH, NCH = R / CH;
    extern __shared__ char smem[];
    const int n = g.n, m = g.n - g.j0, G = g.G;
    // (a problem's workgroups on one XCD where G allows it, as in the panel kernel)
    const int nwg = (int)gridDim.x;
    const int lin = (nwg % 8 == 0 && (nwg / 8) % G == 0) ? (int)(blockIdx.x & 7) * (nwg / 8) + (int)(blockIdx.x >> 3)
                                                      : (int)blockIdx.x;
    const int p = lin / G, gi = lin % G;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, NT = blockDim.x, nwave = NT >> 6;
    T* A = g.A + (size_t)p * n * n + g.j0 + (size_t)g.j0 * n;   // the trailing matrix, ld n
    unsigned long long* ring = g.ring + (size_t)p * 2 * m * NW;
    T* dd = g.d + (size_t)p * n + g.j0;
    T* ee = g.e + (size_t)p * n + g.j0;
    T* tt = g.tau + (size_t)p * n + g.j0;
    T* lx = reinterpret_cast<T*>(smem);   // m: column j
    T* redA = lx + m;                     // RES_WAVES
    T* redB = redA + RES_WAVES;           // RES_WAVES
    T* sc = redB + RES_WAVES;             // [0] w(j) [1] x(j) [2] x(j+1)
    T* acol = sc + 4;                     // R: own rows' entries of column j+1
    T* wown = acol + R;                   // R: own rows' w
    T* part = wown + R;                   // RES_WAVES x R: the waves' parts of own rows' products

    T a[R][C], v[C], x[C], vown[NCH];
#pragma unroll
    for (int q = 0; q < R; q++) {
        const int r = q * G + gi;
#pragma unroll
        for (int k = 0; k < C; k++) {
            const int c = tid + k * NT;
            a[q][k] = r < m && c < m ? (c >= r ? A[c + (size_t)r * n] : A[r + (size_t)c * n]) : T(0);
        }
    }
    // column 0 arrives final
#pragma unroll
    for (int k = 0; k < C; k++) {
        const int c = tid + k * NT;
        v[k] = T(0);
        x[k] = c < m ? A[c] : T(0);
    }
#pragma unroll
    for (int h = 0; h < NCH; h++) vown[h] = T(0);
    const int rlast = gi < m ? (m - 1 - gi) / G * G + gi : -1;   // last own row
    T tau = 0;
    for (int j = 0; j < m - 1 && rlast > j; j++) {
        T wp[C], a2 = 0;
#pragma unroll
        for (int k = 0; k < C; k++) wp[k] = T(0);
        if (j > 0) {
            // w of column j - 1 and the entries of column j from their owners.
            // The words take longer than RES_WAIT to arrive, and polls that
            // fail delay them for everyone (8 problems of order 410: 2.9 ms
            // polled at once, 1.36 ms with a pause of 12 to 16, 1.53 ms with 32)
            __builtin_amdgcn_s_sleep(RES_WAIT);
            const unsigned long long* buf = ring + (size_t)(j & 1) * m * NW;
            T wc[C], ac[C], s1 = 0;
#pragma unroll
            for (int k = 0; k < C; k++) {
                const int c = tid + k * NT;
                wc[k] = ac[k] = T(0);
                if (c >= j && c < m) {
                    unsigned long long q[NW];
                    const unsigned long long* src = buf + (size_t)c * NW;
                    for (long spins = 0;; spins++) {
                        bool ok = true;
#pragma unroll
                        for (int i = 0; i < NW; i++)
                            q[i] = __hip_atomic_load(src + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                        for (int i = 0; i < NW; i++) ok = ok && (unsigned)(q[i] >> 32) == (unsigned)j;
                        if (ok) break;
                        if ((spins & 63) == 63) {
                            if (__hip_atomic_load(g.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) break;
                            if (spins > (1L << 21)) {   // seconds of polling: a lost workgroup
                                atomicExch(g.err, 1);
                                break;
                            }
                        }
                    }
                    res_unpack(q, wc[k], ac[k]);
                    if (c == j) sc[0] = wc[k];
                } else {
                    v[k] = T(0);
                }
                s1 += wc[k] * v[k];
            }
            s1 = wave_total(s1);
            if (lane == 0) redA[wave] = s1;
            lds_barrier();
            s1 = T(0);
            for (int i = 0; i < nwave; i++) s1 += redA[i];
            // a2 = -tau/2 w^T v, w' = w + a2 v, column j less v w'(j) + w' v(j), v(j) = 1
            a2 = T(-0.5) * tau * s1;
            const T wj = sc[0] + a2;
#pragma unroll
            for (int k = 0; k < C; k++) {
                wp[k] = wc[k] + a2 * v[k];
                x[k] = ac[k] - v[k] * wj - wp[k];
            }
        }
        // the column: its head, and the tail's entries xt with their norm
        T nrm = 0, xt[C];
#pragma unroll
        for (int k = 0; k < C; k++) {
            const int c = tid + k * NT;
            xt[k] = c > j + 1 && c < m ? x[k] : T(0);
            nrm += xt[k] * xt[k];
            if (c == j) sc[1] = x[k];
            if (c == j + 1) sc[2] = x[k];
            if (c < m) lx[c] = x[k];
        }
        // own rows: the last column's rank-2 update and the product with the
        // tail (v = scal xt + e_j+1 follows from it once the reflector is
        // known), RES_CH rows at a time; finished rows are skipped by fours
#pragma unroll
        for (int h = 0; h < NCH; h++) {
            const int q0 = h * CH;
            // row q0 + l in lane l (< CH)
            const T vr_l = vown[h], wr_l = j > 0 ? wown[q0 + (lane & (CH - 1))] + a2 * vr_l : T(0);
            T acc[CH];
#pragma unroll
            for (int q = 0; q < CH; q++) acc[q] = T(0);
#pragma unroll
            for (int q4 = 0; q4 < CH; q4 += 4) {
                if ((q0 + q4 + 3) * G + gi <= j) continue;
#pragma unroll
                for (int q = q4; q < q4 + 4; q++) {
                    const T vr = read_lane(vr_l, q), wr = read_lane(wr_l, q);
#pragma unroll
                    for (int k = 0; k < C; k++) {
                        a[q0 + q][k] -= vr * wp[k] + wr * v[k];
                        acc[q] += a[q0 + q][k] * xt[k];
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < C; k++)
                if (tid + k * NT == j + 1) {
#pragma unroll
                    for (int q = 0; q < CH; q++) acol[q0 + q] = a[q0 + q][k];
                }
            const T s = wave_col_sums<CH>(acc, lane);
            constexpr int SH = 6 - ilog2<CH>();
            if ((lane & ((1 << SH) - 1)) == 0) part[wave * R + q0 + (lane >> SH)] = s;
        }
        nrm = wave_total(nrm);
        if (lane == 0) redB[wave] = nrm;
        lds_barrier();
        // the reflector
        T xn2 = 0;
        for (int i = 0; i < nwave; i++) xn2 += redB[i];
        const T alpha = sc[2];
        T beta = alpha, scal = 0;
        tau = 0;
        if (xn2 != T(0)) {
            beta = -copysign(sqrt(alpha * alpha + xn2), alpha);
            tau = (beta - alpha) / beta;
            scal = T(1) / (alpha - beta);
        }
        if (j < m - 2) {
            unsigned long long* buf = ring + (size_t)((j + 1) & 1) * m * NW;
            for (int i = tid; i < 2 * R; i += NT) {
                const int q = i % R, h = i / R, r = q * G + gi;
                T val = acol[q];
                if (h == 0) {
                    T s = 0;
                    for (int w = 0; w < nwave; w++) s += part[w * R + q];
                    val = tau * (scal * s + val);
                    wown[q] = val;
                }
                if (r > j && r < m) res_put(buf + (size_t)r * NW, h, val, (unsigned)(j + 1));
            }
        }
        // the owner of row j + 1 stores the reflector (column 0 waits for
        // step 1: by then every workgroup has loaded its rows)
        const bool writer = (j + 1) % G == gi;
        if (writer && tid == 0) {
            dd[j] = sc[1];
            ee[j] = beta;
            tt[j] = tau;
            // the last diagonal element (sytrd_finish_kernel moves it to d)
            if (j == m - 2) A[(size_t)(m - 1) * n + m - 1] = acol[(m - 1) / G];
        }
#pragma unroll
        for (int k = 0; k < C; k++) {
            const int c = tid + k * NT;
            if (writer && j == 1 && c >= 1 && c < m) A[c] = v[k];
            v[k] = c == j + 1 ? T(1) : scal * xt[k];
            if (writer && c > j && c < m && (j > 0 || m == 2)) A[c + (size_t)j * n] = v[k];
        }
#pragma unroll
        for (int h = 0; h < NCH; h++) {
            const int r = (h * CH + (lane & (CH - 1))) * G + gi;
            vown[h] = r == j + 1 ? T(1) : (r > j + 1 && r < m ? scal * lx[r] : T(0));
        }
    }
}

// Shape of the resident kernel for B problems of trailing order m on ncu
// compute units: C columns per thread, R rows and G workgroups per problem,
// NT threads.  All B G workgroups must be resident at once, one per compute
// unit, and a thread's R C matrix elements must leave it registers to work
// with (R C <= 64: 240 of 256 at FP64, nothing spilled).  The fewest rows
// that fit are the fastest (1024 x 1: R = 8 / 16 / 32 took 4.2 / 4.6 / 5.6 ms).
struct ResShape {
    int R = 0, C = 0, G = 0, NT = 0;
};
inline ResShape res_shape(int m, int B, int ncu)
{
    ResShape s;
    if (m < 2 || m > 4 * RES_THREADS) return s;
    const int C = (m + RES_THREADS - 1) / RES_THREADS;
    const int rmax = C == 1 ? 64 : C == 2 ? 32 : 16;
    for (int R = 8; R <= rmax; R *= 2) {
        const int G = (m + R - 1) / R;
        if ((long)B * G > ncu) continue;
        s.R = R;
        s.C = C;
        s.G = G;
        s.NT = ((m + C - 1) / C + 63) / 64 * 64;
        return s;
    }
    return s;
}
// Largest trailing order the resident kernel takes (0: none).
inline int res_max(int B, int ncu)
{
    int m = 4 * RES_THREADS;
    while (m >= 2 && res_shape(m, B, ncu).R == 0) m--;
    return m >= 2 ? m : 0;
}
template <class T>
const void* res_kernel(int R, int C)
{
    switch (C * 100 + R) {
        case 108: return (const void*)sytrd_resident_kernel<T, 8, 1>;
        case 116: return (const void*)sytrd_resident_kernel<T, 16, 1>;
        case 132: return (const void*)sytrd_resident_kernel<T, 32, 1>;
        case 164: return (const void*)sytrd_resident_kernel<T, 64, 1>;
        case 208: return (const void*)sytrd_resident_kernel<T, 8, 2>;
        case 216: return (const void*)sytrd_resident_kernel<T, 16, 2>;
        case 232: return (const void*)sytrd_resident_kernel<T, 32, 2>;
        case 308: return (const void*)sytrd_resident_kernel<T, 8, 3>;
        case 316: return (const void*)sytrd_resident_kernel<T, 16, 3>;
        case 408: return (const void*)sytrd_resident_kernel<T, 8, 4>;
        case 416: return (const void*)sytrd_resident_kernel<T, 16, 4>;
    }
    return nullptr;
}
