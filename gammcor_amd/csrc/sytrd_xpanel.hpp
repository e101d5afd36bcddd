// Panel of the blocked tridiagonalisation (see sytrd_panel_kernel for the
// algorithm and the row ownership) with its exchanges in self-validating
// words: what a workgroup tells the others travels as 8-byte words of 32 data
// bits and the column's epoch (relaxed agent-scope atomics, polled by the
// reader) instead of plain stores between group barriers.  A barrier costs its fences (write-back and invalidation of
// the L2, after which the panels are read again), its flag and then the loads
// of the data: 27 us per column besides the SYMV at every order.
//
// Per column j, three exchanges, of which two are waited for:
//   A  w_r = tau (A v)_r of column j-1 and b_r, column j less the panel
//      columns before j-1, from the owner of each row r to everyone: every
//      workgroup forms a2, w' = w + a2 v, column j = b - v w'(j) - w' and its
//      reflector from them;
//   D  the owned rows' parts of W'^T v and V^T v, which travel while the SYMV
//      runs;
//   B  the SYMV's scatter parts, to the owners of their rows.
// A word is overwritten one column later at the earliest, by a workgroup that
// has read exchange A of that column from every owner; an owner publishes A
// only after it has read the B and D of the column before, and its B only
// after A, so one buffer of each kind suffices as long as every workgroup owns
// rows of the trailing matrix (the caller sees to it).
//
// Every sum has a fixed order; DET makes the SYMV's scatter one too.
//
// Measured, all panels of a reduction, barriers -> words: FP32 order 860 x 24
// problems 9.5 -> 6.1 ms, 1359 x 5 9.1 -> 6.4, 2664 x 8 61 -> 45, 4524 x 16 299
// -> 254; FP64 700 x 64 14.0 -> 11.5, 1359 x 5 8.2 -> 7.1, 2144 x 32 112 -> 103.
// Of a column of 2664 x 8 in FP32 the SYMV is 15-21 us, the rest 11.
//
// Included by eigen.hip only, inside its namespace.
#pragma once

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

constexpr int XP_DW = 4;  // waves that gather exchange D while the others publish B
constexpr int XP_WAIT = 14;   // pause before exchange A's first poll, in units of 64 clocks
constexpr int XP_C = 5;   // rows per thread in exchange A: orders up to XP_C x SY_THREADS

// x[0] + x[stride] + ... (count of them), eight loads at once: one by one each
// waits for its 130 cycles of LDS, and there are up to G of them on the
// column's path (1359 x 5 7.5 -> 6.9 ms of panels, 730 x 32 6.6 -> 6.0, FP64).
template <class T>
__device__ inline T xp_lds_sum(const T* x, int stride, int count)
{
    constexpr int N = 8;
    T s = 0;
    for (int t0 = 0; t0 < count; t0 += N) {
        T y[N];
#pragma unroll
        for (int t = 0; t < N; t++) y[t] = t0 + t < count ? x[(t0 + t) * stride] : T(0);
#pragma unroll
        for (int h = N / 2; h >= 1; h /= 2)
#pragma unroll
            for (int t = 0; t < h; t++) y[t] += y[t + h];
        s += y[0];
    }
    return s;
}

template <class T>
struct XPanelArgs {
    T *A, *W, *X, *d, *e, *tau;
    unsigned long long *xa, *xb, *xd;   // exchange words per problem: n rows x (w, b); G x n; G x 2 nb
    int* err;
    const T* fro;
    int n, k, kb, nb, G;
    unsigned epoch0;
};
// Words of one value.
template <class T>
constexpr int xp_words() { return (int)(sizeof(T) / 4); }

__device__ inline void xp_put(unsigned long long* q, float x, unsigned ep) { res_put(q, 0, x, ep); }
__device__ inline void xp_put(unsigned long long* q, double x, unsigned ep) { res_put(q, 0, x, ep); }
__device__ inline float xp_value(const unsigned long long (&x)[1]) { return __uint_as_float((unsigned)x[0]); }
__device__ inline double xp_value(const unsigned long long (&x)[2])
{
    return __longlong_as_double((long long)((x[1] << 32) | (x[0] & 0xffffffffull)));
}
// Loads the N W words of N packets src + t * stride (t in pend's bits) until
// all carry the epoch; a bounded poll.
template <int N, int W>
__device__ inline void xp_poll(const unsigned long long* src, size_t stride, unsigned pend, unsigned ep, int* err,
                               unsigned long long (&q)[N][W])
{
    for (long spins = 0; pend != 0; spins++) {
#pragma unroll
        for (int t = 0; t < N; t++)
            if (pend >> t & 1)
#pragma unroll
                for (int i = 0; i < W; i++)
                    q[t][i] = __hip_atomic_load(src + t * stride + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int t = 0; t < N; t++) {
            bool ok = (pend >> t & 1) != 0;
#pragma unroll
            for (int i = 0; i < W; i++) ok = ok && (unsigned)(q[t][i] >> 32) == ep;
            if (ok) pend &= ~(1u << t);
        }
        if ((spins & 63) == 63) {
            if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) break;
            if (spins > (1L << 21)) {   // seconds of polling: a lost workgroup
                atomicExch(err, 1);
                break;
            }
        }
    }
}
// Sum over t = part, part + P, ... < G (t != self) of the value at src + t stride.
template <class T>
__device__ inline T xp_sum(const unsigned long long* src, size_t stride, int part, int P, int G, int self, unsigned ep,
                           int* err)
{
    constexpr int N = 4, W = xp_words<T>();
    T acc = 0;
    for (int t0 = part; t0 < G; t0 += N * P) {
        unsigned pend = 0;
#pragma unroll
        for (int z = 0; z < N; z++)
            if (t0 + z * P < G && t0 + z * P != self) pend |= 1u << z;
        unsigned long long q[N][W] = {};
        xp_poll<N, W>(src + t0 * stride, P * stride, pend, ep, err, q);
#pragma unroll
        for (int z = 0; z < N; z++)
            if (pend >> z & 1) acc += xp_value(q[z]);
    }
    return acc;
}

// Dynamic LDS of the kernel (nsm: row slots of the largest workgroup).
template <class T>
constexpr size_t xp_lds(int n, int nsm, int nb, bool plds)
{
    const int ps = nsm > SY_THREADS ? nsm : SY_THREADS;
    return ((size_t)2 * n + nsm + (plds ? 2 * (size_t)nb * nsm : 0) + 2 * (size_t)nb * nb + 2 * nb + 2 * ps +
            2 * SY_WAVES + 4) * sizeof(T);
}

template <class T, bool PLDS, int KV, int UV, bool DET>
__global__ __launch_bounds__(SY_THREADS) void sytrd_xpanel_kernel(XPanelArgs<T> g)
{
    constexpr int NW = xp_words<T>();
    extern __shared__ char smem[];
    const int n = g.n, k = g.k, kb = g.kb, nb = g.nb, G = g.G;
    // (numbered XCD by XCD where G allows it, as in sytrd_panel_kernel)
    const int nwg = (int)gridDim.x;
    const int lin = (nwg % 8 == 0 && (nwg / 8) % G == 0) ? (int)(blockIdx.x & 7) * (nwg / 8) + (int)(blockIdx.x >> 3)
                                                      : (int)blockIdx.x;
    const int p = lin / G, gi = lin % G;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nunit = (n + SY_OB - 1) / SY_OB;
    const int nslots = owned_slots(nunit, gi, G);
    const int nsm = SY_OB * ((nunit + G - 1) / G);
    const int ps = nsm > SY_THREADS ? nsm : SY_THREADS;

    T* A = g.A + (size_t)p * n * n;
    T* Wg = g.W + (size_t)p * n * nb;
    T* X = g.X + (size_t)p * n * 3 * nb;
    unsigned long long* xa = g.xa + (size_t)p * n * 2 * NW;
    unsigned long long* xb = g.xb + (size_t)p * G * n * NW;
    unsigned long long* xd = g.xd + (size_t)p * G * 2 * nb * NW;
    int* err = g.err;

    T* u = reinterpret_cast<T*>(smem);              // n: scatter sums
    T* v = u + n;                                   // n
    T* y = v + n;                                   // nsm: dot parts of the owned rows
    T* Vp = y + nsm;                                // PLDS: V and W' of the owned rows, nb x nsm each
    T* Wp = Vp + (PLDS ? (size_t)nb * nsm : 0);
    T* Vt = Wp + (PLDS ? (size_t)nb * nsm : 0);     // rows k .. k+nb-1 of V and W': [row - k][column]
    T* Wt = Vt + (size_t)nb * nb;
    T* t12 = Wt + (size_t)nb * nb;                  // 2 nb: W'^T v, V^T v
    T* ps1 = t12 + 2 * nb;                          // ps
    T* ps2 = ps1 + ps;                              // ps
    T* redA = ps2 + ps;                             // SY_WAVES
    T* redB = redA + SY_WAVES;                      // SY_WAVES
    T* sc = redB + SY_WAVES;                        // [0] w(j) [1] x(j) [2] x(j+1)

    auto vpan = [&](int c, int q, int r) -> T {
        if constexpr (PLDS) return Vp[(size_t)c * nsm + q];
        else return A[r + (size_t)(k + c) * n];
    };
    auto wpan = [&](int c, int q, int r) -> T {
        if constexpr (PLDS) return Wp[(size_t)c * nsm + q];
        else return Wg[r + (size_t)c * n];
    };
    auto block_total = [&](T s, T* red) -> T {   // one barrier; red is reused a column later
        s = wave_total(s);
        if (lane == 0) red[wave] = s;
        lds_barrier();
        T t = 0;
#pragma unroll
        for (int w = 0; w < SY_WAVES; w++) t += red[w];
        return t;
    };

    T tau = 0;
    // exchange A of column k + i - 1 (i >= 1): its V and W' into the panel, and
    // column k + i into x (rows c = tid + t SY_THREADS)
    auto gather = [&](int i, T (&x)[XP_C]) {
        const int j = k + i;
        const unsigned ep = g.epoch0 + (unsigned)i;
        T w[XP_C], s1 = 0;   // x holds b until a2 is known
        __builtin_amdgcn_s_sleep(XP_WAIT);
        constexpr int N = 2;   // packets in flight per thread (registers)
#pragma unroll
        for (int t0 = 0; t0 < XP_C; t0 += N) {
            unsigned pend = 0;
#pragma unroll
            for (int t = 0; t < N; t++) {
                const int c = tid + (t0 + t) * SY_THREADS;
                if (t0 + t < XP_C && c >= j && c < n) pend |= 1u << t;
            }
            unsigned long long q[N][2 * NW] = {};
            xp_poll<N, 2 * NW>(xa + (size_t)(tid + t0 * SY_THREADS) * 2 * NW, (size_t)SY_THREADS * 2 * NW, pend, ep, err,
                               q);
#pragma unroll
            for (int t = 0; t < N; t++) {
                if (t0 + t >= XP_C) continue;
                const int c = tid + (t0 + t) * SY_THREADS;
                T wv = 0, bv = 0;
                if (pend >> t & 1) {
                    res_unpack(q[t], wv, bv);
                    if (c == j) sc[0] = wv;
                    s1 += wv * v[c];
                }
                w[t0 + t] = wv;
                x[t0 + t] = bv;
            }
        }
        s1 = block_total(s1, redA);
        const T a2 = T(-0.5) * tau * s1;
        const T wj = sc[0] + a2;
#pragma unroll
        for (int t = 0; t < XP_C; t++) {
            const int c = tid + t * SY_THREADS;
            if (c < j || c >= n) continue;
            const T vv = v[c], wp = w[t] + a2 * vv;
            x[t] = x[t] - vv * wj - wp;
            if (c < k + nb) {
                Vt[(c - k) * nb + i - 1] = vv;
                Wt[(c - k) * nb + i - 1] = wp;
            }
            // the owner's copies
            const int un = c / SY_OB, rd = un / G;
            if (owned_unit(rd, gi, G) == un) {
                const int q = SY_OB * rd + c % SY_OB;
                A[c + (size_t)(j - 1) * n] = vv;
                if constexpr (PLDS) {
                    Vp[(size_t)(i - 1) * nsm + q] = vv;
                    Wp[(size_t)(i - 1) * nsm + q] = wp;
                } else {
                    Wg[c + (size_t)(i - 1) * n] = wp;
                }
            }
        }
    };

    for (int i = 0; i < kb; i++) {
        const int j = k + i;
        const unsigned ep = g.epoch0 + (unsigned)i + 1;
        T x[XP_C];
        if (i > 0) {
            gather(i, x);
        } else {
#pragma unroll
            for (int t = 0; t < XP_C; t++) {
                const int c = tid + t * SY_THREADS;
                x[t] = c >= k && c < n ? A[c + (size_t)k * n] : T(0);   // column k arrives updated
            }
        }
        // reflector of column j
        T nrm = 0;
#pragma unroll
        for (int t = 0; t < XP_C; t++) {
            const int c = tid + t * SY_THREADS;
            if (c == j) sc[1] = x[t];
            if (c == j + 1) sc[2] = x[t];
            if (c > j + 1 && c < n) nrm += x[t] * x[t];
        }
        const T xn2 = block_total(nrm, redB);
        const T alpha = sc[2];
        T beta = alpha, scal = 0;
        tau = 0;
        if (xn2 != T(0)) {
            beta = -copysign(sqrt(alpha * alpha + xn2), alpha);
            tau = (beta - alpha) / beta;
            scal = T(1) / (alpha - beta);
        }
        T dsc = 0;
        if constexpr (DET) {
            // ||v||_2 with v(j+1) = 1 and the rest scal * x
            const T bound = g.fro[p] * sqrt(T(1) + scal * scal * xn2);
            dsc = bound > T(0) && bound < T(INFINITY) ? det_range<T>() / bound : T(1);
        }
        if (gi == 0 && tid == 0) {
            g.d[(size_t)p * n + j] = sc[1];
            g.e[(size_t)p * n + j] = beta;
            g.tau[(size_t)p * n + j] = tau;
        }
#pragma unroll
        for (int t = 0; t < XP_C; t++) {
            const int c = tid + t * SY_THREADS;
            if (c < n) {
                v[c] = c == j + 1 ? T(1) : (c > j + 1 ? scal * x[t] : T(0));
                u[c] = T(0);
            }
        }
        if constexpr (PLDS) lds_barrier();
        else __syncthreads();   // the panels' new column is read back from global memory
        const int qb = first_slot(j + 1, gi, G), nbq = nslots - qb;
        // exchange D: the panel dots over the owned rows, up to four per wave
        // (c < i with W'(:, c), else with V(:, c - i))
        for (int c0 = wave; c0 < 2 * i; c0 += 4 * SY_WAVES) {
            T f[4] = {T(0), T(0), T(0), T(0)};
            for (int q = qb + lane; q < nslots; q += 64) {
                const int r = owned_row(q, gi, G);
                if (r <= j || r >= n) continue;
                const T vv = v[r];
#pragma unroll
                for (int z = 0; z < 4; z++) {
                    const int c = c0 + z * SY_WAVES;
                    if (c < 2 * i) f[z] += (c < i ? wpan(c, q, r) : vpan(c - i, q, r)) * vv;
                }
            }
            const T s = wave_col_sums<4>(f, lane);
            const int c = c0 + (lane >> 4) * SY_WAVES;
            if ((lane & 15) == 0 && c < 2 * i) xp_put(xd + ((size_t)gi * 2 * nb + c) * NW, s, ep);
        }
        sytrd_symv_vec<T, KV, UV, DET>(A, n, j, gi, G, nslots, v, u, y, dsc);
        lds_barrier();
        // exchange B: the scatter sums to the rows' owners; W'^T v and V^T v
        // from everyone's parts.  Loads return in order after the same wave's
        // stores, so the first XP_DW waves read and the others store
        const int dw = i > 0 ? XP_DW : 0;
        if (wave >= dw) {
            for (int c = j + 1 + tid - 64 * dw; c < n; c += SY_THREADS - 64 * dw) {
                if constexpr (DET) u[c] = det_value(&u[c], dsc);
                const int un = c / SY_OB;
                if (owned_unit(un / G, gi, G) != un) xp_put(xb + ((size_t)gi * n + c) * NW, u[c], ep);
            }
        }
        if (i > 0) {
            const int nc = 2 * i, P = max(1, min(G, 64 * XP_DW / nc));
            if (wave < dw)
                for (int idx = tid; idx < nc * P; idx += 64 * dw)
                    ps1[idx] = xp_sum<T>(xd + (size_t)(idx % nc) * NW, (size_t)2 * nb * NW, idx / nc, P, G, -1, ep, err);
            lds_barrier();
            if (tid < nc) t12[tid] = xp_lds_sum(ps1 + tid, nc, P);
        }
        lds_barrier();
        // the owned rows' terms of y and of column j+1, each row's split over
        // P threads: the others' scatter sums, the panel terms
        const bool more = i + 1 < kb;
        if (nbq > 0) {
            const int P = max(1, min(max(G, i), SY_THREADS / nbq));
            for (int idx = tid; idx < nbq * P; idx += SY_THREADS) {
                const int q = qb + idx % nbq, part = idx / nbq;
                const int r = owned_row(q, gi, G);
                T ay = 0, ab = 0;
                if (r > j && r < n) {
                    for (int c = part; c < i; c += P) {
                        const T vv = vpan(c, q, r), ww = wpan(c, q, r);
                        ay -= vv * t12[c] + ww * t12[i + c];
                        if (more) ab -= vv * Wt[(i + 1) * nb + c] + ww * Vt[(i + 1) * nb + c];
                    }
                    if (part == 0) ab += more ? A[r + (size_t)(j + 1) * n] : T(0);
                    ay += xp_sum<T>(xb + (size_t)r * NW, (size_t)n * NW, part, P, G, gi, ep, err);
                }
                ps1[idx] = ay;
                ps2[idx] = ab;
            }
            lds_barrier();
            for (int q0 = tid; q0 < nbq; q0 += SY_THREADS) {
                const int q = qb + q0, r = owned_row(q, gi, G);
                if (r <= j || r >= n) continue;
                const T sy = y[q] + u[r] + xp_lds_sum(ps1 + q0, nbq, P), sb = xp_lds_sum(ps2 + q0, nbq, P);
                res_put(xa + (size_t)r * 2 * NW, 0, tau * sy, ep);
                res_put(xa + (size_t)r * 2 * NW, 1, sb, ep);
            }
        }
    }
    {
        T x[XP_C];
        gather(kb, x);
    }
    __syncthreads();
    // X = [V | W' | V] for the trailing rows owned here
    const int k1 = k + kb;
    for (int q = tid; q < nslots; q += SY_THREADS) {
        const int r = owned_row(q, gi, G);
        if (r < k1 || r >= n) continue;
        for (int c = 0; c < kb; c++) {
            const T vv = vpan(c, q, r), ww = wpan(c, q, r);
            X[r + (size_t)c * n] = vv;
            X[r + (size_t)(kb + c) * n] = ww;
            X[r + (size_t)(2 * kb + c) * n] = vv;
        }
    }
}
