// Tridiagonalisation of trailing problems that fit in the register files of
// the GPU: one persistent launch holds the whole matrix in registers, both
// triangles, and applies every rank-2 update at once (no panels, no trailing
// products).  Workgroup gi of a problem keeps the rows gi, gi + G, ...
//
// What bounds it is the latency of a column's chain (publish, read, reductions,
// update and product), so there is one exchange and one barrier per column,
// made of what the owners have before the reflector is known: for its own rows
// r a workgroup publishes S_r = (A xt)_r (xt: the column's tail) and a_r = A(r,
// j+1).  While these travel everyone forms the reflector v = scal xt + e(j+1)
// from its own copy of the column; then, from the words, w = tau A v = tau (scal
// S + a), w^T v, w' = w - tau/2 (w^T v) v and column j+1 of the updated matrix,
// and updates and multiplies its own rows.
//
// A word that is not there yet is zero, and a zero is published as -0: the
// words are stored and polled at agent scope and need no flag and no fence (a
// flag per column and the data behind it are two trips; words with an epoch
// beside 32 data bits are twice the traffic).  Four buffers: publishing epoch e,
// a wave also clears its words of epoch e - 2, which everyone had read before
// publishing e - 1, whose words this workgroup has read; the clearing store is
// complete (vmcnt) before the same wave publishes e + 1, and nobody polls for e
// + 2 in that buffer before it has read e + 1.  A workgroup whose rows are all
// done has nothing left to read and leaves.
//
// Two layouts of a workgroup's rows over its threads: up to order 512 each
// wave has whole rows (sytrd_resident_rows_kernel: a row's product is one wave's
// sum, reduced columns and rows are skipped, but every wave forms the whole
// column, which costs more than it saves from there on), above each thread has
// some columns of every row (sytrd_resident_kernel).
//
// Every sum is formed in a fixed order, so the result does not depend on
// timing (it serves the deterministic mode as it is).
//
// Measured, tridiagonalisation alone in FP64: panels and trailing updates -> one
// exchange per column with two barriers, reflector before publication -> here
//   order x problems   256 x 64     410 x 8       1024 x 8      1281 x 1      2048 x 1
//   ms                3.4 1.2 0.82  6.7 1.4 1.00  20.7 4.8 3.96 23.5 5.3 3.86 39.3 9.2 7.09
// 1.9 us per column at order 85, 2.4 at 410, 3.0 at 1281 (a word's way from one
// compute unit to another: 0.3 to 0.4 us).
//
// Included by eigen.hip only, inside its namespace.
#pragma once

constexpr int RES_THREADS = 512, RES_WAVES = RES_THREADS / 64;
constexpr int RES_CH = 16;    // own rows whose products are reduced together
constexpr int RES_WAIT = 2;   // pause before a column's first poll, in units of 64 clocks
constexpr int RES_RING = 4;   // buffers of the exchange
constexpr int RES_PG = 4;     // workgroups per problem / 64, at most
constexpr int RES_ROWS_MAX = 512;   // order up to which a wave has whole rows

template <class T>
struct ResArgs {
    T *A, *d, *e, *tau;
    T* ring;                  // per problem RES_RING x res_buf elements, zero on entry
    const unsigned* amax;     // per problem the largest entry (columns-per-thread layout)
    int* err;
    int n, j0, G;             // order (ld and stride of A, d, e, tau), first column, workgroups per problem
};

// Elements of one exchange buffer: (S, a) of every position (gi R + q for row q
// of workgroup gi; in FP64 every S, then every a), then every workgroup's share
// of xt^T A xt (to 16 bytes).
constexpr int res_buf(int G, int R) { return 2 * G * R + (G + 3) / 4 * 4; }

typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

// Agent-scope words of a buffer (byte offsets): a pair (S, a) and one value.
// A value's word or half of a pair is never +0 once published.
//
// A value counts as there when any of its bits is set, so it must become visible
// whole: each travels in an aligned access of its own size, 4 or 8 bytes, which
// is single-copy atomic (the same load and store with the same cache policy that a
// relaxed agent-scope atomic of that size compiles to).  A 16-byte access is not
// promised to be: the pair of FP64 is two accesses, S at o and a at o + plane
// (apart, so that the compiler cannot merge them): as one, 1281 x 1 took
// 3.78 ms for 3.86, 2048 x 1 6.81 for 7.09, 1024 x 8 4.07 for 3.96.  Of the 8-byte
// pair of FP32 each half is tested by itself.
template <class T>
struct ResRing;
template <>
struct ResRing<double> {
    static constexpr int SC1 = 16;   // cache policy: agent scope
    typedef u32x2 word;
    struct pair {
        word s, a;
    };
    static __device__ inline word get1(__amdgpu_buffer_rsrc_t r, int o) { return __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, SC1); }
    static __device__ inline void put1(__amdgpu_buffer_rsrc_t r, int o, word p) { __builtin_amdgcn_raw_buffer_store_b64(p, r, o, 0, SC1); }
    static __device__ inline pair get2(__amdgpu_buffer_rsrc_t r, int o, int plane) { return pair{get1(r, o), get1(r, o + plane)}; }
    static __device__ inline void put2(__amdgpu_buffer_rsrc_t r, int o, int plane, pair p)
    {
        put1(r, o, p.s);
        put1(r, o + plane, p.a);
    }
    static __device__ inline bool there(word p) { return (p.x | p.y) != 0; }
    static __device__ inline bool there(pair p) { return there(p.s) && there(p.a); }
    static __device__ inline double val(word p)
    {
        return __longlong_as_double((long long)(((unsigned long long)p.y << 32) | p.x));
    }
    static __device__ inline double first(pair p) { return val(p.s); }
    static __device__ inline double second(pair p) { return val(p.a); }
    static __device__ inline word bits(double x)
    {
        const unsigned long long b = (unsigned long long)__double_as_longlong(x);
        const unsigned lo = (unsigned)b, hi = (unsigned)(b >> 32);
        return word{lo, (lo | hi) == 0 ? 0x80000000u : hi};
    }
    static __device__ inline pair bits(double x, double y) { return pair{bits(x), bits(y)}; }
    static __device__ inline pair clear() { return pair{word(0), word(0)}; }
};
template <>
struct ResRing<float> {
    static constexpr int SC1 = 16;
    typedef unsigned word;
    typedef u32x2 pair;
    static __device__ inline word get1(__amdgpu_buffer_rsrc_t r, int o) { return __builtin_amdgcn_raw_buffer_load_b32(r, o, 0, SC1); }
    static __device__ inline void put1(__amdgpu_buffer_rsrc_t r, int o, word p) { __builtin_amdgcn_raw_buffer_store_b32(p, r, o, 0, SC1); }
    static __device__ inline pair get2(__amdgpu_buffer_rsrc_t r, int o, int) { return __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, SC1); }
    static __device__ inline void put2(__amdgpu_buffer_rsrc_t r, int o, int, pair p) { __builtin_amdgcn_raw_buffer_store_b64(p, r, o, 0, SC1); }
    static __device__ inline bool there(word p) { return p != 0; }
    static __device__ inline bool there(pair p) { return p.x != 0 && p.y != 0; }
    static __device__ inline float val(word p) { return __uint_as_float(p); }
    static __device__ inline float first(pair p) { return __uint_as_float(p.x); }
    static __device__ inline float second(pair p) { return __uint_as_float(p.y); }
    static __device__ inline word bits(float x)
    {
        const unsigned b = __float_as_uint(x);
        return b == 0 ? 0x80000000u : b;
    }
    static __device__ inline pair bits(float x, float y) { return pair{bits(x), bits(y)}; }
    static __device__ inline pair clear() { return pair(0); }
};

// 1 / x to rounding level: the hardware's estimate and two Newton steps (the
// IEEE division's scaling and fix-up are as long again, on the critical path).
__device__ inline double res_rcp(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}
__device__ inline float res_rcp(float x) { return 1.0f / x; }

// x 2^e, and the exponent of a number from its upper 32 bits without the sign
// (0 for an infinite or NaN one).
__device__ inline double res_scale(double x, int e) { return __builtin_amdgcn_ldexp(x, e); }
__device__ inline float res_scale(float x, int e) { return __builtin_amdgcn_ldexpf(x, e); }
__device__ inline unsigned res_top(double x) { return (unsigned)((unsigned long long)__double_as_longlong(x) >> 32) & 0x7fffffffu; }
__device__ inline unsigned res_top(float x) { return __float_as_uint(x) & 0x7fffffffu; }
template <class T>
__device__ inline int res_exp(unsigned top)
{
    constexpr int MB = sizeof(T) == 8 ? 20 : 23, EMAX = sizeof(T) == 8 ? 0x7ff : 0xff;
    const int e = (int)(top >> MB);
    return e == EMAX ? 0 : e - EMAX / 2;
}

// Zeroes a problem's exchange buffers (words of 32 bits) and finds the largest
// entry of its trailing matrix (lower triangle; amax zero on entry): 12 us at
// 2048 x 1 and 20 at 1024 x 8 in FP64, beside 6.8 and 4.1 ms.
template <class T>
__global__ __launch_bounds__(256) void res_prepare_kernel(ResArgs<T> g, int words, unsigned* amax)
{
    __shared__ unsigned red[4];
    const int n = g.n, m = g.n - g.j0, p = blockIdx.y;
    unsigned* ring = reinterpret_cast<unsigned*>(g.ring) + (size_t)p * words;
    for (int i = blockIdx.x * 256 + threadIdx.x; i < words; i += gridDim.x * 256) ring[i] = 0u;
    const T* A = g.A + (size_t)p * n * n + g.j0 + (size_t)g.j0 * n;
    unsigned top = 0;
    for (int c = blockIdx.x; c < m; c += gridDim.x)
        for (int r = c + threadIdx.x; r < m; r += 256) top = max(top, res_top(A[r + (size_t)c * n]));
    for (int o = 32; o > 0; o >>= 1) top = max(top, (unsigned)__shfl_xor((int)top, o, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = top;
    __syncthreads();
    if (threadIdx.x == 0) atomicMax(&amax[p], max(max(red[0], red[1]), max(red[2], red[3])));
}

// The sum of the waves' values x[0], x[stride], ...: all loads at once, as a
// tree (a loop over the waves there are waits for each load: 700 cycles of 8).
template <class T>
__device__ inline T res_wave_sum(const T* x, int stride)
{
    T s[RES_WAVES];
#pragma unroll
    for (int w = 0; w < RES_WAVES; w++) s[w] = x[w * stride];
#pragma unroll
    for (int h = RES_WAVES / 2; h >= 1; h /= 2)
#pragma unroll
        for (int w = 0; w < h; w++) s[w] += s[w + h];
    return s[0];
}
// The sum over each group of R neighbouring lanes.
template <int R, class T>
__device__ inline T res_group_total(T v)
{
    v += dpp_mov<DPP_XOR1>(v);
    v += dpp_mov<DPP_XOR2>(v);
    v += dpp_mov<DPP_HALF_MIRROR>(v);
    if constexpr (R >= 16) v += dpp_mov<DPP_MIRROR>(v);
    if constexpr (R >= 32) v = swap_add<16>(v, v);
    if constexpr (R >= 64) v = swap_add<32>(v, v);
    return v;
}

// A bounded poll's end: every 64th pass, whether some workgroup has given up,
// and after 2^21 passes (seconds: a lost workgroup) giving up.
__device__ inline bool res_give_up(long spins, int* err, int lane)
{
    if ((spins & 63) != 63) return false;
    if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return true;
    if (spins <= (1L << 21)) return false;
    if (lane == 0) atomicExch(err, 1);
    return true;
}

// Thread t keeps the columns at the positions t, t + blockDim, ... (at most C)
// of R rows: what a wave reads of the exchange is contiguous.  The sum of xt^T A
// xt travels as a share per workgroup: a sum over the column's waves would be a
// second barrier.  It has three factors of the matrix's size, which leave the
// range long before the two of every other sum here do (FP32: entries of 1e13), so
// the matrix is reduced as A 2^-ex, ex the exponent of its largest entry, found
// beforehand (an exchange for it in here cost every column 2-3 % through the
// registers it takes).
// Dynamic LDS for a trailing order m (everything twice: a
// column's writes need no barrier behind the last column's reads).
template <class T>
constexpr size_t res_lds(int m, int R)
{
    return 2 * ((size_t)m + RES_WAVES + 4 + R + (size_t)RES_WAVES * R) * sizeof(T);
}

template <class T, int R, int C>
__global__ __launch_bounds__(RES_THREADS) void sytrd_resident_kernel(ResArgs<T> g)
{
    typedef ResRing<T> Ring;
    constexpr int CH = R < RES_CH ? R : RES_CH, NCH = R / CH, ES = (int)sizeof(T);
    extern __shared__ char smem[];
    const int n = g.n, m = g.n - g.j0, G = g.G;
    // (a problem's workgroups on one XCD where G allows it, as in the panel kernel)
    const int nwg = (int)gridDim.x;
    const int lin = (nwg % 8 == 0 && (nwg / 8) % G == 0) ? (int)(blockIdx.x & 7) * (nwg / 8) + (int)(blockIdx.x >> 3)
                                                      : (int)blockIdx.x;
    const int p = lin / G, gi = lin % G;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, NT = blockDim.x;
    T* A = g.A + (size_t)p * n * n + g.j0 + (size_t)g.j0 * n;   // the trailing matrix, ld n
    const int bufb = res_buf(G, R) * ES, plane = 8 * G * R, share = 2 * G * R * ES;
    const __amdgpu_buffer_rsrc_t ring = __builtin_amdgcn_make_buffer_rsrc(
        g.ring + (size_t)p * RES_RING * res_buf(G, R), 0, RES_RING * bufb, 0x20000);   // (32-bit elements, no stride)
    T* dd = g.d + (size_t)p * n + g.j0;
    T* ee = g.e + (size_t)p * n + g.j0;
    T* tt = g.tau + (size_t)p * n + g.j0;
    T* lx0 = reinterpret_cast<T*>(smem);        // 2 x m: column j
    T* redB0 = lx0 + 2 * m;                     // 2 x RES_WAVES
    T* sc0 = redB0 + 2 * RES_WAVES;             // 2 x 4: [0] x(j) [1] x(j+1)
    T* acol0 = sc0 + 8;                         // 2 x R: own rows' entries of column j+1
    T* part0 = acol0 + 2 * R;                   // 2 x RES_WAVES x R: the waves' parts of own rows' products

    // (the sums over waves run over RES_WAVES of them)
    for (int i = tid; i < 2 * RES_WAVES; i += NT) redB0[i] = T(0);
    for (int i = tid; i < 2 * RES_WAVES * R; i += NT) part0[i] = T(0);
    lds_barrier();

    const int ex = res_exp<T>(g.amax[p]);
    T a[R][C], v[C], x[C], vown[NCH], wown[NCH];
    int col[C];   // (m: none)
#pragma unroll
    for (int k = 0; k < C; k++) {
        const int pos = tid + k * NT, c = (pos % R) * G + pos / R;
        col[k] = pos < G * R && c < m ? c : m;
    }
#pragma unroll
    for (int q = 0; q < R; q++) {
        const int r = q * G + gi;
#pragma unroll
        for (int k = 0; k < C; k++) {
            const int c = col[k];
            a[q][k] = r < m && c < m ? res_scale(c >= r ? A[c + (size_t)r * n] : A[r + (size_t)c * n], -ex) : T(0);
        }
    }
    // column 0 arrives final
#pragma unroll
    for (int k = 0; k < C; k++) {
        v[k] = T(0);
        x[k] = col[k] < m ? res_scale(A[col[k]], -ex) : T(0);
    }
#pragma unroll
    for (int h = 0; h < NCH; h++) vown[h] = wown[h] = T(0);
    const int rlast = gi < m ? (m - 1 - gi) / G * G + gi : -1;   // last own row
    T tau = 0, scal = 0, beta = 0;
    // column j's reflector into A, d, e and tau, by the owner of row j + 1, a
    // step later: the stores' way to memory is then beside the arithmetic, and
    // column 0 is overwritten only when every workgroup has loaded its rows
    auto store_reflector = [&](int j) {
        if ((j + 1) % G != gi) return;
        const T* lx = lx0 + (j & 1) * m;
        if (tid == 0) {
            dd[j] = res_scale(sc0[4 * (j & 1)], ex);
            ee[j] = res_scale(beta, ex);
            tt[j] = tau;
        }
        for (int c = tid; c < m; c += NT)
            if (c > j) A[c + (size_t)j * n] = c == j + 1 ? T(1) : scal * lx[c];
    };
    int j = 0, jg = 0, jq = 0;   // j = jq G + jg
    for (; j < m - 1 && rlast > j; j++) {
        T* lx = lx0 + (j & 1) * m;
        T* redB = redB0 + (j & 1) * RES_WAVES;
        T* sc = sc0 + 4 * (j & 1);
        T* acol = acol0 + (j & 1) * R;
        T* part = part0 + (j & 1) * RES_WAVES * R;
        T wp[C], a2 = 0;
#pragma unroll
        for (int k = 0; k < C; k++) wp[k] = T(0);
        if (j > 0) {
            // S and a of the rows from j on, row j's own, and the shares
            __builtin_amdgcn_s_sleep(RES_WAIT);
            const int base = (j & (RES_RING - 1)) * bufb;
            // (each load under its own condition, so they go out one after the
            // other; all at once is slower, 1281 x 1 3.8 -> 4.4 ms: at these
            // orders everyone's reading is what the words wait for, and the
            // pass then starts before they can have arrived)
            typename Ring::pair pk[C], pj = Ring::bits(T(0), T(0));
            typename Ring::word ps[RES_PG];
            bool need[C], needj = true, needs[RES_PG];
            const int oj = base + 8 * (jg * R + jq);
#pragma unroll
            for (int k = 0; k < C; k++) {
                pk[k] = Ring::bits(T(0), T(0));
                need[k] = col[k] >= j && col[k] < m;
            }
#pragma unroll
            for (int i = 0; i < RES_PG; i++) {
                const int gq = lane + 64 * i;
                ps[i] = Ring::bits(T(0));
                needs[i] = gq < G && (m - 1 - gq) / G * G + gq >= j;
            }
            for (long spins = 0;; spins++) {
                asm volatile("" ::: "memory");   // (every pass loads anew)
#pragma unroll
                for (int k = 0; k < C; k++)
                    if (need[k]) pk[k] = Ring::get2(ring, base + 8 * (tid + k * NT), plane);
                if (needj) pj = Ring::get2(ring, oj, plane);
#pragma unroll
                for (int i = 0; i < RES_PG; i++)
                    if (needs[i]) ps[i] = Ring::get1(ring, base + share + ES * (lane + 64 * i));
                bool more = false;
#pragma unroll
                for (int k = 0; k < C; k++) {
                    need[k] = need[k] && !Ring::there(pk[k]);
                    more = more || need[k];
                }
                needj = needj && !Ring::there(pj);
                more = more || needj;
#pragma unroll
                for (int i = 0; i < RES_PG; i++) {
                    needs[i] = needs[i] && !Ring::there(ps[i]);
                    more = more || needs[i];
                }
                if (__builtin_amdgcn_ballot_w64(more) == 0 || res_give_up(spins, g.err, lane)) break;
            }
            store_reflector(j - 1);
            // xt^T A xt, then w^T v = tau (scal^2 xt^T A xt + 2 scal S(j) + a(j)):
            // xt^T a = S(j) by symmetry
            T q = Ring::val(ps[0]);
#pragma unroll
            for (int i = 1; i < RES_PG; i++) q += Ring::val(ps[i]);
            q = wave_total(q);
            const T Sj = Ring::first(pj), aj = Ring::second(pj);
            a2 = T(-0.5) * tau * tau * (scal * (scal * q + T(2) * Sj) + aj);
            // w' = w + a2 v, column j less v w'(j) + w' v(j), v(j) = 1
            const T wj = tau * (scal * Sj + aj) + a2;
#pragma unroll
            for (int k = 0; k < C; k++) {
                const bool in = col[k] >= j && col[k] < m;
                const T ak = in ? Ring::second(pk[k]) : T(0);
                if (!in) v[k] = T(0);
                wp[k] = in ? tau * (scal * Ring::first(pk[k]) + ak) + a2 * v[k] : T(0);
                x[k] = ak - v[k] * wj - wp[k];
            }
        }
        // the column: its head, and the tail's entries xt with their norm
        T nrm = 0, xt[C];
#pragma unroll
        for (int k = 0; k < C; k++) {
            const int c = col[k];
            xt[k] = c > j + 1 && c < m ? x[k] : T(0);
            nrm += xt[k] * xt[k];
            if (c == j) sc[0] = x[k];
            if (c == j + 1 && c < m) sc[1] = x[k];
            if (c < m) lx[c] = x[k];
        }
        // own rows: the last column's rank-2 update and the product with the
        // tail, RES_CH rows at a time; finished rows are skipped by fours
#pragma unroll
        for (int h = 0; h < NCH; h++) {
            const int q0 = h * CH;
            // row q0 + l in lane l (< CH)
            const T vr_l = vown[h], wr_l = wown[h] + a2 * vr_l;
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
                if (col[k] == j + 1) {
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
        if (wave == 0 && j < m - 2) {
            // publish; the words of two columns ago become free
            const int base = ((j + 1) & (RES_RING - 1)) * bufb, old = ((j + 3) & (RES_RING - 1)) * bufb;
            const int q = lane % R, r = q * G + gi, o = 8 * (gi * R + q);
            const T s = res_wave_sum(part + q, R);
            const bool in = r > j && r < m, on = lane < R && in;
            __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): the last column's clearing stores are complete
            if (on) Ring::put2(ring, base + o, plane, Ring::bits(s, acol[q]));
            const T t = res_group_total<R>(in && r > j + 1 ? s * lx[r] : T(0));
            if (lane == 0) Ring::put1(ring, base + share + ES * gi, Ring::bits(t));
            if (on) Ring::put2(ring, old + o, plane, Ring::clear());
            if (lane == 0) Ring::put1(ring, old + share + ES * gi, typename Ring::word(0));
        }
        // the reflector
        const T xn2 = res_wave_sum(redB, 1);
        const T alpha = sc[1];
        beta = alpha;
        scal = tau = 0;
        if (xn2 != T(0)) {
            // |beta| = sqrt(s) = s rsqrt(s), tau = (beta - alpha) / beta, scal = 1 / (alpha - beta)
            const T s = alpha * alpha + xn2, rs = rsqrt(s);
            T b = s * rs;
            b += T(0.5) * rs * fma(-b, b, s);
            beta = -copysign(b, alpha);
            tau = T(1) + fabs(alpha) * rs;
            scal = res_rcp(alpha - beta);
        }
        if (j == m - 2 && tid == 0)   // the last diagonal element (sytrd_finish_kernel moves it to d)
            A[(size_t)(m - 1) * n + m - 1] = res_scale(acol[(m - 1) / G], ex);
#pragma unroll
        for (int k = 0; k < C; k++) v[k] = col[k] == j + 1 ? T(1) : scal * xt[k];
#pragma unroll
        for (int h = 0; h < NCH; h++) {
            const int q = h * CH + (lane & (CH - 1)), r = q * G + gi;
            const T s = res_wave_sum(part + q, R);
            vown[h] = r == j + 1 ? T(1) : (r > j + 1 && r < m ? scal * lx[r] : T(0));
            wown[h] = tau * (scal * s + acol[q]);
        }
        if (++jg == G) {
            jg = 0;
            jq++;
        }
    }
    if (j > 0) store_reflector(j - 1);
}

// The sums over the wave of RW values per lane: the lane gets that of row lane
// >> (6 - log2 RW).
template <int RW, class T>
__device__ inline T res_row_sums(T (&s)[RW], int lane)
{
    if constexpr (RW == 2) {
        T t = swap_add<32>(s[0], s[1]);
        t = swap_add<16>(t, t);
        t += dpp_mov<DPP_MIRROR>(t);
        t += dpp_mov<DPP_HALF_MIRROR>(t);
        t += dpp_mov<DPP_XOR2>(t);
        return t + dpp_mov<DPP_XOR1>(t);
    } else {
        return wave_col_sums<RW>(s, lane);
    }
}

// Wave w keeps the rows q G + gi, q = i NW + w (RW of them), all their columns:
// lane l the columns l + 64 k, k < K.  The words are read once per workgroup and
// w and a go to LDS, for every wave to form the column.
// Dynamic LDS: w and a, twice (a column's writes need no barrier
// behind the last column's reads).
template <class T>
constexpr size_t res_rows_lds(int K) { return 4 * (size_t)K * 64 * sizeof(T); }

template <class T, int NW, int RW, int K>
__global__ __launch_bounds__(64 * NW) void sytrd_resident_rows_kernel(ResArgs<T> g)
{
    typedef ResRing<T> Ring;
    constexpr int R = NW * RW, NT = 64 * NW, CP = (K + NW - 1) / NW, SH = 6 - ilog2<RW>(), ES = (int)sizeof(T), M = 64 * K;
    constexpr int GS = 2;   // chunks taken together
    extern __shared__ char smem[];
    const int n = g.n, m = g.n - g.j0, G = g.G;
    // (a problem's workgroups on one XCD where G allows it, as in the panel kernel)
    const int nwg = (int)gridDim.x;
    const int lin = (nwg % 8 == 0 && (nwg / 8) % G == 0) ? (int)(blockIdx.x & 7) * (nwg / 8) + (int)(blockIdx.x >> 3)
                                                      : (int)blockIdx.x;
    const int p = lin / G, gi = lin % G;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    T* A = g.A + (size_t)p * n * n + g.j0 + (size_t)g.j0 * n;   // the trailing matrix, ld n
    const int bufb = res_buf(G, R) * ES, plane = 8 * G * R;
    const __amdgpu_buffer_rsrc_t ring = __builtin_amdgcn_make_buffer_rsrc(
        g.ring + (size_t)p * RES_RING * res_buf(G, R), 0, RES_RING * bufb, 0x20000);   // (32-bit elements, no stride)
    T* dd = g.d + (size_t)p * n + g.j0;
    T* ee = g.e + (size_t)p * n + g.j0;
    T* tt = g.tau + (size_t)p * n + g.j0;
    T* lds = reinterpret_cast<T*>(smem);   // 2 x (M of w, M of a), zero where nothing was written

    for (int i = tid; i < 4 * M; i += NT) lds[i] = T(0);
    // positions of the exchange read by this thread, and their columns (m: none)
    int col[CP];
#pragma unroll
    for (int i = 0; i < CP; i++) {
        const int pos = tid + i * NT, s = pos % R, c = ((s % RW) * NW + s / RW) * G + pos / R;
        col[i] = pos < G * R && c < m ? c : m;
    }
    // the row this lane publishes, one of the wave's
    const int il = lane >> SH, rl = (il * NW + wave) * G + gi;
    const int opub = 8 * (gi * R + wave * RW + il);
    T a[RW][K], v[K];
#pragma unroll
    for (int i = 0; i < RW; i++) {
        const int r = (i * NW + wave) * G + gi;
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int c = lane + 64 * k;
            a[i][k] = r < m && c < m ? (c >= r ? A[c + (size_t)r * n] : A[r + (size_t)c * n]) : T(0);
        }
    }
    // column 0 arrives final: into LDS as a (w = 0, v = 0)
#pragma unroll
    for (int k = 0; k < K; k++) v[k] = T(0);
    lds_barrier();
    for (int c = tid; c < m; c += NT) lds[M + c] = A[c];
    lds_barrier();
    T vr_l = 0;   // v of row rl
    const int rlast = gi < m ? (m - 1 - gi) / G * G + gi : -1, khi = (m - 1) >> 6;
    T tau = 0, scal = 0, beta = 0, dj = 0;
    // column j's reflector into A, d, e and tau, by the owner of row j + 1, a
    // step later: the stores' way to memory is then beside the arithmetic, and
    // column 0 is overwritten only when every workgroup has loaded its rows
    auto store_reflector = [&](int j) {
        if ((j + 1) % G != gi) return;
        if (tid == 0) {
            dd[j] = dj;
            ee[j] = beta;
            tt[j] = tau;
        }
#pragma unroll
        for (int k = 0; k < K; k++) {
            const int c = lane + 64 * k;
            if (k % NW == wave && c > j && c < m) A[c + (size_t)j * n] = v[k];
        }
    };
    int j = 0;
    for (; j < m - 1 && rlast > j; j++) {
        T* lw = lds + (j & 1) * 2 * M;
        T* la = lw + M;
        const int kj = j >> 6, k1 = (j + 1) >> 6, l1 = (j + 1) & 63;
        if (j > 0) {
            // S and a of the rows from j on (a word that is not wanted is one past
            // the buffers: no access).  All loads of a pass are issued before
            // the first is waited for
            __builtin_amdgcn_s_sleep(RES_WAIT);
            const int base = (j & (RES_RING - 1)) * bufb, none = RES_RING * bufb;
            typename Ring::pair pk[CP];
            int ok[CP];
#pragma unroll
            for (int i = 0; i < CP; i++) ok[i] = col[i] >= j && col[i] < m ? base + 8 * (tid + i * NT) : none;
            for (long spins = 0;; spins++) {
                asm volatile("" ::: "memory");   // (every pass loads anew)
#pragma unroll
                for (int i = 0; i < CP; i++) pk[i] = Ring::get2(ring, ok[i], plane);
                bool more = false;
#pragma unroll
                for (int i = 0; i < CP; i++) more = more || (ok[i] != none && !Ring::there(pk[i]));
                if (__builtin_amdgcn_ballot_w64(more) == 0) break;
                if (res_give_up(spins, g.err, lane)) break;
            }
            // (finished columns: zeros)
#pragma unroll
            for (int i = 0; i < CP; i++)
                if (col[i] < m) {
                    const bool in = col[i] >= j;
                    const T ak = Ring::second(pk[i]), wk = tau * (scal * Ring::first(pk[i]) + ak);
                    lw[col[i]] = in ? wk : T(0);
                    la[col[i]] = in ? ak : T(0);
                }
            lds_barrier();
            store_reflector(j - 1);
        }
        // all reads of w and a are issued before the first is used (chunk by
        // chunk, a read's 130 cycles came twice for each)
        const T wj = lw[j];
        const T wl = rl < m ? lw[rl] : T(0), al = rl < m ? la[rl] : T(0);
        T wv[K], av[K], q = 0;
#pragma unroll
        for (int h = 0; h < K; h += GS)
            if (h + GS > kj && h <= khi) {
#pragma unroll
                for (int k = h; k < h + GS; k++) wv[k] = lw[lane + 64 * k];
            }
#pragma unroll
        for (int h = 0; h < K; h += GS)
            if (h + GS > kj && h <= khi) {
#pragma unroll
                for (int k = h; k < h + GS; k++) av[k] = la[lane + 64 * k];
            }
        // w^T v, a2 = -tau/2 w^T v
#pragma unroll
        for (int h = 0; h < K; h += GS)
            if (h + GS > kj && h <= khi) {
                T t = 0;
#pragma unroll
                for (int k = h; k < h + GS; k++) t += wv[k] * v[k];
                q += t;
            }
        q = wave_total(q);
        const T a2 = T(-0.5) * tau * q, a22 = a2 + a2;
        // the own rows' entries of the column, and the update's factors: a -=
        // v_r w' + w'_r v = v_r (w + 2 a2 v) + w_r v
        const T xr_l = al - (wl + a22 * vr_l) - vr_l * wj;
        T vr[RW], wr[RW];
#pragma unroll
        for (int i = 0; i < RW; i++) {
            vr[i] = read_lane(vr_l, i << SH);
            wr[i] = read_lane(wl, i << SH);
        }
        T nrm = 0, acc[RW], ac[RW], alpha = 0;
#pragma unroll
        for (int i = 0; i < RW; i++) acc[i] = ac[i] = T(0);
#pragma unroll
        for (int h = 0; h < K; h += GS) {
            if (h + GS <= kj || h > khi) continue;
            T wp[GS], x[GS];
#pragma unroll
            for (int k = 0; k < GS; k++) {
                // column j of the updated matrix (v(j) = 1)
                wp[k] = wv[h + k] + a22 * v[h + k];
                x[k] = av[h + k] - wp[k] - v[h + k] * wj;
            }
            // its head; xt is what is left
            if (kj >= h && kj < h + GS) {
#pragma unroll
                for (int k = 0; k < GS; k++) {
                    if (h + k != kj) continue;
                    dj = read_lane(x[k], j & 63);
                    x[k] = lane == (j & 63) ? T(0) : x[k];
                }
            }
            if (k1 >= h && k1 < h + GS) {
#pragma unroll
                for (int k = 0; k < GS; k++) {
                    if (h + k != k1) continue;
                    alpha = read_lane(x[k], l1);
                    x[k] = lane == l1 ? T(0) : x[k];
                }
            }
#pragma unroll
            for (int i = 0; i < RW; i++) {
                if ((i * NW + wave) * G + gi <= j) continue;
#pragma unroll
                for (int k = 0; k < GS; k++) a[i][h + k] -= vr[i] * wp[k] + wr[i] * v[h + k];
#pragma unroll
                for (int k = 0; k < GS; k++) acc[i] += a[i][h + k] * x[k];
            }
            if (k1 >= h && k1 < h + GS) {
#pragma unroll
                for (int k = 0; k < GS; k++) {
                    if (h + k != k1) continue;
#pragma unroll
                    for (int i = 0; i < RW; i++) ac[i] = a[i][h + k];
                }
            }
#pragma unroll
            for (int k = 0; k < GS; k++) {
                v[h + k] = x[k];
                nrm += x[k] * x[k];
            }
        }
        // a(r, j+1) of the row this lane publishes: lane l1 has them all
        T acl = 0;
#pragma unroll
        for (int i = 0; i < RW; i++) {
            const T t = read_lane(ac[i], l1);
            acl = il == i ? t : acl;
        }
        // publish; the words of two columns ago become free
        const T s = res_row_sums<RW>(acc, lane);
        if (j < m - 2) {
            const int base = ((j + 1) & (RES_RING - 1)) * bufb, old = ((j + 3) & (RES_RING - 1)) * bufb;
            const bool on = (lane & ((1 << SH) - 1)) == 0 && rl > j && rl < m;
            __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): the last column's clearing stores are complete
            if (on) Ring::put2(ring, base + opub, plane, Ring::bits(s, acl));
            if (on) Ring::put2(ring, old + opub, plane, Ring::clear());
        } else if (rl == m - 1 && (lane & ((1 << SH) - 1)) == 0) {
            A[(size_t)(m - 1) * n + m - 1] = acl;   // the last diagonal element (sytrd_finish_kernel moves it to d)
        }
        // the reflector
        nrm = wave_total(nrm);
        beta = alpha;
        scal = tau = 0;
        if (nrm != T(0)) {
            // |beta| = sqrt(s2) = s2 rsqrt(s2), tau = (beta - alpha) / beta, scal = 1 / (alpha - beta)
            const T s2 = alpha * alpha + nrm, rs = rsqrt(s2);
            T b = s2 * rs;
            b += T(0.5) * rs * fma(-b, b, s2);
            beta = -copysign(b, alpha);
            tau = T(1) + fabs(alpha) * rs;
            scal = res_rcp(alpha - beta);
        }
#pragma unroll
        for (int h = 0; h < K; h += GS) {
            if (h + GS <= kj || h > khi) continue;
#pragma unroll
            for (int k = h; k < h + GS; k++) v[k] = lane + 64 * k == j + 1 ? T(1) : scal * v[k];
        }
        vr_l = rl == j + 1 ? T(1) : (rl > j + 1 && rl < m ? scal * xr_l : T(0));
    }
    if (j > 0) store_reflector(j - 1);
}

// Shape of a resident launch for B problems of trailing order m on ncu compute
// units: R rows and G workgroups per problem, NT threads; C columns per thread,
// or, where waves have whole rows, K chunks of 64 columns.  All B G workgroups
// must be resident at once, one per compute unit, and the matrix elements of a
// thread (R C, or R K 64 / NT) leave it registers to work with (at most 64: 256
// registers at FP64, nothing spilled).  The fewest rows that fit are the fastest
// (1024 x 1: R = 8 / 16 / 32 took 4.2 / 4.6 / 5.6 ms), and four waves with whole
// rows where the registers allow it: eight form the column twice as often.
struct ResShape {
    int R = 0, C = 0, K = 0, G = 0, NT = 0;
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
        s.G = G;
        if (m <= RES_ROWS_MAX) {
            s.K = m <= 256 ? 4 : 8;
            s.NT = R * s.K > 256 ? 512 : 256;
        } else {
            s.C = C;
            s.NT = ((G * R + C - 1) / C + 63) / 64 * 64;   // (G R <= 512 C: R divides 512)
        }
        return s;
    }
    return s;
}
// Largest trailing order the resident kernels take (0: none).
inline int res_max(int B, int ncu)
{
    int m = 4 * RES_THREADS;
    while (m >= 2 && res_shape(m, B, ncu).R == 0) m--;
    return m >= 2 ? m : 0;
}
template <class T>
const void* res_kernel(const ResShape& s)
{
    if (s.K > 0) {
        switch (s.K * 100 + s.R) {
            case 408: return (const void*)sytrd_resident_rows_kernel<T, 4, 2, 4>;
            case 416: return (const void*)sytrd_resident_rows_kernel<T, 4, 4, 4>;
            case 432: return (const void*)sytrd_resident_rows_kernel<T, 4, 8, 4>;
            case 464: return (const void*)sytrd_resident_rows_kernel<T, 4, 16, 4>;
            case 808: return (const void*)sytrd_resident_rows_kernel<T, 4, 2, 8>;
            case 816: return (const void*)sytrd_resident_rows_kernel<T, 4, 4, 8>;
            case 832: return (const void*)sytrd_resident_rows_kernel<T, 4, 8, 8>;
            case 864: return (const void*)sytrd_resident_rows_kernel<T, 8, 8, 8>;
        }
        return nullptr;
    }
    switch (s.C * 100 + s.R) {
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
template <class T>
size_t res_lds(int m, const ResShape& s)
{
    return s.K > 0 ? res_rows_lds<T>(s.K) : res_lds<T>(m, s.R);
}
