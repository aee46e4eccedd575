// Stockham transforms of mesh rows (device code): rows of 2^n points in
// registers, rows of other lengths in LDS.
#pragma once
#include "bdk_device.hpp"

namespace bdkx {

// ------------------------------------------------------------------ FFT in LDS
// tw[k] = exp(-2 pi i k / Z), k < Z; the inverse transforms use the conjugates.
// radix-4 butterfly in place, y = DFT4(v) (inverse: conjugate kernel)
template <typename C>
__device__ __forceinline__ void dft4(C *v, bool inv) {
    C t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
    C t2 = cadd(v[1], v[3]), t3 = csub(v[1], v[3]);
    C r3 = inv ? cmul_i(t3) : cmul_mi(t3);
    v[0] = cadd(t0, t2);
    v[2] = csub(t0, t2);
    v[1] = cadd(t1, r3);
    v[3] = csub(t1, r3);
}

// radix-8 butterfly: y[2m] = DFT4(v[t] + v[t+4])[m],
// y[2m+1] = DFT4((v[t] - v[t+4]) W^t)[m], W = exp(-+2 pi i / 8)
template <typename C>
__device__ __forceinline__ void dft8(const C *v, C *y, bool inv) {
    using R = decltype(C::x);
    const R c = (R)0.70710678118654752440;
    C a[4], b[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        a[t] = cadd(v[t], v[t + 4]);
        b[t] = csub(v[t], v[t + 4]);
    }
    // b[1] *= W, b[2] *= W^2, b[3] *= W^3
    if (!inv) {
        b[1] = cm<C>(c * (b[1].x + b[1].y), c * (b[1].y - b[1].x));
        b[2] = cmul_mi(b[2]);
        b[3] = cm<C>(c * (b[3].y - b[3].x), -c * (b[3].x + b[3].y));
    } else {
        b[1] = cm<C>(c * (b[1].x - b[1].y), c * (b[1].x + b[1].y));
        b[2] = cmul_i(b[2]);
        b[3] = cm<C>(-c * (b[3].x + b[3].y), c * (b[3].x - b[3].y));
    }
    dft4(a, inv);
    dft4(b, inv);
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        y[2 * m] = a[m];
        y[2 * m + 1] = b[m];
    }
}

// radix-16 butterfly: y[2m] = DFT8(v[t] + v[t+8])[m],
// y[2m+1] = DFT8((v[t] - v[t+8]) W^t)[m], W = exp(-+2 pi i / 16)
template <typename C>
__device__ __forceinline__ void dft16(const C *v, C *y, bool inv) {
    using R = decltype(C::x);
    const R c1 = (R)0.92387953251128675613, s1 = (R)0.38268343236508977173;  // cos, sin of pi/8
    const R h = (R)0.70710678118654752440;
    // W^t = cos(t pi/8) -+ i sin(t pi/8), t = 1..7
    const R wr[8] = {(R)1, c1, h, s1, (R)0, -s1, -h, -c1};
    const R wi[8] = {(R)0, s1, h, c1, (R)1, c1, h, s1};
    C a[8], b[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        a[t] = cadd(v[t], v[t + 8]);
        b[t] = csub(v[t], v[t + 8]);
    }
    b[4] = inv ? cmul_i(b[4]) : cmul_mi(b[4]);
#pragma unroll
    for (int t = 1; t < 8; ++t) {
        if (t == 4) continue;
        const R si = inv ? wi[t] : -wi[t];
        b[t] = cm<C>(b[t].x * wr[t] - b[t].y * si, b[t].x * si + b[t].y * wr[t]);
    }
    C ya[8], yb[8];
    dft8(a, ya, inv);
    dft8(b, yb, inv);
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        y[2 * m] = ya[m];
        y[2 * m + 1] = yb[m];
    }
}

// ------------------------------------------------------------------ rows of 2^LOGN points
// Sync between the LDS writes and reads of one row: in-order LDS and a fence
// where one wave holds the whole row, else the block's barrier.
template <bool WAVE> __device__ __forceinline__ void row_sync() {
    if (WAVE) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

// Elements per thread of a power-of-two mesh: 16 in FP32 from 1024 points on
// (radix-16 passes, a 1024-point row in one wave), else 8.  It fixes the
// passes and so the rounding: the mesh decides, not the launch, so a
// simulation transforms alike alone and in a batch.
__host__ __device__ constexpr int fft_ept(int Z, bool f32) { return f32 && Z >= 1024 ? 16 : 8; }

// LDS index of element i of a row, one padding element after every E: the
// writes of a pass (strides E, E^2, ...) and the consecutive reads then touch
// every bank once per 32 lanes (8-byte elements) or 16 lanes (16-byte ones).
template <int E> __host__ __device__ __forceinline__ constexpr int lpe(int i) {
    return i + (i >> (E == 16 ? 4 : (E == 8 ? 3 : 2)));
}
// A row of 2^LOGN points, transformed by T = 2^LOGN / E threads with E points
// each in registers: thread t always holds the points t + T u, u < E.
// Stockham passes of radix E (the last one smaller if need be): butterfly
// j = t + T e takes the points j + (N/r) i, which are the thread's own, and
// its outputs k + (j - k) r + Ns i (k = j mod Ns) go through LDS to the
// threads that hold them next; after the last pass they are the thread's own
// points again.  So the first pass reads and the last pass writes global
// memory directly (consecutive threads, consecutive points), and a forward
// transform, a product and an inverse transform need no exchange between them.
// tw[k] = exp(-2 pi i k / Z), Z = 2^LOGZ; the powers a pass needs (1, 2, 4, 8;
// the others as products, up to three roundings deeper) are loaded once by
// load(), ahead of the passes, and serve both directions.
template <typename R, int LOGN, int E, int LOGZ> struct RowFft {
    using C = typename V2<R>::T;
    static constexpr int LE = E == 16 ? 4 : (E == 8 ? 3 : 2);
    static constexpr int N = 1 << LOGN, T = N / E, NP = (LOGN + LE - 1) / LE;
    static constexpr bool WAVE = T <= 64;
    static constexpr int logr(int p) { return p + 1 < NP ? LE : LOGN - LE * (NP - 1); }

    C tb[NP][8];  // base twiddles of pass p: [butterfly][power 1, 2, 4, 8] (tb[0] unused)

    __device__ __forceinline__ void load(const C *__restrict__ tw, int t) {
#pragma unroll
        for (int p = 1; p < NP; ++p) {
            const int lr = logr(p), nb = E >> lr, ns = 1 << (LE * p);
#pragma unroll
            for (int e = 0; e < nb; ++e) {
                const int k = (t + e * T) & (ns - 1);
#pragma unroll
                for (int i = 0; i < lr; ++i) tb[p][e * lr + i] = tw[(k << i) << (LOGZ - LE * p - lr)];
            }
        }
    }

    // pass P on A rows at once (their twiddle products are shared)
    template <int P, int A, bool INV> __device__ __forceinline__ void pass(C (&v)[A][E]) const {
        constexpr int LR = logr(P), RAD = 1 << LR, NB = E / RAD;
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            C w[RAD];
            if (P > 0) {
                const C *b = &tb[P][e * LR];
                w[1] = b[0];
                if (RAD >= 4) {
                    w[2] = b[1];
                    w[3] = cmul(w[1], w[2]);
                }
                if (RAD >= 8) {
                    w[4] = b[2];
                    w[5] = cmul(w[4], w[1]);
                    w[6] = cmul(w[4], w[2]);
                    w[7] = cmul(w[4], w[3]);
                }
                if (RAD == 16) {
                    w[8] = b[3];
#pragma unroll
                    for (int i = 9; i < 16; ++i) w[i] = cmul(w[8], w[i - 8]);
                }
            }
#pragma unroll
            for (int a = 0; a < A; ++a) {
                C x[RAD], y[RAD];
#pragma unroll
                for (int i = 0; i < RAD; ++i) {
                    x[i] = v[a][e + i * NB];
                    if (P > 0 && i > 0) x[i] = cmul(x[i], INV ? cconj(w[i]) : w[i]);
                }
                if constexpr (RAD == 2) {
                    y[0] = cadd(x[0], x[1]);
                    y[1] = csub(x[0], x[1]);
                } else if constexpr (RAD == 4) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) y[i] = x[i];
                    dft4(y, INV);
                } else if constexpr (RAD == 8) {
                    dft8(x, y, INV);
                } else {
                    dft16(x, y, INV);
                }
#pragma unroll
                for (int i = 0; i < RAD; ++i) v[a][e + i * NB] = y[i];
            }
        }
    }

    // the outputs of pass P through LDS to the inputs of pass P + 1; s: A
    // values per element, the row's own part of LDS
    template <int P, int A> __device__ __forceinline__ static void exchange(C (&v)[A][E], C *s, int t) {
        constexpr int LR = logr(P), RAD = 1 << LR, NB = E / RAD, NS = 1 << (LE * P);
#pragma unroll
        for (int e = 0; e < NB; ++e) {
            const int j = t + e * T, k = j & (NS - 1);
            const int base = lpe<E>(((j - k) << LR) + k);
#pragma unroll
            for (int i = 0; i < RAD; ++i) {
                // NS = 1: the E outputs of a butterfly fill one padded group
                C *q = s + A * (base + i * (NS == 1 ? 1 : lpe<E>(NS)));
#pragma unroll
                for (int a = 0; a < A; ++a) q[a] = v[a][e + i * NB];
            }
        }
        row_sync<WAVE>();
        gather<A>(v, s, t);
    }
    // the thread's points t + T u from LDS
    template <int A> __device__ __forceinline__ static void gather(C (&v)[A][E], const C *s, int t) {
#pragma unroll
        for (int u = 0; u < E; ++u) {
            const C *q = s + A * (T % E == 0 ? lpe<E>(t) + u * lpe<E>(T) : lpe<E>(t + T * u));
#pragma unroll
            for (int a = 0; a < A; ++a) v[a][u] = q[a];
        }
    }

    // whole transform of the points in v; every thread of the block calls it.
    // s holds no values still to be read by another thread (FRESH), or may
    // (the previous use ends with reads): then a sync comes first.
    template <int A, bool INV, bool FRESH, int P = 0>
    __device__ __forceinline__ void run(C (&v)[A][E], C *s, int t) const {
        pass<P, A, INV>(v);
        if constexpr (P + 1 < NP) {
            if (P > 0 || !FRESH) row_sync<WAVE>();
            exchange<P, A>(v, s, t);
            run<A, INV, FRESH, P + 1>(v, s, t);
        }
    }
};

// LDS elements from row to row of a block with `rows` rows of n points
// (padded after every E), such that the accesses across rows (row index
// fastest) spread over the banks: `per` elements fill all banks once
__host__ __device__ constexpr int row_stride(int n, int E, int rows, int per) {
    return (n + n / E + per - 1) / per * per + (rows < per ? per / rows : 1);
}

// ------------------------------------------------------------------ rows of any length
// LDS layout of these rows: element i sits at lp(i), one padding element
// after every 8; a row of n elements takes n + n/8 + 1 (odd) elements.
__device__ __forceinline__ int lp(int i) { return i + (i >> 3); }
__host__ __device__ __forceinline__ int lds_row(int n) { return n + n / 8 + 1; }

// radix-3 butterfly, y = DFT3(v): W = exp(-+2 pi i / 3) = -1/2 -+ i sqrt(3)/2
template <typename C>
__device__ __forceinline__ void dft3(const C *v, C *y, bool inv) {
    using R = decltype(C::x);
    const R h = (R)0.86602540378443864676;  // sqrt(3)/2
    const C s = cadd(v[1], v[2]), d = csub(v[1], v[2]);
    const C m = cm<C>(v[0].x - (R)0.5 * s.x, v[0].y - (R)0.5 * s.y);
    const C r = inv ? cm<C>(-h * d.y, h * d.x) : cm<C>(h * d.y, -h * d.x);  // (+-i) sqrt(3)/2 (v1 - v2)
    y[0] = cadd(v[0], s);
    y[1] = cadd(m, r);
    y[2] = csub(m, r);
}

// radix-P butterfly for P = 5, 7 as the P-point DFT, y[u] = sum_t v[t] W^(tu
// mod P), W = exp(-+2 pi i / P) = tw[Z / P] (conjugated for the inverse);
// P divides Z.
template <typename C, int P>
__device__ __forceinline__ void dftp(const C *v, C *y, const C *__restrict__ tw, int Z, bool inv) {
    const int zp = Z / P;
    C w[P];
#pragma unroll
    for (int k = 0; k < P; ++k) {
        w[k] = tw[k * zp];
        if (inv) w[k].y = -w[k].y;
    }
#pragma unroll
    for (int u = 0; u < P; ++u) {
        C acc = v[0];
#pragma unroll
        for (int t = 1; t < P; ++t) acc = cadd(acc, cmul(v[t], w[(t * u) % P]));
        y[u] = acc;
    }
}

// One Stockham pass of radix RAD (2, 3, 4, 5, 7 or 8) over rows of any
// length n divisible by RAD (the meshes whose size is not a power of two),
// with per-element LDS addresses (lp of every index), exact integer division for the butterfly and row indices,
// and every twiddle power loaded from the table: tw[t k Z / (Ns RAD)].
// Inputs are read before the barrier, outputs written after it (in place).
template <typename R, int EPT, int RAD>
__device__ __forceinline__ void fft_pass_g(typename V2<R>::T *buf, int n, int nrows, int stride, int Ns,
                                           const typename V2<R>::T *__restrict__ tw, int Z, bool inv) {
    using C = typename V2<R>::T;
    constexpr int NB = (EPT + RAD - 1) / RAD;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int nb = n / RAD, tot = nb * nrows;
    const int twm = Z / (Ns * RAD);
    const Dv dnb(nb), dns(Ns);
    C v[NB][RAD];
#pragma unroll
    for (int e = 0; e < NB; ++e) {
        const int b = tid + e * nt;
        if (b < tot) {
            const int row = dnb.q(b), j = b - row * nb;
            const C *p = buf + row * stride;
#pragma unroll
            for (int t = 0; t < RAD; ++t) v[e][t] = p[lp(j + t * nb)];
        }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < NB; ++e) {
        const int b = tid + e * nt;
        if (b < tot) {
            const int row = dnb.q(b), j = b - row * nb;
            const int k = dns.r(j);
#pragma unroll
            for (int t = 1; t < RAD; ++t) {
                C ww = tw[t * k * twm];
                if (inv) ww.y = -ww.y;
                v[e][t] = cmul(v[e][t], ww);
            }
            C y[RAD];
            if constexpr (RAD == 2) {
                y[0] = cadd(v[e][0], v[e][1]);
                y[1] = csub(v[e][0], v[e][1]);
            } else if constexpr (RAD == 3) {
                dft3(v[e], y, inv);
            } else if constexpr (RAD == 4) {
#pragma unroll
                for (int t = 0; t < 4; ++t) y[t] = v[e][t];
                dft4(y, inv);
            } else if constexpr (RAD == 8) {
                dft8(v[e], y, inv);
            } else {
                dftp<C, RAD>(v[e], y, tw, Z, inv);
            }
            C *q = buf + row * stride;
            const int base = (j - k) * RAD + k;
#pragma unroll
            for (int t = 0; t < RAD; ++t) q[lp(base + t * Ns)] = y[t];
        }
    }
    __syncthreads();
}

// Transform of rows of length n = 2^p 3^c 5^d 7^f: radix-8 passes over the
// factor 2^p, one radix-4 or radix-2 pass for its remaining bits, then one
// radix-3, -5 or -7 pass per odd factor.
template <typename R, int EPT>
__device__ __forceinline__ void lds_fft_g(typename V2<R>::T *buf, int n, int nrows, int stride,
                                          const typename V2<R>::T *__restrict__ tw, int Z, bool inv) {
    int m = n, c3 = 0, c5 = 0, c7 = 0;
    while (m % 3 == 0) {
        m /= 3;
        ++c3;
    }
    while (m % 5 == 0) {
        m /= 5;
        ++c5;
    }
    while (m % 7 == 0) {
        m /= 7;
        ++c7;
    }
    int Ns = 1;
    while (m >= 8) {
        fft_pass_g<R, EPT, 8>(buf, n, nrows, stride, Ns, tw, Z, inv);
        Ns *= 8;
        m /= 8;
    }
    if (m == 4) {
        fft_pass_g<R, EPT, 4>(buf, n, nrows, stride, Ns, tw, Z, inv);
        Ns *= 4;
    } else if (m == 2) {
        fft_pass_g<R, EPT, 2>(buf, n, nrows, stride, Ns, tw, Z, inv);
        Ns *= 2;
    }
    for (; c3 > 0; --c3) {
        fft_pass_g<R, EPT, 3>(buf, n, nrows, stride, Ns, tw, Z, inv);
        Ns *= 3;
    }
    for (; c5 > 0; --c5) {
        fft_pass_g<R, EPT, 5>(buf, n, nrows, stride, Ns, tw, Z, inv);
        Ns *= 5;
    }
    for (; c7 > 0; --c7) {
        fft_pass_g<R, EPT, 7>(buf, n, nrows, stride, Ns, tw, Z, inv);
        Ns *= 7;
    }
}

constexpr int FFT_THREADS = 256;

// elements per thread: the smallest doubling of want whose block holds `need` elements
static inline int ept_for(int want, int need) {
    int e = want;
    while (e * FFT_THREADS < need && e < 32) e *= 2;
    return e;
}

#define BDK_EPT_SWITCH(E, CALL) \
    switch (E) {                \
    case 8: CALL(8); break;     \
    case 16: CALL(16); break;   \
    default: CALL(32); break;   \
    }


// ------------------------------------------------------------------ the passes
constexpr int FFT_MAX_THREADS = 512;  // power-of-two passes

// G(j, m') = 1/((lap[j] + lap[m']) + 1/lambda^2) (dm:585-593, dm:1384-1394)
template <typename R> __device__ __forceinline__ R green(R lapj, R lapm, bool zero, R lam2inv) {
    if (zero) return (R)0.0;
    if (sizeof(R) == 4)  // FP32: the hardware reciprocal (1 ulp) instead of a correctly rounded division
        return (R)__builtin_amdgcn_rcpf((float)((lapj + lapm) + lam2inv));
    return (R)1.0 / ((lapj + lapm) + lam2inv);
}

// spectral factors of one (j, m') pair: gx = sq[j] G / Z / Z, gy = sq[m'] G / Z / Z
template <typename R>
__device__ __forceinline__ void symbols(int j, int mm, const Geo &g, const R *sq, const R *lap, R &gx, R &gy) {
    const R G = green<R>(lap[j], lap[mm], j == 0 && mm == 0 && g.zero_mode_g, (R)g.lam2inv);
    // x / Z / Z == x * 2^(-2 log2 Z) exactly where Z is a power of two
    const R izz = (R)1.0 / ((R)g.Z * (R)g.Z);
    gx = sq[j] * G * izz;
    gy = sq[mm] * G * izz;
}

// The packed (DC, Nyquist) column at j, from P = S[j] and Q = S[Z - j]:
// i g(., 0) S_dc + i (i g(., Z/2) S_ny) for x and y
template <typename R, typename C>
__device__ __forceinline__ void packed_column(int j, C P, C Q, const Geo &g, const R *sq, const R *lap, C &fx, C &fy) {
    const C Sdc = cscale(cadd(P, cconj(Q)), (R)0.5);
    const C Sny = cmul_mi(cscale(csub(P, cconj(Q)), (R)0.5));
    R gx0, gy0, gxN, gyN;
    symbols<R>(j, 0, g, sq, lap, gx0, gy0);
    symbols<R>(j, g.Z >> 1, g, sq, lap, gxN, gyN);
    fx = cadd(cmul_i(cscale(Sdc, gx0)), cmul_i(cmul_i(cscale(Sny, gxN))));
    fy = cadd(cmul_i(cscale(Sdc, gy0)), cmul_i(cmul_i(cscale(Sny, gyN))));
}

// half spectrum X[m] of a real row from its packed transform: a = z[m],
// b = z[n - m], w = exp(-2 pi i m / Z)
template <typename C> __device__ __forceinline__ C split_real(C a, C b, C w) {
    using R = decltype(C::x);
    const C bc = cconj(b);
    const C E = cscale(cadd(a, bc), (R)0.5);
    const C O = cmul_mi(cscale(csub(a, bc), (R)0.5));
    return cadd(E, cmul(w, O));
}

// ------------------------------------------------------------------ power-of-two meshes
template <typename R, int LOGZ> struct P2Pass {
    using C = typename V2<R>::T;
    static constexpr int Z = 1 << LOGZ, E = fft_ept(Z, sizeof(R) == 4);
    static constexpr int ER = E < Z / 2 ? E : Z / 2;  // of the r2c rows
    static constexpr int per = 256 / (int)sizeof(C);  // elements that fill all LDS banks once
    using Row = RowFft<R, LOGZ - 1, ER, LOGZ>;        // r2c rows: Z/2 complex points
    using Col = RowFft<R, LOGZ, E, LOGZ>;             // columns and c2r rows
    static constexpr int col_stride = 2 * (Z + Z / E) + 2;
};

// Row r2c: rows k0..k0+rows-1 of the real mesh -> half spectrum X[m], m<Z/2,
// with X[0] packing (DC, Nyquist) (both real), written transposed:
// ht[m*Z + k].  Length-Z/2 complex transform of (x[2n], x[2n+1]) + split.
// The stores take the rows of the block together (rows x 8 or 16 bytes).
template <typename R, int LOGZ>
__device__ __forceinline__ void r2c_p2(const R *__restrict__ rho, typename V2<R>::T *__restrict__ ht,
                                       const typename V2<R>::T *__restrict__ tw, int rows, int blk) {
    using P = P2Pass<R, LOGZ>;
    using F = typename P::Row;
    using C = typename P::C;
    constexpr int Z = P::Z, E = P::ER, N = F::N, T = F::T;
    extern __shared__ unsigned char smem_raw[];
    C *s = (C *)smem_raw;
    const int tid = threadIdx.x, row = tid / T, t = tid % T, k0 = blk * rows, na = rows * T;
    const int stride = row_stride(N, E, rows, P::per), lrows = __ffs(rows) - 1;
    C *sr = s + row * stride;
    const bool act = tid < na;
    if (act || !F::WAVE) {
        const C *p = (const C *)(rho + (size_t)(k0 + row) * Z) + t;
        C v[1][E];
#pragma unroll
        for (int u = 0; u < E; ++u) v[0][u] = p[T * u];
        F f;
        f.load(tw, t);
        f.template run<1, false, true>(v, sr, t);
        if (F::NP > 1) row_sync<F::WAVE>();
#pragma unroll
        for (int u = 0; u < E; ++u) sr[T % E == 0 ? lpe<E>(t) + u * lpe<E>(T) : lpe<E>(t + T * u)] = v[0][u];
    }
    C w[E];
#pragma unroll
    for (int u = 0; u < E; ++u) w[u] = tw[((tid + u * na) >> lrows) & (N - 1)];
    __syncthreads();
    if (!act) return;
#pragma unroll
    for (int u = 0; u < E; ++u) {
        const int i = tid + u * na, m = i >> lrows, r = i & (rows - 1);
        const C *p = s + r * stride;
        const C a = p[lpe<E>(m)];
        C o;
        if (m == 0)
            o = cm<C>(a.x + a.y, a.x - a.y);
        else
            o = split_real(a, p[lpe<E>(N - m)], w[u]);
        ht[(size_t)m * Z + k0 + r] = o;
    }
}

// Column pass: rows m0..m0+rows-1 of ht (length Z along x), forward
// transform, times i*gx and i*gy, inverse transform of both together, out
// gt[m*Z+k] = (Fx, Fy).  The spectrum stays in registers in between.
template <typename R, int LOGZ>
__device__ __forceinline__ void col_p2(const typename V2<R>::T *__restrict__ ht, typename V4<R>::T *__restrict__ gt,
                                       const typename V2<R>::T *__restrict__ tw, const R *__restrict__ sq,
                                       const R *__restrict__ lap, const Geo &g, int rows, int blk) {
    using P = P2Pass<R, LOGZ>;
    using F = typename P::Col;
    using C = typename P::C;
    using C4 = typename V4<R>::T;
    constexpr int Z = P::Z, E = P::E, T = F::T;
    extern __shared__ unsigned char smem_raw[];
    C *s = (C *)smem_raw;
    const int tid = threadIdx.x, row = tid / T, t = tid % T, m0 = blk * rows, m = m0 + row;
    const bool act = tid < rows * T;
    C *sr = s + row * P::col_stride;
    F f;
    C v[1][E], xy[2][E];
    if (act || !F::WAVE) {
        const C *p = ht + (size_t)m * Z + t;
#pragma unroll
        for (int u = 0; u < E; ++u) v[0][u] = p[T * u];
        f.load(tw, t);
        f.template run<1, false, true>(v, sr, t);
    }
    if (m0 == 0) {
        // the packed column pairs j with Z - j, held by other threads
        __syncthreads();
        if (act && m == 0)
#pragma unroll
            for (int u = 0; u < E; ++u) sr[t + T * u] = v[0][u];
        __syncthreads();
        if (act && m == 0)
#pragma unroll
            for (int u = 0; u < E; ++u) {
                const int j = t + T * u;
                packed_column<R, C>(j, v[0][u], sr[(Z - j) & (Z - 1)], g, sq, lap, xy[0][u], xy[1][u]);
            }
        __syncthreads();
    }
    if (!act && F::WAVE) return;
    if (m != 0) {
        const R sqm = sq[m], lapm = lap[m], l2 = (R)g.lam2inv, izz = (R)1.0 / ((R)Z * (R)Z);
#pragma unroll
        for (int u = 0; u < E; ++u) {
            const int j = t + T * u;
            const R G = green<R>(lap[j], lapm, false, l2);
            const R gx = sq[j] * G * izz, gy = sqm * G * izz;
            const C S = v[0][u];
            xy[0][u] = cm<C>(-gx * S.y, gx * S.x);
            xy[1][u] = cm<C>(-gy * S.y, gy * S.x);
        }
    }
    f.template run<2, true, F::NP == 1>(xy, sr, t);
    C4 *o = gt + (size_t)m * Z + t;
#pragma unroll
    for (int u = 0; u < E; ++u) {
        C4 q;
        q.x = xy[0][u].x;
        q.y = xy[0][u].y;
        q.z = xy[1][u].x;
        q.w = xy[1][u].y;
        o[T * u] = q;
    }
}

// Row c2r of the two real signals Fx, Fy: rows k0..k0+rows-1, spectrum
// C[m] = X[m] + i Y[m] completed by Hermitian symmetry, inverse transform of
// length Z, out fmesh[k*Z + l] = (Re, Im) = (Fx, Fy).
template <typename R, int LOGZ>
__device__ __forceinline__ void c2r_p2(const typename V4<R>::T *__restrict__ gt, typename V2<R>::T *__restrict__ fm,
                                       const typename V2<R>::T *__restrict__ tw, int rows, int blk) {
    using P = P2Pass<R, LOGZ>;
    using F = typename P::Col;
    using C = typename P::C;
    using C4 = typename V4<R>::T;
    constexpr int Z = P::Z, E = P::E, T = F::T;
    extern __shared__ unsigned char smem_raw[];
    C *s = (C *)smem_raw;
    const int tid = threadIdx.x, row = tid / T, t = tid % T, k0 = blk * rows, na = rows * T;
    const int stride = row_stride(Z, E, rows, P::per), lrows = __ffs(rows) - 1;
    const bool act = tid < na;
    F f;
    if (act) {
        C4 q[E / 2];
#pragma unroll
        for (int u = 0; u < E / 2; ++u) {
            const int i = tid + u * na;
            q[u] = gt[(size_t)(i >> lrows) * Z + k0 + (i & (rows - 1))];
        }
        f.load(tw, t);
#pragma unroll
        for (int u = 0; u < E / 2; ++u) {
            const int i = tid + u * na, m = i >> lrows;
            C *p = s + (i & (rows - 1)) * stride;
            if (m == 0) {
                p[0] = cm<C>(q[u].x, q[u].z);
                p[lpe<E>(Z / 2)] = cm<C>(q[u].y, q[u].w);
            } else {
                p[lpe<E>(m)] = cm<C>(q[u].x - q[u].w, q[u].y + q[u].z);
                p[lpe<E>(Z - m)] = cm<C>(q[u].x + q[u].w, -q[u].y + q[u].z);
            }
        }
    }
    __syncthreads();
    if (!act && F::WAVE) return;
    C *sr = s + row * stride;
    C v[1][E];
    F::template gather<1>(v, sr, t);
    f.template run<1, true, false>(v, sr, t);
    C *o = fm + (size_t)(k0 + row) * Z + t;
#pragma unroll
    for (int u = 0; u < E; ++u) o[T * u] = v[0][u];
}

// ------------------------------------------------------------------ other meshes
// Rows in LDS: the block's rows are read, transformed in place and written.
template <typename R, int EPT>
__device__ __forceinline__ void r2c_any(const R *__restrict__ rho, typename V2<R>::T *__restrict__ ht,
                                        const typename V2<R>::T *__restrict__ tw, int Z, int RB, int stride, int blk) {
    using C = typename V2<R>::T;
    extern __shared__ unsigned char smem_raw[];
    C *s = (C *)smem_raw;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int n = Z >> 1;
    const Dv dn(n), drb(RB);
    const int k0 = blk * RB;
    for (int idx = tid; idx < RB * n; idx += nt) {
        const int row = dn.q(idx), m = dn.r(idx);
        s[row * stride + lp(m)] = ((const C *)(rho + (size_t)(k0 + row) * Z))[m];
    }
    __syncthreads();
    lds_fft_g<R, EPT>(s, n, RB, stride, tw, Z, false);
    for (int idx = tid; idx < RB * n; idx += nt) {
        const int m = drb.q(idx), row = drb.r(idx);
        const C *p = s + row * stride;
        const C a = p[lp(m)];
        ht[(size_t)m * Z + k0 + row] = m == 0 ? cm<C>(a.x + a.y, a.x - a.y) : split_real(a, p[lp(n - m)], tw[m]);
    }
}

template <typename R, int EPT>
__device__ __forceinline__ void col_any(const typename V2<R>::T *__restrict__ ht, typename V4<R>::T *__restrict__ gt,
                                        const typename V2<R>::T *__restrict__ tw, const R *__restrict__ sq,
                                        const R *__restrict__ lap, const Geo &g, int RC, int stride, int blk) {
    using C = typename V2<R>::T;
    using C4 = typename V4<R>::T;
    extern __shared__ unsigned char smem_raw[];
    C *s = (C *)smem_raw;
    C *sB = s + RC * stride;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int Z = g.Z, Zh = Z >> 1;
    const Dv dz(Z);
    const int m0 = blk * RC;
    for (int idx = tid; idx < RC * Z; idx += nt) {
        const int row = dz.q(idx), k = dz.r(idx);
        s[row * stride + lp(k)] = ht[(size_t)(m0 + row) * Z + k];
    }
    __syncthreads();
    lds_fft_g<R, EPT>(s, Z, RC, stride, tw, Z, false);
    for (int idx = tid; idx < RC * Z; idx += nt) {
        const int row = dz.q(idx), j = dz.r(idx);
        const int m = m0 + row;
        if (m == 0) {
            // packed (DC, Nyquist) column: pairs (j, Z-j) by one thread
            if (j > Zh) continue;
            const int jn = j == 0 ? 0 : Z - j;
            const C P = s[lp(j)], Q = s[lp(jn)];
            C fx, fy, gx, gy;
            packed_column<R, C>(j, P, Q, g, sq, lap, fx, fy);
            packed_column<R, C>(jn, Q, P, g, sq, lap, gx, gy);
            s[lp(j)] = fx;
            sB[lp(j)] = fy;
            if (jn != j) {
                s[lp(jn)] = gx;
                sB[lp(jn)] = gy;
            }
        } else {
            R gx, gy;
            symbols<R>(j, m, g, sq, lap, gx, gy);
            const int o = row * stride + lp(j);
            const C S = s[o];
            s[o] = cm<C>(-gx * S.y, gx * S.x);
            sB[o] = cm<C>(-gy * S.y, gy * S.x);
        }
    }
    __syncthreads();
    lds_fft_g<R, EPT>(s, Z, 2 * RC, stride, tw, Z, true);
    for (int idx = tid; idx < RC * Z; idx += nt) {
        const int row = dz.q(idx), k = dz.r(idx);
        const int so = row * stride + lp(k);
        const C a = s[so], b = sB[so];
        C4 o;
        o.x = a.x;
        o.y = a.y;
        o.z = b.x;
        o.w = b.y;
        gt[(size_t)(m0 + row) * Z + k] = o;
    }
}

template <typename R, int EPT>
__device__ __forceinline__ void c2r_any(const typename V4<R>::T *__restrict__ gt, typename V2<R>::T *__restrict__ fm,
                                        const typename V2<R>::T *__restrict__ tw, int Z, int RB2, int stride,
                                        int blk) {
    using C = typename V2<R>::T;
    using C4 = typename V4<R>::T;
    extern __shared__ unsigned char smem_raw[];
    C *s = (C *)smem_raw;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int Zh = Z >> 1;
    const Dv dz(Z), drb(RB2);
    const int k0 = blk * RB2;
    for (int idx = tid; idx < RB2 * Zh; idx += nt) {
        const int m = drb.q(idx), row = drb.r(idx);
        const C4 v = gt[(size_t)m * Z + k0 + row];
        C *p = s + row * stride;
        if (m == 0) {
            p[0] = cm<C>(v.x, v.z);
            p[lp(Zh)] = cm<C>(v.y, v.w);
        } else {
            p[lp(m)] = cm<C>(v.x - v.w, v.y + v.z);
            p[lp(Z - m)] = cm<C>(v.x + v.w, -v.y + v.z);
        }
    }
    __syncthreads();
    lds_fft_g<R, EPT>(s, Z, RB2, stride, tw, Z, true);
    for (int idx = tid; idx < RB2 * Z; idx += nt) {
        const int row = dz.q(idx), l = dz.r(idx);
        fm[(size_t)(k0 + row) * Z + l] = s[row * stride + lp(l)];
    }
}

// a pass over one mesh: rows per block, threads and LDS of a block; for meshes
// whose size is not a power of two also the LDS row stride and the plan of the
// row's passes (ept = 0) or the elements per thread
struct FftLaunch {
    int rows, threads, blocks, ept, stride;
    size_t lds;
    MixPlan mix;
};
FftLaunch fft_launch(const bdk_t *h, int pass);

#define BDK_LOGZ_LOW(CALL) \
    case 3: CALL(3); break;   \
    case 4: CALL(4); break;   \
    case 5: CALL(5); break;   \
    case 6: CALL(6); break;   \
    case 7: CALL(7); break;   \
    case 8: CALL(8); break;   \
    case 9: CALL(9); break;
#define BDK_LOGZ_HIGH(CALL) \
    case 10: CALL(10); break; \
    case 11: CALL(11); break; \
    default: CALL(12); break;

}  // namespace bdkx
