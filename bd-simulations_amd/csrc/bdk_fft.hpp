// Stockham transforms of rows held in LDS (device code).
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

// LDS layout of the FFT rows: element i of a row sits at lp(i), one padding
// element after every 8.  The output strides of the first Stockham passes
// (8 and 64 elements) then spread over the banks instead of piling onto a
// few (measured: half the LDS cycles of the unpadded passes were bank
// conflicts).  A row of n elements takes n + n/8 + 1 (odd) elements.
__device__ __forceinline__ int lp(int i) { return i + (i >> 3); }
__host__ __device__ __forceinline__ int lds_row(int n) { return n + n / 8 + 1; }

// One Stockham pass of radix RAD (2, 4 or 8) over nrows rows of length
// n = 2^logn held in LDS (row stride `stride`, layout lp), in place: every thread reads
// its butterflies' inputs (and, for small register footprints, their
// twiddles: powers 1, 2, 4 from the FP64-built table, 3, 5, 6, 7 as
// products) before the barrier and writes the outputs after it.  Twiddle of input t of butterfly j: tw[(t k) << twsh],
// k = j mod Ns (conjugated for the inverse transform).
// Output index ((j - k) << LR) + k + t Ns with Ns a power of 8 maps to
// lp(base) + t (Ns + Ns/8); input index j + t nb to lp(j) + t (nb + nb/8)
// when nb is a multiple of 8 (SMALL: nb < 8, mapped per element).
template <typename R, int EPT, int RAD, bool SMALL>
__device__ __forceinline__ void fft_pass(typename V2<R>::T *buf, int logn, int nrows, int stride, int logNs,
                                         const typename V2<R>::T *__restrict__ tw, int logZ, bool inv) {
    using C = typename V2<R>::T;
    constexpr int LR = RAD == 16 ? 4 : (RAD == 8 ? 3 : (RAD == 4 ? 2 : 1));
    // butterflies per thread (radix 16 at 8 elements per thread: one, on half
    // of the threads)
    constexpr int NB = EPT >= RAD ? EPT / RAD : 1;
    constexpr bool PRE = sizeof(R) == 4 && NB * (RAD - 1) <= 16;  // twiddles fetched before the barrier
    const int tid = threadIdx.x, nt = blockDim.x;
    const int lognb = logn - LR, nb = 1 << lognb;
    const int tot = nb * nrows;
    const int Ns = 1 << logNs;
    const int twsh = logZ - (logNs + LR);
    const int nbp = nb + (nb >> 3), Nsp = Ns + (Ns >> 3);
    C v[NB][RAD];
    C w[PRE ? NB : 1][RAD - 1];
    // twiddles of butterfly k: tw^1, tw^2, tw^4 (and tw^8) from the table,
    // the other powers as products (one to three roundings deeper; 3 loads
    // instead of 7 for radix 8, 4 instead of 15 for radix 16).  Every tiling
    // forms them the same way -- before the barrier when the registers allow
    // (PRE), else after it -- so the transform's rounding does not depend on
    // the elements per thread.
    auto twiddles = [&](int k, C *ww) {
        ww[0] = tw[k << twsh];
        if (RAD >= 4) {
            ww[1] = tw[(2 * k) << twsh];
            ww[2] = cmul(ww[0], ww[1]);
        }
        if (RAD >= 8) {
            ww[3] = tw[(4 * k) << twsh];
            ww[4] = cmul(ww[3], ww[0]);
            ww[5] = cmul(ww[3], ww[1]);
            ww[6] = cmul(ww[3], ww[2]);
        }
        if (RAD == 16) {
            ww[7] = tw[(8 * k) << twsh];
#pragma unroll
            for (int t = 8; t < 15; ++t) ww[t] = cmul(ww[7], ww[t - 8]);
        }
    };
#pragma unroll
    for (int e = 0; e < NB; ++e) {
        const int b = tid + e * nt;
        if (b < tot) {
            const int row = b >> lognb, j = b & (nb - 1);
            const C *p = buf + row * stride;
            if (SMALL) {
#pragma unroll
                for (int t = 0; t < RAD; ++t) v[e][t] = p[lp(j + t * nb)];
            } else {
                p += lp(j);
#pragma unroll
                for (int t = 0; t < RAD; ++t) v[e][t] = p[t * nbp];
            }
            if (PRE) twiddles(j & (Ns - 1), w[PRE ? e : 0]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < NB; ++e) {
        const int b = tid + e * nt;
        if (b < tot) {
            const int row = b >> lognb, j = b & (nb - 1);
            const int k = j & (Ns - 1);
            C wl[RAD - 1];
            if (!PRE) twiddles(k, wl);
#pragma unroll
            for (int t = 1; t < RAD; ++t) {
                C ww = PRE ? w[PRE ? e : 0][t - 1] : wl[t - 1];
                if (inv) ww.y = -ww.y;
                v[e][t] = cmul(v[e][t], ww);
            }
            C y[RAD];
            if (RAD == 2) {
                y[0] = cadd(v[e][0], v[e][1]);
                y[1] = csub(v[e][0], v[e][1]);
            } else if (RAD == 4) {
#pragma unroll
                for (int t = 0; t < 4; ++t) y[t] = v[e][t];
                dft4(y, inv);
            } else if (RAD == 8) {
                dft8(v[e], y, inv);
            } else {
                dft16(v[e], y, inv);
            }
            if (RAD == 16 && Ns < 8) {
                // the first radix-16 pass (Ns = 1): outputs 16 j + t straddle a
                // padding element, so each takes its own padded index
                C *q = buf + row * stride;
                const int base = (j - k) << LR;
#pragma unroll
                for (int t = 0; t < RAD; ++t) q[lp(base + k + t * Ns)] = y[t];
            } else {
                C *q = buf + row * stride + lp(((j - k) << LR) + k);
#pragma unroll
                for (int t = 0; t < RAD; ++t) q[t * Nsp] = y[t];
            }
        }
    }
    __syncthreads();
}

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
// length n divisible by RAD (the meshes whose size is not a power of two).
// The same butterflies as fft_pass, with per-element LDS addresses (lp of
// every index), exact integer division for the butterfly and row indices,
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
// radix-3, -5 or -7 pass per odd factor.  A power-of-two n takes fft_pass
// (below).
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

// rows of length n: the power-of-two passes below, or lds_fft_g when n has an
// odd factor (tw holds exp(-2 pi i k / Z), k < Z; n divides Z).  R16: the
// kernel's power-of-two rows take radix-16 passes (FP32); a kernel's choice
// does not depend on its elements per thread, so neither does its rounding.
template <typename R, int EPT, bool R16 = false, bool R16T = false>
__device__ __forceinline__ void lds_fft_pow2(typename V2<R>::T *buf, int logn, int nrows, int stride,
                                             const typename V2<R>::T *__restrict__ tw, int logZ, bool inv);
template <typename R, int EPT>
__device__ __forceinline__ void lds_fft(typename V2<R>::T *buf, int n, int nrows, int stride,
                                        const typename V2<R>::T *__restrict__ tw, int Z, bool inv) {
    if ((n & (n - 1)) == 0 && (Z & (Z - 1)) == 0)
        lds_fft_pow2<R, EPT>(buf, __ffs(n) - 1, nrows, stride, tw, __ffs(Z) - 1, inv);
    else
        lds_fft_g<R, EPT>(buf, n, nrows, stride, tw, Z, inv);
}
// the same with the mesh kind known at compile time (P2: n and Z powers of two)
template <typename R, int EPT, bool P2, bool R16 = false, bool R16T = false>
__device__ __forceinline__ void lds_fft_t(typename V2<R>::T *buf, int n, int nrows, int stride,
                                          const typename V2<R>::T *__restrict__ tw, int Z, bool inv) {
    if (P2)
        lds_fft_pow2<R, EPT, R16, R16T>(buf, __ffs(n) - 1, nrows, stride, tw, __ffs(Z) - 1, inv);
    else
        lds_fft_g<R, EPT>(buf, n, nrows, stride, tw, Z, inv);
}

// radix-8 passes (radix-16 passes with R16), then one pass of a smaller radix
// for the remaining bits
template <typename R, int EPT, bool R16, bool R16T>
__device__ __forceinline__ void lds_fft_pow2(typename V2<R>::T *buf, int logn, int nrows, int stride,
                                             const typename V2<R>::T *__restrict__ tw, int logZ, bool inv) {
    int logNs = 0;
    if constexpr (R16T && sizeof(R) == 4) {
        // radix-8 passes, with the last 4 bits (when radix 8 would leave one
        // bit for a radix-2 pass) in one radix-16 pass: 1024 points in passes
        // of 8, 8 and 16
        if (logn >= 7 && logn % 3 == 1) {
            while (logn - logNs > 4) {
                fft_pass<R, EPT, 8, false>(buf, logn, nrows, stride, logNs, tw, logZ, inv);
                logNs += 3;
            }
            fft_pass<R, EPT, 16, false>(buf, logn, nrows, stride, logNs, tw, logZ, inv);
            return;
        }
    }
    if constexpr (R16 && sizeof(R) == 4) {
        // FP32 rows of at least 128: radix-16 passes, then one pass of radix
        // 8, 4 or 2 for the remaining bits (2048 points in 3 passes instead
        // of 4)
        if (logn >= 7) {
            while (logn - logNs >= 4) {
                fft_pass<R, EPT, 16, false>(buf, logn, nrows, stride, logNs, tw, logZ, inv);
                logNs += 4;
            }
            const int rem = logn - logNs;
            if (rem == 3)
                fft_pass<R, EPT, 8, false>(buf, logn, nrows, stride, logNs, tw, logZ, inv);
            else if (rem == 2)
                fft_pass<R, EPT, 4, false>(buf, logn, nrows, stride, logNs, tw, logZ, inv);
            else if (rem == 1)
                fft_pass<R, EPT, 2, false>(buf, logn, nrows, stride, logNs, tw, logZ, inv);
            return;
        }
    }
    const bool small8 = logn - 3 < 3;  // nb = n/8 below 8
    while (logn - logNs >= 3) {
        if (small8)
            fft_pass<R, EPT, 8, true>(buf, logn, nrows, stride, logNs, tw, logZ, inv);
        else
            fft_pass<R, EPT, 8, false>(buf, logn, nrows, stride, logNs, tw, logZ, inv);
        logNs += 3;
    }
    if (logn - logNs == 2) {
        if (logn - 2 < 3)
            fft_pass<R, EPT, 4, true>(buf, logn, nrows, stride, logNs, tw, logZ, inv);
        else
            fft_pass<R, EPT, 4, false>(buf, logn, nrows, stride, logNs, tw, logZ, inv);
    } else if (logn - logNs == 1) {
        if (logn - 1 < 3)
            fft_pass<R, EPT, 2, true>(buf, logn, nrows, stride, logNs, tw, logZ, inv);
        else
            fft_pass<R, EPT, 2, false>(buf, logn, nrows, stride, logNs, tw, logZ, inv);
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


}  // namespace bdkx
