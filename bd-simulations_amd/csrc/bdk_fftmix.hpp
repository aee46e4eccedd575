// Stockham transforms of mesh rows whose length is not a power of two, one
// radix-2 to radix-14 butterfly per thread and pass (device code).
#pragma once
#include "bdk_fft.hpp"

namespace bdkx {

// cos (i = 0) and sin (i = 1) of 2 pi k / N
template <int N> __device__ __forceinline__ constexpr double root(int i, int k) {
    if constexpr (N == 5) {
        constexpr double t[2][5] = {{
        1.0, 0.30901699437494745, -0.8090169943749475, -0.8090169943749475, 0.30901699437494745},
        {
        0.0, 0.9510565162951535, 0.5877852522924731, -0.5877852522924731, -0.9510565162951535}};
        return t[i][k % N];
    }
    if constexpr (N == 6) {
        constexpr double t[2][6] = {{
        1.0, 0.5, -0.5, -1.0, -0.5, 0.5},
        {
        0.0, 0.8660254037844386, 0.8660254037844386, 0.0, -0.8660254037844386, -0.8660254037844386}};
        return t[i][k % N];
    }
    if constexpr (N == 7) {
        constexpr double t[2][7] = {{
        1.0, 0.6234898018587335, -0.2225209339563144, -0.9009688679024191, -0.9009688679024191,
        -0.2225209339563144, 0.6234898018587335},
        {
        0.0, 0.7818314824680298, 0.9749279121818236, 0.4338837391175581, -0.4338837391175581, -0.9749279121818236,
        -0.7818314824680298}};
        return t[i][k % N];
    }
    if constexpr (N == 9) {
        constexpr double t[2][9] = {{
        1.0, 0.766044443118978, 0.17364817766693036, -0.5, -0.9396926207859084, -0.9396926207859084, -0.5,
        0.17364817766693036, 0.766044443118978},
        {
        0.0, 0.6427876096865394, 0.984807753012208, 0.8660254037844386, 0.3420201433256687, -0.3420201433256687,
        -0.8660254037844386, -0.984807753012208, -0.6427876096865394}};
        return t[i][k % N];
    }
    if constexpr (N == 10) {
        constexpr double t[2][10] = {{
        1.0, 0.8090169943749475, 0.30901699437494745, -0.30901699437494745, -0.8090169943749475, -1.0,
        -0.8090169943749475, -0.30901699437494745, 0.30901699437494745, 0.8090169943749475},
        {
        0.0, 0.5877852522924731, 0.9510565162951535, 0.9510565162951535, 0.5877852522924731, 0.0,
        -0.5877852522924731, -0.9510565162951535, -0.9510565162951535, -0.5877852522924731}};
        return t[i][k % N];
    }
    if constexpr (N == 12) {
        constexpr double t[2][12] = {{
        1.0, 0.8660254037844386, 0.5, 0.0, -0.5, -0.8660254037844386, -1.0, -0.8660254037844386, -0.5, 0.0, 0.5,
        0.8660254037844386},
        {
        0.0, 0.5, 0.8660254037844386, 1.0, 0.8660254037844386, 0.5, 0.0, -0.5, -0.8660254037844386, -1.0,
        -0.8660254037844386, -0.5}};
        return t[i][k % N];
    }
    if constexpr (N == 14) {
        constexpr double t[2][14] = {{
        1.0, 0.9009688679024191, 0.6234898018587335, 0.2225209339563144, -0.2225209339563144, -0.6234898018587335,
        -0.9009688679024191, -1.0, -0.9009688679024191, -0.6234898018587335, -0.2225209339563144,
        0.2225209339563144, 0.6234898018587335, 0.9009688679024191},
        {
        0.0, 0.4338837391175581, 0.7818314824680298, 0.9749279121818236, 0.9749279121818236, 0.7818314824680298,
        0.4338837391175581, 0.0, -0.4338837391175581, -0.7818314824680298, -0.9749279121818236,
        -0.9749279121818236, -0.7818314824680298, -0.4338837391175581}};
        return t[i][k % N];
    }
    return 0.0;
}

// x = DFT_N(x) in place, with exp(-2 pi i / N)
template <int N, typename C> __device__ __forceinline__ void dft(C *x);

// N = A B: column transforms of length A, twiddles, row transforms of length B
template <int A, int B, typename C> __device__ __forceinline__ void dft_ab(C *x) {
    using R = decltype(C::x);
    C y[A * B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
        C a[A];
#pragma unroll
        for (int i = 0; i < A; ++i) a[i] = x[i * B + b];
        dft<A>(a);
#pragma unroll
        for (int k = 0; k < A; ++k) {
            const R c = (R)root<A * B>(0, b * k), s = (R)root<A * B>(1, b * k);
            y[k * B + b] = b * k == 0 ? a[k] : cmul(a[k], cm<C>(c, -s));
        }
    }
#pragma unroll
    for (int k = 0; k < A; ++k) {
        C r[B];
#pragma unroll
        for (int b = 0; b < B; ++b) r[b] = y[k * B + b];
        dft<B>(r);
#pragma unroll
        for (int b = 0; b < B; ++b) x[k + A * b] = r[b];
    }
}

// N = 5, 7 from the sums and differences of x[t] and x[N - t]
template <int N, typename C> __device__ __forceinline__ void dft_odd(C *x) {
    using R = decltype(C::x);
    constexpr int H = N / 2;
    C s[H], d[H], y[N];
    y[0] = x[0];
#pragma unroll
    for (int t = 1; t <= H; ++t) {
        s[t - 1] = cadd(x[t], x[N - t]);
        d[t - 1] = csub(x[t], x[N - t]);
        y[0] = cadd(y[0], s[t - 1]);
    }
#pragma unroll
    for (int u = 1; u <= H; ++u) {
        C a = x[0], b = cm<C>((R)0, (R)0);
#pragma unroll
        for (int t = 1; t <= H; ++t) {
            a = cadd(a, cscale(s[t - 1], (R)root<N>(0, t * u)));
            b = cadd(b, cscale(d[t - 1], (R)root<N>(1, t * u)));
        }
        const C r = cmul_mi(b);
        y[u] = cadd(a, r);
        y[N - u] = csub(a, r);
    }
#pragma unroll
    for (int u = 0; u < N; ++u) x[u] = y[u];
}

template <int N, typename C> __device__ __forceinline__ void dft(C *x) {
    if constexpr (N == 2) {
        const C a = x[0];
        x[0] = cadd(a, x[1]);
        x[1] = csub(a, x[1]);
    } else if constexpr (N == 4) {
        dft4(x, false);
    } else if constexpr (N == 5 || N == 7) {
        dft_odd<N>(x);
    } else if constexpr (N == 6 || N == 9) {
        dft_ab<3, N / 3>(x);
    } else if constexpr (N == 10) {
        dft_ab<5, 2>(x);
    } else if constexpr (N == 12) {
        dft_ab<3, 4>(x);
    } else if constexpr (N == 14) {
        dft_ab<7, 2>(x);
    } else {
        C v[N];
#pragma unroll
        for (int i = 0; i < N; ++i) v[i] = x[i];
        if constexpr (N == 3)
            dft3(v, x, false);
        else
            dft8(v, x, false);
    }
}

#define BDK_RADIX_SWITCH(r, CALL) \
    switch (r) {                  \
    case 2: CALL(2); break;       \
    case 3: CALL(3); break;       \
    case 4: CALL(4); break;       \
    case 5: CALL(5); break;       \
    case 6: CALL(6); break;       \
    case 7: CALL(7); break;       \
    case 8: CALL(8); break;       \
    case 9: CALL(9); break;       \
    case 10: CALL(10); break;     \
    case 12: CALL(12); break;     \
    default: CALL(14); break;     \
    }

// powers t < RAD of tw[i] (1, 2, 4 and 8 read, the others products)
template <int RAD, typename C> __device__ __forceinline__ void mix_tw(C (&w)[RAD], const C *__restrict__ tw, int i) {
    w[1] = tw[i];
    if constexpr (RAD > 2) w[2] = tw[2 * i];
    if constexpr (RAD > 4) w[4] = tw[4 * i];
    if constexpr (RAD > 8) w[8] = tw[8 * i];
#pragma unroll
    for (int t = 3; t < RAD; ++t) {
        if (t == 4 || t == 8) continue;
        const int h = t > 8 ? 8 : (t > 4 ? 4 : 2);
        w[t] = cmul(w[h], w[t - h]);
    }
}

template <typename C> __device__ __forceinline__ C cswap(C a) { return cm<C>(a.y, a.x); }

// One row of n points; thread j of its threads does butterfly j of every
// pass: points j + t n/RAD in, (j - k) RAD + k + t Ns out, k = j mod Ns, in the
// row's part s of LDS (point i at lp(i)).  Every thread of the block calls the
// passes; on: it has a row.  Inverse transforms are forward ones with real and
// imaginary parts swapped, when the values come and when they leave.
template <typename R> struct MixRow {
    using C = typename V2<R>::T;
    C *s;
    const C *tw;
    int n, Z, j;
    bool on;

    // the butterfly of the points from f(point)
    template <int RAD, typename F> __device__ __forceinline__ void take(C (&v)[RAD], int Ns, int k, F &&f) const {
        const int nb = n / RAD;
        C w[RAD];
        if (Ns > 1) mix_tw<RAD>(w, tw, k * (Z / (Ns * RAD)));
#pragma unroll
        for (int t = 0; t < RAD; ++t) v[t] = f(j + t * nb);
        if (Ns > 1)
#pragma unroll
            for (int t = 1; t < RAD; ++t) v[t] = cmul(v[t], w[t]);
        dft<RAD>(v);
    }
    template <int RAD> __device__ __forceinline__ void put(const C (&v)[RAD], int Ns, int k) const {
        const int base = (j - k) * RAD + k;
#pragma unroll
        for (int t = 0; t < RAD; ++t) s[lp(base + t * Ns)] = v[t];
    }
    template <int RAD> __device__ __forceinline__ bool mine() const { return on && j * RAD < n; }

    // first pass, from global memory
    template <int RAD> __device__ __forceinline__ void first(const C *__restrict__ p) const {
        if (mine<RAD>()) {
            C v[RAD];
            take<RAD>(v, 1, 0, [&](int i) { return p[i]; });
            put<RAD>(v, 1, 0);
        }
        __syncthreads();
    }
    // LDS to LDS
    template <int RAD> __device__ __forceinline__ void mid(int Ns) const {
        const int k = Dv(Ns).r(j);
        C v[RAD];
        const bool b = mine<RAD>();
        if (b) take<RAD>(v, Ns, k, [&](int i) { return s[lp(i)]; });
        __syncthreads();
        if (b) put<RAD>(v, Ns, k);
        __syncthreads();
    }
    // last pass, to out(point, value)
    template <int RAD, typename F> __device__ __forceinline__ void last(F &&out) const {
        if (!mine<RAD>()) return;
        C v[RAD];
        take<RAD>(v, n / RAD, j, [&](int i) { return s[lp(i)]; });
#pragma unroll
        for (int t = 0; t < RAD; ++t) out(j + t * (n / RAD), v[t]);
    }
    __device__ __forceinline__ void mids(unsigned r, int Ns) const {
#define CALL(RAD) mid<RAD>(Ns)
        BDK_RADIX_SWITCH(r, CALL)
#undef CALL
    }
};

// A mesh whose size is not a power of two and whose rows (Z/2 and Z points)
// split into two to four radices of at most 14, with at most FFT_THREADS / 2
// butterflies each: the rows' first pass reads and last pass writes global
// memory, the columns' product and the passes around it stay in registers.  The
// general passes (rows in LDS throughout, radices 8, 4, 2, 3, 5, 7) run the
// others.  Bound by the chain of a few waves per CU, part of it the fetch of code
// (with radices 15 and 16 in the switch, never chosen, every pass took 0.3 to 1 us more).  Before (the
// general passes) and now, us, r2c / columns / c2r: 144^2 FP32 7.1 / 10.4 / 7.4
// -> 5.1 / 6.7 / 5.2, 250^2 FP64 7.2 / 9.3 / 6.5 -> 5.1 / 9.4 / 6.1, 384^2 FP64
// 6.9 / 10.8 / 7.1 -> 5.4 / 9.7 / 6.2, 600^2 FP32 9.7 / 11.9 / 7.8 -> 6.2 / 9.6 /
// 6.8, 1000^2 FP64 14.1 / 20.4 / 15.1 -> 9.7 / 17.1 / 12.6.  Passes that all go
// through LDS with one piece of code per radix, or tables in LDS, were slower
// (384^2 FP64 columns 11.7 and 10.6 against 10.4 then).
template <typename R>
__device__ __forceinline__ void r2c_mix(const R *__restrict__ rho, typename V2<R>::T *__restrict__ ht,
                                        const typename V2<R>::T *__restrict__ tw, int Z, MixPlan mp, int rows, int stride,
                                        int blk) {
    using C = typename V2<R>::T;
    extern __shared__ unsigned char smem_raw[];
    C *s = (C *)smem_raw;
    const int tid = threadIdx.x, n = Z >> 1, k0 = blk * rows, row = Dv(mp.tpr).q(tid);
    const MixRow<R> f = {s + row * stride, tw, n, Z, tid - row * mp.tpr, row < rows};
    const C *p = (const C *)(rho + (size_t)(k0 + row) * Z);
    int Ns = mp.rad & 255;
#define CALL(RAD) f.template first<RAD>(p)
    BDK_RADIX_SWITCH(Ns, CALL)
#undef CALL
    for (unsigned r = mp.rad >> 8; r; r >>= 8) {
        f.mids(r & 255, Ns);
        Ns *= r & 255;
    }
    const Dv drb(rows);
    for (int idx = tid; idx < rows * n; idx += blockDim.x) {
        const int m = drb.q(idx), w = drb.r(idx);
        const C *q = s + w * stride;
        const C a = q[lp(m)];
        ht[(size_t)m * Z + k0 + w] = m == 0 ? cm<C>(a.x + a.y, a.x - a.y) : split_real(a, q[lp(n - m)], tw[m]);
    }
}

// the columns' last forward pass, product (fy: with the y gradient), swap and
// first inverse pass
template <typename R, int RAD>
__device__ __forceinline__ void col_turn(const MixRow<R> &f, const R *__restrict__ sq, const R *__restrict__ lap,
                                         const Geo &g, int m0, int m, int fy) {
    using C = typename V2<R>::T;
    const int Z = f.n, nb = Z / RAD;
    const bool b = f.template mine<RAD>();
    C v[RAD];
    if (b) f.template take<RAD>(v, nb, f.j, [&](int i) { return f.s[lp(i)]; });
    if (m0 == 0) {
        // the packed column pairs j with Z - j, held by other threads
        __syncthreads();
        if (b && m == 0)
#pragma unroll
            for (int t = 0; t < RAD; ++t) f.s[f.j + t * nb] = v[t];
        __syncthreads();
        if (b && m == 0)
#pragma unroll
            for (int t = 0; t < RAD; ++t) {
                const int j = f.j + t * nb;
                C x, y;
                packed_column<R, C>(j, v[t], f.s[j == 0 ? 0 : Z - j], g, sq, lap, x, y);
                v[t] = cswap(fy ? y : x);
            }
    }
    if (b && m != 0) {
#pragma unroll
        for (int t = 0; t < RAD; ++t) {
            R gx, gy;
            symbols<R>(f.j + t * nb, m, g, sq, lap, gx, gy);
            const R q = fy ? gy : gx;
            v[t] = cm<C>(q * v[t].x, -q * v[t].y);  // i q S, swapped
        }
    }
    __syncthreads();
    if (b) {
        dft<RAD>(v);
        f.template put<RAD>(v, 1, 0);
    }
    __syncthreads();
}

// Two thread groups per column, one for the x and one for the y gradient, each
// with its own forward transform: a third more work than one group for both,
// two thirds of its chain.
template <typename R>
__device__ __forceinline__ void col_mix(const typename V2<R>::T *__restrict__ ht, typename V4<R>::T *__restrict__ gt,
                                        const typename V2<R>::T *__restrict__ tw, const R *__restrict__ sq,
                                        const R *__restrict__ lap, const Geo &g, MixPlan mp, int rows, int stride,
                                        int blk) {
    using C = typename V2<R>::T;
    extern __shared__ unsigned char smem_raw[];
    const int tid = threadIdx.x, Z = g.Z, m0 = blk * rows, w = Dv(mp.tpr).q(tid), fy = w & 1, m = m0 + (w >> 1);
    const MixRow<R> f = {(C *)smem_raw + w * stride, tw, Z, Z, tid - w * mp.tpr, w < 2 * rows};
    int Ns = mp.rad & 255;
    const C *p = ht + (size_t)m * Z;
#define CALL(RAD) f.template first<RAD>(p)
    BDK_RADIX_SWITCH(Ns, CALL)
#undef CALL
    int sh = 8;  // of the radix in turn
    for (; (mp.rad >> sh) >> 8; sh += 8) {
        const int r = (mp.rad >> sh) & 255;
        f.mids(r, Ns);
        Ns *= r;
    }
    Ns = mp.rad >> sh;
#define CALL(RAD) col_turn<R, RAD>(f, sq, lap, g, m0, m, fy)
    BDK_RADIX_SWITCH(Ns, CALL)
#undef CALL
    for (sh -= 8; sh > 0; sh -= 8) {
        const int r = (mp.rad >> sh) & 255;
        f.mids(r, Ns);
        Ns *= r;
    }
    C *o = (C *)(gt + (size_t)m * Z) + fy;
#define CALL(RAD) f.template last<RAD>([&](int i, C v) { o[2 * i] = cswap(v); })
    BDK_RADIX_SWITCH((int)(mp.rad & 255), CALL)
#undef CALL
}

template <typename R>
__device__ __forceinline__ void c2r_mix(const typename V4<R>::T *__restrict__ gt, typename V2<R>::T *__restrict__ fm,
                                        const typename V2<R>::T *__restrict__ tw, int Z, MixPlan mp, int rows, int stride,
                                        int blk) {
    using C = typename V2<R>::T;
    using C4 = typename V4<R>::T;
    extern __shared__ unsigned char smem_raw[];
    C *s = (C *)smem_raw;
    const int tid = threadIdx.x, Zh = Z >> 1, k0 = blk * rows, row = Dv(mp.tpr).q(tid);
    const Dv drb(rows);
    for (int idx = tid; idx < rows * Zh; idx += blockDim.x) {
        const int m = drb.q(idx), w = drb.r(idx);
        const C4 v = gt[(size_t)m * Z + k0 + w];
        C *p = s + w * stride;
        if (m == 0) {
            p[0] = cm<C>(v.z, v.x);
            p[lp(Zh)] = cm<C>(v.w, v.y);
        } else {
            p[lp(m)] = cm<C>(v.y + v.z, v.x - v.w);
            p[lp(Z - m)] = cm<C>(-v.y + v.z, v.x + v.w);
        }
    }
    __syncthreads();
    const MixRow<R> f = {s + row * stride, tw, Z, Z, tid - row * mp.tpr, row < rows};
    int Ns = 1;
    unsigned r = mp.rad;
    for (; r >> 8; r >>= 8) {
        f.mids(r & 255, Ns);
        Ns *= r & 255;
    }
    C *o = fm + (size_t)(k0 + row) * Z;
#define CALL(RAD) f.template last<RAD>([&](int i, C v) { o[i] = cswap(v); })
    BDK_RADIX_SWITCH((int)r, CALL)
#undef CALL
}

// EPT of a launch: 0 by the plan, else the elements per thread
#define BDK_OTHER_SWITCH(E, CALL) \
    if ((E) == 0) {               \
        CALL(0);                  \
    } else                        \
        BDK_EPT_SWITCH(E, CALL)

// by the plan (EPT = 0) or with EPT elements per thread
template <typename R, int EPT>
__device__ __forceinline__ void r2c_other(const R *__restrict__ rho, typename V2<R>::T *__restrict__ ht,
                                          const typename V2<R>::T *__restrict__ tw, int Z, MixPlan mp, int rows,
                                          int stride, int blk) {
    if constexpr (EPT == 0)
        r2c_mix<R>(rho, ht, tw, Z, mp, rows, stride, blk);
    else
        r2c_any<R, EPT>(rho, ht, tw, Z, rows, stride, blk);
}
template <typename R, int EPT>
__device__ __forceinline__ void col_other(const typename V2<R>::T *__restrict__ ht, typename V4<R>::T *__restrict__ gt,
                                          const typename V2<R>::T *__restrict__ tw, const R *__restrict__ sq,
                                          const R *__restrict__ lap, const Geo &g, MixPlan mp, int rows, int stride,
                                          int blk) {
    if constexpr (EPT == 0)
        col_mix<R>(ht, gt, tw, sq, lap, g, mp, rows, stride, blk);
    else
        col_any<R, EPT>(ht, gt, tw, sq, lap, g, rows, stride, blk);
}
template <typename R, int EPT>
__device__ __forceinline__ void c2r_other(const typename V4<R>::T *__restrict__ gt, typename V2<R>::T *__restrict__ fm,
                                          const typename V2<R>::T *__restrict__ tw, int Z, MixPlan mp, int rows,
                                          int stride, int blk) {
    if constexpr (EPT == 0)
        c2r_mix<R>(gt, fm, tw, Z, mp, rows, stride, blk);
    else
        c2r_any<R, EPT>(gt, fm, tw, Z, rows, stride, blk);
}

}  // namespace bdkx
