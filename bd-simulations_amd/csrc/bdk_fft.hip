// The three FFT passes of the mesh force (gfx950), for one simulation and for
// batches:
//   r2c rows   row transforms of the real mesh, transposed half spectrum out;
//   columns    column transform, Green's function x gradient (dm:1210-1216),
//              two inverse column transforms (Fx, Fy);
//   c2r rows   inverse row transform of Fx + i Fy -> the real force mesh.
// Power-of-two meshes: rows in registers (RowFft), sizes known at compile
// time.  Other even meshes: a plan of radices, a butterfly per thread and pass
// (bdk_fftmix.hpp), or rows in LDS, any length 2^a 3^b 5^c 7^d.
//
// The power-of-two passes in one place (us, r2c / columns / c2r; before, rows
// went through LDS for the load, every pass, the product and the store, with
// block barriers, and blocks of 256 threads took up to 16 rows of a small
// mesh): 128^2 FP64 6.6 / 12.9 / 8.9 -> 3.3 / 5.8 / 3.1, 512^2 FP32 6.9 /
// 11.2 / 8.1 -> 3.4 / 4.2 / 3.6, 1024^2 FP64 8.4 / 19.3 / 13.1 -> 5.7 / 10.7 /
// 9.0, 2048^2 FP32 14.3 / 21 / 19 -> 10.1 / 15.4 / 14.9, 4096^2 FP32 104 / 120
// / 86 -> 32 / 52 / 49.  The largest meshes are now bound by memory (134, 201
// and 268 MB at 4096^2: 3.9 to 5.5 TB/s), 2048^2 by memory and LDS about
// equally, the small ones by the chain of one global read, the passes and one
// global write.
#pragma clang fp contract(off)

#include "bdk_device.hpp"
#include "bdk_fft.hpp"
#include "bdk_fftmix.hpp"

namespace bdkx {

// LDS bytes of a block of `rows` rows; pass 0 r2c, 1 columns, 2 c2r
template <typename R, int LOGZ> static size_t p2_lds(int pass, int rows) {
    using P = P2Pass<R, LOGZ>;
    const size_t c = sizeof(typename P::C);
    if (pass == 0) return (size_t)rows * row_stride(P::Z / 2, P::ER, rows, P::per) * c;
    if (pass == 1) return (size_t)rows * P::col_stride * c;
    return (size_t)rows * row_stride(P::Z, P::E, rows, P::per) * c;
}
template <typename R, int LOGZ> static int p2_threads(int pass, int rows) {
    using P = P2Pass<R, LOGZ>;
    return rows * (pass == 0 ? P::Row::T : P::Col::T);
}

template <typename R, int LOGZ>
__global__ __launch_bounds__(FFT_MAX_THREADS) void k_r2c_rows(const R *__restrict__ rho,
                                                              typename V2<R>::T *__restrict__ ht,
                                                              const typename V2<R>::T *__restrict__ tw, int rows,
                                                              int remap) {
    r2c_p2<R, LOGZ>(rho, ht, tw, rows, xcd_block(remap));
}

template <typename R, int LOGZ>
__global__ __launch_bounds__(FFT_MAX_THREADS) void k_col(const typename V2<R>::T *__restrict__ ht,
                                                         typename V4<R>::T *__restrict__ gt,
                                                         const typename V2<R>::T *__restrict__ tw,
                                                         const R *__restrict__ sq, const R *__restrict__ lap, Geo g,
                                                         int rows) {
    col_p2<R, LOGZ>(ht, gt, tw, sq, lap, g, rows, blockIdx.x);
}

template <typename R, int LOGZ>
__global__ __launch_bounds__(FFT_MAX_THREADS) void k_c2r_rows(const typename V4<R>::T *__restrict__ gt,
                                                              typename V2<R>::T *__restrict__ fm,
                                                              const typename V2<R>::T *__restrict__ tw, int rows,
                                                              int remap, Geo g, DevBufs d, int end_step) {
    if (end_step && blockIdx.x == 0) step_end_body(g, d);
    c2r_p2<R, LOGZ>(gt, fm, tw, rows, xcd_block(remap));
}

template <typename R, int EPT>
__global__ __launch_bounds__(FFT_THREADS) void k_r2c_any(const R *__restrict__ rho, typename V2<R>::T *__restrict__ ht,
                                                         const typename V2<R>::T *__restrict__ tw, int Z, int RB,
                                                         int stride, int remap, MixPlan mp) {
    r2c_other<R, EPT>(rho, ht, tw, Z, mp, RB, stride, xcd_block(remap));
}

template <typename R, int EPT>
__global__ __launch_bounds__(FFT_THREADS) void k_col_any(const typename V2<R>::T *__restrict__ ht,
                                                         typename V4<R>::T *__restrict__ gt,
                                                         const typename V2<R>::T *__restrict__ tw,
                                                         const R *__restrict__ sq, const R *__restrict__ lap, Geo g,
                                                         int RC, int stride, MixPlan mp) {
    col_other<R, EPT>(ht, gt, tw, sq, lap, g, mp, RC, stride, blockIdx.x);
}

template <typename R, int EPT>
__global__ __launch_bounds__(FFT_THREADS) void k_c2r_any(const typename V4<R>::T *__restrict__ gt,
                                                         typename V2<R>::T *__restrict__ fm,
                                                         const typename V2<R>::T *__restrict__ tw, int Z, int RB2,
                                                         int stride, int remap, Geo g, DevBufs d, int end_step,
                                                         MixPlan mp) {
    if (end_step && blockIdx.x == 0) step_end_body(g, d);
    c2r_other<R, EPT>(gt, fm, tw, Z, mp, RB2, stride, xcd_block(remap));
}

// ------------------------------------------------------------------ batched
// One map entry per block; the size is the member's, so one launch serves
// every power-of-two mesh with the same points per thread.
// H: FP32 meshes of 1024 points and more (16 points per thread)
template <typename R, bool P, bool H>
__global__ __launch_bounds__(FFT_MAX_THREADS) void kb_r2c(const RepDev *m, const int2 *map, int nmap) {
    using C = typename V2<R>::T;
    for_entries<P, true, true>(nmap, [&](int e_) {
        const int2 t = map[e_];
        const RepDev &r = m[t.x];
#define CALL(LZ) r2c_p2<R, LZ>((const R *)r.d.rho, (C *)r.d.ht, (const C *)r.d.tw, r.rb, t.y)
        if constexpr (H) {
            switch (r.g.logZ) { BDK_LOGZ_HIGH(CALL) }
        } else if constexpr (sizeof(R) == 4) {
            switch (r.g.logZ) { BDK_LOGZ_LOW(CALL) }
        } else {
            switch (r.g.logZ) { BDK_LOGZ_LOW(CALL) BDK_LOGZ_HIGH(CALL) }
        }
#undef CALL
    });
}

template <typename R, bool P, bool H>
__global__ __launch_bounds__(FFT_MAX_THREADS) void kb_col(const RepDev *m, const int2 *map, int nmap) {
    using C = typename V2<R>::T;
    using C4 = typename V4<R>::T;
    for_entries<P, true, false>(nmap, [&](int e_) {
        const int2 t = map[e_];
        const RepDev &r = m[t.x];
        const R *sq = std::is_same<R, float>::value ? (const R *)r.d.sqf : (const R *)r.d.sq;
        const R *lap = std::is_same<R, float>::value ? (const R *)r.d.lapf : (const R *)r.d.lap;
#define CALL(LZ) col_p2<R, LZ>((const C *)r.d.ht, (C4 *)r.d.gt, (const C *)r.d.tw, sq, lap, r.g, r.rc, t.y)
        if constexpr (H) {
            switch (r.g.logZ) { BDK_LOGZ_HIGH(CALL) }
        } else if constexpr (sizeof(R) == 4) {
            switch (r.g.logZ) { BDK_LOGZ_LOW(CALL) }
        } else {
            switch (r.g.logZ) { BDK_LOGZ_LOW(CALL) BDK_LOGZ_HIGH(CALL) }
        }
#undef CALL
    });
}

template <typename R, bool P, bool H>
__global__ __launch_bounds__(FFT_MAX_THREADS) void kb_c2r(const RepDev *m, const int2 *map, int nmap, int end_step) {
    using C = typename V2<R>::T;
    using C4 = typename V4<R>::T;
    for_entries<P, true, true>(nmap, [&](int e_) {
        const int2 t = map[e_];
        const RepDev &r = m[t.x];
        if (end_step && t.y == 0) step_end_body(r.g, r.d);
#define CALL(LZ) c2r_p2<R, LZ>((const C4 *)r.d.gt, (C *)r.d.fmesh, (const C *)r.d.tw, r.rb2, t.y)
        if constexpr (H) {
            switch (r.g.logZ) { BDK_LOGZ_HIGH(CALL) }
        } else if constexpr (sizeof(R) == 4) {
            switch (r.g.logZ) { BDK_LOGZ_LOW(CALL) }
        } else {
            switch (r.g.logZ) { BDK_LOGZ_LOW(CALL) BDK_LOGZ_HIGH(CALL) }
        }
#undef CALL
    });
}

template <typename R, int EPT, bool P>
__global__ __launch_bounds__(FFT_THREADS) void kb_r2c_any(const RepDev *m, const int2 *map, int nmap) {
    using C = typename V2<R>::T;
    for_entries<P, true, true>(nmap, [&](int e_) {
        const int2 t = map[e_];
        const RepDev &r = m[t.x];
        if (r.mixr.rad)
            r2c_mix<R>((const R *)r.d.rho, (C *)r.d.ht, (const C *)r.d.tw, r.g.Z, r.mixr, r.rb, r.sR1, t.y);
        else
            r2c_any<R, EPT>((const R *)r.d.rho, (C *)r.d.ht, (const C *)r.d.tw, r.g.Z, r.rb, r.sR1, t.y);
    });
}

template <typename R, int EPT, bool P>
__global__ __launch_bounds__(FFT_THREADS) void kb_col_any(const RepDev *m, const int2 *map, int nmap) {
    using C = typename V2<R>::T;
    using C4 = typename V4<R>::T;
    for_entries<P, true, false>(nmap, [&](int e_) {
        const int2 t = map[e_];
        const RepDev &r = m[t.x];
        const R *sq = std::is_same<R, float>::value ? (const R *)r.d.sqf : (const R *)r.d.sq;
        const R *lap = std::is_same<R, float>::value ? (const R *)r.d.lapf : (const R *)r.d.lap;
        if (r.mixc.rad)
            col_mix<R>((const C *)r.d.ht, (C4 *)r.d.gt, (const C *)r.d.tw, sq, lap, r.g, r.mixc, r.rc, r.sC, t.y);
        else
            col_any<R, EPT>((const C *)r.d.ht, (C4 *)r.d.gt, (const C *)r.d.tw, sq, lap, r.g, r.rc, r.sC, t.y);
    });
}

template <typename R, int EPT, bool P>
__global__ __launch_bounds__(FFT_THREADS) void kb_c2r_any(const RepDev *m, const int2 *map, int nmap, int end_step) {
    using C = typename V2<R>::T;
    using C4 = typename V4<R>::T;
    for_entries<P, true, true>(nmap, [&](int e_) {
        const int2 t = map[e_];
        const RepDev &r = m[t.x];
        if (end_step && t.y == 0) step_end_body(r.g, r.d);
        if (r.mixc.rad)
            c2r_mix<R>((const C4 *)r.d.gt, (C *)r.d.fmesh, (const C *)r.d.tw, r.g.Z, r.mixc, r.rb2, r.sR2, t.y);
        else
            c2r_any<R, EPT>((const C4 *)r.d.gt, (C *)r.d.fmesh, (const C *)r.d.tw, r.g.Z, r.rb2, r.sR2, t.y);
    });
}

// ------------------------------------------------------------------ launchers
// the largest divisor of m not above cap (at least 1)
static int div_at_most(int m, int cap) {
    cap = std::max(1, std::min(m, cap));
    while (m % cap) --cap;
    return cap;
}

// rows of a pass (of its batch or single launch)
static int pass_rows(int pass, int Z) { return pass == 1 ? Z / 2 : Z; }
// complex values a row of the pass keeps in a block
static int pass_need(int pass, int Z) { return pass == 0 ? Z / 2 : (pass == 1 ? 2 * Z : Z); }

static size_t p2_lds_bytes(bool f32, int Z, int pass, int rows) {
#define CALL(LZ) return f32 ? p2_lds<float, LZ>(pass, rows) : p2_lds<double, LZ>(pass, rows)
    switch (__builtin_ctz(Z)) { BDK_LOGZ_LOW(CALL) BDK_LOGZ_HIGH(CALL) }
#undef CALL
    return 0;
}
static int p2_block(bool f32, int Z, int pass, int rows) {
#define CALL(LZ) return f32 ? p2_threads<float, LZ>(pass, rows) : p2_threads<double, LZ>(pass, rows)
    switch (__builtin_ctz(Z)) { BDK_LOGZ_LOW(CALL) BDK_LOGZ_HIGH(CALL) }
#undef CALL
    return 0;
}

// Rows per block of a power-of-two pass.  The columns need no company (one per
// block).  The r2c rows are stored and the c2r rows read across rows, so 4
// rows of a block make 32 or 64 consecutive bytes; below 1024 points, where
// the mesh lies in the caches, more blocks count for more.  Measured (us, rows
// 1 / 2 / 4 / 8): r2c 2048^2 FP32 15.6 / 11.8 / 10.1 / 10.3, 4096^2 80 / 45 /
// 32 / -, 1024^2 FP64 6.7 / 6.4 / 5.7 / 6.7, 512^2 FP32 3.4 / 3.8 / 3.7 / 4.1;
// c2r 2048^2 18.1 / 15.4 / 14.9 / 15.0, 4096^2 76 / 49 / 49 / -, 1024^2 FP64
// 9.6 / 9.0 / 9.3 / 9.3, 512^2 3.6 / 4.2 / 4.1 / 4.3; columns at 2 instead of
// 1: 15.4 to 15.6, 10.7 to 11.6 and 4.2 to 5.0.  At least a wave per block.
static int p2_rows(bool f32, int Z, int pass) {
    const int all = pass_rows(pass, Z), t = p2_block(f32, Z, pass, 1);
    const int want = pass == 1 || Z < 1024 ? 1 : (pass == 2 && Z < 2048 ? 2 : 4);
    int rows = 1;
    while (rows < all && (rows < want || rows * t < 64)) rows *= 2;
    while (rows > 1 && rows * t > FFT_MAX_THREADS) rows /= 2;
    return rows;
}

// The cheapest passes over n points, a pass of radix r taken to cost r + 4 (its
// chain of loads, products and sums, and its trip through LDS), with at most
// FFT_THREADS / 2 butterflies each (radices of 15 and 16 would never pay).  Largest radix first.  r2c / c2r of 192^2
// FP64 with r + 1.6, r + 4 and r + 8: 6.6 / 7.0, 5.3 / 5.9 and 5.7 / 5.9 us.  A
// wave's worth of threads per block: with two, r2c of 600^2 takes 8.2 instead of
// 7.0.
static void mix_search(int n, int left, int top, unsigned rad, int np, double cost, unsigned &best, double &best_cost) {
    static const int radices[] = {14, 12, 10, 9, 8, 7, 6, 5, 4, 3, 2};
    if (left == 1 && np >= 2 && cost < best_cost) {
        best = rad;
        best_cost = cost;
    }
    if (np == 4) return;
    for (int r : radices)
        if (r <= top && left % r == 0 && n / r <= FFT_THREADS / 2)
            mix_search(n, left / r, r, rad | (unsigned)r << (8 * np), np + 1, cost + r + 4.0, best, best_cost);
}
static MixPlan mix_plan(int n) {
    unsigned best = 0;
    double cost = 1e9;
    mix_search(n, n, 14, 0, 0, 0.0, best, cost);
    int least = 14;
    for (unsigned r = best; r; r >>= 8) least = std::min(least, (int)(r & 255));
    return {best, best ? n / least : 0};
}
void mix_plans(int Z, MixPlan &r, MixPlan &c) {
    r = c = {0, 0};
    if (zp2(Z)) return;
    r = mix_plan(Z / 2);
    c = mix_plan(Z);
    if (!r.rad || !c.rad) r = c = {0, 0};
}

// Threads and elements per thread of a pass over a mesh without a plan of
// radices (750 points a side and more): 128 threads of 8 elements where a row
// fits, else 256 threads of as many as the row needs.  Two exceptions, where
// rows side by side fill the lines that a block writes (r2c) or reads (c2r)
// across rows: r2c takes 256 threads where they hold an even number of rows and
// more than 128 do (us, 128 / 256 threads: 980^2 FP32 13.4 / 12.6, FP64 16.2 /
// 14.4, 1500^2 16.9 / 15.0 and 21.9 / 19.4, 2000^2 22.0 / 19.2 and 28.0 / 25.4;
// odd numbers 750^2 10.1 / 10.8, 1050^2 11.3 / 12.0), and c2r in FP32 from 1800
// points on two rows, 16 elements per thread (one / two rows: 1500^2 21.7 /
// 22.0, 1890^2 35.4 / 33.1, 2016^2 34.4 / 30.6; FP64 1500^2 30.1 / 35.1, 2000^2
// 45.1 / 52.1).
struct AnyCfg {
    int ept, threads, rows, stride;
    size_t lds;
};
static AnyCfg any_cfg(int pass, int Z, size_t csz) {
    const int need = pass_need(pass, Z);
    AnyCfg c;
    c.threads = need <= 8 * 128 ? 128 : FFT_THREADS;
    c.ept = ept_for(pass == 2 && csz == 8 && Z >= 1800 ? 16 : 8, need);
    c.rows = div_at_most(pass_rows(pass, Z), c.ept * c.threads / need);
    if (pass == 0 && c.threads < FFT_THREADS) {
        const int rows = div_at_most(pass_rows(pass, Z), c.ept * FFT_THREADS / need);
        if (rows > c.rows && rows % 2 == 0) {
            c.threads = FFT_THREADS;
            c.rows = rows;
        }
    }
    c.stride = lds_row(pass == 0 ? Z / 2 : Z);
    c.lds = (size_t)(pass == 1 ? 2 : 1) * c.rows * c.stride * csz;
    return c;
}

FftLaunch fft_launch(const bdk_t *h, int pass) {
    const bool f32 = h->p.precision != BDK_FP64;
    const int Z = h->g.Z;
    FftLaunch l = {};
    if (zp2(Z)) {
        l.rows = p2_rows(f32, Z, pass);
        l.threads = std::max(64, p2_block(f32, Z, pass, l.rows));
        l.lds = p2_lds_bytes(f32, Z, pass, l.rows);
    } else {
        l.mix = pass == 0 ? h->mixr : h->mixc;
        if (l.mix.rad) {
            const int per = (pass == 1 ? 2 : 1) * l.mix.tpr;  // threads per row
            l.rows = div_at_most(pass_rows(pass, Z), 64 / per);
            l.threads = 64;
            while (l.threads < l.rows * per) l.threads *= 2;
            l.stride = lds_row(pass == 0 ? Z / 2 : Z);
            l.lds = (size_t)(pass == 1 ? 2 : 1) * l.rows * l.stride * (f32 ? 8 : 16);
        } else {
            const AnyCfg c = any_cfg(pass, Z, f32 ? 8 : 16);
            l = {c.rows, c.threads, 0, c.ept, c.stride, c.lds, {0, 0}};
        }
    }
    l.blocks = pass_rows(pass, Z) / l.rows;
    return l;
}

template <typename R> static void launch_pass_p2(bdk_t *h, int pass, hipStream_t st, int end_step) {
    using C = typename V2<R>::T;
    using C4 = typename V4<R>::T;
    constexpr bool f32 = sizeof(R) == 4;
    const FftLaunch l = fft_launch(h, pass);
    const int rows = l.rows;
    const dim3 grid(l.blocks), blk(l.threads);
    const size_t lds = l.lds;
    const R *sq = f32 ? (const R *)h->d.sqf : (const R *)h->d.sq, *lap = f32 ? (const R *)h->d.lapf : (const R *)h->d.lap;
    const C *tw = (const C *)h->d.tw;
#define R2C(LZ) \
    hipLaunchKernelGGL((k_r2c_rows<R, LZ>), grid, blk, lds, st, (const R *)h->d.rho, (C *)h->d.ht, tw, rows, h->g.xcd)
#define COL(LZ)                                                                                                   \
    hipLaunchKernelGGL((k_col<R, LZ>), grid, blk, lds, st, (const C *)h->d.ht, (C4 *)h->d.gt, tw, sq, lap, h->g, \
                       rows)
#define C2R(LZ)                                                                                               \
    hipLaunchKernelGGL((k_c2r_rows<R, LZ>), grid, blk, lds, st, (const C4 *)h->d.gt, (C *)h->d.fmesh, tw, rows, \
                       h->g.xcd, h->g, h->d, end_step)
    if (pass == 0)
        switch (h->g.logZ) { BDK_LOGZ_LOW(R2C) BDK_LOGZ_HIGH(R2C) }
    else if (pass == 1)
        switch (h->g.logZ) { BDK_LOGZ_LOW(COL) BDK_LOGZ_HIGH(COL) }
    else
        switch (h->g.logZ) { BDK_LOGZ_LOW(C2R) BDK_LOGZ_HIGH(C2R) }
#undef R2C
#undef COL
#undef C2R
}

template <typename R> static void launch_pass_any(bdk_t *h, int pass, hipStream_t st, int end_step) {
    using C = typename V2<R>::T;
    using C4 = typename V4<R>::T;
    const int Z = h->g.Z;
    const FftLaunch c = fft_launch(h, pass);
    const dim3 grid(c.blocks), blk(c.threads);
    const R *sq = sizeof(R) == 4 ? (const R *)h->d.sqf : (const R *)h->d.sq;
    const R *lap = sizeof(R) == 4 ? (const R *)h->d.lapf : (const R *)h->d.lap;
    const C *tw = (const C *)h->d.tw;
#define R2C(E)                                                                                                        \
    hipLaunchKernelGGL((k_r2c_any<R, E>), grid, blk, c.lds, st, (const R *)h->d.rho, (C *)h->d.ht, tw, Z, c.rows,       \
                       c.stride, h->g.xcd, c.mix)
#define COL(E)                                                                                                        \
    hipLaunchKernelGGL((k_col_any<R, E>), grid, blk, c.lds, st, (const C *)h->d.ht, (C4 *)h->d.gt, tw, sq, lap, h->g,   \
                       c.rows, c.stride, c.mix)
#define C2R(E)                                                                                                        \
    hipLaunchKernelGGL((k_c2r_any<R, E>), grid, blk, c.lds, st, (const C4 *)h->d.gt, (C *)h->d.fmesh, tw, Z, c.rows,    \
                       c.stride, h->g.xcd, h->g, h->d, end_step, c.mix)
    if (pass == 0) {
        BDK_OTHER_SWITCH(c.ept, R2C)
    } else if (pass == 1) {
        BDK_OTHER_SWITCH(c.ept, COL)
    } else {
        BDK_OTHER_SWITCH(c.ept, C2R)
    }
#undef R2C
#undef COL
#undef C2R
}

hipError_t launch_fft_pass(bdk_t *h, int pass, hipStream_t st, int end_step) {
    if (!st) st = h->stream;
    const bool f32 = h->p.precision != BDK_FP64;
    if (zp2(h->g.Z))
        f32 ? launch_pass_p2<float>(h, pass, st, end_step) : launch_pass_p2<double>(h, pass, st, end_step);
    else
        f32 ? launch_pass_any<float>(h, pass, st, end_step) : launch_pass_any<double>(h, pass, st, end_step);
    return hipGetLastError();
}

hipError_t launch_fft(bdk_t *h) {
    hipError_t e = hipSuccess;
    for (int p = 0; p < 3 && e == hipSuccess; ++p) e = launch_fft_pass(h, p);
    return e;
}

int batch_min_ept(int stage, int zmax) { return ept_for(8, pass_need(stage, zmax)); }

// rows per block of a member's passes for the batch's block sizes
// (ept x FFT_THREADS complex values per block), and the LDS its launches need
void fft_member(RepDev &r, int Z, const int ept[3], BatchPlan &bp) {
    int rows[3];
    for (int k = 0; k < 3; ++k) {
        const int cap = ept[k] * FFT_THREADS / pass_need(k, Z);
        size_t lds;
        int kind;
        if (zp2(Z)) {
            rows[k] = 1;
            while (2 * rows[k] <= std::min(cap, pass_rows(k, Z)) &&
                   p2_block(bp.f32, Z, k, 2 * rows[k]) <= FFT_MAX_THREADS)
                rows[k] *= 2;
            lds = p2_lds_bytes(bp.f32, Z, k, rows[k]);
            kind = fft_ept(Z, bp.f32) == 16 ? 0 : 1;
            bp.fft_threads[kind][k] = std::max(bp.fft_threads[kind][k], std::max(64, p2_block(bp.f32, Z, k, rows[k])));
        } else {
            const MixPlan &mp = k == 0 ? r.mixr : r.mixc;
            rows[k] = div_at_most(pass_rows(k, Z), mp.rad ? std::min(cap, FFT_THREADS / ((k == 1 ? 2 : 1) * mp.tpr)) : cap);
            lds = (size_t)(k == 1 ? 2 : 1) * rows[k] * lds_row(k == 0 ? Z / 2 : Z) * (bp.f32 ? 8 : 16);
            kind = 2;
            bp.fft_threads[kind][k] = FFT_THREADS;
        }
        bp.fft_lds[kind][k] = std::max(bp.fft_lds[kind][k], lds);
    }
    r.rb = rows[0];
    r.rc = rows[1];
    r.rb2 = rows[2];
    r.sR1 = lds_row(Z / 2);
    r.sC = lds_row(Z);
    r.sR2 = lds_row(Z);
}

// stage 2 r2c, 3 columns, 4 c2r, 12 c2r + step end: one launch per kind of
// mesh present (16 points per thread, other powers of two, other sizes)
template <typename R, bool P> static void batch_fft_t(const BatchPlan &bp, int stage, hipStream_t st) {
    const int pass = stage == 2 ? 0 : (stage == 3 ? 1 : 2), S = pass == 0 ? BS_R2C : (pass == 1 ? BS_COL : BS_C2R);
    const int cut[4] = {0, bp.nblk16[S], bp.nblk2[S], bp.nblk[S]};
    const RepDev *m = bp.reps;
    for (int kind = 0; kind < 3; ++kind) {
        const int n = cut[kind + 1] - cut[kind];
        if (n <= 0) continue;
        const int2 *map = bp.map[S] + cut[kind];
        const dim3 grid(stage_grid(bp, n)), blk(bp.fft_threads[kind][pass]);
        const size_t lds = bp.fft_lds[kind][pass];
        const int end = stage == 12 ? 1 : 0;
        if (kind < 2) {
            auto go = [&](auto h) {
                constexpr bool H = decltype(h)::value && sizeof(R) == 4;
                if (pass == 0)
                    hipLaunchKernelGGL((kb_r2c<R, P, H>), grid, blk, lds, st, m, map, n);
                else if (pass == 1)
                    hipLaunchKernelGGL((kb_col<R, P, H>), grid, blk, lds, st, m, map, n);
                else
                    hipLaunchKernelGGL((kb_c2r<R, P, H>), grid, blk, lds, st, m, map, n, end);
            };
            if (kind == 0)
                go(std::true_type());
            else
                go(std::false_type());
        } else {
#define R2C(E) hipLaunchKernelGGL((kb_r2c_any<R, E, P>), grid, blk, lds, st, m, map, n)
#define COL(E) hipLaunchKernelGGL((kb_col_any<R, E, P>), grid, blk, lds, st, m, map, n)
#define C2R(E) hipLaunchKernelGGL((kb_c2r_any<R, E, P>), grid, blk, lds, st, m, map, n, end)
            if (pass == 0)
                BDK_EPT_SWITCH(bp.ept[0], R2C)
            else if (pass == 1)
                BDK_EPT_SWITCH(bp.ept[1], COL)
            else
                BDK_EPT_SWITCH(bp.ept[2], C2R)
#undef R2C
#undef COL
#undef C2R
        }
    }
}

void batch_fft_stage(const BatchPlan &bp, int stage, hipStream_t st) {
    const bool p = bp.tune.persist > 0;
    if (bp.f32)
        p ? batch_fft_t<float, true>(bp, stage, st) : batch_fft_t<float, false>(bp, stage, st);
    else
        p ? batch_fft_t<double, true>(bp, stage, st) : batch_fft_t<double, false>(bp, stage, st);
}

// dynamic LDS above the default limit
hipError_t fft_set_attributes() {
    hipError_t e = hipSuccess;
    auto big = [&](const void *k) {
        if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    };
#define ONE(R, LZ)                          \
    big((const void *)k_r2c_rows<R, LZ>); \
    big((const void *)k_col<R, LZ>);      \
    big((const void *)k_c2r_rows<R, LZ>);
#define BOTH(LZ) ONE(float, LZ) ONE(double, LZ)
    BOTH(3) BOTH(4) BOTH(5) BOTH(6) BOTH(7) BOTH(8) BOTH(9) BOTH(10) BOTH(11) BOTH(12)
#undef BOTH
#undef ONE
#define ONE(R, E)                              \
    big((const void *)k_r2c_any<R, E>);      \
    big((const void *)k_col_any<R, E>);      \
    big((const void *)k_c2r_any<R, E>);
#define ANY(R, E)                              \
    ONE(R, E)                                  \
    big((const void *)kb_r2c_any<R, E, false>); \
    big((const void *)kb_col_any<R, E, false>); \
    big((const void *)kb_c2r_any<R, E, false>); \
    big((const void *)kb_r2c_any<R, E, true>);  \
    big((const void *)kb_col_any<R, E, true>);  \
    big((const void *)kb_c2r_any<R, E, true>);
    ANY(float, 8) ANY(float, 16) ANY(float, 32) ANY(double, 8) ANY(double, 16) ANY(double, 32)
    ONE(float, 0) ONE(double, 0)
#undef ONE
#undef ANY
#define KB(R, P, H)                       \
    big((const void *)kb_r2c<R, P, H>); \
    big((const void *)kb_col<R, P, H>); \
    big((const void *)kb_c2r<R, P, H>);
    KB(float, false, false) KB(float, true, false) KB(float, false, true) KB(float, true, true)
    KB(double, false, false) KB(double, true, false)
#undef KB
    return e;
}

}  // namespace bdkx
