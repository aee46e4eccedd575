// Device helpers shared by the kernel files: complex arithmetic, Philox noise,
// workgroup order, mesh indices and weights, the WCA pair, a block scan.
#pragma once
#pragma clang fp contract(off)

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <type_traits>

#include "bdk_internal.hpp"

namespace bdkx {


template <typename R> struct V2;
template <> struct V2<float> { using T = float2; };
template <> struct V2<double> { using T = double2; };
template <typename R> struct V4;
template <> struct V4<float> { using T = float4; };
template <> struct V4<double> { using T = double4; };

// Complex helpers of the FFT and spectral arithmetic.  The complex product
// uses explicit fused multiply-adds (the file compiles without automatic
// contraction, so every kernel that inlines it rounds the same way).
template <typename C> __device__ __forceinline__ C cm(decltype(C::x) a, decltype(C::x) b) {
    C r;
    r.x = a;
    r.y = b;
    return r;
}
template <typename C> __device__ __forceinline__ C cadd(C a, C b) { return cm<C>(a.x + b.x, a.y + b.y); }
template <typename C> __device__ __forceinline__ C csub(C a, C b) { return cm<C>(a.x - b.x, a.y - b.y); }
template <typename C> __device__ __forceinline__ C cconj(C a) { return cm<C>(a.x, -a.y); }
template <typename C> __device__ __forceinline__ C cmul(C a, C b) {
    return cm<C>(fma(a.x, b.x, -(a.y * b.y)), fma(a.x, b.y, a.y * b.x));
}
template <typename C> __device__ __forceinline__ C cmul_i(C a) { return cm<C>(-a.y, a.x); }    // i*a
template <typename C> __device__ __forceinline__ C cmul_mi(C a) { return cm<C>(a.y, -a.x); }   // -i*a
template <typename C> __device__ __forceinline__ C cscale(C a, decltype(C::x) s) { return cm<C>(a.x * s, a.y * s); }

__device__ __forceinline__ double dbits(unsigned long long b) { return __longlong_as_double((long long)b); }
__device__ __forceinline__ unsigned long long bitsd(double v) { return (unsigned long long)__double_as_longlong(v); }

// ------------------------------------------------------------------ Philox
// Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11).
__device__ __forceinline__ void philox4x32_10(uint32_t c[4], uint32_t k0, uint32_t k1) {
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r) {
            k0 += 0x9E3779B9u;
            k1 += 0xBB67AE85u;
        }
        // one 32x32 -> 64-bit product each (a single multiply instruction
        // instead of separate low and high halves)
        const uint64_t p0 = (uint64_t)0xD2511F53u * c[0], p1 = (uint64_t)0xCD9E8D57u * c[2];
        const uint32_t hi0 = (uint32_t)(p0 >> 32), lo0 = (uint32_t)p0;
        const uint32_t hi1 = (uint32_t)(p1 >> 32), lo1 = (uint32_t)p1;
        uint32_t n0 = hi1 ^ c[1] ^ k0;
        uint32_t n2 = hi0 ^ c[3] ^ k1;
        c[0] = n0;
        c[1] = lo1;
        c[2] = n2;
        c[3] = lo0;
    }
}

// noise of particle `pid` at step `step`: disc of radius sqrt 5 (variance
// 5/4 per component, the distribution of dm:1321-1325) or Gaussian.
__device__ __forceinline__ double2 philox_noise(unsigned long long seed, uint32_t pid, unsigned long long step,
                                                int gauss, double var) {
    uint32_t c[4] = {pid, (uint32_t)step, (uint32_t)(step >> 32), 0x4244u};
    philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    const double inv53 = 1.0 / 9007199254740992.0;
    double u1 = (double)(((((unsigned long long)c[1]) << 32) | c[0]) >> 11) * inv53;
    double u2 = (double)(((((unsigned long long)c[3]) << 32) | c[2]) >> 11) * inv53;
    double r = gauss ? sqrt(-2.0 * var * log(1.0 - u1)) : sqrt(5.0 * u1);
    double a = 2.0 * M_PI * u2;
    double sa, ca;
    sincos(a, &sa, &ca);
    double2 o;
    o.x = r * ca;
    o.y = r * sa;
    return o;
}

// The same draws in FP32 (FP32 force mode: the random force is a force):
// u1, u2 are the high words of the FP64 path's 64-bit draws rounded to FP32
// (relative error <= 2^-24 + 2^-32/u), r and the angle in FP32.
__device__ __forceinline__ double2 philox_noise_f32(unsigned long long seed, uint32_t pid, unsigned long long step,
                                                    int gauss, double var) {
    uint32_t c[4] = {pid, (uint32_t)step, (uint32_t)(step >> 32), 0x4244u};
    philox4x32_10(c, (uint32_t)seed, (uint32_t)(seed >> 32));
    const float u1 = fminf((float)c[1] * 2.3283064365386963e-10f, 0.99999994f);  // 2^-32, below 1
    const float u2 = (float)c[3] * 2.3283064365386963e-10f;
    const float r = gauss ? sqrtf(-2.0f * (float)var * logf(1.0f - u1)) : sqrtf(5.0f * u1);
    float sa, ca;
    sincospif(2.0f * u2, &sa, &ca);
    double2 o;
    o.x = (double)(r * ca);
    o.y = (double)(r * sa);
    return o;
}

// ------------------------------------------------------------------ launch order
// Workgroups are dispatched round-robin over the 8 XCDs, each with its own
// L2.  Renumbered so that every XCD runs one contiguous range of the logical
// grid, neighbouring tiles (whose inputs overlap) share an L2.
__device__ __forceinline__ int xcd_of(int b, int nb, int on) {  // block b of nb
    if (!on) return b;
    const int x = b & 7, i = b >> 3, base = nb >> 3, rem = nb & 7;
    return x < rem ? x * (base + 1) + i : rem * (base + 1) + (x - rem) * base + i;
}
__device__ __forceinline__ int xcd_block(int on) {
    return xcd_of(blockIdx.x + blockIdx.y * gridDim.x, gridDim.x * gridDim.y, on);
}

// Two kinds of work in one launch: na blocks of the first and nb of the
// second, interleaved evenly in groups of eight, so that block i of either
// kind runs on XCD i mod 8 as in a launch of its own.
struct PairGrid {
    int na, nb;
    unsigned long long share;  // groups of the first kind per group, 32 fractional bits
    PairGrid(int na_, int nb_) : na(na_), nb(nb_) {
        const unsigned long long ga = (na + 7) / 8, all = groups();
        share = ((ga << 32) + all - 1) / all;
    }
    unsigned long long groups() const { return (na + 7) / 8 + (nb + 7) / 8; }
    unsigned blocks() const { return (unsigned)(8 * groups()); }
    // the block's kind and number there; false: nothing to do
    __device__ __forceinline__ bool mine(bool &first, int &i) const {
        const unsigned long long grp = blockIdx.x >> 3;
        const int a0 = (int)((grp * share) >> 32), a1 = (int)(((grp + 1) * share) >> 32);
        first = a1 > a0;
        i = (first ? a0 : (int)grp - a0) * 8 + (int)(blockIdx.x & 7);
        return i < (first ? na : nb);
    }
};

// ------------------------------------------------------------------ geometry
__device__ __forceinline__ int wrapc(int u, int n) {
    int v = u % n;
    return v < 0 ? v + n : v;
}
// u in [-n, 2n)
__device__ __forceinline__ int wrap1(int u, int n) { return u < 0 ? u + n : (u >= n ? u - n : u); }
// Mesh code is compiled for two kinds of mesh size: P2 (Z a power of two:
// masks and shifts) and the other even sizes.  The kind is a template
// parameter of every mesh kernel, chosen by its launcher, so the
// power-of-two instruction stream carries no test of the other.
// mesh index u in [-Z, 2Z) into [0, Z)
template <bool P2> __device__ __forceinline__ int wrapz(int u, int Z) { return P2 ? (u & (Z - 1)) : wrap1(u, Z); }
// any two mesh indices into [0, Z): a state may hold offsets of many boxes (|rel| < 1e9)
template <bool P2> __device__ __forceinline__ void foldz(int &k, int &l, int Z) {
    if (P2) {
        k &= Z - 1;
        l &= Z - 1;
        return;
    }
    const int a = wrap1(k, Z), b = wrap1(l, Z);
    if (__builtin_expect(max((unsigned)a, (unsigned)b) >= (unsigned)Z, 0)) {
        k = wrapc(k, Z);
        l = wrapc(l, Z);
    } else {
        k = a;
        l = b;
    }
}
// x / d and x % d for 0 <= x < 2^22: a shift when d is a power of two, else
// the float reciprocal corrected to the exact quotient
struct Dv {
    int d, sh;
    float inv;
    __device__ explicit Dv(int d_)
        : d(d_), sh((d_ & (d_ - 1)) == 0 ? __ffs(d_) - 1 : -1), inv(__builtin_amdgcn_rcpf((float)d_)) {}
    __device__ int q(int x) const {
        if (sh >= 0) return x >> sh;
        int v = (int)((float)x * inv);
        const int r = x - v * d;
        v += (r >= d) - (r < 0);
        return v;
    }
    __device__ int r(int x) const { return sh >= 0 ? (x & (d - 1)) : x - q(x) * d; }
};
// c / nc for 0 <= c < 2^24 (float reciprocal, corrected to the exact quotient)
__device__ __forceinline__ int div_nc(int c, const Geo &g) {
    int q = (int)((float)c * g.ncinv);
    const int r = c - q * g.nc;
    q += (r >= g.nc) - (r < 0);
    return q;
}

// mesh index and weights along one axis (NGP gr:44-54, CIC gr:154-190,
// TSC gr:435-459), evaluated in FP64 in the reference's operation order
template <int SCHEME>
__device__ __forceinline__ void weights1d(double x, double h, int &k, double w[3]) {
    int kk = (int)(x / h);
    k = kk;
    if (SCHEME == 0) {
        w[0] = 0.0;
        w[1] = 1.0;
        w[2] = 0.0;
    } else if (SCHEME == 1) {
        double tmp = x / h - (kk + 0.5);
        w[1] = 1.0 - fabs(tmp);
        if (tmp < 0.0) {
            w[0] = -tmp;
            w[2] = 0.0;
        } else {
            w[0] = 0.0;
            w[2] = tmp;
        }
    } else {
        double d = x - (kk + 0.5) * h;
        w[1] = 0.75 - d * d / h / h;
        double tmp = fabs((d + h) / h);
        w[0] = 0.5 * (1.5 - tmp) * (1.5 - tmp);
        tmp = fabs((d - h) / h);
        w[2] = 0.5 * (1.5 - tmp) * (1.5 - tmp);
    }
}

// Weights in the precision of the forces: FP64 follows the reference's
// operations exactly; FP32 takes the index from x/h in FP64 and evaluates
// the offset t = x/h - k - 1/2 and the textbook weights (CIC: 1-|t|, -t, t;
// TSC: 3/4-t^2, (1/2-t)^2/2, (1/2+t)^2/2) in FP32.
template <typename R, int SCHEME>
__device__ __forceinline__ void weights_r(double x, const Geo &g, int &k, R w[3]) {
    if (std::is_same<R, double>::value) {
        double wd[3];
        weights1d<SCHEME>(x, g.h, k, wd);
        w[0] = (R)wd[0];
        w[1] = (R)wd[1];
        w[2] = (R)wd[2];
        return;
    }
    if (SCHEME == 0) {
        k = (int)(x / g.h);
        w[0] = 0;
        w[1] = 1;
        w[2] = 0;
        return;
    }
    // CIC/TSC weights are continuous across a cell edge, so x * (1/h) may
    // pick the neighbouring index at an exact edge without changing the sum
    const double u = x * g.hinv;
    const int kk = (int)u;
    k = kk;
    const float t = (float)(u - (kk + 0.5));
    if (SCHEME == 1) {
        w[1] = 1.0f - fabsf(t);
        w[0] = t < 0.0f ? -t : 0.0f;
        w[2] = t < 0.0f ? 0.0f : t;
    } else {
        const float a = 0.5f - t, b = 0.5f + t;
        w[1] = 0.75f - t * t;
        w[0] = 0.5f * a * a;
        w[2] = 0.5f * b * b;
    }
}

// One WCA pair, the arithmetic of dm:640-698 (type 0, pair 11), dm:815-868
// (type 1, pair 22) and dm:987-1040 (type 2, pair 12): force on particle a
// at (xa,ya) from b at (xb,yb).  Minimum image as abstand2 (am:100-166) and
// the shift logic of dm:663-676.  Returns false outside the cutoff.
template <typename R>
__device__ __forceinline__ bool wca_pair(double xa, double ya, double xb, double yb, int type, const Geo &g,
                                         R &fx, R &fy) {
    const double L = g.L;
    double t1 = xa - xb, t2 = xa - xb + L, t3 = xa - xb - L;
    double m23 = (t3 * t3 < t2 * t2) ? t3 * t3 : t2 * t2;
    double dx2 = (m23 < t1 * t1) ? m23 : t1 * t1;
    t1 = ya - yb;
    t2 = ya - yb + L;
    t3 = ya - yb - L;
    m23 = (t3 * t3 < t2 * t2) ? t3 * t3 : t2 * t2;
    double dy2 = (m23 < t1 * t1) ? m23 : t1 * t1;
    double a2 = dx2 + dy2;
    double sig = type == 1 ? g.s22 : g.s12;
    if (type == 0) {
        if (a2 > g.cut2) return false;
    } else {
        if (a2 * sig * sig > g.cut2) return false;
    }
    double x2 = xb, y2 = yb;
    double dx = xa - x2, dy = ya - y2;
    if (dx * dx + dy * dy > a2) {
        if ((dx - L) * (dx - L) < dx * dx)
            x2 += L;
        else if ((dx + L) * (dx + L) < dx * dx)
            x2 -= L;
        dx = xa - x2;
        if ((dy - L) * (dy - L) < dy * dy)
            y2 += L;
        else if ((dy + L) * (dy + L) < dy * dy)
            y2 -= L;
        dy = ya - y2;
    }
    if (type != 0) {
        a2 *= sig * sig;
        dx *= sig;
        dy *= sig;
    }
    const R ra2 = (R)a2;
    const R a_8 = (R)1.0 / (ra2 * ra2 * ra2 * ra2);
    const R a_14 = (R)1.0 / (ra2 * ra2 * ra2 * ra2 * ra2 * ra2 * ra2);
    R absF;
    if (type == 0)
        absF = (R)4.0 * (R)6.0 * ((R)2.0 * a_14 - a_8);
    else
        absF = (R)(type == 1 ? g.e22f : g.e12f) * (R)4.0 * (R)6.0 * ((R)2.0 * a_14 - a_8);
    if (absF > (R)g.maxpair) absF = (R)g.maxpair;
    fx = absF * (R)dx;
    fy = absF * (R)dy;
    return true;
}

// End of a step: step counter + 1, and the per-step scalars of the next
// update re-armed (dt minimum and the 64 slots of dt candidates, excursion
// slot, displacement bound).  Run by threads 0..63 of one block of the
// step's last mesh pass (k_c2r_rows), which follows every reader of these
// scalars in the step.
__device__ __forceinline__ void step_end_body(const Geo &g, const DevBufs &d) {
    const int t = threadIdx.x;
    if (t < 64) {
        d.exo[t * 16] = 0ull;
        d.dts[t * 16] = ~0ull;
    }
    if (t == 0) {
        const unsigned long long s = d.sc->step;
        d.sc->dt_bits = bitsd(g.dt_max);
        d.sc->exc_bits[s & 1] = 0ull;  // filled by the update of step s + 1
        d.sc->step = s + 1;
    }
}


// ------------------------------------------------------------------ block scan
// exclusive scan of a[0..n) in LDS (n <= 4*blockDim.x, blockDim.x <= 1024),
// returns the total; all threads must call it
static __device__ int block_exscan4(int *a, int n, int *wsum) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, nw = (blockDim.x + 63) >> 6;
    int v[4];
    int s = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        int idx = 4 * tid + q;
        v[q] = idx < n ? a[idx] : 0;
        s += v[q];
    }
    int x = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    int woff = 0, total = 0;
    for (int q = 0; q < nw; ++q) {
        if (q < w) woff += wsum[q];
        total += wsum[q];
    }
    int e = woff + x - s;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        int idx = 4 * tid + q;
        if (idx < n) a[idx] = e;
        e += v[q];
    }
    __syncthreads();
    return total;
}

// ------------------------------------------------------------------ batches
// Every batched kernel walks its stage's block map: one map entry per block,
// or in the persistent form (a grid smaller than the map) each block takes
// the entries blockIdx.x, blockIdx.x + gridDim.x, ...  Kernels whose bodies
// use LDS end every entry with a barrier, so the next entry may refill it.
// A member's results do not depend on the grid or on the WCA block size
// (per-particle sums, integer deposit sums, order-free min/max reductions).
// P (persistent) selects the form at compile time: without it a kernel
// handles exactly its own entry (no loop, so the code and its register use
// are those of a plain one-entry kernel).
// XCD: the entries in contiguous ranges per XCD, as the single-simulation
// kernels run, so a member's blocks share an L2 between the particle stages
// and the FFT passes. 32 members of 16,384 particles on 512^2: 176 -> 167 us
// per step. The stages whose single kernels run in plain order (scan, sort,
// column pass) or order their tiles themselves (deposit) pass false.
template <bool P, bool SYNC, bool XCD, typename F> __device__ __forceinline__ void for_entries(int nmap, F &&f) {
    if (!P) {
        f(XCD ? xcd_of((int)blockIdx.x, nmap, 1) : (int)blockIdx.x);
        return;
    }
    for (int e = blockIdx.x; e < nmap; e += gridDim.x) {
        f(e);
        if (SYNC) __syncthreads();
    }
}

static inline bool zp2(int Z) { return (Z & (Z - 1)) == 0; }
static inline unsigned nblk(size_t n, int b) { return (unsigned)((n + b - 1) / b); }

// blocks of a launch over a map of n entries (the persistent form caps them)
static inline unsigned stage_grid(const BatchPlan &bp, int n) {
    const int p = bp.tune.persist;
    return (unsigned)std::max(1, p > 0 ? std::min(n, p) : n);
}

}  // namespace bdkx
