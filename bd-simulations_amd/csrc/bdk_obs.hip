// Device observables: rho(k) by FFT and by direct sums, pair correlations,
// radial profiles, the snapshot density grid.
#pragma clang fp contract(off)

#include "bdk_device.hpp"
#include "bdk_fft.hpp"

namespace bdkx {

// Column sums of part[nrow][ncol] in a fixed order: 32 columns x 32 threads
// per block, thread y adds rows y, y + 32, ..., then its 32 sums are added in
// order.
__global__ __launch_bounds__(1024) void k_sum_rows(const double *__restrict__ part, int nrow, int ncol,
                                                   double *__restrict__ out) {
    __shared__ double sm[32][33];
    const int x = threadIdx.x & 31, y = threadIdx.x >> 5, c = blockIdx.x * 32 + x;
    double v = 0.0;
    if (c < ncol)
        for (int r = y; r < nrow; r += 32) v += part[(size_t)r * ncol + c];
    sm[y][x] = v;
    __syncthreads();
    if (y == 0 && c < ncol) {
        for (int k = 1; k < 32; ++k) v += sm[k][x];
        out[c] = v;
    }
}

static void launch_sum_rows(const double *part, int nrow, int ncol, double *out, hipStream_t st) {
    hipLaunchKernelGGL(k_sum_rows, dim3(nblk(ncol, 32)), dim3(1024), 0, st, part, nrow, ncol, out);
}

// rho(k) of one species (record_rhoFFTW, auswertung.cpp:529-626): the
// species' number density (weights drho, gridRoutinen.cpp:672-1040) is
// transformed (r2c rows + this column pass), multiplied by (-1)^(i+j)
// (the origin moved to the box centre) and the real parts are summed over
// shells bin = (int)(dq_dqFT |k|/dq + 1/2) of the full Z x Z plane: a
// column m of the half spectrum stands for itself and its mirror
// (Z-j, Z-m), whose conjugate adds the same real part (the imaginary parts
// cancel).
//
// Along a column the bin grows with |j|, so a shell is a range of |j| (found
// from its radius, then corrected with the binning expression itself): one
// thread per shell sums the range in order into the column's partial row
// [sums][lattice points], and k_sum_rows adds the rows in order.  One thread
// per column over all j took 850 us at Z = 2048 (its add waits on the
// previous one's LDS round trip) and the host counted the plane's lattice
// points for 7 ms; a call is now bound by the deposit and the two passes:
// 16.6 ms -> 0.17 ms for both species of 2M particles.
__device__ __forceinline__ int shell_bin(int a, double m2, double dqr) {
    return (int)(dqr * sqrt((double)a * a + m2) + 0.5);
}
// the first a in [0, Zh + 1] whose bin is at least b
__device__ __forceinline__ int shell_begin(int b, double m2, double dqr, int Zh) {
    const double r = ((double)b - 0.5) / dqr, a2 = r * r - m2;
    int a = r <= 0.0 || a2 <= 0.0 ? 0 : (int)fmin(sqrt(a2), (double)Zh + 1.0);
    while (a > 0 && shell_bin(a - 1, m2, dqr) >= b) --a;
    while (a <= Zh && shell_bin(a, m2, dqr) < b) ++a;
    return a;
}

// the shells of column m's transform, point i at s[at(i)]
template <typename C, typename F>
__device__ __forceinline__ void shell_sums(const C *s, F &&at, int m, int Z, double dqr, int nbins, double *part) {
    const int tid = threadIdx.x, Zh = Z >> 1;
    // column m > 0, or the DC (col = 0) and Nyquist (col = Z/2) columns that
    // share the packed column 0
    for (int t = tid; t < (m == 0 ? 2 : 1) * nbins; t += blockDim.x) {
        const int b = t < nbins ? t : t - nbins, col = m > 0 ? m : (t < nbins ? 0 : Zh);
        const double m2 = (double)col * col;
        const int a0 = shell_begin(b, m2, dqr, Zh), a1 = shell_begin(b + 1, m2, dqr, Zh);
        double v = 0.0, n = 0.0;
        for (int a = a0; a < a1; ++a) {
            // |j| = a: j = a and Z - a (one of them for a = 0 and Z/2)
            const bool two = a > 0 && a < Zh;
            const C P = s[at(a)], Q = s[at(a == 0 ? 0 : Z - a)];
            double w = two ? (double)P.x + (double)Q.x : (double)P.x;
            if (m > 0)
                w *= 2.0;
            else if (col == 0)  // real parts of the DC column: (P + conj Q)/2
                w = (two ? 1.0 : 0.5) * ((double)P.x + (double)Q.x);
            else
                w = (two ? 1.0 : 0.5) * ((double)P.y + (double)Q.y);
            v += ((a + col) & 1) ? -w : w;  // (-1)^(j + col), Z even
            n += two ? 2.0 : 1.0;
        }
        double *p = part + (size_t)col * 2 * nbins;
        p[b] = v;
        p[nbins + b] = m > 0 ? 2.0 * n : n;
    }
}

// power-of-two meshes: one column per block, the transform by its first Z/E
// threads (all of them where several waves take part)
template <typename R, int LOGZ>
__global__ __launch_bounds__(512) void k_col_rhok(const typename V2<R>::T *__restrict__ ht,
                                                  const typename V2<R>::T *__restrict__ tw, double dqr, int nbins,
                                                  double *part) {
    using C = typename V2<R>::T;
    constexpr int Z = 1 << LOGZ, E = fft_ept(Z, sizeof(R) == 4);
    using F = RowFft<R, LOGZ, E, LOGZ>;
    extern __shared__ unsigned char smem_raw[];
    C *s = (C *)smem_raw;
    const int m = blockIdx.x, t = threadIdx.x;
    if (t < F::T) {
        C v[1][E];
#pragma unroll
        for (int u = 0; u < E; ++u) v[0][u] = ht[(size_t)m * Z + t + F::T * u];
        F f;
        f.load(tw, t);
        f.template run<1, false, true>(v, s, t);
        if (F::NP > 1) row_sync<F::WAVE>();
#pragma unroll
        for (int u = 0; u < E; ++u) s[lpe<E>(t + F::T * u)] = v[0][u];
    }
    __syncthreads();
    shell_sums(s, [](int i) { return lpe<E>(i); }, m, Z, dqr, nbins, part);
}

// other meshes
template <typename R, int EPT>
__global__ __launch_bounds__(FFT_THREADS) void k_col_rhok_any(const typename V2<R>::T *__restrict__ ht,
                                                              const typename V2<R>::T *__restrict__ tw, int Z,
                                                              double dqr, int nbins, double *part) {
    using C = typename V2<R>::T;
    extern __shared__ unsigned char smem_raw[];
    C *s = (C *)smem_raw;
    const int m = blockIdx.x;
    for (int k = threadIdx.x; k < Z; k += blockDim.x) s[lp(k)] = ht[(size_t)m * Z + k];
    __syncthreads();
    lds_fft_g<R, EPT>(s, Z, 1, lds_row(Z), tw, Z, false);
    shell_sums(s, [](int i) { return lp(i); }, m, Z, dqr, nbins, part);
}

template <typename R> static void launch_rhok_t(bdk_t *h, double dqr, int nbins, double *part, double *out) {
    using C = typename V2<R>::T;
    const int Z = h->g.Z;
    const C *ht = (const C *)h->d.ht, *tw = (const C *)h->d.tw;
    const size_t lds = (size_t)(Z + Z / 8 + 1) * sizeof(C);
    auto big = [](const void *k) {
        (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    };
    if (zp2(Z)) {
        // blocks whose barriers every thread reaches: exactly the row's
        // threads where they are more than a wave
        const int T = Z / fft_ept(Z, sizeof(R) == 4), nt = T > 64 ? T : 256;
#define RHOK(LZ)                                                                                                 \
    big((const void *)k_col_rhok<R, LZ>);                                                                        \
    hipLaunchKernelGGL((k_col_rhok<R, LZ>), dim3(Z / 2), dim3(nt), lds, h->stream, ht, tw, dqr, nbins, part)
        switch (h->g.logZ) {
        case 3: RHOK(3); break;
        case 4: RHOK(4); break;
        case 5: RHOK(5); break;
        case 6: RHOK(6); break;
        case 7: RHOK(7); break;
        case 8: RHOK(8); break;
        case 9: RHOK(9); break;
        case 10: RHOK(10); break;
        case 11: RHOK(11); break;
        default: RHOK(12); break;
        }
#undef RHOK
    } else {
        const int ept = ept_for(8, Z);
#define RHOK(E)                                                                                                    \
    big((const void *)k_col_rhok_any<R, E>);                                                                       \
    hipLaunchKernelGGL((k_col_rhok_any<R, E>), dim3(Z / 2), dim3(FFT_THREADS), lds, h->stream, ht, tw, Z, dqr, nbins, \
                       part)
        BDK_EPT_SWITCH(ept, RHOK)
#undef RHOK
    }
    launch_sum_rows(part, Z / 2 + 1, 2 * nbins, out, h->stream);
}

// species density -> rho, r2c rows, column pass + shells
hipError_t launch_rhok(bdk_t *h, int species, double dqr, int nbins, double *part, double *out) {
    hipError_t e = launch_species_deposit(h, species);
    if (e == hipSuccess) e = launch_fft_pass(h, 0);
    if (e != hipSuccess) return e;
    if (h->p.precision != BDK_FP64)
        launch_rhok_t<float>(h, dqr, nbins, part, out);
    else
        launch_rhok_t<double>(h, dqr, nbins, part, out);
    return hipGetLastError();
}

// Pair correlation g11, g12, g22 (record_korrelationsfunktion11/12/22,
// auswertung.cpp:110-188): minimum-image distances (abstand2, am:100-166)
// of all pairs closer than nbins*dr, binned by (int)(r/dr).  Every unordered
// pair is visited once and counted with integer atomics in LDS per block, a
// same-species pair as two (both orders) and a 12 pair as one, then added to
// the global histograms: the counts are exact and deterministic.
//
// Bound by the pair arithmetic (FP64 distances; 8.0M pairs at N = 4000).
// The bin comes from an FP32 square root and a multiplication; only a value
// within its error of a bin edge (a fraction 1e-6 to 1e-3 of the pairs) takes
// the FP64 square root and division that define it.
//
// N = 4000, r up to L/2 (751 bins): 12.5 ms -> 24 us for the kernel.  One
// thread per particle over all 71,000 cells had 16 blocks on the chip and
// read two list starts per mostly empty cell.  Jobs of 1024 x 64 pairs on 256
// blocks, four pairs of a thread in flight: 24 us; one at a time 36; 512 x 64
// 30, 256 x 64 on 512 blocks 27 (more bins cleared and added per pair), 256 x
// 128 49.
constexpr int PH_THREADS = 1024;   // particles i per job, one per thread
constexpr int PH_J = 64;          // particles j per job, staged in LDS
constexpr long long PH_JOB_MAX = (1LL << 30) / (PH_THREADS * PH_J);  // jobs per block: 2 counts each in 32 bits

struct PairBins {
    int nbins;
    double dr;
    float inv;   // 1/dr
    float umax;  // beyond it no bin
};

// bin of a squared distance d2 (FP64); nbins or more: none
__device__ __forceinline__ int pair_bin(double d2, const PairBins &pb) {
    const float u = __builtin_amdgcn_sqrtf((float)d2) * pb.inv;
    if (!(u < pb.umax)) return pb.nbins;
    const int b = (int)u;
    // u is within 2^-21 u of sqrt(d2)/dr (three roundings and a 1-ulp root):
    // away from the bin's edges its integer part is the exact one
    const float fr = u - (float)b, eps = 1e-6f + 5e-7f * u;
    if (fr < eps || fr > 1.0f - eps) return (int)(sqrt(d2) / pb.dr);
    return b;
}
// counts one pair; type 0: 11, 1: 12, 2: 22
__device__ __forceinline__ void pair_count(double d2, int type, const PairBins &pb, unsigned int *sh) {
    const int b = pair_bin(d2, pb);
    if (b < pb.nbins) atomicAdd(&sh[type * pb.nbins + b], type == 1 ? 1u : 2u);
}

// min over the images of t, t + L, t - L of the square (|t| below 2 L: the
// nearer image is |t| - L)
__device__ __forceinline__ double image2(double t, double L) {
    const double u = fabs(t), v = u - L;
    const double a = u * u, b = v * v;
    return b < a ? b : a;
}

__device__ __forceinline__ void pair_flush(const unsigned int *sh, int nbins, unsigned long long *hist) {
    for (int b = threadIdx.x; b < 3 * nbins; b += blockDim.x)
        if (sh[b]) atomicAdd(&hist[b], (unsigned long long)sh[b]);
}

// All pairs (the cells within R cells cover the box): jobs of PH_THREADS
// particles i (one per thread) times PH_J particles j > i in LDS; tile I of
// particles i meets the j tiles from its own first position on.
__global__ __launch_bounds__(PH_THREADS) void k_pair_hist_all(Geo g, DevBufs d, PairBins pb,
                                                              unsigned long long *hist) {
    extern __shared__ unsigned int shist[];  // [3][nbins]
    __shared__ double2 sx[PH_J];
    __shared__ int ss[PH_J];
    const int tid = threadIdx.x;
    for (int b = tid; b < 3 * pb.nbins; b += PH_THREADS) shist[b] = 0u;
    const int nj = (g.N + PH_J - 1) / PH_J;
    constexpr int STEP = PH_THREADS / PH_J;
    auto load = [&](int q, double2 &x, int &s2) {
        const int c = d.lcell[q], cx = div_nc(c, g), cy = c - cx * g.nc;
        const double2 r = d.lrel[q];
        x.x = cx * g.B + r.x;
        x.y = cy * g.B + r.y;
        s2 = d.lpid[q] >= g.n1 ? 1 : 0;
    };
    long long job = blockIdx.x;
    int I = 0, have = -1;
    double2 xi = make_double2(0.0, 0.0);
    int s2i = 0;
    for (;;) {
        while (I * STEP < nj && job >= nj - I * STEP) {
            job -= nj - I * STEP;
            ++I;
        }
        if (I * STEP >= nj) break;
        const int qi = I * PH_THREADS + tid;
        if (have != I) {
            have = I;
            if (qi < g.N) load(qi, xi, s2i);
        }
        const int j0 = (I * STEP + (int)job) * PH_J, jn = min(PH_J, g.N - j0);
        __syncthreads();
        if (tid < jn) load(j0 + tid, sx[tid], ss[tid]);
        __syncthreads();
        if (qi < g.N) {
            // four pairs at a time: their LDS reads and square roots overlap
            int k = max(0, qi + 1 - j0);
            for (; k + 4 <= jn; k += 4) {
                double d2[4];
                int ty[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const double2 xj = sx[k + e];
                    ty[e] = s2i + ss[k + e];
                    d2[e] = image2(xi.x - xj.x, g.L) + image2(xi.y - xj.y, g.L);
                }
                int b[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) b[e] = pair_bin(d2[e], pb);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (b[e] < pb.nbins) atomicAdd(&shist[ty[e] * pb.nbins + b[e]], ty[e] == 1 ? 1u : 2u);
            }
            for (; k < jn; ++k) {
                const double2 xj = sx[k];
                pair_count(image2(xi.x - xj.x, g.L) + image2(xi.y - xj.y, g.L), s2i + ss[k], pb, shist);
            }
        }
        job += gridDim.x;
    }
    __syncthreads();
    pair_flush(shist, pb.nbins, hist);
}

// Pairs within R cells, 2 R + 1 < nc: one thread per particle (list
// position) and range of row offsets.  The cells (cx + a, cy - R .. cy + R)
// of a row are one range of the list, two where y wraps; rows a > 0 hold
// each pair once, row 0 is taken from the particle on.
__global__ __launch_bounds__(256) void k_pair_hist_near(Geo g, DevBufs d, PairBins pb, int R, int rows_per,
                                                        unsigned long long *hist) {
    extern __shared__ unsigned int shist[];  // [3][nbins]
    for (int b = threadIdx.x; b < 3 * pb.nbins; b += blockDim.x) shist[b] = 0u;
    __syncthreads();
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < g.N) {
        const int nc = g.nc, c = d.lcell[q];
        const int cx = div_nc(c, g), cy = c - cx * nc;
        const double2 ri = d.lrel[q];
        const double xi = cx * g.B + ri.x, yi = cy * g.B + ri.y, L = g.L;
        const int s2i = d.lpid[q] >= g.n1 ? 1 : 0;
        const int a0 = blockIdx.y * rows_per, a1 = min(a0 + rows_per, R + 1);
        for (int a = a0; a < a1; ++a) {
            const int ux = wrap1(cx + a, nc), row = ux * nc;
            const double xr = ux * g.B;
            // row 0: the rest of the own cell, then the cells above it
            const int lo = a == 0 ? cy : cy - R, hi = cy + R;
            for (int part = 0; part < 2; ++part) {
                int y0, y1;  // inclusive cells of this part
                if (part == 0) {
                    y0 = max(lo, 0);
                    y1 = min(hi, nc - 1);
                } else if (lo < 0) {
                    y0 = lo + nc;
                    y1 = nc - 1;
                } else if (hi >= nc) {
                    y0 = 0;
                    y1 = hi - nc;
                } else {
                    break;
                }
                const int je = d.start[row + y1 + 1];
                int j = d.start[row + y0];
                if (a == 0 && part == 0) j = q + 1;
                for (; j < je; ++j) {
                    const double2 rj = d.lrel[j];
                    const int uy = d.lcell[j] - row;
                    const int s2j = d.lpid[j] >= g.n1 ? 1 : 0;
                    pair_count(image2(xi - (xr + rj.x), L) + image2(yi - (uy * g.B + rj.y), L), s2i + s2j, pb, shist);
                }
            }
        }
    }
    __syncthreads();
    pair_flush(shist, pb.nbins, hist);
}

// All pairs where the cells within R cover the box, else the rows of cells.
hipError_t launch_pair_hist(bdk_t *h, int nbins, double dr, unsigned long long *hist) {
    const Geo &g = h->g;
    int R = (int)std::min(ceil(nbins * dr / g.B), (double)g.nc);
    if (R < 1) R = 1;
    // (outside FP32's comfortable range 1/dr is left 0: every bin from FP64)
    const PairBins pb = {nbins, dr, dr > 1e-12 && dr < 1e12 ? (float)(1.0 / dr) : 0.0f,
                         (float)nbins * 1.00001f + 1.0f};
    const size_t lds = (size_t)3 * nbins * sizeof(unsigned int);
    if (2 * R + 1 >= g.nc) {
        const long long nj = nblk(g.N, PH_J), ni = nblk(g.N, PH_THREADS);
        const long long jobs = ni * nj - (PH_THREADS / PH_J) * (ni * (ni - 1) / 2);
        // one block per compute unit, more where the 32-bit counts need it
        const long long grid = std::max(std::min(jobs, 256LL), (jobs + PH_JOB_MAX - 1) / PH_JOB_MAX);
        hipLaunchKernelGGL(k_pair_hist_all, dim3((unsigned)grid), dim3(PH_THREADS), lds, h->stream, g, h->d, pb, hist);
    } else {
        // rows split over blocks while the particles alone leave the chip idle
        const int nb = (int)nblk(g.N, 256), want = std::max(1, std::min(R + 1, 1024 / nb));
        const int per = (int)nblk(R + 1, want);
        hipLaunchKernelGGL(k_pair_hist_near, dim3(nb, nblk(R + 1, per)), dim3(256), lds, h->stream, g, h->d, pb, R,
                           per, hist);
    }
    return hipGetLastError();
}

// ------------------------------------------------------------------ observables
// Radial density profiles of the blob (berechne_dichteprofile,
// observablen_auswertung.cpp:227-330) around the circular-mean centres of
// the species (berechne_mittelpunkte, observablen_auswertung.cpp:140-223).
// Sums use a fixed-order reduction (per-block tree, then one block over the
// block partials in order) and the histograms integer atomics, so the
// result is deterministic.
constexpr int OBS_THREADS = 256;
constexpr int OBS_PER_THREAD = 8;
constexpr int OBS_COPIES = 8;  // copies of a global histogram, added on the host
constexpr size_t OBS_LDS = 48 * 1024;  // largest histogram counted in LDS

// absolute position and species of list position q
__device__ __forceinline__ double2 list_position(const Geo &g, const DevBufs &d, int q, bool &s2) {
    const int c = d.lcell[q], gx = div_nc(c, g), gy = c - gx * g.nc;
    const double2 r = d.lrel[q];
    s2 = d.lpid[q] >= g.n1;
    return make_double2(gx * g.B + r.x, gy * g.B + r.y);
}

// block partial sums of cos/sin(2 pi x / L), cos/sin(2 pi y / L) per species:
// OBS_PER_THREAD positions per thread (bound by the FP64 sincos)
__global__ __launch_bounds__(OBS_THREADS) void k_circ_partial(Geo g, DevBufs d, double *part) {
    __shared__ double sm[OBS_THREADS / 64][8];
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    const double k = 2.0 * M_PI / g.L;
    const int q0 = blockIdx.x * (OBS_THREADS * OBS_PER_THREAD) + threadIdx.x;
    for (int e = 0; e < OBS_PER_THREAD; ++e) {
        const int q = q0 + e * OBS_THREADS;
        if (q >= g.N) break;
        bool s2;
        const double2 x = list_position(g, d, q, s2);
        double cx, sx, cy, sy;
        sincos(x.x * k, &sx, &cx);
        sincos(x.y * k, &sy, &cy);
        v[0] += s2 ? 0.0 : cx;
        v[1] += s2 ? 0.0 : sx;
        v[2] += s2 ? 0.0 : cy;
        v[3] += s2 ? 0.0 : sy;
        v[4] += s2 ? cx : 0.0;
        v[5] += s2 ? sx : 0.0;
        v[6] += s2 ? cy : 0.0;
        v[7] += s2 ? sy : 0.0;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) v[i] += __shfl_xor(v[i], o, 64);
        if ((threadIdx.x & 63) == 0) sm[threadIdx.x >> 6][i] = v[i];
    }
    __syncthreads();
    if (threadIdx.x < 8) {
        double t = 0.0;
        for (int w = 0; w < OBS_THREADS / 64; ++w) t += sm[w][threadIdx.x];
        part[blockIdx.x * 8 + threadIdx.x] = t;
    }
}

// centres S1, S2, Sgamma = (S1+S2)/2 from the block partials (one block):
// thread t adds sum t % 8 of the blocks t / 8, t / 8 + 32, ...
__global__ __launch_bounds__(OBS_THREADS) void k_circ_final(Geo g, const double *part, int nb, double *centers) {
    __shared__ double sm[OBS_THREADS];
    __shared__ double S[4];
    const int t = threadIdx.x;
    double v = 0.0;
    for (int b = t >> 3; b < nb; b += OBS_THREADS / 8) v += part[b * 8 + (t & 7)];
    sm[t] = v;
    __syncthreads();
    if (t < 8) {
        for (int w = 1; w < OBS_THREADS / 8; ++w) v += sm[w * 8 + t];
        sm[t] = v;
    }
    __syncthreads();
    const double k = 2.0 * M_PI / g.L;
    if (t < 4) S[t] = (atan2(-sm[2 * t + 1], -sm[2 * t]) + M_PI) / k;  // (S1x, S1y, S2x, S2y)
    __syncthreads();
    if (t < 6) centers[t] = t < 4 ? S[t] : 0.5 * (S[t - 4] + S[t - 2]);
}

// counts per bin: rho1ring (Sgamma), rho2ring (S2), rho1zen1, rho1zen2,
// rho2zen1, rho2zen2; distances without periodic images, beyond the last
// bin into the last bin (as the reference).  A block counts a contiguous part
// of the list in LDS and adds its non-zero bins to one of OBS_COPIES copies
// of the histogram: 4.0 ms -> 17 us at 2M particles and 256 bins.  (Every
// particle straight into one global histogram is 6M atomics on 1536 counters,
// some 30 ns each where they meet; half of what is left is FP64 square roots
// and divisions.)
// LDS: false where 6 nbins counters exceed OBS_LDS
// (then one copy).
template <bool LDS>
__global__ __launch_bounds__(OBS_THREADS) void k_radial_hist(Geo g, DevBufs d, const double *centers, int nbins,
                                                             double dr, int per, int *hist) {
    extern __shared__ int rhist[];  // [6][nbins]
    int *out = LDS ? hist + (size_t)(blockIdx.x % OBS_COPIES) * 6 * nbins : hist;
    int *h = LDS ? rhist : out;
    if (LDS) {
        for (int b = threadIdx.x; b < 6 * nbins; b += OBS_THREADS) rhist[b] = 0;
        __syncthreads();
    }
    double2 ce[3];  // S1, S2, Sgamma
    for (int i = 0; i < 3; ++i) ce[i] = make_double2(centers[2 * i], centers[2 * i + 1]);
    const int q0 = blockIdx.x * per, q1 = min(q0 + per, g.N);
    for (int q = q0 + threadIdx.x; q < q1; q += OBS_THREADS) {
        bool s2;
        const double2 x = list_position(g, d, q, s2);
        int bin[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double dx = x.x - ce[i].x, dy = x.y - ce[i].y;
            const int b = (int)(sqrt(dx * dx + dy * dy) / dr);
            bin[i] = b < 0 || b >= nbins ? nbins - 1 : b;
        }
        atomicAdd(&h[(s2 ? 1 : 0) * nbins + (s2 ? bin[1] : bin[2])], 1);
        atomicAdd(&h[(s2 ? 4 : 2) * nbins + bin[0]], 1);
        atomicAdd(&h[(s2 ? 5 : 3) * nbins + bin[1]], 1);
    }
    if (!LDS) return;
    __syncthreads();
    for (int b = threadIdx.x; b < 6 * nbins; b += OBS_THREADS)
        if (rhist[b]) atomicAdd(&out[b], rhist[b]);
}

int radial_blocks(const bdk_t *h) { return (int)nblk(h->g.N, OBS_THREADS * OBS_PER_THREAD); }
int radial_copies(int nbins) { return (size_t)6 * nbins * sizeof(int) <= OBS_LDS ? OBS_COPIES : 1; }

hipError_t launch_radial(bdk_t *h, int nbins, double dr, double *part, double *centers, int *hist) {
    const int nb = radial_blocks(h);
    hipLaunchKernelGGL(k_circ_partial, dim3(nb), dim3(OBS_THREADS), 0, h->stream, h->g, h->d, part);
    hipLaunchKernelGGL(k_circ_final, dim3(1), dim3(OBS_THREADS), 0, h->stream, h->g, part, nb, centers);
    hipError_t e = launch_zero_ints(hist, radial_copies(nbins) * 6 * nbins, h->stream);
    if (e != hipSuccess) return e;
    // at most about 4 blocks per compute unit, so that few counters are added
    const int per = std::max(OBS_THREADS * OBS_PER_THREAD, (int)nblk(h->g.N, 1024 * OBS_THREADS) * OBS_THREADS);
    const dim3 grid(nblk(h->g.N, per));
    const size_t lds = (size_t)6 * nbins * sizeof(int);
    if (radial_copies(nbins) > 1)
        hipLaunchKernelGGL(k_radial_hist<true>, grid, dim3(OBS_THREADS), lds, h->stream, h->g, h->d, centers, nbins,
                           dr, per, hist);
    else
        hipLaunchKernelGGL(k_radial_hist<false>, grid, dim3(OBS_THREADS), 0, h->stream, h->g, h->d, centers, nbins,
                           dr, per, hist);
    return hipGetLastError();
}

// ------------------------------------------------------------------ snapshot grid
// Local densities on an m x m grid of width w = L/m (main_auswertung.cpp:
// 214-320): each particle adds its TSC weights times 1/w^2 to the nine cells
// around cell (int)(x/w) mod m of its species' grid.  The weight products are
// summed as 2^-40 fixed point in 64-bit integers, so the grid does not depend
// on the order of the additions.  The offset d from the cell centre uses the
// unwrapped cell index (the reference wraps first, which only differs when
// x/w rounds up to m).
//
// A block owns a tile of ts x ts grid cells and sums both species' weights
// there in LDS: it visits the particles of the list cells around the tile
// (each row of them is one range of the list, two where y wraps) and keeps
// what falls into the tile.  Then it turns its cells into densities and
// counts their statistics at once.  2M particles on 1414^2: 427 -> 62 us,
// against nine global 64-bit atomics per particle, a cleared accumulator and
// a second pass over it.
constexpr double SNAP_SCALE = 1099511627776.0;  // 2^40
constexpr int SNAP_TILE = 32;                   // grid cells per tile side, at most
constexpr int SNAP_CELLS = 48;                  // list cells under a tile's side, about, at most
constexpr int SNAP_SEG = 512;                   // list ranges per round
constexpr int SNAP_COPIES = 8;                  // copies of the counters, added on the host

__device__ __forceinline__ void snap_tsc(double x, double w, int m, int &k, double wt[3]) {
    const int k0 = (int)(x / w);
    k = k0 >= m || k0 <= -m ? k0 % m : k0;
    const double dd = x - (k0 + 0.5) * w;
    wt[1] = 0.75 - dd * dd / (w * w);
    double t = fabs((dd + w) / w);
    wt[0] = 0.5 * (1.5 - t) * (1.5 - t);
    t = fabs((dd - w) / w);
    wt[2] = 0.5 * (1.5 - t) * (1.5 - t);
}

// bin of a histogram value (main_auswertung.cpp:324-375)
__device__ __forceinline__ int snap_bin(double t, int nbins) {
    if (!(t > -1.0)) return 0;  // (int) truncates toward zero; below 0 clamps to 0
    if (t >= (double)nbins) return nbins - 1;
    const int b = (int)t;
    return b < 0 ? 0 : (b >= nbins ? nbins - 1 : b);
}

// one count at sh[i] by every active lane; lanes that share one i (most grid
// cells of a dilute state are empty) count together
__device__ __forceinline__ void snap_count(unsigned int *sh, int i) {
    const int first = __builtin_amdgcn_readfirstlane(i);
    if (__all(i == first)) {
        const unsigned long long act = __ballot(1);
        if ((int)(threadIdx.x & 63) == __ffsll((unsigned long long)act) - 1) atomicAdd(&sh[first], (unsigned)__popcll(act));
    } else {
        atomicAdd(&sh[i], 1u);
    }
}

// list cells that hold every particle which can reach grid cells [p0, p1) of
// an axis: those of x / w in [p0 - 1, p1 + 1), widened by the excursion e of
// offsets outside their cell and a cell of margin
__device__ __forceinline__ void snap_span(int p0, int p1, double w, double e, const Geo &g, int &c0, int &n) {
    const int lo = (int)floor(((p0 - 1) * w - e) / g.B) - 1, hi = (int)floor(((p1 + 1) * w + e) / g.B) + 1;
    n = hi - lo + 1;
    c0 = lo;
    if (n >= g.nc) {
        n = g.nc;
        c0 = 0;
    }
}

struct SnapArgs {
    int m, ts, tiles;  // grid cells per side, per tile side, tiles per side
    double w, drho;
    int stats, nbins;
    double dbin;
    SnapThresh th;
};

__global__ __launch_bounds__(256) void k_snap_tiles(Geo g, DevBufs d, SnapArgs a, double *rho, unsigned int *cnt) {
    extern __shared__ unsigned int sh[];  // [4 * nbins + 7] counts
    __shared__ unsigned long long acc[2 * SNAP_TILE * SNAP_TILE];
    __shared__ int seg_q[SNAP_SEG], seg_pre[SNAP_SEG + 1], wsum[4];
    const int tid = threadIdx.x, nsh = 4 * a.nbins + 7, nc = g.nc, m = a.m;
    if (a.stats)
        for (int i = tid; i < nsh; i += 256) sh[i] = 0u;
    // excursion bound of the current state
    const double e = dbits(d.sc->exc_bits[d.sc->step & 1]) + 1e-9 * g.L;
    const size_t mm = (size_t)m * m;
    for (int tile = blockIdx.x; tile < a.tiles * a.tiles; tile += gridDim.x) {
        const int k0 = (tile / a.tiles) * a.ts, l0 = (tile % a.tiles) * a.ts;
        const int nk = min(a.ts, m - k0), nl = min(a.ts, m - l0), nown = nk * nl;
        __syncthreads();
        for (int i = tid; i < 2 * nown; i += 256) acc[i] = 0ull;
        int cx0, nx, cy0, ny;
        snap_span(k0, k0 + nk, a.w, e, g, cx0, nx);
        snap_span(l0, l0 + nl, a.w, e, g, cy0, ny);
        cx0 = wrapc(cx0, nc);
        cy0 = wrapc(cy0, nc);
        const int parts = cy0 + ny > nc ? 2 : 1;  // a row's y range wraps
        const int nseg = nx * parts;
        for (int s0 = 0; s0 < nseg; s0 += SNAP_SEG) {
            const int ns = min(SNAP_SEG, nseg - s0);
            __syncthreads();
            for (int i = tid; i < ns; i += 256) {
                const int r = (s0 + i) / parts, part = (s0 + i) - r * parts;
                int ux = cx0 + r;
                if (ux >= nc) ux -= nc;
                const int ya = part == 0 ? cy0 : 0, yb = part == 0 ? min(cy0 + ny, nc) : cy0 + ny - nc;
                const int q = d.start[ux * nc + ya];
                seg_q[i] = q;
                seg_pre[i] = max(d.start[ux * nc + yb] - q, 0);
            }
            __syncthreads();
            const int total = block_exscan4(seg_pre, ns, wsum);
            for (int t = tid; t < total; t += 256) {
                int lo = 0, hi = ns - 1;  // last range that begins at or before t
                while (lo < hi) {
                    const int mid = (lo + hi + 1) >> 1;
                    if (seg_pre[mid] <= t) lo = mid;
                    else hi = mid - 1;
                }
                const int q = seg_q[lo] + (t - seg_pre[lo]);
                bool s2;
                const double2 x = list_position(g, d, q, s2);
                int k, l;
                double wx[3], wy[3];
                snap_tsc(x.x, a.w, m, k, wx);
                snap_tsc(x.y, a.w, m, l, wy);
                unsigned long long *p = acc + (s2 ? nown : 0);
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const int kk = wrap1(k - 1 + i, m) - k0;
                    if ((unsigned)kk >= (unsigned)nk) continue;
#pragma unroll
                    for (int j = 0; j < 3; ++j) {
                        const int ll = wrap1(l - 1 + j, m) - l0;
                        if ((unsigned)ll >= (unsigned)nl) continue;
                        const long long v = __double2ll_rn(wx[i] * wy[j] * SNAP_SCALE);
                        atomicAdd(&p[kk * nl + ll], (unsigned long long)v);
                    }
                }
            }
        }
        __syncthreads();
        for (int i = tid; i < nown; i += 256) {
            const double r1 = ((double)acc[i] / SNAP_SCALE) * a.drho;
            const double r2 = ((double)acc[nown + i] / SNAP_SCALE) * a.drho;
            if (rho) {
                const int kk = i / nl;
                const size_t o = (size_t)(k0 + kk) * m + l0 + (i - kk * nl);
                rho[o] = r1;
                rho[mm + o] = r2;
            }
            if (!a.stats) continue;
            const int nbins = a.nbins;
            const double rs = r1 + r2, dr = r1 - r2;
            for (int t = 0; t < 3; ++t)
                if (rs > a.th.rho[t]) snap_count(sh, 4 * nbins + t);
            const double f = rs > 0.0 ? fabs(dr) / rs : 0.0;  // 0/0 passes no threshold
            for (int t = 0; t < 4; ++t)
                if (rs > 0.0 && f > a.th.drho[t]) snap_count(sh, 4 * nbins + 3 + t);
            snap_count(sh, snap_bin(r1 / a.dbin - 0.5, nbins));
            snap_count(sh, nbins + snap_bin(r2 / a.dbin - 0.5, nbins));
            snap_count(sh, 2 * nbins + snap_bin(rs / a.dbin - 0.5, nbins));
            snap_count(sh, 3 * nbins + snap_bin(dr / a.dbin - 0.5 + (double)(nbins / 2), nbins));
        }
    }
    if (!a.stats) return;
    __syncthreads();
    unsigned int *out = cnt + (size_t)(blockIdx.x % SNAP_COPIES) * nsh;
    for (int i = tid; i < nsh; i += 256)
        if (sh[i]) atomicAdd(&out[i], sh[i]);
}

int snap_copies() { return SNAP_COPIES; }

hipError_t launch_snap(bdk_t *h, int m, double *rho, int stats, int nbins, double dbin, SnapThresh th,
                       unsigned int *cnt) {
    SnapArgs a = {};
    a.m = m;
    a.w = h->p.L / m;
    a.drho = 1.0 / (a.w * a.w);
    // a wide grid cell covers many list cells: smaller tiles, so that a coarse
    // grid still spreads over the chip
    a.ts = std::max(1, std::min(SNAP_TILE, (int)std::min(SNAP_CELLS * h->g.B / a.w, 1e6)));
    a.tiles = (int)nblk(m, a.ts);
    a.stats = stats;
    a.nbins = stats ? nbins : 0;
    a.dbin = dbin;
    a.th = th;
    const size_t lds = stats ? (size_t)(4 * nbins + 7) * sizeof(unsigned int) : 0;
    (void)hipFuncSetAttribute((const void *)k_snap_tiles, hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);
    const unsigned grid = (unsigned)std::min((long long)a.tiles * a.tiles, 2048LL);
    hipLaunchKernelGGL(k_snap_tiles, dim3(grid), dim3(256), lds, h->stream, h->g, h->d, a, rho, cnt);
    return hipGetLastError();
}

// ------------------------------------------------------------------ direct rho(k)
// record_ftrho_unkorrigiert (au:307-360): for each wave-vector index pair
// (i, j) the sums over one species of cos and sin(dq (x i + y j)).  For
// species 1 the reference takes y = git_y B + rel_x (au:333), unless the
// parameters ask for rel_y (ftrho_fix); species 2 uses rel_y.
//
// exp(i dq (x i + y j)) is a product of a factor of x and a factor of y, so
// the sums over the particles are one complex product X^T Y of the factors
// of all i and all j, taken by the FP64 matrix units: 2 q sine/cosine pairs
// per particle instead of one per (i, j).  Each angle is reduced to
// [-pi, pi] before the sine and cosine without rounding (i u - 2 rint(i u / 2)
// with u = x dq / pi kept in two doubles), so the sums come out nearer to
// exact arithmetic than with one rounded angle per pair (against extended
// precision: at most 4e-16 of their norm, the other way up to 3e-14).
//
// A block takes a tile of P x P index pairs (P = 32; 16 or 8 for qbins up to
// that) and a part of the list: it queues the species' particles in list order,
// writes both factors of every FtTile::K of them to LDS, and its four waves
// multiply: a 16 x 16 quarter each (P = 32), or every fourth of the particles
// each (P = 16: real and imaginary parts as two products; P = 8: one product
// of [cos | sin] by [cos | sin]), added in order of the waves at the end.  The
// parts are added in order (k_sum_rows).  Bound by the FP64 sine/cosine
// evaluations, 2 P per particle.
// Both species of 2 x 500,000 particles (us a pair of calls): 5 bins 112, 16
// bins 181, 30 bins 375.  With P = 32 for all: 374 throughout; one sine/cosine
// pair per particle and wave vector: 1 bin 176, 5 bins 250, 8 bins 414, 16 bins
// 1236.  2 x 10,000: 47 / 51 / 57, P = 32 for all 55, one pair each 105 to 180.
// (One factor per thread instead of both costs P = 32 a sixth: 438.)
constexpr int FT_THREADS = 256, FT_TILE = 32;
template <int P> struct FtTile {
    static constexpr int K = P == 8 ? 64 : 32;  // particles per round
    // LDS row of one particle's factors: P cosines, P sines, padded to 16 mod 32
    // doubles, so that two consecutive rows' parts read by half a wave lie in
    // different banks
    static constexpr int ROW = P == 32 ? 80 : (P == 16 ? 48 : 16);
};

typedef double ft_acc __attribute__((ext_vector_type(4)));

// cos and sin of (k u) pi, u = uh + ul
__device__ __forceinline__ void ft_factor(int k, double uh, double ul, double *cs, double *sn) {
    const double t = k * uh, te = fma((double)k, uh, -t) + k * ul;
    sincospi((t - 2.0 * rint(0.5 * t)) + te, sn, cs);
}

template <int P>
__global__ __launch_bounds__(FT_THREADS) void k_ftrho(Geo g, DevBufs d, int species, int fix, int qbins, int nt,
                                                      double ch, double cl, int per, double *part) {
    constexpr int K = FtTile<P>::K, ROW = FtTile<P>::ROW, WAVES = FT_THREADS / 64;
    __shared__ double S[2 * K * ROW];
    __shared__ double2 queue[FT_THREADS + K];
    __shared__ int wcnt[WAVES];
    double *X = S, *Y = S + K * ROW;
    const int ti = (int)blockIdx.y / nt, tj = (int)blockIdx.y - ti * nt;
    if (P * P * (ti * ti + tj * tj) > qbins * qbins) return;  // beyond the quarter circle
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wi = (wave >> 1) * 16, wj = (wave & 1) * 16;
    const int q0 = blockIdx.x * per, q1 = min(q0 + per, g.N);
    const double ydrop = species == 1 && !fix ? 1.0 : 0.0;
    ft_acc re = {0.0, 0.0, 0.0, 0.0}, im = {0.0, 0.0, 0.0, 0.0};
    int n = 0;  // queued particles
    for (int base = q0; base < q1; base += FT_THREADS) {
        const int t = base + tid;
        bool want = false;
        double2 x;
        if (t < q1) {
            want = (d.lpid[t] >= g.n1) == (species == 2);
            const int cell = d.lcell[t], gx = div_nc(cell, g), gy = cell - gx * g.nc;
            const double2 r = d.lrel[t];
            x.x = gx * g.B + r.x;
            x.y = gy * g.B + (ydrop != 0.0 ? r.x : r.y);
        }
        const unsigned long long mask = __ballot(want);
        if (lane == 0) wcnt[wave] = __popcll(mask);
        __syncthreads();
        int pos = n + __popcll(mask & ((1ull << lane) - 1ull));
        for (int w = 0; w < WAVES; ++w) {
            if (w < wave) pos += wcnt[w];
            n += wcnt[w];
        }
        if (want) queue[pos] = x;
        __syncthreads();
        int head = 0;
        const bool last = base + FT_THREADS >= q1;
        while (n - head >= K || (last && n > head)) {
            const int m = min(K, n - head);
            if constexpr (P == 32) {
                // both factors: index tid % 32, particles tid / 32 + 8 e
                for (int e = 0; e < K / 8; ++e) {
                    const int i = tid & 31, k = (tid >> 5) + 8 * e;
                    double cx = 0.0, sx = 0.0, cy = 0.0, sy = 0.0;
                    if (k < m) {
                        const double2 p = queue[head + k];
                        const double ux = p.x * ch, uy = p.y * ch;
                        ft_factor(P * ti + i, ux, fma(p.x, ch, -ux) + p.x * cl, &cx, &sx);
                        ft_factor(P * tj + i, uy, fma(p.y, ch, -uy) + p.y * cl, &cy, &sy);
                    }
                    X[k * ROW + i] = cx;
                    X[k * ROW + P + i] = sx;
                    Y[k * ROW + i] = cy;
                    Y[k * ROW + P + i] = sy;
                }
            } else {
                // one factor: of x by the first P of 2 P threads, of y by the others
                const int i = tid & (P - 1), iy = (tid / P) & 1;
                double *row = (iy ? Y : X) + i;
                for (int k = tid / (2 * P); k < K; k += FT_THREADS / (2 * P)) {
                    double c = 0.0, s = 0.0;
                    if (k < m) {
                        const double2 p = queue[head + k];
                        const double v = iy ? p.y : p.x, u = v * ch;
                        ft_factor(i, u, fma(v, ch, -u) + v * cl, &c, &s);
                    }
                    row[k * ROW] = c;
                    row[k * ROW + P] = s;
                }
            }
            __syncthreads();
            // operands: row (column) lane % 16 of particle k + lane / 16
            if constexpr (P == 32) {
#pragma unroll
                for (int k = 0; k < K; k += 4) {
                    const int o = (k + (lane >> 4)) * ROW + (lane & 15);
                    const double xc = X[o + wi], xs = X[o + wi + P], yc = Y[o + wj], ys = Y[o + wj + P];
                    re = __builtin_amdgcn_mfma_f64_16x16x4f64(xc, yc, re, 0, 0, 0);
                    re = __builtin_amdgcn_mfma_f64_16x16x4f64(-xs, ys, re, 0, 0, 0);
                    im = __builtin_amdgcn_mfma_f64_16x16x4f64(xs, yc, im, 0, 0, 0);
                    im = __builtin_amdgcn_mfma_f64_16x16x4f64(xc, ys, im, 0, 0, 0);
                }
            } else {
#pragma unroll
                for (int k = 4 * wave; k < K; k += 4 * WAVES) {
                    const int o = (k + (lane >> 4)) * ROW + (lane & 15);
                    if constexpr (P == 16) {
                        const double xc = X[o], xs = X[o + P], yc = Y[o], ys = Y[o + P];
                        re = __builtin_amdgcn_mfma_f64_16x16x4f64(xc, yc, re, 0, 0, 0);
                        re = __builtin_amdgcn_mfma_f64_16x16x4f64(-xs, ys, re, 0, 0, 0);
                        im = __builtin_amdgcn_mfma_f64_16x16x4f64(xs, yc, im, 0, 0, 0);
                        im = __builtin_amdgcn_mfma_f64_16x16x4f64(xc, ys, im, 0, 0, 0);
                    } else {
                        re = __builtin_amdgcn_mfma_f64_16x16x4f64(X[o], Y[o], re, 0, 0, 0);
                    }
                }
            }
            __syncthreads();
            head += m;
        }
        // what is left (fewer than K) moves to the front
        n -= head;
        double2 keep;
        if (tid < n) keep = queue[head + tid];
        __syncthreads();
        if (tid < n) queue[tid] = keep;
    }
    // results: column lane % 16, rows lane / 16 + 4 r
    const int qp = P * nt;
    double *out = part + (size_t)blockIdx.x * 2 * qp * qp;
    if constexpr (P == 32) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const size_t o = (size_t)(P * ti + wi + (lane >> 4) + 4 * r) * qp + P * tj + wj + (lane & 15);
            out[o] = re[r];
            out[(size_t)qp * qp + o] = im[r];
        }
    } else {
        constexpr int TILE = P == 16 ? 512 : 256;  // values of a wave
        static_assert(WAVES * TILE <= 2 * K * ROW, "the waves' sums lie where the factors were");
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int o = wave * TILE + ((lane >> 4) + 4 * r) * 16 + (lane & 15);
            S[o] = re[r];
            if (P == 16) S[o + 256] = im[r];
        }
        __syncthreads();
        auto sum = [&](int o) { return ((S[o] + S[o + TILE]) + S[o + 2 * TILE]) + S[o + 3 * TILE]; };
        if (P == 16) {
            out[tid] = sum(tid);
            out[256 + tid] = sum(256 + tid);
        } else if (tid < 64) {
            const int o = (tid >> 3) * 16 + (tid & 7);
            out[tid] = sum(o) - sum(o + 8 * 16 + 8);
            out[64 + tid] = sum(o + 8 * 16) + sum(o + 8);
        }
    }
}

// the tile's side: one tile of 8 or 16 where that holds all indices, so that a
// few wave vectors do not pay for 32 factors per axis; parts of the list (a
// multiple of 64 positions each) such that about 1024 blocks run, 512 of a
// small tile (5 / 16 bins, 2 x 500,000 and 2 x 100,000 particles, us: 256 parts
// 132 / 223, 62 / 82; 512 111 / 182, 61 / 78; 1024 112 / 178, 68 / 86); side of
// the padded square of index pairs
FtPlan ftrho_plan(const bdk_t *h, int qbins) {
    FtPlan f;
    const int tile = qbins <= 8 ? 8 : (qbins <= 16 ? 16 : FT_TILE), nt = (int)nblk(qbins, tile);
    f.side = tile * nt;
    const int want = tile < FT_TILE ? 512 : std::max(1, std::min(256, 1024 / (nt * nt)));
    f.per = (int)nblk(nblk(h->g.N, want), 64) * 64;
    f.parts = (int)nblk(h->g.N, f.per);
    return f;
}

// sums of the species: out[2][side][side] = cos and sin sums of (i, j); part
// [parts][2][side][side].  Entries outside the quarter circle hold nothing.
hipError_t launch_ftrho(bdk_t *h, const FtPlan &f, int qbins, int species, double dq, double *part, double *out) {
    const long double c = (long double)dq / 3.14159265358979323846264338327950288L;
    const double ch = (double)c, cl = (double)(c - (long double)ch);
    auto go = [&](auto tile) {
        constexpr int P = decltype(tile)::value;
        const int nt = f.side / P;
        hipLaunchKernelGGL(k_ftrho<P>, dim3(f.parts, nt * nt), dim3(FT_THREADS), 0, h->stream, h->g, h->d, species,
                           h->p.ftrho_fix ? 1 : 0, qbins, nt, ch, cl, f.per, part);
    };
    if (f.side == 8)
        go(std::integral_constant<int, 8>());
    else if (f.side == 16)
        go(std::integral_constant<int, 16>());
    else
        go(std::integral_constant<int, FT_TILE>());
    launch_sum_rows(part, f.parts, 2 * f.side * f.side, out, h->stream);
    return hipGetLastError();
}

}  // namespace bdkx
