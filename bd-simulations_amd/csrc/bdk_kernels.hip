// HIP kernels of the MI355X Brownian-dynamics timestep (gfx950).
//
// One step (dynamik_methoden.cpp:74-163) starts from a state whose forces
// are on the device and leaves the next state with its forces:
//   k_update    gather (gr:81-668), noise (dm:1317-1339), Euler step
//               (dm:116-157), refresh (dm:216-325); the cell counts are
//               updated by the particles that change cell;
// then on two streams side by side:
//   k_scan      exclusive scan of the cell counts (the update ranked the
//               particles that stay in their cell, without atomics);
//   k_fill      cell list = slots grouped by cell, species in bit 31, and
//               the particle state in list order (lcell, lrel, lpid, lrelf);
//   k_sort_cells  the arrivals of each cell in slot order;
//   k_wca       WCA forces (dm:617-1059) of the new lists;
// and
//   k_deposit   charge deposit (gr:31-547) per tile of cells into the tile's
//               own mesh points, integer LDS accumulation, here from the
//               slot arrays (grouped by the previous cells);
//   k_r2c_rows  row FFTs of the real mesh, transposed half-spectrum out;
//   k_col       column FFT, Green's function x gradient (dm:1210-1216), two
//               inverse column FFTs (Fx, Fy);
//   k_c2r_rows  inverse row FFT of (Fx + i Fy) -> real Fx, Fy mesh
//               (the three passes: bdk_fft.hip).
// Every force, gather and update kernel runs over list positions q and
// reads the list-ordered state; k_update writes the new state to slot q.
// The slots are therefore re-sorted by cell every step: consecutive threads
// handle particles of neighbouring cells for the whole run.
// With a finite max_travel, k_gather (forces and the dt candidates,
// dm:1420-1491) runs before a non-fused k_update, which reduces them.
//
// Position arithmetic (x = git*B + rel, mesh indices, weights, refresh) is
// compiled without FP contraction so it rounds like the reference's x86-64
// build; cell indices are therefore bit-exact.
#pragma clang fp contract(off)

#include <mutex>

#include "bdk_device.hpp"
#include "bdk_fft.hpp"
#include "bdk_particles.hpp"

namespace bdkx {

__device__ int first_owned(int c, const Geo &g) {
    if (c <= 0) return 0;
    if (c >= g.nc) return g.Z;
    int k = (int)ceil(c * g.B / g.h - 0.5);
    if (k < 0) k = 0;
    if (k > g.Z) k = g.Z;
    auto owner = [&](int kk) { return (int)floor(((kk + 0.5) * g.h) / g.B); };
    while (k > 0 && owner(k - 1) >= c) --k;
    while (k < g.Z && owner(k) < c) ++k;
    return k;
}

__global__ void k_own(Geo g, int *own) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c <= g.nc) own[c] = first_owned(c, g);
}

template <typename R>
__global__ __launch_bounds__(256) void k_wca(Geo g, DevBufs d) {
    wca_ref_body<R>(g, d, xcd_block(g.xcd));
}

constexpr int WCA64_BLOCK = 256, WCA64_PER = WCA64_BLOCK / WCA_LANES;  // particles per block
__global__ __launch_bounds__(WCA64_BLOCK) void k_wca_f64(Geo g, DevBufs d) {
    const int first = xcd_block(g.xcd) * WCA64_PER;
    wca_f64_body(g, d, first, min(WCA64_PER, g.N - first));
}

template <bool UNIT>
__global__ __launch_bounds__(256) void k_wca_f32(Geo g, DevBufs d) {
    __shared__ float2 sp[WCA_STAGE + 1];
    __shared__ unsigned se[UNIT ? 1 : WCA_STAGE + 1];
    __shared__ int hdr[8];
    wca_f32_body<UNIT>(g, d, xcd_block(g.xcd), sp, se, hdr);
}

// hardware block order: measured faster than per-XCD ranges for this kernel
// P2: the mesh kind (chosen by the launcher; one body per kernel keeps the
// scalar registers of the power-of-two path as they were)
template <typename R, int SCHEME, bool P2>
__global__ __launch_bounds__(DP_THREADS) void k_deposit(Geo g, DevBufs d, DepArgs a) {
    deposit_body<R, SCHEME, P2>(g, d, a, blockIdx.x);
}

// per-step scalar re-arm when no deposit runs (ideal-gas runs), at the start
// of the step; one wave
__global__ void k_rearm(Geo g, DevBufs d) {
    d.dts[threadIdx.x * 16] = ~0ull;
    if (threadIdx.x == 0) {
        const unsigned long long step = d.sc->step;
        d.sc->dt_bits = bitsd(g.dt_max);
        d.sc->exc_bits[(step + 1) & 1] = 0ull;
    }
}

// ------------------------------------------------------------------ gather, update
template <typename R, int SCHEME, bool P2>
__device__ __forceinline__ void gather_kap(double x, double y, bool s2, const typename V2<R>::T *__restrict__ fm,
                                           const Geo &g, double &fx, double &fy) {
    using R2 = typename V2<R>::T;
    const int Z = g.Z;
    int k, l;
    R wx[3], wy[3];
    weights_r<R, SCHEME>(x, g, k, wx);
    weights_r<R, SCHEME>(y, g, l, wy);
    foldz<P2>(k, l, Z);
    if (SCHEME == 0) {
        R2 f = fm[(size_t)k * Z + l];
        if (!s2) {
            fx = (double)f.x;
            fy = (double)f.y;
        } else {
            fx = (double)((R)g.f2_f1 * f.x);
            // gr:123 reads Fx[..][1], the imaginary part of the x force (zero
            // up to rounding); ngp_fix reads Fy
            fy = g.ngp_fix ? (double)((R)g.f2_f1 * f.y) : 0.0;
        }
        return;
    }
    const int kx[3] = {wrapz<P2>(k - 1, Z), k, wrapz<P2>(k + 1, Z)};
    const int ly[3] = {wrapz<P2>(l - 1, Z), l, wrapz<P2>(l + 1, Z)};
    R ax = 0, ay = 0;
    // weighted sums of the mesh forces with explicit fused multiply-adds
    // (the weights and indices above follow the reference's rounding)
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const R2 *row = fm + (size_t)kx[a] * Z;
        R2 f0 = row[ly[0]], f1 = row[ly[1]], f2 = row[ly[2]];
        const R sx = fma(wy[2], f2.x, fma(wy[1], f1.x, wy[0] * f0.x));
        const R sy = fma(wy[2], f2.y, fma(wy[1], f1.y, wy[0] * f0.y));
        if (a == 0) {
            ax = wx[0] * sx;
            ay = wx[0] * sy;
        } else {
            ax = fma(wx[a], sx, ax);
            ay = fma(wx[a], sy, ay);
        }
    }
    if (s2) {
        ax *= (R)g.f2_f1;
        ay *= (R)g.f2_f1;
    }
    fx = (double)ax;
    fy = (double)ay;
}

__device__ __forceinline__ double dt_candidate(double F, double n, const Geo &g) {
    if (fabs(F) < 1.0e-5) return g.mrd * g.mrd / (2.0 * g.T * n * n);
    double u = n * sqrt(0.5 * g.T) / F;
    double w = sqrt(u * u + g.mrd / fabs(F));
    return (w - fabs(u)) * (w - fabs(u));
}

__device__ __forceinline__ double2 particle_noise(const Geo &g, const DevBufs &d, int pid, unsigned long long step) {
    double2 n;
    if (g.nowca) {
        n.x = 0.0;
        n.y = 0.0;
    } else if (g.noise_mode == BDK_NOISE_UPLOAD) {
        n = d.noise_up[pid];
    } else if (g.f32noise) {
        n = philox_noise_f32(g.seed, (uint32_t)pid, step, g.noise_mode == BDK_NOISE_GAUSS, g.noise_var);
    } else {
        n = philox_noise(g.seed, (uint32_t)pid, step, g.noise_mode == BDK_NOISE_GAUSS, g.noise_var);
    }
    return n;
}

// forces only: fkap (and dt candidates when with_dt) of block blk of list
// positions; the block minimum of the candidates goes to dts slot `slot`
template <typename R, int SCHEME, bool P2>
__device__ __forceinline__ void gather_body(const Geo &g, const DevBufs &d, int with_dt, int blk, int slot) {
    using R2 = typename V2<R>::T;
    const int s = blk * blockDim.x + threadIdx.x;  // list position
    double cand = INFINITY;
    if (s < g.N) {
        const int c = d.lcell[s];
        const int gx = div_nc(c, g), gy = c - gx * g.nc;
        const double2 r = d.lrel[s];
        const int pid = d.lpid[s];
        // the WCA force and the noise before the mesh gather: their loads
        // overlap the gather's instead of waiting behind the fkap store
        R2 fw;
        double2 n;
        if (with_dt) {
            fw = ((const R2 *)d.fwca)[s];
            n = particle_noise(g, d, pid, d.sc->step);
        }
        double fx = 0.0, fy = 0.0;
        if (!g.idgas) gather_kap<R, SCHEME, P2>(gx * g.B + r.x, gy * g.B + r.y, pid >= g.n1, (const R2 *)d.fmesh, g, fx, fy);
        R2 o;
        o.x = (R)fx;
        o.y = (R)fy;
        ((R2 *)d.fkap)[s] = o;
        if (with_dt) {
            double c0 = dt_candidate((double)fw.x + (double)o.x, n.x, g);
            double c1 = dt_candidate((double)fw.y + (double)o.y, n.y, g);
            if (c0 < cand) cand = c0;
            if (c1 < cand) cand = c1;
        }
    }
    if (with_dt) {
        // NaN candidates never win (std::min semantics of dm:1420-1491).
        // Minimum over the block, then one atomicMin into one of 64 slots
        // (128 bytes apart), skipped when the slot already holds less.
        __shared__ double wmin[4];
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            double v = __shfl_xor(cand, o, 64);
            if (v < cand) cand = v;
        }
        if ((threadIdx.x & 63) == 0) wmin[threadIdx.x >> 6] = cand;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int w = 1; w < (int)(blockDim.x >> 6); ++w)
                if (wmin[w] < cand) cand = wmin[w];
            if (cand < INFINITY && cand >= 0.0) {
                unsigned long long *sp = &d.dts[(slot & 63) * 16];
                const unsigned long long b = bitsd(cand);
                if (b < *(volatile unsigned long long *)sp) atomicMin(sp, b);
            }
        }
    }
}

template <typename R, int SCHEME, bool P2>
__global__ __launch_bounds__(256) void k_gather(Geo g, DevBufs d, int with_dt) {
    gather_body<R, SCHEME, P2>(g, d, with_dt, xcd_block(g.xcd), blockIdx.x);
}

// dt for bdk_optimal_dt (the step's update reduces the slots itself):
// dt_max and the 64 slot minima of k_gather folded into
// sc->dt_bits and logged by step; the slots are re-armed (all ones) for the
// next reduction.  One wave.
__device__ __forceinline__ void dt_fold_body(const Geo &g, const DevBufs &d) {
    const int t = threadIdx.x;
    unsigned long long m = d.dts[t * 16];
    d.dts[t * 16] = ~0ull;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const unsigned long long v = __shfl_xor(m, o, 64);
        if (v < m) m = v;
    }
    if (t == 0) {
        const unsigned long long dm = bitsd(g.dt_max);
        const unsigned long long dt = m < dm ? m : dm;
        d.sc->dt_bits = dt;
        d.dtlog[d.sc->step & (kDtLog - 1)] = dbits(dt);
    }
}

__global__ __launch_bounds__(64) void k_dt_fold(Geo g, DevBufs d) { dt_fold_body(g, d); }

// fmod(y, B) for the refresh's y = rel + B (dm:249-250): for |y| < 2B the
// quotient is 0 or 1 and the remainder y or y - B, which is exact (y and B
// within a factor of two); larger moves take fmod itself.  Equal to fmod
// bit for bit everywhere (IEEE fmod is exact too).
__device__ __forceinline__ double fmod_cell(double y, double B) {
    if (y >= 0.0 && y < B) return y;
    if (y >= B && y < 2.0 * B) return y - B;
    if (y > -B && y < 0.0) return y;
    return fmod(y, B);
}

// Euler step (dm:116-157) + refresh (dm:216-325) + cell counting of list
// position s (written to slot s).  Returns how far the stored new position
// (cell and offset) lies outside the particle's previous cell (<= 0 inside).
// FUSED: capillary force gathered here (fixed dt); else read from fkap.
// cell: the particle's previous cell if it stays there, else -1 - that cell.
template <typename R, int SCHEME, bool FUSED, bool P2>
__device__ __forceinline__ double update_one(const Geo &g, const DevBufs &d, int s, double dt, int &cell) {
    using R2 = typename V2<R>::T;
    const unsigned long long step = d.sc->step;
    const int c = d.lcell[s];
    int gx = div_nc(c, g), gy = c - gx * g.nc;
    double2 r = d.lrel[s];
    const int pid = d.lpid[s];
    const bool s2 = pid >= g.n1;
    double fwx = 0.0, fwy = 0.0, fkx = 0.0, fky = 0.0;
    if (!g.idgas) {
        const R2 fw = ((const R2 *)d.fwca)[s];
        fwx = (double)fw.x;
        fwy = (double)fw.y;
        if (FUSED) {
            gather_kap<R, SCHEME, P2>(gx * g.B + r.x, gy * g.B + r.y, s2, (const R2 *)d.fmesh, g, fkx, fky);
        } else {
            const R2 fk = ((const R2 *)d.fkap)[s];
            fkx = (double)fk.x;
            fky = (double)fk.y;
        }
    }
    const double2 n = particle_noise(g, d, pid, step);
    const double sq = g.adaptive ? sqrt(2.0 * g.T * dt) : g.sq_fixed;  // same expression, correctly rounded
    const double dx = dt * (fwx + fkx) + sq * n.x;
    const double dy = dt * (fwy + fky) + sq * n.y;
    double2 rn;
    float2 kc = make_float2(0.f, 0.f);  // Kahan compensation (pos_mode 2)
    if (g.pos_mode == 0) {
        rn.x = r.x + dx;
        rn.y = r.y + dy;
    } else {
        // FP32 in-cell positions: the increment rounded to FP32 and added in
        // FP32 (pos_mode 2: Kahan summation, c = (t - r) - y carries the
        // low-order part lost by the addition into the next step)
        const float rx = (float)r.x, ry = (float)r.y;
        if (g.pos_mode == 1) {
            rn.x = (double)(rx + (float)dx);
            rn.y = (double)(ry + (float)dy);
        } else {
            const float2 c = d.lcomp[s];
            const float yx = (float)dx - c.x, yy = (float)dy - c.y;
            const float tx = rx + yx, ty = ry + yy;
            kc.x = (tx - rx) - yx;
            kc.y = (ty - ry) - yy;
            rn.x = (double)tx;
            rn.y = (double)ty;
        }
    }
    if (s2 && g.restrict_radial) {  // dm:138-155
        const double mitte = 0.5 * g.L;
        const int i2 = pid - g.n1;
        double x = gx * g.B + rn.x, y = gy * g.B + rn.y;
        double dxm = mitte - x, dym = mitte - y;
        double abst = sqrt(dxm * dxm + dym * dym);
        double xs = mitte + abst * cos(2 * M_PI * (int)i2 / g.n2);
        double ys = mitte + abst * sin(2 * M_PI * (int)i2 / g.n2);
        rn.x += (xs - x);
        rn.y += (ys - y);
    }
    const double B = g.B;
    int nc_new = c;
    const bool finite = fabs(rn.x) < 1e9 && fabs(rn.y) < 1e9;
    if (!finite) {
        // non-finite or runaway position: keep the old state, raise the flag
        atomicOr(&d.sc->nonfinite, 1);
        rn = r;
    }
    // the stored new position (cell, offset) relative to the previous cell's
    // corner: the bound the deposit beside the rebuild stages by
    double ox = rn.x, oy = rn.y;
    if (finite && (rn.x < 0.0 || rn.x > B || rn.y < 0.0 || rn.y > B)) {
        const int ic0 = (int)floor((gx * B + rn.x) / B);
        const int jc0 = (int)floor((gy * B + rn.y) / B);
        const int ic = wrapc(ic0 + g.nc, g.nc);
        const int jc = wrapc(jc0 + g.nc, g.nc);
        rn.x = fmod_cell(rn.x + B, B);
        rn.y = fmod_cell(rn.y + B, B);
        // a move of more than one cell downwards keeps a negative offset
        // (fmod takes the sign of rel + B, dm:216-325): the stored position
        // then lies one cell below the moved one, so the bound follows the
        // stored cell and offset
        ox = (ic0 - gx) * B + rn.x;
        oy = (jc0 - gy) * B + rn.y;
        gx = ic;
        gy = jc;
        nc_new = gx * g.nc + gy;
        if (g.pos_mode) {
            // back to FP32 storage; the rounding of the shifted value joins
            // the compensation (the position is t - c)
            const float wx = (float)rn.x, wy = (float)rn.y;
            kc.x += (float)((double)wx - rn.x);
            kc.y += (float)((double)wy - rn.y);
            ox += (double)wx - rn.x;
            oy += (double)wy - rn.y;
            rn.x = (double)wx;
            rn.y = (double)wy;
        }
    }
    const double ex_prev = fmax(fmax(-ox, ox - B), fmax(-oy, oy - B));
    d.cell[s] = nc_new;
    d.rel[s] = rn;
    d.pid[s] = pid;
    if (g.pos_mode == 2) d.comp[s] = kc;
    if (nc_new != c) {
        // a cell change (a few percent of the particles per step): the
        // counts follow, and the rank among the new cell's arrivals comes
        // from arr; particles that stay are ranked without atomics
        atomicSub(&d.count[c], 1);
        atomicAdd(&d.count[nc_new], 1);
        if ((c >> SCAN_SHIFT) != (nc_new >> SCAN_SHIFT)) {
            atomicSub(&d.bcount[(c >> SCAN_SHIFT) * BCOUNT_STRIDE], 1);
            atomicAdd(&d.bcount[(nc_new >> SCAN_SHIFT) * BCOUNT_STRIDE], 1);
        }
        d.rank[s] = RANK_MOVED | atomicAdd(&d.arr[nc_new], 1);
    }
    cell = nc_new == c ? c : -1 - c;
    double ex = fmax(fmax(-rn.x, rn.x - B), fmax(-rn.y, rn.y - B));
    if (ex > 0.0) atomicMax(&d.sc->exc_bits[(step + 1) & 1], bitsd(ex));
    if (s == 0) d.sc->dt_last = bitsd(dt);
    return ex_prev;
}

// The update of one block of list positions.  The largest distance of a new
// position outside its previous cell bounds where the next deposit finds the
// particles when it stages them by their previous cells (during the list
// rebuild): reduced per wave, then one atomicMax per wave into one of 64
// slots (128 bytes apart), skipped when the slot already holds as much.
template <typename R, int SCHEME, bool FUSED, bool P2>
__device__ __forceinline__ void update_body(const Geo &g, const DevBufs &d, int blk) {
    const int s = blk * blockDim.x + threadIdx.x;  // list position in, slot out
    // the starts that group the slot arrays after this update (the previous
    // list order), kept for the deposit beside the rebuild
    const int stride = ((g.N + blockDim.x - 1) / blockDim.x) * blockDim.x;
    for (int c = s; c <= g.ncell; c += stride) d.start_old[c] = d.start[c];
    double dt = g.dt_max;
    if (!FUSED && g.adaptive) {
        // the step's dt (dm:1420-1491): dt_max and the 64 slot minima of the
        // candidates from k_gather (all ones = none), reduced by every wave;
        // the step's last mesh pass re-arms the slots (k_rearm at the start
        // of the step when no mesh pass runs)
        unsigned long long mm = d.dts[(threadIdx.x & 63) * 16];
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) {
            const unsigned long long v = __shfl_xor(mm, o, 64);
            if (v < mm) mm = v;
        }
        const unsigned long long dm = bitsd(g.dt_max);
        dt = dbits(mm < dm ? mm : dm);
        if (blk == 0 && threadIdx.x == 0) {
            d.sc->dt_bits = bitsd(dt);
            d.dtlog[d.sc->step & (kDtLog - 1)] = dt;
            if (d.hdt) __hip_atomic_store(d.hdt, dt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    double m = 0.0;
    int cell = -1 - g.ncell;  // (no particle: a cell of its own, not a stayer)
    if (s < g.N) m = update_one<R, SCHEME, FUSED, P2>(g, d, s, dt, cell);
    // Rank of a particle that stays: the stayers of its cell before it.  A
    // wave holds 64 consecutive list positions, so the cell's entries are
    // neighbouring lanes; the fill adds the stayers before the wave for the
    // wave's first cell.  (A pass of its own that compared the cells of each
    // particle's predecessors took 16 us at 2M particles.)
    {
        const int lane = threadIdx.x & 63, c = cell >= 0 ? cell : -1 - cell;
        const int prev = __shfl_up(c, 1, 64);
        const unsigned long long heads = __ballot(lane == 0 || prev != c), stay = __ballot(cell >= 0);
        const unsigned long long upto = ~0ull >> (63 - lane);
        const int first = 63 - __clzll((long long)(heads & upto));  // the cell's first lane
        const int r = __popcll(stay & (upto >> 1) & (~0ull << first));
        if (cell >= 0) d.rank[s] = first == 0 ? r | RANK_OPEN : r;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0 && m > 0.0) {
        unsigned long long *slot = &d.exo[((s >> 6) & 63) * 16];
        const unsigned long long b = bitsd(m);
        if (b > *(volatile unsigned long long *)slot) atomicMax(slot, b);
    }
}

// (without the fused gather the mesh kind plays no part: P2 = true).
// 128-thread blocks: measured a little faster than 256 (and 512 slower).
template <typename R, int SCHEME, bool FUSED, bool P2>
__global__ __launch_bounds__(128) void k_update(Geo g, DevBufs d) {
    update_body<R, SCHEME, FUSED, P2>(g, d, xcd_block(g.xcd));
}

// refresh (dm:216-325) without motion + counting; used by bdk_refresh
__global__ void k_refresh(Geo g, DevBufs d) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.N) return;
    const int c = d.cell[s];
    int gx = c / g.nc, gy = c - gx * g.nc;
    double2 rn = d.rel[s];
    const double B = g.B;
    int nc_new = c;
    if (!(fabs(rn.x) < 1e9 && fabs(rn.y) < 1e9)) {
        atomicOr(&d.sc->nonfinite, 1);
    } else if (rn.x < 0.0 || rn.x > B || rn.y < 0.0 || rn.y > B) {
        int ic = (int)floor((gx * B + rn.x) / B);
        int jc = (int)floor((gy * B + rn.y) / B);
        ic = wrapc(ic + g.nc, g.nc);
        jc = wrapc(jc + g.nc, g.nc);
        rn.x = fmod(rn.x + B, B);
        rn.y = fmod(rn.y + B, B);
        nc_new = ic * g.nc + jc;
    }
    d.cell[s] = nc_new;
    d.rel[s] = rn;
    d.rank[s] = atomicAdd(&d.count[nc_new], 1);
    double ex = fmax(fmax(-rn.x, rn.x - B), fmax(-rn.y, rn.y - B));
    if (ex > 0.0) atomicMax(&d.sc->exc_bits[d.sc->step & 1], bitsd(ex));
}

// counting: rank and excursion of a particle in slot s
__device__ __forceinline__ void bin_slot(const Geo &g, const DevBufs &d, int s, int c, double2 rn) {
    d.rank[s] = atomicAdd(&d.count[c], 1);
    const double B = g.B;
    double ex = fmax(fmax(-rn.x, rn.x - B), fmax(-rn.y, rn.y - B));
    if (ex > 0.0) atomicMax(&d.sc->exc_bits[d.sc->step & 1], bitsd(ex));
}

// counting only (after a state's load)
__global__ void k_bin(Geo g, DevBufs d) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < g.N) bin_slot(g, d, s, d.cell[s], d.rel[s]);
}

// A new state: cells and offsets by id (device memory, or the pinned staging
// read over the bus) into the slots of the same number, counted on the way.
// The flags and counters start cleared (k_place_clear).
__global__ __launch_bounds__(256) void k_place(Geo g, DevBufs d, const int2 *__restrict__ git,
                                               const double2 *__restrict__ rel) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= g.N) return;
    const int2 gi = git[s];
    double2 r = rel[s];
    if (g.pos_mode) r = make_double2((double)(float)r.x, (double)(float)r.y);  // FP32 storage of the in-cell positions
    const int c = gi.x * g.nc + gi.y;
    d.cell[s] = c;
    d.pid[s] = s;
    d.rel[s] = r;
    if (d.comp) d.comp[s] = make_float2(0.f, 0.f);
    bin_slot(g, d, s, c, r);
}

__global__ __launch_bounds__(256) void k_place_clear(int *count, int ncell, DevScalars *sc) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < ncell) count[i] = 0;
    if (i == 0) {
        sc->exc_bits[sc->step & 1] = 0ull;
        sc->nonfinite = 0;  // the flags describe a run from the state before
    }
}

// clears the excursion slot that k_bin / k_refresh fill
__global__ void k_reset_exc(DevScalars *sc) { sc->exc_bits[sc->step & 1] = 0ull; }

// noise of the next step, by particle id (bdk_get_noise)
__global__ void k_noise_out(Geo g, DevBufs d) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= g.N) return;
    d.noise_out[p] = particle_noise(g, d, p, d.sc->step);
}

// Cells and offsets of one species (ids id0 .. id0 + n - 1) in id order, for
// the host, and the error flags (null: not wanted): the scatter by id that a
// host thread would do over the whole state runs here (a random 24 B write
// per particle; 20 us at 2M particles against 15 ms), and only the species
// asked for crosses to the host.
__global__ void k_by_id(Geo g, DevBufs d, int id0, int n, ByIdHead *head, int2 *git, double2 *rel) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s == 0 && head) head->flags = d.sc->nonfinite;
    if (s >= g.N) return;
    const int i = d.pid[s] - id0;
    if ((unsigned)i >= (unsigned)n) return;
    const int c = d.cell[s], gx = div_nc(c, g);
    if (git) git[i] = make_int2(gx, c - gx * g.nc);
    if (rel) rel[i] = d.rel[s];
}

// n 16-byte words into pinned host memory, a wave's 1 KB per store; bound by
// the bus (2.7 MB: 60 us, 46 GB/s)
__global__ __launch_bounds__(256) void k_to_host(const uint4 *__restrict__ src, uint4 *__restrict__ dst, int n) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) dst[i] = src[i];
}

// list-ordered forces as doubles in id order
template <typename R>
__global__ void k_force_by_id(Geo g, DevBufs d, const typename V2<R>::T *__restrict__ f, double2 *out) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= g.N) return;
    out[d.lpid[q]] = make_double2((double)f[q].x, (double)f[q].y);
}

// ------------------------------------------------------------------ scan + fill
// Full recount of bcount from the cell counts (after an upload or a
// refresh; during steps the update keeps bcount current).
__device__ __forceinline__ void scan_reduce_body(const int *__restrict__ count, int ncell, int *__restrict__ bcount,
                                                 int blk) {
    __shared__ int ws[SCAN_THREADS / 64];
    const int base = blk * SCAN_BLOCK;
    int s = 0;
    for (int q = threadIdx.x; q < SCAN_BLOCK; q += SCAN_THREADS) {
        int i = base + q;
        if (i < ncell) s += count[i];
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        int t = 0;
        for (int w = 0; w < SCAN_THREADS / 64; ++w) t += ws[w];
        bcount[blk * BCOUNT_STRIDE] = t;
    }
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_reduce(const int *__restrict__ count, int ncell,
                                                              int *__restrict__ bcount) {
    scan_reduce_body(count, ncell, bcount, blockIdx.x);
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan(const int *__restrict__ count, const int *__restrict__ bcount,
                                                       int *__restrict__ start, int ncell, int nb, int nmax,
                                                       DevScalars *sc, int inc_step) {
    scan_body(count, bcount, start, ncell, nb, nmax, sc, inc_step, blockIdx.x);
}

__global__ void k_fill(Geo g, DevBufs d, int moved_ranks) { fill_body(g, d, moved_ranks, blockIdx.x); }

__global__ void k_zero_int(int *p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void k_sort_cells(Geo g, DevBufs d, int moved_ranks) { sort_cells_body(g, d, moved_ranks, blockIdx.x); }


// ------------------------------------------------------------------ batches
// A batch advances many independent simulations (members) with one launch
// per stage.  A batched kernel maps its block through the stage's table to
// (member, block of that member) and runs the same device body as the
// single-simulation kernel on that member's geometry and buffers, so every
// member's results are bit-identical alone and in a batch.

template <typename R, bool P>
__global__ __launch_bounds__(512) void kb_wca(const RepDev *m, const int2 *map, int nmap) {
    constexpr int S = std::is_same<R, float>::value ? WCA_STAGE + 1 : 1;  // FP64 members read the list directly
    __shared__ float2 sp[S];
    __shared__ unsigned se[S];
    __shared__ int hdr[8];
    for_entries<P, true, true>(nmap, [&](int e_) {
        const int2 t = map[e_];
        const RepDev &r = m[t.x];
        if (std::is_same<R, float>::value && r.g.fast_wca) {
            if (r.unit)
                wca_f32_body<true>(r.g, r.d, t.y, sp, se, hdr);
            else
                wca_f32_body<false>(r.g, r.d, t.y, sp, se, hdr);
        } else {
            if constexpr (std::is_same<R, float>::value) {
                wca_ref_body<R>(r.g, r.d, t.y);
            } else {
                const int first = t.y * blockDim.x;
                wca_f64_body(r.g, r.d, first, min((int)blockDim.x, r.g.N - first));
            }
        }
    });
}

template <typename R, bool P, bool P2>
__global__ __launch_bounds__(DP_THREADS) void kb_deposit(const RepDev *m, const int2 *map, int nmap, int slot) {
    for_entries<P, true, false>(nmap, [&](int e_) {
        const int2 t = map[e_];
        const RepDev &r = m[t.x];
        DepArgs a = r.dep;
        if (slot) {  // beside the rebuild: the step's end re-arms the scalars
            a.slot = 1;
            a.reset = 0;
        }
        switch (r.g.scheme) {
        case 0: deposit_body<R, 0, P2>(r.g, r.d, a, t.y); break;
        case 1: deposit_body<R, 1, P2>(r.g, r.d, a, t.y); break;
        default: deposit_body<R, 2, P2>(r.g, r.d, a, t.y); break;
        }
    });
}

// Members with a fixed dt gather the mesh force inside the update; members
// with adaptive dt read the forces of kb_gather and reduce its dt
// candidates, as their single-simulation steps do.
template <typename R, bool P, bool P2>
__global__ __launch_bounds__(256) void kb_update(const RepDev *m, const int2 *map, int nmap) {
    for_entries<P, false, true>(nmap, [&](int e_) {
        const int2 t = map[e_];
        const RepDev &r = m[t.x];
        if (r.g.adaptive) {
            switch (r.g.scheme) {
            case 0: update_body<R, 0, false, true>(r.g, r.d, t.y); break;
            case 1: update_body<R, 1, false, true>(r.g, r.d, t.y); break;
            default: update_body<R, 2, false, true>(r.g, r.d, t.y); break;
            }
        } else {
            switch (r.g.scheme) {
            case 0: update_body<R, 0, true, P2>(r.g, r.d, t.y); break;
            case 1: update_body<R, 1, true, P2>(r.g, r.d, t.y); break;
            default: update_body<R, 2, true, P2>(r.g, r.d, t.y); break;
            }
        }
    });
}

// capillary forces and dt candidates of the adaptive members (their
// particle blocks only)
template <typename R, bool P, bool P2>
__global__ __launch_bounds__(256) void kb_gather(const RepDev *m, const int2 *map, int nmap) {
    for_entries<P, true, true>(nmap, [&](int e_) {
        const int2 t = map[e_];
        const RepDev &r = m[t.x];
        switch (r.g.scheme) {
        case 0: gather_body<R, 0, P2>(r.g, r.d, 1, t.y, e_); break;
        case 1: gather_body<R, 1, P2>(r.g, r.d, 1, t.y, e_); break;
        default: gather_body<R, 2, P2>(r.g, r.d, 1, t.y, e_); break;
        }
    });
}

template <bool P>
__global__ __launch_bounds__(SCAN_THREADS) void kb_scan(const RepDev *m, const int2 *map, int nmap) {
    for_entries<P, true, false>(nmap, [&](int e_) {
        const int2 t = map[e_];
        const RepDev &r = m[t.x];
        scan_body(r.d.count, r.d.bcount, r.d.start, r.g.ncell, r.scan_nb, r.g.N, r.d.sc, 0, t.y);
    });
}

template <bool P>
__global__ __launch_bounds__(256) void kb_fill(const RepDev *m, const int2 *map, int nmap) {
    for_entries<P, false, true>(nmap, [&](int e_) {
        const int2 t = map[e_];
        fill_body(m[t.x].g, m[t.x].d, 1, t.y);
    });
}

template <bool P>
__global__ __launch_bounds__(256) void kb_sort_cells(const RepDev *m, const int2 *map, int nmap) {
    for_entries<P, false, false>(nmap, [&](int e_) {
        const int2 t = map[e_];
        sort_cells_body(m[t.x].g, m[t.x].d, 1, t.y);
    });
}

// ------------------------------------------------------------------ launchers
// Dynamic LDS above the default limit, once per device: some 200 kernels, 1 us
// each, which every bdk_create paid.
hipError_t set_kernel_attributes(int dev) {
    static std::mutex mu;
    static std::vector<char> done;
    std::lock_guard<std::mutex> lock(mu);
    if (dev < (int)done.size() && done[dev]) return hipSuccess;
    hipError_t e = fft_set_attributes();
    if (e == hipSuccess) e = pairs_set_attributes();
#define BDK_ATTR_D(K) \
    if (e == hipSuccess) e = hipFuncSetAttribute((const void *)K, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
#define BDK_ATTR_DQ(Q)                      \
    BDK_ATTR_D((k_deposit<float, 0, Q>))    \
    BDK_ATTR_D((k_deposit<float, 1, Q>))    \
    BDK_ATTR_D((k_deposit<float, 2, Q>))    \
    BDK_ATTR_D((k_deposit<double, 0, Q>))   \
    BDK_ATTR_D((k_deposit<double, 1, Q>))   \
    BDK_ATTR_D((k_deposit<double, 2, Q>))   \
    BDK_ATTR_D((kb_deposit<float, false, Q>))  \
    BDK_ATTR_D((kb_deposit<double, false, Q>)) \
    BDK_ATTR_D((kb_deposit<float, true, Q>))   \
    BDK_ATTR_D((kb_deposit<double, true, Q>))
    BDK_ATTR_DQ(true)
    BDK_ATTR_DQ(false)
#undef BDK_ATTR_DQ
#undef BDK_ATTR_D
    if (e == hipSuccess) {
        if (dev >= (int)done.size()) done.resize(dev + 1, 0);
        done[dev] = 1;
    }
    return e;
}

hipError_t launch_wca(bdk_t *h, hipStream_t st) {
    // FP32 forces use the cell-relative displacement when the box holds at
    // least 6 cells per side (the neighbour offset is then the minimum image)
    const dim3 grid(nblk(h->g.N, 256)), blk(256);
    if (!st) st = h->stream;
    if (h->g.fast_wca) {
        const bool unit = h->p.sigma11_22 == 1.0 && h->p.sigma11_12 == 1.0 && h->p.eps22_11 == 1.0 &&
                          h->p.eps12_11 == 1.0;
        if (unit)
            hipLaunchKernelGGL(k_wca_f32<true>, grid, blk, 0, st, h->g, h->d);
        else
            hipLaunchKernelGGL(k_wca_f32<false>, grid, blk, 0, st, h->g, h->d);
    } else if (h->p.precision != BDK_FP64) {
        hipLaunchKernelGGL(k_wca<float>, grid, blk, 0, st, h->g, h->d);
    } else {
        hipLaunchKernelGGL(k_wca_f64, dim3(nblk(h->g.N, WCA64_PER)), dim3(WCA64_BLOCK), 0, st, h->g, h->d);
    }
    return hipGetLastError();
}

// Deposit tiling: tcx x tcy list cells such that a tile owns about tile_pts^2
// mesh points; fixed-point scales chosen so that no sum of N charges can
// overflow 63 bits.  Without a batch's choice the side is 38 points, less on
// meshes below 532 points, so that there are some 200 tiles.  Deposit alone
// (us) at sides 16 / 24 / 30 / 38 / 46: 128^2 FP64 5.0 / 5.2 / 6.4 / 6.8 / 8.5,
// 384^2 FP64 6.8 / 6.2 / 5.2 / 6.9 / 7.9, 512^2 6.0 / 6.0 / 6.0 / 6.5 / 9.3,
// 1024^2 FP64 20.6 / 17.7 / 14.0 / 13.0 / 15.3, 2048^2 45 / 29 / 24.8 / 22.6 /
// 23.8, 4096^2 156 / 82 / 68 / 53 / 60; square tiles of side 38: 7.0, 8.4, 8.2,
// 16.9, 25.6 and 66.
struct DepPlan {
    DepArgs a;
    dim3 grid;
    size_t lds;
};

static DepPlan dep_plan(const bdk_t *h, int reset, int tile_pts = 0) {
    const Geo &g = h->g;
    const bool f64 = h->p.precision == BDK_FP64;
    DepPlan pl;
    if (tile_pts <= 0) tile_pts = std::max(16, std::min(38, g.Z / 14));
    // 1.6 times the side along y, so that a wave's lanes cover a row of the
    // tile and the rows of cells make longer ranges, but at most a wave's 64
    const double py = std::min(62.0, 1.6 * tile_pts), px = (double)tile_pts * tile_pts / py;
    auto cells = [&](double pts) { return std::max(1, std::min(g.nc, (int)std::floor(pts * g.h / g.B))); };
    pl.a.tcx = cells(px);
    pl.a.tcy = cells(py);
    auto points = [&](int tc) { return (int)std::floor(tc * g.B / g.h) + 2 + 4; };  // with the rim
    // the window stays below 64 KB of LDS
    while (pl.a.tcx > 1 && (size_t)points(pl.a.tcx) * points(pl.a.tcy) * (f64 ? 16 : 8) > 64 * 1024) --pl.a.tcx;
    while (pl.a.tcy > 1 && (size_t)points(pl.a.tcx) * points(pl.a.tcy) * (f64 ? 16 : 8) > 64 * 1024) --pl.a.tcy;
    pl.a.win_cap = points(pl.a.tcx) * points(pl.a.tcy);
    const double cmax = g.drho * std::max(1.0, std::fabs(g.f2_f1));
    const double nlog = std::log2((double)g.N * cmax + 1.0);
    int s1 = (int)std::floor(62.0 - nlog);
    if (!f64) s1 = std::min(s1, 40);
    const int gap = std::min(40, 61 - (int)std::ceil(std::log2((double)g.N + 1.0)));
    const int s2 = s1 + gap;
    pl.a.scale_hi = std::ldexp(1.0, s1);
    pl.a.iscale_hi = std::ldexp(1.0, -s1);
    pl.a.scale_lo = std::ldexp(1.0, s2);
    pl.a.iscale_lo = std::ldexp(1.0, -s2);
    pl.a.reset = reset;
    pl.a.q1 = 1.0;  // species charges of the capillary deposit (gr:31-547)
    pl.a.q2 = g.f2_f1;
    pl.a.slot = 0;
    pl.a.scale_f = 1.0f;
    pl.a.iscale_f = 1.0;
    if (!f64) {
        const int sf = (int)std::floor(30.0 - std::log2(cmax));
        pl.a.scale_f = std::ldexp(1.0f, sf);
        pl.a.iscale_f = std::ldexp(1.0, -sf);
    }
    pl.a.ty = (int)nblk(g.nc, pl.a.tcy);
    pl.grid = dim3(nblk(g.nc, pl.a.tcx) * pl.a.ty);
    pl.lds = (size_t)pl.a.win_cap * (f64 ? 16 : 8);
    return pl;
}

DepLaunch deposit_launch(const bdk_t *h) {
    DepPlan pl = dep_plan(h, 0);
    pl.a.slot = 1;
    return {pl.a, (int)pl.grid.x, pl.lds};
}


template <typename R, int SCHEME> static void launch_deposit_t(bdk_t *h, const DepPlan &pl, hipStream_t st) {
    if (zp2(h->g.Z))
        hipLaunchKernelGGL((k_deposit<R, SCHEME, true>), pl.grid, dim3(DP_THREADS), pl.lds, st, h->g, h->d, pl.a);
    else
        hipLaunchKernelGGL((k_deposit<R, SCHEME, false>), pl.grid, dim3(DP_THREADS), pl.lds, st, h->g, h->d, pl.a);
}

hipError_t launch_deposit(bdk_t *h, int reset, int slot, hipStream_t st) {
    DepPlan pl = dep_plan(h, reset);
    pl.a.slot = slot;
    if (!st) st = h->stream;
    const bool f32 = h->p.precision != BDK_FP64;
    switch (h->g.scheme) {
    case 0: f32 ? launch_deposit_t<float, 0>(h, pl, st) : launch_deposit_t<double, 0>(h, pl, st); break;
    case 1: f32 ? launch_deposit_t<float, 1>(h, pl, st) : launch_deposit_t<double, 1>(h, pl, st); break;
    default: f32 ? launch_deposit_t<float, 2>(h, pl, st) : launch_deposit_t<double, 2>(h, pl, st); break;
    }
    return hipGetLastError();
}

// number density of one species (charges 1 and 0) -> rho, from the list order
hipError_t launch_species_deposit(bdk_t *h, int species) {
    DepPlan pl = dep_plan(h, 0);
    pl.a.q1 = species == 1 ? 1.0 : 0.0;
    pl.a.q2 = species == 2 ? 1.0 : 0.0;
    hipStream_t st = h->stream;
    const bool f32 = h->p.precision != BDK_FP64;
    switch (h->g.scheme) {
    case 0: f32 ? launch_deposit_t<float, 0>(h, pl, st) : launch_deposit_t<double, 0>(h, pl, st); break;
    case 1: f32 ? launch_deposit_t<float, 1>(h, pl, st) : launch_deposit_t<double, 1>(h, pl, st); break;
    default: f32 ? launch_deposit_t<float, 2>(h, pl, st) : launch_deposit_t<double, 2>(h, pl, st); break;
    }
    return hipGetLastError();
}

hipError_t launch_by_id(bdk_t *h, int id0, int n, ByIdHead *head, int2 *git, double2 *rel) {
    hipLaunchKernelGGL(k_by_id, dim3(nblk(h->g.N, 256)), dim3(256), 0, h->stream, h->g, h->d, id0, n, head, git, rel);
    return hipGetLastError();
}

hipError_t launch_force_by_id(bdk_t *h, const void *f, double2 *out) {
    const dim3 grid(nblk(h->g.N, 256)), blk(256);
    if (h->p.precision != BDK_FP64)
        hipLaunchKernelGGL(k_force_by_id<float>, grid, blk, 0, h->stream, h->g, h->d, (const float2 *)f, out);
    else
        hipLaunchKernelGGL(k_force_by_id<double>, grid, blk, 0, h->stream, h->g, h->d, (const double2 *)f, out);
    return hipGetLastError();
}

hipError_t launch_to_host(const void *src, size_t bytes, void *dst, hipStream_t st) {
    const int n = (int)((bytes + 15) / 16);
    hipLaunchKernelGGL(k_to_host, dim3(std::max(1u, std::min(256u, nblk(n, 256)))), dim3(256), 0, st,
                       (const uint4 *)src, (uint4 *)dst, n);
    return hipGetLastError();
}

hipError_t launch_zero_ints(int *p, int n, hipStream_t st) {
    hipLaunchKernelGGL(k_zero_int, dim3(nblk(n, 256)), dim3(256), 0, st, p, n);
    return hipGetLastError();
}

hipError_t launch_rearm(bdk_t *h) {
    hipLaunchKernelGGL(k_rearm, dim3(1), dim3(64), 0, h->stream, h->g, h->d);
    return hipGetLastError();
}

template <typename R, int SCHEME> static void launch_gather_t(bdk_t *h, int with_dt, int fold) {
    if (zp2(h->g.Z))
        hipLaunchKernelGGL((k_gather<R, SCHEME, true>), dim3(nblk(h->g.N, 256)), dim3(256), 0, h->stream, h->g, h->d,
                           with_dt);
    else
        hipLaunchKernelGGL((k_gather<R, SCHEME, false>), dim3(nblk(h->g.N, 256)), dim3(256), 0, h->stream, h->g,
                           h->d, with_dt);
    if (with_dt && fold) hipLaunchKernelGGL(k_dt_fold, dim3(1), dim3(64), 0, h->stream, h->g, h->d);
}

hipError_t launch_gather(bdk_t *h, int with_dt, int fold) {
    const bool f32 = h->p.precision != BDK_FP64;
    switch (h->g.scheme) {
    case 0: f32 ? launch_gather_t<float, 0>(h, with_dt, fold) : launch_gather_t<double, 0>(h, with_dt, fold); break;
    case 1: f32 ? launch_gather_t<float, 1>(h, with_dt, fold) : launch_gather_t<double, 1>(h, with_dt, fold); break;
    default: f32 ? launch_gather_t<float, 2>(h, with_dt, fold) : launch_gather_t<double, 2>(h, with_dt, fold); break;
    }
    return hipGetLastError();
}

template <typename R, int SCHEME> static void launch_update_t(bdk_t *h, int fused) {
    if (fused && zp2(h->g.Z))
        hipLaunchKernelGGL((k_update<R, SCHEME, true, true>), dim3(nblk(h->g.N, 128)), dim3(128), 0, h->stream,
                           h->g, h->d);
    else if (fused)
        hipLaunchKernelGGL((k_update<R, SCHEME, true, false>), dim3(nblk(h->g.N, 128)), dim3(128), 0, h->stream,
                           h->g, h->d);
    else
        hipLaunchKernelGGL((k_update<R, SCHEME, false, true>), dim3(nblk(h->g.N, 128)), dim3(128), 0, h->stream,
                           h->g, h->d);
}

hipError_t launch_update(bdk_t *h, int fused) {
    const bool f32 = h->p.precision != BDK_FP64;
    switch (h->g.scheme) {
    case 0: f32 ? launch_update_t<float, 0>(h, fused) : launch_update_t<double, 0>(h, fused); break;
    case 1: f32 ? launch_update_t<float, 1>(h, fused) : launch_update_t<double, 1>(h, fused); break;
    default: f32 ? launch_update_t<float, 2>(h, fused) : launch_update_t<double, 2>(h, fused); break;
    }
    return hipGetLastError();
}

static void launch_scan_fill(bdk_t *h) {
    const int ncell = h->g.ncell;
    const int nb = (int)nblk(ncell, SCAN_BLOCK);
    hipLaunchKernelGGL(k_scan_reduce, dim3(nb), dim3(SCAN_THREADS), 0, h->stream, h->d.count, ncell, h->d.bcount);
    hipLaunchKernelGGL(k_scan, dim3(nb), dim3(SCAN_THREADS), 0, h->stream, h->d.count, h->d.bcount, h->d.start, ncell,
                       nb, h->g.N, h->d.sc, 0);
    hipLaunchKernelGGL(k_fill, dim3(nblk(h->g.N, 256)), dim3(256), 0, h->stream, h->g, h->d, 0);
    hipLaunchKernelGGL(k_sort_cells, dim3(nblk(ncell, 256 * SORT_CELLS)), dim3(256), 0, h->stream, h->g, h->d, 0);
}

hipError_t launch_own(bdk_t *h) {
    hipLaunchKernelGGL(k_own, dim3(nblk(h->g.nc + 1, 256)), dim3(256), 0, h->stream, h->g, h->d.own);
    return hipGetLastError();
}

hipError_t launch_bin(bdk_t *h) {
    hipLaunchKernelGGL(k_reset_exc, dim3(1), dim3(1), 0, h->stream, h->d.sc);
    hipLaunchKernelGGL(k_bin, dim3(nblk(h->g.N, 256)), dim3(256), 0, h->stream, h->g, h->d);
    launch_scan_fill(h);
    return hipGetLastError();
}

hipError_t launch_place(bdk_t *h, const int2 *git, const double2 *rel) {
    hipLaunchKernelGGL(k_place_clear, dim3(nblk(h->g.ncell, 256)), dim3(256), 0, h->stream, h->d.count, h->g.ncell,
                       h->d.sc);
    hipLaunchKernelGGL(k_place, dim3(nblk(h->g.N, 256)), dim3(256), 0, h->stream, h->g, h->d, git, rel);
    launch_scan_fill(h);
    return hipGetLastError();
}

hipError_t launch_refresh(bdk_t *h) {
    hipLaunchKernelGGL(k_reset_exc, dim3(1), dim3(1), 0, h->stream, h->d.sc);
    hipLaunchKernelGGL(k_zero_int, dim3(nblk(h->g.ncell, 256)), dim3(256), 0, h->stream, h->d.count, h->g.ncell);
    hipLaunchKernelGGL(k_refresh, dim3(nblk(h->g.N, 256)), dim3(256), 0, h->stream, h->g, h->d);
    launch_scan_fill(h);
    return hipGetLastError();
}

hipError_t launch_noise_out(bdk_t *h) {
    hipLaunchKernelGGL(k_noise_out, dim3(nblk(h->g.N, 256)), dim3(256), 0, h->stream, h->g, h->d);
    return hipGetLastError();
}

// ------------------------------------------------------------------ step counters
// TimestepInfo (signaturen2.h:71-145, filled by zeitschritt_debug,
// dm:168-211): the largest force of each kind by |F|^2 with its particle,
// the number of candidate pairs the cell lists present, and the particles
// that changed cell.  Maxima are 64-bit keys (|F|^2 as FP32 bits, list
// position) under atomicMax, so the result does not depend on the order.
template <typename R>
__global__ __launch_bounds__(256) void k_info_forces(Geo g, DevBufs d, StepInfoDev *info) {
    using R2 = typename V2<R>::T;
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    unsigned long long cand = 0;
    if (q < g.N) {
        const R2 fw = ((const R2 *)d.fwca)[q], fk = ((const R2 *)d.fkap)[q];
        const double2 n = particle_noise(g, d, d.lpid[q], d.sc->step);
        const double v[3] = {(double)fw.x * fw.x + (double)fw.y * fw.y, (double)fk.x * fk.x + (double)fk.y * fk.y,
                             n.x * n.x + n.y * n.y};
        for (int k = 0; k < 3; ++k) {
            const unsigned long long key = ((unsigned long long)__float_as_uint((float)v[k]) << 32) | (unsigned)q;
            atomicMax(&info->key[k], key);
        }
        // as the reference counts them: a species-1 particle against both
        // lists, a species-2 particle against list 2 (the 12 pairs once)
        const bool s2 = d.lpid[q] >= g.n1;
        const int c = d.lcell[q], cx = div_nc(c, g), cy = c - cx * g.nc;
        for (int a = -1; a <= 1; ++a)
            for (int b = -1; b <= 1; ++b) {
                const int cc = wrap1(cx + a, g.nc) * g.nc + wrap1(cy + b, g.nc);
                if (!s2) {
                    cand += d.start[cc + 1] - d.start[cc];
                } else {
                    for (int j = d.start[cc]; j < d.start[cc + 1]; ++j)
                        cand += ((const unsigned *)d.list)[j] >> 31;
                }
            }
        cand -= 1;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) cand += __shfl_xor(cand, o, 64);
    if ((threadIdx.x & 63) == 0 && cand) atomicAdd(&info->num_wca, cand);
}

// the vectors and particles of the maxima (one thread), before the update
template <typename R>
__global__ void k_info_fetch(Geo g, DevBufs d, StepInfoDev *info) {
    using R2 = typename V2<R>::T;
    for (int k = 0; k < 3; ++k) {
        const int q = (int)(info->key[k] & 0xffffffffull);
        info->pid[k] = d.lpid[q];
        if (k == 0) {
            const R2 f = ((const R2 *)d.fwca)[q];
            info->wca[0] = f.x;
            info->wca[1] = f.y;
            const int c = d.lcell[q], cx = div_nc(c, g), cy = c - cx * g.nc;
            int n1 = 0, n2 = 0;
            for (int a = -1; a <= 1; ++a)
                for (int b = -1; b <= 1; ++b) {
                    const int cc = wrap1(cx + a, g.nc) * g.nc + wrap1(cy + b, g.nc);
                    for (int j = d.start[cc]; j < d.start[cc + 1]; ++j) {
                        if (((const unsigned *)d.list)[j] >> 31) ++n2;
                        else ++n1;
                    }
                }
            info->nlist[0] = n1;
            info->nlist[1] = n2;
        } else if (k == 1) {
            const R2 f = ((const R2 *)d.fkap)[q];
            info->kap[0] = f.x;
            info->kap[1] = f.y;
        } else {
            const double2 n = particle_noise(g, d, d.lpid[q], d.sc->step);
            info->rnd[0] = n.x;
            info->rnd[1] = n.y;
        }
    }
}

// after the update, before the list rebuild: cell changes per species
__global__ void k_info_moves(Geo g, DevBufs d, StepInfoDev *info) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= g.N) return;
    if (d.cell[q] != d.lcell[q]) atomicAdd(&info->moves[d.lpid[q] >= g.n1 ? 1 : 0], 1);
}

// Event marks for per-kernel timing: with ev != nullptr an event is
// recorded on the main stream after every launch and everything runs on the
// main stream in order; names receives the labels.
struct Marks {
    bdk_t *h;
    std::vector<std::string> *names;
    std::vector<hipEvent_t> *ev;
    hipError_t e = hipSuccess;
    void chk(hipError_t r) {
        if (e == hipSuccess && r != hipSuccess) e = r;
    }
    void mark(const char *nm) {
        if (names) names->push_back(nm);
        if (ev) {
            hipEvent_t x;
            if (hipEventCreate(&x) == hipSuccess) {
                chk(hipEventRecord(x, h->stream));
                ev->push_back(x);
            }
        }
    }
};

// Forces of the current state.  The WCA forces and the mesh chain (deposit
// from the list order, FFTs) only read the particle state: the WCA runs on
// the second stream beside the chain (fork and join by events).
hipError_t enqueue_forces(bdk_t *h, std::vector<std::string> *names, std::vector<hipEvent_t> *ev) {
    Marks m{h, names, ev};
    if (ev) m.mark("begin");
    if (h->g.idgas) return hipSuccess;  // no forces
    const bool fork = !ev && h->aux;
    if (fork) {
        m.chk(hipEventRecord(h->ev_fork, h->stream));
        m.chk(hipStreamWaitEvent(h->aux, h->ev_fork, 0));
        m.chk(launch_wca(h, h->aux));
        m.chk(hipEventRecord(h->ev_join, h->aux));
    } else {
        m.chk(launch_wca(h));
        m.mark("k_wca");
    }
    m.chk(launch_deposit(h, 1));
    m.mark("k_deposit");
    for (int p = 0; p < 3; ++p) {
        m.chk(launch_fft_pass(h, p));
        m.mark(p == 0 ? "k_r2c_rows" : p == 1 ? "k_col" : "k_c2r_rows");
    }
    if (fork) m.chk(hipStreamWaitEvent(h->stream, h->ev_join, 0));
    m.chk(hipGetLastError());
    return m.e;
}

// One step from a state whose forces are ready: the update (gather, noise,
// Euler step, refresh), then the two halves that only need its output side
// by side:
//   main stream: the list rebuild (scan, fill, sort), then the WCA
//                forces of the new lists;
//   second stream: the deposit from the slot arrays (grouped by the previous
//                starts, which the update kept; halo widened by the
//                update's displacement bound), the FFT passes, the last of
//                which ends the step (counter, per-step scalars);
// joined.  The new state leaves with its forces ready.  Without forces (an
// ideal gas) the scan ends the step.
hipError_t enqueue_step(bdk_t *h, std::vector<std::string> *names, std::vector<hipEvent_t> *ev,
                        StepInfoDev *info, hipEvent_t dt_known) {
    Marks m{h, names, ev};
    if (ev) m.mark("begin");
    const bool kap = !h->g.idgas;
    const int ncell = h->g.ncell, nb = (int)nblk(ncell, SCAN_BLOCK);
    if (!kap) {
        m.chk(launch_rearm(h));
        m.mark("k_rearm");
    }
    if (info) {
        // capillary forces on their own (the step fuses them into the update)
        if (kap && !h->g.adaptive) m.chk(launch_gather(h, 0, 0));
        const bool f32 = h->p.precision != BDK_FP64;
        if (f32) {
            hipLaunchKernelGGL(k_info_forces<float>, dim3(nblk(h->g.N, 256)), dim3(256), 0, h->stream, h->g, h->d, info);
            hipLaunchKernelGGL(k_info_fetch<float>, dim3(1), dim3(1), 0, h->stream, h->g, h->d, info);
        } else {
            hipLaunchKernelGGL(k_info_forces<double>, dim3(nblk(h->g.N, 256)), dim3(256), 0, h->stream, h->g, h->d, info);
            hipLaunchKernelGGL(k_info_fetch<double>, dim3(1), dim3(1), 0, h->stream, h->g, h->d, info);
        }
    }
    if (h->g.adaptive) {
        m.chk(launch_gather(h, 1, 0));  // the update reduces the candidates itself
        m.mark("k_gather");
        m.chk(launch_update(h, 0));
    } else {
        m.chk(launch_update(h, kap ? 1 : 0));
    }
    m.mark("k_update");
    if (dt_known) m.chk(hipEventRecord(dt_known, h->stream));
    if (info) hipLaunchKernelGGL(k_info_moves, dim3(nblk(h->g.N, 256)), dim3(256), 0, h->stream, h->g, h->d, info);
    if (kap && !ev && pairs_apply(h)) {
        m.chk(launch_pairs(h));
        return m.e;
    }
    const bool fork = kap && !ev && h->aux;
    hipStream_t side = fork ? h->aux : h->stream;
    if (kap) {
        if (fork) {
            m.chk(hipEventRecord(h->ev_fork, h->stream));
            m.chk(hipStreamWaitEvent(h->aux, h->ev_fork, 0));
        }
        m.chk(launch_deposit(h, 0, 1, side));
        m.mark("k_deposit");
        for (int p = 0; p < 3; ++p) {
            m.chk(launch_fft_pass(h, p, side, p == 2));
            m.mark(p == 0 ? "k_r2c_rows" : p == 1 ? "k_col" : "k_c2r_rows");
        }
        if (fork) m.chk(hipEventRecord(h->ev_join, side));
    }
    // bcount is current (the update adjusted it with the counts)
    hipLaunchKernelGGL(k_scan, dim3(nb), dim3(SCAN_THREADS), 0, h->stream, h->d.count, h->d.bcount, h->d.start, ncell,
                       nb, h->g.N, h->d.sc, kap ? 0 : 1);
    m.mark("k_scan");
    hipLaunchKernelGGL(k_fill, dim3(nblk(h->g.N, 256)), dim3(256), 0, h->stream, h->g, h->d, 1);
    m.mark("k_fill");
    hipLaunchKernelGGL(k_sort_cells, dim3(nblk(ncell, 256 * SORT_CELLS)), dim3(256), 0, h->stream, h->g, h->d, 1);
    m.mark("k_sort_cells");
    if (kap) {
        m.chk(launch_wca(h));
        m.mark("k_wca");
    }
    if (fork) m.chk(hipStreamWaitEvent(h->stream, h->ev_join, 0));
    m.chk(hipGetLastError());
    return m.e;
}

// ------------------------------------------------------------------ batch plans

hipError_t batch_build(const std::vector<bdk_t *> &mem, const BatchTuning &tune, BatchPlan &bp,
                       std::vector<RepDev> &reps, std::vector<int2> maps[BS_COUNT]) {
    const int n = (int)mem.size();
    reps.assign(n, RepDev());
    for (int k = 0; k < BS_COUNT; ++k) {
        maps[k].clear();
        bp.nblk2[k] = 0;
        bp.nblk16[k] = 0;
    }
    bp.nmem = n;
    bp.f32 = mem.empty() ? 1 : (mem[0]->p.precision != BDK_FP64);
    bp.tune = tune;
    int zmax = 8;
    for (const bdk_t *h : mem) zmax = std::max(zmax, h->g.Z);
    for (int k = 0; k < 3; ++k) bp.ept[k] = std::max(tune.ept[k], batch_min_ept(k, zmax));
    const int *ept = bp.ept;
    bp.dep_lds = 0;
    std::fill(&bp.fft_lds[0][0], &bp.fft_lds[0][0] + 9, (size_t)0);
    std::fill(&bp.fft_threads[0][0], &bp.fft_threads[0][0] + 9, 0);
    // entries of the members with a power-of-two mesh first, those with 16
    // mesh points per FFT thread (FP32) before the others: the mesh stages
    // launch once per mesh kind present (the kind is a template parameter)
    auto cls = [&](const bdk_t *h) { return zp2(h->g.Z) ? (fft_ept(h->g.Z, bp.f32) == 16 ? 0 : 1) : 2; };
    std::vector<int> order;
    for (int pass = 0; pass < 3; ++pass)
        for (int i = 0; i < n; ++i)
            if (cls(mem[i]) == pass) order.push_back(i);
    for (int oi = 0; oi < n; ++oi) {
        const int i = order[oi];
        const bdk_t *h = mem[i];
        RepDev &r = reps[i];
        r.g = h->g;
        r.d = h->d;
        const DepPlan pl = dep_plan(h, 1, tune.dep_tile);
        r.dep = pl.a;
        bp.dep_lds = std::max(bp.dep_lds, pl.lds);
        const int Z = h->g.Z;
        r.mixr = h->mixr;
        r.mixc = h->mixc;
        fft_member(r, Z, ept, bp);
        r.scan_nb = (int)nblk(h->g.ncell, SCAN_BLOCK);
        r.unit = h->p.sigma11_22 == 1.0 && h->p.sigma11_12 == 1.0 && h->p.eps22_11 == 1.0 && h->p.eps12_11 == 1.0;
        const int ad = h->g.adaptive ? 1 : 0;
        const int nb[BS_COUNT] = {(int)nblk(h->g.N, 256), (int)nblk(h->g.ncell, 256 * SORT_CELLS), r.scan_nb,
                                  (int)pl.grid.x, Z / r.rb, (Z / 2) / r.rc, Z / r.rb2,
                                  ad * (int)nblk(h->g.N, 256), (int)nblk(h->g.N, tune.wca_block)};
        for (int k = 0; k < BS_COUNT; ++k)
            for (int b = 0; b < nb[k]; ++b) maps[k].push_back(make_int2(i, b));
        if (zp2(h->g.Z))
            for (int k = 0; k < BS_COUNT; ++k) bp.nblk2[k] = (int)maps[k].size();
        if (cls(h) == 0)
            for (int k = 0; k < BS_COUNT; ++k) bp.nblk16[k] = (int)maps[k].size();
    }
    for (int k = 0; k < BS_COUNT; ++k) bp.nblk[k] = (int)maps[k].size();
    return hipSuccess;
}

template <typename R, bool P> static void batch_stage_tp(const BatchPlan &bp, int stage, hipStream_t st) {
    const RepDev *m = bp.reps;
    // f(kind, map, entries) once per mesh kind present in stage S's map
    auto kinds = [&](int S, auto &&f) {
        const int n2 = bp.nblk2[S], nall = bp.nblk[S];
        if (n2 > 0) f(std::true_type(), (const int2 *)bp.map[S], n2);
        if (nall > n2) f(std::false_type(), (const int2 *)bp.map[S] + n2, nall - n2);
    };
#define BDK_G(S) dim3(stage_grid(bp, bp.nblk[S]))
    switch (stage) {
    case 0:
        hipLaunchKernelGGL((kb_wca<R, P>), BDK_G(BS_WCA), dim3(bp.tune.wca_block), 0, st, m, bp.map[BS_WCA],
                           bp.nblk[BS_WCA]);
        break;
    case 1:  // from the list order
    case 8:  // from the slot arrays, beside the rebuild
        kinds(BS_DEP, [&](auto q, const int2 *mp, int nm) {
            constexpr bool Q = decltype(q)::value;
            hipLaunchKernelGGL((kb_deposit<R, P, Q>), dim3(stage_grid(bp, nm)), dim3(DP_THREADS), bp.dep_lds, st, m,
                               mp, nm, stage == 8 ? 1 : 0);
        });
        break;
    case 2:
    case 3:
    case 4:
    case 12:  // 12: c2r, also the end of the step
        batch_fft_stage(bp, stage, st);
        break;
    case 5:
        kinds(BS_PART, [&](auto q, const int2 *mp, int nm) {
            constexpr bool Q = decltype(q)::value;
            hipLaunchKernelGGL((kb_update<R, P, Q>), dim3(stage_grid(bp, nm)), dim3(256), 0, st, m, mp, nm);
        });
        break;
    case 13:  // adaptive members: forces and dt candidates (their updates reduce them)
        if (bp.nblk[BS_GATHER] > 0) {
            kinds(BS_GATHER, [&](auto q, const int2 *mp, int nm) {
                constexpr bool Q = decltype(q)::value;
                hipLaunchKernelGGL((kb_gather<R, P, Q>), dim3(stage_grid(bp, nm)), dim3(256), 0, st, m, mp, nm);
            });
        }
        break;
    case 6:
        hipLaunchKernelGGL(kb_scan<P>, BDK_G(BS_SCAN), dim3(SCAN_THREADS), 0, st, m, bp.map[BS_SCAN], bp.nblk[BS_SCAN]);
        break;
    default: {  // 11: fill, sort
        hipLaunchKernelGGL(kb_fill<P>, BDK_G(BS_PART), dim3(256), 0, st, m, bp.map[BS_PART], bp.nblk[BS_PART]);
        hipLaunchKernelGGL(kb_sort_cells<P>, BDK_G(BS_CELL), dim3(256), 0, st, m, bp.map[BS_CELL], bp.nblk[BS_CELL]);
        break;
    }
    }
#undef BDK_G
}

template <typename R> static void batch_stage_t(const BatchPlan &bp, int stage, hipStream_t st) {
    if (bp.tune.persist > 0)
        batch_stage_tp<R, true>(bp, stage, st);
    else
        batch_stage_tp<R, false>(bp, stage, st);
}

// stage 0 WCA, 1 deposit (list order), 2 r2c, 3 col, 4 c2r, 5 update,
// 6 scan, 8 deposit (slot arrays), 11 fill + sort, 12 c2r + step end,
// 13 gather (forces and dt candidates) of the adaptive members
hipError_t batch_stage(const BatchPlan &bp, int stage, hipStream_t st) {
    if (bp.f32)
        batch_stage_t<float>(bp, stage, st);
    else
        batch_stage_t<double>(bp, stage, st);
    return hipGetLastError();
}

// The members' forces: the WCA stage on aux beside the mesh stages.
hipError_t batch_enqueue_forces(const BatchPlan &bp, hipStream_t st, hipStream_t aux, hipEvent_t fork,
                                hipEvent_t join) {
    hipError_t e = hipSuccess;
    if (aux) {
        e = hipEventRecord(fork, st);
        if (e == hipSuccess) e = hipStreamWaitEvent(aux, fork, 0);
        if (e == hipSuccess) e = batch_stage(bp, 0, aux);
        if (e == hipSuccess) e = hipEventRecord(join, aux);
    } else {
        e = batch_stage(bp, 0, st);
    }
    for (int k = 1; k <= 4 && e == hipSuccess; ++k) e = batch_stage(bp, k, st);
    if (aux && e == hipSuccess) e = hipStreamWaitEvent(st, join, 0);
    return e;
}

// One batched step, laid out like the single-simulation step: (the adaptive
// members' gather,) update, then
// the rebuild and the WCA on st beside the slot-order deposit and the FFT
// stages on aux (the last of which ends the step), joined.
hipError_t batch_enqueue_step(const BatchPlan &bp, hipStream_t st, hipStream_t aux, hipEvent_t fork,
                              hipEvent_t join) {
    hipError_t e = bp.nblk[BS_GATHER] > 0 ? batch_stage(bp, 13, st) : hipSuccess;
    if (e == hipSuccess) e = batch_stage(bp, 5, st);
    hipStream_t side = aux ? aux : st;
    if (aux && e == hipSuccess) e = hipEventRecord(fork, st);
    if (aux && e == hipSuccess) e = hipStreamWaitEvent(aux, fork, 0);
    if (e == hipSuccess) e = batch_stage(bp, 8, side);
    for (int k = 2; k <= 3 && e == hipSuccess; ++k) e = batch_stage(bp, k, side);
    if (e == hipSuccess) e = batch_stage(bp, 12, side);
    if (aux && e == hipSuccess) e = hipEventRecord(join, side);
    if (e == hipSuccess) e = batch_stage(bp, 6, st);
    if (e == hipSuccess) e = batch_stage(bp, 11, st);
    if (e == hipSuccess) e = batch_stage(bp, 0, st);
    if (aux && e == hipSuccess) e = hipStreamWaitEvent(st, join, 0);
    return e;
}

}  // namespace bdkx
