// The two halves of a step after the update, paired stage by stage: each
// launch runs the blocks of a mesh stage and of a list stage side by side,
//   deposit (slot arrays) | scan of the cell counts
//   r2c rows              | fill of the new lists
//   columns               | sort of the arrivals
//   c2r rows + step end   | WCA forces of the new lists
// so that one stream carries the step.  The halves only meet at the next
// update, so the pairs need no order among themselves.  For small
// simulations, whose steps are bound by launches (see pairs_apply).
#pragma clang fp contract(off)

#include "bdk_device.hpp"
#include "bdk_fft.hpp"
#include "bdk_fftmix.hpp"
#include "bdk_particles.hpp"

namespace bdkx {

template <typename R, int SCHEME, bool P2>
__global__ __launch_bounds__(DP_THREADS) void k_deposit_scan(Geo g, DevBufs d, DepArgs a, PairGrid pg) {
    bool dep;
    int i;
    if (!pg.mine(dep, i)) return;
    if (dep)
        deposit_body<R, SCHEME, P2>(g, d, a, i);
    else
        scan_body(d.count, d.bcount, d.start, g.ncell, pg.nb, g.N, d.sc, 0, i);
}

// LZ: log2 of a power-of-two mesh, or 0: another size, by its plan (EPT = 0) or
// with EPT elements per thread
template <typename R, int LZ, int EPT>
__global__ __launch_bounds__(LZ ? FFT_MAX_THREADS : FFT_THREADS) void k_r2c_fill(Geo g, DevBufs d, int rows, int stride,
                                                                                 MixPlan mp, PairGrid pg) {
    using C = typename V2<R>::T;
    bool mesh;
    int i;
    if (!pg.mine(mesh, i)) return;
    if (!mesh) {
        fill_body(g, d, 1, i);
        return;
    }
    const int blk = xcd_of(i, pg.na, g.xcd);
    if constexpr (LZ > 0)
        r2c_p2<R, LZ>((const R *)d.rho, (C *)d.ht, (const C *)d.tw, rows, blk);
    else
        r2c_other<R, EPT>((const R *)d.rho, (C *)d.ht, (const C *)d.tw, g.Z, mp, rows, stride, blk);
}

template <typename R, int LZ, int EPT>
__global__ __launch_bounds__(LZ ? FFT_MAX_THREADS : FFT_THREADS) void k_col_sort(Geo g, DevBufs d, int rows, int stride,
                                                                                 MixPlan mp, PairGrid pg) {
    using C = typename V2<R>::T;
    using C4 = typename V4<R>::T;
    bool mesh;
    int i;
    if (!pg.mine(mesh, i)) return;
    if (!mesh) {
        sort_cells_body(g, d, 1, i);
        return;
    }
    const R *sq = sizeof(R) == 4 ? (const R *)d.sqf : (const R *)d.sq;
    const R *lap = sizeof(R) == 4 ? (const R *)d.lapf : (const R *)d.lap;
    if constexpr (LZ > 0)
        col_p2<R, LZ>((const C *)d.ht, (C4 *)d.gt, (const C *)d.tw, sq, lap, g, rows, i);
    else
        col_other<R, EPT>((const C *)d.ht, (C4 *)d.gt, (const C *)d.tw, sq, lap, g, mp, rows, stride, i);
}

// UNIT: FP32 with all sigma and epsilon ratios 1
template <typename R, int LZ, int EPT, bool UNIT>
__global__ __launch_bounds__(LZ ? FFT_MAX_THREADS : FFT_THREADS) void k_c2r_wca(Geo g, DevBufs d, int rows, int stride,
                                                                                MixPlan mp, int stage, PairGrid pg) {
    using C = typename V2<R>::T;
    using C4 = typename V4<R>::T;
    bool mesh;
    int i;
    if (!pg.mine(mesh, i)) return;
    if (!mesh) {
        const int blk = xcd_of(i, pg.nb, g.xcd);
        if constexpr (sizeof(R) == 4) {
            extern __shared__ unsigned char smem_raw[];
            int *hdr = (int *)smem_raw;
            float2 *sp = (float2 *)(smem_raw + 64);
            wca_f32_body<UNIT>(g, d, blk, sp, (unsigned *)(sp + stage + 1), hdr, stage);
        } else {
            const int per = blockDim.x / WCA_LANES, first = blk * per;
            wca_f64_body(g, d, first, min(per, g.N - first));
        }
        return;
    }
    if (i == 0) step_end_body(g, d);
    const int blk = xcd_of(i, pg.na, g.xcd);
    if constexpr (LZ > 0)
        c2r_p2<R, LZ>((const C4 *)d.gt, (C *)d.fmesh, (const C *)d.tw, rows, blk);
    else
        c2r_other<R, EPT>((const C4 *)d.gt, (C *)d.fmesh, (const C *)d.tw, g.Z, mp, rows, stride, blk);
}

// candidates staged by a WCA block of `threads` particles, and its LDS
static int wca_stage(int threads) { return std::max(WCA_STAGE, 4 * threads); }
static size_t wca_lds(int threads, bool unit) {
    const size_t n = (size_t)wca_stage(threads) + 1;
    return 64 + n * 8 + (unit ? 0 : n * 4);
}

// Below 30 MB of a step's compulsory bytes (64 N + 36 Z^2 in FP32, 80 N + 72
// Z^2 in FP64; one simulation with forces of k_wca_f32 or FP64) the launches
// and the waits between two streams cost more than the stages: paired.  Above
// it the stages fill the chip by themselves, and the mesh stage's LDS and
// registers then cost the list stage its occupancy: two streams.  Step,
// two streams / paired (us): 2000 on 128^2 FP64 37 / 27, 16,000 on 256^2 40 /
// 28, 64,000 on 512^2 with travel cap 48.5 / 39.0, 64,000 on 512^2 FP64 44.2 /
// 41.6 (24 MB), 256,000 on 512^2 50.9 / 46.7 (26 MB), 128,000 on 512^2 FP64
// 52.5 / 53.6 (29 MB), 500,000 on 512^2
// 59.5 / 61.7 (41 MB), 128,000 on 1024^2 48.8 / 48.6 (46 MB), 200,000 on 1024^2
// FP64 71 / 73, 2M on 2048^2 164 / 191.
bool pairs_apply(const bdk_t *h) {
    if (h->p.precision != BDK_FP64 && !h->g.fast_wca) return false;
    const double f64 = h->p.precision == BDK_FP64, z2 = (double)h->g.Z * h->g.Z;
    return (64.0 + 16.0 * f64) * h->g.N + 36.0 * (1.0 + f64) * z2 < 30e6;
}

template <typename R> static void launch_deposit_scan(bdk_t *h) {
    const DepLaunch dl = deposit_launch(h);
    const PairGrid pg(dl.blocks, (int)nblk(h->g.ncell, SCAN_BLOCK));
    const dim3 grid(pg.blocks()), blk(DP_THREADS);
#define DS(S)                                                                                                        \
    if (zp2(h->g.Z))                                                                                                 \
        hipLaunchKernelGGL((k_deposit_scan<R, S, true>), grid, blk, dl.lds, h->stream, h->g, h->d, dl.a, pg);         \
    else                                                                                                             \
        hipLaunchKernelGGL((k_deposit_scan<R, S, false>), grid, blk, dl.lds, h->stream, h->g, h->d, dl.a, pg)
    switch (h->g.scheme) {
    case 0: DS(0); break;
    case 1: DS(1); break;
    default: DS(2); break;
    }
#undef DS
}

template <typename R, int LZ, int EPT> static void launch_mesh_pair(bdk_t *h, int pass, const FftLaunch &l) {
    const bool unit = h->p.sigma11_22 == 1.0 && h->p.sigma11_12 == 1.0 && h->p.eps22_11 == 1.0 && h->p.eps12_11 == 1.0;
    const dim3 blk(l.threads);
    if (pass == 0) {
        const PairGrid pg(l.blocks, (int)nblk(h->g.N, l.threads));
        hipLaunchKernelGGL((k_r2c_fill<R, LZ, EPT>), dim3(pg.blocks()), blk, l.lds, h->stream, h->g, h->d, l.rows, l.stride,
                           l.mix, pg);
    } else if (pass == 1) {
        const PairGrid pg(l.blocks, (int)nblk(h->g.ncell, l.threads * SORT_CELLS));
        hipLaunchKernelGGL((k_col_sort<R, LZ, EPT>), dim3(pg.blocks()), blk, l.lds, h->stream, h->g, h->d, l.rows, l.stride,
                           l.mix, pg);
    } else if constexpr (sizeof(R) == 4) {
        const PairGrid pg(l.blocks, (int)nblk(h->g.N, l.threads));
        const size_t lds = std::max(l.lds, wca_lds(l.threads, unit));
        if (unit)
            hipLaunchKernelGGL((k_c2r_wca<R, LZ, EPT, true>), dim3(pg.blocks()), blk, lds, h->stream, h->g, h->d, l.rows,
                               l.stride, l.mix, wca_stage(l.threads), pg);
        else
            hipLaunchKernelGGL((k_c2r_wca<R, LZ, EPT, false>), dim3(pg.blocks()), blk, lds, h->stream, h->g, h->d, l.rows,
                               l.stride, l.mix, wca_stage(l.threads), pg);
    } else {
        const PairGrid pg(l.blocks, (int)nblk(h->g.N, l.threads / WCA_LANES));
        hipLaunchKernelGGL((k_c2r_wca<R, LZ, EPT, true>), dim3(pg.blocks()), blk, l.lds, h->stream, h->g, h->d, l.rows,
                           l.stride, l.mix, 0, pg);
    }
}

template <typename R> static void launch_mesh_pairs(bdk_t *h) {
    for (int pass = 0; pass < 3; ++pass) {
        const FftLaunch l = fft_launch(h, pass);
        if (zp2(h->g.Z)) {
#define CALL(LZ) launch_mesh_pair<R, LZ, 8>(h, pass, l)
            switch (h->g.logZ) { BDK_LOGZ_LOW(CALL) BDK_LOGZ_HIGH(CALL) }
#undef CALL
        } else {
#define CALL(E) launch_mesh_pair<R, 0, E>(h, pass, l)
            BDK_OTHER_SWITCH(l.ept, CALL)
#undef CALL
        }
    }
}

hipError_t launch_pairs(bdk_t *h) {
    if (h->p.precision != BDK_FP64) {
        launch_deposit_scan<float>(h);
        launch_mesh_pairs<float>(h);
    } else {
        launch_deposit_scan<double>(h);
        launch_mesh_pairs<double>(h);
    }
    return hipGetLastError();
}

hipError_t pairs_set_attributes() {
    hipError_t e = hipSuccess;
    auto big = [&](const void *k, int kb = 160) {
        if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kb * 1024);
    };
#define MESH(R, LZ, E)                               \
    big((const void *)k_r2c_fill<R, LZ, E>);       \
    big((const void *)k_col_sort<R, LZ, E>);       \
    big((const void *)k_c2r_wca<R, LZ, E, true>);
#define CALL(LZ)                                        \
    MESH(float, LZ, 8) MESH(double, LZ, 8)            \
    big((const void *)k_c2r_wca<float, LZ, 8, false>);
    CALL(3) CALL(4) CALL(5) CALL(6) CALL(7) CALL(8) CALL(9) CALL(10) CALL(11) CALL(12)
#undef CALL
#define CALL(E)                                         \
    MESH(float, 0, E) MESH(double, 0, E)              \
    big((const void *)k_c2r_wca<float, 0, E, false>);
    CALL(0) CALL(8) CALL(16) CALL(32)
#undef CALL
#undef MESH
#define DS(S, Q)                                          \
    big((const void *)k_deposit_scan<float, S, Q>, 156);  /* the scan has a little static LDS */ \
    big((const void *)k_deposit_scan<double, S, Q>, 156);
    DS(0, true) DS(0, false) DS(1, true) DS(1, false) DS(2, true) DS(2, false)
#undef DS
    return e;
}

}  // namespace bdkx
