// Device code of the particle stages (WCA forces, deposit, list rebuild),
// shared by the kernels of one stage, of paired stages and of batches.
#pragma once
#include "bdk_device.hpp"

namespace bdkx {

// ------------------------------------------------------------------ WCA
// One thread per list position.  Neighbours come from the cell list of
// the 3x3 cells around the particle's own cell (the extended-list semantics
// of dm:459-526): entries are slot | species << 31, each cell's entries
// sorted by slot, so every sum has a fixed order.  Same-species and
// cross-species contributions are summed separately and then added, the
// grouping of dm:617-702 + dm:973-1059.
constexpr unsigned LIST_SLOT = 0x7fffffffu;
// rank of a particle that changed cell during the step: its arrival index
// in the new cell, marked (ranks stay below 2^30).  RANK_OPEN marks the rank
// of a stayer whose cell begins before its wave's first list position: the
// stayers there are still to be added.
constexpr int RANK_MOVED = 1 << 30;
constexpr int RANK_OPEN = 1 << 31;
// Scan of the cell counts: blocks of SCAN_BLOCK cells, SCAN_PER_THREAD
// consecutive cells per thread; bcount[c >> SCAN_SHIFT] is the particle count
// of the block holding cell c
constexpr int SCAN_THREADS = 256;
constexpr int SCAN_SHIFT = 12;
constexpr int SCAN_BLOCK = 1 << SCAN_SHIFT;  // 4096 cells per block
constexpr int SCAN_PER_THREAD = SCAN_BLOCK / SCAN_THREADS;
static_assert(SCAN_PER_THREAD % 4 == 0, "int4 loads");
// bcount entries sit 128 bytes apart: the movers' atomics on the blocks of
// a dense region then spread over many L2 lines instead of a few
constexpr int BCOUNT_STRIDE = 32;

template <typename R>
__device__ __forceinline__ void wca_ref_body(const Geo &g, const DevBufs &d, int blk) {
    using R2 = typename V2<R>::T;
    const int qi = blk * blockDim.x + threadIdx.x;
    if (qi >= g.N) return;
    const int nc = g.nc;
    const unsigned *list = (const unsigned *)d.list;
    const int s = (int)(list[qi] & LIST_SLOT);
    const int c = d.lcell[qi];
    const int cx = div_nc(c, g), cy = c - cx * nc;
    const double2 ri = d.lrel[qi];
    const bool s2i = d.lpid[qi] >= g.n1;
    R fsx = 0, fsy = 0, fcx = 0, fcy = 0;
    {
        // the reference's FP64 arithmetic on absolute positions (am:100-166,
        // dm:640-698); the S2 side of a 12 pair is the negated S1 side
        const double xi = cx * g.B + ri.x, yi = cy * g.B + ri.y;
        for (int da = -1; da <= 1; ++da)
            for (int db = -1; db <= 1; ++db) {
                const int ux = wrap1(cx + da, nc), uy = wrap1(cy + db, nc);
                const int cc = ux * nc + uy;
                const int qe = d.start[cc + 1];
                for (int q = d.start[cc]; q < qe; ++q) {
                    const unsigned ent = list[q];
                    const int sj = (int)(ent & LIST_SLOT);
                    if (sj == s) continue;
                    const bool s2j = (ent >> 31) != 0;
                    const double2 rj = d.lrel[q];
                    const double xj = ux * g.B + rj.x, yj = uy * g.B + rj.y;
                    R fx, fy;
                    if (!s2i && !s2j) {
                        if (wca_pair<R>(xi, yi, xj, yj, 0, g, fx, fy)) { fsx += fx; fsy += fy; }
                    } else if (s2i && s2j) {
                        if (wca_pair<R>(xi, yi, xj, yj, 1, g, fx, fy)) { fsx += fx; fsy += fy; }
                    } else if (!s2i) {
                        if (wca_pair<R>(xi, yi, xj, yj, 2, g, fx, fy)) { fcx += fx; fcy += fy; }
                    } else {
                        if (wca_pair<R>(xj, yj, xi, yi, 2, g, fx, fy)) { fcx -= fx; fcy -= fy; }
                    }
                }
            }
    }
    R2 o;
    o.x = fsx + fcx;
    o.y = fsy + fcy;
    ((R2 *)d.fwca)[qi] = o;
}

// FP64 forces: four lanes per particle (list positions first .. first + n -
// 1 of the block).  A row's candidates (cells cy - 1 .. cy + 1, one range of
// the list or two where y wraps) go to the four lanes in turn, so a lane
// meets about one per row, and the rows' loads are in flight together; the
// lanes' sums are added pairwise.  A candidate costs its two coordinate
// differences unless it lies within the cutoff.  Where a difference exceeds
// L/2 the images are compared as the reference does (wca_pair); below it the
// nearest image is the difference itself, and the arithmetic is that of
// wca_pair bit for bit.
//
// Bound by its chain of dependent loads (list starts, candidates) at small N
// and by FP64 issue (two divisions per partner within the cutoff) at large
// N.  One lane per particle and cell by cell: 2000 particles 28 us, 4000
// (dilute) 12.4, 200,000 45; so 5.9, 4.5 and 14.6.
constexpr int WCA_LANES = 4;

__device__ __forceinline__ void wca_f64_body(const Geo &g, const DevBufs &d, int first, int n) {
    const int nc = g.nc, sub = threadIdx.x & (WCA_LANES - 1);
    const unsigned *list = (const unsigned *)d.list;
    const double hl = 0.5 * g.L;
    for (int i = threadIdx.x / WCA_LANES; i < n; i += blockDim.x / WCA_LANES) {
        const int qi = first + i;
        const int c = d.lcell[qi];
        const int cx = div_nc(c, g), cy = c - cx * nc;
        const double2 ri = d.lrel[qi];
        const bool s2i = d.lpid[qi] >= g.n1;
        const double xi = cx * g.B + ri.x, yi = cy * g.B + ri.y;
        // the rows' ranges: qa[r] + k for k < na[r], then qb[r] + k
        int qa[3], na[3], qb[3], nt[3];
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const int *st = d.start + wrap1(cx + r - 1, nc) * nc;
            if (cy >= 1 && cy <= nc - 2) {
                qa[r] = st[cy - 1];
                na[r] = nt[r] = st[cy + 2] - qa[r];
                qb[r] = 0;
            } else {
                const int ya = cy == 0 ? nc - 1 : cy - 1;  // first part: up to the edge
                qa[r] = st[ya];
                na[r] = st[nc] - qa[r];
                const int yb = cy == 0 ? 2 : 1;  // second part: cells 0 .. yb - 1
                qb[r] = st[0] - na[r];
                nt[r] = na[r] + st[yb] - st[0];
            }
        }
        double fsx = 0, fsy = 0, fcx = 0, fcy = 0;
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            const int ux = wrap1(cx + r - 1, nc), row = ux * nc;
            const double xr = ux * g.B;
            for (int k = sub; k < nt[r]; k += WCA_LANES) {
                const int q = (k < na[r] ? qa[r] : qb[r]) + k;
                if (q == qi) continue;
                const double2 rj = d.lrel[q];
                const int uy = d.lcell[q] - row;
                const bool s2j = (list[q] >> 31) != 0;
                const double xj = xr + rj.x, yj = uy * g.B + rj.y;
                double dx = xi - xj, dy = yi - yj, fx, fy;
                const int type = s2i == s2j ? (s2i ? 1 : 0) : 2;
                if (fabs(dx) > hl || fabs(dy) > hl) {
                    if (type < 2 || !s2i) {
                        if (!wca_pair<double>(xi, yi, xj, yj, type, g, fx, fy)) continue;
                    } else {  // the S2 side of a 12 pair is the negated S1 side
                        if (!wca_pair<double>(xj, yj, xi, yi, 2, g, fx, fy)) continue;
                        fx = -fx;
                        fy = -fy;
                    }
                } else {
                    double a2 = dx * dx + dy * dy;
                    const double sig = type == 1 ? g.s22 : g.s12;
                    if ((type == 0 ? a2 : a2 * sig * sig) > g.cut2) continue;
                    if (type != 0) {
                        a2 *= sig * sig;
                        dx *= sig;
                        dy *= sig;
                    }
                    const double a_8 = 1.0 / (a2 * a2 * a2 * a2);
                    const double a_14 = 1.0 / (a2 * a2 * a2 * a2 * a2 * a2 * a2);
                    double absF = type == 0 ? 4.0 * 6.0 * (2.0 * a_14 - a_8)
                                            : (type == 1 ? g.e22f : g.e12f) * 4.0 * 6.0 * (2.0 * a_14 - a_8);
                    if (absF > g.maxpair) absF = g.maxpair;
                    fx = absF * dx;
                    fy = absF * dy;
                }
                if (type < 2) {
                    fsx += fx;
                    fsy += fy;
                } else {
                    fcx += fx;
                    fcy += fy;
                }
            }
        }
#pragma unroll
        for (int o = 1; o < WCA_LANES; o <<= 1) {
            fsx += __shfl_xor(fsx, o, 64);
            fsy += __shfl_xor(fsy, o, 64);
            fcx += __shfl_xor(fcx, o, 64);
            fcy += __shfl_xor(fcy, o, 64);
        }
        if (sub == 0) ((double2 *)d.fwca)[qi] = make_double2(fsx + fcx, fsy + fcy);
    }
}

// FP32 forces for boxes of at least 6 cells per side: the displacement is
// the difference of the in-cell offsets (FP32 copies centred on the cell,
// lrelf) plus the cell offset, the minimum image by construction.  UNIT: all
// sigma and epsilon ratios are 1, so the per-type factors drop out and one
// sum collects all partners; otherwise same-species and cross-species
// partners are summed apart and added at the end (the grouping of
// dm:617-702 + dm:973-1059).  Partners are visited in list order, cell by
// cell, row by row.
//
// A block handles consecutive list positions.  Their neighbour cells in row
// da (da = -1, 0, 1: the cells (cx + da, cy - 1 .. cy + 1)) form one
// contiguous range of the list when no particle's row wraps around the box
// in x; the block copies the three ranges' offsets (and entries) to LDS once
// and every particle away from the y edge reads its candidates there.  The
// rest (the first and last cell columns, rows wrapping in y, ranges beyond
// the LDS capacity) read the list directly.  Both loops evaluate a candidate
// with the same code, so a particle's force has the same bits either way
// (and therefore for every block size).
// staged candidates per block: 8 KB of offsets, small enough to share a CU
// with the FFT passes of the other stream (measured in the two-stream step:
// 2048 entries 185.5 us, 1024 180.7 us, 768 183.4 us per step; a dense
// 256-particle block stages about 800)
constexpr int WCA_STAGE = 1024;

// One candidate (entry e, centred offset r) at list position q.  The cell
// offset is folded into this particle's coordinates: y + B below m1 (yb), y
// below m2 (ym), y - B from m2 on (ya), x + ox (xo).  SELF: the row holds
// this particle (position qi, excluded).  Outside the cutoff the force is
// selected away rather than branched around (every wave holds some partner
// inside, so the branch would not skip the arithmetic).  Contraction into
// FMAs is allowed in the FP32 force arithmetic, unlike the FP64 position
// arithmetic.
template <bool UNIT, bool SELF>
__device__ __forceinline__ void wca_f32_cand(unsigned e, float2 r, int q, int qi, bool s2i, int m1, int m2, float xo,
                                             float yb, float ym, float ya, float cut2, float cap, float sigA,
                                             float prefA, float sigB, float prefB, float &fsx, float &fsy,
                                             float &fcx, float &fcy) {
#pragma clang fp contract(fast)
    const float yo = q < m1 ? yb : (q < m2 ? ym : ya);
    const float dx = xo - r.x, dy = yo - r.y;
    const float r2 = dx * dx + dy * dy;
    if (UNIT) {
        const float inv = __builtin_amdgcn_rcpf(r2);
        const float i2 = inv * inv, i4 = i2 * i2;
        float absF = fminf(24.0f * (2.0f * (i4 * i2 * inv) - i4), cap);
        absF = (r2 <= cut2 && (!SELF || q != qi)) ? absF : 0.0f;
        fsx += absF * dx;
        fsy += absF * dy;
    } else {
        const bool s2j = (e >> 31) != 0;
        const float sig = s2j ? sigB : sigA;
        const float r2s = r2 * sig * sig;
        const float inv = __builtin_amdgcn_rcpf(r2s);
        const float i2 = inv * inv, i4 = i2 * i2;
        float absF = fminf((s2j ? prefB : prefA) * 24.0f * (2.0f * (i4 * i2 * inv) - i4), cap);
        absF = (r2s <= cut2 && (!SELF || q != qi)) ? absF : 0.0f;
        const float fx = absF * dx * sig, fy = absF * dy * sig;
        if (s2i == s2j) {
            fsx += fx;
            fsy += fy;
        } else {
            fcx += fx;
            fcy += fy;
        }
    }
}

// candidates q0..qe-1 read from the list, loaded one candidate ahead of the
// arithmetic (the list arrays carry one padding entry).  (Scalar arguments:
// a parameter struct here was placed in LDS by the compiler.)
template <bool UNIT, bool SELF>
__device__ __forceinline__ void wca_f32_row(const unsigned *__restrict__ list, const float2 *__restrict__ rf, int qi,
                                            bool s2i, int q0, int qe, int m1, int m2, float xo, float yb, float ym,
                                            float ya, float cut2, float cap, float sigA, float prefA, float sigB,
                                            float prefB, float &fsx, float &fsy, float &fcx, float &fcy) {
    unsigned ent = list[q0];
    float2 rj = rf[q0];
    for (int q = q0; q < qe; ++q) {
        const unsigned e = ent;
        const float2 r = rj;
        ent = list[q + 1];  // q + 1 <= N: padding entry
        rj = rf[q + 1];
        wca_f32_cand<UNIT, SELF>(e, r, q, qi, s2i, m1, m2, xo, yb, ym, ya, cut2, cap, sigA, prefA, sigB, prefB, fsx,
                                 fsy, fcx, fcy);
    }
}

// the same candidates read from the staged copy (list position q at q + delta)
template <bool UNIT, bool SELF>
__device__ __forceinline__ void wca_f32_row_lds(const float2 *sp, const unsigned *se, int delta, int qi, bool s2i,
                                                int q0, int qe, int m1, int m2, float xo, float yb, float ym,
                                                float ya, float cut2, float cap, float sigA, float prefA, float sigB,
                                                float prefB, float &fsx, float &fsy, float &fcx, float &fcy) {
    float2 rn = sp[q0 + delta];
    unsigned en = UNIT ? 0u : se[q0 + delta];
    for (int q = q0; q < qe; ++q) {
        const float2 r = rn;
        const unsigned e = en;
        rn = sp[q + 1 + delta];  // one ahead: the arrays hold one entry more than the stage
        if (!UNIT) en = se[q + 1 + delta];
        wca_f32_cand<UNIT, SELF>(e, r, q, qi, s2i, m1, m2, xo, yb, ym, ya, cut2, cap, sigA, prefA, sigB, prefB, fsx,
                                 fsy, fcx, fcy);
    }
}

// LDS of the staged rows: offsets sp[cap + 1], entries
// se[cap + 1] (not UNIT; the extra entry is read ahead, never used),
// and hdr[8] (each row's first list position and length, and whether the
// block stages).  Every thread of the block calls this.
template <bool UNIT>
__device__ __forceinline__ void wca_f32_body(const Geo &g, const DevBufs &d, int blk, float2 *sp, unsigned *se,
                                             int *hdr, int cap_stage = WCA_STAGE) {
    const int nb = blockDim.x, tid = threadIdx.x;
    const int q_first = blk * nb;
    const int q_last = min(q_first + nb, g.N) - 1;
    const int nc = g.nc;
    const unsigned *list = (const unsigned *)d.list;
    const float2 *rf = d.lrelf;
    if (tid < 3) {
        // lane da + 1: the list range of the cells (cx + da, cy - 1 .. cy + 1)
        // over the block's cells c_first..c_last (list order is cell order)
        const int cf = d.lcell[q_first], cl = d.lcell[q_last];
        const int ok = div_nc(cf, g) >= 1 && div_nc(cl, g) <= nc - 2;
        int g0 = 0, len = 0;
        if (ok) {
            const int da = tid - 1;
            const int lo = max(cf + da * nc - 1, 0), hi = min(cl + da * nc + 1, g.ncell - 1);
            g0 = d.start[lo];
            len = d.start[hi + 1] - g0;
        }
        hdr[tid] = g0;
        hdr[3 + tid] = len;
        if (tid == 0) hdr[6] = ok;
    }
    __syncthreads();
    const int l0 = hdr[3], l1 = hdr[4], total = l0 + l1 + hdr[5];
    const bool staged = hdr[6] && total <= cap_stage;
    if (staged) {
        for (int t = tid; t < total; t += nb) {
            const int r = (t >= l0) + (t >= l0 + l1);
            const int q = hdr[r] + t - (r == 0 ? 0 : (r == 1 ? l0 : l0 + l1));
            sp[t] = rf[q];
            if (!UNIT) se[t] = list[q];
        }
    }
    __syncthreads();
    const int qi = q_first + tid;
    if (qi > q_last) return;
    const int c = d.lcell[qi];
    const int cx = div_nc(c, g), cy = c - cx * nc;
    const float2 ri = rf[qi];
    const bool s2i = d.lpid[qi] >= g.n1;
    const float B = (float)g.B, cut2 = (float)g.cut2, cap = (float)g.maxpair;
    // factors for a partner of species 1 (A) or species 2 (B)
    const float sigA = s2i ? (float)g.s12 : 1.0f, prefA = s2i ? (float)g.e12f : 1.0f;
    const float sigB = s2i ? (float)g.s22 : (float)g.s12, prefB = s2i ? (float)g.e22f : (float)g.e12f;
    const float yb = ri.y + B, ym = ri.y, ya = ri.y - B;
    float fsx = 0, fsy = 0, fcx = 0, fcy = 0;
    // cells cy-1, cy, cy+1 of a row are adjacent in the list
    const bool inner = cy >= 1 && cy <= nc - 2;
    if (staged && inner) {
#define BDK_WCA_ROW(SELF)                                                                                       \
    wca_f32_row_lds<UNIT, SELF>(sp, se, delta, qi, s2i, s0, s3, s1, s2, xo, yb, ym, ya, cut2, cap, sigA, prefA, \
                                sigB, prefB, fsx, fsy, fcx, fcy)
        for (int da = -1; da <= 1; ++da) {
            const float xo = ri.x - da * B;
            const int *st = d.start + (cx + da) * nc + cy - 1;
            const int s0 = st[0], s1 = st[1], s2 = st[2], s3 = st[3];
            const int delta = (da < 0 ? 0 : (da == 0 ? l0 : l0 + l1)) - hdr[da + 1];
            if (da == 0)
                BDK_WCA_ROW(true);
            else
                BDK_WCA_ROW(false);
        }
#undef BDK_WCA_ROW
    } else {
#define BDK_WCA_ROW(SELF, Q0, QE, M1, M2)                                                                    \
    wca_f32_row<UNIT, SELF>(list, rf, qi, s2i, Q0, QE, M1, M2, xo, yb, ym, ya, cut2, cap, sigA, prefA, sigB, \
                            prefB, fsx, fsy, fcx, fcy)
        for (int da = -1; da <= 1; ++da) {
            const int row = wrap1(cx + da, nc) * nc;
            const float xo = ri.x - da * B;
            if (inner) {
                const int *st = d.start + row + cy - 1;
                const int s0 = st[0], s1 = st[1], s2 = st[2], s3 = st[3];
                if (da == 0)
                    BDK_WCA_ROW(true, s0, s3, s1, s2);
                else
                    BDK_WCA_ROW(false, s0, s3, s1, s2);
            } else {
                for (int db = -1; db <= 1; ++db) {
                    const int cc = row + wrap1(cy + db, nc);
                    const int q0 = d.start[cc], qe = d.start[cc + 1];
                    const int m1 = db < 0 ? qe : q0, m2 = db > 0 ? q0 : qe;
                    if (da == 0 && db == 0)
                        BDK_WCA_ROW(true, q0, qe, m1, m2);
                    else
                        BDK_WCA_ROW(false, q0, qe, m1, m2);
                }
            }
        }
#undef BDK_WCA_ROW
    }
    float2 o;
    o.x = fsx + fcx;
    o.y = fsy + fcy;
    ((float2 *)d.fwca)[qi] = o;
}

// ------------------------------------------------------------------ deposit
// Charge assignment (gr:31-547) per tile of tcx x tcy list cells.  A mesh
// point belongs to the tile whose cells contain its centre,
// owner(k) = floor((k+1/2)h/B).  Every particle near enough adds its (up to
// 9) weighted charges in LDS to a window of the tile's own points and two
// more on every side, so a particle has one base index and fixed offsets: one
// whose stencil misses the own points is skipped, and what falls beside them
// is not written out.  The particles come row by row of list cells (each
// row's cells are one range of the list, two where y wraps), DP_LANES lanes
// per row.
//
// The additions are integer (fixed point, scale 2^S), so the sums do not
// depend on the order of the atomics: the deposit is deterministic without
// floating-point atomics.  FP32 charges are truncated to 32-bit fixed point
// (|charge| 2^S < 2^31: a truncation error of 2^-31 of the largest charge,
// far below FP32 resolution) and summed in 64 bits.  FP64 mode splits every
// charge into a coarse and a fine integer part (two accumulators), which
// keeps the sum exact to ~2^-(S+40).
//
// Bound by its phases' latency (bounds, list starts, particles, write-out)
// and the 64-bit LDS atomics.  Before (square tiles, a window over all that the
// staged cells could reach, particles through a prefix sum and a segment
// table): 26.3 us at 2M particles on 2048^2, now 22.6; 4M on 4096^2 74.6 ->
// 53.4; 64,000 on 512^2 8.2 -> 6.0; 200,000 FP64 on 1024^2 14.9 -> 13.0.  With 8,
// 32 or 64 lanes per row: 25.8, 21.7 and 23.0 us on 2048^2, 63, 55 and 55 on
// 4096^2, 9.0, 7.1 and 7.5 on 512^2; 512 threads: 26.1, 69 and 6.8.
constexpr int DP_THREADS = 256;
constexpr int DP_LANES = 16;     // lanes per row of list cells

// one mesh point's charge into the accumulators at w
template <typename R>
__device__ __forceinline__ void deposit_add(const DepArgs &a, float cf, double cd, int w, unsigned long long *hi,
                                            unsigned long long *lo) {
    if (std::is_same<R, float>::value) {
        atomicAdd(&hi[w], (unsigned long long)(long long)(int)cf);
    } else {
        const long long Xh = __double2ll_rn(cd * a.scale_hi);
        const double rem = cd - (double)Xh * a.iscale_hi;
        const long long Xl = __double2ll_rn(rem * a.scale_lo);
        atomicAdd(&hi[w], (unsigned long long)Xh);
        atomicAdd(&lo[w], (unsigned long long)Xl);
    }
}

// The window of a tile: mesh rows kw0 .. kw0 + nwx - 1, columns lw0 ..
// (unwrapped), its own points klo .. khi - 1, llo .. lhi - 1; and the points
// that a particle of the visited cells may reach (kr0, nrx, ...), beyond
// which the displacement bound was wrong.
struct DepWin {
    int klo, khi, llo, lhi, kw0, lw0, nwx, nwy, kr0, nrx, lr0, nry;
    bool win;  // the window's points are distinct (else only own points, tested one by one)
    bool chk;  // the reachable points are well short of the whole mesh
    // a particle may lie a quarter of the box or more outside its cell, so that a mesh index
    // may leave the range that wrapz takes (not P2); a branch of the whole block costs 0.2 us
    // of 9 at 300,000 particles on 1000^2, a fold of every particle's index 0.6
    bool far;
};

// one particle at (x, y) with fixed-point charge dqs (FP32: drho q 2^S) or q (FP64)
template <typename R, int SCHEME, bool P2>
__device__ __forceinline__ void deposit_particle(const Geo &g, const DevBufs &d, const DepArgs &a, const DepWin &v,
                                                 float dqs, double q, double x, double y, unsigned long long *hi,
                                                 unsigned long long *lo) {
    int kp, lp;
    R wx[3], wy[3];
    weights_r<R, SCHEME>(x, g, kp, wx);
    weights_r<R, SCHEME>(y, g, lp, wy);
    if (!P2 && v.far) foldz<P2>(kp, lp, g.Z);
    constexpr bool F32 = std::is_same<R, float>::value;
    auto charge = [&](int ia, int ib, float &cf, double &cd) {
        if (F32)
            cf = SCHEME == 0 ? dqs : ((float)wx[ia] * (float)wy[ib]) * dqs;
        else
            cd = SCHEME == 0 ? g.drho * q : (double)wx[ia] * (double)wy[ib] * g.drho * q;
    };
    if (v.win) {
        // (unsigned: a last tile's window of a particle below 0 comes out below 0, rightly
        // beside; P2: masked)
        const int kb = wrapz<P2>(kp - 1 - v.kw0, g.Z), lb = wrapz<P2>(lp - 1 - v.lw0, g.Z);
        if ((unsigned)kb > (unsigned)(v.nwx - 3) || (unsigned)lb > (unsigned)(v.nwy - 3)) {  // none of the own points
            if (v.chk && (wrapz<P2>(kp - v.kr0, g.Z) >= v.nrx || wrapz<P2>(lp - v.lr0, g.Z) >= v.nry))
                atomicOr(&d.sc->nonfinite, 4);
            return;
        }
        const int w = kb * v.nwy + lb;
#pragma unroll
        for (int ia = 0; ia < 3; ++ia) {
            if (SCHEME == 0 && ia != 1) continue;
            if (SCHEME == 1 && wx[ia] == 0) continue;
#pragma unroll
            for (int ib = 0; ib < 3; ++ib) {
                if (SCHEME == 0 && ib != 1) continue;
                if (SCHEME == 1 && wy[ib] == 0) continue;
                float cf = 0.f;
                double cd = 0.0;
                charge(ia, ib, cf, cd);
                deposit_add<R>(a, cf, cd, w + ia * v.nwy + ib, hi, lo);
            }
        }
        return;
    }
#pragma unroll
    for (int ia = 0; ia < 3; ++ia) {
        if (SCHEME == 0 && ia != 1) continue;
        const int k = wrapz<P2>(kp + ia - 1, g.Z);
        if (k < v.klo || k >= v.khi) continue;
#pragma unroll
        for (int ib = 0; ib < 3; ++ib) {
            if (SCHEME == 0 && ib != 1) continue;
            const int l = wrapz<P2>(lp + ib - 1, g.Z);
            if (l < v.llo || l >= v.lhi) continue;
            float cf = 0.f;
            double cd = 0.0;
            charge(ia, ib, cf, cd);
            deposit_add<R>(a, cf, cd, (k - v.kw0) * v.nwy + (l - v.lw0), hi, lo);
        }
    }
}

// list cells that hold every particle which can reach mesh points [p0, p1) of
// an axis: those of x / h in [p0 - 1, p1 + 1), widened by the bound e on how
// far a particle lies outside its cell; c0 in [-nc, nc), n <= nc
__device__ __forceinline__ void deposit_span(int p0, int p1, double e, const Geo &g, int &c0, int &n) {
    const int lo = (int)floor(((p0 - 1) * g.h - e) / g.B), hi = (int)floor(((p1 + 1) * g.h + e) / g.B);
    c0 = lo;
    n = hi - lo + 1;
    if (n >= g.nc) {
        c0 = 0;
        n = g.nc;
    }
}

// lb: tile index, tiles numbered y fastest over a.ty tiles per row
template <typename R, int SCHEME, bool P2>
__device__ __forceinline__ void deposit_body(const Geo &g, const DevBufs &d, const DepArgs &a, int lb) {
    extern __shared__ unsigned char smem_raw[];
    constexpr bool F32 = std::is_same<R, float>::value;
    unsigned long long *hi = (unsigned long long *)smem_raw, *lo = hi + a.win_cap;
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63;
    const int nc = g.nc;
    const int cx0 = (lb / a.ty) * a.tcx, cy0 = (lb % a.ty) * a.tcy;
    const int nx = min(a.tcx, nc - cx0), ny = min(a.tcy, nc - cy0);
    const unsigned long long step = d.sc->step;
    // bound on how far a particle lies outside the cell it is listed in: the
    // excursion of rel outside [0, B] (list order), or during a rebuild the
    // distance of the new positions outside their previous cells
    double e = a.slot ? dbits(d.exo[lane * 16]) : dbits(d.sc->exc_bits[step & 1]);
    DepWin v;
    v.klo = d.own[cx0];
    v.khi = d.own[cx0 + nx];
    v.llo = d.own[cy0];
    v.lhi = d.own[cy0 + ny];
    v.win = v.khi - v.klo + 4 <= g.Z && v.lhi - v.llo + 4 <= g.Z;
    const int rim = v.win ? 2 : 0;
    v.kw0 = v.klo - rim;
    v.lw0 = v.llo - rim;
    v.nwx = v.khi - v.klo + 2 * rim;
    v.nwy = v.lhi - v.llo + 2 * rim;
    for (int w = tid; w < v.nwx * v.nwy; w += nt) {
        hi[w] = 0ull;
        if (!F32) lo[w] = 0ull;
    }
    if (a.reset && lb == 0 && tid == 0) {
        // per-step scalars for the kernels that follow this one
        d.sc->dt_bits = bitsd(g.dt_max);
        d.sc->exc_bits[(step + 1) & 1] = 0ull;
    }
    if (a.slot) {
#pragma unroll
        for (int o = 32; o >= 1; o >>= 1) e = fmax(e, __shfl_xor(e, o, 64));
    }
    e += 1e-9 * g.L;
    v.far = !P2 && __builtin_amdgcn_readfirstlane(!(e <= 0.25 * g.L));
    int rx0, nrows, ry0, ncols;
    deposit_span(v.klo, v.khi, e, g, rx0, nrows);
    deposit_span(v.llo, v.lhi, e, g, ry0, ncols);
    // mesh indices of the visited cells' particles (with a margin of one)
    v.kr0 = (int)floor((rx0 * g.B - e) * g.hinv) - 1;
    v.nrx = (int)floor(((rx0 + nrows) * g.B + e) * g.hinv) + 2 - v.kr0;
    v.lr0 = (int)floor((ry0 * g.B - e) * g.hinv) - 1;
    v.nry = (int)floor(((ry0 + ncols) * g.B + e) * g.hinv) + 2 - v.lr0;
    v.chk = nrows < nc && ncols < nc && 2 * v.nrx <= g.Z && 2 * v.nry <= g.Z;
    rx0 = wrapc(rx0, nc);
    ry0 = wrapc(ry0, nc);
    const int *st = a.slot ? d.start_old : d.start;
    // FP32: the species charges in fixed point, drho q 2^S (2^S exact)
    const float dqs1 = ((float)g.drho * (float)a.q1) * a.scale_f, dqs2 = ((float)g.drho * (float)a.q2) * a.scale_f;
    const int *cells = a.slot ? d.cell : d.lcell, *ids = a.slot ? d.pid : d.lpid;
    const double2 *rels = a.slot ? d.rel : d.lrel;
    const int yend = ry0 + ncols, ye = min(yend, nc), wrapped = max(yend - nc, 0);
    __syncthreads();  // accumulators cleared before the first atomic
    for (int r = tid / DP_LANES; r < nrows; r += nt / DP_LANES) {
        const int *row = st + wrap1(rx0 + r, nc) * nc;
        const int qa = row[ry0], na = row[ye] - qa, qb = row[0], nb = wrapped ? row[wrapped] - qb : 0;
        for (int k = tid & (DP_LANES - 1); k < na + nb; k += DP_LANES) {
            const int q = k < na ? qa + k : qb + (k - na);
            const int c = cells[q];  // during a rebuild the new cell, not that of the row
            const double2 rr = rels[q];
            const bool s2 = ids[q] >= g.n1;
            const int gx = div_nc(c, g), gy = c - gx * nc;
            deposit_particle<R, SCHEME, P2>(g, d, a, v, s2 ? dqs2 : dqs1, s2 ? a.q2 : a.q1, gx * g.B + rr.x,
                                            gy * g.B + rr.y, hi, lo);
        }
    }
    __syncthreads();
    // the own points, a wave per mesh row
    R *rho = (R *)d.rho;
    const int nl = v.lhi - v.llo;
    for (int k = v.klo + (tid >> 6); k < v.khi; k += nt >> 6) {
        const int w = (k - v.kw0) * v.nwy + rim;
        for (int l = lane; l < nl; l += 64) {
            double val;
            if (F32)
                val = (double)(long long)hi[w + l] * a.iscale_f;
            else
                val = (double)(long long)hi[w + l] * a.iscale_hi + (double)(long long)lo[w + l] * a.iscale_lo;
            rho[(size_t)k * g.Z + v.llo + l] = (R)val;
        }
    }
}

// Exclusive scan of the cell counts into start[] in one pass: a block scans
// its SCAN_BLOCK cells (int4 loads, wave scans, one LDS exchange) and adds
// the particles of the blocks before it, summed from bcount.  The last
// thread of the last block closes the step: start[ncell] = total, step
// counter += inc_step.
__device__ __forceinline__ void scan_body(const int *__restrict__ count, const int *__restrict__ bcount,
                                          int *__restrict__ start, int ncell, int nb, int nmax, DevScalars *sc,
                                          int inc_step, int blk) {
    constexpr int NW = SCAN_THREADS / 64;
    __shared__ int ws[2 * NW];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    int p = 0;
    for (int i = tid; i < blk; i += SCAN_THREADS) p += bcount[i * BCOUNT_STRIDE];
    const int base = blk * SCAN_BLOCK + tid * SCAN_PER_THREAD;
    const bool full = base + SCAN_PER_THREAD <= ncell;
    int loc[SCAN_PER_THREAD];
    if (full) {
        const int4 *c4 = (const int4 *)(count + base);
#pragma unroll
        for (int k = 0; k < SCAN_PER_THREAD / 4; ++k) {
            const int4 v = c4[k];
            loc[4 * k] = v.x;
            loc[4 * k + 1] = v.y;
            loc[4 * k + 2] = v.z;
            loc[4 * k + 3] = v.w;
        }
    } else {
#pragma unroll
        for (int q = 0; q < SCAN_PER_THREAD; ++q) loc[q] = base + q < ncell ? count[base + q] : 0;
    }
    int s = 0;
#pragma unroll
    for (int q = 0; q < SCAN_PER_THREAD; ++q) s += loc[q];
    int x = s;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) p += __shfl_xor(p, o, 64);
    if (lane == 63) ws[w] = x;
    if (lane == 0) ws[NW + w] = p;
    __syncthreads();
    int e = x - s;
#pragma unroll
    for (int k = 0; k < NW; ++k) e += ws[NW + k] + (k < w ? ws[k] : 0);
    // starts are clamped into [0, total of the recount]: list ranges stay
    // inside the arrays even if the counts were inconsistent (then flagged)
    int out[SCAN_PER_THREAD];
#pragma unroll
    for (int q = 0; q < SCAN_PER_THREAD; ++q) {
        out[q] = min(max(e, 0), nmax);
        e += loc[q];
    }
    if (full) {
        int4 *s4 = (int4 *)(start + base);
#pragma unroll
        for (int k = 0; k < SCAN_PER_THREAD / 4; ++k)
            s4[k] = make_int4(out[4 * k], out[4 * k + 1], out[4 * k + 2], out[4 * k + 3]);
    } else {
#pragma unroll
        for (int q = 0; q < SCAN_PER_THREAD; ++q)
            if (base + q < ncell) start[base + q] = out[q];
    }
    if (blk == nb - 1 && tid == SCAN_THREADS - 1) {
        start[ncell] = min(max(e, 0), nmax);
        if (e != nmax) atomicOr(&sc->nonfinite, 2);
        if (inc_step) sc->step += 1;
    }
}

// List entries and the list-ordered state from the ranks.  After a step
// (moved_ranks) a cell holds its stayers first (ascending slot, ranked by
// the update), then its arrivals (marked ranks, ordered by k_sort_cells); after
// a full binning every rank is the position in the cell (ordered by
// k_sort_cells).
__device__ __forceinline__ void fill_body(const Geo &g, const DevBufs &d, int moved_ranks, int blk) {
    const int s = blk * blockDim.x + threadIdx.x;
    if (s >= g.N) return;
    const int pid = d.pid[s];
    const int c = d.cell[s];
    const int rk = d.rank[s];
    // what a mover (start of the next cell, arrivals) or an open rank (the cell's
    // previous start) needs besides is loaded together, one trip to memory (an
    // ideal gas of 64,000 18.4 -> 18.0 us a step, of 4000 15.7 -> 15.4)
    const bool moved = moved_ranks && (rk & RANK_MOVED), open = moved_ranks && (rk & RANK_OPEN);
    const int b = d.start[c];
    int end = 0, arr = 0, from = s;
    if (moved) {
        end = d.start[c + 1];
        arr = d.arr[c];
    }
    if (open) from = d.start_old[c];
    int pos = b + (rk & (RANK_MOVED - 1));
    if (moved) pos += end - b - arr;
    if (open)  // the stayers of the cell before the update's wave
        for (int p = from; p < (s & ~63); ++p) pos += d.cell[p] == c;
    if ((unsigned)pos >= (unsigned)g.N) {  // inconsistent counts: flagged, nothing written
        atomicOr(&d.sc->nonfinite, 2);
        return;
    }
    const double2 r = d.rel[s];
    ((unsigned *)d.list)[pos] = (unsigned)s | ((pid >= g.n1 ? 1u : 0u) << 31);
    d.lcell[pos] = c;
    d.lrel[pos] = r;
    d.lpid[pos] = pid;
    if (g.fast_wca) d.lrelf[pos] = make_float2((float)(r.x - 0.5 * g.B), (float)(r.y - 0.5 * g.B));
    if (g.pos_mode == 2) d.lcomp[pos] = d.comp[s];
}

// Fixed order inside each cell: after a step only the arrivals (the last
// arr[c] entries) need sorting by slot, after a full binning the whole cell.
// Entries move together with their list-ordered state.
// entries lo .. n - 1 of the cell that begins at list position b, by slot
__device__ __forceinline__ void sort_entries(const Geo &g, const DevBufs &d, int b, int lo, int n) {
    unsigned *l = (unsigned *)d.list + b;
    double2 *rl = d.lrel + b;
    int *pl = d.lpid + b;
    float2 *fl = d.lrelf + b;
    const bool f = g.fast_wca, kah = g.pos_mode == 2;
    float2 *cl = kah ? d.lcomp + b : nullptr;
    for (int i = lo + 1; i < n; ++i) {
        const unsigned v = l[i];
        const double2 vr = rl[i];
        const int vp = pl[i];
        const float2 vf = f ? fl[i] : make_float2(0.f, 0.f);
        const float2 vc = kah ? cl[i] : make_float2(0.f, 0.f);
        int j = i - 1;
        while (j >= lo && (l[j] & LIST_SLOT) > (v & LIST_SLOT)) {
            l[j + 1] = l[j];
            rl[j + 1] = rl[j];
            pl[j + 1] = pl[j];
            if (f) fl[j + 1] = fl[j];
            if (kah) cl[j + 1] = cl[j];
            --j;
        }
        l[j + 1] = v;
        rl[j + 1] = vr;
        pl[j + 1] = vp;
        if (f) fl[j + 1] = vf;
        if (kah) cl[j + 1] = vc;
    }
}

// arrivals of a cell after a step: most cells had none and one or two had
// one; only cells with two or more read their range and sort
__device__ __forceinline__ void sort_arrivals(const Geo &g, const DevBufs &d, int c, int a) {
    if (a < 2) return;
    const int b = d.start[c], n = d.start[c + 1] - b;
    if (n < a) return;  // inconsistent counts, flagged by the scan
    sort_entries(g, d, b, n - a, n);
}

// SORT_CELLS consecutive cells per thread: a thread whose cells had no arrival
// is done after two loads
constexpr int SORT_CELLS = 8;
__device__ __forceinline__ void sort_cells_body(const Geo &g, const DevBufs &d, int moved_ranks, int blk) {
    const int c0 = (blk * blockDim.x + threadIdx.x) * SORT_CELLS;
    if (c0 >= g.ncell) return;
    if (moved_ranks && c0 + SORT_CELLS <= g.ncell) {
        const int4 u = *(const int4 *)(d.arr + c0), v = *(const int4 *)(d.arr + c0 + 4);
        if ((u.x | u.y | u.z | u.w | v.x | v.y | v.z | v.w) == 0) return;
        *(int4 *)(d.arr + c0) = make_int4(0, 0, 0, 0);  // consumed by k_fill
        *(int4 *)(d.arr + c0 + 4) = make_int4(0, 0, 0, 0);
        const int a[SORT_CELLS] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
#pragma unroll
        for (int k = 0; k < SORT_CELLS; ++k) sort_arrivals(g, d, c0 + k, a[k]);
        return;
    }
    for (int c = c0; c < min(c0 + SORT_CELLS, g.ncell); ++c) {
        const int a = d.arr[c];
        d.arr[c] = 0;
        if (moved_ranks) {
            sort_arrivals(g, d, c, a);
        } else {
            const int b = d.start[c], n = d.start[c + 1] - b;
            sort_entries(g, d, b, 0, n);
        }
    }
}

}  // namespace bdkx
