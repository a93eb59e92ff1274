// Geometric-multigrid kernels for gfx950: FP32 Chebyshev smoothing with the
// coarse-grid correction fused into the first post-smoothing step, one-pass
// pairs of steps (and of the last step with the restriction), residual +
// restriction, FP64 Galerkin coarsening over 2x2x2 aggregates, the dense
// coarsest solve. (The small levels' launches are in mg_tile.hip.)
//
// Threads map to cells with z (the unit-stride axis of the reference layout)
// across the 64 lanes of a wavefront and y across the 4 wavefronts of a
// block; each block covers one x plane of its tile (see cell_tile).
#include "device_util.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <initializer_list>
#include <type_traits>

namespace sfp {

Launch cell_launch(Dims d, int planes, int max_planes) {
    Launch L;
    unsigned tz = 64;
    while (tz > 1 && (int)tz / 2 >= d.nz) tz /= 2;
    const unsigned ty = kBlock / tz;
    L.cg.gx = (d.nz + tz - 1) / tz;
    L.cg.gy = (d.ny + ty - 1) / ty;
    if (planes <= 0) {
        // march over several x planes per block (x-neighbour reuse in
        // registers) while keeping >= ~2048 blocks to fill 256 CUs
        const long long tiles = (long long)L.cg.gx * L.cg.gy * d.nx;
        planes = (int)std::min<long long>(max_planes, std::max<long long>(1, tiles / 2048));
    }
    L.cg.planes = planes;
    const unsigned gz = (d.nx + L.cg.planes - 1) / L.cg.planes;
    L.block = dim3(tz, ty, 1);
    L.grid = dim3(L.cg.gx * L.cg.gy * gz, 1, 1);
    return L;
}

namespace {

// true when a batched solve has already converged (see KrylovScalars::stop)
__device__ __forceinline__ bool gated(const double *gate) { return gate && *gate != 0.0; }


template <bool FROM64>
__global__ __launch_bounds__(kBlock) void k_smooth_first(CellGrid cg, Dims d, Op32 A, const double *r64,
                                                         float *b, float *x, float c0,
                                                         const double *gate) {
    if (gated(gate)) return;
    int k, j, i0;
    cell_tile(cg, k, j, i0);
    if (k >= d.nz || j >= d.ny) return;
    for (int i = i0, ie = min(i0 + cg.planes, d.nx); i < ie; i++) {
        const size_t c = d.idx(i, j, k);
        float bv;
        if constexpr (FROM64) {
            bv = (float)r64[c];
            b[c] = bv;
        } else {
            bv = b[c];
        }
        x[c] = c0 * rcp_or_zero(A.diag[c]) * bv;
    }
}

// One Chebyshev step xout = x + d', d' = cd d + cr D^{-1} (b - A x), marching
// over the block's x planes with the x-direction neighbours kept in
// registers and the z-direction neighbours (iterate and z coupling) taken
// from the adjacent lanes of the tile row (only the row's end lanes load
// them). The input iterate x is, by mode:
//   SM_FIRST   : the zero-start first step c0 D^{-1} b, recomputed at every
//                stencil point (b read from r64 and rounded when r64 != null,
//                which also stores b); the previous direction equals it
//   SM_PROLONG : xin + P e (piecewise-constant coarse correction)
// (the other modes run over the flat cell index, k_smooth_flat, as SM_PROLONG
// does where z rows hold whole groups). Every lane of a row takes part in the shuffles, so lanes past the grid
// edge stay in the loop with their loads and stores masked.
template <int MODE>
__global__ __launch_bounds__(kBlock) void k_smooth(CellGrid cg, Dims d, Op32 A,
                                                   const double *__restrict__ r64,
                                                   float *__restrict__ b,
                                                   const float *__restrict__ xin,
                                                   float *__restrict__ xout, float *dvec,
                                                   float c0, float cd, float cr,
                                                   const float *__restrict__ e, Dims dc,
                                                   const double *gate) {
    if (gated(gate)) return;
    constexpr bool kFirst = (MODE & SM_FIRST) != 0;
    constexpr bool kProlong = (MODE & SM_PROLONG) != 0;
    static_assert(kFirst != kProlong && (MODE & ~(SM_FIRST | SM_PROLONG | SM_WRITE_D)) == 0, "k_smooth's modes");
    int k, j, i0;
    cell_tile(cg, k, j, i0);
    const int tz = blockDim.x;
    const int lane = threadIdx.x;  // position in the tile row
    const bool on = k < d.nz && j < d.ny;
    if (i0 >= d.nx) return;  // uniform over the block
    const Strides s(d);
    auto bval = [&](size_t q) -> float { return r64 ? (float)r64[q] : b[q]; };
    // coarse-grid offsets (prolongation): plane stride, and this thread's
    // column and its y neighbours' columns within a coarse plane
    const size_t dcsx = (size_t)dc.ny * dc.nz;
    size_t eo = 0, eym = 0, eyp = 0;
    if constexpr (kProlong) {
        if (on) {
            eo = dc.idx(0, j >> 1, k >> 1);
            if (j > 0) eym = dc.idx(0, (j - 1) >> 1, k >> 1);
            if (j + 1 < d.ny) eyp = dc.idx(0, (j + 1) >> 1, k >> 1);
        }
    }
    // iterate value at a neighbour point q (cell coordinates qi, qj, qk; for
    // the prolongation, ecol = the point's column offset on the coarse grid)
    auto xval = [&](size_t q, int qi, size_t ecol) -> float {
        if constexpr (kFirst) {
            return c0 * rcp_or_zero(A.diag[q]) * bval(q);
        } else {
            return xin[q] + e[(size_t)(qi >> 1) * dcsx + ecol];
        }
    };
    const int ie = min(i0 + cg.planes, d.nx);
    const bool zlo = k > 0, zhi = k + 1 < d.nz;
    size_t c = on ? d.idx(i0, j, k) : 0;
    float xm = 0.f, xc = 0.f, cxc = 0.f;
    bool primed = false;  // xm, xc, cxc hold this plane's values
    const bool ylo = on && j > 0, yhi = on && j + 1 < d.ny;
    for (int i = i0; i < ie; i++, c += s.sx) {
        const float dg = on ? A.diag[c] : 0.f;
        // a wavefront whose cells are all inactive has nothing to update (their
        // vectors hold zeros and couple with weight 0): skip it whole
        if (!__any(on && dg > 0.f)) {
            primed = false;
            continue;
        }
        if (!primed) {
            xm = (on && i > 0) ? xval(c - s.sx, i - 1, eo) : 0.f;
            xc = on ? xval(c, i, eo) : 0.f;
            cxc = on ? A.cpl[0][c] : 0.f;
            primed = true;
        }
        // every load of the plane is issued before the lane exchange
        const bool up = i + 1 < d.nx;
        const float xp = (on && up) ? xval(c + s.sx, i + 1, eo) : 0.f;
        const float cxp = (on && up) ? A.cpl[0][c + s.sx] : 0.f;
        const float czm = on ? A.cpl[2][c] : 0.f;
        const float cym = ylo ? A.cpl[1][c] : 0.f;
        const float xym = ylo ? xval(c - s.sy, i, eym) : 0.f;
        const float cyp = yhi ? A.cpl[1][c + s.sy] : 0.f;
        const float xyp = yhi ? xval(c + s.sy, i, eyp) : 0.f;
        float bc = 0.f;
        if constexpr (kFirst) {
            bc = on ? bval(c) : 0.f;
        } else {
            bc = on ? b[c] : 0.f;
        }
        float dprev = 0.f;
        float xin_c = 0.f;
        if constexpr (kProlong) xin_c = on ? xin[c] : 0.f;
        float xzm = __shfl_up(xc, 1, tz);
        float xzp = __shfl_down(xc, 1, tz);
        float czp = __shfl_down(czm, 1, tz);
        if (lane == 0) xzm = (on && zlo) ? xval(c - 1, i, kProlong ? dc.idx(0, j >> 1, (k - 1) >> 1) : 0) : 0.f;
        if (lane == tz - 1) {
            xzp = (on && zhi) ? xval(c + 1, i, kProlong ? dc.idx(0, j >> 1, (k + 1) >> 1) : 0) : 0.f;
            czp = (on && zhi) ? A.cpl[2][c + 1] : 0.f;
        }
        if (on) {
            float off = fmaf(cxc, xm, cxp * xp);
            if (j > 0) off = fmaf(cym, xym, off);
            if (j + 1 < d.ny) off = fmaf(cyp, xyp, off);
            if (zlo) off = fmaf(czm, xzm, off);
            if (zhi) off = fmaf(czp, xzp, off);
            if constexpr (kFirst) {
                if (r64) b[c] = bc;
            }
            // centre iterate: the coarse correction only lands on active cells
            float x0 = xc;
            if constexpr (kProlong) {
                if (!(dg > 0.f)) x0 = xin_c;
            }
            const float r = bc - fmaf(dg, x0, -off);
            if constexpr (kFirst) dprev = x0;
            const float dn = fmaf(cd, dprev, cr * rcp_or_zero(dg) * r);
            xout[c] = x0 + dn;
            if constexpr ((MODE & SM_WRITE_D) != 0) dvec[c] = dn;
        }
        xm = xc;
        xc = xp;
        cxc = cxp;
    }
}

// The step in every mode but SM_FIRST over the flat cell index, four
// consecutive cells per lane (of one z row where nz is a multiple of 4; else
// wherever they lie, kAny): 16-byte loads of every array at the cell, its x and
// y neighbours and the upper x and y couplings, one more iterate value and z
// coupling at each end of the group. With SM_XFIRST the iterate is the
// zero-start first step and the previous direction too; with SM_PROLONG the
// coarse correction (two coarse cells per group and row) is added to every
// iterate value read and, on active cells, to the centre, as k_prolong_add
// followed by a plain step would. A cell's off-diagonal sum has the order x-,
// x+, y-, y+, z-, z+ (one fmaf each, the first two products paired), as
// k_smooth's. A wavefront whose 256 cells are all inactive writes nothing, or 0.
constexpr unsigned kSmoothFlatCells = 4 * kBlock;
constexpr size_t kEagerCells = (size_t)1 << 21;

// Row-sum FP32 diagonal (Op32::pinned_rowsum) of one cell from its six
// couplings in the order -x, +x, -y, +y, -z, +z (0 where there is no
// neighbour): summed in FP64 (exact for couplings within 2^27 of each other)
// and rounded once, the assembly's arithmetic, so the bits are the stored
// diagonal's.
__device__ __forceinline__ float rowsum_diag(float xl, float xh, float yl, float yh, float zl, float zh) {
    return (float)(((((((double)xl + (double)xh) + (double)yl) + (double)yh) + (double)zl) + (double)zh));
}
// The same for the four cells of a group: the lower x and y couplings (cxc,
// cym), the upper ones (cxp, cyp: the next plane's and row's lower), the
// lower z ones (cz) and the one above the group (czhi).
typedef float f4v __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f4v rowsum_diag4(f4v cxc, f4v cxp, f4v cym, f4v cyp, f4v cz, float czhi) {
    f4v dg;
#pragma unroll
    for (int q = 0; q < 4; q++) dg[q] = rowsum_diag(cxc[q], cxp[q], cym[q], cyp[q], cz[q], q < 3 ? cz[q + 1] : czhi);
    return dg;
}
// The group of four cells from c on holds none of the cells whose diagonal is
// not the row sum (0, 1, nz, nz*ny); kAny: it may start at any cell. For
// operators of Op32::pinned_rowsum only (the kernels' kRowsum): the condition
// guards a load, so it holds nothing uniform beside the lane's part, and no
// branch of its own (see load_operands).
template <bool kAny = false>
__device__ __forceinline__ bool rowsum_group(size_t c, Dims d) {
    if constexpr (!kAny) return (c != 0) & (c != (size_t)d.nz) & (c != (size_t)d.ny * d.nz);
    const unsigned sy = (unsigned)d.nz, sx = (unsigned)d.ny * sy, cu = (unsigned)c;
    return (cu > 1) & (sy - cu >= 4) & (sx - cu >= 4);  // (differences below 0 are large)
}

// The operands of one group, which (kAny: nz no multiple of 4) need not lie
// within a z row: a neighbour is sx, sy or 1 cells on in the array wherever the
// row or the plane ends, since the coupling to what lies across an end is 0 as
// stored (the lower one of the first cell there). A missing neighbour group's
// address is the group's own, and the upper couplings past the array are put to
// 0 by selection, so the loads need no branches and are all in flight together.
// With kAny a neighbour's group is at any 4-byte address. One that crosses the
// array's end is loaded past it (an allocation reaches 64 bytes past its array)
// and one that crosses its start is loaded from the start and moved; the cells
// outside are put to 0 (end_cells). (Branches of the lanes here, on these rare
// groups, cost 20 registers; with a uniform part in their condition they were
// compiled to loads at undefined addresses.)
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
struct GroupOperands {
    f4v xc, xm, xp, ym, yp, cx, cxp, cy, cyp, cz, b;
    float zlo, zhi, czhi;
};
// the first `k` cells of a group stay, the others are put to 0
__device__ __forceinline__ f4v first_cells(f4v v, unsigned k) {
#pragma unroll
    for (unsigned q = 0; q < 4; q++) v[q] = q < k ? v[q] : 0.f;
    return v;
}
// a group moved up by k cells, 0 below
__device__ __forceinline__ f4v moved_up(f4v v, unsigned k) {
    if (k & 1) v = f4v{0.f, v.x, v.y, v.z};
    if (k & 2) v = f4v{0.f, 0.f, v.x, v.y};
    return k < 4 ? v : f4v{0.f, 0.f, 0.f, 0.f};
}
// a group's own cells of an array, 0 past its end
template <bool kAny>
__device__ __forceinline__ f4v own_cells(const float *__restrict__ a, unsigned c, unsigned n) {
    const f4v v = *(const f4u *)(a + c);
    return kAny ? first_cells(v, n - c) : v;
}
template <bool kAny>
__device__ __forceinline__ void store_cells(float *__restrict__ a, unsigned c, unsigned n, f4v v) {
    if (!kAny || n - c >= 4) {
        *(f4u *)(a + c) = v;
    } else {
#pragma unroll
        for (unsigned q = 0; q < 4; q++)
            if (c + q < n) a[c + q] = v[q];
    }
}
template <bool kAny>
__device__ __forceinline__ GroupOperands load_operands(const Op32 &A, const float *__restrict__ b,
                                                       const float *__restrict__ x, Dims d, unsigned c) {
    const unsigned n = (unsigned)d.cells(), sy = (unsigned)d.nz, sx = (unsigned)d.ny * sy, left = n - c;
    const unsigned cxm = c >= sx ? c - sx : 0, cym = c >= sy ? c - sy : 0;
    const unsigned cxu = left > sx ? c + sx : c, cyu = left > sy ? c + sy : c;
    const unsigned czl = c > 0 ? c - 1 : c, czu = left > 4 ? c + 4 : c;
    GroupOperands g;
    g.xc = *(const f4u *)(x + c);
    g.xm = *(const f4u *)(x + cxm);
    g.xp = *(const f4u *)(x + cxu);
    g.ym = *(const f4u *)(x + cym);
    g.yp = *(const f4u *)(x + cyu);
    g.cx = *(const f4u *)(A.cpl[0] + c);
    g.cxp = *(const f4u *)(A.cpl[0] + cxu);
    g.cy = *(const f4u *)(A.cpl[1] + c);
    g.cyp = *(const f4u *)(A.cpl[1] + cyu);
    g.cz = *(const f4u *)(A.cpl[2] + c);
    g.b = *(const f4u *)(b + c);
    g.zlo = x[czl];
    g.zhi = x[czu];
    g.czhi = A.cpl[2][czu];
    return g;
}
__device__ __forceinline__ void pin(const GroupOperands &g) {
    for (const f4v &v : {g.xc, g.xm, g.xp, g.ym, g.yp, g.cx, g.cxp, g.cy, g.cyp, g.cz, g.b}) sfp::pin(v);
    sfp::pin(g.zlo);
    sfp::pin(g.zhi);
    sfp::pin(g.czhi);
}
// What lies past the array put to 0: the upper couplings and (kAny) the cells of
// groups that cross its ends.
template <bool kAny>
__device__ __forceinline__ void end_cells(GroupOperands &g, Dims d, unsigned c) {
    const unsigned sy = (unsigned)d.nz, sx = (unsigned)d.ny * sy, left = (unsigned)d.cells() - c;
    if constexpr (kAny) {
        const unsigned xu = left > sx ? left - sx : 0, yu = left > sy ? left - sy : 0;  // cells there are
        g.cxp = first_cells(g.cxp, xu);
        g.xp = first_cells(g.xp, xu);
        g.cyp = first_cells(g.cyp, yu);
        g.yp = first_cells(g.yp, yu);
        const unsigned xd = c < sx ? sx - c : 0, yd = c < sy ? sy - c : 0;  // (from 4 on: none, coupled with 0)
        if (__any((xd - 1 < 3) | (yd - 1 < 3))) {
            g.xm = moved_up(g.xm, xd);
            g.ym = moved_up(g.ym, yd);
        }
        g.xc = first_cells(g.xc, left);
        g.cx = first_cells(g.cx, left);
        g.cy = first_cells(g.cy, left);
        g.cz = first_cells(g.cz, left);
        g.b = first_cells(g.b, left);
    } else {
        const f4v z4 = {0.f, 0.f, 0.f, 0.f};
        if (!(left > sx)) g.cxp = z4;
        if (!(left > sy)) g.cyp = z4;
    }
    if (!(left > 4)) g.czhi = 0.f;
}

// kEagerRun (levels of at most kEagerCells cells, where a launch is one round of
// wavefronts bound by its chain of memory latencies): the gate, the diagonal
// and every operand are loaded at once and the launch leaves after them, on a
// closed gate or an inactive wavefront; else (large levels, bound by the bytes)
// before the operands' loads. kListRun (levels with a list of active chunks):
// as many blocks as run at once share the listed chunks, a
// wavefront one at a time; with a wavefront per chunk of the grid those of the
// inactive chunks have to be dispatched and to wait for a diagonal (256^3 pool,
// 26 % active: 61 us a first post-smoothing step, 43 so, the list's bytes at the
// copy rate being 31; its 128^3 level 11.8, 6.5 so).
enum FlatRun { kBytesRun, kEagerRun, kListRun };
// (wavefronts per SIMD the registers of a mode allow: blocks of a list run per CU)
constexpr int list_waves(int mode, bool any) { return (mode & SM_PROLONG) || any ? 7 : 8; }

template <int MODE, bool kRowsum, FlatRun kRun, bool kAny>
__global__ __launch_bounds__(kBlock, kRun == kListRun ? list_waves(MODE, kAny) : 1) void k_smooth_flat(
                                                        Dims d, Op32 A, const float *__restrict__ b,
                                                        const float *__restrict__ xin,
                                                        float *__restrict__ xout, float *dvec,
                                                        float cd, float cr,
                                                        const float *__restrict__ e, Dims dc,
                                                        const double *gate) {
    static_assert((MODE & SM_FIRST) == 0, "flat step: no fused first step");
    constexpr bool kProlong = (MODE & SM_PROLONG) != 0;
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    constexpr bool kEager = kRun == kEagerRun;
    static_assert(kRun != kListRun || !kRowsum, "no list where every cell is active");
    static_assert(!kAny || !kProlong, "the prolongation reads z rows of whole groups");
    const double stop = load_gate(gate, A.diag);
    const unsigned n = (unsigned)d.cells();  // below 2^32
    auto group = [&](unsigned ct) {  // the group of cells from ct on
        const bool on = ct < n;
        const unsigned c = on ? ct : (n - 1) & ~3u;
        const bool rs = kRowsum && rowsum_group<kAny>(c, d);  // every group there has an active cell
        f4 dg = {0.f, 0.f, 0.f, 0.f};
        if (!rs) dg = own_cells<kAny>(A.diag, c, n);
        if constexpr (kRun == kBytesRun) {
            if (stop != 0.0) return;
            const bool act = on && (rs || dg.x > 0.f || dg.y > 0.f || dg.z > 0.f || dg.w > 0.f);
            if (!__any(act)) return;
        }
        GroupOperands g = load_operands<kAny>(A, b, xin, d, c);
        f4 dprev = {0.f, 0.f, 0.f, 0.f};
        if constexpr ((MODE & SM_READ_D) != 0) dprev = own_cells<kAny>(dvec, c, n);
        f2 ec, e_xm, e_xp, e_ym, e_yp;
        float ezlo = 0.f, ezhi = 0.f;
        if constexpr (kProlong) {
            // (i, j, k) of the first cell (z rows of whole groups)
            const unsigned t = c / (unsigned)d.nz;
            const int k = (int)(c - t * (unsigned)d.nz);
            const unsigned iu = t / (unsigned)d.ny;
            const int i = (int)iu, j = (int)(t - iu * (unsigned)d.ny);
            // coarse values of the group's two coarse cells in this row and in the
            // neighbouring rows and planes (16-byte aligned groups: k >> 1 even)
            const int kc = k >> 1, jl = max(j - 1, 0) >> 1, jh = min(j + 1, d.ny - 1) >> 1, il = max(i - 1, 0) >> 1,
                      ih = min(i + 1, d.nx - 1) >> 1;
            auto e2 = [&](int ii, int jj) { return *(const f2 *)(e + dc.idx(ii, jj, kc)); };
            ec = e2(i >> 1, j >> 1);
            e_xm = e2(il, j >> 1);
            e_xp = e2(ih, j >> 1);
            e_ym = e2(i >> 1, jl);
            e_yp = e2(i >> 1, jh);
            ezlo = e[dc.idx(i >> 1, j >> 1, max(kc - 1, 0))];
            ezhi = e[dc.idx(i >> 1, j >> 1, min(kc + 2, dc.nz - 1))];
        }
        if constexpr (kEager) {
            pin(g);
            sfp::pin(dg);
            if constexpr ((MODE & SM_READ_D) != 0) sfp::pin(dprev);
            if constexpr (kProlong) {
                for (const f2 &v : {ec, e_xm, e_xp, e_ym, e_yp}) sfp::pin(v);
                sfp::pin(ezlo);
                sfp::pin(ezhi);
            }
            if (stop != 0.0) return;
        }
        end_cells<kAny>(g, d, c);
        if (rs) dg = rowsum_diag4(g.cx, g.cxp, g.cy, g.cyp, g.cz, g.czhi);
        const f4 xin_c = g.xc;
        if constexpr (kProlong) {
    #pragma unroll
            for (int q = 0; q < 4; q++) {
                g.xc[q] = g.xc[q] + ec[q >> 1];
                g.xm[q] = g.xm[q] + e_xm[q >> 1];
                g.xp[q] = g.xp[q] + e_xp[q >> 1];
                g.ym[q] = g.ym[q] + e_ym[q >> 1];
                g.yp[q] = g.yp[q] + e_yp[q >> 1];
            }
            g.zlo = g.zlo + ezlo;
            g.zhi = g.zhi + ezhi;
        }
        f4 xo, dno;
    #pragma unroll
        for (int q = 0; q < 4; q++) {
            const float xzm = q > 0 ? g.xc[q - 1] : g.zlo;
            const float xzp = q < 3 ? g.xc[q + 1] : g.zhi;
            const float czp = q < 3 ? g.cz[q + 1] : g.czhi;
            float off = fmaf(g.cx[q], g.xm[q], g.cxp[q] * g.xp[q]);
            off = fmaf(g.cy[q], g.ym[q], off);
            off = fmaf(g.cyp[q], g.yp[q], off);
            off = fmaf(g.cz[q], xzm, off);
            off = fmaf(czp, xzp, off);
            // centre iterate: the coarse correction only lands on active cells
            const float x0 = (kProlong && !(dg[q] > 0.f)) ? xin_c[q] : g.xc[q];
            const float r = g.b[q] - fmaf(dg[q], x0, -off);
            const float dp = (MODE & SM_XFIRST) != 0 ? x0 : dprev[q];
            const float dn = fmaf(cd, dp, cr * rcp_or_zero(dg[q]) * r);
            xo[q] = x0 + dn;
            dno[q] = dn;
        }
        if (!on) return;
        store_cells<kAny>(xout, c, n, xo);
        if constexpr ((MODE & SM_WRITE_D) != 0) store_cells<kAny>(dvec, c, n, dno);
    };
    if constexpr (kRun == kListRun) {
        if (stop != 0.0) return;
        const unsigned units = A.chunks.list[0], waves = flat_waves();
        for (unsigned u = flat_wave(); u < units; u += waves) group(list_cell<4>(A.chunks.list, u));
    } else {
        group(blockIdx.x * kSmoothFlatCells + 4 * (unsigned)flat_tid());
    }
}

// Two passes over the grid in one (temporal blocking). Step A is a
// Chebyshev step from iterate x1 and direction d1:
//   d2 = cdA d1 + crA D^{-1} (b - A x1),   x2 = x1 + d2.
// Step B is, with kRestrict false, a second Chebyshev step
//   x3 = x2 + cdB d2 + crB D^{-1} (b - A x2)   (written to xo; d2 not stored),
// and with kRestrict true the restriction of the residual of x2,
//   bc = R (b - A x2)   (x2 written to xo),
// with the per-cell arithmetic of the separate launches (k_smooth_flat with
// SM_READ_D | SM_WRITE_D, then SM_READ_D; or with SM_READ_D, then
// k_restrict_flat), so results agree bit for bit.
//
// A block of 64 lanes (z) x kPairRows wavefronts (y) marches over x planes,
// computing x2 on its whole 64 x kPairRows tile one plane ahead of step B;
// the rows exchange x2 through LDS, and step B covers the tile's interior
// (lanes 1..62, rows 1..kPairRows-2), so adjacent tiles overlap by one cell
// on each side. The interior starts on even z, y and x and has even extents,
// so each coarse cell's 8 children lie in one block: z pairs through the lane
// pair, y pairs through LDS, x pairs in a register. A wavefront whose row is
// inactive on a plane skips its work there (x2 there is 0, as the buffers
// already hold). xo must not alias x1.
//
// LDS holds x2 (and cpl_y) of three consecutive planes: the one barrier per
// plane then also separates a plane's reads from the store that reuses its
// buffer (issued two planes later, by a wavefront at most one barrier ahead).
constexpr int kPairRows = 16;
constexpr int kPairZ = 62, kPairY = kPairRows - 2;  // interior extents (tile strides)

template <bool kRestrict, bool kRowsum>
__global__ __launch_bounds__(64 * kPairRows, 8) void k_smooth_pair(
    CellGrid cg, Dims d, Op32 A, const float *__restrict__ b, const float *__restrict__ x1,
    float *__restrict__ xo, const float *__restrict__ d1, float cdA, float crA, float cdB,
    float crB, Dims dc, float *__restrict__ bc, const double *gate) {
    if (gated(gate)) return;
    __shared__ float sx2[3][kPairRows][64];
    __shared__ float scy[3][kPairRows][64];  // cpl_y of the same three planes
    __shared__ float sres[kRestrict ? kPairRows : 1][64];
    // Blocks go to the 8 XCDs in turn (block b to XCD b % 8); renumbered so
    // that each XCD takes a contiguous run of tiles, the rows, planes and
    // cache lines that neighbouring tiles share are read into one L2 (the
    // tiles overlap, and their z extents are not line-aligned). A tail of
    // fewer than 8 blocks keeps its numbers.
    unsigned L = blockIdx.x;
    {
        const unsigned q = gridDim.x / 8;
        if (L < 8 * q) L = (L % 8) * q + L / 8;
    }
    const unsigned per = cg.gx * cg.gy;
    const unsigned bx = L / per, rem = L - bx * per;
    const unsigned by = rem / cg.gx, bz = rem - by * cg.gx;
    const int lane = threadIdx.x, row = threadIdx.y;
    const int k = (int)bz * kPairZ - 1 + lane;
    const int j = (int)by * kPairY - 1 + row;
    const int i0 = (int)bx * cg.planes;
    if (i0 >= d.nx) return;  // uniform over the block
    const int ie = min(i0 + cg.planes, d.nx);
    const bool on = k >= 0 && k < d.nz && j >= 0 && j < d.ny;
    const bool interior = on && lane >= 1 && lane <= kPairZ && row >= 1 && row <= kPairY;
    const bool zlo = k > 0, zhi = k + 1 < d.nz, ylo = on && j > 0, yhi = on && j + 1 < d.ny;
    const Strides s(d);
    const size_t c0 = on ? d.idx(0, j, k) : 0;  // cell (i, j, k) = c0 + i sx when on

    // one plane of step A, kept for step B. Step B takes the couplings of the
    // upper faces from where they are stored: cpl_x(i+1) from the next
    // plane, cpl_y(j+1) from the next row (LDS), cpl_z(k+1) from the next
    // lane; where that cell is inactive the coupling is 0 either way.
    struct Plane {
        float x2, d2, dg, bc, cxc, cym, czm;
        bool live;
    };
    // step-A pipeline for the next plane q: x1 at q-1 and q, cpl_x at q
    float xm = 0.f, xc = 0.f, cxc = 0.f;
    bool primed = false;
    auto step_a = [&](int q) -> Plane {
        Plane P{};
        if (q >= d.nx) return P;
        const size_t c = c0 + q * s.sx;
        // a row-sum diagonal is rebuilt below (cells 1, nz and nz*ny read it)
        const bool rs = kRowsum && (on & (c != 1) & (c != (size_t)d.nz) & (c != s.sx));
        float dg = (on && !rs) ? A.diag[c] : 0.f;
        P.live = __any(on && (rs || dg > 0.f));
        if (!P.live) {
            primed = false;
            return P;
        }
        if (!primed) {
            xm = (on && q > 0) ? x1[c - s.sx] : 0.f;
            xc = on ? x1[c] : 0.f;
            cxc = on ? A.cpl[0][c] : 0.f;
            primed = true;
        }
        const bool up = q + 1 < d.nx;
        const float xp = (on && up) ? x1[c + s.sx] : 0.f;
        const float cxp = (on && up) ? A.cpl[0][c + s.sx] : 0.f;
        const float czm = on ? A.cpl[2][c] : 0.f;
        const float cym = ylo ? A.cpl[1][c] : 0.f;
        const float xym = ylo ? x1[c - s.sy] : 0.f;
        const float cyp = yhi ? A.cpl[1][c + s.sy] : 0.f;
        const float xyp = yhi ? x1[c + s.sy] : 0.f;
        const float bc = on ? b[c] : 0.f;
        const float dprev = on ? d1[c] : 0.f;
        float xzm = __shfl_up(xc, 1, 64);
        float xzp = __shfl_down(xc, 1, 64);
        float czp = __shfl_down(czm, 1, 64);
        if (lane == 0) xzm = (on && zlo) ? x1[c - 1] : 0.f;
        if (lane == 63) {
            xzp = (on && zhi) ? x1[c + 1] : 0.f;
            czp = (on && zhi) ? A.cpl[2][c + 1] : 0.f;
        }
        if (rs) dg = rowsum_diag(cxc, cxp, cym, cyp, czm, czp);
        if (on) {
            float off = fmaf(cxc, xm, cxp * xp);
            if (j > 0) off = fmaf(cym, xym, off);
            if (j + 1 < d.ny) off = fmaf(cyp, xyp, off);
            if (zlo) off = fmaf(czm, xzm, off);
            if (zhi) off = fmaf(czp, xzp, off);
            const float r = bc - fmaf(dg, xc, -off);
            const float dn = fmaf(cdA, dprev, crA * rcp_or_zero(dg) * r);
            P.x2 = xc + dn;
            if constexpr (kRestrict) {
                if (interior) xo[c] = P.x2;
            } else {
                P.d2 = dn;
            }
        }
        P.dg = dg;
        P.bc = bc;
        P.cxc = cxc;
        P.cym = cym;
        P.czm = czm;
        xm = xc;
        xc = xp;
        cxc = cxp;
        return P;
    };

    Plane pm{}, pc{};  // x2 at planes i - 1 and i
    if (i0 > 0) pm = step_a(i0 - 1);
    pc = step_a(i0);
    int bcur = i0 % 3;  // LDS buffer of plane i
    sx2[bcur][row][lane] = pc.x2;
    scy[bcur][row][lane] = pc.cym;
    float acc = 0.f;  // restriction: sum over the x pair
    // the lane of each coarse cell's first child stores the sum
    const bool writer = kRestrict && interior && (k & 1) == 0 && (j & 1) == 0;
    const size_t bco = writer ? dc.idx(0, j >> 1, k >> 1) : 0;
    const size_t dcsx = (size_t)dc.ny * dc.nz;
    for (int i = i0; i < ie; i++) {
        const int bnext = bcur == 2 ? 0 : bcur + 1;  // buffer of plane i + 1
        const Plane pn = step_a(i + 1);
        sx2[bnext][row][lane] = pn.x2;
        scy[bnext][row][lane] = pn.cym;
        __syncthreads();
        const float cxp = pn.cxc;
        const float czp = __shfl_down(pc.czm, 1, 64);  // lane 63 is never interior
        if constexpr (!kRestrict) {
            if (pc.live) {
                const float xzm = __shfl_up(pc.x2, 1, 64);
                const float xzp = __shfl_down(pc.x2, 1, 64);
                if (interior) {
                    const float xym = sx2[bcur][row - 1][lane];
                    const float xyp = sx2[bcur][row + 1][lane];
                    const float cyp = scy[bcur][row + 1][lane];
                    float off = fmaf(pc.cxc, pm.x2, cxp * pn.x2);
                    if (j > 0) off = fmaf(pc.cym, xym, off);
                    if (j + 1 < d.ny) off = fmaf(cyp, xyp, off);
                    if (zlo) off = fmaf(pc.czm, xzm, off);
                    if (zhi) off = fmaf(czp, xzp, off);
                    const float r = pc.bc - fmaf(pc.dg, pc.x2, -off);
                    const float dn = fmaf(cdB, pc.d2, crB * rcp_or_zero(pc.dg) * r);
                    xo[c0 + i * s.sx] = pc.x2 + dn;
                }
            }
        } else {
            // residual of x2 on the interior's active cells (the operand
            // order of k_restrict_flat), then the 2 x 2 x 2 sums
            float r = 0.f;
            if (pc.live) {
                const float xzm = __shfl_up(pc.x2, 1, 64);
                const float xzp = __shfl_down(pc.x2, 1, 64);
                if (interior && pc.dg > 0.f) {
                    const float xym = sx2[bcur][row - 1][lane];
                    const float xyp = sx2[bcur][row + 1][lane];
                    const float cyp = scy[bcur][row + 1][lane];
                    float off = 0.f;
                    if (i > 0) off = fmaf(pc.cxc, pm.x2, off);
                    if (i + 1 < d.nx) off = fmaf(cxp, pn.x2, off);
                    if (j > 0) off = fmaf(pc.cym, xym, off);
                    if (j + 1 < d.ny) off = fmaf(cyp, xyp, off);
                    if (zlo) off = fmaf(pc.czm, xzm, off);
                    if (zhi) off = fmaf(czp, xzp, off);
                    r = pc.bc - fmaf(pc.dg, pc.x2, -off);
                }
            }
            r += __shfl_down(r, 1, 64);  // z pair: lanes of even k take k + 1
            sres[row][lane] = r;
            __syncthreads();
            if (row < kPairRows - 1) r += sres[row + 1][lane];  // y pair (rows of even j)
            acc += r;                                             // x pair
            if ((i & 1) == 1 || i + 1 == d.nx) {
                if (writer) bc[bco + (size_t)(i >> 1) * dcsx] = acc;
                acc = 0.f;
            }
        }
        pm = pc;
        pc = pn;
        bcur = bnext;
    }
}

// The same pair of steps (step A, then step B with kRestrict false) on grids
// whose z rows hold at most 256 cells, in groups of four: a lane holds four
// consecutive cells of a z row (16-byte accesses), a wavefront a whole row or
// two, a block kRows rows of y, and the block marches over its run of x
// planes. Tiles overlap by one row on each side in y (rows 0 and
// kRows - 1 are step A's halo) and not at all in z. The per-cell
// arithmetic is k_smooth_flat's (two launches: SM_READ_D | SM_WRITE_D, or
// SM_XFIRST | SM_WRITE_D when d1 is x1 (kDx), then SM_READ_D), bit for bit.
//
// Each iteration of the march, for plane i:
//   1. puts x1, cpl_x and cpl_y of plane i + 2 (loaded kEarlyAhead - 2
//      iterations earlier) in LDS, with the out-of-tile rows next to the tile;
//   2. issues the loads of x1, cpl_x, cpl_y of plane i + kEarlyAhead and of
//      cpl_z, b, d1 and the diagonal of plane i + kRestAhead;
//   3. computes step A on plane i + 1 (x1 of the rows above and below and
//      their cpl_y from LDS) and puts x2 in LDS; one barrier;
//   4. computes step B on plane i (x2 of the three planes and of the rows
//      above and below from LDS) and stores it on the tile's interior rows.
// LDS rings: x1 two planes deep (written an iteration before it is read, and
// rewritten only after the next barrier), x2 three (written before the
// barrier that precedes its readers, which a wavefront one barrier ahead must
// not disturb), cpl_y four (read by step A in one iteration and by step B
// in the next) and cpl_x three (read by the wavefront that wrote it only).
// `rowact` (null: every row active) marks the (plane, row) z rows holding an
// active cell: the others load nothing and stay 0, as the vectors hold there.
//
// One block per CU (152 KB of LDS, 160 registers) has to keep enough loads in
// flight for its share of the memory's rate: what bounds it is their latency.
// 256^3, every row active: 94 us a pair (28 B per cell) and 87 with d1 = x1
// (24 B), 5.1-5.5 TB/s with the rows read twice; 110 and 108 with the loads
// behind branches and one plane ahead, 99 and 94 one plane ahead.
//
// kSub: z rows a wavefront holds, each in 64 / kSub lanes (2 where rows hold at
// most 128 cells). 128^3: 20 us a pair, 22 with a row a wavefront and half its
// lanes idle, two flat steps 23; runs of 4 planes a block, so the loads of the
// two planes around them and the first step's latency are half of it. Listed
// levels (pressure, 128^3, 26 % of the rows active) keep their flat steps: 13
// us for two, 20-23 a pair.
constexpr int kRowPairWaves = 12;
constexpr int row_pair_y(int sub) { return kRowPairWaves * sub - 2; }  // interior rows: the tiles' stride in y
// A byte offset past every run's planes; two of them add up without wrapping.
constexpr unsigned kPairOut = 0x40000000u;

template <bool kRowsum, bool kDx, int kSub>
__global__ __launch_bounds__(64 * kRowPairWaves, 1) void k_smooth_pair_rows(
    Dims d, Op32 A, const float *__restrict__ b, const float *__restrict__ x1,
    float *__restrict__ xo, const float *__restrict__ d1, float cdA, float crA, float cdB,
    float crB, const unsigned char *__restrict__ rowact, const int *__restrict__ segments, int planes,
    unsigned ytiles, const double *gate) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    if (gated(gate)) return;
    constexpr int kLanes = 64 / kSub, kRows = kRowPairWaves * kSub, kRowsY = row_pair_y(kSub);
    // the out-of-tile rows take one value per thread: 3 parts of 4 kLanes z values
    constexpr int kHaloWaves = 4 / kSub;
    static_assert(3 * kHaloWaves <= kRowPairWaves, "too few wavefronts for the halo rows");
    const unsigned runs = segments ? (unsigned)segments[0] : gridDim.x;
    if (blockIdx.x >= runs) return;
    __shared__ f4 sx1[2][kRows + 2][kLanes];  // x1 of rows -1 .. kRows (index row + 1)
    __shared__ f4 scy[4][kRows + 1][kLanes];  // cpl_y of rows 0 .. kRows
    __shared__ f4 sx2[3][kRows][kLanes];      // x2 of rows 0 .. kRows - 1
    // the stored diagonal of lane 0's group on planes 0 and 1: a row-sum
    // diagonal is rebuilt but in the groups of cells 1, nz and nz*ny
    __shared__ f4 sdg[2][kRowsum ? kRows : 1];
    __shared__ f4 scx[3][kRows][kLanes];      // cpl_x, read by the wavefront that wrote it
    // logical tiles run y fastest; each XCD (block b goes to XCD b % 8) takes
    // a contiguous run of them, so the rows two tiles share meet in one L2
    unsigned L = blockIdx.x;
    {
        const unsigned q = runs / 8;
        if (L < 8 * q) L = (L % 8) * q + L / 8;
    }
    unsigned by = L % ytiles;
    int i0 = (int)(L / ytiles) * planes, ie = min(i0 + planes, d.nx);
    if (segments) {
        by = (unsigned)segments[1 + 3 * L];
        i0 = segments[2 + 3 * L];
        ie = segments[3 + 3 * L];
    }
    if (i0 >= d.nx) return;  // uniform over the block
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.y), wlane = threadIdx.x;
    const int lane = wlane % kLanes, sub = kSub > 1 ? wlane / kLanes : 0, row = kSub * wave + sub;
    const int k = 4 * lane;
    const int j = (int)by * kRowsY - 1 + row;
    const bool zon = k < d.nz;
    const bool yin = j >= 0 && j < d.ny;
    const bool interior = row >= 1 && row <= kRowsY;
    const bool ylo = j > 0, yhi = j + 1 < d.ny;
    const bool zl = k > 0, zh = k + 4 < d.nz;
    const Strides s(d);
    // element offsets fit 32 bits (the launcher keeps cells() < 2^32); lanes
    // past the row's end read its last group (a cache hit) and drop it
    const unsigned c0 = yin ? (unsigned)d.idx(0, j, min(k, d.nz - 4)) : 0u;
    const unsigned sx = (unsigned)s.sx;
    // Every load is a buffer load over planes p0 .. of the run, issued on every
    // row and lane: one that has nothing to load (an inactive row, a plane
    // outside, a lane past the row) passes an offset past the buffer, which
    // reads 0 and moves nothing. (Behind branches, or with a select on what
    // they loaded, the loads were waited for where they were issued: the
    // compiler cannot count those in flight. 256^3: 110 us a pair so.)
    const int p0 = max(i0 - 2, 0);
    const unsigned plane_bytes = 4 * sx;
    const unsigned run_bytes = (unsigned)(min(ie + 6, d.nx) - p0) * plane_bytes;  // (< kPairOut)
    auto rsrc = [&](const float *p) { return buf_rsrc(p + (size_t)p0 * sx, run_bytes); };
    const auto rx1 = rsrc(x1), rcx = rsrc(A.cpl[0]), rcy = rsrc(A.cpl[1]), rcz = rsrc(A.cpl[2]), rb = rsrc(b),
               rd1 = rsrc(d1), rdg = rsrc(A.diag), rxo = rsrc(xo);
    const unsigned o0 = yin && zon ? 4 * c0 : kPairOut;  // bytes within a plane
    // the out-of-tile rows next to the tile (x1 of rows j0 - 1 and
    // j0 + kRows - 2, cpl_y of the latter), one value per thread: thread
    // t of the block takes z = t mod 256 of part t / 256
    const int hpart = wave / kHaloWaves, hz = wave % kHaloWaves * 64 + wlane;
    const int jt = (int)by * kRowsY - 1;  // the tile's row 0
    const int jh = hpart == 0 ? jt - 1 : jt + kRows;
    const bool hon_any = hpart < 3 && jh >= 0 && jh < d.ny;  // uniform over the wavefront
    const unsigned oh = hon_any && hz < d.nz ? 4 * (unsigned)d.idx(0, jh, hz) : kPairOut;
    const f4 z4 = {0.f, 0.f, 0.f, 0.f};
    // activity of this row and of the out-of-tile row for planes i0 - 2 ..
    // i0 + 61 (bit q - i0 + 2), one lane per plane, read once
    auto row_mask = [&](int jj) -> unsigned long long {
        const int q = i0 - 2 + wlane;
        const bool a = q >= 0 && q < d.nx && q <= ie + 1 && jj >= 0 && jj < d.ny &&
                       (!rowact || rowact[(size_t)q * d.ny + jj] != 0);
        return __ballot(a);
    };
    // (of the wavefront's rows: its first and, kSub 2, its second)
    const int jw = (int)by * kRowsY - 1 + kSub * wave;
    const unsigned long long amask = row_mask(jw), amask2 = kSub > 1 ? row_mask(jw + 1) : 0ull;
    const unsigned long long hmask_lo = row_mask(jt - 1), hmask_hi = row_mask(jt + kRows);
    const unsigned long long hmask = hpart == 0 ? hmask_lo : hmask_hi;
    auto active = [&](int q, unsigned long long m) { return ((m >> (q - i0 + 2)) & 1ull) != 0; };
    auto mine = [&](int q) { return sub ? active(q, amask2) : active(q, amask); };
    auto any_active = [&](int q) { return active(q, amask | amask2); };
    auto at_row = [&](int q) {
        const unsigned o = active(q, amask) ? (unsigned)(q - p0) * plane_bytes : kPairOut;
        if constexpr (kSub == 1) return o;
        const unsigned o2 = active(q, amask2) ? (unsigned)(q - p0) * plane_bytes : kPairOut;
        return sub ? o2 : o;
    };
    auto at = [&](int q, unsigned long long m) { return active(q, m) ? (unsigned)(q - p0) * plane_bytes : kPairOut; };
    auto ld = [&](__amdgpu_buffer_rsrc_t p, unsigned o) {
        return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(p, o0 + o, 0, 0));
    };

    struct Early {
        f4 x, cx, cy;  // x1, cpl_x, cpl_y
        float h;       // this thread's value of the out-of-tile rows
    };
    struct Rest {
        f4 cz, bv, dv, dg;
    };
    auto load_early = [&](int q) {
        Early e;
        const unsigned o = at_row(q);
        e.x = ld(rx1, o);
        e.cx = ld(rcx, o);
        e.cy = ld(rcy, o);
        e.h = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(hpart == 2 ? rcy : rx1,
                                                                             oh + at(q, hmask), 0, 0));
        return e;
    };
    auto load_rest = [&](int q) {
        Rest r;
        const unsigned o = at_row(q);
        r.cz = ld(rcz, o);
        r.bv = ld(rb, o);
        r.dv = r.dg = z4;
        if constexpr (!kDx) r.dv = ld(rd1, o);
        if constexpr (!kRowsum) r.dg = ld(rdg, o);
        return r;
    };
    auto put_early = [&](int q, const Early &e) {
        sx1[q & 1][row + 1][lane] = e.x;
        scy[q & 3][row][lane] = e.cy;
        scx[(q + 3) % 3][row][lane] = e.cx;
        if (hpart == 0) ((float *)&sx1[q & 1][0][0])[hz] = e.h;
        else if (hpart == 1) ((float *)&sx1[q & 1][kRows + 1][0])[hz] = e.h;
        else if (hpart == 2) ((float *)&scy[q & 3][kRows][0])[hz] = e.h;
    };
    // one Chebyshev step of the four cells at plane q from iterate xc (x
    // neighbours xm, xp; y neighbours and couplings given), direction dp
    auto cheb = [&](f4 xc, f4 xm, f4 xp, f4 xym, f4 xyp, f4 cxc, f4 cxp, f4 cym, f4 cyp, f4 cz,
                    f4 bv, f4 dg, f4 rdg, f4 dp, float cd, float cr, f4 &dn_out) {
        // every lane takes part in the shuffles: a lane outside the exec mask
        // does not supply its value to ds_bpermute (the reader gets 0)
        const float xzlo = __shfl_up(xc.w, 1, 64);
        const float xzhi = __shfl_down(xc.x, 1, 64);
        const float czdn = __shfl_down(cz.x, 1, 64);
        const float czhi = zh ? czdn : 0.f;
        f4 xo4;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float xzm = q > 0 ? xc[q - 1] : xzlo;
            const float xzp = q < 3 ? xc[q + 1] : xzhi;
            const float czp = q < 3 ? cz[q + 1] : czhi;
            float off = fmaf(cxc[q], xm[q], cxp[q] * xp[q]);
            if (ylo) off = fmaf(cym[q], xym[q], off);
            if (yhi) off = fmaf(cyp[q], xyp[q], off);
            if (q > 0 || zl) off = fmaf(cz[q], xzm, off);
            if (q < 3 || zh) off = fmaf(czp, xzp, off);
            const float r = bv[q] - fmaf(dg[q], xc[q], -off);
            const float dn = fmaf(cd, dp[q], cr * rdg[q] * r);
            xo4[q] = xc[q] + dn;
            dn_out[q] = dn;
        }
        return xo4;
    };
    // the diagonal at plane q: loaded, or rebuilt from the couplings
    auto diag_at = [&](int q, f4 cxc, f4 cxp, f4 cym, f4 cyp, const Rest &r) {
        f4 dg = r.dg;
        if constexpr (kRowsum) {
            const float czdn = __shfl_down(r.cz.x, 1, 64);  // all lanes (see cheb)
            const float czhi = zh ? czdn : 0.f;
            dg = rowsum_diag4(cxc, cxp, cym, cyp, r.cz, czhi);
            if (q <= 1 && jw <= 1) {  // uniform
                const f4 stored = sdg[q & 1][row];
                if (!rowsum_group(c0 + (unsigned)q * sx, d)) dg = stored;
            }
        }
        return dg;
    };
    // step A at plane q: x2 (returned) and d2; x1 of this row at planes q and
    // q + 1 is read back from LDS (this wavefront wrote it). Step B forms the
    // plane's diagonal and its reciprocal again from the same operands (bit
    // for bit the same values): carried in registers for an iteration they
    // made the kernel spill.
    auto step_a = [&](int q, f4 xm, const Rest &r, f4 &d2, f4 &xc) {
        const f4 cym = scy[q & 3][row][lane], cyp = scy[q & 3][row + 1][lane];
        const f4 cxc = scx[(q + 3) % 3][row][lane], cxp = scx[(q + 4) % 3][row][lane];
        const f4 dg = diag_at(q, cxc, cxp, cym, cyp, r);
        // (the FP64 row sums' registers are free again before x1 is read)
        if constexpr (kRowsum) __builtin_amdgcn_sched_barrier(0);
        xc = sx1[q & 1][row + 1][lane];
        const f4 xp = sx1[(q + 1) & 1][row + 1][lane];
        const f4 xym = sx1[q & 1][row][lane], xyp = sx1[q & 1][row + 2][lane];
        f4 rdg;
#pragma unroll
        for (int k = 0; k < 4; k++) rdg[k] = rcp_or_zero(dg[k]);
        d2 = z4;
        if (!any_active(q)) return z4;  // uniform over the wavefront
        f4 x2 = cheb(xc, xm, xp, xym, xyp, cxc, cxp, cym, cyp, r.cz, r.bv, dg, rdg, kDx ? xc : r.dv,
                     cdA, crA, d2);
        if (!zon || (kSub > 1 && !mine(q))) x2 = z4;
        return x2;
    };

    // ---- prologue: planes i0 - 1 and i0 through step A, plane i0 + 1 in LDS
    // E: planes i + 2 and i + 3 in flight, by the parity of i - i0; R: planes i
    // and i + 1 and, in flight, i + 2, by their distance from i0 mod 4; D: the
    // direction of planes i and i + 1 from step A. (The march is unrolled by
    // four, so every index is a constant and nothing in flight is copied.)
    // (three planes ahead for R beside the diagonal, or four for E beside d1, spills)
    constexpr int kEarlyAhead = kDx ? 4 : 3, kRestAhead = kRowsum ? 3 : 2;
    if constexpr (kRowsum) {
        if (i0 <= 2 && yin && j <= 1 && lane == 0)
            for (int q = 0; q < min(2, d.nx); q++) sdg[q][row] = *(const f4 *)(A.diag + c0 + (size_t)q * sx);
    }
    Early E[2];
    Rest R[4];
    f4 D[2];
    const f4 xpre = load_early(i0 - 2).x;
    const Early em = load_early(i0 - 1), e0 = load_early(i0), e1 = load_early(i0 + 1);
    R[3] = load_rest(i0 - 1);
    R[0] = load_rest(i0);
    E[0] = load_early(i0 + 2);
    R[1] = load_rest(i0 + 1);
    if constexpr (kEarlyAhead == 4) E[1] = load_early(i0 + 3);
    if constexpr (kRestAhead == 3) R[2] = load_rest(i0 + 2);
    // step A at i0 - 1 reads planes i0 - 1 and i0 from the x1 ring, step A at
    // i0 planes i0 and i0 + 1 (which takes the buffer of i0 - 1)
    put_early(i0 - 1, em);
    put_early(i0, e0);
    __syncthreads();
    f4 xa, xb;  // x1 at planes i and i + 1 (this row)
    f4 x2prev = step_a(i0 - 1, xpre, R[3], D[0], xa);  // x2 at plane i - 1 (this row)
    __syncthreads();
    put_early(i0 + 1, e1);
    __syncthreads();
    {
        const f4 x2c = step_a(i0, xa, R[0], D[0], xb);
        sx2[(i0 + 2) % 3][row][lane] = x2prev;  // (i0 - 1) mod 3
        sx2[i0 % 3][row][lane] = x2c;
    }
    xa = xb;
    __syncthreads();
    auto iter = [&](auto Uc, int i) {
        constexpr int U = decltype(Uc)::value;
        // 1. what was loaded two iterations ago: x1 and the couplings of plane
        // i + 2 into LDS
        put_early(i + 2, E[U & 1]);
        // 2. loads into registers just read, in flight for two iterations
        E[(U + kEarlyAhead) & 1] = load_early(i + kEarlyAhead);
        R[(U + kRestAhead) & 3] = load_rest(i + kRestAhead);
        // 3. step A on plane i + 1
        const f4 x2n = step_a(i + 1, xa, R[(U + 1) & 3], D[(U + 1) & 1], xb);
        sx2[(i + 1) % 3][row][lane] = x2n;
        __syncthreads();
        // 4. step B on plane i (the tile's interior rows)
        if (kSub > 1 || interior) {
            const int bi = i % 3;
            const f4 xc = sx2[bi][row][lane];
            if (any_active(i)) {
                const Rest &r = R[U];
                const int rb = kSub > 1 ? max(row - 1, 0) : row - 1, ra = kSub > 1 ? min(row + 1, kRows - 1) : row + 1;
                const f4 xym = sx2[bi][rb][lane], xyp = sx2[bi][ra][lane];
                const f4 cym = scy[i & 3][row][lane], cyp = scy[i & 3][row + 1][lane];
                const f4 cxc = scx[bi][row][lane], cxp = scx[(i + 1) % 3][row][lane];
                const f4 dgB = diag_at(i, cxc, cxp, cym, cyp, r);
                f4 rdgB;
#pragma unroll
                for (int k = 0; k < 4; k++) rdgB[k] = rcp_or_zero(dgB[k]);
                f4 dn;
                const f4 x3 = cheb(xc, x2prev, x2n, xym, xyp, cxc, cxp, cym, cyp, r.cz, r.bv, dgB, rdgB, D[U & 1],
                                   cdB, crB, dn);
                __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, x3), rxo,
                                                       kSub == 1 ? o0 + (unsigned)(i - p0) * plane_bytes
                                                                 : interior ? o0 + at_row(i) : kPairOut,
                                                       0, 0);
            }
            x2prev = xc;
        }
        xa = xb;
    };
    for (int i = i0; i < ie; i += 4) {  // uniform over the block
        iter(std::integral_constant<int, 0>{}, i);
        if (i + 1 >= ie) break;
        iter(std::integral_constant<int, 1>{}, i + 1);
        if (i + 2 >= ie) break;
        iter(std::integral_constant<int, 2>{}, i + 2);
        if (i + 3 >= ie) break;
        iter(std::integral_constant<int, 3>{}, i + 3);
    }
}

// x += P e on active cells (the piecewise-constant coarse correction), in
// place, before a plain first post-smoothing step: on large grids this pass
// and the step cost less than the step that adds the correction at every
// neighbour it reads (the coarse values' gathers cost a third of that step).
// Groups of four cells over the flat cell index, as k_smooth_flat; kList: of the
// listed chunks.
template <bool kList>
__global__ __launch_bounds__(kBlock) void k_prolong_add(Dims d, const unsigned *__restrict__ list,
                                                        const float *__restrict__ diag32,
                                                        const float *__restrict__ e, Dims dc,
                                                        float *__restrict__ x, const double *gate) {
    if (gated(gate)) return;
    const unsigned n = (unsigned)d.cells();
    auto group = [&](unsigned c) {
        if (c >= n) return;
        const f4v dg = own_cells<true>(diag32, c, n);
        if (!(dg.x > 0.f || dg.y > 0.f || dg.z > 0.f || dg.w > 0.f)) return;
        f4v v = own_cells<true>(x, c, n);
        const unsigned t = c / (unsigned)d.nz, iu = t / (unsigned)d.ny;
        int i = (int)iu, j = (int)(t - iu * (unsigned)d.ny), k = (int)(c - t * (unsigned)d.nz);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if (dg[q] > 0.f) v[q] = v[q] + e[dc.idx(i >> 1, j >> 1, k >> 1)];
            if (++k == d.nz) {  // the next row
                k = 0;
                if (++j == d.ny) {
                    j = 0;
                    i++;
                }
            }
        }
        store_cells<true>(x, c, n, v);
    };
    if constexpr (kList) {
        const unsigned units = list[0], waves = flat_waves();
        for (unsigned u = flat_wave(); u < units; u += waves) group(list_cell<4>(list, u));
    } else {
        group(blockIdx.x * kSmoothFlatCells + 4 * (unsigned)flat_tid());
    }
}

// Residual b - A x on the fine grid, summed over each coarse cell's (up to 8)
// children, over the flat cell index: a wavefront covers 64 cells of a z row in
// two rows and two planes, four cells per lane (lanes 0-15: row j, plane i;
// 16-31: row j+1; 32-63: plane i+1). The children are added as the z pairs (in
// the lane), the y pairs (across lanes 16 apart) and the x pair (32 apart) onto
// a zero, and the first 16 lanes store two coarse values each. A residual's
// off-diagonal sum has the order x-, x+, y-, y+, z-, z+, one fmaf each. A
// wavefront whose 256 cells are all inactive only
// stores zeros.
constexpr int kRestrictFlatZ = 64;  // z cells per wavefront

template <bool kRowsum, bool kEager, bool kList, bool kAny>
__global__ __launch_bounds__(kBlock) void k_restrict_flat(Dims df, Op32 A, const float *__restrict__ b,
                                                          const float *__restrict__ x, Dims dc,
                                                          float *__restrict__ bc, float *__restrict__ x0c,
                                                          const float *__restrict__ diag32c, float c0,
                                                          const double *gate) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    const double stop = load_gate(gate, A.diag);
    const int lane = threadIdx.x & 63;
    unsigned wave = flat_wave();
    if constexpr (kList) {  // (an inactive coarse cell's values are 0 already)
        if (stop != 0.0 || wave >= A.chunks.quads[0]) return;
        wave = A.chunks.quads[1 + wave];
    }
    const unsigned zch = (unsigned)(df.nz + kRestrictFlatZ - 1) / kRestrictFlatZ;
    const unsigned yp = (unsigned)(df.ny + 1) / 2;
    const unsigned kz = wave % zch, t = wave / zch;
    const unsigned jp = t % yp, ip = t / yp;
    if (ip >= (unsigned)(df.nx + 1) / 2) return;  // uniform over the wavefront (no barriers follow)
    const int iw = 2 * (int)ip + (lane >> 5), jw = 2 * (int)jp + ((lane >> 4) & 1);
    const int kw = kRestrictFlatZ * (int)kz + 4 * (lane & 15);
    const bool on = iw < df.nx && jw < df.ny && kw < df.nz;
    // lanes outside the grid load the nearest cells and drop them
    const int i = min(iw, df.nx - 1), j = min(jw, df.ny - 1), k = min(kw, (df.nz - 1) & ~3);
    const unsigned c = (unsigned)df.idx(i, j, k), n = (unsigned)df.cells();
    const bool rs = kRowsum && rowsum_group<kAny>(c, df);  // every group there has an active cell
    f4 dg = {0.f, 0.f, 0.f, 0.f};
    if (!rs) dg = own_cells<kAny>(A.diag, c, n);
    f4 r = {0.f, 0.f, 0.f, 0.f};
    bool any = true;
    if constexpr (!kEager && !kList) {
        if (stop != 0.0) return;
        any = __any(on && (rs || dg.x > 0.f || dg.y > 0.f || dg.z > 0.f || dg.w > 0.f));
    }
    if (any) {
        GroupOperands g = load_operands<kAny>(A, b, x, df, c);
        if constexpr (kEager) {
            pin(g);
            sfp::pin(dg);
            if (stop != 0.0) return;
        }
        end_cells<kAny>(g, df, c);
        if (rs) dg = rowsum_diag4(g.cx, g.cxp, g.cy, g.cyp, g.cz, g.czhi);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const float xzm = q > 0 ? g.xc[q - 1] : g.zlo;
            const float xzp = q < 3 ? g.xc[q + 1] : g.zhi;
            const float czp = q < 3 ? g.cz[q + 1] : g.czhi;
            float off = fmaf(g.cx[q], g.xm[q], 0.f);
            off = fmaf(g.cxp[q], g.xp[q], off);
            off = fmaf(g.cy[q], g.ym[q], off);
            off = fmaf(g.cyp[q], g.yp[q], off);
            off = fmaf(g.cz[q], xzm, off);
            off = fmaf(czp, xzp, off);
            const float rr = g.b[q] - fmaf(dg[q], g.xc[q], -off);
            // (past the row: the next one's)
            r[q] = on && (!kAny || kw + q < df.nz) && dg[q] > 0.f ? rr : 0.f;
        }
    }
    float s0 = r.x + r.y, s1 = r.z + r.w;  // z pairs
    s0 += __shfl_xor(s0, 16);              // y pairs
    s1 += __shfl_xor(s1, 16);
    const float o0 = __shfl_xor(s0, 32), o1 = __shfl_xor(s1, 32);  // the other plane's
    if (lane < 16 && on) {
        f2 v;
        v.x = 0.f;
        v.x += s0;
        v.x += o0;
        v.y = 0.f;
        v.y += s1;
        v.y += o1;
        const size_t q = dc.idx((int)ip, (int)jp, k >> 1);
        if constexpr (!kAny) {
            *(f2 *)(bc + q) = v;
            if (x0c) {
                const f2 dgc = *(const f2 *)(diag32c + q);
                f2 x0;
                x0.x = c0 * rcp_or_zero(dgc.x) * v.x;
                x0.y = c0 * rcp_or_zero(dgc.y) * v.y;
                *(f2 *)(x0c + q) = x0;
            }
        } else {
#pragma unroll
            for (int h = 0; h < 2; h++)
                if ((k >> 1) + h < dc.nz) {
                    bc[q + h] = v[h];
                    if (x0c) x0c[q + h] = c0 * rcp_or_zero(diag32c[q + h]) * v[h];
                }
        }
    }
}

// Zeros the level vectors (and, if given, one FP64 vector of the first
// level) at the inactive cells (FP32 diagonal 0): a new operator may make
// inactive cells that were unknowns before, and the values left there would
// survive in the groups of inactive cells the stencil kernels skip. Active
// cells are written before they are read in every cycle, so they need no
// clearing. Every level in one launch (the small levels' launches would each
// cost more than their bytes), one cell per lane (consecutive lanes,
// consecutive cells: the sparse stores stay coalesced).
__global__ __launch_bounds__(kBlock) void k_clear_inactive(ClearArgs a) {
    const unsigned gid = blockIdx.x * kBlock + threadIdx.x;
    if (gid >= a.start[a.nlev]) return;
    int l = 0;
    while (gid >= a.start[l + 1]) l++;
    const unsigned c = gid - a.start[l];
    if (a.diag32[l][c] > 0.f) return;
#pragma unroll
    for (int k = 0; k < 4; k++) a.v[l][k][c] = 0.f;
    if (l == 0 && a.w) a.w[c] = 0.0;
}

// Whether the assembly before the launch has formed rows (see RowsFlag; null:
// it has), which one thread tells the host.
__device__ __forceinline__ bool tell_rows(const RowsFlag &rows) {
    if (!rows.host) return true;
    const bool any = *rows.seen == rows.epoch;  // uniform
    if (blockIdx.x == 0 && flat_tid() == 0)
        __hip_atomic_store(rows.host, 2u * rows.epoch + (any ? 1u : 0u), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
    return any;
}

// Galerkin coarsening over the fine grid (the mapping of k_smooth): each
// fine cell forms its contributions to its aggregate -- the active cell's
// row sum diag - (its 6 couplings), its lower-face couplings where it lies on
// the aggregate's lower layer of an axis, its upper-face couplings where it
// lies on the upper layer -- and the 8 children are added pairwise (z through
// the lane pair, y through LDS, x over the block's plane pairs). Same operator
// as a per-aggregate loop over the children, up to the order of the sums.
// The coarse couplings are the summed ones times `scale`, the coarse diagonal
// the summed row sum times `rs_scale` plus the coarse couplings.
constexpr int kCoarsenSums = 8;  // row sum, 3 lower, 3 upper, active count

__global__ __launch_bounds__(kBlock) void k_coarsen_fine(CellGrid cg, Dims df, Op64 Af,
                                                         const float *__restrict__ diag32f, Dims dc,
                                                         double scale, double rs_scale, double *diag64c,
                                                         MutFaces cpl64c, float *diag32c,
                                                         float *cpl32c0, float *cpl32c1,
                                                         float *cpl32c2, RowsFlag rows) {
    if (!tell_rows(rows)) return;
    __shared__ double sh[kCoarsenSums][kBlock];
    int k, j, i0;
    cell_tile(cg, k, j, i0);
    const int tz = blockDim.x, lane = threadIdx.x, row = threadIdx.y;
    if (i0 >= df.nx) return;  // uniform over the block
    const bool on = k < df.nz && j < df.ny;
    const bool writer = on && (k & 1) == 0 && (j & 1) == 0;
    const Strides s(df);
    const int ie = min(i0 + cg.planes, df.nx);
    const int t = row * tz + lane;
    float *cpl32c[3] = {cpl32c0, cpl32c1, cpl32c2};
    double acc[kCoarsenSums];
#pragma unroll
    for (int q = 0; q < kCoarsenSums; q++) acc[q] = 0.0;
    for (int i = i0; i < ie; i++) {
        double v[kCoarsenSums];
#pragma unroll
        for (int q = 0; q < kCoarsenSums; q++) v[q] = 0.0;
        if (on) {
            const size_t c = df.idx(i, j, k);
            const bool up[3] = {i + 1 < df.nx, j + 1 < df.ny, k + 1 < df.nz};
            const double cl[3] = {Af.cpl[0][c], Af.cpl[1][c], Af.cpl[2][c]};
            const double cu[3] = {up[0] ? Af.cpl[0][c + s.sx] : 0.0, up[1] ? Af.cpl[1][c + s.sy] : 0.0,
                                  up[2] ? Af.cpl[2][c + 1] : 0.0};
            const int idx[3] = {i, j, k};
            if (diag32f[c] > 0.f) {
                double off = cl[0] + cl[1] + cl[2];
                if (up[0]) off += cu[0];
                if (up[1]) off += cu[1];
                if (up[2]) off += cu[2];
                v[0] = Af.diag[c] - off;
                v[7] = 1.0;
            }
#pragma unroll
            for (int a = 0; a < 3; a++) {
                if ((idx[a] & 1) == 0) v[1 + a] = cl[a];  // lower layer: the face below
                else v[4 + a] = cu[a];                     // upper layer: the face above
            }
        }
        if (tz > 1) {
#pragma unroll
            for (int q = 0; q < kCoarsenSums; q++) v[q] += __shfl_xor(v[q], 1, tz);  // z pair
        }
#pragma unroll
        for (int q = 0; q < kCoarsenSums; q++) sh[q][t] = v[q];
        __syncthreads();
        if ((row & 1) == 0) {
#pragma unroll
            for (int q = 0; q < kCoarsenSums; q++) v[q] += sh[q][t + tz];  // y pair
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kCoarsenSums; q++) acc[q] += v[q];  // x pair
        if ((i & 1) == 1 || i + 1 == df.nx) {
            if (writer) {
                const int I = i >> 1, J = j >> 1, K = k >> 1;
                const int IC[3] = {I, J, K};
                double lower[3], upper[3];
                for (int a = 0; a < 3; a++) {
                    lower[a] = IC[a] > 0 ? scale * acc[1 + a] : 0.0;
                    upper[a] = IC[a] + 1 < dc.n(a) ? scale * acc[4 + a] : 0.0;
                }
                const bool active = acc[7] > 0.0;
                const size_t cc = dc.idx(I, J, K);
                if (active) {
                    const double dg = rs_scale * acc[0] + lower[0] + upper[0] + lower[1] + upper[1] +
                                      lower[2] + upper[2];
                    diag64c[cc] = dg;
                    diag32c[cc] = dg > 0.0 ? (float)dg : 0.f;
                } else {
                    diag64c[cc] = 1.0;
                    diag32c[cc] = 0.f;
                }
                for (int a = 0; a < 3; a++) {
                    const double cv = active ? lower[a] : 0.0;
                    cpl64c.a[a][cc] = cv;
                    cpl32c[a][cc] = (float)cv;
                }
            }
#pragma unroll
            for (int q = 0; q < kCoarsenSums; q++) acc[q] = 0.0;
        }
    }
}

// The same coarsening over the flat cell index (grids with nz a multiple of
// 4), in k_restrict_flat's mapping: a wavefront covers 64 cells of a z row in
// two rows and two planes, four cells per lane (lanes 0-15: row j, plane i;
// 16-31: row j+1; 32-63: plane i+1). Each cell's contributions are
// k_coarsen_fine's, and the children are added in its order -- the z pair in
// the lane, the y pair across lanes 16 apart, the x pair across lanes 32
// apart onto a zero -- so the coarse operator is the same to the bit; the
// first 16 lanes store two coarse cells each.
__global__ __launch_bounds__(kBlock) void k_coarsen_flat(Dims df, Op64 Af, const float *__restrict__ diag32f,
                                                         Dims dc, double scale, double rs_scale,
                                                         double *diag64c, MutFaces cpl64c,
                                                         float *diag32c, float *cpl32c0, float *cpl32c1,
                                                         float *cpl32c2, RowsFlag rows) {
    if (!tell_rows(rows)) return;
    typedef double d2 __attribute__((ext_vector_type(2)));
    typedef float f4 __attribute__((ext_vector_type(4)));
    const int lane = threadIdx.x & 63;
    const unsigned wave = (unsigned)(blockIdx.x * kBlock + threadIdx.x) >> 6;
    const unsigned zch = (unsigned)(df.nz + 63) / 64;
    const unsigned yp = (unsigned)(df.ny + 1) / 2;
    const unsigned kz = wave % zch, t = wave / zch;
    const unsigned jp = t % yp, ip = t / yp;
    if (ip >= (unsigned)(df.nx + 1) / 2) return;  // uniform over the wavefront (no barriers follow)
    const int i = 2 * (int)ip + (lane >> 5), j = 2 * (int)jp + ((lane >> 4) & 1);
    const int k = 64 * (int)kz + 4 * (lane & 15);
    const bool on = i < df.nx && j < df.ny && k < df.nz;
    const Strides s(df);
    // v[h][q]: the sums of coarse z cell k / 2 + h (row sum, 3 lower, 3 upper, active count)
    double v[2][kCoarsenSums];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int q = 0; q < kCoarsenSums; q++) v[h][q] = 0.0;
    if (on) {
        const size_t c = df.idx(i, j, k);
        const bool upx = i + 1 < df.nx, upy = j + 1 < df.ny;
        auto ld4 = [&](const double *p, double (&o)[4]) {
            const d2 a = *(const d2 *)p, b = *(const d2 *)(p + 2);
            o[0] = a.x;
            o[1] = a.y;
            o[2] = b.x;
            o[3] = b.y;
        };
        double cl0[4], cl1[4], cl2[4], cu0[4] = {0.0, 0.0, 0.0, 0.0}, cu1[4] = {0.0, 0.0, 0.0, 0.0}, dg[4];
        ld4(Af.cpl[0] + c, cl0);
        ld4(Af.cpl[1] + c, cl1);
        ld4(Af.cpl[2] + c, cl2);
        if (upx) ld4(Af.cpl[0] + c + s.sx, cu0);
        if (upy) ld4(Af.cpl[1] + c + s.sy, cu1);
        const double cz4 = k + 4 < df.nz ? Af.cpl[2][c + 4] : 0.0;  // the face above the group
        ld4(Af.diag + c, dg);
        const f4 d32 = *(const f4 *)(diag32f + c);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int kq = k + q;
            const bool upz = kq + 1 < df.nz;
            const double cl[3] = {cl0[q], cl1[q], cl2[q]};
            const double cu[3] = {upx ? cu0[q] : 0.0, upy ? cu1[q] : 0.0,
                                  upz ? (q < 3 ? cl2[q + 1] : cz4) : 0.0};
            const bool upv[3] = {upx, upy, upz};
            const int idx[3] = {i, j, kq};
            double w[kCoarsenSums];
#pragma unroll
            for (int e = 0; e < kCoarsenSums; e++) w[e] = 0.0;
            if (d32[q] > 0.f) {
                double off = cl[0] + cl[1] + cl[2];
                if (upv[0]) off += cu[0];
                if (upv[1]) off += cu[1];
                if (upv[2]) off += cu[2];
                w[0] = dg[q] - off;
                w[7] = 1.0;
            }
#pragma unroll
            for (int a = 0; a < 3; a++) {
                if ((idx[a] & 1) == 0) w[1 + a] = cl[a];  // lower layer: the face below
                else w[4 + a] = cu[a];                     // upper layer: the face above
            }
            // the z pair: the even cell's sums first, then the odd cell's added
#pragma unroll
            for (int e = 0; e < kCoarsenSums; e++) v[q >> 1][e] = (q & 1) ? v[q >> 1][e] + w[e] : w[e];
        }
    }
    // y pair (the row-j lanes keep row j's sums first), then the x pair onto 0
    double acc[2][kCoarsenSums];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int e = 0; e < kCoarsenSums; e++) {
            const double y = v[h][e] + __shfl_xor(v[h][e], 16, 64);
            const double o = __shfl_xor(y, 32, 64);
            double a = 0.0;
            a += y;
            if (2 * (int)ip + 1 < df.nx) a += o;
            acc[h][e] = a;
        }
    if (lane < 16 && on) {
        float *cpl32c[3] = {cpl32c0, cpl32c1, cpl32c2};
        const int I = (int)ip, J = (int)jp;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int K = (k >> 1) + h;
            const int IC[3] = {I, J, K};
            double lower[3], upper[3];
            for (int a = 0; a < 3; a++) {
                lower[a] = IC[a] > 0 ? scale * acc[h][1 + a] : 0.0;
                upper[a] = IC[a] + 1 < dc.n(a) ? scale * acc[h][4 + a] : 0.0;
            }
            const bool active = acc[h][7] > 0.0;
            const size_t cc = dc.idx(I, J, K);
            if (active) {
                const double dgc =
                    rs_scale * acc[h][0] + lower[0] + upper[0] + lower[1] + upper[1] + lower[2] + upper[2];
                diag64c[cc] = dgc;
                diag32c[cc] = dgc > 0.0 ? (float)dgc : 0.f;
            } else {
                diag64c[cc] = 1.0;
                diag32c[cc] = 0.f;
            }
            for (int a = 0; a < 3; a++) {
                const double cv = active ? lower[a] : 0.0;
                cpl64c.a[a][cc] = cv;
                cpl32c[a][cc] = (float)cv;
            }
        }
    }
}

// Dense inverse of the coarsest operator (n <= 64 cells; SPD up to
// pure-Neumann blocks) by in-place Gauss-Jordan. Pivots below 1e-12 of the
// largest diagonal (the pure-Neumann direction) are dropped: their row and
// column stay 0.
//
// The 64 pivot steps are a serial chain, so what counts is the length of one:
// the matrix is in registers, wavefront w of four holding rows 16 w .. 16 w +
// 15 and lane c column c. A step reads the pivot row and the pivot's
// reciprocal from LDS and the pivot column of its own rows from lane kk's
// registers; the wavefront with the next pivot row updates that one first and
// publishes it (two buffers, one barrier), so its division overlaps the other
// rows' updates. In column kk the row counts as 1 and the matrix as 0, which
// leaves one product and one sum per element whatever its place. One block at
// 4^3 cells: 36 us (66 with the division between the rows' updates and the
// barrier and a choice of four forms per element; 77 with the matrix in LDS).
constexpr int kInvertThreads = 256;

__global__ __launch_bounds__(kInvertThreads) void k_coarse_invert(Dims d, Op64 A, float *ainv) {
    constexpr int S = kMaxCoarse, R = S / (kInvertThreads / 64);  // rows per wavefront
    static_assert(S == 64 && R == 16, "lane c holds column c");
    __shared__ double M[S * S];
    __shared__ double rowk[2][S], pivk[2];  // the pivot row; the pivot's reciprocal, 0 for a dropped one
    const int n = (int)d.cells();
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const Strides s(d);
    for (int e = tid; e < S * S; e += kInvertThreads) M[e] = 0.0;
    __syncthreads();
    for (int c = tid; c < n; c += kInvertThreads) {
        const int i = c / (d.ny * d.nz), j = (c / d.nz) % d.ny, k = c % d.nz;
        M[c * S + c] = A.diag[c];
        if (i > 0) M[c * S + (c - (int)s.sx)] = -A.cpl[0][c];
        if (i + 1 < d.nx) M[c * S + (c + (int)s.sx)] = -A.cpl[0][c + s.sx];
        if (j > 0) M[c * S + (c - (int)s.sy)] = -A.cpl[1][c];
        if (j + 1 < d.ny) M[c * S + (c + (int)s.sy)] = -A.cpl[1][c + s.sy];
        if (k > 0) M[c * S + (c - 1)] = -A.cpl[2][c];
        if (k + 1 < d.nz) M[c * S + (c + 1)] = -A.cpl[2][c + 1];
    }
    __syncthreads();
    double m = fabs(M[lane * S + lane]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    const double tiny = 1e-12 * m;
    double a[R];
#pragma unroll
    for (int r = 0; r < R; r++) a[r] = M[(R * wave + r) * S + lane];
    auto at_lane = [](double v, int l) {
        typedef int i2 __attribute__((ext_vector_type(2)));
        const i2 h = __builtin_bit_cast(i2, v);
        return __builtin_bit_cast(double, i2{__builtin_amdgcn_readlane(h.x, l), __builtin_amdgcn_readlane(h.y, l)});
    };
    auto publish = [&](double row, int kk) {
        const double p = at_lane(row, kk);
        rowk[kk & 1][lane] = row;
        const double pinv = fabs(p) <= tiny ? 0.0 : 1.0 / p;
        if (lane == 0) pivk[kk & 1] = pinv;
    };
    if (wave == 0) publish(a[0], 0);
    __syncthreads();
    for (int w = 0; w < S / R; w++) {
#pragma unroll
        for (int ki = 0; ki < R; ki++) {
            const int kk = R * w + ki;
            if (kk >= n) break;  // uniform over the block
            const int kn = (ki + 1) % R;  // the next pivot row's place in its wavefront
            const bool next = wave == (ki + 1 < R ? w : w + 1) && kk + 1 < n;
            const double pinv = pivk[kk & 1], row = rowk[kk & 1][lane];
            const double rk = lane == kk ? 1.0 : row;
            auto step = [&](double v) {
                const double ck = at_lane(v, kk);
                const double v0 = lane == kk ? 0.0 : v;
                return pinv == 0.0 ? v0 : v0 - ck * rk * pinv;
            };
            if (next) {
                a[kn] = step(a[kn]);
                publish(a[kn], kk + 1);
            }
            // (the pivot row itself, and the next one where it is done, are put
            // right after the loop)
            const double done = a[kn];
#pragma unroll
            for (int r = 0; r < R; r++) a[r] = step(a[r]);
            if (next) a[kn] = done;
            if (wave == w) a[ki] = pinv == 0.0 ? 0.0 : rk * pinv;
            __syncthreads();
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int row = R * wave + r;
        if (row < n && lane < n) ainv[row * n + lane] = (float)a[r];
    }
}

__global__ __launch_bounds__(kBlock) void k_coarse_solve(int n, const float *ainv, const float *b,
                                                         float *x, const double *gate) {
    if (gated(gate)) return;
    __shared__ float bs[kMaxCoarse];
    const int tid = threadIdx.x;
    for (int t = tid; t < n; t += kBlock) bs[t] = b[t];
    __syncthreads();
    for (int r = tid; r < n; r += kBlock) {
        float acc = 0.f;
        for (int c = 0; c < n; c++) acc = fmaf(ainv[r * n + c], bs[c], acc);
        x[r] = acc;
    }
}

}  // namespace

void launch_smooth_first(hipStream_t st, Dims d, Op32 A, const double *r64, float *b, float *x,
                         float c0, const double *gate) {
    Launch L = cell_launch(d);
    if (r64)
        hipLaunchKernelGGL(k_smooth_first<true>, L.grid, L.block, 0, st, L.cg, d, A, r64, b, x, c0, gate);
    else
        hipLaunchKernelGGL(k_smooth_first<false>, L.grid, L.block, 0, st, L.cg, d, A, r64, b, x, c0, gate);
    SFP_LAUNCH_CHECK();
}

unsigned restrict_quads(Dims d) {
    return (unsigned)((d.nz + kRestrictFlatZ - 1) / kRestrictFlatZ) * (unsigned)((d.ny + 1) / 2) *
           (unsigned)((d.nx + 1) / 2);
}

bool flat_step(Dims d) { return d.cells() < (size_t(1) << 32) - 64; }
bool whole_groups(Dims d) { return d.nz % 4 == 0 && flat_step(d); }

// The flat step where it applies: no fused first step, 16-byte aligned arrays;
// with the prolongation z rows of whole 4-cell groups (8-byte aligned coarse
// values). On MI355X 12 % faster than x-plane tiles at 256^3, 17 % at 128^3, and
// 14.5 us instead of 26 at 131 x 129 x 133 (the restriction 13 instead of 29).
static bool smooth_flat(Dims d, int mode, const double *r64, const float *ecoarse,
                        std::initializer_list<const float *> arrays) {
    if ((mode & SM_FIRST) || r64 || !flat_step(d)) return false;
    if ((mode & SM_PROLONG) && (!whole_groups(d) || (uintptr_t)ecoarse % 8)) return false;
    for (const float *a : arrays)
        if ((uintptr_t)a % 16) return false;
    return true;
}

void launch_smooth(hipStream_t st, int mode, Dims d, Op32 A, const double *r64, float *b,
                   const float *xin, float *xout, float *dvec, float c0, float cd, float cr,
                   const float *ecoarse, const double *gate) {
    if (smooth_flat(d, mode, r64, ecoarse, {A.diag, A.cpl[0], A.cpl[1], A.cpl[2], b, xin, xout, dvec})) {
        const unsigned nb = (unsigned)((d.cells() + kSmoothFlatCells - 1) / kSmoothFlatCells);
        const Dims dc = d.coarse();
        const bool eager = d.cells() <= kEagerCells, any = !whole_groups(d);
#define SFP_FLAT_RUN(M, RS, RUN, ANY)                                                                \
    hipLaunchKernelGGL((k_smooth_flat<M, RS, RUN, ANY>),                                               \
                       dim3(RUN == kListRun ? std::min(nb, 256u * list_waves(M, ANY)) : nb), dim3(kBlock), 0, st, d, A, b, \
                       xin, xout, dvec, cd, cr, ecoarse, dc, gate)
#define SFP_FLAT_LAUNCH(M, RS, RUN)                                                                  \
    do {                                                                                             \
        if constexpr (((M) & SM_PROLONG) != 0) SFP_FLAT_RUN(M, RS, RUN, false);                      \
        else if (any) SFP_FLAT_RUN(M, RS, RUN, true);                                                \
        else SFP_FLAT_RUN(M, RS, RUN, false);                                                        \
    } while (0)
#define SFP_FLAT_CASE(M)                                                                           \
    case M:                                                                                        \
        if (A.pinned_rowsum) {                                                                     \
            if (eager) SFP_FLAT_LAUNCH(M, true, kEagerRun); else SFP_FLAT_LAUNCH(M, true, kBytesRun); \
        } else if (A.chunks.list) {                                                                \
            SFP_FLAT_LAUNCH(M, false, kListRun);                                                   \
        } else {                                                                                   \
            if (eager) SFP_FLAT_LAUNCH(M, false, kEagerRun); else SFP_FLAT_LAUNCH(M, false, kBytesRun); \
        }                                                                                          \
        break;
        switch (mode) {
            SFP_FLAT_CASE(SM_PROLONG)
            SFP_FLAT_CASE(SM_PROLONG | SM_WRITE_D)
            SFP_FLAT_CASE(SM_XFIRST)
            SFP_FLAT_CASE(SM_XFIRST | SM_WRITE_D)
            SFP_FLAT_CASE(SM_READ_D)
            SFP_FLAT_CASE(SM_READ_D | SM_WRITE_D)
            SFP_FLAT_CASE(0)
            SFP_FLAT_CASE(SM_WRITE_D)
            default:
                throw ArgError("unsupported smoother mode");
        }
#undef SFP_FLAT_CASE
#undef SFP_FLAT_LAUNCH
#undef SFP_FLAT_RUN
        SFP_LAUNCH_CHECK();
        return;
    }
    // 8 planes per block measured best for the shuffle-based step (256^3:
    // 122 us vs 124 us at 16 and 123 us at 4)
    Launch L = cell_launch(d, 0, 8);
    Dims dc = d.coarse();
#define SFP_SMOOTH_CASE(M)                                                                    \
    case M:                                                                                   \
        hipLaunchKernelGGL(k_smooth<M>, L.grid, L.block, 0, st, L.cg, d, A, r64, b, xin, xout, \
                           dvec, c0, cd, cr, ecoarse, dc, gate);                              \
        break;
    switch (mode) {
        SFP_SMOOTH_CASE(SM_FIRST)
        SFP_SMOOTH_CASE(SM_FIRST | SM_WRITE_D)
        SFP_SMOOTH_CASE(SM_PROLONG)
        SFP_SMOOTH_CASE(SM_PROLONG | SM_WRITE_D)
        default:  // (a flat mode on arrays or a grid it does not take)
            throw ArgError("unsupported smoother mode, arrays or grid");
    }
#undef SFP_SMOOTH_CASE
    SFP_LAUNCH_CHECK();
}

Launch pair_launch(Dims d, bool even_planes) {
    Launch L;
    L.cg.gx = (d.nz + kPairZ - 1) / kPairZ;
    L.cg.gy = (d.ny + kPairY - 1) / kPairY;
    const long long tiles = (long long)L.cg.gx * L.cg.gy * d.nx;
    L.cg.planes = (int)std::min<long long>(16, std::max<long long>(1, tiles / 1024));
    if (even_planes && (L.cg.planes & 1)) L.cg.planes++;  // x pairs stay in one block
    L.block = dim3(64, kPairRows, 1);
    L.grid = dim3(L.cg.gx * L.cg.gy * ((d.nx + L.cg.planes - 1) / L.cg.planes), 1, 1);
    return L;
}

// Rows of a wavefront, or of half a wavefront (row_pair_sub 2) from 80 cells: 180
// x 180 x 132 to 192 magnetic solves 1.04-1.11x against the x-plane pair, 120 x
// 124 x 80 1.02x and x 72 0.98x against flat steps. k_smooth_pair_rows addresses a run's planes, at
// most 64 with their neighbours, by byte offsets below kPairOut.
static int row_pair_sub(Dims d) { return d.nz <= 128 ? 2 : 1; }
bool row_pair(Dims d) {
    return d.nz % 4 == 0 && d.nz >= 80 && d.nz <= 256 && d.cells() < (size_t(1) << 32) &&
           64 * 4 * (size_t)d.ny * d.nz < kPairOut;
}

// Compute units of the current device (cached per device).
static int device_cus() {
    static int cus[64] = {0};
    int dev = 0;
    SFP_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= 64) return 256;
    if (!cus[dev]) {
        int v = 0;
        SFP_HIP(hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev));
        cus[dev] = v > 0 ? v : 256;
    }
    return cus[dev];
}

// rowact[i ny + j] = 1 when the z row (i, j) holds an active cell: one
// wavefront per row.
__global__ __launch_bounds__(kBlock) void k_row_activity(Dims d, const float *__restrict__ diag32,
                                                         unsigned char *__restrict__ act) {
    const size_t row = ((size_t)blockIdx.x * kBlock + threadIdx.x) / 64;
    const int lane = threadIdx.x & 63;
    if (row >= (size_t)d.nx * d.ny) return;  // uniform over the wavefront
    const size_t c = row * (size_t)d.nz;
    bool a = false;
    for (int k = lane; k < d.nz; k += 64) a = a || diag32[c + k] > 0.f;
    const unsigned long long m = __ballot(a);
    if (lane == 0) act[row] = m != 0ull ? 1 : 0;
}

void launch_row_activity(hipStream_t st, Dims d, const float *diag32, unsigned char *act) {
    const size_t threads = (size_t)d.nx * d.ny * 64;
    hipLaunchKernelGGL(k_row_activity, dim3((unsigned)((threads + kBlock - 1) / kBlock)), dim3(kBlock), 0, st,
                       d, diag32, act);
    SFP_LAUNCH_CHECK();
}

// flags[q]: whether chunk q (256 cells) holds an active cell. A wavefront per
// chunk.
__global__ __launch_bounds__(kBlock) void k_chunk_flags(unsigned n, const float *__restrict__ diag32,
                                                        unsigned char *__restrict__ flags) {
    const unsigned q = (blockIdx.x * kBlock + threadIdx.x) / 64, lane = threadIdx.x & 63;
    const unsigned c = q * kChunk + 4 * lane;
    bool a = false;
    if (c < n) {
        const f4v v = own_cells<true>(diag32, c, n);
        a = v.x > 0.f || v.y > 0.f || v.z > 0.f || v.w > 0.f;
    }
    const unsigned long long m = __ballot(a);
    if (lane == 0 && q * kChunk < n) flags[q] = m != 0ull ? 1 : 0;
}

// The set flags' indices in ascending order (so sums over the listed chunks
// have a fixed order), list[0] their number. A block for each list: a thread counts a run
// of flags, 16 at a time, the counts are summed over the threads before it, and
// it writes its run's (65536 chunks of a 256^3 grid: 12 us, beside the clears).
constexpr int kListThreads = 1024;
__global__ __launch_bounds__(kListThreads) void k_chunk_list(unsigned nch, unsigned nq, unsigned nbl, ActiveLists a) {
    if (blockIdx.x == 1) nch = nq;
    if (blockIdx.x == 2) nch = nbl;
    const unsigned char *const flags = blockIdx.x == 0 ? a.flags : blockIdx.x == 1 ? a.quad_flags : a.block_flags;
    unsigned *const list = blockIdx.x == 0 ? a.list : blockIdx.x == 1 ? a.quads : a.blocks;
    __shared__ unsigned sums[kListThreads / 64];
    const unsigned tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const unsigned per = ((nch + kListThreads - 1) / kListThreads + 15) / 16 * 16;
    const unsigned b0 = tid * per, b1 = min(b0 + per, nch);
    auto each = [&](auto f) {
        for (unsigned b = b0; b < b1; b += 16) {  // (an allocation reaches 64 bytes past its array)
            const uint4 v = *(const uint4 *)(flags + b);
            const unsigned w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (unsigned k = 0; k < 16; k++)
                if (b + k < b1 && ((w[k / 4] >> (8 * (k % 4))) & 0xffu)) f(b + k);
        }
    };
    unsigned own = 0;
    each([&](unsigned) { own++; });
    unsigned sum = own;  // inclusive over the wavefront
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned v = __shfl_up(sum, o, 64);
        if ((int)lane >= o) sum += v;
    }
    if (lane == 63) sums[wave] = sum;
    __syncthreads();
    unsigned before = 0, total = 0;
    for (unsigned w = 0; w < kListThreads / 64; w++) {
        if (w < wave) before += sums[w];
        total += sums[w];
    }
    unsigned at = 1 + before + sum - own;
    each([&](unsigned q) { list[at++] = q; });
    if (tid == 0) list[0] = total;
}

// flags[u]: whether quad u of the restriction (k_restrict_flat's 64 cells of z
// in two rows and two planes) meets an active chunk; then whether an FCG block
// (two chunks) holds one.
__global__ __launch_bounds__(kBlock) void k_unit_flags(Dims d, unsigned quads, unsigned blocks, unsigned nch,
                                                       const unsigned char *__restrict__ chunk_flags,
                                                       unsigned char *__restrict__ quad_flags,
                                                       unsigned char *__restrict__ block_flags) {
    static_assert(kListCells == 2 * kChunk, "an FCG block is two chunks");
    const unsigned u = blockIdx.x * kBlock + threadIdx.x;
    if (u < blocks) block_flags[u] = chunk_flags[2 * u] | (2 * u + 1 < nch ? chunk_flags[2 * u + 1] : 0);
    if (u >= quads) return;
    const unsigned zch = (unsigned)(d.nz + kRestrictFlatZ - 1) / kRestrictFlatZ, yp = (unsigned)(d.ny + 1) / 2;
    const int k0 = kRestrictFlatZ * (int)(u % zch), k1 = min(k0 + kRestrictFlatZ, d.nz) - 1;
    const int j0 = 2 * (int)(u / zch % yp), i0 = 2 * (int)(u / zch / yp);
    unsigned char a = 0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int i = min(i0 + (q >> 1), d.nx - 1), j = min(j0 + (q & 1), d.ny - 1);
        a |= chunk_flags[(unsigned)d.idx(i, j, k0) / kChunk] | chunk_flags[(unsigned)d.idx(i, j, k1) / kChunk];
    }
    quad_flags[u] = a;
}

void launch_active_chunks(hipStream_t st, Dims d, const float *diag32, const ActiveLists &a) {
    if (!flat_step(d)) throw ArgError("launch_active_chunks: not a flat level");
    const unsigned n = (unsigned)d.cells(), nch = (n + kChunk - 1) / kChunk, nq = restrict_quads(d),
                   nbl = (n + kListCells - 1) / kListCells;
    hipLaunchKernelGGL(k_chunk_flags, dim3((nch + kBlock / 64 - 1) / (kBlock / 64)), dim3(kBlock), 0, st, n, diag32,
                       a.flags);
    SFP_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_unit_flags, dim3((std::max(nq, nbl) + kBlock - 1) / kBlock), dim3(kBlock), 0, st, d, nq, nbl,
                       nch, a.flags, a.quad_flags, a.block_flags);
    SFP_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_chunk_list, dim3(3), dim3(kListThreads), 0, st, nch, nq, nbl, a);
    SFP_LAUNCH_CHECK();
}

// The runs of planes that hold k_smooth_pair_rows' work where z rows are
// inactive: one block per compute unit runs at a time and marches over its run,
// so equal runs of whole tile columns leave the CUs of the air idle while the
// liquid's set the time (256^3 pool, 26 % of the rows active: 76 us a pair, 40
// with this). Runs start at an active plane of their column and take P planes,
// P the least with which there are no more runs than CUs.
constexpr int kSegTiles = 128, kSegPlanes = 1024, kSegMin = 8, kSegMax = 56;
unsigned pair_segments_max(Dims d) {
    const int rows = row_pair_y(row_pair_sub(d));
    const unsigned ytiles = (unsigned)((d.ny + rows - 1) / rows);
    if (!row_pair(d) || row_pair_sub(d) > 1 || ytiles > (unsigned)kSegTiles || d.nx > kSegPlanes) return 0;
    return ytiles * (unsigned)((d.nx + kSegMin - 1) / kSegMin);
}
__global__ __launch_bounds__(kListThreads) void k_pair_segments(Dims d, int ytiles, int rows, int cus,
                                                                const unsigned char *__restrict__ rowact,
                                                                int *__restrict__ segments) {
    __shared__ unsigned long long mask[kSegTiles][kSegPlanes / 64];
    __shared__ int count[kSegTiles];
    __shared__ int total;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int words = (d.nx + 63) / 64;
    if (tid == 0) total = 0;
    __syncthreads();
    for (int e = wave; e < ytiles * words; e += kListThreads / 64) {
        const int by = e / words, w = e % words, q = 64 * w + lane;
        const int j1 = min((by + 1) * rows, d.ny);
        bool a = false;
        if (q < d.nx)
            for (int j = by * rows; j < j1; j++) a |= rowact[(size_t)q * d.ny + j] != 0;
        const unsigned long long m = __ballot(a);
        if (lane == 0) {
            mask[by][w] = m;
            atomicAdd(&total, __popcll(m));
        }
    }
    __syncthreads();
    int P = min(kSegMax, max(kSegMin, (total + cus - 1) / cus));
    auto next_active = [&](int q) {  // the first active plane from q on, or nx
        for (int w = q / 64; w < words; w++) {
            const unsigned long long m = mask[tid][w] & (w == q / 64 ? ~0ull << (q % 64) : ~0ull);
            if (m) return 64 * w + __ffsll(m) - 1;
        }
        return d.nx;
    };
    while (true) {
        __syncthreads();
        if (tid == 0) total = 0;
        __syncthreads();
        if (tid < ytiles) {
            int n = 0;
            for (int q = next_active(0); q < d.nx; q = q + P < d.nx ? next_active(q + P) : d.nx) n++;
            count[tid] = n;
            atomicAdd(&total, n);
        }
        __syncthreads();
        if (total <= cus || P >= kSegMax) break;  // uniform
        P++;
    }
    if (tid < ytiles) {
        int at = 0;
        for (int y = 0; y < tid; y++) at += count[y];
        for (int q = next_active(0); q < d.nx; q = q + P < d.nx ? next_active(q + P) : d.nx) {
            segments[1 + 3 * at] = tid;
            segments[2 + 3 * at] = q;
            segments[3 + 3 * at] = min(q + P, d.nx);
            at++;
        }
        if (tid == ytiles - 1) segments[0] = at;
    }
}
void launch_pair_segments(hipStream_t st, Dims d, const unsigned char *rowact, int *segments) {
    const int rows = row_pair_y(row_pair_sub(d)), ytiles = (d.ny + rows - 1) / rows;
    if (!pair_segments_max(d)) throw ArgError("launch_pair_segments: not a row-pair level");
    hipLaunchKernelGGL(k_pair_segments, dim3(1), dim3(kListThreads), 0, st, d, ytiles, rows, device_cus(), rowact,
                       segments);
    SFP_LAUNCH_CHECK();
}

void launch_smooth_pair(hipStream_t st, Dims d, Op32 A, const float *b, const float *x1, float *x3,
                        const float *d1, float cdA, float crA, float cdB, float crB,
                        const double *gate, const unsigned char *rowact, const int *segments) {
    if (x1 == x3) throw ArgError("launch_smooth_pair: x3 aliases x1");
    bool rows = row_pair(d);
    for (const float *a : {A.diag, A.cpl[0], A.cpl[1], A.cpl[2], b, x1, (const float *)x3, d1})
        rows = rows && (uintptr_t)a % 16 == 0;
    if (rows) {
        // one block per compute unit, in one round: as many x runs per tile
        // column as the columns leave CUs for (at most 56 planes a run, the
        // activity masks' reach)
        const int sub = row_pair_sub(d), ty = row_pair_y(sub);
        const unsigned ytiles = (unsigned)((d.ny + ty - 1) / ty);
        const int runs_max = std::max(1, device_cus() / (int)ytiles);
        int planes = std::min(56, std::max(1, (d.nx + runs_max - 1) / runs_max));
        const unsigned runs = (unsigned)((d.nx + planes - 1) / planes);
        const bool dx = d1 == x1;
        const unsigned char *ra = A.pinned_rowsum ? nullptr : rowact;
        const int *sg = ra ? segments : nullptr;
        const dim3 grid(sg ? pair_segments_max(d) : ytiles * runs), block(64, kRowPairWaves);
#define SFP_ROWPAIR(RS, DX)                                                                      \
    if (sub == 2)                                                                                \
        hipLaunchKernelGGL((k_smooth_pair_rows<RS, DX, 2>), grid, block, 0, st, d, A, b, x1, x3, \
                           d1, cdA, crA, cdB, crB, ra, sg, planes, ytiles, gate);                \
    else                                                                                         \
        hipLaunchKernelGGL((k_smooth_pair_rows<RS, DX, 1>), grid, block, 0, st, d, A, b, x1, x3, \
                           d1, cdA, crA, cdB, crB, ra, sg, planes, ytiles, gate)
        if (A.pinned_rowsum) {
            if (dx) { SFP_ROWPAIR(true, true); } else { SFP_ROWPAIR(true, false); }
        } else {
            if (dx) { SFP_ROWPAIR(false, true); } else { SFP_ROWPAIR(false, false); }
        }
#undef SFP_ROWPAIR
        SFP_LAUNCH_CHECK();
        return;
    }
    const Launch L = pair_launch(d, false);
    if (A.pinned_rowsum)
        hipLaunchKernelGGL((k_smooth_pair<false, true>), L.grid, L.block, 0, st, L.cg, d, A, b, x1, x3,
                           d1, cdA, crA, cdB, crB, Dims{}, nullptr, gate);
    else
        hipLaunchKernelGGL((k_smooth_pair<false, false>), L.grid, L.block, 0, st, L.cg, d, A, b, x1, x3,
                           d1, cdA, crA, cdB, crB, Dims{}, nullptr, gate);
    SFP_LAUNCH_CHECK();
}

void launch_smooth_restrict(hipStream_t st, Dims d, Op32 A, const float *b, const float *x1,
                            float *x2, const float *d1, float cd, float cr, float *bc,
                            const double *gate) {
    if (x1 == x2) throw ArgError("launch_smooth_restrict: x2 aliases x1");
    const Launch L = pair_launch(d, true);
    if (A.pinned_rowsum)
        hipLaunchKernelGGL((k_smooth_pair<true, true>), L.grid, L.block, 0, st, L.cg, d, A, b, x1, x2,
                           d1, cd, cr, 0.f, 0.f, d.coarse(), bc, gate);
    else
        hipLaunchKernelGGL((k_smooth_pair<true, false>), L.grid, L.block, 0, st, L.cg, d, A, b, x1, x2,
                           d1, cd, cr, 0.f, 0.f, d.coarse(), bc, gate);
    SFP_LAUNCH_CHECK();
}

void launch_prolong_add(hipStream_t st, Dims d, const float *diag32, const unsigned *list, const float *ecoarse,
                        float *x, const double *gate) {
    if (!flat_step(d)) throw ArgError("launch_prolong_add: grid too large");
    const unsigned nb = (unsigned)((d.cells() + kSmoothFlatCells - 1) / kSmoothFlatCells);
    if (list)
        hipLaunchKernelGGL(k_prolong_add<true>, dim3(std::min(nb, 2048u)), dim3(kBlock), 0, st, d, list, diag32,
                           ecoarse, d.coarse(), x, gate);
    else
        hipLaunchKernelGGL(k_prolong_add<false>, dim3(nb), dim3(kBlock), 0, st, d, list, diag32, ecoarse,
                           d.coarse(), x, gate);
    SFP_LAUNCH_CHECK();
}

void launch_clear_inactive(hipStream_t st, const ClearArgs &a) {
    if (a.nlev < 1 || a.nlev > kClearMaxLevels) throw ArgError("launch_clear_inactive: bad level count");
    const unsigned groups = a.start[a.nlev];
    const unsigned nb = (groups + kBlock - 1) / kBlock;
    hipLaunchKernelGGL(k_clear_inactive, dim3(nb), dim3(kBlock), 0, st, a);
    SFP_LAUNCH_CHECK();
}

void launch_restrict(hipStream_t st, Dims df, Op32 A, const float *b, const float *x, float *bc,
                     const double *gate, float *x0c, const float *diag32c, float c0) {
    if (x0c && !diag32c) throw ArgError("launch_restrict: x0c needs the coarse diagonal");
    Dims dc = df.coarse();
    bool flat = flat_step(df) && (uintptr_t)bc % 8 == 0 && (uintptr_t)x0c % 8 == 0 &&
                (uintptr_t)diag32c % 8 == 0;
    for (const float *a : {A.diag, A.cpl[0], A.cpl[1], A.cpl[2], b, x}) flat = flat && (uintptr_t)a % 16 == 0;
    if (!flat) throw ArgError("launch_restrict: grid too large or arrays not aligned");
    const unsigned nb = (unsigned)(((size_t)restrict_quads(df) * 64 + kBlock - 1) / kBlock);
    const bool eager = df.cells() <= kEagerCells;
#define SFP_RESTRICT_RUN(RS, EA, LI, ANY)                                                              \
    hipLaunchKernelGGL((k_restrict_flat<RS, EA, LI, ANY>), dim3(nb), dim3(kBlock), 0, st, df, A, b, x, dc, \
                       bc, x0c, diag32c, c0, gate)
#define SFP_RESTRICT_LAUNCH(RS, EA, LI)                      \
    do {                                                     \
        if (whole_groups(df)) SFP_RESTRICT_RUN(RS, EA, LI, false); \
        else SFP_RESTRICT_RUN(RS, EA, LI, true);             \
    } while (0)
    if (A.pinned_rowsum) {
        if (eager) SFP_RESTRICT_LAUNCH(true, true, false); else SFP_RESTRICT_LAUNCH(true, false, false);
    } else if (A.chunks.quads) {
        SFP_RESTRICT_LAUNCH(false, false, true);
    } else {
        if (eager) SFP_RESTRICT_LAUNCH(false, true, false); else SFP_RESTRICT_LAUNCH(false, false, false);
    }
#undef SFP_RESTRICT_LAUNCH
#undef SFP_RESTRICT_RUN
    SFP_LAUNCH_CHECK();
}

void launch_coarsen(hipStream_t st, Dims df, Op64 Af, const float *diag32f, Dims dc,
                    double scale, double rs_scale, double *diag64c, double *const cpl64c[3],
                    float *diag32c, float *const cpl32c[3], RowsFlag rows) {
    MutFaces m{{cpl64c[0], cpl64c[1], cpl64c[2]}};
    bool flat = whole_groups(df) && (uintptr_t)diag32f % 16 == 0;
    for (const double *a : {Af.diag, Af.cpl[0], Af.cpl[1], Af.cpl[2]}) flat = flat && (uintptr_t)a % 16 == 0;
    if (flat) {
        const size_t waves = (size_t)((df.nz + 63) / 64) * ((df.ny + 1) / 2) * ((df.nx + 1) / 2);
        const unsigned nb = (unsigned)((waves * 64 + kBlock - 1) / kBlock);
        hipLaunchKernelGGL(k_coarsen_flat, dim3(nb), dim3(kBlock), 0, st, df, Af, diag32f, dc, scale, rs_scale,
                           diag64c, m, diag32c, cpl32c[0], cpl32c[1], cpl32c[2], rows);
        SFP_LAUNCH_CHECK();
        return;
    }
    // over the fine grid, with even plane pairs per block (as the restriction)
    Launch L = cell_launch(df, 0, 8);
    if (L.cg.planes & 1) L = cell_launch(df, L.cg.planes + 1);
    hipLaunchKernelGGL(k_coarsen_fine, L.grid, L.block, 0, st, L.cg, df, Af, diag32f, dc, scale, rs_scale,
                       diag64c, m, diag32c, cpl32c[0], cpl32c[1], cpl32c[2], rows);
    SFP_LAUNCH_CHECK();
}

void launch_coarse_invert(hipStream_t st, Dims d, Op64 A, float *ainv) {
    if ((int)d.cells() > kMaxCoarse) throw ArgError("coarsest level too large for the dense solve");
    hipLaunchKernelGGL(k_coarse_invert, dim3(1), dim3(kInvertThreads), 0, st, d, A, ainv);
    SFP_LAUNCH_CHECK();
}

void launch_coarse_solve(hipStream_t st, int n, const float *ainv, const float *b, float *x,
                         const double *gate) {
    if (n > kMaxCoarse) throw ArgError("coarsest level too large for the dense solve");
    hipLaunchKernelGGL(k_coarse_solve, dim3(1), dim3(kBlock), 0, st, n, ainv, b, x, gate);
    SFP_LAUNCH_CHECK();
}

}  // namespace sfp
