// The small levels of a V-cycle in few launches: several Chebyshev steps of a
// level in one launch over overlapping tiles (k_tile_steps), and the coarse
// end of the cycle in one block (k_vcycle_tail).
//
// Separate launches on levels of up to some hundred thousand cells cost about
// 4.4 us each however little they compute (3.3 us from dispatch to the end of
// the write-back, of which most is two or three dependent memory latencies,
// and 1 us to the next): so the operator is read once into registers, the
// iterate goes between the threads through LDS, and a step costs an LDS round
// trip and a barrier.
//
// The mapping of both: a thread holds G groups of four consecutive z cells
// (z rows padded to whole groups with inactive cells) with their seven
// couplings, right-hand side, direction and iterate in registers; the iterate
// of every cell is also in LDS, twice (a step reads one copy and writes the
// other, so one barrier a step). Outside the grid and in the padding the
// couplings, the diagonal and the values are 0, which leaves every sum as the
// separate launches form it: each cell's arithmetic is k_smooth_flat's,
// k_restrict_flat's and k_coarse_solve's, in their order, and the results agree
// bit for bit.
#include "device_util.hpp"
#include "kernels.hpp"

#include <algorithm>

namespace sfp {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f2 __attribute__((ext_vector_type(2)));

// The pending ||r||^2 (see FoldArgs): true when the solve stops here. (stop_rr:
// f.sc->stop_rr, loaded with the partials.)
__device__ __forceinline__ bool fold_stop(const FoldArgs &f, const FoldLoad<1> &l, double stop_rr) {
    double v[1];
    fold_sum<1>(f.partials, f.nb, l, v);
    const bool stop = v[0] <= stop_rr;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        f.sc->rr = v[0];
        f.sc->iters += 1.0;
        if (stop) f.sc->stop = 1.0;
    }
    return stop;
}

// Guard floats before and after an LDS iterate (the z neighbours of its first
// and last group; any finite value, their coupling is 0).
constexpr int kGuard = 4;

// A level's extent in the padded z-fastest order of the LDS arrays.
struct Geo {
    int nx, ny, zp;  // zp: z row of whole groups
    int sx, sy;
    __device__ Geo(int x, int y, int z) : nx(x), ny(y), zp((z + 3) & ~3), sx(y * ((z + 3) & ~3)), sy((z + 3) & ~3) {}
    __device__ int groups() const { return nx * (sx >> 2); }
};

// Four values of a z row from element offset o, and those past the row's end
// (all but the first m) set to 0. Rows need not be aligned (gfx950 loads 16 bytes
// from any multiple of four), and the up to three values read past the last
// row are inside the buffer's allocation (DevBuf::ensure).
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ f4 ld_row(const float *__restrict__ p, unsigned o) {
    return *(const f4u *)((const char *)p + 4u * o);
}
__device__ __forceinline__ f4 in_row(f4 v, int m) {
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = q < m ? v[q] : 0.f;
    return v;
}
__device__ __forceinline__ void st_row(float *__restrict__ p, unsigned o, int m, f4 v) {
    if (m >= 4) {
        *(f4u *)((char *)p + 4u * o) = v;
        return;
    }
#pragma unroll
    for (int q = 0; q < 4; q++)
        if (q < m) p[o + q] = v[q];
}

// G groups of four cells of one thread.
template <int G>
struct Groups {
    f4 cx[G], cxp[G], cy[G], cyp[G], cz[G], dg[G], rd[G], b[G], d[G], x[G];  // (rd: 1 / dg, 0 on inactive cells)
    float czp[G];                            // the coupling above the group
    int c[G];                                // LDS offset of the group (-1: none)
    // of its x and y neighbours (its own where there is none), the upper one
    // in the upper half
    unsigned nx[G], ny[G];
};

// The operator (but rd) and right-hand side of group q at grid cell (i, j, k),
// element offset o (0 outside the grid), as stored; mask_group then zeroes what
// lies outside the grid (m: its cells inside the z row, 0 outside the grid).
// Loads first, selections after: the loads of all of a thread's groups are
// then in flight together.
template <int G>
__device__ __forceinline__ void load_group(Groups<G> &g, int q, const Op32 &A, const float *__restrict__ b, Dims d,
                                           int i, int j, unsigned o, int m) {
    const unsigned sy = (unsigned)d.nz, sx = (unsigned)d.ny * sy;
    g.dg[q] = ld_row(A.diag, o);
    g.cx[q] = ld_row(A.cpl[0], o);
    g.cxp[q] = ld_row(A.cpl[0], m > 0 && i + 1 < d.nx ? o + sx : o);
    g.cy[q] = ld_row(A.cpl[1], o);
    g.cyp[q] = ld_row(A.cpl[1], m > 0 && j + 1 < d.ny ? o + sy : o);
    g.cz[q] = ld_row(A.cpl[2], o);
    g.czp[q] = A.cpl[2][m > 4 ? o + 4 : o];
    g.b[q] = ld_row(b, o);
}
template <int G>
__device__ __forceinline__ void pin_group(const Groups<G> &g, int q) {
    pin(g.dg[q]);
    pin(g.cx[q]);
    pin(g.cxp[q]);
    pin(g.cy[q]);
    pin(g.cyp[q]);
    pin(g.cz[q]);
    pin(g.czp[q]);
    pin(g.b[q]);
}
template <int G>
__device__ __forceinline__ void mask_group(Groups<G> &g, int q, Dims d, int i, int j, int m) {
    g.dg[q] = in_row(g.dg[q], m);
    g.cx[q] = in_row(g.cx[q], m);
    g.cxp[q] = in_row(g.cxp[q], i + 1 < d.nx ? m : 0);
    g.cy[q] = in_row(g.cy[q], m);
    g.cyp[q] = in_row(g.cyp[q], j + 1 < d.ny ? m : 0);
    g.cz[q] = in_row(g.cz[q], m);
    g.czp[q] = m > 4 ? g.czp[q] : 0.f;
    g.b[q] = in_row(g.b[q], m);
#pragma unroll
    for (int s = 0; s < 4; s++) g.rd[q][s] = rcp_or_zero(g.dg[q][s]);
}

// LDS offsets of group t of a (tile or level) extent.
template <int G>
__device__ __forceinline__ void place_group(Groups<G> &g, int q, int t, const Geo &e, int &i, int &j, int &k) {
    const int gz = e.zp >> 2;
    const int r = t / gz;
    k = 4 * (t - r * gz);
    i = r / e.ny;
    j = r - i * e.ny;
    const int c = kGuard + 4 * t;
    g.c[q] = c;
    g.nx[q] = (unsigned)(i > 0 ? c - e.sx : c) | (unsigned)(i + 1 < e.nx ? c + e.sx : c) << 16;
    g.ny[q] = (unsigned)(j > 0 ? c - e.sy : c) | (unsigned)(j + 1 < e.ny ? c + e.sy : c) << 16;
}

// The off-diagonal sums and the step of one group from the iterate in X:
// d = cd d + cr D^-1 (b - A x), x += d (k_smooth_flat's arithmetic).
__device__ __forceinline__ void cheb_group(const f4 &cx, const f4 &cxp, const f4 &cy, const f4 &cyp, const f4 &cz,
                                           float czp, const f4 &dg, const f4 &rd, const f4 &b, f4 &d, f4 &x, f4 xm,
                                           f4 xp, f4 ym, f4 yp, float zl, float zh, float cd, float cr) {
    f4 xn;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float xzm = e > 0 ? x[e - 1] : zl, xzp = e < 3 ? x[e + 1] : zh;
        const float czu = e < 3 ? cz[e + 1] : czp;
        float off = fmaf(cx[e], xm[e], cxp[e] * xp[e]);
        off = fmaf(cy[e], ym[e], off);
        off = fmaf(cyp[e], yp[e], off);
        off = fmaf(cz[e], xzm, off);
        off = fmaf(czu, xzp, off);
        const float r = b[e] - fmaf(dg[e], x[e], -off);
        const float dn = fmaf(cd, d[e], cr * rd[e] * r);
        d[e] = dn;
        xn[e] = x[e] + dn;
    }
    x = xn;
}

// The residual's z-pair sums of one group (k_restrict_flat's residual, 0 on
// inactive cells).
__device__ __forceinline__ f2 residual_pairs(const f4 &cx, const f4 &cxp, const f4 &cy, const f4 &cyp, const f4 &cz,
                                             float czp, const f4 &dg, const f4 &b, const f4 &x, f4 xm, f4 xp, f4 ym,
                                             f4 yp, float zl, float zh) {
    f4 r = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float xzm = e > 0 ? x[e - 1] : zl, xzp = e < 3 ? x[e + 1] : zh;
        const float czu = e < 3 ? cz[e + 1] : czp;
        float off = fmaf(cx[e], xm[e], 0.f);
        off = fmaf(cxp[e], xp[e], off);
        off = fmaf(cy[e], ym[e], off);
        off = fmaf(cyp[e], yp[e], off);
        off = fmaf(cz[e], xzm, off);
        off = fmaf(czu, xzp, off);
        const float rr = b[e] - fmaf(dg[e], x[e], -off);
        r[e] = dg[e] > 0.f ? rr : 0.f;
    }
    return f2{r.x + r.y, r.z + r.w};
}

template <int G>
__device__ __forceinline__ void put_x(const Groups<G> &g, float *X) {
#pragma unroll
    for (int q = 0; q < G; q++)
        if (g.c[q] >= 0) *(f4 *)(X + g.c[q]) = g.x[q];
    __syncthreads();
}

// One Chebyshev step of every group: reads Xin, writes Xout, ends at a barrier.
template <int G>
__device__ __forceinline__ void step_groups(Groups<G> &g, const float *Xin, float *Xout, float cd, float cr) {
#pragma unroll
    for (int q = 0; q < G; q++) {
        if (g.c[q] < 0) continue;
        const int c = g.c[q];
        cheb_group(g.cx[q], g.cxp[q], g.cy[q], g.cyp[q], g.cz[q], g.czp[q], g.dg[q], g.rd[q], g.b[q], g.d[q],
                   g.x[q], *(const f4 *)(Xin + (g.nx[q] & 0xffffu)), *(const f4 *)(Xin + (g.nx[q] >> 16)), *(const f4 *)(Xin + (g.ny[q] & 0xffffu)),
                   *(const f4 *)(Xin + (g.ny[q] >> 16)), Xin[c - 1], Xin[c + 4], cd, cr);
        *(f4 *)(Xout + c) = g.x[q];
    }
    __syncthreads();
}

// The z-pair sums of every group's residual into S (two floats a group, in
// group order), ends at a barrier.
template <int G>
__device__ __forceinline__ void residual_groups(const Groups<G> &g, const float *X, float *S) {
#pragma unroll
    for (int q = 0; q < G; q++) {
        if (g.c[q] < 0) continue;
        const int c = g.c[q];
        const f2 s = residual_pairs(g.cx[q], g.cxp[q], g.cy[q], g.cyp[q], g.cz[q], g.czp[q], g.dg[q], g.b[q], g.x[q],
                                    *(const f4 *)(X + (g.nx[q] & 0xffffu)), *(const f4 *)(X + (g.nx[q] >> 16)),
                                    *(const f4 *)(X + (g.ny[q] & 0xffffu)), *(const f4 *)(X + (g.ny[q] >> 16)), X[c - 1], X[c + 4]);
        *(f2 *)(S + ((c - kGuard) >> 1)) = s;
    }
    __syncthreads();
}

// Sum of a coarse cell's children: its z-pair sums S at the fine (or tile)
// rows (i, j) and (i, j + 1) of planes i and i + 1 (k_restrict_flat's order: the y
// pair, then the x pair onto 0).
__device__ __forceinline__ float child_sum(const float *S, int i, int j, int K, int nx, int ny, int zh) {
    const float *p = S + (i * ny + j) * zh + K;
    const bool jy = j + 1 < ny, ix = i + 1 < nx;
    float acc = 0.f;
    acc += p[0] + (jy ? p[zh] : 0.f);
    if (ix) acc += p[ny * zh] + (jy ? p[ny * zh + zh] : 0.f);
    return acc;
}

// ---------------------------------------------------------------- tiles
// Up to eight steps of one level (and the restriction after them) in one
// launch: a block takes a tile of tx x ty x tz cells with a halo of as many
// cells as it makes stencil applications (in z whole groups, or none where
// the tile holds whole rows), computes every step on all of it (the outer
// cells of the halo go wrong by one layer a step, the tile's own cells never
// see them) and stores its own cells.
template <int G, int START>
__global__ __launch_bounds__(1024) void k_tile_steps(TileArgs a, const double *gate) {
    __shared__ __attribute__((aligned(16))) float lds[2][G * 4096 + 2 * kGuard];
    const Dims d = a.d;
    const TilePlan &P = a.plan;
    unsigned t = blockIdx.x;
    const int kb = (int)(t % (unsigned)P.bz);
    t /= (unsigned)P.bz;
    const int jb = (int)(t % (unsigned)P.by), ib = (int)(t / (unsigned)P.by);
    const int i0 = ib * P.tx - P.hx, j0 = jb * P.ty - P.hy, k0 = kb * P.tz - P.hz;
    const Geo e(P.tx + 2 * P.hx, P.ty + 2 * P.hy, P.tz + 2 * P.hz);
    const int ng = e.groups();
    // every load is issued before any is waited for: the gate's and the pending
    // norm's, the operator's, the iterate's and the coarse correction's
    const double stop = load_gate(gate, a.b);
    FoldLoad<1> fl;
    double stop_rr = 0.0;
    if (START == TILE_FIRST && a.fold.nb) {
        fold_load<1>(a.fold.partials, a.fold.nb, fl);
        stop_rr = a.fold.sc->stop_rr;
    }
    Groups<G> g;
    float e0[G], e1[G];
    int gi[G], gj[G], m[G];
#pragma unroll
    for (int q = 0; q < G; q++) {
        const int t = (int)threadIdx.x + q * (int)blockDim.x;
        int i, j, k;
        place_group(g, q, min(t, ng - 1), e, i, j, k);
        if (t >= ng) g.c[q] = -1;
        gi[q] = i0 + i;
        gj[q] = j0 + j;
        const int gk = k0 + k;
        const bool in = t < ng && gi[q] >= 0 && gi[q] < d.nx && gj[q] >= 0 && gj[q] < d.ny && gk >= 0 && gk < d.nz;
        const unsigned o = in ? ((unsigned)gi[q] * d.ny + gj[q]) * (unsigned)d.nz + gk : 0u;
        m[q] = in ? d.nz - gk : 0;
        load_group(g, q, a.A, a.b, d, gi[q], gj[q], o, m[q]);
        if constexpr (START != TILE_FIRST) g.x[q] = ld_row(a.xin, o);
        if constexpr (START == TILE_CONTINUE) g.d[q] = ld_row(a.din, o);
        if constexpr (START == TILE_PROLONG) {
            const unsigned er =
                in ? ((unsigned)(gi[q] >> 1) * a.dc.ny + (gj[q] >> 1)) * (unsigned)a.dc.nz + (gk >> 1) : 0u;
            e0[q] = a.e[er];
            e1[q] = a.e[m[q] > 2 ? er + 1 : er];
        }
    }
#pragma unroll
    for (int q = 0; q < G; q++) {
        pin_group(g, q);
        if constexpr (START != TILE_FIRST) pin(g.x[q]);
        if constexpr (START == TILE_CONTINUE) pin(g.d[q]);
        if constexpr (START == TILE_PROLONG) pin(e0[q]), pin(e1[q]);
    }
    if (stop != 0.0) return;
    if (START == TILE_FIRST && a.fold.nb && fold_stop(a.fold, fl, stop_rr)) return;  // uniform
#pragma unroll
    for (int q = 0; q < G; q++) {
        mask_group(g, q, d, gi[q], gj[q], m[q]);
        if constexpr (START != TILE_FIRST) g.x[q] = in_row(g.x[q], m[q]);
        if constexpr (START == TILE_CONTINUE) g.d[q] = in_row(g.d[q], m[q]);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            if (START == TILE_FIRST) g.x[q][s] = a.c0 * g.rd[q][s] * g.b[q][s];
            if (START == TILE_PROLONG && g.dg[q][s] > 0.f) g.x[q][s] = g.x[q][s] + (s < 2 ? e0[q] : e1[q]);
        }
        if (START == TILE_FIRST) g.d[q] = g.x[q];
        if (START == TILE_PROLONG) g.d[q] = f4{0.f, 0.f, 0.f, 0.f};  // (cd[0] is 0)
    }
    if (threadIdx.x < 2 * kGuard) {
        const int o = threadIdx.x < kGuard ? threadIdx.x : 4 * ng + threadIdx.x;
        lds[0][o] = lds[1][o] = 0.f;
    }
    float *X = lds[0], *Y = lds[1];
    put_x(g, X);
#pragma nounroll
    for (int s = 0; s < a.nsteps; s++) {
        step_groups(g, X, Y, a.cd[s], a.cr[s]);
        float *tmp = X;
        X = Y;
        Y = tmp;
    }
    // the tile's own cells
    auto own = [&](int q, int &gi, int &gj, int &gk) {
        if (g.c[q] < 0) return false;
        const int t = (g.c[q] - kGuard) >> 2, gz = e.zp >> 2;
        const int r = t / gz, k = 4 * (t - r * gz), i = r / e.ny, j = r - i * e.ny;
        gi = i0 + i;
        gj = j0 + j;
        gk = k0 + k;
        return i >= P.hx && i < P.hx + P.tx && j >= P.hy && j < P.hy + P.ty && k >= P.hz && k < P.hz + P.tz &&
               gi < d.nx && gj < d.ny && gk < d.nz;
    };
#pragma unroll
    for (int q = 0; q < G; q++) {
        int gi, gj, gk;
        if (!own(q, gi, gj, gk)) continue;
        const unsigned o = ((unsigned)gi * d.ny + gj) * (unsigned)d.nz + gk;
        st_row(a.xout, o, d.nz - gk, g.x[q]);
        if (a.dout) st_row(a.dout, o, d.nz - gk, g.d[q]);
    }
    if (!a.bc) return;  // uniform
    residual_groups(g, X, Y);
    // coarse cells of the tile (its extents and origin are even)
    const int cx = (P.tx + 1) >> 1, cy = (P.ty + 1) >> 1, cz = (P.tz + 1) >> 1;
    for (int t = threadIdx.x; t < cx * cy * cz; t += blockDim.x) {
        const int r = t / cz, K = t - r * cz, I = r / cy, J = r - I * cy;
        const int gI = ib * (P.tx >> 1) + I, gJ = jb * (P.ty >> 1) + J, gK = kb * (P.tz >> 1) + K;
        if (gI >= a.dc.nx || gJ >= a.dc.ny || gK >= a.dc.nz) continue;
        const float s = child_sum(Y, P.hx + 2 * I, P.hy + 2 * J, (P.hz >> 1) + K, e.nx, e.ny, e.zp >> 1);
        a.bc[((size_t)gI * a.dc.ny + gJ) * a.dc.nz + gK] = s;
    }
}

// ---------------------------------------------------------------- V-cycle tail
// The levels below the tail's first keep 8 arrays in LDS (operator, b,
// direction, two iterates), each padded to whole groups; their steps read
// everything from LDS (at most a few groups per thread, a few hundred
// threads).
struct LdsLevel {
    Geo e;
    int nz, n;  // real z extent, padded cells
    float *dg, *cx, *cy, *cz, *b, *d, *x0, *x1;
};

__device__ __forceinline__ LdsLevel lds_level(float *pool, const TailArgs &t, int l) {
    int off = 0;
    for (int q = 1; q < l; q++) {
        const Geo e(t.lv[q].d.nx, t.lv[q].d.ny, t.lv[q].d.nz);
        off += tail_level_floats(e.nx * e.sx);
    }
    const Dims d = t.lv[l].d;
    const Geo e(d.nx, d.ny, d.nz);
    const int n = e.nx * e.sx;
    float *p = pool + off;
    const int w = n + 2 * kGuard;
    return LdsLevel{e, d.nz, n, p, p + n, p + 2 * n, p + 3 * n, p + 4 * n, p + 5 * n, p + 6 * n + kGuard,
                    p + 6 * n + w + kGuard};
}

// x = c0 D^-1 b, d = x.
__device__ __forceinline__ void lds_first(const LdsLevel &L, float *x, float c0) {
    for (int g = threadIdx.x; 4 * g < L.n; g += blockDim.x) {
        const f4 dg = *(const f4 *)(L.dg + 4 * g), bv = *(const f4 *)(L.b + 4 * g);
        f4 xv;
#pragma unroll
        for (int q = 0; q < 4; q++) xv[q] = c0 * rcp_or_zero(dg[q]) * bv[q];
        *(f4 *)(x + 4 * g) = xv;
        *(f4 *)(L.d + 4 * g) = xv;
    }
    __syncthreads();
}

// x += P e on active cells; e on the next level's padded rows.
__device__ __forceinline__ void lds_prolong(const LdsLevel &L, float *x, const float *e, const Geo &ce) {
    for (int g = threadIdx.x; 4 * g < L.n; g += blockDim.x) {
        const int gz = L.e.zp >> 2;
        const int r = g / gz, k = 4 * (g - r * gz), i = r / L.e.ny, j = r - i * L.e.ny;
        const f2 ev = *(const f2 *)(e + ((i >> 1) * ce.ny + (j >> 1)) * ce.sy + (k >> 1));
        const f4 dg = *(const f4 *)(L.dg + 4 * g);
        f4 xv = *(const f4 *)(x + 4 * g);
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (dg[q] > 0.f) xv[q] = xv[q] + (q < 2 ? ev.x : ev.y);
        *(f4 *)(x + 4 * g) = xv;
    }
    __syncthreads();
}

// One step (kPairs false), or the residual's z-pair sums into out (kPairs).
template <bool kPairs>
__device__ __forceinline__ void lds_step(const LdsLevel &L, const float *x, float *out, float cd, float cr) {
    const f4 z4 = {0.f, 0.f, 0.f, 0.f};
    for (int g = threadIdx.x; 4 * g < L.n; g += blockDim.x) {
        const int c = 4 * g, gz = L.e.zp >> 2;
        const int r = g / gz, k = 4 * (g - r * gz), i = r / L.e.ny, j = r - i * L.e.ny;
        const bool xl = i > 0, xh = i + 1 < L.e.nx, yl = j > 0, yh = j + 1 < L.e.ny;
        const int xm = xl ? c - L.e.sx : c, xp = xh ? c + L.e.sx : c, ym = yl ? c - L.e.sy : c, yp = yh ? c + L.e.sy : c;
        f4 xc = *(const f4 *)(x + c);
        const f4 cx = *(const f4 *)(L.cx + c), cy = *(const f4 *)(L.cy + c), cz = *(const f4 *)(L.cz + c);
        const f4 ux = *(const f4 *)(L.cx + xp), uy = *(const f4 *)(L.cy + yp);
        const f4 cxp = xh ? ux : z4, cyp = yh ? uy : z4;
        const float uz = L.cz[c + 4 < L.n ? c + 4 : c];
        const float czp = k + 4 < L.nz ? uz : 0.f;
        const f4 dg = *(const f4 *)(L.dg + c), b = *(const f4 *)(L.b + c);
        const f4 vxm = *(const f4 *)(x + xm), vxp = *(const f4 *)(x + xp), vym = *(const f4 *)(x + ym),
                 vyp = *(const f4 *)(x + yp);
        if constexpr (kPairs) {
            *(f2 *)(out + (c >> 1)) =
                residual_pairs(cx, cxp, cy, cyp, cz, czp, dg, b, xc, vxm, vxp, vym, vyp, x[c - 1], x[c + 4]);
        } else {
            f4 dv = *(const f4 *)(L.d + c), rd;
#pragma unroll
            for (int q = 0; q < 4; q++) rd[q] = rcp_or_zero(dg[q]);
            cheb_group(cx, cxp, cy, cyp, cz, czp, dg, rd, b, dv, xc, vxm, vxp, vym, vyp, x[c - 1], x[c + 4], cd, cr);
            *(f4 *)(L.d + c) = dv;
            *(f4 *)(out + c) = xc;
        }
    }
    __syncthreads();
}

// The coarse right-hand side from the z-pair sums S of a level of extent
// (nx, ny) and zh pairs a row (0 in the coarse level's padding).
__device__ __forceinline__ void lds_restrict(const LdsLevel &C, const float *S, int nx, int ny, int zh) {
    for (int t = threadIdx.x; t < C.n; t += blockDim.x) {
        const int r = t / C.e.zp, K = t - r * C.e.zp, I = r / C.e.ny, J = r - I * C.e.ny;
        C.b[t] = K < C.nz ? child_sum(S, 2 * I, 2 * J, K, nx, ny, zh) : 0.f;
    }
    __syncthreads();
}

__global__ __launch_bounds__(1024) void k_vcycle_tail(TailArgs t, const double *gate) {
    __shared__ __attribute__((aligned(16))) float lds[2][kTailMaxCells + 2 * kGuard];
    __shared__ __attribute__((aligned(16))) float pool[kTailPoolFloats];
    __shared__ __attribute__((aligned(16))) float inv[kMaxCoarse * kInvStride];
    __shared__ __attribute__((aligned(16))) float bs[kMaxCoarse];
    const int tid = threadIdx.x;
    const int last = t.nlev - 1;
    const Dims d = t.lv[0].d;
    const Geo e(d.nx, d.ny, d.nz);
    const int ng = e.groups();
    // every load of the copy-in is issued before any is waited for: the first
    // level's operator and b into registers, the others' into LDS
    const double stop = load_gate(gate, t.ainv);
    FoldLoad<1> fl;
    double stop_rr = 0.0;
    if (t.fold.nb) {
        fold_load<1>(t.fold.partials, t.fold.nb, fl);
        stop_rr = t.fold.sc->stop_rr;
    }
    Groups<1> g;
    int gi, gj, gk;
    place_group(g, 0, min(tid, ng - 1), e, gi, gj, gk);
    if (tid >= ng) g.c[0] = -1;
    const int gm = tid < ng ? d.nz - gk : 0;
    load_group(g, 0, t.lv[0].A, t.lv[0].b, d, gi, gj, tid < ng ? (unsigned)((gi * d.ny + gj) * d.nz + gk) : 0u, gm);
    {
        const int nC = (int)t.lv[last].d.cells();
        f4 a4 = {0.f, 0.f, 0.f, 0.f};  // row r, columns c .. c + 3
        const int r = tid >> 4, c = 4 * (tid & 15);
        if (r < nC)
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (c + q < nC) a4[q] = t.ainv[r * nC + c + q];
        for (int l = 1; l <= last; l++) {
            const LdsLevel L = lds_level(pool, t, l);
            const Op32 A = t.lv[l].A;
            for (int o = tid; o < L.n; o += 1024) {
                const int row = o / L.e.zp, k = o - row * L.e.zp;
                const bool in = k < L.nz;
                const int s = row * L.nz + k;
                const float vd = in ? A.diag[s] : 0.f, vx = in ? A.cpl[0][s] : 0.f, vy = in ? A.cpl[1][s] : 0.f,
                            vz = in ? A.cpl[2][s] : 0.f;
                L.dg[o] = vd;
                L.cx[o] = vx;
                L.cy[o] = vy;
                L.cz[o] = vz;
            }
            if (tid < 2 * kGuard) {
                const int o = tid < kGuard ? tid - kGuard : L.n + tid - kGuard;
                L.x0[o] = L.x1[o] = 0.f;
            }
        }
        *(f4 *)(inv + r * kInvStride + c) = a4;
    }
    pin_group(g, 0);
    if (stop != 0.0) return;
    if (t.fold.nb && fold_stop(t.fold, fl, stop_rr)) return;  // uniform
    mask_group(g, 0, d, gi, gj, gm);
    if (tid < 2 * kGuard) {
        const int o = tid < kGuard ? tid : 4 * ng + tid;
        lds[0][o] = lds[1][o] = 0.f;
    }
    // ---- first level, down
    float *X = lds[0], *Y = lds[1];
#pragma unroll
    for (int s = 0; s < 4; s++) g.x[0][s] = t.cr[0][0] * g.rd[0][s] * g.b[0][s];
    g.d[0] = g.x[0];
    put_x(g, X);
#pragma nounroll
    for (int s = 1; s < t.deg[0]; s++) {
        step_groups(g, X, Y, t.cd[0][s], t.cr[0][s]);
        float *tmp = X;
        X = Y;
        Y = tmp;
    }
    residual_groups(g, X, Y);
    lds_restrict(lds_level(pool, t, 1), Y, e.nx, e.ny, e.zp >> 1);
    // ---- levels below, down
    unsigned in_x1 = 0;  // bit l: level l's pre-smoothed iterate is in x1
    for (int l = 1; l < last; l++) {
        const LdsLevel L = lds_level(pool, t, l);
        float *x = L.x0, *y = L.x1;
        lds_first(L, x, t.cr[1][0]);
#pragma nounroll
        for (int s = 1; s < t.deg[1]; s++) {
            lds_step<false>(L, x, y, t.cd[1][s], t.cr[1][s]);
            float *tmp = x;
            x = y;
            y = tmp;
        }
        if (x == L.x1) in_x1 |= 1u << l;
        lds_step<true>(L, x, y, 0.f, 0.f);
        lds_restrict(lds_level(pool, t, l + 1), y, L.e.nx, L.e.ny, L.e.zp >> 1);
    }
    // ---- coarsest: the dense inverse times b, a thread a row (k_coarse_solve's
    // order; the columns past the last are 0)
    {
        const LdsLevel C = lds_level(pool, t, last);
        const int nC = (int)t.lv[last].d.cells();
        const int o = tid < nC ? (tid / C.nz) * C.e.zp + tid % C.nz : 0;  // the cell's place
        if (tid < kMaxCoarse) bs[tid] = tid < nC ? C.b[o] : 0.f;
        __syncthreads();
        if (tid < nC) {
            float acc = 0.f;
#pragma unroll
            for (int c = 0; c < kMaxCoarse; c += 4) {
                const f4 m = *(const f4 *)(inv + tid * kInvStride + c), v = *(const f4 *)(bs + c);
#pragma unroll
                for (int q = 0; q < 4; q++) acc = fmaf(m[q], v[q], acc);
            }
            // (the padding after a row's last cell is prolonged to no cell)
            C.x0[o] = acc;
        }
        __syncthreads();
    }
    // ---- up
    const float *ev = lds_level(pool, t, last).x0;
    for (int l = last - 1; l >= 1; l--) {
        const LdsLevel L = lds_level(pool, t, l);
        float *x = (in_x1 >> l) & 1u ? L.x1 : L.x0, *y = x == L.x0 ? L.x1 : L.x0;
        lds_prolong(L, x, ev, lds_level(pool, t, l + 1).e);
#pragma nounroll
        for (int s = 0; s < t.deg[1]; s++) {
            lds_step<false>(L, x, y, s == 0 ? 0.f : t.cd[1][s], t.cr[1][s]);
            float *tmp = x;
            x = y;
            y = tmp;
        }
        ev = x;
    }
    if (tid < ng) {
        const Geo ce = lds_level(pool, t, 1).e;
        const f2 v = *(const f2 *)(ev + ((gi >> 1) * ce.ny + (gj >> 1)) * ce.sy + (gk >> 1));
#pragma unroll
        for (int s = 0; s < 4; s++)
            if (g.dg[0][s] > 0.f) g.x[0][s] = g.x[0][s] + (s < 2 ? v.x : v.y);
    }
    put_x(g, X);
#pragma nounroll
    for (int s = 0; s < t.deg[0]; s++) {
        step_groups(g, X, Y, s == 0 ? 0.f : t.cd[0][s], t.cr[0][s]);
        float *tmp = X;
        X = Y;
        Y = tmp;
    }
    // the first level's result
    if (tid < ng) st_row(t.lv[0].x1, (unsigned)((gi * d.ny + gj) * d.nz + gk), d.nz - gk, g.x[0]);
}

int padded_z(Dims d) { return (d.nz + 3) & ~3; }

}  // namespace

// ---------------------------------------------------------------- plans
// Modelled time of one launch (us), fitted to sweeps of every tile at 64^3 and
// 32^3 for 1 to 5 steps (within 10 % of the measured times of the best 20
// tiles; 64^3, two steps and the restriction: 4 x 4 x 64 tiles 7.8 us,
// 8 x 8 x 16 tiles 10.1 us; 32^3, three steps: 4.6 us against 9.4 us for three
// launches): 2.6 us of launch and first latency; 1.45 ns per group for the
// loads, more where a z row's part fills its 128-byte lines badly; 0.15 us and
// 0.52 ns per group a step (the compute unit's vector units: a step is about
// 330 cycles of a SIMD for 64 groups).
static double tile_cost(long long blocks, int groups, int zcells, bool rows, int steps) {
    const int threads = (groups > 1024 ? (groups + 1) / 2 : groups) + 63;
    const int fit = std::max(1, (groups > 1024 ? 16 : 24) / (threads / 64));
    const long long per_cu = (blocks + 255) / 256;
    const long long together = std::min<long long>(per_cu, fit);
    const double rounds = (double)((per_cu + together - 1) / together);
    const double bytes = 4.0 * zcells, lines = rows ? bytes : 128.0 * (1.0 + bytes / 128.0);
    const double g = (double)groups * (double)together;
    return 2.6 + rounds * (0.2 + 1.45e-3 * g * std::max(1.0, lines / bytes) + steps * (0.15 + 0.52e-3 * g));
}

TilePlan choose_tile(Dims d, int steps, bool restrict_after, double *cost) {
    const int H = steps + (restrict_after ? 1 : 0);
    const int zp = padded_z(d);
    TilePlan best;
    double best_cost = 1e30;
    static const int sizes[] = {2, 4, 6, 8, 10, 12, 16, 20, 24, 32, 48, 64};
    const int nz_opts[] = {zp, 64, 48, 32, 24, 16, 8};
    for (int tz : nz_opts) {
        if (tz > zp || (tz < zp && tz % 4)) continue;
        const int bz = (d.nz + tz - 1) / tz;
        if (tz != zp && bz == 1) continue;
        const int hz = bz == 1 ? 0 : (H + 3) & ~3;
        const int gz = (tz + 2 * hz) / 4;
        for (int sx : sizes) {
            const int tx = std::min(sx, (d.nx + 1) & ~1);
            const int bx = (d.nx + tx - 1) / tx, hx = bx == 1 ? 0 : H;
            for (int sy : sizes) {
                const int ty = std::min(sy, (d.ny + 1) & ~1);
                const int by = (d.ny + ty - 1) / ty, hy = by == 1 ? 0 : H;
                const long long groups = (long long)(tx + 2 * hx) * (ty + 2 * hy) * gz;
                if (groups > kTileMaxGroups) continue;
                const double c = tile_cost((long long)bx * by * bz, (int)groups, tz + 2 * hz, bz == 1,
                                           steps + (restrict_after ? 1 : 0));
                if (c < best_cost) {
                    best_cost = c;
                    best = TilePlan{tx, ty, tz, hx, hy, hz, bx, by, bz, (int)groups};
                }
            }
        }
    }
    if (cost) *cost = best_cost;
    return best;
}

void launch_tile_steps(hipStream_t st, const TileArgs &a, const double *gate) {
    const TilePlan &P = a.plan;
    if (a.nsteps < 0 || a.nsteps > 8) throw ArgError("tile steps: bad step count");
    if (P.groups < 1 || P.groups > kTileMaxGroups || P.tz % 4 || P.hz % 4 || (P.tx & 1) || (P.ty & 1))
        throw ArgError("tile steps: bad tile");
    const int reach = a.nsteps + (a.bc ? 1 : 0);
    if ((P.bx > 1 && P.hx < reach) || (P.by > 1 && P.hy < reach) || (P.bz > 1 && P.hz < reach))
        throw ArgError("tile steps: halo narrower than the steps");
    if (a.d.cells() >= ((size_t)1 << 30)) throw ArgError("tile steps: level too large");
    if (!a.b || !a.xout || (a.start != TILE_FIRST && !a.xin) || (a.start == TILE_PROLONG && !a.e) ||
        (a.start == TILE_CONTINUE && !a.din) || a.start < TILE_FIRST || a.start > TILE_CONTINUE)
        throw ArgError("tile steps: missing input");
    if (a.fold.nb > kFoldMax || (a.fold.nb && a.start != TILE_FIRST)) throw ArgError("tile steps: bad fold");
    if (a.xout == a.xin || (a.dout && a.dout == a.din) || (a.bc && a.dout))
        throw ArgError("tile steps: outputs alias inputs");
    const unsigned nb = (unsigned)(P.bx * P.by * P.bz);
    const dim3 grid(nb), block(((P.groups <= 1024 ? P.groups : (P.groups + 1) / 2) + 63) / 64 * 64);
#define SFP_TILE(G, S) hipLaunchKernelGGL((k_tile_steps<G, S>), grid, block, 0, st, a, gate)
    if (P.groups <= 1024) {
        if (a.start == TILE_FIRST) SFP_TILE(1, TILE_FIRST);
        else if (a.start == TILE_PROLONG) SFP_TILE(1, TILE_PROLONG);
        else SFP_TILE(1, TILE_CONTINUE);
    } else {
        if (a.start == TILE_FIRST) SFP_TILE(2, TILE_FIRST);
        else if (a.start == TILE_PROLONG) SFP_TILE(2, TILE_PROLONG);
        else SFP_TILE(2, TILE_CONTINUE);
    }
#undef SFP_TILE
    SFP_LAUNCH_CHECK();
}

bool tail_fits(const Dims *lv, int nlev) {
    if (nlev < 2 || nlev > kTailMaxLevels) return false;
    if ((size_t)lv[0].nx * lv[0].ny * padded_z(lv[0]) > kTailMaxCells) return false;
    if (lv[nlev - 1].cells() > (size_t)kMaxCoarse) return false;
    size_t pool = 0;
    for (int l = 1; l < nlev; l++) pool += tail_level_floats(lv[l].nx * lv[l].ny * padded_z(lv[l]));
    return pool <= (size_t)kTailPoolFloats;
}

void launch_vcycle_tail(hipStream_t st, const TailArgs &t, const double *gate) {
    Dims dims[kTailMaxLevels];
    if (t.nlev < 2 || t.nlev > kTailMaxLevels) throw ArgError("vcycle tail: bad level count");
    for (int l = 0; l < t.nlev; l++) dims[l] = t.lv[l].d;
    if (!tail_fits(dims, t.nlev)) throw ArgError("vcycle tail: levels too large");
    for (int k = 0; k < 2; k++)
        if (t.deg[k] < 1 || t.deg[k] > 8) throw ArgError("vcycle tail: bad degree");
    hipLaunchKernelGGL(k_vcycle_tail, dim3(1), dim3(1024), 0, st, t, gate);
    SFP_LAUNCH_CHECK();
}

}  // namespace sfp
