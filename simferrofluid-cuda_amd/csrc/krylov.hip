// FP64 kernels of the outer flexible CG (Notay's FCG with one stored
// direction): residual, matvec fused with its inner products, and the fused
// vector update. Each reduction writes per-block partial sums; a one-block
// finalize kernel adds them in block order (deterministic) and runs the
// scalar recurrences on the device, so the host only reads ||r||^2.
#include "device_util.hpp"
#include "kernels.hpp"
#include "solver.hpp"

#include <algorithm>

namespace sfp {
namespace {

enum FinalizeOp : int { FIN_RESIDUAL = 0, FIN_MATVEC = 1, FIN_UPDATE = 2 };

// true when a batched solve has already converged (see KrylovScalars::stop)
__device__ __forceinline__ bool gated(const double *gate) { return gate && *gate != 0.0; }

// Streams that no other thread of the launch reads again (FCG vectors) go
// through non-temporal loads and stores: measured 5-10 % faster on MI355X
// for the matvec and the update than cached accesses.
template <class T>
__device__ __forceinline__ T ld_stream(const T *a) {
    return __builtin_nontemporal_load(a);
}
template <class T>
__device__ __forceinline__ void st_stream(T *a, T v) {
    __builtin_nontemporal_store(v, a);
}
typedef double double2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));

// The x-plane stencils, for grids with odd nz whose sums keep their order: the
// constant mode of a magnetic potential hangs on one pinned cell, which carries
// the last bits of an iteration's sums into it 10^5 times larger (131 x 129 x
// 133: the flat kernels' order moves the field at the pin by 2e-8 of its rms).
// The stencil kernels below march over the block's x planes with the
// x-neighbours in registers and take the z-neighbours (value and z coupling)
// from the adjacent lanes of the tile row; only the row's end lanes load
// them. The off-diagonal sum keeps the order x-, x+, y-, y+, z-, z+.
__global__ __launch_bounds__(kBlock) void k_residual64(CellGrid cg, Dims d, Op64 A,
                                                       const double *__restrict__ b,
                                                       const double *__restrict__ x,
                                                       double *__restrict__ r,
                                                       double *__restrict__ partials,
                                                       float *__restrict__ b32,
                                                       float *__restrict__ x0,
                                                       const float *__restrict__ diag32,
                                                       float c0, const double *need) {
    if (need && *need == 0.0) return;
    int k, j, i0;
    cell_tile(cg, k, j, i0);
    const Strides s(d);
    const int tz = blockDim.x, lane = threadIdx.x;
    const bool on = k < d.nz && j < d.ny && i0 < d.nx;
    const bool zlo = k > 0, zhi = k + 1 < d.nz;
    const int ie = min(i0 + cg.planes, d.nx);
    double v[3] = {0.0, 0.0, 0.0};  // r.r, b.b, active cells (with diag32)
    size_t c = on ? d.idx(i0, j, k) : 0;
    // the FP32 copy of r and the cycle's first iterate (the FCG update's arithmetic)
    auto store32 = [&](size_t q, double rq) {
        const float dq = diag32 ? diag32[q] : 0.f;
        if (dq > 0.f) v[2] += 1.0;
        if (!b32) return;
        const float bf = (float)rq;
        b32[q] = bf;
        if (x0) x0[q] = c0 * rcp_or_zero(dq) * bf;
    };
    if (!x) {
        if (on)
            for (int i = i0; i < ie; i++, c += s.sx) {
                const double bc = b[c];
                if (r) r[c] = bc;
                store32(c, bc);
                v[0] += bc * bc;
                v[1] += bc * bc;
            }
        block_partials<3>(v, partials);
        return;
    }
    double xm = (on && i0 > 0) ? x[c - s.sx] : 0.0;
    double xc = on ? x[c] : 0.0;
    double cxc = on ? A.cpl[0][c] : 0.0;
    for (int i = i0; i < ie; i++, c += s.sx) {
        const bool up = i + 1 < d.nx;
        const double xp = (on && up) ? x[c + s.sx] : 0.0;
        const double cxp = (on && up) ? A.cpl[0][c + s.sx] : 0.0;
        const double czm = on ? A.cpl[2][c] : 0.0;
        double xzm = __shfl_up(xc, 1, tz);
        double xzp = __shfl_down(xc, 1, tz);
        double czp = __shfl_down(czm, 1, tz);
        if (lane == 0) xzm = (on && zlo) ? x[c - 1] : 0.0;
        if (lane == tz - 1) {
            xzp = (on && zhi) ? x[c + 1] : 0.0;
            czp = (on && zhi) ? A.cpl[2][c + 1] : 0.0;
        }
        if (on) {
            double off = 0.0;
            if (i > 0) off += cxc * xm;
            if (up) off += cxp * xp;
            if (j > 0) off += A.cpl[1][c] * x[c - s.sy];
            if (j + 1 < d.ny) off += A.cpl[1][c + s.sy] * x[c + s.sy];
            if (zlo) off += czm * xzm;
            if (zhi) off += czp * xzp;
            const double bc = b[c];
            const double rc = bc - (A.diag[c] * xc - off);
            if (r) r[c] = rc;
            store32(c, rc);
            v[0] += rc * rc;
            v[1] += bc * bc;
        }
        xm = xc;
        xc = xp;
        cxc = cxp;
    }
    block_partials<3>(v, partials);
}

__global__ __launch_bounds__(kBlock) void k_fcg_matvec(CellGrid cg, Dims d, Op64 A,
                                                       const float *__restrict__ active,
                                                       const float *__restrict__ z,
                                                       const double *__restrict__ r,
                                                       const double *__restrict__ qprev,
                                                       double *__restrict__ w, int first,
                                                       double *__restrict__ partials,
                                                       const double *gate) {
    if (gated(gate)) return;
    int k, j, i0;
    cell_tile(cg, k, j, i0);
    const Strides s(d);
    const int tz = blockDim.x, lane = threadIdx.x;
    const bool on = k < d.nz && j < d.ny && i0 < d.nx;
    const bool zlo = k > 0, zhi = k + 1 < d.nz, ylo = on && j > 0, yhi = on && j + 1 < d.ny;
    const int ie = min(i0 + cg.planes, d.nx);
    double v[3] = {0.0, 0.0, 0.0};  // z.w, z.q_prev, z.r
    size_t c = on ? d.idx(i0, j, k) : 0;
    float zm = 0.f, zc = 0.f;
    double cxc = 0.0;
    bool primed = false;  // zm, zc, cxc hold this plane's values
    float act_next = (active && on) ? active[c] : 0.f;
    for (int i = i0; i < ie; i++, c += s.sx) {
        float act = 1.f;
        if (active) {
            act = act_next;
            act_next = (on && i + 1 < ie) ? active[c + s.sx] : 0.f;
            if (!__any(on && act > 0.f)) {
                primed = false;
                continue;
            }
        }
        if (!primed) {
            zm = (on && i > 0) ? z[c - s.sx] : 0.f;
            zc = on ? z[c] : 0.f;
            cxc = on ? A.cpl[0][c] : 0.0;
            primed = true;
        }
        const bool up = i + 1 < d.nx;
        const float zp = (on && up) ? z[c + s.sx] : 0.f;
        const double cxp = (on && up) ? A.cpl[0][c + s.sx] : 0.0;
        const double czm = on ? A.cpl[2][c] : 0.0;
        const double cym = ylo ? A.cpl[1][c] : 0.0;
        const double cyp = yhi ? A.cpl[1][c + s.sy] : 0.0;
        const float zym = ylo ? z[c - s.sy] : 0.f;
        const float zyp = yhi ? z[c + s.sy] : 0.f;
        const double dg = on ? A.diag[c] : 0.0;
        // (an inactive cell's q may be an earlier system's: the update skips
        // groups of 128 cells of the array, not of this row)
        const double qp = (on & (act > 0.f) & !first) ? ld_stream(qprev + c) : 0.0;
        const double rc = on ? ld_stream(r + c) : 0.0;
        float zzm = __shfl_up(zc, 1, tz);
        float zzp = __shfl_down(zc, 1, tz);
        double czp = __shfl_down(czm, 1, tz);
        if (lane == 0) zzm = (on && zlo) ? z[c - 1] : 0.f;
        if (lane == tz - 1) {
            zzp = (on && zhi) ? z[c + 1] : 0.f;
            czp = (on && zhi) ? A.cpl[2][c + 1] : 0.0;
        }
        if (on) {
            double off = 0.0;
            if (i > 0) off += cxc * (double)zm;
            if (up) off += cxp * (double)zp;
            if (j > 0) off += cym * (double)zym;
            if (j + 1 < d.ny) off += cyp * (double)zyp;
            if (zlo) off += czm * (double)zzm;
            if (zhi) off += czp * (double)zzp;
            const double zd = act > 0.f ? (double)zc : 0.0;
            const double wc = dg * zd - off;
            st_stream(w + c, wc);
            v[0] += zd * wc;
            if (!first) v[1] += zd * qp;
            v[2] += zd * rc;
        }
        zm = zc;
        zc = zp;
        cxc = cxp;
    }
    block_partials<3>(v, partials);
}

// The flat stencils run over the flat cell index, two consecutive cells of one z
// row per lane (nz even): 16-byte loads of the FP64 operator and vectors at the
// pair and at its x and y neighbour pairs, one extra value and z coupling at
// each end. A neighbour is sx, sy or 1 cells on in the array also where a row or
// a plane ends: the coupling to it is 0 there as stored (the lower coupling of
// the first cell across), and only a neighbour past the array has its couplings
// put to 0 (its value is any other). The off-diagonal sum has the order x-, x+,
// y-, y+, z-, z+; a row-sum diagonal is rebuilt from the couplings (the same
// sums in the same order as the assembly's, so the same bits), except in the
// pairs that hold cell 0 or its upper neighbours.
struct PairAt {
    unsigned n, sx, sy, c;
    __device__ __forceinline__ PairAt(Dims d, size_t cell)
        : n((unsigned)d.cells()), sx((unsigned)d.ny * (unsigned)d.nz), sy((unsigned)d.nz), c((unsigned)cell) {}
    // a at this pair and at the pair k cells before and after it
    __device__ __forceinline__ double2v at(const double *__restrict__ a) const { return *(const double2v *)(a + c); }
    __device__ __forceinline__ float2v at(const float *__restrict__ a) const { return *(const float2v *)(a + c); }
    __device__ __forceinline__ double2v below(const double *__restrict__ a, unsigned k) const {
        return *(const double2v *)(a + (c >= k ? c - k : 0));
    }
    __device__ __forceinline__ float2v below(const float *__restrict__ a, unsigned k) const {
        return *(const float2v *)(a + (c >= k ? c - k : 0));
    }
    __device__ __forceinline__ double2v above(const double *__restrict__ a, unsigned k) const {
        return *(const double2v *)(a + (n - c > k ? c + k : c));
    }
    __device__ __forceinline__ float2v above(const float *__restrict__ a, unsigned k) const {
        return *(const float2v *)(a + (n - c > k ? c + k : c));
    }
    // the cell below the pair's first, and the one above its second
    template <class T>
    __device__ __forceinline__ T one_below(const T *__restrict__ a) const {
        return a[c > 0 ? c - 1 : 0];
    }
    template <class T>
    __device__ __forceinline__ T one_above(const T *__restrict__ a) const {
        return a[n - c > 2 ? c + 2 : c];
    }
    // whether the pair holds a cell whose diagonal is not the row sum (0, 1, nz, nz*ny)
    __device__ __forceinline__ bool pinned() const { return (c == 0) | (c == sy) | (c == sx); }
};
// The operator at a pair: its couplings and diagonal.
struct PairOperator {
    double2v cxm, cxp, cym, cyp, cz, dg;
    double czp;
    __device__ __forceinline__ PairOperator(const Op64 &A, const PairAt &P) {
        cxm = P.at(A.cpl[0]);
        cxp = P.above(A.cpl[0], P.sx);
        cym = P.at(A.cpl[1]);
        cyp = P.above(A.cpl[1], P.sy);
        cz = P.at(A.cpl[2]);          // below each cell of the pair
        czp = P.one_above(A.cpl[2]);  // above the second
        const unsigned left = P.n - P.c;
        if (!(left > P.sx)) cxp = double2v{0.0, 0.0};
        if (!(left > P.sy)) cyp = double2v{0.0, 0.0};
        if (!(left > 2)) czp = 0.0;
        // (one condition, by bit operations: a short circuit between its uniform
        // and its lanes' part has been compiled to loads at undefined addresses)
        if ((A.pinned_rowsum != 0) & !P.pinned()) {
            dg.x = ((((cxm.x + cxp.x) + cym.x) + cyp.x) + cz.x) + cz.y;
            dg.y = ((((cxm.y + cxp.y) + cym.y) + cyp.y) + cz.y) + czp;
        } else {
            dg = P.at(A.diag);
        }
    }
    // (A v) of the pair, whose values are vc, the neighbours' the rest
    __device__ __forceinline__ double2v apply(double2v vc, double2v vxm, double2v vxp, double2v vym, double2v vyp,
                                              double vzm, double vzp) const {
        double o0 = 0.0, o1 = 0.0;
        o0 += cxm.x * vxm.x;
        o1 += cxm.y * vxm.y;
        o0 += cxp.x * vxp.x;
        o1 += cxp.y * vxp.y;
        o0 += cym.x * vym.x;
        o1 += cym.y * vym.y;
        o0 += cyp.x * vyp.x;
        o1 += cyp.y * vyp.y;
        o0 += cz.x * vzm;
        o0 += cz.y * vc.y;
        o1 += cz.y * vc.x;
        o1 += czp * vzp;
        return double2v{dg.x * vc.x - o0, dg.y * vc.y - o1};
    }
};
__device__ __forceinline__ double2v widen(float2v v) { return double2v{(double)v.x, (double)v.y}; }

// The same residual (r, and b32 with x0, may be null: then not stored; a
// convergence check needs only the sums, and with kList takes them of the listed
// blocks, as the matvec below).
constexpr unsigned kResidualCells = kListCells;

template <bool kList>
__global__ __launch_bounds__(kBlock) void k_residual64_flat(Dims d, Op64 A, const double *__restrict__ b,
                                                            const double *__restrict__ x,
                                                            double *__restrict__ r, double *__restrict__ partials,
                                                            float *__restrict__ b32, float *__restrict__ x0,
                                                            const float *__restrict__ diag32, float c0,
                                                            unsigned nb, const double *need) {
    if (need && *need == 0.0) return;
    const unsigned count = kList ? A.chunks.blocks[0] : nb;
    for (unsigned u = blockIdx.x; u < count; u += kList ? gridDim.x : nb) {
        const unsigned block = kList ? A.chunks.blocks[1 + u] : u;
        const size_t c = (size_t)block * kResidualCells + 2 * (size_t)flat_tid();
        double v[3] = {0.0, 0.0, 0.0};  // r.r, b.b, active cells (with diag32)
        if (c < d.cells()) {            // cells() is even: then c + 1 is a cell too
            const PairAt P(d, c);
            const double2v bc = ld_stream((const double2v *)(b + c));
            double2v rc = bc;
            if (x) {
                const double2v xc = P.at(x), xxm = P.below(x, P.sx), xxp = P.above(x, P.sx), xym = P.below(x, P.sy),
                               xyp = P.above(x, P.sy);
                const double xzm = P.one_below(x), xzp = P.one_above(x);
                const PairOperator op(A, P);
                const double2v ax = op.apply(xc, xxm, xxp, xym, xyp, xzm, xzp);
                rc.x = bc.x - ax.x;
                rc.y = bc.y - ax.y;
            }
            if (r) st_stream((double2v *)(r + c), rc);
            const float2v dd = diag32 ? *(const float2v *)(diag32 + c) : float2v{0.f, 0.f};
            v[2] = (dd.x > 0.f ? 1.0 : 0.0) + (dd.y > 0.f ? 1.0 : 0.0);
            if (b32) {
                const float2v bf = {(float)rc.x, (float)rc.y};
                *(float2v *)(b32 + c) = bf;
                if (x0) {
                    const float2v xf = {c0 * rcp_or_zero(dd.x) * bf.x, c0 * rcp_or_zero(dd.y) * bf.y};
                    *(float2v *)(x0 + c) = xf;
                }
            }
            v[0] = rc.x * rc.x + rc.y * rc.y;
            v[1] = bc.x * bc.x + bc.y * bc.y;
        }
        block_sum<3>(v);
        if (flat_tid() == 0)
#pragma unroll
            for (int q = 0; q < 3; q++) partials[(size_t)q * nb + block] = v[q];
    }
}

// The same matvec. kList: the launch's blocks share the listed blocks of
// kMatvecCells cells (Chunks::blocks), each with its own place among the partial
// sums (0 in the others', as its cells would give), so the sums keep their order
// to the bit. 256^3 pool, 26 % of the rows active: 70 us so, 80 with a block for
// each (the list's bytes at the copy rate: 62).
constexpr unsigned kMatvecCells = kListCells;
static_assert(kMatvecCells == 2 * kBlock, "two cells per lane");

template <bool kList>
__global__ __launch_bounds__(kBlock, kList ? 8 : 1) void k_fcg_matvec_flat(Dims d, Op64 A,
                                                            const float *__restrict__ active,
                                                            const float *__restrict__ z,
                                                            const double *__restrict__ r,
                                                            const double *__restrict__ qprev,
                                                            double *__restrict__ w, int first,
                                                            double *__restrict__ partials, unsigned nb,
                                                            const double *gate) {
    if (gated(gate)) return;
    const unsigned count = kList ? A.chunks.blocks[0] : nb;
    for (unsigned u = blockIdx.x; u < count; u += kList ? gridDim.x : nb) {
        const unsigned block = kList ? A.chunks.blocks[1 + u] : u;
        const size_t c = (size_t)block * kMatvecCells + 2 * (size_t)flat_tid();
        const bool on = c < d.cells();  // cells() is even: then c + 1 is a cell too
        double v[3] = {0.0, 0.0, 0.0};  // z.w, z.q_prev, z.r
        bool act = on, on0 = true, on1 = true;  // the pair's cells are active
        if (active && on) {
            const float2v a = *(const float2v *)(active + c);
            on0 = a.x > 0.f;
            on1 = a.y > 0.f;
            act = on0 || on1;
        }
        if (__any(act) && on) {
            const PairAt P(d, c);
            const float2v zl = P.at(z);
            const float2v zxm = P.below(z, P.sx), zxp = P.above(z, P.sx), zym = P.below(z, P.sy),
                          zyp = P.above(z, P.sy);
            const float zzm = P.one_below(z), zzp = P.one_above(z);
            const PairOperator op(A, P);
            const double2v qp = first ? double2v{0.0, 0.0} : ld_stream((const double2v *)(qprev + c));
            const double2v rc = ld_stream((const double2v *)(r + c));
            const double2v zc = {on0 ? (double)zl.x : 0.0, on1 ? (double)zl.y : 0.0};
            const double2v wc =
                op.apply(zc, widen(zxm), widen(zxp), widen(zym), widen(zyp), (double)zzm, (double)zzp);
            st_stream((double2v *)(w + c), wc);
            v[0] = zc.x * wc.x + zc.y * wc.y;
            if (!first) v[1] = zc.x * qp.x + zc.y * qp.y;
            v[2] = zc.x * rc.x + zc.y * rc.y;
        }
        block_sum<3>(v);
        if (flat_tid() == 0)
#pragma unroll
            for (int q = 0; q < 3; q++) partials[(size_t)q * nb + block] = v[q];
    }
}

// The iteration's scalars from its dots: p = z - beta p_prev with beta =
// z.q_prev / p_prev.q_prev makes p A-orthogonal to p_prev; then p.q = z.w -
// beta z.q_prev, and p.r = z.r because p_prev.r = 0 after the previous step.
struct Recurrence {
    double alpha, beta, pq;
};
__device__ __forceinline__ Recurrence recurrence(const double (&v)[3], double pq_prev, int first) {
    Recurrence c{0.0, 0.0, v[0]};
    if (!first && pq_prev != 0.0) {
        c.beta = v[1] / pq_prev;
        c.pq = v[0] - c.beta * v[1];
    }
    c.alpha = c.pq != 0.0 ? v[2] / c.pq : 0.0;
    return c;
}

// The update is pointwise: it runs over the flat cell index with two
// consecutive cells per lane (16-byte loads and stores of the FP64 vectors),
// one pair per thread (kUpdateCells per block). A wavefront whose 128 cells
// are all inactive is skipped (q, r stay 0 there). With b32 it also
// stores the new residual rounded to FP32: the right-hand side the next
// V-cycle starts from, which then need not read the FP64 residual.
//
// Neither the direction p nor the solution x is formed here: both are sums of
// the iterations' z with scalars, so the z are kept (FP32, as the V-cycle
// stores them) and k_fcg_flush runs p = z - beta p, x += alpha p for up to
// kRing iterations in one pass. The update then moves 40 B per cell and the
// FP32 copies' 12 instead of 80 (z, p in and out, x every other iteration).
//
// kFold: the block adds the matvec's partials (mv, nb_mv of them) and forms
// the scalars itself (and block 0 stores them) instead of a finalize launch
// before it.
constexpr unsigned kUpdateCells = 2 * kBlock;

template <bool kFold>
__global__ __launch_bounds__(kBlock) void k_fcg_update(size_t n, const float *__restrict__ active,
                                                       const double *__restrict__ w,
                                                       double *__restrict__ q,
                                                       double *__restrict__ r,
                                                       float *__restrict__ b32,
                                                       float *__restrict__ x0, float c0, int first, int iter,
                                                       const double *__restrict__ mv, unsigned nb_mv,
                                                       double *__restrict__ partials,
                                                       KrylovScalars *sc,
                                                       const double *gate) {
    const int ci = iter % kCoefs;
    const size_t c = (size_t)blockIdx.x * kUpdateCells + 2 * (size_t)flat_tid();
    const bool pair = c + 1 < n;  // else at most the grid's last cell
    double alpha, beta;
    double2v wc = {0.0, 0.0}, r0 = {0.0, 0.0}, qq = {0.0, 0.0};
    if constexpr (kFold) {
        // every load at once: the vectors' beside the gate's and the partials'
        const double stop = load_gate(gate, sc);
        FoldLoad<3> f;
        fold_load<3>(mv, nb_mv, f);
        const double pq_prev = sc->pq[(iter + kCoefs - 1) % kCoefs];
        const size_t cl = pair ? c : 0;  // (a grid of one cell: the allocations hold a pair)
        wc = ld_stream((const double2v *)(w + cl));
        r0 = ld_stream((const double2v *)(r + cl));
        qq = ld_stream((const double2v *)(q + cl));
        pin(stop);
        pin(f);
        pin(pq_prev);
        pin(wc);
        pin(r0);
        pin(qq);
        if (stop != 0.0) return;
        double v[3];
        fold_sum<3>(mv, nb_mv, f, v);
        const Recurrence c = recurrence(v, first ? 0.0 : pq_prev, first);
        alpha = c.alpha;
        beta = c.beta;
        if (blockIdx.x == 0 && threadIdx.x == 0) {
            sc->alpha[ci] = alpha;
            sc->beta[ci] = beta;
            sc->pq[ci] = c.pq;
        }
    } else {
        if (gated(gate)) return;
        alpha = sc->alpha[ci];
        beta = sc->beta[ci];
    }
    double v[1] = {0.0};
    bool act = c < n;
    float2v dg = {0.f, 0.f};  // FP32 diagonal (the activity flag)
    if (active) {
        if (pair) dg = *(const float2v *)(active + c);
        else if (c < n) dg.x = active[c];
        act = dg.x > 0.f || dg.y > 0.f;
    }
    if (__any(act)) {
        if (pair) {
            if constexpr (!kFold) {
                wc = ld_stream((const double2v *)(w + c));
                r0 = ld_stream((const double2v *)(r + c));
                if (!first) qq = ld_stream((const double2v *)(q + c));
            }
            double2v qc = wc;
            if (!first) {
                qc.x = wc.x - beta * qq.x;
                qc.y = wc.y - beta * qq.y;
            }
            double2v rc;
            rc.x = r0.x - alpha * qc.x;
            rc.y = r0.y - alpha * qc.y;
            st_stream((double2v *)(q + c), qc);
            st_stream((double2v *)(r + c), rc);
            if (b32) {
                const float2v bf = {(float)rc.x, (float)rc.y};
                *(float2v *)(b32 + c) = bf;
                if (x0) {
                    const float2v xf = {c0 * rcp_or_zero(dg.x) * bf.x, c0 * rcp_or_zero(dg.y) * bf.y};
                    *(float2v *)(x0 + c) = xf;
                }
            }
            v[0] += rc.x * rc.x;
            v[0] += rc.y * rc.y;
        } else if (c < n) {
            const double qc = first ? w[c] : w[c] - beta * q[c];
            q[c] = qc;
            const double rc = r[c] - alpha * qc;
            r[c] = rc;
            if (b32) {
                b32[c] = (float)rc;
                if (x0) x0[c] = c0 * rcp_or_zero(dg.x) * b32[c];
            }
            v[0] += rc * rc;
        }
    }
    block_partials<1>(v, partials);
}

// The same update on the listed blocks of kUpdateCells cells, as the matvec's
// (256^3 pool: 46 us, 50 with a block for each; the list's bytes: 51).
static_assert(kUpdateCells == kListCells, "the lists' blocks");
__global__ __launch_bounds__(kBlock) void k_fcg_update_list(size_t n, const unsigned *__restrict__ blocks,
                                                            const float *__restrict__ active,
                                                            const double *__restrict__ w, double *__restrict__ q,
                                                            double *__restrict__ r, float *__restrict__ b32,
                                                            float *__restrict__ x0, float c0, int first, int iter,
                                                            double *__restrict__ partials,
                                                            const KrylovScalars *__restrict__ sc,
                                                            const double *gate) {
    if (gated(gate)) return;
    const double alpha = sc->alpha[iter % kCoefs], beta = sc->beta[iter % kCoefs];
    const unsigned count = blocks[0];
    for (unsigned u = blockIdx.x; u < count; u += gridDim.x) {
        const unsigned block = blocks[1 + u];
        const size_t c = (size_t)block * kUpdateCells + 2 * (size_t)flat_tid();
        const bool pair = c + 1 < n;  // else at most the grid's last cell
        double v[1] = {0.0};
        float2v dg = {0.f, 0.f};
        if (pair) dg = *(const float2v *)(active + c);
        else if (c < n) dg.x = active[c];
        if (__any(dg.x > 0.f || dg.y > 0.f)) {
            if (pair) {
                const double2v wc = ld_stream((const double2v *)(w + c)), r0 = ld_stream((const double2v *)(r + c));
                double2v qc = wc;
                if (!first) {
                    const double2v qq = ld_stream((const double2v *)(q + c));
                    qc.x = wc.x - beta * qq.x;
                    qc.y = wc.y - beta * qq.y;
                }
                double2v rc;
                rc.x = r0.x - alpha * qc.x;
                rc.y = r0.y - alpha * qc.y;
                st_stream((double2v *)(q + c), qc);
                st_stream((double2v *)(r + c), rc);
                if (b32) {
                    const float2v bf = {(float)rc.x, (float)rc.y};
                    *(float2v *)(b32 + c) = bf;
                    if (x0) {
                        const float2v xf = {c0 * rcp_or_zero(dg.x) * bf.x, c0 * rcp_or_zero(dg.y) * bf.y};
                        *(float2v *)(x0 + c) = xf;
                    }
                }
                v[0] += rc.x * rc.x;
                v[0] += rc.y * rc.y;
            } else if (c < n) {
                const double qc = first ? w[c] : w[c] - beta * q[c];
                q[c] = qc;
                const double rc = r[c] - alpha * qc;
                r[c] = rc;
                if (b32) {
                    b32[c] = (float)rc;
                    if (x0) x0[c] = c0 * rcp_or_zero(dg.x) * b32[c];
                }
                v[0] += rc * rc;
            }
        }
        block_sum<1>(v);
        if (flat_tid() == 0) partials[block] = v[0];
    }
}

// p = z_k - beta_k p, x += alpha_k p for K iterations (numbers i0 .. i0 + K - 1,
// their z at z + k stride), in the order and arithmetic of an update per
// iteration. K is k0 or, with `need` (the stop flag: the launch returns while
// it is down), k0 plus the iterations of the batch before it. has_p: p0 holds
// the direction before them; store_p: it receives the last one. zero_x: x
// starts from 0 (and every cell is written); else a wavefront without active
// cells is skipped. z counts as 0 at inactive cells.
__global__ __launch_bounds__(kBlock) void k_fcg_flush(size_t n, const float *__restrict__ active,
                                                      const float *__restrict__ z, size_t stride,
                                                      double *__restrict__ p0, int has_p, int store_p,
                                                      double *__restrict__ x, int zero_x, int i0, int k0,
                                                      const KrylovScalars *__restrict__ sc, const double *need) {
    if (need && *need == 0.0) return;
    const int K = min(need ? k0 + (int)sc->iters : k0, kRing);  // uniform
    const size_t c = (size_t)blockIdx.x * kUpdateCells + 2 * (size_t)flat_tid();
    const bool pair = c + 1 < n;
    bool act = c < n;
    float2v dg = {1.f, 1.f};
    if (active) {
        dg = float2v{0.f, 0.f};
        if (pair) dg = *(const float2v *)(active + c);
        else if (c < n) dg.x = active[c];
        act = dg.x > 0.f || dg.y > 0.f;
    }
    if (zero_x ? !(c < n) : !__any(act)) return;
    if (pair) {
        float2v zk[kRing];
#pragma unroll
        for (int k = 0; k < kRing; k++)
            zk[k] = k < K && act ? ld_stream((const float2v *)(z + k * stride + c)) : float2v{0.f, 0.f};
        double2v p = {0.0, 0.0}, xn = {0.0, 0.0};
        if (has_p) p = ld_stream((const double2v *)(p0 + c));
        if (!zero_x) xn = ld_stream((const double2v *)(x + c));
#pragma unroll
        for (int k = 0; k < kRing; k++) {
            if (k >= K) break;
            const double alpha = sc->alpha[(i0 + k) % kCoefs], beta = sc->beta[(i0 + k) % kCoefs];
            p.x = (double)(dg.x > 0.f ? zk[k].x : 0.f) - beta * p.x;
            p.y = (double)(dg.y > 0.f ? zk[k].y : 0.f) - beta * p.y;
            xn.x += alpha * p.x;
            xn.y += alpha * p.y;
        }
        if (store_p) st_stream((double2v *)(p0 + c), p);
        st_stream((double2v *)(x + c), xn);
    } else if (c < n) {
        double p = has_p ? p0[c] : 0.0, xn = zero_x ? 0.0 : x[c];
        for (int k = 0; k < K; k++) {
            const double zc = dg.x > 0.f ? (double)z[k * stride + c] : 0.0;
            p = zc - sc->beta[(i0 + k) % kCoefs] * p;
            xn += sc->alpha[(i0 + k) % kCoefs] * p;
        }
        if (store_p) p0[c] = p;
        x[c] = xn;
    }
}

__global__ __launch_bounds__(kBlock) void k_jacobi(CellGrid cg, Dims d, Op32 A,
                                                   const double *__restrict__ r,
                                                   float *__restrict__ z, const double *gate) {
    if (gated(gate)) return;
    int k, j, i0;
    cell_tile(cg, k, j, i0);
    if (k >= d.nz || j >= d.ny) return;
    for (int i = i0, ie = min(i0 + cg.planes, d.nx); i < ie; i++) {
        const size_t c = d.idx(i, j, k);
        const float dg = A.diag[c];
        z[c] = dg > 0.f ? (float)(r[c] / (double)dg) : 0.f;
    }
}

// One block: add the partials and advance the scalar recurrences.
// The finalize kernel is one block of kFinalizeThreads (wide, so the partial
// sums of the largest grids take few rounds of loads).
constexpr int kFinalizeThreads = 1024;

// Start of a batch of gated iterations: the threshold on ||r||^2 (tol2 times
// the ||b||^2 of the solve's first residual), the counters and the stop flag
// cleared (one thread; the host need not know ||b|| yet). first: nor has it
// seen that residual, so the flag is up where no iteration is needed.
__global__ __launch_bounds__(64) void k_batch_begin(KrylovScalars *sc, double tol2, double stall_rr, int first) {
    if (threadIdx.x == 0) {
        const double stop_rr = tol2 * sc->bb;
        sc->stop = first && (sc->bb == 0.0 || sc->rr <= stop_rr) ? 1.0 : 0.0;
        sc->stop_rr = stop_rr;
        sc->iters = 0.0;
        sc->ok = 0.0;
        sc->stall_rr = stall_rr;
        sc->stalled = 0.0;
    }
}

__global__ __launch_bounds__(kFinalizeThreads) void k_finalize(int op, unsigned nb, int first, int iter,
                                                     const double *__restrict__ partials,
                                                     KrylovScalars *sc, const double *gate,
                                                     KrylovScalars *host, const double *need, double tol) {
    if (need && *need == 0.0) return;
    // what the host reads after this launch (host: its pinned copy, or null)
    auto tell_host = [&] {
        if (!host) return;
        host->rr = sc->rr;
        host->bb = sc->bb;
        host->active = sc->active;
        host->iters = sc->iters;
        host->stalled = sc->stalled;
        host->stop = sc->stop;
        host->check_rr = sc->check_rr;
        host->ok = sc->ok;
    };
    if (gated(gate)) {
        if (flat_tid() == 0) tell_host();
        return;
    }
    double v[3] = {0.0, 0.0, 0.0};
    if (op != FIN_UPDATE) {
        sum_partials<3, kFinalizeThreads, 16>(partials, nb, v);
    } else {
        double t[1];
        sum_partials<1, kFinalizeThreads, 16>(partials, nb, t);
        v[0] = t[0];
    }
    if (flat_tid() != 0) return;
    if (op == FIN_RESIDUAL) {
        sc->rr = v[0];
        sc->bb = v[1];
        sc->active = v[2];
        sc->check_rr = v[0];
        sc->ok = sqrt(v[0] / v[1]) <= tol ? 1.0 : 0.0;
    } else if (op == FIN_MATVEC) {
        const Recurrence c = recurrence(v, first ? 0.0 : sc->pq[(iter + kCoefs - 1) % kCoefs], first);
        sc->zw = v[0];
        sc->zq = v[1];
        sc->zr = v[2];
        sc->alpha[iter % kCoefs] = c.alpha;
        sc->beta[iter % kCoefs] = c.beta;
        sc->pq[iter % kCoefs] = c.pq;
    } else {
        const double rr_prev = sc->rr;
        sc->rr = v[0];
        sc->iters += 1.0;
        if (gate && v[0] <= sc->stop_rr) sc->stop = 1.0;  // later gated kernels return at once
        if (gate && sc->stall_rr > 0.0 && v[0] > sc->stall_rr * rr_prev) {
            sc->stalled = 1.0;  // the host switches to the plain V-cycle after the batch
            sc->stop = 1.0;
        }
    }
    tell_host();
}

// Above kStageMin partials the sums take two launches: kStageThreads-wide
// blocks add fixed chunks of kStageChunk partials each (every block one
// round of loads instead of the single block's many), the finalize adds the
// chunks' sums. The order is fixed by nb, so results stay deterministic.
constexpr unsigned kStageMin = 4096, kStageChunk = 1024, kStageMaxBlocks = 64;
constexpr int kStageThreads = 1024;

template <int N>
__global__ __launch_bounds__(kStageThreads) void k_partials_stage(unsigned nb, unsigned chunk,
                                                                  const double *__restrict__ partials,
                                                                  double *__restrict__ out,
                                                                  const double *gate) {
    if (gated(gate)) return;
    const unsigned b0 = blockIdx.x * chunk;  // < nb: the launcher sizes the grid
    const unsigned n = min(chunk, nb - b0);
    double v[N];
    sum_partials<N, kStageThreads, 8>(partials + b0, n, v, nb);
    if (flat_tid() == 0)
#pragma unroll
        for (int q = 0; q < N; q++) out[(size_t)q * gridDim.x + blockIdx.x] = v[q];
}

// `partials` holds the N sums of op for nb blocks ([q * nb + b]); the stage
// writes its sums after them (reduction_partials leaves room).
void finalize(hipStream_t st, int op, unsigned nb, int first, int iter, double *partials, KrylovScalars *sc,
              const double *gate = nullptr, KrylovScalars *host = nullptr, const double *need = nullptr,
              double tol = 0.0) {
    const int N = op == FIN_UPDATE ? 1 : 3;
    if (nb > kStageMin) {
        const unsigned chunk = std::max(kStageChunk, (nb + kStageMaxBlocks - 1) / kStageMaxBlocks);
        const unsigned G = (nb + chunk - 1) / chunk;
        double *out = partials + (size_t)N * nb;
        if (N == 3)
            hipLaunchKernelGGL(k_partials_stage<3>, dim3(G), dim3(kStageThreads), 0, st, nb, chunk, partials, out,
                               gate);
        else
            hipLaunchKernelGGL(k_partials_stage<1>, dim3(G), dim3(kStageThreads), 0, st, nb, chunk, partials, out,
                               gate);
        SFP_LAUNCH_CHECK();
        partials = out;
        nb = G;
    }
    hipLaunchKernelGGL(k_finalize, dim3(1), dim3(kFinalizeThreads), 0, st, op, nb, first, iter,
                       partials, sc, gate, host, need, tol);
    SFP_LAUNCH_CHECK();
}

}  // namespace

// FCG matvec: the flat kernel where z rows hold whole cell pairs (nz even;
// 11 % faster than x-plane tiles at 256^3 and 9 % at 384^3 on MI355X), else
// x-plane tiles of 4 planes per block (more blocks in flight than the 16 of the
// other reductions: 6 % faster at 256^3). (With odd nz the flat order of the
// sums is not for use: see the x-plane stencils.)
static bool matvec_flat(Dims d) { return d.nz % 2 == 0; }
static Launch matvec_launch(Dims d) { return cell_launch(d, 0, 4); }
static unsigned matvec_blocks(Dims d) {
    return matvec_flat(d) ? (unsigned)((d.cells() + kMatvecCells - 1) / kMatvecCells)
                          : matvec_launch(d).blocks();
}
// Blocks of a launch over the listed ones: as many as run at once (eight of four
// wavefronts per CU), or the grid's where that is less.
static unsigned list_launch(unsigned nb) { return std::min(nb, 8u * 256); }
static unsigned update_blocks(Dims d) { return (unsigned)((d.cells() + kUpdateCells - 1) / kUpdateCells); }

size_t reduction_partials(Dims d) {
    // The matvec's partials, the update's after them (a folded update reads
    // the former while it writes the latter) or the largest other set, then
    // room for the two-stage finalize's chunk sums.
    return std::max(3 * (size_t)cell_launch(d, kReducePlanes).blocks(),
                    3 * (size_t)matvec_blocks(d) + (size_t)update_blocks(d)) +
           3 * (size_t)kStageMaxBlocks;
}

size_t list_sums(Dims d) { return 3 * (size_t)matvec_blocks(d) + update_blocks(d) + 4 * (size_t)kStageMaxBlocks; }

bool fold_pays(Dims d) { return std::max(matvec_blocks(d), update_blocks(d)) <= kFoldMax; }
FoldArgs update_fold(Dims d, double *partials, KrylovScalars *sc) {
    return FoldArgs{partials + 3 * (size_t)matvec_blocks(d), update_blocks(d), sc};
}

void launch_batch_begin(hipStream_t st, KrylovScalars *sc, double tol2, double stall_rr, bool first) {
    hipLaunchKernelGGL(k_batch_begin, dim3(1), dim3(64), 0, st, sc, tol2, stall_rr, first ? 1 : 0);
    SFP_LAUNCH_CHECK();
}

void launch_residual64(hipStream_t st, Dims d, Op64 A, const double *b, const double *x,
                       double *r, double *partials, KrylovScalars *sc, KrylovScalars *host, float *b32,
                       float *x0, const float *diag32, float c0, const double *need, double tol) {
    if (x0 && (!b32 || !diag32)) throw ArgError("launch_residual64: x0 needs b32 and the diagonal");
    if (d.cells() >= (size_t(1) << 32) - 64) throw ArgError("launch_residual64: grid too large");
    for (const void *a : {(const void *)A.diag, (const void *)A.cpl[0], (const void *)A.cpl[1],
                          (const void *)A.cpl[2], (const void *)b, (const void *)x, (const void *)r})
        if ((uintptr_t)a % 16) throw ArgError("launch_residual64: FP64 array not 16-byte aligned");
    if ((uintptr_t)b32 % 8 || (uintptr_t)x0 % 8 || (uintptr_t)diag32 % 8)
        throw ArgError("launch_residual64: b32, x0 or the diagonal not 8-byte aligned");
    if (matvec_flat(d)) {
        const unsigned nb = (unsigned)((d.cells() + kResidualCells - 1) / kResidualCells);
        if (A.chunks.blocks && !r && !b32) {
            partials = A.chunks.sums;
            hipLaunchKernelGGL(k_residual64_flat<true>, dim3(list_launch(nb)), dim3(kBlock), 0, st, d, A, b, x, r,
                               partials, b32, x0, diag32, c0, nb, need);
        } else {
            hipLaunchKernelGGL(k_residual64_flat<false>, dim3(nb), dim3(kBlock), 0, st, d, A, b, x, r, partials,
                               b32, x0, diag32, c0, nb, need);
        }
        SFP_LAUNCH_CHECK();
        finalize(st, FIN_RESIDUAL, nb, 0, 0, partials, sc, nullptr, host, need, tol);
        return;
    }
    const Launch L = cell_launch(d, kReducePlanes);
    hipLaunchKernelGGL(k_residual64, L.grid, L.block, 0, st, L.cg, d, A, b, x, r, partials, b32, x0, diag32, c0,
                       need);
    SFP_LAUNCH_CHECK();
    finalize(st, FIN_RESIDUAL, L.blocks(), 0, 0, partials, sc, nullptr, host, need, tol);
}

void launch_fcg_matvec(hipStream_t st, Dims d, Op64 A, const float *active, const float *z,
                       const double *r, const double *qprev, double *w, int first, int iter, bool fold,
                       double *partials, KrylovScalars *sc, const double *gate, hipEvent_t kernel_done) {
    const bool list = A.chunks.blocks && matvec_flat(d);
    const unsigned nb = matvec_blocks(d);
    if (list) partials = A.chunks.sums;
    if (d.cells() >= (size_t(1) << 32) - 64) throw ArgError("launch_fcg_matvec: grid too large");
    // pairs of cells: 16-byte (8-byte for z and the flags) aligned vectors
    for (const void *a : {(const void *)A.diag, (const void *)A.cpl[0], (const void *)A.cpl[1],
                          (const void *)A.cpl[2], (const void *)r, (const void *)qprev, (const void *)w})
        if ((uintptr_t)a % 16) throw ArgError("launch_fcg_matvec: FP64 array not 16-byte aligned");
    if ((uintptr_t)z % 8 || (uintptr_t)active % 8)
        throw ArgError("launch_fcg_matvec: z or the diagonal not 8-byte aligned");
    if (list) {
        hipLaunchKernelGGL(k_fcg_matvec_flat<true>, dim3(list_launch(nb)), dim3(kBlock), 0, st, d, A, active, z, r,
                           qprev, w, first, partials, nb, gate);
    } else if (matvec_flat(d)) {
        hipLaunchKernelGGL(k_fcg_matvec_flat<false>, dim3(nb), dim3(kBlock), 0, st, d, A, active, z, r, qprev, w,
                           first, partials, nb, gate);
    } else {
        const Launch L = matvec_launch(d);
        hipLaunchKernelGGL(k_fcg_matvec, L.grid, L.block, 0, st, L.cg, d, A, active, z, r, qprev, w, first,
                           partials, gate);
    }
    SFP_LAUNCH_CHECK();
    if (kernel_done) SFP_HIP(hipEventRecord(kernel_done, st));
    if (!fold) finalize(st, FIN_MATVEC, nb, first, iter, partials, sc, gate);
}

void launch_fcg_update(hipStream_t st, Dims d, const float *active, const Chunks &chunks, const double *w, double *q, double *r,
                       float *b32, float *x0, float c0, int first, int iter, bool fold, double *partials,
                       KrylovScalars *sc, const double *gate, hipEvent_t kernel_done, KrylovScalars *host) {
    // two cells per lane: 16-byte (8-byte for the FP32 ones) aligned vectors
    for (const void *a : {(const void *)w, (const void *)q, (const void *)r})
        if ((uintptr_t)a % 16) throw ArgError("launch_fcg_update: FP64 vector not 16-byte aligned");
    if ((uintptr_t)active % 8 || (uintptr_t)b32 % 8 || (uintptr_t)x0 % 8)
        throw ArgError("launch_fcg_update: the diagonal, b32 or x0 not 8-byte aligned");
    if (x0 && (!b32 || !active)) throw ArgError("launch_fcg_update: x0 needs b32 and the diagonal");
    if (chunks.blocks && (fold || !active)) throw ArgError("launch_fcg_update: no list here");
    const unsigned nb = update_blocks(d), nb_mv = matvec_blocks(d);
    double *out = partials + 3 * (size_t)nb_mv;
    if (chunks.blocks) {
        out = chunks.sums + 3 * (size_t)nb_mv + 3 * kStageMaxBlocks;
        hipLaunchKernelGGL(k_fcg_update_list, dim3(list_launch(nb)), dim3(kBlock), 0, st, d.cells(), chunks.blocks,
                           active, w, q, r, b32, x0, c0, first, iter, out, sc, gate);
    } else if (fold)
        hipLaunchKernelGGL(k_fcg_update<true>, dim3(nb), dim3(kBlock), 0, st, d.cells(), active, w, q, r, b32, x0,
                           c0, first, iter, partials, nb_mv, out, sc, gate);
    else
        hipLaunchKernelGGL(k_fcg_update<false>, dim3(nb), dim3(kBlock), 0, st, d.cells(), active, w, q, r, b32, x0,
                           c0, first, iter, partials, nb_mv, out, sc, gate);
    SFP_LAUNCH_CHECK();
    if (kernel_done) SFP_HIP(hipEventRecord(kernel_done, st));
    if (!fold)
        finalize(st, FIN_UPDATE, nb, 0, 0, out, sc, gate, host);
}

void launch_fcg_norm(hipStream_t st, Dims d, double *partials, KrylovScalars *sc, const double *gate,
                     KrylovScalars *host) {
    finalize(st, FIN_UPDATE, update_blocks(d), 0, 0, partials + 3 * (size_t)matvec_blocks(d), sc, gate, host);
}

void launch_fcg_flush(hipStream_t st, Dims d, const float *active, const float *z, size_t stride, int K, int i0,
                      double *p, bool has_p, bool store_p, double *x, bool zero_x, const KrylovScalars *sc,
                      const double *need) {
    if (K < (need ? 0 : 1) || K > kRing) throw ArgError("launch_fcg_flush: bad iteration count");
    if ((has_p || store_p) && !p) throw ArgError("launch_fcg_flush: no direction");
    if ((uintptr_t)z % 8 || stride % 2 || (uintptr_t)active % 8 || (uintptr_t)p % 16 || (uintptr_t)x % 16)
        throw ArgError("launch_fcg_flush: vectors not aligned");
    hipLaunchKernelGGL(k_fcg_flush, dim3(update_blocks(d)), dim3(kBlock), 0, st, d.cells(), active, z, stride, p,
                       has_p ? 1 : 0, store_p ? 1 : 0, x, zero_x ? 1 : 0, i0, K, sc, need);
    SFP_LAUNCH_CHECK();
}

void launch_jacobi(hipStream_t st, Dims d, Op32 A, const double *r, float *z, const double *gate) {
    Launch L = cell_launch(d);
    hipLaunchKernelGGL(k_jacobi, L.grid, L.block, 0, st, L.cg, d, A, r, z, gate);
    SFP_LAUNCH_CHECK();
}

}  // namespace sfp
