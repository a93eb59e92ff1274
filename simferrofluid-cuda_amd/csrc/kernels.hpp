// Host-side launchers of the gfx950 kernels (defined in the .hip files).
#pragma once
#include "sfp_internal.hpp"

namespace sfp {

// Iteration kernels take an optional `gate` (&KrylovScalars::stop): when it
// points at a nonzero value the kernel returns at once (batched iterations
// after convergence). Null = always run.

// ---------------------------------------------------------------- multigrid (mg.hip)
// Chebyshev step modes.
enum SmoothMode : int {
    SM_FIRST = 1,      // input iterate is the zero-start first step c0 D^{-1} b, fused in
    SM_READ_D = 2,     // previous direction read from dvec
    SM_WRITE_D = 4,    // store the new direction
    SM_PROLONG = 8,    // input iterate is x + P e (coarse correction fused in)
    SM_XFIRST = 16     // input iterate is the zero-start first step c0 D^{-1} b, stored
                       // in xin (by the FCG kernels on the fine level, the restriction on
                       // the coarse ones); the previous direction equals it
};

// x = c0 * D^{-1} b from a zero start; at the fine level b is first rounded
// from the FP64 residual r64 (and stored to b).
void launch_smooth_first(hipStream_t s, Dims d, Op32 A, const double *r64, float *b, float *x,
                         float c0, const double *gate = nullptr);
// xout = x + d', d' = cd * d + cr * D^{-1} (b - A x) with x = xin, xin + P e,
// or the fused zero-start step c0 D^{-1} b (SM_FIRST; b from r64 when given).
void launch_smooth(hipStream_t s, int mode, Dims d, Op32 A, const double *r64, float *b,
                   const float *xin, float *xout, float *dvec, float c0, float cd, float cr,
                   const float *ecoarse, const double *gate = nullptr);
// Two steps in one pass: x2 = x1 + d2, d2 = cdA d1 + crA D^{-1} (b - A x1), then
// x3 = x2 + cdB d2 + crB D^{-1} (b - A x2); d2 is not stored. x3 must differ
// from x1. Same results as the two launch_smooth calls, bit for bit.
// With x1 == d1 (the stored zero-start iterate, which is also the previous
// direction) the pair is the first two steps of a cycle.
// pair_pays: grids on which it beats the two launches on MI355X. The 64 x 16
// tiles overlap by one cell per side: equal at 128^3, faster above. Whole rows
// of 80..128 cells: 20 us against 23 at 128^3, 45 against 82 at 256 x 256 x 128
// (magnetic solves 1.03x and 1.17x), 1.01x at 100 x 105 x 100.
bool row_pair(Dims d);
inline bool pair_pays(Dims d) {
    return d.nz >= 64 && d.cells() > ((size_t)1 << (row_pair(d) && d.nz <= 128 ? 20 : 21));
}
// Grids on which launch_smooth runs its steps (all but the fused first step)
// over the flat cell index: fewer than 2^32 cells. whole_groups: with the
// prolongation too (nz a multiple of 4).
bool flat_step(Dims d);
bool whole_groups(Dims d);
// Grids with z rows of 80..256 cells in groups of four run it over whole rows (k_smooth_pair_rows); rowact (null: all active) marks the z rows
// holding an active cell (launch_row_activity), whose loads the others skip.
void launch_smooth_pair(hipStream_t s, Dims d, Op32 A, const float *b, const float *x1, float *x3,
                        const float *d1, float cdA, float crA, float cdB, float crB,
                        const double *gate = nullptr, const unsigned char *rowact = nullptr,
                        const int *segments = nullptr);
// The lists of a level's active chunks, restriction units and FCG blocks (see
// Chunks; flags: a byte for each, lists: an entry for each and one more).
unsigned restrict_quads(Dims d);
struct ActiveLists {
    unsigned char *flags, *quad_flags, *block_flags;
    unsigned *list, *quads, *blocks;
};
void launch_active_chunks(hipStream_t s, Dims d, const float *diag32, const ActiveLists &a);
// Doubles of Chunks::sums.
size_t list_sums(Dims d);
// k_smooth_pair_rows' work on a level with inactive rows: segments[0] runs of x
// planes of a tile column, each (column, first plane, end) from segments[1 + 3 q]
// on. pair_segments_max: the most of them, 0 where they are not used.
unsigned pair_segments_max(Dims d);
void launch_pair_segments(hipStream_t s, Dims d, const unsigned char *rowact, int *segments);
// rowact[i ny + j] = 1 when the z row (i, j) holds an active cell (diag32 > 0)
void launch_row_activity(hipStream_t s, Dims d, const float *diag32, unsigned char *rowact);
// The last pre-smoothing step and the restriction in one pass:
// x2 = x1 + cd d1 + cr D^{-1} (b - A x1), then bc = R (b - A x2) (the coarse
// right-hand side, as launch_restrict). Same results as launch_smooth
// (SM_READ_D) then launch_restrict, bit for bit; x2 must differ from x1.
void launch_smooth_restrict(hipStream_t s, Dims d, Op32 A, const float *b, const float *x1,
                            float *x2, const float *d1, float cd, float cr, float *bc,
                            const double *gate = nullptr);
// x += P e on active cells (diag32 > 0), in place.
void launch_prolong_add(hipStream_t s, Dims d, const float *diag32, const unsigned *list, const float *ecoarse,
                        float *x, const double *gate = nullptr);
// bc = R (b - A x): sum of the residuals of the (up to 8) children. With
// x0c, also x0c = c0 Dc^-1 bc (diag32c: the coarse FP32 diagonal), the first
// Chebyshev iterate of the coarse level's cycle, as the FCG update stores it
// on the fine level.
void launch_restrict(hipStream_t s, Dims df, Op32 A, const float *b, const float *x, float *bc,
                     const double *gate = nullptr, float *x0c = nullptr,
                     const float *diag32c = nullptr, float c0 = 0.f);
// Galerkin coarsening by 2x2x2 aggregation, scaled: writes the coarse FP64
// and FP32 operators, the couplings scaled by `scale` and each row's sum
// (diagonal minus couplings) by `rs_scale` (scale: scale * P^T A P).
// (rows: of the assembly before it, which it tells the host of as it starts)
void launch_coarsen(hipStream_t s, Dims df, Op64 Af, const float *diag32f, Dims dc,
                    double scale, double rs_scale, double *diag64c, double *const cpl64c[3],
                    float *diag32c, float *const cpl32c[3], RowsFlag rows = {});
// Dense inverse of the coarsest operator (n = cells <= kMaxCoarse) into ainv (n*n floats).
constexpr int kMaxCoarse = 64;

// The coarse end of a V-cycle in one launch of one block: from its first level
// (cells, z rows padded to groups of four, <= kTailMaxCells) down to the
// coarsest and back, with the per-cell arithmetic of the separate smoothing,
// restriction and dense-solve launches. The level's result is left in lv[0].x1
// (tail_result); the other level vectors are not touched. The first level's b
// must already hold its right-hand side. The first level lives in registers (a
// group of four cells for each of 1024 threads), the others in LDS. (Two groups
// a thread, 8192 cells, spilled and took 33 us at 20^3, where two tile launches
// and the tail from 10^3 take 17.)
constexpr size_t kTailMaxCells = 4096;
constexpr int kTailMaxLevels = 8;
struct TailLevel {
    Dims d;
    Op32 A;
    float *b, *x0, *x1, *dv;
};
// The ||r||^2 of the update before a cycle, added by the cycle's first launch:
// nb partials (0: nothing to add), counted and compared to stop_rr as
// launch_fcg_norm does; the launch returns when that raises `stop`.
struct FoldArgs {
    const double *partials = nullptr;
    unsigned nb = 0;
    KrylovScalars *sc = nullptr;
};
struct TailArgs {
    int nlev = 0;  // levels in the tail, the last the coarsest
    TailLevel lv[kTailMaxLevels];
    // Chebyshev degree and coefficients: [0] for the first level, [1] below it
    int deg[2] = {3, 3};
    float cd[2][8] = {}, cr[2][8] = {};
    const float *ainv = nullptr;
    FoldArgs fold;
};
// LDS of the levels below the first: 8 padded arrays each (two with guards).
constexpr int kTailPoolFloats = 16384;
constexpr int kInvStride = 68;  // row stride of the dense inverse in LDS
constexpr __host__ __device__ int tail_level_floats(int padded_cells) { return 8 * padded_cells + 16; }
// Whether levels lv[0..nlev) (first to coarsest) can run as a tail.
bool tail_fits(const Dims *lv, int nlev);
void launch_vcycle_tail(hipStream_t s, const TailArgs &t, const double *gate = nullptr);
// The buffer that holds the tail's result for its first level.
inline float *tail_result(const TailArgs &t) { return t.lv[0].x1; }

// Several Chebyshev steps of one level in one launch, over overlapping tiles
// held in registers and LDS. start:
//   TILE_FIRST    from x = c0 D^-1 b, which is also the previous direction
//   TILE_PROLONG  from xin + P e (e on the coarse extents dc), cd[0] = 0
//   TILE_CONTINUE from xin with direction din
// then nsteps steps with coefficients cd[], cr[]; x to xout and, when dout is
// given, the direction to dout; with bc the restriction of the residual (the
// coarse right-hand side). Same results as launch_smooth and launch_restrict,
// bit for bit. xout must not alias xin, nor dout din.
enum TileStart : int { TILE_FIRST = 0, TILE_PROLONG = 1, TILE_CONTINUE = 2 };
constexpr int kTileMaxGroups = 2048;
struct TilePlan {
    int tx = 0, ty = 0, tz = 0;  // own cells of a tile (even; tz a multiple of 4)
    int hx = 0, hy = 0, hz = 0;  // halo (0 where one tile spans the axis)
    int bx = 0, by = 0, bz = 0;  // tiles along each axis
    int groups = 0;              // groups of four cells with the halo
};
struct TileArgs {
    Dims d, dc;
    Op32 A;
    TilePlan plan;
    const float *b = nullptr, *xin = nullptr, *din = nullptr, *e = nullptr;
    float *xout = nullptr, *dout = nullptr, *bc = nullptr;
    int start = TILE_FIRST, nsteps = 0;
    float c0 = 0.f, cd[8] = {}, cr[8] = {};
    FoldArgs fold;
};
// The tile of the least modelled cost for `steps` steps (and the restriction)
// on level d; its cost in microseconds.
TilePlan choose_tile(Dims d, int steps, bool restrict_after, double *cost = nullptr);
void launch_tile_steps(hipStream_t s, const TileArgs &a, const double *gate = nullptr);
void launch_coarse_invert(hipStream_t s, Dims d, Op64 A, float *ainv);
// On every level l < nlev: v[l][0..3][c] = 0 (and on level 0 w[c] = 0 when
// w is given) at the cells with diag32[l][c] == 0. start[l] is the first
// cell of level l in the launch (start[l + 1] = start[l] + n[l]).
constexpr int kClearMaxLevels = 16;
struct ClearArgs {
    int nlev = 0;
    unsigned start[kClearMaxLevels + 1] = {};
    unsigned n[kClearMaxLevels] = {};
    const float *diag32[kClearMaxLevels] = {};
    float *v[kClearMaxLevels][4] = {};
    double *w = nullptr;
};
void launch_clear_inactive(hipStream_t s, const ClearArgs &a);
void launch_coarse_solve(hipStream_t s, int n, const float *ainv, const float *b, float *x,
                         const double *gate = nullptr);

// ---------------------------------------------------------------- Krylov (krylov.hip)
// `host` (the residual, the update and the norm): a pinned copy of the scalars
// that the launch's finalize fills in (all but the recurrences' scalars; also
// behind a closed gate), so that the host reads them after a stream
// synchronization, without a copy (a launch of its own, 3 us, before it).
// Reduction kernels cover this many x planes per block (fewer partials).
constexpr int kReducePlanes = 0;  // automatic
// Doubles of partial-sum scratch a reduction over grid d needs.
size_t reduction_partials(Dims d);
// Before a batch of gated iterations: scalars->stop_rr = tol2 ||b||^2,
// ->stall_rr = stall_rr (0: no stall test), ->iters, ->ok, ->stalled and ->stop
// = 0; first (batch of a solve): stop is raised where ||r||^2 needs no iteration.
void launch_batch_begin(hipStream_t s, KrylovScalars *sc, double tol2, double stall_rr, bool first);
// r = b - A x (x may be null = 0); scalars->rr = r.r, scalars->bb = b.b;
// r may be null (only the sums).
// With b32, also b32 = r rounded to FP32 and, with x0, x0 = c0 D32^-1 b32
// (diag32: the FP32 diagonal): the right-hand side and first Chebyshev
// iterate of a V-cycle on r, as the FCG update stores them. With diag32 the
// active cells are counted too (scalars->active). scalars->check_rr = r.r, ->ok
// whether its root over ||b|| is at most tol. need: the launches return while
// *need is 0.
void launch_residual64(hipStream_t s, Dims d, Op64 A, const double *b, const double *x,
                       double *r, double *partials, KrylovScalars *sc, KrylovScalars *host = nullptr,
                       float *b32 = nullptr, float *x0 = nullptr, const float *diag32 = nullptr,
                       float c0 = 0.f, const double *need = nullptr, double tol = 0.0);
// w = A z; dots z.w, z.q_prev, z.r, and with them alpha, beta and p.q of
// iteration number iter (scalars->alpha[iter % kCoefs], ...). fold: only the
// partial sums (the update adds them).
// active: the FP32 diagonal (0 = inactive cell, where z counts as 0) to skip
// all-inactive wavefronts; null = every cell.
void launch_fcg_matvec(hipStream_t s, Dims d, Op64 A, const float *active, const float *z,
                       const double *r, const double *qprev, double *w, int first, int iter, bool fold,
                       double *partials, KrylovScalars *sc, const double *gate = nullptr,
                       hipEvent_t kernel_done = nullptr);
// q = w - beta q; r -= alpha q; rr = r.r (all-inactive wavefronts skipped when
// `active` is given); b32 (or null) receives r rounded to FP32 and x0 (or null)
// the first Chebyshev iterate c0 D^{-1} b32, with D the FP32 diagonal
// `active`. fold: the scalars are formed from the matvec's partials in the
// kernel, and of rr only the partial sums (launch_fcg_norm, or the next cycle's
// first launch, adds them).
void launch_fcg_update(hipStream_t s, Dims d, const float *active, const Chunks &chunks, const double *w, double *q, double *r,
                       float *b32, float *x0, float c0, int first, int iter, bool fold, double *partials,
                       KrylovScalars *sc, const double *gate = nullptr,
                       hipEvent_t kernel_done = nullptr, KrylovScalars *host = nullptr);
// (kernel_done, if given, is recorded after the stencil kernel and before
// the one-block finalize that forms the scalars.)
// rr from the update's partials; counts the update and raises `stop`.
void launch_fcg_norm(hipStream_t s, Dims d, double *partials, KrylovScalars *sc, const double *gate = nullptr,
                     KrylovScalars *host = nullptr);
// Grids whose reductions' partials the kernels that need the sums add
// themselves.
bool fold_pays(Dims d);
FoldArgs update_fold(Dims d, double *partials, KrylovScalars *sc);
// x += alpha_k p_k, p_k = z_k - beta_k p_{k-1} for the K <= kRing iterations
// i0 .. i0 + K - 1 whose z_k are at z + (k - i0) stride (see k_fcg_flush; need:
// K counts those before the current batch).
void launch_fcg_flush(hipStream_t s, Dims d, const float *active, const float *z, size_t stride, int K, int i0,
                      double *p, bool has_p, bool store_p, double *x, bool zero_x, const KrylovScalars *sc,
                      const double *need = nullptr);
// z = D^{-1} r on active cells (Jacobi preconditioner).
void launch_jacobi(hipStream_t s, Dims d, Op32 A, const double *r, float *z,
                   const double *gate = nullptr);

// ---------------------------------------------------------------- assembly (assemble.hip)
struct Faces {
    const double *a[3];
};
struct MutFaces {
    double *a[3];
};
// Post-projection steps (post.hip).
// valid[f] (face grid axis) = fraction < 1 and a liquid cell on either side.
void launch_velocity_valid(hipStream_t s, Dims d, int axis, const double *phi, const double *frac,
                           unsigned char *valid);
// `steps` sweeps of Extrapolation::Solve on one grid: valid (the mask) and
// scratch (same size) are both overwritten.
void launch_extrapolate(hipStream_t s, Dims g, double *data, unsigned char *valid,
                        unsigned char *scratch, double clear, int steps);
// Collider::Enforce; old is the velocity before the call (not aliasing vel).
void launch_collider_enforce(hipStream_t s, Dims d, double spacing, const double origin[3], Faces old,
                             Faces frac, Faces normal, Faces colvel, MutFaces vel);
// Geometry of MagneticField's own StaggeredGrid (core/MagneticField.cpp:11-16).
struct MagGeom {
    double face_origin[3][3];
    double ls_origin[3];  // cell grid of the level set
    double spacing, inv;
};
MagGeom mag_geometry(Dims d, double spacing, const double origin[3]);

// Pressure::SetUnKnowns + BuildProjectionMatrix; liquid[c] = phi <= 0;
// *err set to 1 when a liquid cell has an open face on the grid boundary.
void launch_pressure_assemble(hipStream_t s, Dims d, const double *phi, Faces frac, Faces vel,
                              Faces us, const Faces *jump, double vol_error, double *diag64,
                              double *const cpl64[3], double *rhs, float *diag32,
                              float *const cpl32[3], unsigned char *liquid, int *err, RowsFlag rows);
// Pressure::SetRightHandSide on the stored unknowns.
void launch_pressure_rhs(hipStream_t s, Dims d, const unsigned char *liquid, Faces frac,
                         Faces vel, Faces us, double vol_error, double *rhs);
// Pressure::ApplyProjection (p on the full grid, 0 at air cells); p_out (or
// null) receives a copy of p. need: the launches return while *need is 0.
void launch_pressure_apply(hipStream_t s, Dims d, const double *phi, Faces frac,
                           const Faces *jump, const unsigned char *liquid, const double *p,
                           MutFaces vel, int *err, double *p_out, const double *need);
// MagneticField::BuildMatrix coefficients, matrix and AssembleRHS.
void launch_magnetic_mu(hipStream_t s, Dims d, const MagGeom &g, const double *phi, double chi,
                        double band, MutFaces mu);
// dirichlet: the opt-in box condition phi = 0 (no pinned cell) instead of
// the reference's Neumann box faces with cell 0 pinned.
void launch_magnetic_assemble(hipStream_t s, Dims d, Faces mu, Faces hext, double spacing,
                              double *diag64, double *const cpl64[3], double *rhs,
                              float *diag32, float *const cpl32[3], int dirichlet = 0);
// MagneticField::AssignTotalField; copies of the potential to pot_out and of
// the field to out (each null: none). need as above.
void launch_magnetic_total_field(hipStream_t s, Dims d, double inv, const double *pot,
                                 Faces hext, MutFaces htot, double *pot_out, MutFaces out,
                                 const double *need);
// MagneticField::CalculateVertexPressures.
void launch_vertex_pressures(hipStream_t s, Dims d, const MagGeom &g, Faces htot, double chi,
                             int nverts, const double *pos, const double *nrm, double *out);

}  // namespace sfp
