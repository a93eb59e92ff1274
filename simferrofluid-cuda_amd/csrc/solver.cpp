// Hierarchy setup, V-cycle orchestration and the FP64 flexible CG.
#include "solver.hpp"

#include "learned.hpp"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>

namespace sfp {

void hip_fail(hipError_t e, const char *what, const char *file, int line) {
    char buf[512];
    std::snprintf(buf, sizeof(buf), "%s failed: %s (%s:%d)", what, hipGetErrorString(e), file, line);
    (void)hipGetLastError();  // (else the next launch's check would report it again)
    throw HipError(buf);
}

static thread_local int t_fail_after = -1;
void fail_allocation(int after) { t_fail_after = after; }
bool allocation_fails() { return t_fail_after >= 0 && t_fail_after-- == 0; }

// ---------------------------------------------------------------- Chebyshev
Cheby Cheby::make(int degree, double ratio) {
    // D^{-1}A of these weakly diagonally dominant M-matrices has spectrum in
    // (0, 2] (Gershgorin), so lambda_max = 2 is a safe bound needing no estimate.
    Cheby c;
    c.degree = std::max(1, std::min(degree, 8));
    const double lmax = 2.0, lmin = lmax / ratio;
    const double theta = 0.5 * (lmax + lmin), delta = 0.5 * (lmax - lmin);
    const double sigma = theta / delta;
    double rho = 1.0 / sigma;
    c.cd[0] = 0.f;
    c.cr[0] = (float)(1.0 / theta);
    for (int s = 1; s < c.degree; s++) {
        const double rn = 1.0 / (2.0 * sigma - rho);
        c.cd[s] = (float)(rn * rho);
        c.cr[s] = (float)(2.0 * rn / delta);
        rho = rn;
    }
    return c;
}

// ---------------------------------------------------------------- timers
void KernelTimer::begin(hipStream_t s, double b) {
    if (used + 2 > ev.size()) {
        for (int t = 0; t < 64; t++) {
            hipEvent_t e;
            SFP_HIP(hipEventCreate(&e));
            ev.push_back(e);
        }
    }
    if (bytes.size() < ev.size() / 2) bytes.resize(ev.size() / 2);
    bytes[used / 2] = b;
    SFP_HIP(hipEventRecord(ev[used], s));
}
void KernelTimer::end(hipStream_t s) {
    SFP_HIP(hipEventRecord(ev[used + 1], s));
    used += 2;
}
void KernelTimer::harvest() {
    // launches of a batch past its stop return at once: a duration under a
    // fifth of the median is such a launch, not a measurement of the kernel
    std::vector<float> ms(used / 2);
    for (size_t t = 0; t + 1 < used; t += 2) SFP_HIP(hipEventElapsedTime(&ms[t / 2], ev[t], ev[t + 1]));
    std::vector<float> sorted = ms;
    std::sort(sorted.begin(), sorted.end());
    const float med = sorted.empty() ? 0.f : sorted[sorted.size() / 2];
    for (size_t q = 0; q < ms.size(); q++) {
        if (ms[q] < 0.2f * med) continue;
        total_ms += ms[q];
        total_bytes += bytes[q];
        launches++;
    }
    used = 0;
}
void KernelTimer::reset() {
    used = 0;
    launches = 0;
    total_ms = total_bytes = 0.0;
}
KernelTimer::~KernelTimer() {
    for (auto e : ev) (void)hipEventDestroy(e);
}

// ---------------------------------------------------------------- System
// Levels whose steps run in pairs: large ones, and of those with a list of
// active chunks the ones the row-pair kernel takes (131 x 129 x 133 pool: two
// listed steps 15 us, the x-plane pair 24).
static bool pairs(const Level &L) { return pair_pays(L.d) && (!L.sparse || pair_segments_max(L.d) > 0); }

// Grids whose kernels are bound by launch latency rather than bytes.
static bool small_grid(Dims d) { return d.cells() <= ((size_t)1 << 19); }

// The stencil kernels skip wavefront rows whose cells are all inactive; the
// skipped cells of the level vectors then keep the zeros written here.
static void zero_vectors(Level &L, hipStream_t st) {
    const size_t n = L.d.cells();
    for (auto *v : {&L.x0, &L.x1, &L.dv, &L.b}) SFP_HIP(hipMemsetAsync(v->p, 0, n * sizeof(float), st));
}

void System::allocate(Dims d, hipStream_t st) {
    if (d_.nx == d.nx && d_.ny == d.ny && d_.nz == d.nz && !lv_.empty()) return;
    d_ = Dims{};  // (of a system whose every vector is there)
    lv_.clear();
    lv_.emplace_back();
    Level &L = lv_[0];
    L.d = d;
    const size_t n = d.cells();
    L.diag64.ensure(n);
    L.diag32.ensure(n);
    for (int a = 0; a < 3; a++) {
        L.cpl64[a].ensure(n);
        L.cpl32[a].ensure(n);
    }
    L.x0.ensure(n);
    L.x1.ensure(n);
    L.dv.ensure(n);
    L.b.ensure(n);
    zero_vectors(L, st);
    rhs_.ensure(n);
    x_.ensure(n);
    r_.ensure(n);
    q_.ensure(n);
    w_.ensure(n);
    for (auto *v : {&r_, &q_, &w_}) SFP_HIP(hipMemsetAsync(v->p, 0, n * sizeof(double), st));
    // The ring (48 B per cell) and the direction p, which a solve of more than
    // ring_ iterations needs, are allocated here, so that no solve runs out of
    // memory on the way. Where memory is short the ring takes fewer vectors, and
    // p and x are formed more often (the same bits): it and p leave three quarters
    // of what is free to the coarse levels, the other system and the caller.
    zring_stride_ = (n + 63) / 64 * 64;
    const auto ring_bytes = [&](int slots) { return slots * zring_stride_ * sizeof(float) + n * sizeof(double); };
    ring_ = kRing;
    if (ring_bytes(kRing) > (size_t)1 << 30) {  // (the query takes as long as a small solve)
        size_t free_bytes = 0, total_bytes = 0;
        SFP_HIP(hipMemGetInfo(&free_bytes, &total_bytes));
        for (int slots : {kBatch, 1})
            if (ring_bytes(ring_) > free_bytes / 4) ring_ = slots;
    }
    // (one allocation: each costs some 0.3 ms above 2 MiB)
    zring_.ensure(ring_ * zring_stride_ + 2 * n);
    p_ = (double *)(zring_.p + ring_ * zring_stride_);
    SFP_HIP(hipMemsetAsync(zring_.p, 0, ring_ * zring_stride_ * sizeof(float), st));
    SFP_HIP(hipMemsetAsync(x_.p, 0, n * sizeof(double), st));
    built_coarsest_ = -1;
    d_ = d;
}

void System::join_ainv(Workspace &ws) {
    if (!ainv_pending_) return;
    SFP_HIP(hipStreamWaitEvent(ws.stream, ws.side_out, 0));
    ainv_pending_ = false;
}

// The assembly is known to have formed no row, or to have raised an error: a
// look at pinned memory, whose answer may still be on its way.
bool System::nothing_to_solve(const Workspace &ws) const {
    return input_err_ && (__atomic_load_n(input_err_, __ATOMIC_ACQUIRE) != 0 ||
                          __atomic_load_n(ws.rows.host, __ATOMIC_ACQUIRE) == 2u * ws.rows.epoch);
}

// Waits for that answer (or the end of the stream's work, failed or not).
void System::await_rows(const Workspace &ws) const {
    for (unsigned look = 1; __atomic_load_n(ws.rows.host, __ATOMIC_ACQUIRE) >> 1 != ws.rows.epoch % 0x80000000u; look++)
        if (look % (1u << 22) == 0) {  // every few milliseconds
            const hipError_t e = hipStreamQuery(ws.stream);
            (void)hipGetLastError();
            if (e != hipErrorNotReady) return;
        }
}

bool System::build_hierarchy(Workspace &ws, const SolverConfig &cfg, bool known_rows) {
    // an inverse still being formed reads the coarsest operator rebuilt below
    join_ainv(ws);
    const int coarsest = std::max(2, std::min(cfg.coarsest, 4));
    if (built_coarsest_ != coarsest) {
        built_coarsest_ = -1;
        lv_.resize(1);
        while (true) {
            Dims dl = lv_.back().d;
            if (std::max({dl.nx, dl.ny, dl.nz}) <= coarsest) break;
            Level L;
            L.d = dl.coarse();
            const size_t n = L.d.cells();
            L.diag64.ensure(n);
            L.diag32.ensure(n);
            for (int a = 0; a < 3; a++) {
                L.cpl64[a].ensure(n);
                L.cpl32[a].ensure(n);
            }
            L.x0.ensure(n);
            L.x1.ensure(n);
            L.dv.ensure(n);
            L.b.ensure(n);
            zero_vectors(L, ws.stream);
            lv_.push_back(std::move(L));
        }
        if ((int)lv_.back().d.cells() > kMaxCoarse) throw ArgError("coarsest level too large");
        ainv_.ensure((size_t)lv_.back().d.cells() * lv_.back().d.cells());
        stages_.clear();
        built_coarsest_ = coarsest;
    }
    for (size_t l = 1; l < lv_.size(); l++) {
        Level &F = lv_[l - 1];
        Level &C = lv_[l];
        double *c64[3] = {C.cpl64[0].p, C.cpl64[1].p, C.cpl64[2].p};
        float *c32[3] = {C.cpl32[0].p, C.cpl32[1].p, C.cpl32[2].p};
        launch_coarsen(ws.stream, F.d, F.op64(), F.diag32.p, C.d, cfg.coarse_scale,
                       pinned_ ? 1.0 : cfg.coarse_scale, C.diag64.p, c64, C.diag32.p, c32,
                       l == 1 && !known_rows ? ws.rows : RowsFlag{});
    }
    // On the side stream, overlapping the clears below: which rows and chunks of
    // cells are active (one-block kernels but for the flags), then the dense
    // inverse of the coarsest level (one block bound by its pivot steps), which
    // overlaps the initial residual too; the first reader of the inverse joins it.
    const hipStream_t side = ws.side ? ws.side : ws.stream;
    if (ws.side) {
        SFP_HIP(hipEventRecord(ws.side_in, ws.stream));
        SFP_HIP(hipStreamWaitEvent(side, ws.side_in, 0));
    }
    // Large systems wait for the assembly here, hidden by the coarsening (0.1 ms
    // at 256^3), so that an empty one costs no more than these launches; on smaller
    // ones the host is the slower, and only looks, here and in the first batch. A
    // projection without liquid at 20^3, 64^3, 128^3 and 256^3: 60, 66, 90 and
    // 360 us (210, 240, 370 and 1015 with the whole set-up and a batch before the
    // host knew); with liquid as fast as without the look, where 20^3 and 64^3
    // took 50 us longer if they waited here.
    if (!known_rows) {
        if (lv_[0].d.cells() > (size_t)1 << 21) await_rows(ws);
        if (nothing_to_solve(ws)) return false;
    }
    bool lists = false;
    for (Level &L : lv_) {
        // a system of part of the grid: the flat kernels run on the chunks that
        // hold an active cell (small grids' launches cost the same either way)
        L.sparse = sparse_ && !(ws.fused_pairs & 32) && flat_step(L.d) && !small_grid(L.d);
        // and the row-tiled step pairs skip the loads of z rows without one
        // (on levels of rows up to 128 cells only where there are such pairs:
        // the launch took 35 us of 180 x 180 x 72's 1740)
        if (sparse_ && row_pair(L.d) && (L.d.nz > 128 || pairs(L))) {
            L.rowact.ensure((size_t)L.d.nx * L.d.ny);
            launch_row_activity(side, L.d, L.diag32.p, L.rowact.p);
            lists = true;
        } else {
            L.rowact.release();
        }
        if (L.sparse) {
            const size_t nch = (L.d.cells() + kChunk - 1) / kChunk, nq = restrict_quads(L.d);
            const size_t nbl = (L.d.cells() + kListCells - 1) / kListCells;
            L.chunk_flags.ensure(nch);
            L.chunk_list.ensure(nch + 1);
            L.quad_flags.ensure(nq);
            L.quad_list.ensure(nq + 1);
            L.block_flags.ensure(nbl);
            L.block_list.ensure(nbl + 1);
            launch_active_chunks(side, L.d, L.diag32.p,
                                 ActiveLists{L.chunk_flags.p, L.quad_flags.p, L.block_flags.p, L.chunk_list.p,
                                             L.quad_list.p, L.block_list.p});
            L.list_sums.ensure(list_sums(L.d));
            SFP_HIP(hipMemsetAsync(L.list_sums.p, 0, list_sums(L.d) * sizeof(double), side));
            if (const unsigned segs = pair_segments_max(L.d)) {
                L.segments.ensure(1 + 3 * (size_t)segs);
                launch_pair_segments(side, L.d, L.rowact.p, L.segments.p);
            }
            lists = true;
        }
    }
    if (ws.side && lists) SFP_HIP(hipEventRecord(ws.side_lists, side));
    launch_coarse_invert(side, lv_.back().d, lv_.back().op64(), ainv_.p);
    if (ws.side) {
        SFP_HIP(hipEventRecord(ws.side_out, side));
        ainv_pending_ = true;
    }
    // Every kernel skips groups of inactive cells (rows, tiles, pairs of
    // rows) and writes 0 at the inactive cells of the groups it processes
    // only if their inputs are 0 there; the groups differ between kernels.
    // A new operator may have a new active set, so the vectors are cleared at
    // the inactive cells (values left on cells that were active before would
    // otherwise leak into z, w, q and the inner products). Active cells are
    // written before they are read in every cycle; q is written at every cell
    // of the update's groups by the first iteration, and read in those groups
    // (the flat matvec's are the same) or, by the x-plane matvec, at active
    // cells only. The ring of z needs none: z counts as 0 at inactive cells
    // wherever it is read for its own cell, and elsewhere couples with weight 0.
    if (lv_.size() > (size_t)kClearMaxLevels) throw ArgError("too many multigrid levels");
    ClearArgs ca;
    ca.nlev = (int)lv_.size();
    size_t total = 0;
    for (size_t l = 0; l < lv_.size(); l++) {
        Level &L = lv_[l];
        total += L.d.cells();
        if (total >= ((size_t)1 << 32)) throw ArgError("grid too large for the level clear");
        ca.n[l] = (unsigned)L.d.cells();
        ca.start[l + 1] = (unsigned)total;
        ca.diag32[l] = L.diag32.p;
        float *const v[4] = {L.x0.p, L.x1.p, L.dv.p, L.b.p};
        for (int k = 0; k < 4; k++) ca.v[l][k] = v[k];
    }
    ca.w = w_.p;
    launch_clear_inactive(ws.stream, ca);
    if (ws.side && lists) SFP_HIP(hipStreamWaitEvent(ws.stream, ws.side_lists, 0));
    return true;
}

bool System::tail_at(const Workspace &ws, int l) const {
    const int nlev = (int)lv_.size() - l;
    if (!ws.vcycle_tail || nlev < 2 || nlev > kTailMaxLevels) return false;
    Dims dims[kTailMaxLevels];
    for (int q = 0; q < nlev; q++) dims[q] = lv_[l + q].d;
    return tail_fits(dims, nlev);
}

bool System::fold_at(const Workspace &ws, const Smoothing &sm, int l) {
    if (!fold_pays(lv_[l].d) || l + 1 >= (int)lv_.size()) return false;
    return tail_at(ws, l) || tile_stages(ws, l, sm.at(l).degree - 1, true).n > 0;
}

float *System::vcycle_tail(Workspace &ws, const Smoothing &sm, int l) {
    if (!tail_at(ws, l)) return nullptr;
    const int nlev = (int)lv_.size() - l;
    TailArgs t;
    t.nlev = nlev;
    for (int q = 0; q < nlev; q++) {
        Level &L = lv_[l + q];
        t.lv[q] = TailLevel{L.d, L.op32(), L.b.p, L.x0.p, L.x1.p, L.dv.p};
    }
    for (int set = 0; set < 2; set++) {
        const Cheby &cb = set == 0 ? sm.at(l) : sm.coarse;  // the first level's, the others'
        t.deg[set] = cb.degree;
        for (int q = 0; q < 8; q++) {
            t.cd[set][q] = cb.cd[q];
            t.cr[set][q] = cb.cr[q];
        }
    }
    t.lv[0].x1 = last_out(ws, l, t.lv[0].x1);
    t.ainv = ainv_.p;
    if (l == ws.z_level) t.fold = ws.fold;
    join_ainv(ws);
    launch_vcycle_tail(ws.stream, t, ws.gate);
    return tail_result(t);
}

// One separate launch of a step or the restriction on a level (us): 3.1 us
// up to 64^3 whatever it computes, 5.6 ns per thousand cells above (measured:
// 32^3 and 64^3 3.0-3.2, 80^3 3.7-4.4, 96^3 5.1-7.0, 128^3 12.0-12.4 us).
static double separate_cost(Dims d) { return std::max(3.1, 0.6 + 5.6e-6 * (double)d.cells()); }

const System::TileStages &System::tile_stages(const Workspace &ws, int l, int steps, bool restrict_after) {
    static const TileStages none;
    if (!ws.vcycle_tail) return none;
    if (stages_.size() != lv_.size()) stages_.assign(lv_.size(), {});
    for (const TileStages &t : stages_[l])
        if (t.steps == steps && t.restrict_after == restrict_after) return t;
    TileStages t;
    t.steps = steps;
    t.restrict_after = restrict_after;
    const Dims d = lv_[l].d;
    // (above 2^19 cells the tiles' repeated loads are bound by the caches, which
    // the model does not hold: 128^3, five steps 96 us against 60 us separately)
    if (!small_grid(d)) return none;
    double best = separate_cost(d) * (steps + (restrict_after ? 1 : 0));
    double c = 0.0;
    const TilePlan one = choose_tile(d, steps, restrict_after, &c);
    if (c < best) {
        best = c;
        t.n = 1;
        t.count[0] = steps;
        t.plan[0] = one;
    }
    for (int a = 1; a < steps; a++) {
        double c0 = 0.0, c1 = 0.0;
        const TilePlan p0 = choose_tile(d, a, false, &c0), p1 = choose_tile(d, steps - a, restrict_after, &c1);
        if (c0 + c1 < best) {
            best = c0 + c1;
            t.n = 2;
            t.count[0] = a;
            t.count[1] = steps - a;
            t.plan[0] = p0;
            t.plan[1] = p1;
        }
    }
    stages_[l].push_back(t);
    return stages_[l].back();
}


// Algorithmic bytes per cell of one single Chebyshev step: x, b, diag and 3
// couplings in and x out, plus the direction in and out by mode and the
// coarse correction (an eighth of a value per cell). rowsum: the flat
// kernels rebuild the diagonal instead of reading it.
static double step_bytes(int mode, bool rowsum) {
    double b = 4.0 * (rowsum ? 6 : 7);
    if (mode & SM_READ_D) b += 4.0;
    if (mode & SM_WRITE_D) b += 4.0;
    if (mode & SM_PROLONG) b += 0.5;
    return b;
}

// x0_ready: the level's x0 holds c0 D^-1 b, stored by the restriction that
// formed its b (coarse levels) or by the FCG kernels (ws.x0_level).
float *System::vlevel(Workspace &ws, const Smoothing &sm, int l, const double *r64, bool x0_ready) {
    if (!r64) {
        if (float *z = vcycle_tail(ws, sm, l)) return z;
    }
    const Cheby &cb = sm.at(l);
    Level &L = lv_[l];
    const hipStream_t st = ws.stream;
    const bool fine = (l == 0);
    const double cells = (double)L.d.cells();
    if (l + 1 == (int)lv_.size()) {
        if (r64) launch_smooth_first(st, L.d, L.op32(), r64, L.b.p, L.x1.p, 0.f, ws.gate);
        join_ainv(ws);
        float *out = last_out(ws, l, L.x0.p);
        launch_coarse_solve(st, (int)L.d.cells(), ainv_.p, L.b.p, out, ws.gate);
        return out;
    }
    const Op32 A = L.op32();
    // the flat kernels (nz a multiple of 4) and the pair kernels rebuild a
    // row-sum diagonal instead of reading it
    const bool diag_rebuilt = L.pinned_rowsum && flat_step(L.d);
    const double diag_bytes = diag_rebuilt ? 0.0 : 4.0, pair_diag_bytes = L.pinned_rowsum ? 0.0 : 4.0;
    float *cur = L.x0.p, *oth = L.x1.p;
    const int deg = cb.degree;
    auto smooth = [&](int mode, float cd, float cr, const double *r, const float *e) {
        // timed: the fine-level single steps but the fused first step
        const bool track = fine && ws.profiling && !(mode & SM_FIRST);
        if (track) ws.timers[K_SMOOTH].begin(st, step_bytes(mode, diag_rebuilt) * cells);
        launch_smooth(st, mode, L.d, A, r, L.b.p, cur, oth, L.dv.p, cb.cr[0], cd, cr, e, ws.gate);
        if (track) ws.timers[K_SMOOTH].end(st);
        std::swap(cur, oth);
    };
    // the whole descent of a small level in one or two launches
    if (const TileStages &T = tile_stages(ws, l, deg - 1, true); T.n > 0) {
        if (r64) launch_smooth_first(st, L.d, A, r64, L.b.p, cur, cb.cr[0], ws.gate);  // (b)
        Level &C = lv_[l + 1];
        int s = 1;
        for (int q = 0; q < T.n; q++) {
            TileArgs t;
            t.d = L.d;
            t.dc = C.d;
            t.A = A;
            t.plan = T.plan[q];
            t.b = L.b.p;
            t.start = q == 0 ? TILE_FIRST : TILE_CONTINUE;
            t.c0 = cb.cr[0];
            t.nsteps = T.count[q];
            for (int e = 0; e < t.nsteps; e++) {
                t.cd[e] = cb.cd[s + e];
                t.cr[e] = cb.cr[s + e];
            }
            s += t.nsteps;
            if (q > 0) {
                t.xin = cur;
                t.din = L.dv.p;
            }
            t.xout = oth;
            if (q == 0 && l == ws.z_level) t.fold = ws.fold;
            if (q + 1 < T.n) t.dout = L.dv.p;
            else t.bc = C.b.p;
            launch_tile_steps(st, t, ws.gate);
            std::swap(cur, oth);
        }
        const float *e = vlevel(ws, sm, l + 1, nullptr, false);
        return post_smooth(ws, sm, l, cur, e);
    }
    // the last step and the restriction run as one pass where the grid pays
    // for the pass's tile overlap
    const bool fuse_restrict =
        deg >= 3 && (((ws.fused_pairs & 1) && pairs(L)) || ((ws.fused_pairs & 4) && small_grid(L.d)));
    if (deg == 1) {
        launch_smooth_first(st, L.d, A, r64, L.b.p, cur, cb.cr[0], ws.gate);
    } else {
        // steps 0 and 1 in one pass (step 0 read from x0 when the FCG update
        // stored it); then steps 2 .. deg-1
        const int first = (!r64 && (x0_ready || ws.x0_level == l)) ? SM_XFIRST : SM_FIRST;
        // at degree 3 the two passes from the stored first iterate can run as
        // one: the iterate is also step 1's previous direction
        const bool pre_pair = deg == 3 && !fuse_restrict && first == SM_XFIRST &&
                              (ws.fused_pairs & 16) && pairs(L);
        if (pre_pair) {
            // reads x0, b, diag, 3 couplings; writes x
            if (fine && ws.profiling) ws.timers[K_SMOOTH_PAIR].begin(st, (24.0 + pair_diag_bytes) * cells);
            launch_smooth_pair(st, L.d, A, L.b.p, cur, oth, cur, cb.cd[1], cb.cr[1], cb.cd[2], cb.cr[2],
                               ws.gate, L.rowact.p, L.sparse ? L.segments.p : nullptr);
            if (fine && ws.profiling) ws.timers[K_SMOOTH_PAIR].end(st);
            std::swap(cur, oth);
        } else {
            smooth(first | (deg > 2 ? SM_WRITE_D : 0), cb.cd[1], cb.cr[1], r64, nullptr);
            // from degree 4 the last two steps can (the first of them reads the
            // direction the step before stored)
            const bool last_pair = deg >= 4 && !fuse_restrict && (ws.fused_pairs & 16) && pairs(L);
            for (int s = 2; s < deg - (fuse_restrict ? 1 : last_pair ? 2 : 0); s++)
                smooth(SM_READ_D | (s < deg - 1 ? SM_WRITE_D : 0), cb.cd[s], cb.cr[s], nullptr, nullptr);
            if (last_pair) {
                // reads x, b, d, diag, 3 couplings; writes x
                if (fine && ws.profiling) ws.timers[K_SMOOTH_PAIR].begin(st, (28.0 + pair_diag_bytes) * cells);
                launch_smooth_pair(st, L.d, A, L.b.p, cur, oth, L.dv.p, cb.cd[deg - 2], cb.cr[deg - 2],
                                   cb.cd[deg - 1], cb.cr[deg - 1], ws.gate, L.rowact.p,
                                   L.sparse ? L.segments.p : nullptr);
                if (fine && ws.profiling) ws.timers[K_SMOOTH_PAIR].end(st);
                std::swap(cur, oth);
            }
        }
    }
    bool store_x0 = false;  // the restriction stores the coarse level's first iterate
    if (fuse_restrict) {
        // reads x, b, d, diag, 3 couplings; writes x and the coarse b
        if (fine && ws.profiling) ws.timers[K_SMOOTH_RESTRICT].begin(st, (28.0 + pair_diag_bytes + 0.5) * cells);
        launch_smooth_restrict(st, L.d, A, L.b.p, cur, oth, L.dv.p, cb.cd[deg - 1], cb.cr[deg - 1],
                               lv_[l + 1].b.p, ws.gate);
        if (fine && ws.profiling) ws.timers[K_SMOOTH_RESTRICT].end(st);
        std::swap(cur, oth);
    } else {
        // the coarse level's first iterate too, where its cycle's first step reads it
        Level &C = lv_[l + 1];
        store_x0 = l + 2 < (int)lv_.size() && sm.at(l + 1).degree >= 2;
        // reads x, b, diag, 3 couplings; writes the coarse b (and reads the
        // coarse diagonal, writes the coarse x0): per fine cell
        if (fine && ws.profiling) ws.timers[K_RESTRICT].begin(st, (20.0 + diag_bytes + 0.5 + (store_x0 ? 1.0 : 0.0)) * cells);
        launch_restrict(st, L.d, A, L.b.p, cur, C.b.p, ws.gate, store_x0 ? C.x0.p : nullptr,
                        C.diag32.p, sm.at(l + 1).cr[0]);
        if (fine && ws.profiling) ws.timers[K_RESTRICT].end(st);
    }
    const float *e = vlevel(ws, sm, l + 1, nullptr, store_x0);
    return post_smooth(ws, sm, l, cur, e);
}

float *System::post_smooth(Workspace &ws, const Smoothing &sm, int l, float *cur, const float *e) {
    const Cheby &cb = sm.at(l);
    Level &L = lv_[l];
    const hipStream_t st = ws.stream;
    const Op32 A = L.op32();
    float *oth = cur == L.x0.p ? L.x1.p : L.x0.p;
    const int deg = cb.degree;
    const bool track = l == 0 && ws.profiling;
    if (const TileStages &T = tile_stages(ws, l, deg, false); T.n > 0) {
        int s = 0;
        for (int q = 0; q < T.n; q++) {
            TileArgs t;
            t.d = L.d;
            t.dc = lv_[l + 1].d;
            t.A = A;
            t.plan = T.plan[q];
            t.b = L.b.p;
            t.start = q == 0 ? TILE_PROLONG : TILE_CONTINUE;
            t.nsteps = T.count[q];
            for (int v = 0; v < t.nsteps; v++) {
                t.cd[v] = s + v == 0 ? 0.f : cb.cd[s + v];
                t.cr[v] = cb.cr[s + v];
            }
            s += t.nsteps;
            t.xin = cur;
            t.e = e;
            if (q > 0) t.din = L.dv.p;
            if (q + 1 < T.n) t.dout = L.dv.p;
            else oth = last_out(ws, l, oth);
            t.xout = oth;
            launch_tile_steps(st, t, ws.gate);
            std::swap(cur, oth);
        }
        return cur;
    }
    // the last two steps run as one pass where the grid is large enough to
    // pay for the pass's tile overlap (the direction they leave is not stored:
    // nothing reads it before the next cycle rewrites it)
    const int fused = (deg >= 3 && (((ws.fused_pairs & 2) && pairs(L)) ||
                                    ((ws.fused_pairs & 8) && small_grid(L.d)))) ? 2 : 0;
    // step 0 adds the coarse correction: in the flat step's gathers, else on
    // large grids by its own pointwise pass before a plain step (cheaper than
    // the x-plane tiles' gathers at every neighbour); equal values every way
    const bool add_first = !whole_groups(L.d) && !small_grid(L.d);
    if (add_first) launch_prolong_add(st, L.d, L.diag32.p, A.chunks.list, e, cur, ws.gate);
    for (int s = 0; s < deg - fused; s++) {
        // step 0 adds the prolonged correction; the fine-level steps are timed
        const int mode = (s == 0 ? (add_first ? 0 : SM_PROLONG) : SM_READ_D) | (s < deg - 1 ? SM_WRITE_D : 0);
        const bool t = track;
        if (s == deg - 1) oth = last_out(ws, l, oth);
        if (t) ws.timers[K_SMOOTH].begin(st, step_bytes(mode, L.pinned_rowsum && flat_step(L.d)) * (double)L.d.cells());
        launch_smooth(st, mode, L.d, A, nullptr, L.b.p, cur, oth, L.dv.p, cb.cr[0], s == 0 ? 0.f : cb.cd[s],
                      s == 0 ? cb.cr[0] : cb.cr[s], s == 0 ? e : nullptr, ws.gate);
        if (t) ws.timers[K_SMOOTH].end(st);
        std::swap(cur, oth);
    }
    if (fused) {
        // reads x, b, d, diag (unless rebuilt), 3 couplings and writes x
        oth = last_out(ws, l, oth);
        if (track) ws.timers[K_SMOOTH_PAIR].begin(st, (L.pinned_rowsum ? 28.0 : 32.0) * (double)L.d.cells());
        launch_smooth_pair(st, L.d, A, L.b.p, cur, oth, L.dv.p, cb.cd[deg - 2], cb.cr[deg - 2],
                           cb.cd[deg - 1], cb.cr[deg - 1], ws.gate, L.rowact.p, L.sparse ? L.segments.p : nullptr);
        if (track) ws.timers[K_SMOOTH_PAIR].end(st);
        std::swap(cur, oth);
    }
    return cur;
}

float *System::precondition(Workspace &ws, const SolverConfig &cfg, const double *r64) {
    if (cfg.precond == 2) {  // SFP_PRECOND_JACOBI
        float *z = last_out(ws, 0, lv_[0].x0.p);
        launch_jacobi(ws.stream, d_, lv_[0].op32(), r64, z, ws.gate);
        return z;
    }
    if (cfg.precond == 3 && lv_.size() > 1) return learned_cycle(ws, cfg, r64, kCycleSmooth);
    return vlevel(ws, Smoothing::make(cfg), 0, r64);
}

float *System::learned_cycle(Workspace &ws, const SolverConfig &cfg, const double *r64, Cycle c) {
    // the smoother the network was trained under
    const Smoothing sm = Smoothing::make_learned(cfg);
    Level &L = lv_[0], &C = lv_[1];
    const hipStream_t st = ws.stream;
    // (the V-cycle's result stays in the level; the last smoothing's goes to zout)
    float *const zout = ws.zout;
    ws.zout = nullptr;
    float *z = vlevel(ws, sm, 0, r64);
    ws.zout = zout;
    // residual the V-cycle leaves, restricted to the first coarse level
    launch_restrict(st, L.d, L.op32(), L.b.p, z, C.b.p, ws.gate);
    if (c == kCycleRestrictOnly) return C.b.p;
    if (c == kCycleLearned) {
        network_correction(ws, C.x0.p);
    } else {  // the same cycle without the network: a zero correction
        SFP_HIP(hipMemsetAsync(C.x0.p, 0, C.d.cells() * sizeof(float), st));
    }
    return post_smooth(ws, sm, 0, z, C.x0.p);
}

bool System::learned_ok(const Workspace &ws) const {
    if (!ws.net || lv_.size() < 2) return false;
    const Dims c = lv_[1].d;
    return c.nx % 4 == 0 && c.ny % 4 == 0 && c.nz % 4 == 0;
}

void System::coarse_phi(Workspace &ws) {
    if (!ws.phi) return;
    phic_.ensure(lv_[1].d.cells());
    launch_restrict_phi(ws.stream, d_, ws.phi, lv_[1].d, phic_.p);
}

void System::prepare_learned(Workspace &ws) {
    const Level &C = lv_[1];
    ws.net->ensure(UNetShape{1, C.d.nx, C.d.ny, C.d.nz}, false);
    coarse_phi(ws);
    launch_learned_features(ws.stream, C.d, C.op64(), C.diag32.p, ws.phi ? phic_.p : nullptr,
                            2.0 * ws.spacing, ws.net->input_buffer(), nullptr);
}

void System::learned_features(Workspace &ws, float *f3) {
    if (lv_.size() < 2) throw StateError("the hierarchy has a single level");
    const Level &C = lv_[1];
    coarse_phi(ws);
    launch_learned_features(ws.stream, C.d, C.op64(), C.diag32.p, ws.phi ? phic_.p : nullptr,
                            2.0 * ws.spacing, nullptr, f3);
}

void System::network_correction(Workspace &ws, float *x) {
    Level &C = lv_[1];
    const hipStream_t st = ws.stream;
    UNet &net = *ws.net;
    launch_pack_residual32(st, C.d, C.b.p, C.diag32.p, ws.partials.p, ws.scalars.p, net.input_buffer(),
                           ws.gate);
    net.forward(st, net.input_buffer(), net.output_buffer(), ws.gate);
    launch_scaled_correction(st, C.d, C.op32(), net.output_buffer(), C.b.p, ws.partials.p,
                             ws.scalars.p, x, ws.gate);
}

float *System::precondition_learned(Workspace &ws, const SolverConfig &cfg, const double *r64) {
    return learned_cycle(ws, cfg, r64, kCycleLearned);
}

const float *System::restrict_smoothed(Workspace &ws, const SolverConfig &cfg, const double *r64) {
    if (lv_.size() < 2) throw StateError("the hierarchy has a single level");
    return learned_cycle(ws, cfg, r64, kCycleRestrictOnly);
}

// A z of infinities or NaN (from input that holds them) must not outlive its
// solve: on cells that are active there and inactive in a later system, which
// skips writing them, their neighbours couple with weight 0, and 0 times them
// is NaN.
void System::clear_ring(Workspace &ws) {
    SFP_HIP(hipMemsetAsync(zring_.p, 0, ring_ * zring_stride_ * sizeof(float), ws.stream));
}

SolveInfo System::fcg(Workspace &ws, const SolverConfig &cfg, int level, bool warm, const Finish &finish) {
    SolveInfo info;
    info.precond_used = cfg.precond;
    const hipStream_t st = ws.stream;
    const Dims d = lv_[level].d;
    const size_t n = d.cells();
    const Op64 A = lv_[level].op64();
    const bool fine = level == 0;
    const bool profiling = fine && ws.profiling;
    // a cold solve's x is 0 until the first flush, which then does not read it
    bool zero_x = !warm;
    // The V-cycle preconditioners start from the residual rounded to FP32 in
    // the level's b, with the cycle's first Chebyshev iterate in the level's
    // x0: the residual kernels and the FCG update store both, so no cycle
    // reads the FP64 residual (the Jacobi preconditioner reads r).
    float *b32 = cfg.precond != 2 ? lv_[level].b.p : nullptr;
    float *x0 = b32 ? lv_[level].x0.p : nullptr;
    // learned preconditioner until an iteration reduces the residual by less
    // than stall_ratio; then the plain V-cycle with the plain smoother
    bool learned = fine && cfg.precond == 1 && learned_ok(ws);
    // the first Chebyshev iterate the residual and update kernels store is
    // that of the cycle which reads it next
    const Smoothing plain = Smoothing::make(cfg), net_sm = Smoothing::make_learned(cfg);
    auto first_coef = [&](bool l) {
        return ((l || (fine && cfg.precond == 3)) ? net_sm : plain).at(level).cr[0];
    };
    float c0 = first_coef(learned);
    launch_residual64(st, d, A, rhs_.p, warm ? x_.p : nullptr, r_.p, ws.partials.p,
                      ws.scalars.p, ws.host_sc, b32, x0, lv_[level].diag32.p, c0);
    // The host reads the first residual (||b||, the system's size and its input
    // errors) with the first batch's, which the device gates where no
    // iteration is needed.
    bool known = false;
    double bb = 0.0, rel = 0.0;
    bool first = true;
    bool checked = false;  // rel is a true residual
    const double cells = (double)n;
    if (learned) prepare_learned(ws);
    bool b_ready = b32 != nullptr;  // lv_[level].b holds r rounded (and lv_[level].x0 its first iterate)
    // iterations to enqueue before the host reads the residual; the first
    // learned iteration runs alone: it decides whether the network pays,
    // and iterations enqueued behind a stall would still launch every
    // kernel of the learned cycle (each returning at once)
    const int ring = std::min(ring_, ws.ring_limit), full_batch = std::min(kBatch, ring);
    int next_batch = learned ? 1 : full_batch;
    bool predicted = false;  // next_batch is expected to reach the tolerance
    // iterations whose z is in the ring and whose alpha p is not yet in x, and
    // the number of the next iteration (its scalars' place)
    int pending = 0, iter = 0;
    bool has_p = false;  // p_ holds the direction before the pending iterations
    const float *flags = A.pinned_rowsum ? nullptr : lv_[level].diag32.p;
    auto bring_x_up_to_date = [&](bool keep_p) {
        if (pending > 0) {
            launch_fcg_flush(st, d, flags, zring_.p, zring_stride_, pending, iter - pending, p_,
                             has_p, keep_p, x_.p, zero_x, ws.scalars.p);
            zero_x = false;
            has_p = keep_p;
        }
        pending = 0;
    };
    // the recurrence restarts from the true residual
    auto restart = [&] {
        launch_residual64(st, d, A, rhs_.p, x_.p, r_.p, ws.partials.p, ws.scalars.p, nullptr, b32, x0,
                          lv_[level].diag32.p, c0);
        first = true;
        b_ready = b32 != nullptr;
    };
    // small grids: the reductions' partials are added by the launches that
    // need the sums (the update, and the next cycle's first) instead of
    // finalize launches between
    const bool fold = !profiling && cfg.precond == 0 && fold_at(ws, plain, level);
    ws.z_level = level;
    info.precond_used = learned ? 1 : (cfg.precond == 1 ? 0 : cfg.precond);
    while (true) {
        if (known && rel <= cfg.tol) {
            if (checked) break;
            // recursive residual reached tol: recompute its norm from x in
            // FP64 (the sums only), and restart from the true residual if the
            // two have drifted apart
            bring_x_up_to_date(false);
            launch_residual64(st, d, A, rhs_.p, x_.p, nullptr, ws.partials.p, ws.scalars.p, ws.host_sc);
            ws.wait();
            rel = std::sqrt(ws.host_sc->rr / bb);
            checked = true;
            if (rel > cfg.tol) restart();
            continue;
        }
        if (known && info.iterations >= cfg.max_iters) break;
        // Iterations are enqueued in batches (the first kBatch, then as many
        // as the residual's rate of decrease predicts are left) before the host
        // looks at the residual: the update's finalize raises `stop` on the
        // device once ||r|| <= tol ||b||, or (learned preconditioner) once an
        // iteration reduced ||r|| by less than stall_ratio, and every kernel
        // of the remaining iterations of the batch then returns at once
        // (profiled launches among them are dropped from the timings).
        if (pending + next_batch > ring) bring_x_up_to_date(true);
        const int batch = std::min(next_batch, cfg.max_iters - info.iterations);
        // Behind a batch expected to be the last, the check above and what
        // follows the solve are enqueued too, behind the stop flag and the
        // check's own result: one wait instead of three (each leaves the GPU
        // idle for some 20 us).
        const bool check_here = predicted && finish && !learned && !profiling && batch == next_batch;
        if (batch > 0) {
            launch_batch_begin(st, ws.scalars.p, cfg.tol * cfg.tol,
                               learned ? cfg.stall_ratio * cfg.stall_ratio : 0.0, !known);
            ws.gate = &ws.scalars.p->stop;
        }
        for (int it = 0; it < batch; it++) {
            if (!known && nothing_to_solve(ws)) break;  // (found below)
            const double *r64 = b_ready ? nullptr : r_.p;  // null: the cycle reads b
            ws.x0_level = b_ready ? level : -1;
            ws.zout = zring_.p + (size_t)(pending + it) * zring_stride_;
            // (within a batch, the update before this cycle left its norm's
            // partials)
            ws.fold = fold && it > 0 ? update_fold(d, ws.partials.p, ws.scalars.p) : FoldArgs{};
            const float *z;
            if (learned)
                z = precondition_learned(ws, cfg, r64);
            else if (fine)
                z = precondition(ws, cfg, r64);
            else
                z = vlevel(ws, Smoothing::make(cfg), level, r64);
            // z, the couplings, r, q_prev (after the first iteration) in; w
            // out; and the diagonal and the FP32 one (skips inactive cells)
            // unless the operator has the row-sum structure, where every cell
            // but cell 0 is active and the diagonal is rebuilt
            // (the timings cover the stencil kernels, not the finalize after them)
            hipEvent_t done = nullptr;
            if (profiling) {
                ws.timers[K_MATVEC64].begin(st, (4.0 + (A.pinned_rowsum ? 24.0 : 4.0 + 32.0) + 8.0 +
                                                 (first ? 0.0 : 8.0) + 8.0) * cells);
                done = ws.timers[K_MATVEC64].pending_end();
            }
            ws.zout = nullptr;
            ws.fold = FoldArgs{};
            launch_fcg_matvec(st, d, A, flags, z, r_.p, q_.p, w_.p, first ? 1 : 0, iter + it, fold,
                              ws.partials.p, ws.scalars.p, ws.gate, done);
            if (profiling) ws.timers[K_MATVEC64].end_recorded();
            // w, q, r in; q, r out (and diag in, b and x0 out)
            if (profiling) {
                ws.timers[K_UPDATE64].begin(st, (8.0 * 3 + 8.0 * 2 + (x0 ? 4.0 + 4.0 + 4.0 : 0.0)) * cells);
                done = ws.timers[K_UPDATE64].pending_end();
            }
            ws.x0_level = -1;
            // (a cycle whose first launch folds forms its first iterate itself)
            float *const x0_next = fold ? nullptr : x0;
            launch_fcg_update(st, d, x0_next ? lv_[level].diag32.p : flags, A.chunks, w_.p, q_.p, r_.p, b32, x0_next, c0,
                              first ? 1 : 0, iter + it, fold, ws.partials.p, ws.scalars.p, ws.gate, done,
                              it + 1 == batch ? ws.host_sc : nullptr);
            if (profiling) ws.timers[K_UPDATE64].end_recorded();
            first = false;
            b_ready = b32 != nullptr;
        }
        if (fold && batch > 0) launch_fcg_norm(st, d, ws.partials.p, ws.scalars.p, ws.gate, ws.host_sc);
        ws.gate = nullptr;
        if (check_here) {
            const double *stop = &ws.scalars.p->stop;
            launch_fcg_flush(st, d, flags, zring_.p, zring_stride_, pending, iter - pending, p_, has_p, false,
                             x_.p, zero_x, ws.scalars.p, stop);
            launch_residual64(st, d, A, rhs_.p, x_.p, nullptr, ws.partials.p, ws.scalars.p, ws.host_sc, nullptr,
                              nullptr, nullptr, 0.f, stop, cfg.tol);
            finish(&ws.scalars.p->ok);
        }
        ws.wait();
        const KrylovScalars &h = *ws.host_sc;
        if (!known) {
            known = true;
            info.active = (long long)h.active;
            // (launches that returned at once are no measurement)
            const bool bad_input = input_err_ && *input_err_;
            if (profiling && (h.iters == 0.0 || bad_input))
                for (auto &t : ws.timers) t.used = 0;
            if (bad_input) {
                info.input_error = true;
                clear_ring(ws);
                return info;
            }
            bb = h.bb;
            if (bb == 0.0) {  // zero right-hand side: x = 0
                SFP_HIP(hipMemsetAsync(x_.p, 0, n * sizeof(double), st));
                info.converged = true;
                info.rel = 0.0;
                info.precond_used = cfg.precond;
                return info;
            }
            rel = std::sqrt(h.check_rr / bb);
            checked = true;
            if (batch == 0) continue;
        }
        const bool stalled = h.stalled != 0.0;
        const int done = (int)h.iters;
        pending += done;
        iter += done;
        info.iterations += done;
        if (!learned && cfg.precond == 1 && info.precond_used == 1) info.fallback += done;
        const double prev = rel;
        if (done > 0) {
            rel = std::sqrt(h.rr / bb);
            checked = false;
        }
        if (check_here && h.stop != 0.0) {  // the flush and the check have run
            zero_x = has_p = false;
            pending = 0;
            rel = std::sqrt(h.check_rr / bb);
            checked = true;
            info.finished = h.ok != 0.0;
            if (info.finished) break;
            restart();
            continue;
        }
        // The next batch: as many iterations as the last ones' mean residual
        // reduction predicts are left. Enqueued past convergence an iteration
        // still launches every kernel, which returns at once: some 10 launches
        // or 25 us where the levels run in tiles, 45 launches or 110 us on
        // larger grids (a magnetic 256^3 solve predicts 7 where 4 are left),
        // so there a batch is kBatch at most and the host waits again. A wait
        // costs some 20 us, as do the check and the Finish behind a batch that
        // then needs another.
        next_batch = full_batch;
        predicted = false;
        if (done > 0 && rel > 0.0 && rel < prev) {
            const double rate = std::pow(rel / prev, 1.0 / done);
            const double left = std::log(cfg.tol / rel) / std::log(rate);
            const int cap = small_grid(d) ? ring : full_batch;
            if (left <= cap) next_batch = std::max(1, (int)std::ceil(left));
            predicted = left <= 1.5 * next_batch;
        }
        if (learned && (stalled || (batch == 1 && done == 1 && rel > cfg.stall_ratio * prev))) {
            // fall back to the plain V-cycle, restarting the recurrence from
            // the current iterate (a direction built with the other
            // preconditioner slows the V-cycle's iterations down); the first
            // iterate stored by the last update belongs to the learned
            // cycle's smoother
            learned = false;
            bring_x_up_to_date(false);
            first = true;
            const float c0_plain = first_coef(false);
            if (c0_plain != c0) b_ready = false;
            c0 = c0_plain;
            next_batch = full_batch;
            predicted = false;
        }
    }
    bring_x_up_to_date(false);
    if (zero_x) SFP_HIP(hipMemsetAsync(x_.p, 0, n * sizeof(double), st));  // (no iteration)
    if (!checked) {
        launch_residual64(st, d, A, rhs_.p, x_.p, nullptr, ws.partials.p, ws.scalars.p, ws.host_sc);
        ws.wait();
        rel = std::sqrt(ws.host_sc->rr / bb);
    }
    info.rel = rel;
    info.converged = rel <= cfg.tol;
    if (!std::isfinite(rel)) clear_ring(ws);
    if (info.fallback > 0) info.precond_used = 0;
    if (profiling)
        for (auto &t : ws.timers) t.harvest();
    return info;
}

}  // namespace sfp
