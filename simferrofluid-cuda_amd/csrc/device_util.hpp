// Device helpers shared by the gfx950 kernels: 64-lane wavefront reductions,
// a deterministic grid-wide reduction (last block finishes), and the 7-point
// operator applies in FP32 and FP64.
#pragma once
#include "sfp_internal.hpp"

namespace sfp {

constexpr int kBlock = 256;          // every kernel runs 256 threads = 4 wavefronts
constexpr int kWaves = kBlock / 64;

__device__ __forceinline__ int flat_tid() {
    return threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
}
__device__ __forceinline__ unsigned flat_bid() {
    return blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
}
__device__ __forceinline__ unsigned num_blocks() { return gridDim.x * gridDim.y * gridDim.z; }

// 1 / dg on active cells (dg > 0), 0 on inactive ones. Every kernel that
// scales by the inverse diagonal uses this one approximation.
__device__ __forceinline__ float rcp_or_zero(float dg) {
    return dg > 0.f ? __builtin_amdgcn_rcpf(dg) : 0.f;
}

// A load whose value is used on one side of a branch only is moved down to
// that side, and then its latency is not shared with the loads before the
// branch. `pin` counts as a use where it stands: a kernel that wants all of its
// loads in flight together pins them before its first branch on one of them.
template <class T>
__device__ __forceinline__ void pin(const T &v) {
    asm volatile("" ::"v"(v));
}
// The gate of a batch of iterations (KrylovScalars::stop; null: open), without
// a branch around the load: `other` is any readable address.
__device__ __forceinline__ double load_gate(const double *gate, const void *other) {
    const double v = *(gate ? gate : (const double *)other);
    return gate ? v : 0.0;
}

// The wavefront's number in the grid of a kernel over the flat cell index
// (uniform), and a grid's number of them.
__device__ __forceinline__ unsigned flat_wave() {
    return blockIdx.x * (kBlock / 64) + (unsigned)__builtin_amdgcn_readfirstlane((int)(flat_tid() >> 6));
}
__device__ __forceinline__ unsigned flat_waves() { return gridDim.x * (kBlock / 64); }
// The first of this lane's N consecutive cells, 64 N of a listed chunk to a
// unit of work: unit `u` of list[0] * list_units<N>().
template <int N>
constexpr unsigned list_units() {
    return kChunk / (64 * N);
}
template <int N>
__device__ __forceinline__ unsigned list_cell(const unsigned *list, unsigned u) {
    constexpr unsigned per = list_units<N>();
    return list[1 + u / per] * kChunk + (u % per) * 64 * N + N * (flat_tid() & 63);
}

// Sum over the wavefront, the same in every lane: halves 32 lanes apart, then
// 16, 8, 4, 2 and 1, the tree of shuffles down in lane 0 (so the same bits
// there). The exchanges are register moves (v_permlane32_swap,
// v_permlane16_swap, DPP rotations of 16-lane rows and quads): a shuffle
// through the LDS unit waits about 130 cycles, six of them for each sum.
__device__ __forceinline__ double wave_sum(double v) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    auto halves = [](double a) { return __builtin_bit_cast(u2, a); };
    auto whole = [](unsigned lo, unsigned hi) { return __builtin_bit_cast(double, u2{lo, hi}); };
    {
        const u2 h = halves(v);
        const auto l = __builtin_amdgcn_permlane32_swap(h.x, h.x, false, false);
        const auto u = __builtin_amdgcn_permlane32_swap(h.y, h.y, false, false);
        v = whole(l[0], u[0]) + whole(l[1], u[1]);
    }
    {
        const u2 h = halves(v);
        const auto l = __builtin_amdgcn_permlane16_swap(h.x, h.x, false, false);
        const auto u = __builtin_amdgcn_permlane16_swap(h.y, h.y, false, false);
        v = whole(l[0], u[0]) + whole(l[1], u[1]);
    }
#define SFP_DPP_ADD(CTRL)                                                                             \
    {                                                                                                 \
        const u2 h = halves(v);                                                                       \
        v += whole((unsigned)__builtin_amdgcn_mov_dpp((int)h.x, CTRL, 0xf, 0xf, true),                \
                   (unsigned)__builtin_amdgcn_mov_dpp((int)h.y, CTRL, 0xf, 0xf, true));               \
    }
    SFP_DPP_ADD(0x128)  // row_ror:8
    SFP_DPP_ADD(0x124)  // row_ror:4 (the lanes 8 apart agree)
    SFP_DPP_ADD(0x4e)   // quad_perm 2,3,0,1
    SFP_DPP_ADD(0xb1)   // quad_perm 1,0,3,2
#undef SFP_DPP_ADD
    return v;
}

// Sums v[q] over a block of T threads; the totals are valid in thread 0.
template <int N, int T = kBlock>
__device__ __forceinline__ void block_sum(double (&v)[N]) {
    constexpr int W = T / 64;
    __shared__ double sh[N][W];
    const int tid = flat_tid();
#pragma unroll
    for (int q = 0; q < N; q++) v[q] = wave_sum(v[q]);
    if ((tid & 63) == 0) {
#pragma unroll
        for (int q = 0; q < N; q++) sh[q][tid >> 6] = v[q];
    }
    __syncthreads();
    if (tid == 0) {
#pragma unroll
        for (int q = 0; q < N; q++) {
            double s = sh[q][0];
#pragma unroll
            for (int w = 1; w < W; w++) s += sh[q][w];
            v[q] = s;
        }
    }
    __syncthreads();
}

// Block-level partial sums: block b stores its totals at partials[q*nb + b]
// (nb = gridDim.x). A one-block finalize kernel adds them in block order, so
// every reduction is deterministic for a given grid. (A last-block-done
// scheme needs a device-scope fence per block, which on a multi-XCD chip
// writes back L2 and serializes the blocks.)
template <int N>
__device__ __forceinline__ void block_partials(double (&v)[N], double *partials) {
    block_sum<N>(v);
    if (flat_tid() == 0) {
#pragma unroll
        for (int q = 0; q < N; q++) partials[(size_t)q * gridDim.x + blockIdx.x] = v[q];
    }
}

// A raw buffer over `bytes` bytes from p: a load at an offset past them reads 0
// and a store there is dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *p, unsigned bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00020000);
}

// Inside a one-block kernel of T threads: totals of nb block partials, valid
// in thread 0. Each thread keeps U running sums so U loads per sum are in
// flight at a time (tens of thousands of partials in a few microseconds);
// the order is fixed by nb and T.
// (stride: the distance between the N arrays, nb when 0)
template <int N, int T = kBlock, unsigned U = 8>
__device__ __forceinline__ void sum_partials(const double *partials, unsigned nb, double (&v)[N],
                                             size_t stride = 0) {
    if (stride == 0) stride = nb;
    static_assert(U == 8 || U == 16, "U is 8 or 16");
    double acc[N][U];
#pragma unroll
    for (int q = 0; q < N; q++)
#pragma unroll
        for (unsigned u = 0; u < U; u++) acc[q][u] = 0.0;
    unsigned b = flat_tid();
    for (; b + (U - 1) * T < nb; b += U * T) {
#pragma unroll
        for (unsigned u = 0; u < U; u++)
#pragma unroll
            for (int q = 0; q < N; q++) acc[q][u] += partials[(size_t)q * stride + b + u * T];
    }
    for (; b < nb; b += T)
#pragma unroll
        for (int q = 0; q < N; q++) acc[q][0] += partials[(size_t)q * stride + b];
#pragma unroll
    for (int q = 0; q < N; q++) {
        if constexpr (U == 16) {
#pragma unroll
            for (unsigned u = 0; u < 8; u++) acc[q][u] += acc[q][u + 8];
        }
        v[q] = ((acc[q][0] + acc[q][1]) + (acc[q][2] + acc[q][3])) +
               ((acc[q][4] + acc[q][5]) + (acc[q][6] + acc[q][7]));
    }
    block_sum<N, T>(v);
}

// The sums of N arrays of nb <= kFoldMax block partials ([q * nb + b]) in every
// thread of a block (of whole wavefronts, at least 64 kFoldMax / 1024 threads),
// in the order of a 1024-thread sum_partials: bit for bit the one-block
// finalize's. A kernel that needs a reduction's result adds the partials
// itself where they are few, which costs it little beside its other loads
// (fold_load, issued with them; then fold_sum) instead of a launch of 3 to 4
// us between.
constexpr unsigned kFoldMax = 1024;
constexpr int kFoldLoads = 4;  // a thread's values of each array in registers (256 threads: all)

template <int N>
struct FoldLoad {
    double a[N][kFoldLoads];
};
template <int N>
__device__ __forceinline__ void fold_load(const double *__restrict__ partials, unsigned nb, FoldLoad<N> &f) {
    const unsigned tid = (unsigned)flat_tid(), nt = blockDim.x * blockDim.y * blockDim.z;
#pragma unroll
    for (int u = 0; u < kFoldLoads; u++) {
        const unsigned b = tid + u * nt;
#pragma unroll
        for (int q = 0; q < N; q++) f.a[q][u] = partials[(size_t)q * nb + min(b, nb - 1)];
    }
}
template <int N>
__device__ __forceinline__ void pin(const FoldLoad<N> &f) {
#pragma unroll
    for (int u = 0; u < kFoldLoads; u++)
#pragma unroll
        for (int q = 0; q < N; q++) pin(f.a[q][u]);
}
template <int N>
__device__ __forceinline__ void fold_sum(const double *__restrict__ partials, unsigned nb, const FoldLoad<N> &f,
                                         double (&v)[N]) {
    __shared__ double sh[N][kFoldMax / 64];
    const unsigned tid = (unsigned)flat_tid(), nt = blockDim.x * blockDim.y * blockDim.z;
    const unsigned waves = (nb + 63u) / 64u;  // wavefronts of 64 partials
#pragma unroll
    for (int u = 0; u < kFoldLoads; u++) {
        const unsigned vt = tid + u * nt;
        if (vt >= 64u * waves) break;  // uniform over the wavefront
#pragma unroll
        for (int q = 0; q < N; q++) {
            const double a = wave_sum(vt < nb ? f.a[q][u] : 0.0);
            if ((tid & 63u) == 0) sh[q][vt >> 6] = a;
        }
    }
    for (unsigned vt = tid + kFoldLoads * nt; vt < 64u * waves; vt += nt)  // (blocks of fewer than 256 threads)
#pragma unroll
        for (int q = 0; q < N; q++) {
            const double a = wave_sum(vt < nb ? partials[(size_t)q * nb + vt] : 0.0);
            if ((tid & 63u) == 0) sh[q][vt >> 6] = a;
        }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < N; q++) {
        double s = sh[q][0];
        for (unsigned w = 1; w < waves; w++) s += sh[q][w];
        v[q] = s;
    }
}

// Tile of a cell-parallel block: z index k (lanes), y index j (wavefronts)
// and the first of its cg.planes consecutive x planes. Blocks are taken in
// launch order (tiles of one plane, then the next chunk of planes); a
// renumbering that keeps each XCD on one contiguous slab measured slower for
// these stencils on MI355X, so none is applied.
__device__ __forceinline__ void cell_tile(CellGrid cg, int &k, int &j, int &i0) {
    const unsigned L = blockIdx.x;
    const unsigned per = cg.gx * cg.gy;
    const unsigned bz = L / per, rem = L - bz * per;
    const unsigned by = rem / cg.gx, bx = rem - by * cg.gx;
    k = (int)(bx * blockDim.x + threadIdx.x);
    j = (int)(by * blockDim.y + threadIdx.y);
    i0 = (int)bz * cg.planes;
}

// Strides of the z-fastest layout.
struct Strides {
    size_t sx, sy;
    __device__ __host__ explicit Strides(Dims d) : sx((size_t)d.ny * d.nz), sy((size_t)d.nz) {}
};

// -(off-diagonal part) of A x at cell c: sum of coupling * neighbour value.
template <class T, class Load>
__device__ __forceinline__ T offdiag_sum(const T *const cpl[3], Dims d, Strides s, int i, int j,
                                         int k, size_t c, Load xv) {
    T acc = 0;
    if (i > 0) acc += cpl[0][c] * (T)xv(c - s.sx);
    if (i + 1 < d.nx) acc += cpl[0][c + s.sx] * (T)xv(c + s.sx);
    if (j > 0) acc += cpl[1][c] * (T)xv(c - s.sy);
    if (j + 1 < d.ny) acc += cpl[1][c + s.sy] * (T)xv(c + s.sy);
    if (k > 0) acc += cpl[2][c] * (T)xv(c - 1);
    if (k + 1 < d.nz) acc += cpl[2][c + 1] * (T)xv(c + 1);
    return acc;
}

}  // namespace sfp
