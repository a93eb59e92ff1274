// Kernels of the 3-D U-Net preconditioner on gfx950.
//
// Tensors are channels-last [batch][x][y][z][c], activations BF16 (stored as
// uint16), activation gradients FP32, master weights FP32 with BF16 copies
// [tap][cout][cin] for the convolutions.
//
// k_conv3r is an implicit GEMM: M = output channels (blocks of 16), N = output
// voxels (z rows of 16), K = 27 taps x input channels, on
// v_mfma_f32_16x16x32_bf16 with FP32 accumulation. Lane layouts (checked on
// the device): A[m][k] from lane m%16 + 16*(k/8), B[k][n] from lane
// n + 16*(k/8), D[m][n] in lane n + 16*(m/4), element m%4.
#include "device_util.hpp"
#include "unet.hpp"

#include <type_traits>

namespace sfp {
namespace {

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float(((unsigned)h) << 16); }
__device__ __forceinline__ uint16_t f2bf(float f) {
    // round to nearest even; NaN stays NaN
    const unsigned u = __float_as_uint(f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (uint16_t)((u >> 16) | 0x40);
    return (uint16_t)((u + 0x7fffu + ((u >> 16) & 1u)) >> 16);
}

struct ConvArgs {
    const uint16_t *in;   // [B][X][Y][Z][CIN]
    const uint16_t *w;    // [tap][COUT][CIN]
    const float *bias;    // [COUT] or null
    const uint16_t *skip; // [B][X][Y][Z][COUT] or null: added after the ReLU, or (mask) an activation
                          // whose ReLU the gradient passes: out is 0 where it is not positive
    uint16_t *out;        // BF16 output or null
    float *out32;         // FP32 output or null
    uint16_t *relu_copy;  // relu(acc + bias) before the skip, or null
    int B, X, Y, Z;
    int relu;
    int mask;
    int up;  // 1: `in` is [B][X/2][Y/2][Z/2][CIN], read nearest-up-sampled
    const double *gate;  // nonzero *gate: return at once (a stopped batch of FCG iterations)
    unsigned in_bytes;   // size of `in` (at most kInLimit)
    unsigned out_elems;  // B X Y Z COUT: the elements of out, out32, relu_copy and skip
};

// Raw buffer resources over the tensors: a load at an offset past the
// buffer's size reads 0 and a store there is dropped, so the padding and the
// partial tiles need no branches or address selects. An input offset is the
// sum of a row part and a (z, channel) part, either of which is kInOutside
// when outside the volume: with the input at most kInLimit bytes, the sum is
// then past it too. Output offsets outside the volume are kOutOutside (the
// outputs are at most 2 GiB).
constexpr unsigned kInLimit = 0x40000000u, kInOutside = 0x40000000u, kOutOutside = 0x80000000u;
typedef unsigned u4v __attribute__((ext_vector_type(4)));
typedef unsigned u2v __attribute__((ext_vector_type(2)));
typedef uint16_t h4v __attribute__((ext_vector_type(4)));
typedef __bf16 v4bf __attribute__((ext_vector_type(4)));
// four values as BF16 bits, rounded to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ u2v bf16_bits4(v4f f) {
    return __builtin_bit_cast(u2v, v4bf{(__bf16)f[0], (__bf16)f[1], (__bf16)f[2], (__bf16)f[3]});
}

// The 3x3x3 convolution (zero padding), optionally reading its input
// nearest-up-sampled, with bias, ReLU, a skip tensor added after the ReLU and
// BF16 or FP32 output. Each input row's fragments are reused in registers by
// every output row it is a tap of. A wavefront owns one 16-channel block of
// outputs (nb) on PY z rows (y0 .. y0 + PY - 1, 16 voxels of z each) and
// marches along x over a run of output planes [xa, xe). Its weight fragments
// (9 x KC, all 27 taps of its output channels) stay in VGPRs for the march.
// At each step it loads the fragments of input plane gx (PY + 2 rows, each
// row shifted by dz = -1, 0, 1 in z, times the channel chunks: KC per row)
// straight from global memory (neighbouring wavefronts' rows meet in L1/L2),
// one plane ahead of their use, and each fragment feeds the MFMAs of up to 9
// output rows: planes gx + 1, gx, gx - 1 (dx = 0, 1, 2) times the rows it
// neighbours in y. Accumulators of three output planes rotate; plane gx - 1
// is complete after the step and goes through the epilogue. The weights are
// operand A, so a lane's four results are four channels of one voxel: one
// 8-byte store (16 for FP32) and one load of the skip or mask tensor instead of
// four of 2 bytes each.
// Small volumes are bound by the march's chain of loads (a step of 36 MFMAs
// waits about 1 us for the next plane), large ones by the MFMAs and their
// fragments. 16 -> 16 channels on 8 crops of 32^3: 13.4 -> 11.7 us with these
// stores and the wavefront's indices in scalar registers. Measured and not
// taken: fragments two planes ahead (25.9 us), a march rolled to one step per
// iteration (16.7), twice the wavefronts (17.3).
template <int CIN>
constexpr int kchunks() {
    return CIN == 8 ? 1 : CIN == 16 ? 2 : CIN == 32 ? 3 : 6;
}
// K chunk kc of an input row, lane group g (8 of the MFMA's 32 K values): the
// z shift dz (0..2), the first channel c, and whether the slice exists.
template <int CIN>
__device__ __forceinline__ void kslice(int kc, int g, int &dz, int &c, bool &ok) {
    if constexpr (CIN == 8) {  // dz = g, all 8 channels; group 3 empty
        dz = g;
        c = 0;
        ok = g < 3;
    } else if constexpr (CIN == 16) {  // two z shifts per chunk, 8 channels per group
        dz = 2 * kc + (g >> 1);
        c = 8 * (g & 1);
        ok = dz < 3;
    } else if constexpr (CIN == 32) {
        dz = kc;
        c = 8 * g;
        ok = true;
    } else {
        dz = kc % 3;
        c = 32 * (kc / 3) + 8 * g;
        ok = true;
    }
}

// 16 zero bytes: lanes whose operand lies outside the volume (or outside
// the K chunk) load from here, so no loaded register is overwritten later.
__device__ __attribute__((aligned(16))) uint16_t g_zero8[8] = {0, 0, 0, 0, 0, 0, 0, 0};

// An input row is loaded once per plane: fragment C holds voxel z0 + m of
// lane m (its channel slice), and H the two halo voxels, z0 - 1 in lane m = 0
// and z0 + 16 in lane m = 15 (of each 16-lane row). The z-shifted fragments
// of the K chunks come from C by DPP shifts within the 16-lane rows (lane m
// takes lane m - 1, or m + 1), with H at the row's end, so they equal the
// fragments a load of the shifted voxels would give, bit for bit.
template <int CIN>
constexpr int kcentres() {  // C fragments per row: the channel halves of CIN = 64
    return CIN == 64 ? 2 : 1;
}
// the channel offset of lane group g's slice in centre fragment h
template <int CIN>
__device__ __forceinline__ int centre_channel(int h, int g) {
    if constexpr (CIN == 8) return 0;
    else if constexpr (CIN == 16) return 8 * (g & 1);
    else if constexpr (CIN == 32) return 8 * g;
    else return 32 * h + 8 * g;
}
// whether lane group g of centre fragment h needs the halo below (z0 - 1) or above (z0 + 16)
template <int CIN>
__device__ __forceinline__ bool halo_lo(int g) {
    return CIN == 8 ? g == 0 : CIN == 16 ? g < 2 : true;
}
template <int CIN>
__device__ __forceinline__ bool halo_hi(int g) {
    return CIN == 8 ? g == 2 : CIN == 16 ? g < 2 : true;
}
// x of lane m - 1 (from_below) or m + 1 within each 16-lane row; the lane at
// the row's end, which has no such neighbour, keeps `end` (bound_ctrl off:
// the DPP move leaves it unwritten), so the halo needs no select.
__device__ __forceinline__ v8bf dpp_shift(v8bf x, v8bf end, bool from_below) {
    const u4v u = __builtin_bit_cast(u4v, x), e = __builtin_bit_cast(u4v, end);
    u4v r;
#pragma unroll
    for (int q = 0; q < 4; q++)
        r[q] = from_below ? (unsigned)__builtin_amdgcn_update_dpp((int)e[q], (int)u[q], 0x111, 0xf, 0xf, false)
                          : (unsigned)__builtin_amdgcn_update_dpp((int)e[q], (int)u[q], 0x101, 0xf, 0xf, false);
    return __builtin_bit_cast(v8bf, r);
}
// The KC chunks of one row (kslice's layout) from its centre and halo fragments.
template <int CIN>
__device__ __forceinline__ void row_chunks(const v8bf (&c)[kcentres<CIN>()], const v8bf (&h)[kcentres<CIN>()],
                                           int g, v8bf (&out)[kchunks<CIN>()]) {
    const v8bf zero = __builtin_bit_cast(v8bf, u4v{0u, 0u, 0u, 0u});
#pragma unroll
    for (int q = 0; q < kcentres<CIN>(); q++) {
        const v8bf lo = dpp_shift(c[q], h[q], true);   // voxel z0 + m - 1 (row_shr:1; m = 0: the halo)
        const v8bf hi = dpp_shift(c[q], h[q], false);  // voxel z0 + m + 1 (row_shl:1; m = 15: the halo)
        if constexpr (CIN == 8) {
            out[0] = g == 0 ? lo : g == 1 ? c[0] : g == 2 ? hi : zero;
        } else if constexpr (CIN == 16) {
            out[0] = g < 2 ? lo : c[0];
            out[1] = g < 2 ? hi : zero;
        } else {  // 32, 64: chunk dz + 3 q
            out[3 * q] = lo;
            out[3 * q + 1] = c[q];
            out[3 * q + 2] = hi;
        }
    }
}

// UP: the input is read nearest-up-sampled (a.up set) and PY is even, so y0
// is even and rows y0 + 2k - 1 and y0 + 2k (k >= 1) read the same source row:
// the second takes the first's fragments instead of a load.
template <int PY, bool UP>
constexpr int src_row(int iy) {
    return UP && PY % 2 == 0 && iy >= 2 && iy <= PY && iy % 2 == 0 ? iy - 1 : iy;
}

template <int CIN, int COUT, int PY, int WPS, bool UP = false>
__global__ __launch_bounds__(256, WPS) void k_conv3r(ConvArgs a, int run, int xruns) {
    static_assert(!UP || PY % 2 == 0, "the shared source rows need an even row count");
    constexpr int KC = kchunks<CIN>();
    constexpr int NB = COUT / 16;
    if (a.gate && *a.gate != 0.0) return;
    const uint16_t *__restrict__ wts = a.w;
    const int X = a.X, Y = a.Y, Z = a.Z;
    const int lane = threadIdx.x & 63, g = lane >> 4, r16 = lane & 15;
    const int ypn = (Y + PY - 1) / PY, zbn = (Z + 15) / 16;
    // (in scalar registers, as all that follows from it)
    unsigned w = blockIdx.x * 4 + (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int nb = (int)(w % NB);
    w /= NB;
    const int yp = (int)(w % (unsigned)ypn);
    w /= (unsigned)ypn;
    const int zb = (int)(w % (unsigned)zbn);
    w /= (unsigned)zbn;
    const int xr = (int)(w % (unsigned)xruns);
    const int b = (int)(w / (unsigned)xruns);
    if (b >= a.B) return;  // uniform over the wavefront
    const int y0 = yp * PY, z0 = zb * 16, xa = xr * run;
    if (xa >= X) return;
    const int xe = min(xa + run, X);
    // weights [dx][dy][kc]: A[m][k] of lane m + 16 (k / 8), m the output channel
    v8bf wf[3][3][KC];
#pragma unroll
    for (int dx = 0; dx < 3; dx++)
#pragma unroll
        for (int dy = 0; dy < 3; dy++)
#pragma unroll
            for (int kc = 0; kc < KC; kc++) {
                int dz, c;
                bool ok;
                kslice<CIN>(kc, g, dz, c, ok);
                const uint16_t *p =
                    ok ? wts + ((size_t)((dx * 9 + dy * 3 + dz) * COUT + nb * 16 + r16) * CIN + c) : g_zero8;
                wf[dx][dy][kc] = __builtin_bit_cast(v8bf, *reinterpret_cast<const uint4 *>(p));
            }
    // this lane's input voxel (z) and channel byte offset per chunk within an
    // (x, y) row of the (possibly half-resolution) input: B[k][n] of lane
    // n + 16 (k / 8), n = z - z0 of the output row
    const int up = UP ? 1 : a.up;
    const int Xs = up ? X >> 1 : X, Ys = up ? Y >> 1 : Y, Zs = up ? Z >> 1 : Z;
    const auto rin = buf_rsrc(a.in, a.in_bytes);
    // 16 input channels and more: one centre and one halo fragment per row
    // and channel half (the chunks derived by DPP); 8 channels: the single
    // chunk, which already holds the three z shifts, loaded directly
    constexpr bool kDpp = CIN >= 16;
    constexpr int NC = kDpp ? kcentres<CIN>() : KC;
    // byte offsets within an (x, y) row: of the centre and halo fragments, or
    // of the chunks
    unsigned zc[NC], zh[NC];
#pragma unroll
    for (int q = 0; q < NC; q++) {
        if constexpr (kDpp) {
            const int c = centre_channel<CIN>(q, g);
            auto zoff = [&](int zi) { return (unsigned)(((up ? zi >> 1 : zi) * CIN + c) * 2); };
            const int zi = z0 + r16;
            zc[q] = zi < Z ? zoff(zi) : kInOutside;
            zh[q] = kInOutside;
            if (r16 == 0 && halo_lo<CIN>(g) && z0 > 0) zh[q] = zoff(z0 - 1);
            if (r16 == 15 && halo_hi<CIN>(g) && z0 + 16 < Z) zh[q] = zoff(z0 + 16);
        } else {
            int dz, c;
            bool ok;
            kslice<CIN>(q, g, dz, c, ok);
            const int zi = z0 + r16 + dz - 1;
            zc[q] = ok && zi >= 0 && zi < Z ? (unsigned)(((up ? zi >> 1 : zi) * CIN + c) * 2) : kInOutside;
            zh[q] = kInOutside;
        }
    }
    const unsigned row_bytes = (unsigned)(Zs * CIN * 2);
    // Offsets that do not change along the march: the input rows y0 - 1 .. y0 +
    // PY (kInOutside where outside the volume; scalars), and per lane the
    // output values' (y, z, channel) part (kOutOutside outside). Each step adds
    // its plane's part, a scalar too: one vector add per load or store.
    unsigned ry[PY + 2];
#pragma unroll
    for (int iy = 0; iy < PY + 2; iy++) {
        const int gy = y0 + iy - 1;
        ry[iy] = gy >= 0 && gy < Y ? (unsigned)(up ? gy >> 1 : gy) * row_bytes : kInOutside;
    }
    unsigned ob[PY];  // byte offsets of the 16-bit outputs within a plane: voxel z0 + r16, channels 4 g .. 4 g + 3
#pragma unroll
    for (int oy = 0; oy < PY; oy++) {
        const int gy = y0 + oy, gz = z0 + r16;
        ob[oy] = gy < Y && gz < Z ? (unsigned)((gy * Z + gz) * COUT + nb * 16 + 4 * g) * 2 : kOutOutside;
    }
    v4f acc[3][PY];
#pragma unroll
    for (int s = 0; s < 3; s++)
#pragma unroll
        for (int oy = 0; oy < PY; oy++) acc[s][oy] = v4f{0.f, 0.f, 0.f, 0.f};
    const int steps = xe - xa + 2;  // input planes xa - 1 .. xe
    // The centre and halo fragments of input plane gx: rows y0 - 1 .. y0 +
    // PY, zero outside the volume (offsets past the buffer), so the next
    // plane's loads stay in flight during this plane's MFMAs.
    auto load_plane = [&](v8bf(&fc)[PY + 2][NC], v8bf(&fh)[PY + 2][NC], int gx) {
        // the plane's part (every term below 1 GiB or kInOutside: the sum of
        // three stays below 4 GiB, and past the buffer if any term is outside)
        const unsigned po = gx >= 0 && gx < X ? (unsigned)((b * Xs + (up ? gx >> 1 : gx)) * Ys) * row_bytes
                                              : kInOutside;
#pragma unroll
        for (int iy = 0; iy < PY + 2; iy++)
#pragma unroll
            for (int q = 0; q < NC; q++) {
                if (src_row<PY, UP>(iy) != iy) continue;  // (known after unrolling)
                fc[iy][q] = __builtin_bit_cast(v8bf, __builtin_amdgcn_raw_buffer_load_b128(rin, po + ry[iy] + zc[q], 0, 0));
                if constexpr (kDpp)
                    fh[iy][q] =
                        __builtin_bit_cast(v8bf, __builtin_amdgcn_raw_buffer_load_b128(rin, po + ry[iy] + zh[q], 0, 0));
            }
    };
    v4f bias = {0.f, 0.f, 0.f, 0.f};
    if (a.bias) {
#pragma unroll
        for (int j = 0; j < 4; j++) bias[j] = a.bias[nb * 16 + 4 * g + j];
    }
    const auto rskip = buf_rsrc(a.skip, a.skip ? 2 * a.out_elems : 0);
    const auto rout = buf_rsrc(a.out, a.out ? 2 * a.out_elems : 0);
    const auto rout32 = buf_rsrc(a.out32, a.out32 ? 4 * a.out_elems : 0);
    const auto rrelu = buf_rsrc(a.relu_copy, a.relu_copy ? 2 * a.out_elems : 0);
    const bool has_skip = a.skip != nullptr, has_relu_copy = a.relu_copy != nullptr;
    const bool relu = a.relu != 0, f32 = a.out32 != nullptr, mask = a.mask != 0;
    // Two fragment buffers alternate with the step's parity and three
    // accumulator slots rotate with the step mod 3: the march is unrolled by
    // six, so every index is a constant and no fragment is copied. Step t
    // reads input plane gx = xa - 1 + t; output plane gx + 1 - dx
    // accumulates in slot (t - dx) mod 3.
    v8bf fc[2][PY + 2][NC], fh[2][PY + 2][NC];
    load_plane(fc[0], fh[0], xa - 1);
    // Lc: whether this step loads the next plane (with UP, every other step:
    // planes 2k - 1 and 2k read the same source plane, see below)
    auto step = [&](auto Pc, auto Uc, auto Lc, int t) {
        constexpr int P = decltype(Pc)::value, U = decltype(Uc)::value;
        constexpr bool L = decltype(Lc)::value;
        const int gx = xa - 1 + t;
        // byte offset of output plane gx - 1 (the plane this step completes)
        // in the 16-bit outputs
        const unsigned pb = (unsigned)((b * X + (gx - 1)) * Y * Z * COUT) * 2;
        // the skip values of that plane, loaded before the next plane's
        // fragments so that waiting for them leaves those in flight
        u2v skv[PY];
        if (has_skip && t >= 2) {
#pragma unroll
            for (int oy = 0; oy < PY; oy++)
                skv[oy] = __builtin_bit_cast(u2v, __builtin_amdgcn_raw_buffer_load_b64(rskip, pb + ob[oy], 0, 0));
        }
        if constexpr (L) load_plane(fc[1 - P], fh[1 - P], gx + 1);  // (one past the run at the end: unused)
#pragma unroll
        for (int iy = 0; iy < PY + 2; iy++) {
            v8bf ck[KC];
            if constexpr (kDpp)
                row_chunks<CIN>(fc[P][src_row<PY, UP>(iy)], fh[P][src_row<PY, UP>(iy)], g, ck);
            else
#pragma unroll
                for (int kc = 0; kc < KC; kc++) ck[kc] = fc[P][src_row<PY, UP>(iy)][kc];
#pragma unroll
            for (int dx = 0; dx < 3; dx++)
#pragma unroll
                for (int dy = 0; dy < 3; dy++) {
                    const int oy = iy - dy;
                    if (oy < 0 || oy >= PY) continue;  // known after unrolling
#pragma unroll
                    for (int kc = 0; kc < KC; kc++)
                        acc[(U - dx + 3) % 3][oy] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            wf[dx][dy][kc], ck[kc], acc[(U - dx + 3) % 3][oy], 0, 0, 0);
                }
        }
        // planes before the run (gx + 1 - dx < xa) took contributions in
        // the first two steps: clear their slots
        if (t == 0) {
#pragma unroll
            for (int oy = 0; oy < PY; oy++) acc[(U + 1) % 3][oy] = acc[(U + 2) % 3][oy] = v4f{0.f, 0.f, 0.f, 0.f};
        } else if (t == 1) {
#pragma unroll
            for (int oy = 0; oy < PY; oy++) acc[(U + 1) % 3][oy] = v4f{0.f, 0.f, 0.f, 0.f};
        }
        // output plane gx - 1 has had its three input planes
        if (t >= 2) {
            constexpr int S = (U + 1) % 3;
#pragma unroll
            for (int oy = 0; oy < PY; oy++) {
                const unsigned o = pb + ob[oy];  // past the buffers where outside the volume
                v4f v = acc[S][oy] + bias;
                if (relu)
#pragma unroll
                    for (int j = 0; j < 4; j++) v[j] = v[j] > 0.f ? v[j] : 0.f;
                if (has_relu_copy) __builtin_amdgcn_raw_buffer_store_b64(bf16_bits4(v), rrelu, o, 0, 0);
                const h4v sk = __builtin_bit_cast(h4v, skv[oy]);
                if (has_skip && !mask)
#pragma unroll
                    for (int j = 0; j < 4; j++) v[j] += bf2f(sk[j]);
                if (mask) {
                    h4v m = __builtin_bit_cast(h4v, bf16_bits4(v));
#pragma unroll
                    for (int j = 0; j < 4; j++) m[j] = bf2f(sk[j]) > 0.f ? m[j] : (uint16_t)0;
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2v, m), rout, o, 0, 0);
                }
                if (f32)  // (FP32 output: twice the 16-bit offset)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4v, v), rout32,
                                                           ob[oy] == kOutOutside ? kOutOutside : 2 * o, 0, 0);
                else if (!mask)
                    __builtin_amdgcn_raw_buffer_store_b64(bf16_bits4(v), rout, o, 0, 0);
                acc[S][oy] = v4f{0.f, 0.f, 0.f, 0.f};
            }
        }
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using LD = std::true_type;
    using NL = std::false_type;
    if constexpr (UP) {
        // The run starts on an even plane (the launcher makes runs even), so
        // step t's plane xa - 1 + t reads source plane (xa - 1 + t) >> 1: the
        // same as step t - 1's for even t >= 2. Steps with even t load the
        // next source plane, into the other buffer; odd steps load nothing,
        // and the next step reads their buffer again. Buffer of step t:
        // ((t + 1) >> 1) mod 2, period 4; with the accumulator slots' period
        // 3 the march is unrolled by twelve.
        for (int t0 = 0; t0 < steps; t0 += 12) {  // uniform over the wavefront
            step(I0{}, I0{}, LD{}, t0);
            if (t0 + 1 >= steps) break;
            step(I1{}, I1{}, NL{}, t0 + 1);
            if (t0 + 2 >= steps) break;
            step(I1{}, I2{}, LD{}, t0 + 2);
            if (t0 + 3 >= steps) break;
            step(I0{}, I0{}, NL{}, t0 + 3);
            if (t0 + 4 >= steps) break;
            step(I0{}, I1{}, LD{}, t0 + 4);
            if (t0 + 5 >= steps) break;
            step(I1{}, I2{}, NL{}, t0 + 5);
            if (t0 + 6 >= steps) break;
            step(I1{}, I0{}, LD{}, t0 + 6);
            if (t0 + 7 >= steps) break;
            step(I0{}, I1{}, NL{}, t0 + 7);
            if (t0 + 8 >= steps) break;
            step(I0{}, I2{}, LD{}, t0 + 8);
            if (t0 + 9 >= steps) break;
            step(I1{}, I0{}, NL{}, t0 + 9);
            if (t0 + 10 >= steps) break;
            step(I1{}, I1{}, LD{}, t0 + 10);
            if (t0 + 11 >= steps) break;
            step(I0{}, I2{}, NL{}, t0 + 11);
        }
    } else {
        for (int t0 = 0; t0 < steps; t0 += 6) {  // uniform over the wavefront
            step(I0{}, I0{}, LD{}, t0);
            if (t0 + 1 >= steps) break;
            step(I1{}, I1{}, LD{}, t0 + 1);
            if (t0 + 2 >= steps) break;
            step(I0{}, I2{}, LD{}, t0 + 2);
            if (t0 + 3 >= steps) break;
            step(I1{}, I0{}, LD{}, t0 + 3);
            if (t0 + 4 >= steps) break;
            step(I0{}, I1{}, LD{}, t0 + 4);
            if (t0 + 5 >= steps) break;
            step(I1{}, I2{}, LD{}, t0 + 5);
        }
    }
}

// Weight gradient partials as an implicit GEMM on MFMA (M = 16 output channels,
// N = 16 input channels, K = voxels; BF16 products, exact in FP32, FP32
// accumulation): part[chunk][tile][tap][co][ci] = sum_v g[v][co] x[v + tap][ci]
// for the voxels of a chunk and the channel tile blockIdx.y; "tap" 27 has x = 1
// and gives the bias sums. up: x has half the resolution and is read
// nearest-up-sampled.
//
// A block stages one plane of a column (yt x zt voxels, up to kDwVoxels) of g
// and three planes of x with their one-voxel frame in LDS, as the tensors lie
// (16 channels of a voxel together), and marches along x, a plane's loads in
// flight while the one before is used: x is read from memory 1.3 times and once
// more per run instead of 27 times. Both MFMA operands need 8 voxels of one
// channel per lane; ds_read_b64_tr_b16 transposes on the way (a 16-lane group
// reads 4 voxels x 16 channels, lane n gets channel n's 4), so a tap is an
// address offset. The 28 taps are split over 7 wavefronts, which all pass over
// every voxel: no sum over wavefronts, 16 accumulator registers each. What
// bounds it is LDS reads, 68 of 512 B per 32 voxels for 28 MFMAs. Voxels past
// the volume, or past the column in its last 32, read the zero row in both.
//
// 32^3 x 8 crops, all ten convolutions: 127 us (607 with a block per tap and
// both tensors transposed by 2-byte LDS stores), their partials' sums 15 us in
// one launch (305 in twenty).
constexpr int kDwVoxels = 256;  // voxels of a column plane
constexpr int kDwFramed = 340;  // the most with the frame: sides up to 32, product up to 256
constexpr int kDwThreads = 448, kDwTaps = 28;
constexpr int kDwPart = kDwTaps * 256;  // floats of a partial tile

typedef short v4s __attribute__((ext_vector_type(4)));
typedef short v8s __attribute__((ext_vector_type(8)));

template <int CIN, int COUT>
__global__ __launch_bounds__(kDwThreads) void k_conv_dw(const uint16_t *__restrict__ x,
                                                        const uint16_t *__restrict__ g, DwPlan p, int up,
                                                        float *__restrict__ part) {
    constexpr int NB = CIN < 16 ? 1 : CIN / 16;
    constexpr int kZero = 3 * kDwFramed;  // the zero row
    __shared__ __attribute__((aligned(16))) uint16_t sx[kZero + 1][16];
    __shared__ __attribute__((aligned(16))) uint16_t sg[kDwVoxels][16];
    typedef __attribute__((address_space(3))) v4s *lds4;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mb = (int)blockIdx.y / NB, nb = (int)blockIdx.y % NB;
    const int fz = p.zt + 2, framed = (p.yt + 2) * fz, voxels = p.yt * p.zt;
    // this lane's voxels in a unit of 32: kq and kq + 16 (any assignment of
    // voxels to K will do, as long as both operands have it)
    const int kq = 4 * (lane >> 4) + ((lane & 15) >> 2), pc = 4 * (lane & 3);
    if (tid < 16) sx[kZero][tid] = 0;
    // pieces of 16 bytes: (voxel, half) = (e / 2, e % 2)
    constexpr int RX = (2 * kDwFramed + kDwThreads - 1) / kDwThreads;
    constexpr int RG = (2 * kDwVoxels + kDwThreads - 1) / kDwThreads;
    uint4 rx[RX], rg[RG];
    const int Xs = p.X >> up, Ys = p.Y >> up, Zs = p.Z >> up;
    v4f acc[4];
#pragma unroll
    for (int j = 0; j < 4; j++) acc[j] = v4f{0.f, 0.f, 0.f, 0.f};
    const uint4 none = make_uint4(0, 0, 0, 0);
    for (int item = blockIdx.x; item < p.items; item += gridDim.x) {
        const int col = item / p.segs, seg = item - col * p.segs;
        const int tz = col % p.nzt, ty = (col / p.nzt) % p.nyt, bb = col / (p.nzt * p.nyt);
        const int y0 = ty * p.yt, z0 = tz * p.zt;
        const int xa = seg * p.seg, xe = min(xa + p.seg, p.X);
        auto load_x = [&](int plane) {
            const uint16_t *px = x + (size_t)(bb * (long long)Xs + (plane >> up)) * Ys * Zs * CIN + 16 * nb;
#pragma unroll
            for (int r = 0; r < RX; r++) {
                const int e = tid + r * kDwThreads, vi = e >> 1;
                const int yy = (int)(((unsigned)vi * p.magic_f) >> 16), zz = vi - yy * fz;
                const int gy = y0 + yy - 1, gz = z0 + zz - 1;
                rx[r] = none;
                if (vi < framed && (CIN >= 16 || !(e & 1)) && plane >= 0 && plane < p.X && gy >= 0 && gy < p.Y &&
                    gz >= 0 && gz < p.Z)
                    rx[r] = *reinterpret_cast<const uint4 *>(px + ((size_t)(gy >> up) * Zs + (gz >> up)) * CIN +
                                                              8 * (e & 1));
            }
        };
        auto store_x = [&](int plane) {
            const int base = ((plane + 1) % 3) * kDwFramed;
#pragma unroll
            for (int r = 0; r < RX; r++) {
                const int e = tid + r * kDwThreads;
                if (e >> 1 < framed) *reinterpret_cast<uint4 *>(&sx[base + (e >> 1)][8 * (e & 1)]) = rx[r];
            }
        };
        auto load_g = [&](int plane) {
            const uint16_t *pg = g + (size_t)(bb * (long long)p.X + plane) * p.Y * p.Z * COUT + 16 * mb;
#pragma unroll
            for (int r = 0; r < RG; r++) {
                const int e = tid + r * kDwThreads, vi = e >> 1;
                const int yy = (int)(((unsigned)vi * p.magic) >> 16), zz = vi - yy * p.zt;
                const int gy = y0 + yy, gz = z0 + zz;
                rg[r] = none;
                if (vi < voxels && gy < p.Y && gz < p.Z)
                    rg[r] = *reinterpret_cast<const uint4 *>(pg + ((size_t)gy * p.Z + gz) * COUT + 8 * (e & 1));
            }
        };
        auto store_g = [&] {
#pragma unroll
            for (int r = 0; r < RG; r++) {
                const int e = tid + r * kDwThreads;
                if (e < 2 * kDwVoxels) *reinterpret_cast<uint4 *>(&sg[e >> 1][8 * (e & 1)]) = rg[r];
            }
        };
        // the corner (tap 0) of each of this lane's voxels in a staged plane
        int corner[kDwVoxels / 32][2];
#pragma unroll
        for (int u = 0; u < kDwVoxels / 32; u++)
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int q = 32 * u + kq + 16 * h;
                const int yy = (int)(((unsigned)q * p.magic) >> 16), zz = q - yy * p.zt;
                const bool in = q < voxels && y0 + yy < p.Y && z0 + zz < p.Z;
                corner[u][h] = in ? (yy * fz + zz) * 16 + pc : -1;
            }
        load_x(xa - 1);
        __syncthreads();  // the item before is done with LDS
        store_x(xa - 1);
        load_x(xa);
        store_x(xa);
        load_x(xa + 1);
        load_g(xa);
        for (int xp = xa; xp < xe; xp++) {
            __syncthreads();  // the plane before is done with
            store_x(xp + 1);
            store_g();
            __syncthreads();
            if (xp + 1 < xe) {
                load_x(xp + 2);
                load_g(xp + 1);
            }
            int off[4];  // this wavefront's taps: the plane's slot and the offset in it (uniform)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int t = 4 * wave + j, dx = t / 9, dy = (t / 3) % 3, dz = t % 3;
                off[j] = (((xp + dx) % 3) * kDwFramed + dy * fz + dz) * 16;
            }
#pragma unroll
            for (int u = 0; u < kDwVoxels / 32; u++) {
                if (32 * u >= voxels) break;  // uniform
                auto read = [](const uint16_t *a, const uint16_t *b) {
                    const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)a);
                    const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4)b);
                    return __builtin_bit_cast(v8bf, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
                };
                const uint16_t *sgu = &sg[0][0] + (32 * u + kq) * 16 + pc, *sxu = &sx[0][0];
                const v8bf ga = read(sgu, sgu + 256);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    v8bf xb;
                    if (j == 3 && wave == 6) {  // the bias: x = 1
                        const short one = 0x3f80;
                        xb = __builtin_bit_cast(v8bf, v8s{one, one, one, one, one, one, one, one});
                    } else {
                        const int c0 = corner[u][0], c1 = corner[u][1];
                        xb = read(sxu + (c0 < 0 ? kZero * 16 + pc : c0 + off[j]),
                                  sxu + (c1 < 0 ? kZero * 16 + pc : c1 + off[j]));
                    }
                    acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ga, xb, acc[j], 0, 0, 0);
                }
            }
        }
    }
    // D[co][ci]: row 4 (lane / 16) + i, column lane % 16
    float *out = part + ((size_t)blockIdx.x * gridDim.y + blockIdx.y) * kDwPart;
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int i = 0; i < 4; i++)
            out[(4 * wave + j) * 256 + (4 * (lane >> 4) + i) * 16 + (lane & 15)] = acc[j][i];
}

// The sums over the chunks of every convolution's partials, in a fixed order: a
// block per tap of a tile, wavefront w adding the chunks w, w + 8, .. and their
// eight sums added at the end.
constexpr int kDwSumWaves = 8;
__global__ __launch_bounds__(64 * kDwSumWaves) void k_dw_sums(DwSums s, const float *__restrict__ part,
                                                              float *__restrict__ grad) {
    __shared__ v4f red[kDwSumWaves][64];
    int k = 0;
    while (k + 1 < kUNetConvs && (int)blockIdx.x >= s.first[k + 1]) k++;
    const int rem = (int)blockIdx.x - s.first[k], tile = rem / kDwTaps, t = rem % kDwTaps;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int nb = tile % s.nb[k], mb = tile / s.nb[k];
    const float *src = part + s.off[k] + (size_t)tile * kDwPart + t * 256 + 4 * lane;
    const size_t stride = (size_t)s.tiles[k] * kDwPart;
    v4f sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int c = wave; c < s.chunks[k]; c += kDwSumWaves) sum += *reinterpret_cast<const v4f *>(src + c * stride);
    red[wave][lane] = sum;
    __syncthreads();
    if (wave == 0) {
        for (int w = 1; w < kDwSumWaves; w++) sum += red[w][lane];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int e = 4 * lane + i, co = 16 * mb + e / 16, ci = 16 * nb + e % 16;
            if (t < 27) {
                if (ci < s.cin[k]) grad[s.off_w[k] + ((size_t)t * s.cout[k] + co) * s.cin[k] + ci] = sum[i];
            } else if (ci == 0) {
                grad[s.off_b[k] + co] = sum[i];
            }
        }
    }
}

// The passes between the convolutions are bound by the bytes they move: a
// thread takes 8 channels of a voxel (16-byte loads and stores), and the
// backward ones end with the activation's ReLU and the rounding the next
// convolution reads, so no FP32 gradient is stored for a pass of its own.
struct Voxel8 {
    int c, z, y, x, b;  // first channel; position in a volume of the pass's own extents
};
__device__ __forceinline__ Voxel8 voxel8(unsigned i, int X, int Y, int Z, int C) {
    Voxel8 v;
    unsigned r = i;
    const unsigned c8 = (unsigned)C / 8;
    v.c = 8 * (int)(r % c8);
    r /= c8;
    v.z = (int)(r % (unsigned)Z);
    r /= (unsigned)Z;
    v.y = (int)(r % (unsigned)Y);
    r /= (unsigned)Y;
    v.x = (int)(r % (unsigned)X);
    v.b = (int)(r / (unsigned)X);
    return v;
}
struct Half8 {
    uint16_t h[8];
};
__device__ __forceinline__ Half8 load_half8(const uint16_t *p) {
    return __builtin_bit_cast(Half8, *reinterpret_cast<const uint4 *>(p));
}
__device__ __forceinline__ void store_half8(uint16_t *p, const Half8 &v) {
    *reinterpret_cast<uint4 *>(p) = __builtin_bit_cast(uint4, v);
}
struct Float8 {
    float f[8];
};
__device__ __forceinline__ Float8 load_float8(const float *p) {
    Float8 v;
    const v4f a = reinterpret_cast<const v4f *>(p)[0], b = reinterpret_cast<const v4f *>(p)[1];
#pragma unroll
    for (int c = 0; c < 4; c++) v.f[c] = a[c], v.f[4 + c] = b[c];
    return v;
}
// bf16(g) where the activation is positive, else 0
__device__ __forceinline__ Half8 relu_masked(const Float8 &g, const Half8 &act) {
    Half8 o;
#pragma unroll
    for (int c = 0; c < 8; c++) o.h[c] = bf2f(act.h[c]) > 0.f ? f2bf(g.f[c]) : (uint16_t)0;
    return o;
}
// child d of a coarse voxel, as an offset into the fine tensor
__device__ __forceinline__ size_t child8(const Voxel8 &v, int d, int X, int Y, int Z, int C) {
    return ((((size_t)v.b * X + 2 * v.x + (d >> 2)) * Y + 2 * v.y + ((d >> 1) & 1)) * Z + 2 * v.z + (d & 1)) * C +
           v.c;
}

__global__ __launch_bounds__(256) void k_pool2(const uint16_t *__restrict__ in, unsigned n8, int X, int Y,
                                               int Z, int C, uint16_t *__restrict__ out, const double *gate) {
    if (gate && *gate != 0.0) return;
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n8) return;
    const Voxel8 v = voxel8(i, X / 2, Y / 2, Z / 2, C);
    Half8 o;
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < 8; d++) {
        const Half8 h = load_half8(in + child8(v, d, X, Y, Z, C));
#pragma unroll
        for (int c = 0; c < 8; c++) s[c] += bf2f(h.h[c]);
    }
#pragma unroll
    for (int c = 0; c < 8; c++) o.h[c] = f2bf(s[c] * 0.125f);
    store_half8(out + 8 * (size_t)i, o);
}

// g16[fine] = g[coarse] / 8 + add[fine], through the ReLU of act[fine]
__global__ __launch_bounds__(256) void k_pool2_bwd(const float *__restrict__ g, const float *__restrict__ add,
                                                   const uint16_t *__restrict__ act, unsigned n8, int X, int Y,
                                                   int Z, int C, uint16_t *__restrict__ g16) {
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n8) return;
    const Voxel8 v = voxel8(i, X, Y, Z, C);
    const size_t vc = (((size_t)v.b * (X / 2) + v.x / 2) * (Y / 2) + v.y / 2) * (Z / 2) + v.z / 2;
    const Float8 gc = load_float8(g + vc * C + v.c), ad = load_float8(add + 8 * (size_t)i);
    Float8 o;
#pragma unroll
    for (int c = 0; c < 8; c++) {
        float t = 0.125f * gc.f[c];
        t += ad.f[c];
        o.f[c] = t;
    }
    store_half8(g16 + 8 * (size_t)i, relu_masked(o, load_half8(act + 8 * (size_t)i)));
}

// g16[coarse] = the sum of the 8 children of g[fine], through the ReLU of act[coarse]
__global__ __launch_bounds__(256) void k_up2_bwd(const float *__restrict__ g, const uint16_t *__restrict__ act,
                                                 unsigned n8, int Xc, int Yc, int Zc, int C,
                                                 uint16_t *__restrict__ g16) {
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n8) return;
    const Voxel8 v = voxel8(i, Xc, Yc, Zc, C);
    Float8 s = {{0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int d = 0; d < 8; d++) {
        const Float8 h = load_float8(g + child8(v, d, 2 * Xc, 2 * Yc, 2 * Zc, C));
#pragma unroll
        for (int c = 0; c < 8; c++) s.f[c] += h.f[c];
    }
    store_half8(g16 + 8 * (size_t)i, relu_masked(s, load_half8(act + 8 * (size_t)i)));
}

// z[v] = bo + sum_c wo[c] d0[v][c]
__global__ __launch_bounds__(256) void k_head_fwd(const uint16_t *__restrict__ d0, const float *__restrict__ wb,
                                                  size_t nv, float *__restrict__ z, const double *gate) {
    if (gate && *gate != 0.0) return;
    const size_t v = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (v >= nv) return;
    float s = wb[16];
#pragma unroll
    for (int q = 0; q < 2; q++) {
        const Half8 h = load_half8(d0 + v * 16 + 8 * q);
#pragma unroll
        for (int c = 0; c < 8; c++) s += wb[8 * q + c] * bf2f(h.h[c]);
    }
    z[v] = s;
}

// g16[v][c] = dz[v] wo[c] through the ReLU of d0; per-block partials of sum dz
// d0[v][c] (16) and sum dz
__global__ __launch_bounds__(256) void k_head_bwd(const uint16_t *__restrict__ d0, const float *__restrict__ wb,
                                                  const float *__restrict__ dz, size_t nv,
                                                  uint16_t *__restrict__ g16, double *__restrict__ part) {
    const size_t v = (size_t)blockIdx.x * 256 + threadIdx.x;
    double acc[17];
#pragma unroll
    for (int c = 0; c < 17; c++) acc[c] = 0.0;
    if (v < nv) {
        const float d = dz[v];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const Half8 h = load_half8(d0 + v * 16 + 8 * q);
            Float8 gd;
#pragma unroll
            for (int c = 0; c < 8; c++) {
                gd.f[c] = d * wb[8 * q + c];
                acc[8 * q + c] = (double)d * bf2f(h.h[c]);
            }
            store_half8(g16 + v * 16 + 8 * q, relu_masked(gd, h));
        }
        acc[16] = d;
    }
    block_partials<17>(acc, part);
}

// per-block partials of (mask (z - t)^2, mask)
__global__ __launch_bounds__(256) void k_mse(const float *__restrict__ z, const float *__restrict__ t,
                                             const float *__restrict__ m, size_t nv,
                                             double *__restrict__ part) {
    const size_t v = (size_t)blockIdx.x * 256 + threadIdx.x;
    double acc[2] = {0.0, 0.0};
    if (v < nv) {
        const double mm = m ? m[v] : 1.0;
        const double d = (double)z[v] - t[v];
        acc[0] = mm * d * d;
        acc[1] = mm;
    }
    block_partials<2>(acc, part);
}

// out[q] = the sum of column q's nb partials (a block per column); out32 (or
// null) receives it rounded
__global__ __launch_bounds__(256) void k_sum_partials(const double *__restrict__ part, unsigned nb,
                                                      double *__restrict__ out, float *__restrict__ out32) {
    const int q = blockIdx.x;
    double v[1] = {0.0};
#pragma unroll 4
    for (unsigned b = threadIdx.x; b < nb; b += 256) v[0] += part[(size_t)q * nb + b];
    block_sum<1>(v);
    if (threadIdx.x == 0) {
        out[q] = v[0];
        if (out32) out32[q] = (float)v[0];
    }
}

__global__ __launch_bounds__(256) void k_mse_grad(const float *__restrict__ z, const float *__restrict__ t,
                                                  const float *__restrict__ m, size_t nv,
                                                  const double *__restrict__ sums, float *__restrict__ dz) {
    const size_t v = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (v >= nv) return;
    const double cnt = sums[1];
    const float mm = m ? m[v] : 1.f;
    dz[v] = cnt > 0 ? (float)(mm * 2.0 * ((double)z[v] - t[v]) / cnt) : 0.f;
}

__global__ __launch_bounds__(256) void k_adam(float *__restrict__ w, const float *__restrict__ g,
                                              float *__restrict__ m, float *__restrict__ v, size_t n,
                                              float lr, float b1, float b2, float eps, float c1, float c2) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// BF16 forward weights [tap][cout][cin] (taps padded with zeros) and the
// flipped, transposed copy for the input gradient: wt[tap'][ci][co] = w[26-tap'][co][ci].
__global__ __launch_bounds__(256) void k_cast_weights(const float *__restrict__ w, int cin, int cout,
                                                      int taps_fwd, int taps_bwd,
                                                      uint16_t *__restrict__ wf,
                                                      uint16_t *__restrict__ wt) {
    const size_t n = 27 * (size_t)cin * cout;
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < (size_t)taps_fwd * cin * cout) wf[i] = i < n ? f2bf(w[i]) : (uint16_t)0;
    if (wt && i < (size_t)taps_bwd * cin * cout) {
        uint16_t val = 0;
        if (i < n) {
            const int tp = (int)(i / ((size_t)cin * cout));
            const int rem = (int)(i - (size_t)tp * cin * cout);
            const int ci = rem / cout, co = rem - ci * cout;  // wt index [tp][ci][co]
            val = f2bf(w[((size_t)(26 - tp) * cout + co) * cin + ci]);
        }
        wt[i] = val;
    }
}

// FP32 [nv][4] -> BF16 [nv][8] (channels 4..7 zero)
__global__ __launch_bounds__(256) void k_pack_input(const float *__restrict__ in, size_t nv,
                                                    uint16_t *__restrict__ out) {
    const size_t v = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (v >= nv) return;
    Half8 o = {{0, 0, 0, 0, 0, 0, 0, 0}};
#pragma unroll
    for (int c = 0; c < 4; c++) o.h[c] = f2bf(in[v * 4 + c]);
    store_half8(out + v * 8, o);
}

unsigned blocks_for(size_t n) { return (unsigned)((n + 255) / 256); }

template <int CIN, int COUT>
void conv_dispatch(hipStream_t st, const ConvArgs &a) {
    // rows per wavefront and the wavefronts per SIMD the launch bound asks
    // for, fastest of PY = 1..4 measured on MI355X for each shape at its
    // U-Net level (128^3, 64^3, 32^3); more rows reuse each loaded fragment
    // more often but hold more VGPRs (the weight fragments alone take 36 to
    // 216)
    constexpr int PY = CIN == 8 ? 4 : COUT == 64 ? 1 : 2;
    constexpr int WPS = CIN <= 32 ? 2 : 1;
    // x runs: WPS wavefronts per SIMD of the 256 CUs. With 64 input channels
    // one fits, and a second round of them loads its weights (54 KB each) again:
    // 64 -> 64 on 8 volumes of 8^3 in 21.6 us with 2048 wavefronts, 13.3 with 1024
    const long long base = (long long)a.B * ((a.Z + 15) / 16) * ((a.Y + PY - 1) / PY) * (COUT / 16);
    const long long target = 1024 * WPS;
    int xruns = (int)std::min<long long>(a.X, std::max<long long>(1, (target + base - 1) / base));
    const int run = (a.X + xruns - 1) / xruns;
    xruns = (a.X + run - 1) / run;
    const long long waves = base * xruns;
    // the decoder's up-sampled inputs (32 -> 16 and 64 -> 32 channels) take
    // the kernel that reads each shared source row once
    // (its runs start on even planes: each loaded source plane serves two)
    if constexpr (PY % 2 == 0 && ((CIN == 32 && COUT == 16) || (CIN == 64 && COUT == 32))) {
        if (a.up) {
            const int run2 = (run + 1) & ~1;
            const int xruns2 = (a.X + run2 - 1) / run2;
            const long long waves2 = base * xruns2;
            hipLaunchKernelGGL((k_conv3r<CIN, COUT, PY, WPS, true>), dim3((unsigned)((waves2 + 3) / 4)), dim3(256), 0,
                               st, a, run2, xruns2);
            SFP_LAUNCH_CHECK();
            return;
        }
    }
    hipLaunchKernelGGL((k_conv3r<CIN, COUT, PY, WPS>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, st, a,
                       run, xruns);
    SFP_LAUNCH_CHECK();
}

template <int CIN, int COUT>
void dw_dispatch(hipStream_t st, const uint16_t *x, const uint16_t *g, const DwPlan &p, int up, float *part) {
    hipLaunchKernelGGL((k_conv_dw<CIN, COUT>), dim3(p.chunks, p.tiles), dim3(kDwThreads), 0, st, x, g, p, up,
                       part);
    SFP_LAUNCH_CHECK();
}

}  // namespace

void unet_conv(hipStream_t st, int cin, int cout, const uint16_t *in, const uint16_t *w,
               const float *bias, const uint16_t *skip, uint16_t *out, float *out32,
               uint16_t *relu_copy, int B, int X, int Y, int Z, bool relu, bool up_input,
               const double *gate, const uint16_t *mask) {
    if (mask && (skip || relu_copy)) throw ArgError("a masked convolution has no skip tensor");
    if (up_input && (X % 2 || Y % 2 || Z % 2)) throw ArgError("up-sampled input needs even extents");
    const size_t in_bytes = (size_t)B * (up_input ? (size_t)(X / 2) * (Y / 2) * (Z / 2) : (size_t)X * Y * Z) * cin * 2;
    const size_t out_elems = (size_t)B * X * Y * Z * cout;
    if (in_bytes > kInLimit || out_elems * 4 > kOutOutside)
        throw ArgError("convolution tensors too large for 32-bit buffer offsets");
    ConvArgs a{in, w, bias, mask ? mask : skip, out, out32, relu_copy, B, X, Y, Z, relu ? 1 : 0, mask ? 1 : 0,
               up_input ? 1 : 0, gate,
               (unsigned)in_bytes, (unsigned)out_elems};
#define SFP_CONV(CI, CO) \
    if (cin == CI && cout == CO) return conv_dispatch<CI, CO>(st, a);
    SFP_CONV(8, 16)
    SFP_CONV(16, 16)
    SFP_CONV(16, 32)
    SFP_CONV(32, 16)
    SFP_CONV(32, 32)
    SFP_CONV(32, 64)
    SFP_CONV(64, 32)
    SFP_CONV(64, 64)
#undef SFP_CONV
    throw ArgError("unsupported convolution shape");
}

DwPlan unet_dw_plan(int cin, int cout, int B, int X, int Y, int Z) {
    DwPlan p{};
    p.X = X, p.Y = Y, p.Z = Z;
    const auto share = [](int n, int most) {  // the size of equal parts of at most `most`
        const int parts = (n + most - 1) / most;
        return (n + parts - 1) / parts;
    };
    p.zt = share(Z, 32);
    p.yt = share(Y, std::min(32, kDwVoxels / p.zt));
    p.nyt = (Y + p.yt - 1) / p.yt;
    p.nzt = (Z + p.zt - 1) / p.zt;
    // q / zt as q * magic >> 16: exact for q < 1024 and divisors up to 34
    p.magic = 65536u / (unsigned)p.zt + 1;
    p.magic_f = 65536u / (unsigned)(p.zt + 2) + 1;
    p.tiles = (cout / 16) * std::max(1, cin / 16);
    const long long columns = (long long)B * p.nyt * p.nzt;
    // blocks: one per CU (each more adds its partial tile's 28 KB to write and
    // sum; a run's first plane costs three of x)
    const int want = std::max(1, kDwBlocks / p.tiles);
    const int segs = (int)std::min<long long>(X, std::max<long long>(1, (want + columns - 1) / columns));
    p.seg = (X + segs - 1) / segs;
    p.segs = (X + p.seg - 1) / p.seg;
    if (columns * p.segs > 0x7fffffff) throw ArgError("weight gradient: volume too large");
    p.items = (int)(columns * p.segs);
    const int rounds = (p.items + want - 1) / want;
    p.chunks = (p.items + rounds - 1) / rounds;
    return p;
}

size_t unet_dw_part(const DwPlan &p) { return (size_t)p.chunks * p.tiles * kDwPart; }

void unet_conv_dw(hipStream_t st, int cin, int cout, const uint16_t *x, const uint16_t *g, const DwPlan &p,
                  bool up_input, float *part) {
    if (up_input && (p.X % 2 || p.Y % 2 || p.Z % 2)) throw ArgError("up-sampled input needs even extents");
    if (p.yt > 32 || p.zt > 32 || p.yt * p.zt > kDwVoxels) throw ArgError("weight gradient: plane too large");
#define SFP_DW(CI, CO) \
    if (cin == CI && cout == CO) return dw_dispatch<CI, CO>(st, x, g, p, up_input ? 1 : 0, part);
    SFP_DW(8, 16)
    SFP_DW(16, 16)
    SFP_DW(16, 32)
    SFP_DW(32, 16)
    SFP_DW(32, 32)
    SFP_DW(32, 64)
    SFP_DW(64, 32)
    SFP_DW(64, 64)
#undef SFP_DW
    throw ArgError("unsupported convolution shape");
}

void unet_dw_sums(hipStream_t st, const DwPlan plan[kUNetConvs], const long long off_w[kUNetConvs],
                  const long long off_b[kUNetConvs], const float *part, float *grad) {
    DwSums s{};
    size_t off = 0;
    for (int k = 0; k < kUNetConvs; k++) {
        s.off[k] = off;
        off += unet_dw_part(plan[k]);
        s.chunks[k] = plan[k].chunks;
        s.tiles[k] = plan[k].tiles;
        s.cin[k] = kConvCin[k];
        s.cout[k] = kConvCout[k];
        s.nb[k] = std::max(1, kConvCin[k] / 16);
        s.off_w[k] = off_w[k];
        s.off_b[k] = off_b[k];
        s.first[k + 1] = s.first[k] + plan[k].tiles * kDwTaps;
    }
    hipLaunchKernelGGL(k_dw_sums, dim3(s.first[kUNetConvs]), dim3(64 * kDwSumWaves), 0, st, s, part, grad);
    SFP_LAUNCH_CHECK();
}

// 8-channel groups of a tensor (the passes over them index in 32 bits)
static unsigned groups8(int B, int X, int Y, int Z, int C) {
    const size_t n = (size_t)B * X * Y * Z * (C / 8);
    if (C % 8 || n > 0xffffff00u) throw ArgError("U-Net tensor too large");
    return (unsigned)n;
}

void unet_pool2(hipStream_t st, const uint16_t *in, int B, int X, int Y, int Z, int C, uint16_t *out,
                const double *gate) {
    const unsigned n = groups8(B, X / 2, Y / 2, Z / 2, C);
    hipLaunchKernelGGL(k_pool2, dim3(blocks_for(n)), dim3(256), 0, st, in, n, X, Y, Z, C, out, gate);
    SFP_LAUNCH_CHECK();
}

void unet_pool2_bwd(hipStream_t st, const float *g, const float *add, const uint16_t *act, int B, int X, int Y,
                    int Z, int C, uint16_t *g16) {
    const unsigned n = groups8(B, X, Y, Z, C);
    hipLaunchKernelGGL(k_pool2_bwd, dim3(blocks_for(n)), dim3(256), 0, st, g, add, act, n, X, Y, Z, C, g16);
    SFP_LAUNCH_CHECK();
}

void unet_up2_bwd(hipStream_t st, const float *g, const uint16_t *act, int B, int Xc, int Yc, int Zc, int C,
                  uint16_t *g16) {
    const unsigned n = groups8(B, Xc, Yc, Zc, C);
    hipLaunchKernelGGL(k_up2_bwd, dim3(blocks_for(n)), dim3(256), 0, st, g, act, n, Xc, Yc, Zc, C, g16);
    SFP_LAUNCH_CHECK();
}

void unet_head_fwd(hipStream_t st, const uint16_t *d0, const float *wb, size_t nv, float *z,
                   const double *gate) {
    hipLaunchKernelGGL(k_head_fwd, dim3(blocks_for(nv)), dim3(256), 0, st, d0, wb, nv, z, gate);
    SFP_LAUNCH_CHECK();
}

void unet_head_bwd(hipStream_t st, const uint16_t *d0, const float *wb, const float *dz, size_t nv,
                   uint16_t *g16, double *part, double *sums, float *gwb) {
    const unsigned nb = blocks_for(nv);
    hipLaunchKernelGGL(k_head_bwd, dim3(nb), dim3(256), 0, st, d0, wb, dz, nv, g16, part);
    SFP_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_sum_partials, dim3(17), dim3(256), 0, st, part, nb, sums, gwb);
    SFP_LAUNCH_CHECK();
}

void unet_mse(hipStream_t st, const float *z, const float *t, const float *m, size_t nv,
              double *part, double *sums, float *dz) {
    const unsigned nb = blocks_for(nv);
    hipLaunchKernelGGL(k_mse, dim3(nb), dim3(256), 0, st, z, t, m, nv, part);
    SFP_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_sum_partials, dim3(2), dim3(256), 0, st, part, nb, sums, (float *)nullptr);
    SFP_LAUNCH_CHECK();
    if (dz) {
        hipLaunchKernelGGL(k_mse_grad, dim3(nb), dim3(256), 0, st, z, t, m, nv, sums, dz);
        SFP_LAUNCH_CHECK();
    }
}

void unet_adam(hipStream_t st, float *w, const float *g, float *m, float *v, size_t n, float lr,
               int step) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_adam, dim3(blocks_for(n)), dim3(256), 0, st, w, g, m, v, n, lr, b1, b2, eps, c1, c2);
    SFP_LAUNCH_CHECK();
}

void unet_cast_weights(hipStream_t st, const float *w, int cin, int cout, uint16_t *wf, uint16_t *wt) {
    const int tf = conv_taps(cin), tb = conv_taps(cout);
    const size_t n = (size_t)std::max(tf, tb) * cin * cout;
    hipLaunchKernelGGL(k_cast_weights, dim3(blocks_for(n)), dim3(256), 0, st, w, cin, cout, tf, tb, wf, wt);
    SFP_LAUNCH_CHECK();
}

void unet_pack_input(hipStream_t st, const float *in, size_t nv, uint16_t *out) {
    hipLaunchKernelGGL(k_pack_input, dim3(blocks_for(nv)), dim3(256), 0, st, in, nv, out);
    SFP_LAUNCH_CHECK();
}

}  // namespace sfp
