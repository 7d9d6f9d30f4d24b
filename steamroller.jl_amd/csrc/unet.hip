// libsrmg, learned coarse-level initial guess.
//
// A U-Net of 3^D convolutions maps the right-hand side f of the level-1
// (uniform, coarsest) problem L_1 u = f to an approximation of u. Activations
// and weights are BF16 and every product runs on the matrix cores
// (v_mfma_f32_16x16x32_bf16, FP32 accumulation). Forward pass, backward pass
// (data and weight gradients) and the Adam update are kernels of this file,
// driven from the host code below; nothing here calls a library GEMM.
//
// Layouts
//   activations  [batch][voxel][channel] BF16 (channels last, x fastest),
//                channels a power of two >= 8, so one lane loads the 8
//                channels of one stencil tap as one 16-byte vector;
//   parameters   FP32, per convolution W[cout][tap][cin] then b[cout], taps
//                ordered t = (dx+1) + 3 (dy+1) + 9 (dz+1);
//   packed       BF16 GEMM operands: forward Wf[cout (16-padded)][tap*cin
//                (32-padded)], data gradient Wb[cin][tap'*cout] with the taps
//                mirrored (the transposed convolution).
//
// Network (levels L, widths w_0..w_{L-1}): per level two ReLU convolutions
// (encoder; 2^D average pooling between levels); per decoder level a linear
// convolution at the coarse level, nearest upsampling added to the encoder
// output of the same level (skip connection) and one ReLU convolution; a last
// linear convolution to one FP32 channel. Input channels: f / max|f|, the
// normalized cell-centre coordinates, zeros. Output: u / (max|f| c_out).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <memory>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/srmg.h"
#include "common.h"
#include "unet.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int TPB = 256;
// convolutions over fewer voxels split their K loop over the waves of a work group
constexpr int64_t SPLITK_NVOX = 65536;
// ... and lower the voxels per work group until there are this many
constexpr int64_t SPLIT_WGS = 1024;
constexpr int MAXLEV = 6;
constexpr int FEAT = 8;  // input channels
constexpr int LOSS_WGS = 1024;

__device__ inline float bf2f(uint32_t b) { return __uint_as_float(b << 16); }
// round to nearest even; NaN stays NaN
__device__ inline uint32_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    if ((u & 0x7f800000u) == 0x7f800000u) return (u >> 16) | ((u & 0xffffu) ? 0x40u : 0u);
    u += 0x7fffu + ((u >> 16) & 1u);
    return u >> 16;
}
__device__ inline bool bf_pos(uint32_t b) { return (b & 0xffffu) != 0 && !(b & 0x8000u); }

__device__ inline void unpack8(uint4 q, float *o) {
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int i = 0; i < 4; i++) {
        o[2 * i] = bf2f(w[i] & 0xffffu);
        o[2 * i + 1] = bf2f(w[i] >> 16);
    }
}
__device__ inline uint4 pack8(const float *o) {
    uint32_t w[4];
#pragma unroll
    for (int i = 0; i < 4; i++) w[i] = f2bf(o[2 * i]) | (f2bf(o[2 * i + 1]) << 16);
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// ---------------------------------------------------------------------------
// convolution as an implicit GEMM on the matrix cores
// ---------------------------------------------------------------------------

// Epilogue of the convolutions: a lane holds D[4 g + j][col], the output
// channels 16 r + 4 g + j of its voxel v in column group q.
template <int R, int OUT, int Q>
__device__ __forceinline__ void conv_store(const f32x4 (&acc)[R][Q], int q, int g, int64_t v,
                                           const float *__restrict__ bias, int nbias, int relu,
                                           const uint16_t *__restrict__ mask, void *__restrict__ out, int cout_s,
                                           int row0 = 0) {
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int co0 = row0 + 16 * r + 4 * g;
        if (co0 >= cout_s) continue;
        float o[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float val = acc[r][q][j];
            if (bias && co0 + j < nbias) val += bias[co0 + j];
            if (relu) val = fmaxf(val, 0.f);
            o[j] = val;
        }
        if constexpr (OUT == 0) {
            if (mask) {
                const uint2 mm = *reinterpret_cast<const uint2 *>(mask + v * cout_s + co0);
                if (!bf_pos(mm.x)) o[0] = 0.f;
                if (!bf_pos(mm.x >> 16)) o[1] = 0.f;
                if (!bf_pos(mm.y)) o[2] = 0.f;
                if (!bf_pos(mm.y >> 16)) o[3] = 0.f;
            }
            uint2 pk;
            pk.x = f2bf(o[0]) | (f2bf(o[1]) << 16);
            pk.y = f2bf(o[2]) | (f2bf(o[3]) << 16);
            *reinterpret_cast<uint2 *>(static_cast<uint16_t *>(out) + v * cout_s + co0) = pk;
        } else {
            if (co0 == 0) static_cast<float *>(out)[v] = o[0];
        }
    }
}

// out[v][co] = act(sum_{t, ci} W[co][t][ci] in[v + off(t)][ci] + bias[co]),
// zero outside the grid. GEMM view: D (cout x voxels) = W (cout x K) *
// Xcol (K x voxels), K = taps * cin. A wave owns 16 R output channels x 64
// voxels (R x 4 accumulators of 16 x 16); one 16x16x32 MFMA consumes, per
// lane, 8 consecutive k (one tap, 8 channels) of one voxel (B) and of one
// output channel (A). The same kernel is the data gradient when given the
// mirrored, transposed weights; `mask` then applies the ReLU derivative of
// the layer that produced the gradient's target (out *= mask > 0).
// OUT 0: BF16 output with cout_s stored channels; OUT 1: FP32, one channel.
// SK > 1 (grids with few voxels, where a launch of one wave per 64 voxels
// leaves the chip idle and each wave walks the whole K loop): the SK waves of
// a work group share 16 Q voxels and take every SK-th 32-wide K step; waves
// 1..SK-1 hand their accumulators to wave 0 through LDS, which adds them in
// wave order before the epilogue. Output channels are split over blockIdx.y
// (16 R per work group) and Q is lowered until the launch has a work group for
// every CU; neither changes a product's place in its sum. A wave's chain of
// dependent loads bounds these launches: U steps' operands are loaded before
// their products. 64 to 64 channels on 8^3: 25 us on 8 work groups, 6 us on
// 128; 32 to 32 on 16^3 14 against 5, 16 to 16 on 32^3 9 against 7.
template <int D, int R, int OUT, int SK = 1, int Q = 4, int U = 1>
__global__ __launch_bounds__(TPB) void k_conv(const uint16_t *__restrict__ in, int cin_log2,
                                              const uint16_t *__restrict__ w, int kp, int ktot,
                                              const float *__restrict__ bias, int nbias, int relu,
                                              const uint16_t *__restrict__ mask, void *__restrict__ out, int cout_s,
                                              int n0, int n1, int n2, int64_t nvox) {
    static_assert(SK == 1 || SK == TPB / 64, "split K over the waves of a work group");
    const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
    const int wv = threadIdx.x >> 6;
    const int row0 = 16 * R * blockIdx.y;
    const int64_t vbase = (SK > 1 ? (int64_t)blockIdx.x : (int64_t)blockIdx.x * (TPB / 64) + wv) * (16 * Q);
    const int64_t V = (int64_t)n0 * n1 * n2;
    int px[Q], py[Q], pz[Q];
    int64_t pn[Q];
    bool ok[Q];
#pragma unroll
    for (int q = 0; q < Q; q++) {
        const int64_t v = vbase + 16 * q + col;
        ok[q] = v < nvox;
        const int64_t nn = ok[q] ? v / V : 0;
        const int r = ok[q] ? (int)(v - nn * V) : 0;
        pn[q] = nn * V;
        px[q] = r % n0;
        py[q] = (r / n0) % n1;
        pz[q] = r / (n0 * n1);
    }
    f32x4 acc[R][Q];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int q = 0; q < Q; q++) acc[r][q] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int cin = 1 << cin_log2;
    auto load_a = [&](int kk, int r) {
        return __builtin_bit_cast(bf16x8,
                                  *reinterpret_cast<const uint4 *>(w + (size_t)(row0 + 16 * r + col) * kp + kk));
    };
    auto load_b = [&](int kk, int q) {
        const int t = kk >> cin_log2, ci = kk & (cin - 1);
        const int dx = t % 3 - 1, dy = (t / 3) % 3 - 1, dz = D == 3 ? t / 9 - 1 : 0;
        const int x = px[q] + dx, y = py[q] + dy, z = pz[q] + dz;
        uint4 val = make_uint4(0u, 0u, 0u, 0u);
        if (ok[q] && kk < ktot && x >= 0 && x < n0 && y >= 0 && y < n1 && z >= 0 && z < n2)
            val = *reinterpret_cast<const uint4 *>(in + (pn[q] + x + (int64_t)n0 * (y + (int64_t)n1 * z)) * cin + ci);
        return __builtin_bit_cast(bf16x8, val);
    };
    const int k0 = SK > 1 ? 32 * wv : 0;
    int kc = k0;
    for (; kc + 32 * SK * (U - 1) < kp; kc += 32 * SK * U) {
        bf16x8 a[U][R], b[U][Q];
#pragma unroll
        for (int i = 0; i < U; i++) {
            const int kk = kc + 32 * SK * i + 8 * g;
#pragma unroll
            for (int r = 0; r < R; r++) a[i][r] = load_a(kk, r);
#pragma unroll
            for (int q = 0; q < Q; q++) b[i][q] = load_b(kk, q);
        }
#pragma unroll
        for (int i = 0; i < U; i++)
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int q = 0; q < Q; q++)
                    acc[r][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i][r], b[i][q], acc[r][q], 0, 0, 0);
    }
    if constexpr (U > 1) {
        for (; kc < kp; kc += 32 * SK) {
            bf16x8 a[R], b[Q];
#pragma unroll
            for (int r = 0; r < R; r++) a[r] = load_a(kc + 8 * g, r);
#pragma unroll
            for (int q = 0; q < Q; q++) b[q] = load_b(kc + 8 * g, q);
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int q = 0; q < Q; q++)
                    acc[r][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r], b[q], acc[r][q], 0, 0, 0);
        }
    }
    if constexpr (SK > 1) {
        __shared__ f32x4 red[SK - 1][R][Q][64];
        if (wv > 0) {
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int q = 0; q < Q; q++) red[wv - 1][r][q][lane] = acc[r][q];
        }
        __syncthreads();
        if (wv > 0) return;
#pragma unroll
        for (int k = 0; k < SK - 1; k++)
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int q = 0; q < Q; q++) acc[r][q] += red[k][r][q][lane];
    }
#pragma unroll
    for (int q = 0; q < Q; q++)
        if (ok[q]) conv_store<R, OUT>(acc, q, g, vbase + 16 * q + col, bias, nbias, relu, mask, out, cout_s, row0);
}

// ---------------------------------------------------------------------------
// tiles of a channels-last grid in LDS
// ---------------------------------------------------------------------------

// TX x TY x TZ voxels and a halo of one, kept as one plane per 8 channels:
// 16 bytes per voxel, so that 16 lanes on 16 consecutive voxels read 256
// contiguous bytes whatever the channel count. The tile shrinks with the
// channel count so that a work group's tile stays under 56 KB.
template <int D, int CIN>
struct ConvTile {
    static constexpr int C8 = CIN / 8;
    static constexpr int TX = D == 3 ? (CIN <= 16 ? 16 : 8) : (CIN <= 16 ? 32 : 16);
    static constexpr int TY = D == 3 ? (CIN == 64 ? 4 : 8) : (CIN == 64 ? 8 : 16);
    static constexpr int TZ = D == 3 ? 4 : 1;
    static constexpr int NV = TX * TY * TZ;
    static constexpr int HX = TX + 2, HY = TY + 2, HZ = D == 3 ? TZ + 2 : 1;
    static constexpr int HV = HX * HY * HZ;
    static constexpr int NTAP = D == 3 ? 27 : 9;
    // plane offset of tap t relative to the tap at the tile's lowest corner
    __device__ static __forceinline__ int tap(int t) {
        const int dx = t % 3, dy = (t / 3) % 3, dz = t / 9;
        return (dz * HY + dy) * HX + dx;
    }
    // halo position (lowest tap) of tile voxel t, x fastest
    __device__ static __forceinline__ int base(int t) {
        return ((t / (TX * TY)) * HY + (t / TX) % TY) * HX + t % TX;
    }
};

// where tile `id` of a batch of grids lies
struct TileAt {
    int64_t n;       // first voxel of its grid
    int x, y, z;     // first voxel of the tile in the grid
};
template <class TL>
__device__ __forceinline__ TileAt tile_at(int id, int n0, int n1, int n2) {
    const int tx = (n0 + TL::TX - 1) / TL::TX, ty = (n1 + TL::TY - 1) / TL::TY, tz = (n2 + TL::TZ - 1) / TL::TZ;
    TileAt a;
    a.x = id % tx * TL::TX;
    id /= tx;
    a.y = id % ty * TL::TY;
    id /= ty;
    a.z = id % tz * TL::TZ;
    a.n = (int64_t)(id / tz) * n0 * n1 * n2;
    return a;
}

// the tile and its halo into the planes xs; zero outside the grid
template <int D, int CIN>
__device__ __forceinline__ void load_tile(uint4 *xs, const uint16_t *__restrict__ in, const TileAt &at, int n0, int n1,
                                          int n2) {
    using TL = ConvTile<D, CIN>;
    constexpr int N = TL::HV * TL::C8, IT = (N + TPB - 1) / TPB;
    uint4 v[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const int i = k * TPB + (int)threadIdx.x, c = i % TL::C8, h = i / TL::C8;
        const int x = at.x + h % TL::HX - 1, y = at.y + (h / TL::HX) % TL::HY - 1;
        const int z = D == 3 ? at.z + h / (TL::HX * TL::HY) - 1 : 0;
        v[k] = make_uint4(0u, 0u, 0u, 0u);
        if (i < N && x >= 0 && x < n0 && y >= 0 && y < n1 && z >= 0 && z < n2)
            v[k] = *reinterpret_cast<const uint4 *>(in + (at.n + x + (int64_t)n0 * (y + (int64_t)n1 * z)) * CIN + 8 * c);
    }
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const int i = k * TPB + (int)threadIdx.x;
        if (i < N) xs[(i % TL::C8) * TL::HV + i / TL::C8] = v[k];
    }
}

// consecutive tiles (which share halos) on one XCD: work group i of n takes
// tile xcd_tile(i, n)
__device__ __forceinline__ int xcd_tile(int i, int n) {
    const int q = n >> 3;
    return i < 8 * q ? (i & 7) * q + (i >> 3) : i;
}

// k_conv on tiles in LDS: the same products in the same order (the same bits),
// with the taps' operands read from the tile instead of gathered once per tap
// from the caches. Taken where K is not split and the weights of a K step fit
// (up to 32 channels): 8 to 8 channels on 16 grids of 64^3 take 82 us against
// 136 us gathered, on one grid 11.5 against 17; bound by the LDS reads and the
// address arithmetic about equally, then by the 134 to 200 MB it moves.
template <int D, int CIN, int R, int OUT>
__global__ __launch_bounds__(TPB) void k_conv_tile(const uint16_t *__restrict__ in, const uint16_t *__restrict__ w,
                                                   int kp, const float *__restrict__ bias, int nbias, int relu,
                                                   const uint16_t *__restrict__ mask, void *__restrict__ out,
                                                   int cout_s, int n0, int n1, int n2) {
    using TL = ConvTile<D, CIN>;
    constexpr int KS = (TL::NTAP * CIN + 31) / 32;  // 32-wide K steps
    constexpr int IT = TL::NV / TPB;                // groups of 64 voxels per wave
    static_assert(IT >= 1, "a tile holds 64 voxels for every wave");
    constexpr bool AREG = KS * R <= 16;             // the weights stay in registers
    __shared__ uint4 xs[TL::C8 * TL::HV + 1];
    const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4, wv = threadIdx.x >> 6;
    const TileAt at = tile_at<TL>(xcd_tile(blockIdx.x, gridDim.x), n0, n1, n2);
    auto load_a = [&](int s, int r) {
        return __builtin_bit_cast(bf16x8,
                                  *reinterpret_cast<const uint4 *>(w + (size_t)(16 * r + col) * kp + 32 * s + 8 * g));
    };
    bf16x8 areg[AREG ? KS : 1][R];
    if constexpr (AREG) {
#pragma unroll
        for (int s = 0; s < KS; s++)
#pragma unroll
            for (int r = 0; r < R; r++) areg[s][r] = load_a(s, r);
    }
    load_tile<D, CIN>(xs, in, at, n0, n1, n2);
    if (threadIdx.x == 0) xs[TL::C8 * TL::HV] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
#pragma unroll
    for (int it = 0; it < IT; it++) {
        int hb[4];
#pragma unroll
        for (int q = 0; q < 4; q++) hb[q] = TL::base(it * TPB + 64 * wv + 16 * q + col);
        f32x4 acc[R][4];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int q = 0; q < 4; q++) acc[r][q] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const int kk = 32 * s + 8 * g, t = kk / CIN, c = (kk % CIN) / 8;
            const bool in_k = t < TL::NTAP;
            const int off = c * TL::HV + TL::tap(t);
            bf16x8 a[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                if constexpr (AREG) a[r] = areg[s][r];
                else a[r] = load_a(s, r);
            }
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const bf16x8 b = __builtin_bit_cast(bf16x8, xs[in_k ? hb[q] + off : TL::C8 * TL::HV]);
#pragma unroll
                for (int r = 0; r < R; r++)
                    acc[r][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[r], b, acc[r][q], 0, 0, 0);
            }
        }
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int t = it * TPB + 64 * wv + 16 * q + col;
            const int x = at.x + t % TL::TX, y = at.y + (t / TL::TX) % TL::TY, z = at.z + t / (TL::TX * TL::TY);
            if (x >= n0 || y >= n1 || z >= n2) continue;
            conv_store<R, OUT>(acc, q, g, at.n + x + (int64_t)n0 * (y + (int64_t)n1 * z), bias, nbias, relu, mask, out,
                               cout_s);
        }
    }
}

// Weight and bias gradient of one convolution over a chunk of voxels:
// partial[chunk][co][k] = sum_v dz[v][co] Xcol[v][k], k < ktot, and the bias
// column k = ktot (Xcol = 1). GEMM view with the voxels as the reduction
// dimension: a wave owns 16 output channels x 4 tiles of 16 k. For grids whose
// z planes are no multiple of 32 voxels; k_wgrad takes the others.
template <int D>
__global__ __launch_bounds__(TPB) void k_wgrad_gather(const uint16_t *__restrict__ dz, int cg, int cout,
                                               const uint16_t *__restrict__ x, int cin_log2, int ktot, int kx,
                                               int n0, int n1, int n2, int64_t nvox, int64_t chunk,
                                               float *__restrict__ partial) {
    const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4;
    const int kt0 = (blockIdx.x * (TPB / 64) + (threadIdx.x >> 6)) * 4;
    if (16 * kt0 >= kx) return;
    const int co = 16 * blockIdx.y + col;
    const int64_t v0 = (int64_t)blockIdx.z * chunk, v1 = min(nvox, v0 + chunk);
    const int64_t V = (int64_t)n0 * n1 * n2;
    const int cin = 1 << cin_log2;
    int kdx[4], kdy[4], kdz[4], kci[4], kmode[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int k = 16 * (kt0 + j) + col;
        const int t = k >> cin_log2;
        kci[j] = k & (cin - 1);
        kdx[j] = t % 3 - 1;
        kdy[j] = (t / 3) % 3 - 1;
        kdz[j] = D == 3 ? t / 9 - 1 : 0;
        kmode[j] = k < ktot ? 1 : (k == ktot ? 2 : 0);
    }
    f32x4 acc[4];
#pragma unroll
    for (int j = 0; j < 4; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // rows of a multiple of 8 voxels: each lane's 8 consecutive voxels lie in
    // one row (chunks start at multiples of 32), so their coordinates are
    // found once per step
    const bool rows8 = (n0 & 7) == 0;
    for (int64_t vs = v0; vs < v1 && rows8; vs += 32) {
        const int64_t vb = vs + 8 * g;
        uint32_t av[8], bv[4][8];
        const bool okv = vb < v1;
        const int64_t nn = okv ? vb / V : 0, r = okv ? vb - nn * V : 0;
        const int rr = (int)r, px0 = rr % n0, py = (rr / n0) % n1, pz = rr / (n0 * n1);
#pragma unroll
        for (int i = 0; i < 8; i++) av[i] = (okv && co < cg) ? dz[(vb + i) * cg + co] : 0u;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int yy = py + kdy[j], zz = pz + kdz[j];
            const bool rowok = okv && kmode[j] == 1 && yy >= 0 && yy < n1 && zz >= 0 && zz < n2;
            const int64_t base = (nn * V + (int64_t)n0 * (yy + (int64_t)n1 * zz)) * cin + kci[j];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int xx = px0 + i + kdx[j];
                uint32_t val = 0u;
                if (okv && kmode[j] == 2) val = 0x3f80u;  // 1.0
                else if (rowok && xx >= 0 && xx < n0) val = x[base + (int64_t)xx * cin];
                bv[j][i] = val;
            }
        }
        const uint4 aq = make_uint4(av[0] | (av[1] << 16), av[2] | (av[3] << 16), av[4] | (av[5] << 16),
                                    av[6] | (av[7] << 16));
        const bf16x8 a = __builtin_bit_cast(bf16x8, aq);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint4 bq = make_uint4(bv[j][0] | (bv[j][1] << 16), bv[j][2] | (bv[j][3] << 16),
                                        bv[j][4] | (bv[j][5] << 16), bv[j][6] | (bv[j][7] << 16));
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, bq), acc[j], 0, 0, 0);
        }
    }
    for (int64_t vs = v0; vs < v1 && !rows8; vs += 32) {
        uint32_t av[8], bv[4][8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int64_t vox = vs + 8 * g + i;
            const bool okv = vox < v1;
            av[i] = (okv && co < cg) ? dz[vox * cg + co] : 0u;
            const int64_t nn = okv ? vox / V : 0, r = okv ? vox - nn * V : 0;
            const int px = (int)(r % n0), py = (int)((r / n0) % n1), pz = (int)(r / ((int64_t)n0 * n1));
#pragma unroll
            for (int j = 0; j < 4; j++) {
                uint32_t val = 0u;
                if (okv) {
                    if (kmode[j] == 2) {
                        val = 0x3f80u;  // 1.0
                    } else if (kmode[j] == 1) {
                        const int xx = px + kdx[j], yy = py + kdy[j], zz = pz + kdz[j];
                        if (xx >= 0 && xx < n0 && yy >= 0 && yy < n1 && zz >= 0 && zz < n2)
                            val = x[(nn * V + xx + (int64_t)n0 * (yy + (int64_t)n1 * zz)) * cin + kci[j]];
                    }
                }
                bv[j][i] = val;
            }
        }
        const uint4 aq = make_uint4(av[0] | (av[1] << 16), av[2] | (av[3] << 16), av[4] | (av[5] << 16),
                                    av[6] | (av[7] << 16));
        const bf16x8 a = __builtin_bit_cast(bf16x8, aq);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const uint4 bq = make_uint4(bv[j][0] | (bv[j][1] << 16), bv[j][2] | (bv[j][3] << 16),
                                        bv[j][4] | (bv[j][5] << 16), bv[j][6] | (bv[j][7] << 16));
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, __builtin_bit_cast(bf16x8, bq), acc[j], 0, 0, 0);
        }
    }
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
            const int coo = 16 * blockIdx.y + 4 * g + jj, k = 16 * (kt0 + j) + col;
            if (coo < cout && k < kx) partial[((int64_t)blockIdx.z * cout + coo) * kx + k] = acc[j][jj];
        }
}

// The same sums in the same order (the same bits) with both operands from LDS.
// They want 8 consecutive voxels of one channel per lane, which channels-last
// memory holds a voxel apart: the LDS transpose reads deliver them (16 lanes
// read 4 voxels x 16 channels, each lane gets 4 voxels of one channel). Every
// lane gives its own address, so a tap is an offset into the staged rows, and
// with 8 channels two taps share one MFMA's 16 columns. A work group takes the
// chunk in runs of at most `tl` voxels inside one z plane: the grid rows of the
// run, one row above and below, in the three planes (two halo columns per row
// stay zero), as one LDS plane of 16 bytes per voxel and 8 channels; the next
// run's rows are loaded into registers while this one is used. The eight waves
// split the columns, the last one takes the bias; 16 output channels per
// blockIdx.y. Bound by the LDS reads (two per MFMA operand) and, with two work
// groups per CU, by their latency: 8 to 8 channels on 16 grids of 64^3 take
// 84 us (k_wgrad_gather: 670 us), 16 to 16 on 32^3 22 us (127 us). Longer
// chunks of cubic tiles took 56 us but moved the sums' rounding.
constexpr int WGT = 512;  // threads
constexpr int WG_LDS = 48 << 10;  // rows and gradients of a run: three work groups per CU
constexpr int WG_RUN = 512;  // voxels of a run at most

// LDS plane size of `rows` rows of n0 voxels with halos, in 16-byte words:
// 4 mod 16, so that the two planes of a transpose read fall on different banks
template <int D>
__host__ __device__ inline int wgrad_plane(int n0, int rows) {
    const int h = (D == 3 ? 3 : 1) * (rows + 2) * (n0 + 2);
    return h + ((20 - h % 16) % 16);
}
template <int D, int CIN>
__host__ __device__ inline size_t wgrad_lds(int n0, int rows, int tl) {
    return ((size_t)wgrad_plane<D>(n0, rows) * (CIN / 8) + 2 * (tl + 4)) * 16 + (size_t)(tl + n0) * 2;
}

template <int D, int CIN>
__global__ __launch_bounds__(WGT) void k_wgrad(const uint16_t *__restrict__ dz, int cg, int cout,
                                               const uint16_t *__restrict__ x, int ktot, int kx, int n0, int n1, int n2,
                                               int64_t nvox, int64_t chunk, int tl, int rows,
                                               float *__restrict__ partial) {
    constexpr int C8 = CIN / 8, NTAP = D == 3 ? 27 : 9, NDZ = D == 3 ? 3 : 1;
    constexpr int NT = (NTAP * CIN + 15) / 16;              // 16-column tiles
    constexpr int NTW = CIN == 8 ? (NT + 6) / 7 : (NT + 7) / 8;  // per wave
    constexpr int IT = WG_LDS / 16 / WGT;                   // 16-byte words per thread of a run's rows
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    extern __shared__ uint4 lds[];
    const int HX = n0 + 2, HP = (rows + 2) * HX, plane = wgrad_plane<D>(n0, rows), zp = tl + 4;
    uint4 *xs = lds, *zs = xs + plane * C8;
    uint16_t *pos = reinterpret_cast<uint16_t *>(zs + 2 * zp);  // run voxel -> its lowest tap in a plane
    const int lane = threadIdx.x & 63, col = lane & 15, g = lane >> 4, wv = threadIdx.x >> 6;
    const int co0 = 16 * blockIdx.y;
    const bool two = co0 + 8 < cg;  // the second plane of dz holds channels
    // this lane's part of a 16-column row: 8 bytes (half), in plane or tap hi
    const int hi = (col >> 1) & 1, half = col & 1, row = col >> 2;
    int off[NTW];
#pragma unroll
    for (int j = 0; j < NTW; j++) {
        const int k = 16 * (wv * NTW + j) + 8 * hi, t = k / CIN, c = (k % CIN) / 8;
        // columns past the last tap are not written
        off[j] = t < NTAP ? c * plane + (t / 9) * HP + (t / 3 % 3) * HX + t % 3 : 0;
    }
    f32x4 acc[NTW], accb = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NTW; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int i = threadIdx.x; i < plane * C8 + 2 * zp; i += WGT) lds[i] = make_uint4(0u, 0u, 0u, 0u);
    for (int i = threadIdx.x; i < tl + n0; i += WGT) pos[i] = (uint16_t)(i / n0 * HX + i % n0);
    const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u));
    auto tr = [&](const uint4 *p) {
        return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (lds_s16x4 *)((__attribute__((address_space(3))) char *)p + 8 * half));
    };
    auto both = [](s16x4 lo, s16x4 hi4) {
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    const int P = n0 * n1, rw = n0 * C8;
    const int64_t v0 = (int64_t)blockIdx.x * chunk, v1 = min(nvox, v0 + chunk);
    // a run: first voxel va, its plane's first voxel vp and z, its offset o in
    // the plane, its length, its first row
    struct Run {
        int64_t va, vp;
        int z, o, len, y0;
    };
    auto run_at = [&](int64_t va) {
        Run r;
        r.va = va;
        const int64_t pl = va / P;
        r.vp = pl * P;
        r.z = (int)(pl % n2);
        r.o = (int)(va - r.vp);
        r.len = (int)min((int64_t)min(tl, P - r.o), v1 - va);
        r.y0 = r.o / n0;
        return r;
    };
    uint4 xv[IT], zv[2];
    auto load = [&](const Run &r) {
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const int i = k * WGT + (int)threadIdx.x, rr = i / rw, e = i - rr * rw;
            const int y = r.y0 - 1 + rr % (rows + 2), z = D == 3 ? r.z - 1 + rr / (rows + 2) : 0;
            xv[k] = make_uint4(0u, 0u, 0u, 0u);
            if (rr < NDZ * (rows + 2) && y >= 0 && y < n1 && z >= 0 && z < n2)
                xv[k] = *reinterpret_cast<const uint4 *>(x + (r.vp + (int64_t)(z - (D == 3 ? r.z : 0)) * P +
                                                              (int64_t)y * n0) * CIN + 8 * e);
        }
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int i = k * WGT + (int)threadIdx.x, t = i >> 1, c = i & 1;
            zv[k] = make_uint4(0u, 0u, 0u, 0u);
            if (t < r.len && (c == 0 || two))
                zv[k] = *reinterpret_cast<const uint4 *>(dz + (r.va + t) * cg + co0 + 8 * c);
        }
    };
    if (v0 < v1) load(run_at(v0));
    for (int64_t va = v0; va < v1;) {
        const Run r = run_at(va);
        __syncthreads();  // the previous run has been used (first: the zeros are written)
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const int i = k * WGT + (int)threadIdx.x, rr = i / rw, e = i - rr * rw;
            if (rr < NDZ * (rows + 2)) xs[(e % C8) * plane + rr * HX + 1 + e / C8] = xv[k];
        }
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int i = k * WGT + (int)threadIdx.x, t = i >> 1, c = i & 1;
            if (t < tl) zs[c * zp + t] = zv[k];
        }
        __syncthreads();
        va += r.len;
        if (va < v1) load(run_at(va));
        const int o = r.o - r.y0 * n0;
        // 32 voxels per step: element 8 g + i of a lane is voxel 8 g + i
#pragma unroll 2
        for (int s = 0; s < r.len; s += 32) {
            const int t0 = s + 8 * g + row, t1 = t0 + 4;
            const bf16x8 a = both(tr(zs + hi * zp + t0), tr(zs + hi * zp + t1));
            const uint4 *x0 = xs + pos[o + t0], *x1 = xs + pos[o + t1];
#pragma unroll
            for (int j = 0; j < NTW; j++)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, both(tr(x0 + off[j]), tr(x1 + off[j])), acc[j], 0, 0,
                                                                 0);
            if (wv == WGT / 64 - 1) accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, ones, accb, 0, 0, 0);
        }
    }
    float *p = partial + (int64_t)blockIdx.x * cout * kx;
#pragma unroll
    for (int j = 0; j < NTW; j++)
#pragma unroll
        for (int jj = 0; jj < 4; jj++) {
            const int co = co0 + 4 * g + jj, k = 16 * (wv * NTW + j) + col;
            if (co < cout && k < ktot) p[(int64_t)co * kx + k] = acc[j][jj];
        }
    if (wv == WGT / 64 - 1 && col == 0)
#pragma unroll
        for (int jj = 0; jj < 4; jj++)
            if (co0 + 4 * g + jj < cout) p[(int64_t)(co0 + 4 * g + jj) * kx + ktot] = accb[jj];
}

// sum of the chunk partials, in chunk order, into the weight and bias
// gradients: a work group takes 32 outputs, its loads of all chunks go to LDS
// together and one thread per output adds them (with 16 loads in flight per
// thread the walk over 512 chunks took 15-39 us)
constexpr int WRED_OUT = 32, MAX_CHUNKS = 512;
__global__ __launch_bounds__(1024) void k_wgrad_reduce(const float *__restrict__ partial, int nchunk, int cout, int kx,
                                                       int ktot, float *__restrict__ gw, float *__restrict__ gb) {
    __shared__ float red[MAX_CHUNKS][WRED_OUT];
    const int o = threadIdx.x % WRED_OUT, part = threadIdx.x / WRED_OUT;
    const int i = blockIdx.x * WRED_OUT + o;
    const int64_t stride = (int64_t)cout * kx;
#pragma unroll
    for (int k = 0; k < MAX_CHUNKS * WRED_OUT / 1024; k++) {
        const int c = k * (1024 / WRED_OUT) + part;
        red[c][o] = (c < nchunk && i < cout * kx) ? partial[c * stride + i] : 0.f;
    }
    __syncthreads();
    if (part || i >= cout * kx) return;
    float s = 0.f;
#pragma unroll 16
    for (int c = 0; c < nchunk; c++) s += red[c][o];
    const int co = i / kx, k = i - co * kx;
    if (k < ktot)
        gw[co * ktot + k] = s;
    else
        gb[co] = s;
}

// ---------------------------------------------------------------------------
// pooling, upsampling, skip connections (8 channels per thread)
// ---------------------------------------------------------------------------

struct Ext {
    int n0, n1, n2;
};

// I: the type of the index arithmetic. 32 bits where the tensor's offsets fit
// (for_index): 64-bit divisions were a third of what pooling and upsampling of
// 64^3 x 8 took: 5.2 -> 3.4 and 4.3 -> 3.7 us, a forward pass 151 -> 146
template <class I>
__device__ inline I vindex(const Ext &e, int x, int y, int z) {
    return x + (I)e.n0 * (y + (I)e.n1 * z);
}
template <class Fn>
void for_index(int64_t values, Fn &&fn) {
    if (values < ((int64_t)1 << 31)) fn((uint32_t)0);
    else fn((int64_t)0);
}

// coarse voxel -> its 2^D children
template <int D, class I>
__global__ __launch_bounds__(TPB) void k_pool(const uint16_t *__restrict__ in, uint16_t *__restrict__ out, int c8,
                                              Ext ec, Ext ef, I total) {
    const I i = (I)blockIdx.x * TPB + threadIdx.x;
    if (i >= total) return;
    const int cg = (int)(i % c8);
    const I vc = i / c8, Vc = (I)ec.n0 * ec.n1 * ec.n2, Vf = (I)ef.n0 * ef.n1 * ef.n2;
    const I n = vc / Vc, r = vc - n * Vc;
    const int xc = (int)(r % ec.n0), yc = (int)((r / ec.n0) % ec.n1), zc = (int)(r / ((I)ec.n0 * ec.n1));
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < (1 << D); c++) {
        const int xf = 2 * xc + (c & 1), yf = 2 * yc + ((c >> 1) & 1), zf = D == 3 ? 2 * zc + (c >> 2) : 0;
        float v[8];
        unpack8(*reinterpret_cast<const uint4 *>(in + ((n * Vf + vindex<I>(ef, xf, yf, zf)) * c8 + cg) * 8), v);
        for (int k = 0; k < 8; k++) acc[k] += v[k];
    }
    for (int k = 0; k < 8; k++) acc[k] *= 1.0f / (1 << D);
    *reinterpret_cast<uint4 *>(out + i * 8) = pack8(acc);
}

// fine voxel: out = coarse(parent) + skip
template <int D, class I>
__global__ __launch_bounds__(TPB) void k_up_add(const uint16_t *__restrict__ coarse, const uint16_t *__restrict__ skip,
                                                uint16_t *__restrict__ out, int c8, Ext ec, Ext ef, I total) {
    const I i = (I)blockIdx.x * TPB + threadIdx.x;
    if (i >= total) return;
    const int cg = (int)(i % c8);
    const I vf = i / c8, Vc = (I)ec.n0 * ec.n1 * ec.n2, Vf = (I)ef.n0 * ef.n1 * ef.n2;
    const I n = vf / Vf, r = vf - n * Vf;
    const int x = (int)(r % ef.n0), y = (int)((r / ef.n0) % ef.n1), z = (int)(r / ((I)ef.n0 * ef.n1));
    float a[8], b[8];
    unpack8(*reinterpret_cast<const uint4 *>(coarse + ((n * Vc + vindex<I>(ec, x >> 1, y >> 1, z >> 1)) * c8 + cg) * 8),
            a);
    unpack8(*reinterpret_cast<const uint4 *>(skip + i * 8), b);
    for (int k = 0; k < 8; k++) a[k] += b[k];
    *reinterpret_cast<uint4 *>(out + i * 8) = pack8(a);
}

// coarse voxel: d coarse = sum of the children's d fine (adjoint of nearest upsampling)
template <int D, class I>
__global__ __launch_bounds__(TPB) void k_up_bwd(const uint16_t *__restrict__ dfine, uint16_t *__restrict__ dcoarse,
                                                int c8, Ext ec, Ext ef, I total) {
    const I i = (I)blockIdx.x * TPB + threadIdx.x;
    if (i >= total) return;
    const int cg = (int)(i % c8);
    const I vc = i / c8, Vc = (I)ec.n0 * ec.n1 * ec.n2, Vf = (I)ef.n0 * ef.n1 * ef.n2;
    const I n = vc / Vc, r = vc - n * Vc;
    const int xc = (int)(r % ec.n0), yc = (int)((r / ec.n0) % ec.n1), zc = (int)(r / ((I)ec.n0 * ec.n1));
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int c = 0; c < (1 << D); c++) {
        const int xf = 2 * xc + (c & 1), yf = 2 * yc + ((c >> 1) & 1), zf = D == 3 ? 2 * zc + (c >> 2) : 0;
        float v[8];
        unpack8(*reinterpret_cast<const uint4 *>(dfine + ((n * Vf + vindex<I>(ef, xf, yf, zf)) * c8 + cg) * 8), v);
        for (int k = 0; k < 8; k++) acc[k] += v[k];
    }
    *reinterpret_cast<uint4 *>(dcoarse + i * 8) = pack8(acc);
}

// fine voxel: d e = (d skip + d pooled(parent) / 2^D) * (e > 0)
template <int D, class I>
__global__ __launch_bounds__(TPB) void k_pool_bwd(const uint16_t *__restrict__ dskip, const uint16_t *__restrict__ dp,
                                                  const uint16_t *__restrict__ e, uint16_t *__restrict__ de, int c8,
                                                  Ext ec, Ext ef, I total) {
    const I i = (I)blockIdx.x * TPB + threadIdx.x;
    if (i >= total) return;
    const int cg = (int)(i % c8);
    const I vf = i / c8, Vc = (I)ec.n0 * ec.n1 * ec.n2, Vf = (I)ef.n0 * ef.n1 * ef.n2;
    const I n = vf / Vf, r = vf - n * Vf;
    const int x = (int)(r % ef.n0), y = (int)((r / ef.n0) % ef.n1), z = (int)(r / ((I)ef.n0 * ef.n1));
    float a[8], b[8];
    unpack8(*reinterpret_cast<const uint4 *>(dskip + i * 8), a);
    unpack8(*reinterpret_cast<const uint4 *>(dp + ((n * Vc + vindex<I>(ec, x >> 1, y >> 1, z >> 1)) * c8 + cg) * 8), b);
    const uint4 m = *reinterpret_cast<const uint4 *>(e + i * 8);
    const uint32_t mw[4] = {m.x, m.y, m.z, m.w};
    for (int k = 0; k < 8; k++) {
        const uint32_t bits = (mw[k >> 1] >> (16 * (k & 1))) & 0xffffu;
        a[k] = bf_pos(bits) ? a[k] + b[k] * (1.0f / (1 << D)) : 0.f;
    }
    *reinterpret_cast<uint4 *>(de + i * 8) = pack8(a);
}

// ---------------------------------------------------------------------------
// input normalization, loss, output, optimizer
// ---------------------------------------------------------------------------

// scale[n] = max |f[n]| (1 for an all-zero grid); one work group per grid
// maximum over the work group (all threads get it)
__device__ __forceinline__ double wg_max(double m) {
    __shared__ double red[TPB];
    red[threadIdx.x] = m;
    __syncthreads();
    for (int s = TPB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    return red[0];
}

// max |f| per grid in two stages: work groups per grid reduce contiguous chunks,
// then one work group per grid reduces the chunk maxima (a maximum does not
// depend on the order: the same value as one pass). One per 1,024 cells, so that a
// large batch of small grids does not launch mostly empty ones (4,096 grids of 4^3
// with 256 each: 400 us of a forward pass); 64^3 takes 4 us in 256, 7 us in 64
constexpr int ABSMAX_PARTS = 256;  // at most
inline int absmax_parts(int64_t V) { return (int)std::min<int64_t>(ABSMAX_PARTS, std::max<int64_t>(1, V / 1024)); }
template <typename TF>
__global__ __launch_bounds__(TPB) void k_absmax_part(const TF *__restrict__ f, int64_t V,
                                                     double *__restrict__ part) {
    const int64_t chunk = (V + gridDim.x - 1) / gridDim.x;
    const TF *p = f + (int64_t)blockIdx.y * V;
    const int64_t i0 = (int64_t)blockIdx.x * chunk, i1 = min(V, i0 + chunk);
    double m = 0.0;
    for (int64_t i = i0 + threadIdx.x; i < i1; i += TPB) m = fmax(m, fabs((double)p[i]));
    m = wg_max(m);
    if (threadIdx.x == 0) part[(int64_t)blockIdx.y * gridDim.x + blockIdx.x] = m;
}

__global__ __launch_bounds__(TPB) void k_absmax(const double *__restrict__ part, int parts,
                                                double *__restrict__ scale) {
    static_assert(ABSMAX_PARTS <= TPB, "a chunk's maximum for each thread");
    const double m = wg_max((int)threadIdx.x < parts ? part[(int64_t)blockIdx.x * parts + threadIdx.x] : 0.0);
    if (threadIdx.x == 0) scale[blockIdx.x] = m > 0.0 ? m : 1.0;
}

template <int D, class I, typename TF>
__global__ __launch_bounds__(TPB) void k_features(const TF *__restrict__ f, const double *__restrict__ scale,
                                                  uint16_t *__restrict__ x, Ext e, I nvox) {
    const I v = (I)blockIdx.x * TPB + threadIdx.x;
    if (v >= nvox) return;
    const I V = (I)e.n0 * e.n1 * e.n2, n = v / V, r = v - n * V;
    const int px = (int)(r % e.n0), py = (int)((r / e.n0) % e.n1), pz = (int)(r / ((I)e.n0 * e.n1));
    float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    o[0] = (float)((double)f[v] / scale[n]);
    o[1] = 2.0f * ((float)px + 0.5f) / (float)e.n0 - 1.0f;
    o[2] = 2.0f * ((float)py + 0.5f) / (float)e.n1 - 1.0f;
    if (D == 3) o[3] = 2.0f * ((float)pz + 0.5f) / (float)e.n2 - 1.0f;
    *reinterpret_cast<uint4 *>(x + v * FEAT) = pack8(o);
}

// d = y - u / (scale c_out); dy[v][0] = 2 d / nvox (other channels 0);
// partial[wg] = sum d^2 over a fixed grid-stride set of voxels
template <typename TU>
__global__ __launch_bounds__(TPB) void k_mse(const float *__restrict__ y, const TU *__restrict__ u,
                                             const double *__restrict__ scale, double c_out, int64_t V, int64_t nvox,
                                             uint16_t *__restrict__ dy, double *__restrict__ partial) {
    __shared__ double red[TPB];
    double acc = 0.0;
    const float gs = (float)(2.0 / (double)nvox);
    for (int64_t v = (int64_t)blockIdx.x * TPB + threadIdx.x; v < nvox; v += (int64_t)gridDim.x * TPB) {
        const double t = (double)u[v] / (scale[v / V] * c_out);
        const double d = (double)y[v] - t;
        acc += d * d;
        *reinterpret_cast<uint4 *>(dy + v * 8) = make_uint4(f2bf(gs * (float)d), 0u, 0u, 0u);
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = TPB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ __launch_bounds__(TPB) void k_loss_total(const double *__restrict__ partial, int n, double inv,
                                                    double *__restrict__ out) {
    __shared__ double red[TPB];
    double acc = 0.0;
    for (int i = threadIdx.x; i < n; i += TPB) acc += partial[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int s = TPB / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = red[0] * inv;
}

template <typename TO>
__global__ __launch_bounds__(TPB) void k_output(const float *__restrict__ y, const double *__restrict__ scale,
                                                double c_out, int64_t V, int64_t nvox, TO *__restrict__ u) {
    const int64_t v = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (v >= nvox) return;
    u[v] = (TO)((double)y[v] * scale[v / V] * c_out);
}

__global__ __launch_bounds__(TPB) void k_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                                              float *__restrict__ v, int64_t n, float lr, float b1, float b2, float eps,
                                              float c1, float c2) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

// Wf[row][k] (rows16 x kp) from W[cout][ktot]
__global__ __launch_bounds__(TPB) void k_pack_fwd(const float *__restrict__ W, int cout, int ktot, int rows16, int kp,
                                                  uint16_t *__restrict__ wf) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= (int64_t)rows16 * kp) return;
    const int r = (int)(i / kp), k = (int)(i - (int64_t)r * kp);
    wf[i] = (uint16_t)((r < cout && k < ktot) ? f2bf(W[(int64_t)r * ktot + k]) : 0u);
}

// Wb[ci][t' cg + co] = W[co][ntap - 1 - t'][ci]: the transposed convolution
__global__ __launch_bounds__(TPB) void k_pack_bwd(const float *__restrict__ W, int cout, int cin, int ntap, int cg,
                                                  int rows16, int kp, uint16_t *__restrict__ wb) {
    const int64_t i = (int64_t)blockIdx.x * TPB + threadIdx.x;
    if (i >= (int64_t)rows16 * kp) return;
    const int ci = (int)(i / kp), kb = (int)(i - (int64_t)ci * kp);
    const int t = kb / cg, co = kb - t * cg;
    uint32_t val = 0u;
    if (ci < cin && t < ntap && co < cout) val = f2bf(W[((int64_t)co * ntap + (ntap - 1 - t)) * cin + ci]);
    wb[i] = (uint16_t)val;
}

inline unsigned nblocks(int64_t n) { return (unsigned)((n + TPB - 1) / TPB); }
inline int ilog2(int x) {
    int l = 0;
    while ((1 << l) < x) l++;
    return l;
}
inline int round_up(int x, int m) { return (x + m - 1) / m * m; }

struct ConvL {
    int level = 0;           // grid level of input and output (0 = full grid)
    int cin = 0, cout = 0;   // channels; cin a power of two >= 8
    int cout_s = 0;          // stored output channels (1: the FP32 output)
    int cg = 0;              // channels of the output gradient (>= 8)
    bool relu = false;
    int ktot = 0, kp = 0, rows = 0;    // forward GEMM
    int ktot_b = 0, kp_b = 0, rows_b = 0;  // data-gradient GEMM
    size_t woff = 0, boff = 0;
    DevBuf wf, wb;
};

struct Tensor {
    int level = 0, c = 0;
    DevBuf v, g;
};

}  // namespace

struct srmg_unet {
    int D = 3, L = 4, ntap = 27;
    Ext ext[MAXLEV];
    int64_t V[MAXLEV];
    std::vector<int> w;
    std::vector<ConvL> conv;
    std::vector<int> cA, cE, cC, cDd;
    int cY = -1;
    size_t nparam = 0;
    DevBuf p, gr, m, v;
    int64_t steps = 0;
    double c_out = 1.0;
    bool has_problem = false;
    int geometry = 0, disc = 0;
    double k2 = 0.0;
    int8_t bc[27] = {0};
    hipStream_t stream = nullptr;
    int cap = 0;
    Tensor X;
    std::vector<Tensor> A, E, P, C, S, Dd;
    DevBuf Y, gY, scale, absmax_part, lossp, loss, partial;
    bool packed = false;
};

namespace {

void alloc_tensor(Tensor &t, int level, int c, int64_t nvox, bool grad) {
    t.level = level;
    t.c = c;
    t.v.alloc((size_t)nvox * c * 2);
    if (grad) t.g.alloc((size_t)nvox * c * 2);
}

void ensure_batch(srmg_unet *n, int B) {
    if (B <= n->cap) return;
    const int L = n->L;
    auto nv = [&](int l) { return (int64_t)B * n->V[l]; };
    alloc_tensor(n->X, 0, FEAT, nv(0), false);
    n->A.resize(L);
    n->E.resize(L);
    n->P.resize(L);
    n->C.resize(L);
    n->S.resize(L);
    n->Dd.resize(L);
    for (int l = 0; l < L; l++) {
        alloc_tensor(n->A[l], l, n->w[l], nv(l), true);
        alloc_tensor(n->E[l], l, n->w[l], nv(l), true);
        if (l > 0) alloc_tensor(n->P[l], l, n->w[l - 1], nv(l), true);
        if (l < L - 1) {
            alloc_tensor(n->C[l], l + 1, n->w[l], nv(l + 1), true);
            alloc_tensor(n->S[l], l, n->w[l], nv(l), true);
            alloc_tensor(n->Dd[l], l, n->w[l], nv(l), true);
        }
    }
    n->Y.alloc((size_t)nv(0) * sizeof(float));
    n->gY.alloc((size_t)nv(0) * 8 * 2);
    n->scale.alloc((size_t)B * sizeof(double));
    n->absmax_part.alloc((size_t)B * ABSMAX_PARTS * sizeof(double));
    n->lossp.alloc(LOSS_WGS * sizeof(double));
    n->loss.alloc(sizeof(double));
    n->cap = B;
}

void pack(srmg_unet *n, hipStream_t st) {
    for (ConvL &cv : n->conv) {
        const float *W = n->p.as<float>() + cv.woff;
        hipLaunchKernelGGL(k_pack_fwd, dim3(nblocks((int64_t)cv.rows * 16 * cv.kp)), dim3(TPB), 0, st, W, cv.cout,
                           cv.ktot, cv.rows * 16, cv.kp, cv.wf.as<uint16_t>());
        hipLaunchKernelGGL(k_pack_bwd, dim3(nblocks((int64_t)cv.rows_b * 16 * cv.kp_b)), dim3(TPB), 0, st, W, cv.cout,
                           cv.cin, n->ntap, cv.cg, cv.rows_b * 16, cv.kp_b, cv.wb.as<uint16_t>());
    }
    n->packed = true;
}

// tiles of every grid of a batch
template <class TL>
int64_t tile_count(const Ext &e, int64_t nvox) {
    const int64_t per = (int64_t)((e.n0 + TL::TX - 1) / TL::TX) * ((e.n1 + TL::TY - 1) / TL::TY) *
                        ((e.n2 + TL::TZ - 1) / TL::TZ);
    return per * (nvox / ((int64_t)e.n0 * e.n1 * e.n2));
}

// k_conv_tile where at least 45% of its tiles' voxels are the grid's: a tile costs
// what it costs when full. A forward pass on two levels of 2^18 voxels (2D: 2^17),
// gathered / tiles, 16 channels: 4^3 grids (12% of the tiles) 658 / 799 us, 18 x 10
// x 6 (26%) 178 / 222, 2D 18^2 (32%) 140 / 148; 20 x 12 x 28 (47%) 156 / 154, 2D 16^2
// (50%) 155 / 149, 12^3 (56%) 168 / 158, 24^3 (75%) 147 / 118; 32 channels: 18 x 10
// x 6 (35%) 288 / 298, 6^3 (42%) 424 / 426, 12^3 (56%) 281 / 233.
template <class TL>
bool tile_fits(const Ext &e) {
    const int64_t V = (int64_t)e.n0 * e.n1 * e.n2;
    return 100 * V >= 45 * tile_count<TL>(e, V) * TL::NV;
}

template <int D, int OUT>
void conv_launch_r(int R, unsigned grid, hipStream_t st, const uint16_t *in, int cin_log2, const uint16_t *w, int kp,
                   int ktot, const float *bias, int nbias, int relu, const uint16_t *mask, void *out, int cout_s,
                   const Ext &e, int64_t nvox) {
    const bool split = nvox < SPLITK_NVOX;
    if (split) {
        // 64, 32 or 16 voxels and 16 output channels per work group
        auto go = [&](auto q) {
            constexpr int Q = decltype(q)::value;
            hipLaunchKernelGGL((k_conv<D, 1, OUT, TPB / 64, Q, 4>), dim3((unsigned)((nvox + 16 * Q - 1) / (16 * Q)), R),
                               dim3(TPB), 0, st, in, cin_log2, w, kp, ktot, bias, nbias, relu, mask, out, cout_s, e.n0,
                               e.n1, e.n2, nvox);
        };
        const int64_t wgs = (nvox + 63) / 64 * R;
        if (wgs >= SPLIT_WGS) go(std::integral_constant<int, 4>());
        else if (2 * wgs >= SPLIT_WGS) go(std::integral_constant<int, 2>());
        else go(std::integral_constant<int, 1>());
        return;
    }
#define SRMG_TILE(CC, RR)                                                                                          \
    if (cin_log2 == ilog2(CC) && R == RR && tile_fits<ConvTile<D, CC>>(e)) {                             \
        hipLaunchKernelGGL((k_conv_tile<D, CC, RR, OUT>), dim3((unsigned)tile_count<ConvTile<D, CC>>(e, nvox)),    \
                           dim3(TPB), 0, st, in, w, kp, bias, nbias, relu, mask, out, cout_s, e.n0, e.n1, e.n2);   \
        return;                                                                                                    \
    }
    SRMG_TILE(8, 1)
    SRMG_TILE(16, 1)
    SRMG_TILE(32, 1)
    if constexpr (OUT == 0) {
        SRMG_TILE(8, 2)
        SRMG_TILE(16, 2)
        SRMG_TILE(32, 2)
    }
#undef SRMG_TILE
#define SRMG_CONV(RR)                                                                                          \
    hipLaunchKernelGGL((k_conv<D, RR, OUT>), dim3(grid), dim3(TPB), 0, st, in, cin_log2, w, kp, ktot, bias,    \
                       nbias, relu, mask, out, cout_s, e.n0, e.n1, e.n2, nvox)
    if (R == 1)
        SRMG_CONV(1);
    else if (R == 2)
        SRMG_CONV(2);
    else if (R == 4)
        SRMG_CONV(4);
    else
        fail("unsupported channel count");
#undef SRMG_CONV
}

template <int D>
void conv_fwd(srmg_unet *n, hipStream_t st, const ConvL &cv, const uint16_t *in, void *out, int B) {
    const int64_t nvox = (int64_t)B * n->V[cv.level];
    const unsigned grid = (unsigned)((nvox + TPB - 1) / TPB);
    const float *bias = n->p.as<float>() + cv.boff;
    if (cv.cout_s == 1)
        conv_launch_r<D, 1>(cv.rows, grid, st, in, ilog2(cv.cin), cv.wf.as<uint16_t>(), cv.kp, cv.ktot, bias, cv.cout,
                            0, nullptr, out, 1, n->ext[cv.level], nvox);
    else
        conv_launch_r<D, 0>(cv.rows, grid, st, in, ilog2(cv.cin), cv.wf.as<uint16_t>(), cv.kp, cv.ktot, bias, cv.cout,
                            cv.relu ? 1 : 0, nullptr, out, cv.cout_s, n->ext[cv.level], nvox);
}

// gradient w.r.t. the convolution's input from the gradient dz of its output
template <int D>
void conv_bwd_data(srmg_unet *n, hipStream_t st, const ConvL &cv, const uint16_t *dz, uint16_t *din,
                   const uint16_t *mask, int B) {
    const int64_t nvox = (int64_t)B * n->V[cv.level];
    const unsigned grid = (unsigned)((nvox + TPB - 1) / TPB);
    conv_launch_r<D, 0>(cv.rows_b, grid, st, dz, ilog2(cv.cg), cv.wb.as<uint16_t>(), cv.kp_b, cv.ktot_b, nullptr, 0,
                        0, mask, din, cv.cin, n->ext[cv.level], nvox);
}

template <int D, int CIN>
bool wgrad_rows(const ConvL &cv, hipStream_t st, const uint16_t *dz, const uint16_t *x, const Ext &e, int64_t nvox,
                int64_t chunk, unsigned nchunk, float *partial) {
    // runs of whole 32-voxel steps inside a z plane; as long as their rows fit
    if ((int64_t)e.n0 * e.n1 % 32) return false;
    int tl = WG_RUN, rows = 0;
    size_t need = 0;
    for (;; tl /= 2) {
        if (tl < 32) return false;
        const bool aligned = tl % e.n0 == 0 && chunk % e.n0 == 0;
        rows = std::min(aligned ? tl / e.n0 : (tl + e.n0 - 2) / e.n0 + 1, e.n1);
        need = wgrad_lds<D, CIN>(e.n0, rows, tl);
        if (need <= (size_t)WG_LDS) break;
    }
    hipLaunchKernelGGL((k_wgrad<D, CIN>), dim3(nchunk, (unsigned)((cv.cout + 15) / 16)), dim3(WGT), need, st, dz, cv.cg, cv.cout, x, cv.ktot, cv.ktot + 1, e.n0, e.n1,
                       e.n2, nvox, chunk, tl, rows, partial);
    return true;
}

template <int D>
void conv_bwd_weights(srmg_unet *n, hipStream_t st, const ConvL &cv, const uint16_t *dz, const uint16_t *x, int B) {
    const int64_t nvox = (int64_t)B * n->V[cv.level];
    const int kx = cv.ktot + 1;
    int64_t nchunk = std::min<int64_t>(MAX_CHUNKS, (nvox + 255) / 256);
    int64_t chunk = (nvox + nchunk - 1) / nchunk;
    chunk = (chunk + 31) / 32 * 32;
    nchunk = (nvox + chunk - 1) / chunk;
    const size_t need = (size_t)nchunk * cv.cout * kx * sizeof(float);
    if (n->partial.bytes < need) n->partial.alloc(need);
    const Ext &e = n->ext[cv.level];
    float *part = n->partial.as<float>();
    const unsigned nc = (unsigned)nchunk;
    const bool done = cv.cin == 8    ? wgrad_rows<D, 8>(cv, st, dz, x, e, nvox, chunk, nc, part)
                      : cv.cin == 16 ? wgrad_rows<D, 16>(cv, st, dz, x, e, nvox, chunk, nc, part)
                      : cv.cin == 32 ? wgrad_rows<D, 32>(cv, st, dz, x, e, nvox, chunk, nc, part)
                      : cv.cin == 64 ? wgrad_rows<D, 64>(cv, st, dz, x, e, nvox, chunk, nc, part)
                                     : false;
    if (!done) {
        dim3 grid((unsigned)((kx + 255) / 256), (unsigned)((cv.cout + 15) / 16), nc);
        hipLaunchKernelGGL((k_wgrad_gather<D>), grid, dim3(TPB), 0, st, dz, cv.cg, cv.cout, x, ilog2(cv.cin), cv.ktot,
                           kx, e.n0, e.n1, e.n2, nvox, chunk, part);
    }
    hipLaunchKernelGGL(k_wgrad_reduce, dim3((unsigned)((cv.cout * kx + WRED_OUT - 1) / WRED_OUT)), dim3(1024), 0, st,
                       part, (int)nchunk, cv.cout, kx, cv.ktot, n->gr.as<float>() + cv.woff,
                       n->gr.as<float>() + cv.boff);
}

template <int D>
void forward(srmg_unet *n, hipStream_t st, int B) {
    const int L = n->L;
    for (int l = 0; l < L; l++) {
        const uint16_t *in;
        if (l == 0) {
            in = n->X.v.as<uint16_t>();
        } else {
            const int64_t total = (int64_t)B * n->V[l] * (n->w[l - 1] / 8);
            for_index(8 * total << D, [&](auto ix) {
                using I = decltype(ix);
                hipLaunchKernelGGL((k_pool<D, I>), dim3(nblocks(total)), dim3(TPB), 0, st, n->E[l - 1].v.as<uint16_t>(),
                                   n->P[l].v.as<uint16_t>(), n->w[l - 1] / 8, n->ext[l], n->ext[l - 1], (I)total);
            });
            in = n->P[l].v.as<uint16_t>();
        }
        conv_fwd<D>(n, st, n->conv[n->cA[l]], in, n->A[l].v.p, B);
        conv_fwd<D>(n, st, n->conv[n->cE[l]], n->A[l].v.as<uint16_t>(), n->E[l].v.p, B);
    }
    for (int l = L - 2; l >= 0; l--) {
        const uint16_t *src = (l == L - 2) ? n->E[L - 1].v.as<uint16_t>() : n->Dd[l + 1].v.as<uint16_t>();
        conv_fwd<D>(n, st, n->conv[n->cC[l]], src, n->C[l].v.p, B);
        const int64_t total = (int64_t)B * n->V[l] * (n->w[l] / 8);
        for_index(8 * total, [&](auto ix) {
            using I = decltype(ix);
            hipLaunchKernelGGL((k_up_add<D, I>), dim3(nblocks(total)), dim3(TPB), 0, st, n->C[l].v.as<uint16_t>(),
                               n->E[l].v.as<uint16_t>(), n->S[l].v.as<uint16_t>(), n->w[l] / 8, n->ext[l + 1], n->ext[l],
                               (I)total);
        });
        conv_fwd<D>(n, st, n->conv[n->cDd[l]], n->S[l].v.as<uint16_t>(), n->Dd[l].v.p, B);
    }
    conv_fwd<D>(n, st, n->conv[n->cY], n->Dd[0].v.as<uint16_t>(), n->Y.p, B);
}

template <int D>
void backward(srmg_unet *n, hipStream_t st, int B) {
    const int L = n->L;
    auto g16 = [](Tensor &t) { return t.g.as<uint16_t>(); };
    auto v16 = [](Tensor &t) { return t.v.as<uint16_t>(); };
    {
        const ConvL &cv = n->conv[n->cY];
        conv_bwd_weights<D>(n, st, cv, n->gY.as<uint16_t>(), v16(n->Dd[0]), B);
        conv_bwd_data<D>(n, st, cv, n->gY.as<uint16_t>(), g16(n->Dd[0]), v16(n->Dd[0]), B);
    }
    for (int l = 0; l <= L - 2; l++) {
        const ConvL &cd = n->conv[n->cDd[l]];
        conv_bwd_weights<D>(n, st, cd, g16(n->Dd[l]), v16(n->S[l]), B);
        conv_bwd_data<D>(n, st, cd, g16(n->Dd[l]), g16(n->S[l]), nullptr, B);
        const int64_t total = (int64_t)B * n->V[l + 1] * (n->w[l] / 8);
        for_index(8 * total << D, [&](auto ix) {
            using I = decltype(ix);
            hipLaunchKernelGGL((k_up_bwd<D, I>), dim3(nblocks(total)), dim3(TPB), 0, st, g16(n->S[l]), g16(n->C[l]),
                               n->w[l] / 8, n->ext[l + 1], n->ext[l], (I)total);
        });
        const ConvL &cc = n->conv[n->cC[l]];
        Tensor &src = (l == L - 2) ? n->E[L - 1] : n->Dd[l + 1];
        conv_bwd_weights<D>(n, st, cc, g16(n->C[l]), v16(src), B);
        conv_bwd_data<D>(n, st, cc, g16(n->C[l]), g16(src), v16(src), B);
    }
    for (int l = L - 1; l >= 0; l--) {
        const ConvL &ce = n->conv[n->cE[l]];
        conv_bwd_weights<D>(n, st, ce, g16(n->E[l]), v16(n->A[l]), B);
        conv_bwd_data<D>(n, st, ce, g16(n->E[l]), g16(n->A[l]), v16(n->A[l]), B);
        const ConvL &ca = n->conv[n->cA[l]];
        const uint16_t *in = (l == 0) ? n->X.v.as<uint16_t>() : v16(n->P[l]);
        conv_bwd_weights<D>(n, st, ca, g16(n->A[l]), in, B);
        if (l > 0) {
            conv_bwd_data<D>(n, st, ca, g16(n->A[l]), g16(n->P[l]), nullptr, B);
            const int64_t total = (int64_t)B * n->V[l - 1] * (n->w[l - 1] / 8);
            for_index(8 * total, [&](auto ix) {
                using I = decltype(ix);
                hipLaunchKernelGGL((k_pool_bwd<D, I>), dim3(nblocks(total)), dim3(TPB), 0, st, g16(n->S[l - 1]),
                                   g16(n->P[l]), v16(n->E[l - 1]), g16(n->E[l - 1]), n->w[l - 1] / 8, n->ext[l],
                                   n->ext[l - 1], (I)total);
            });
        }
    }
}

template <typename TF>
void features(srmg_unet *n, hipStream_t st, const TF *f, int B) {
    const int parts = absmax_parts(n->V[0]);
    hipLaunchKernelGGL((k_absmax_part<TF>), dim3(parts, B), dim3(TPB), 0, st, f, n->V[0],
                       n->absmax_part.as<double>());
    hipLaunchKernelGGL(k_absmax, dim3(B), dim3(TPB), 0, st, n->absmax_part.as<double>(), parts,
                       n->scale.as<double>());
    const int64_t nvox = (int64_t)B * n->V[0];
    for_index(nvox * FEAT, [&](auto ix) {
        using I = decltype(ix);
        const auto go = [&](auto k) {
            hipLaunchKernelGGL(k, dim3(nblocks(nvox)), dim3(TPB), 0, st, f, n->scale.as<double>(),
                               n->X.v.as<uint16_t>(), n->ext[0], (I)nvox);
        };
        if (n->D == 3) go(k_features<3, I, TF>);
        else go(k_features<2, I, TF>);
    });
}

void run_forward(srmg_unet *n, hipStream_t st, int B) {
    if (!n->packed) pack(n, st);
    if (n->D == 3)
        forward<3>(n, st, B);
    else
        forward<2>(n, st, B);
}

// loss and gradient of one batch into n->gr (and n->loss)
void loss_grad(srmg_unet *n, const float *f, const float *u, int B) {
    hipStream_t st = n->stream;
    ensure_batch(n, B);
    features<float>(n, st, f, B);
    run_forward(n, st, B);
    const int64_t nvox = (int64_t)B * n->V[0];
    hipLaunchKernelGGL(k_mse<float>, dim3(LOSS_WGS), dim3(TPB), 0, st, n->Y.as<float>(), u, n->scale.as<double>(),
                       n->c_out, n->V[0], nvox, n->gY.as<uint16_t>(), n->lossp.as<double>());
    hipLaunchKernelGGL(k_loss_total, dim3(1), dim3(TPB), 0, st, n->lossp.as<double>(), LOSS_WGS, 1.0 / (double)nvox,
                       n->loss.as<double>());
    if (n->D == 3)
        backward<3>(n, st, B);
    else
        backward<2>(n, st, B);
}

// splitmix64 + Box-Muller: reproducible He-normal initialization
struct Rng {
    uint64_t s;
    uint64_t next() {
        uint64_t z = (s += 0x9e3779b97f4a7c15ull);
        z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
        z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
        return z ^ (z >> 31);
    }
    double uniform() { return ((next() >> 11) + 0.5) * (1.0 / 9007199254740992.0); }
    double normal() { return std::sqrt(-2.0 * std::log(uniform())) * std::cos(6.283185307179586 * uniform()); }
};

srmg_unet *checked(srmg_unet *n) {
    if (!n) fail("null network");
    return n;
}

void check_batch(const srmg_unet *n, int B) {
    if (B < 1) fail("batch must be >= 1");
    if ((int64_t)B * n->V[0] > (int64_t)1 << 31) fail("batch too large for one launch");
}

}  // namespace

namespace srmg_guess {

void extents(const srmg_unet *net, int *D, int n[3]) {
    *D = net->D;
    n[0] = net->ext[0].n0;
    n[1] = net->ext[0].n1;
    n[2] = net->ext[0].n2;
}

bool matches(const srmg_unet *net, int geometry, int disc, double k2, const int8_t bc[27]) {
    return net->has_problem && net->geometry == geometry && net->disc == disc && net->k2 == k2 &&
           std::memcmp(net->bc, bc, 27) == 0;
}

void infer(srmg_unet *n, const double *f, double *u, int ngrid, hipStream_t st) {
    check_batch(n, ngrid);
    ensure_batch(n, ngrid);
    features<double>(n, st, f, ngrid);
    run_forward(n, st, ngrid);
    const int64_t nvox = (int64_t)ngrid * n->V[0];
    hipLaunchKernelGGL(k_output<double>, dim3(nblocks(nvox)), dim3(TPB), 0, st, n->Y.as<float>(),
                       n->scale.as<double>(), n->c_out, n->V[0], nvox, u);
}

}  // namespace srmg_guess

extern "C" {

int srmg_unet_create(srmg_unet **out, int D, const int *n, int levels, const int *widths, uint64_t seed) {
    return guarded([&] {
        if (!out || !n || !widths) fail("null argument");
        if (D != 2 && D != 3) fail("D must be 2 or 3");
        if (levels < 2 || levels > MAXLEV) fail("levels must be in 2.." + std::to_string(MAXLEV));
        for (int l = 0; l < levels; l++) {
            const int w = widths[l];
            if (w < 8 || w > 64 || (w & (w - 1))) fail("widths must be powers of two in 8..64");
        }
        for (int d = 0; d < D; d++)
            if (n[d] < 1 || n[d] % (1 << (levels - 1))) fail("grid extents must be divisible by 2^(levels-1)");
        auto net = std::make_unique<srmg_unet>();
        net->D = D;
        net->L = levels;
        net->ntap = D == 3 ? 27 : 9;
        net->w.assign(widths, widths + levels);
        for (int l = 0; l < levels; l++) {
            net->ext[l] = Ext{n[0] >> l, n[1] >> l, D == 3 ? (n[2] >> l) : 1};
            net->V[l] = (int64_t)net->ext[l].n0 * net->ext[l].n1 * net->ext[l].n2;
        }
        auto add = [&](int level, int cin, int cout, bool relu) {
            ConvL cv;
            cv.level = level;
            cv.cin = cin;
            cv.cout = cout;
            cv.cout_s = cout == 1 ? 1 : cout;
            cv.cg = std::max(cout, 8);
            cv.relu = relu;
            cv.ktot = net->ntap * cin;
            cv.kp = round_up(cv.ktot, 32);
            cv.rows = (cout + 15) / 16;
            if (cv.rows == 3) cv.rows = 4;
            cv.ktot_b = net->ntap * cv.cg;
            cv.kp_b = round_up(cv.ktot_b, 32);
            cv.rows_b = (cin + 15) / 16;
            if (cv.rows_b == 3) cv.rows_b = 4;
            cv.woff = net->nparam;
            net->nparam += (size_t)cout * cv.ktot;
            cv.boff = net->nparam;
            net->nparam += cout;
            net->conv.push_back(std::move(cv));
            return (int)net->conv.size() - 1;
        };
        net->cA.resize(levels);
        net->cE.resize(levels);
        net->cC.assign(levels, -1);
        net->cDd.assign(levels, -1);
        for (int l = 0; l < levels; l++) {
            net->cA[l] = add(l, l == 0 ? FEAT : widths[l - 1], widths[l], true);
            net->cE[l] = add(l, widths[l], widths[l], true);
        }
        for (int l = levels - 2; l >= 0; l--) {
            net->cC[l] = add(l + 1, widths[l + 1], widths[l], false);
            net->cDd[l] = add(l, widths[l], widths[l], true);
        }
        net->cY = add(0, widths[0], 1, false);
        for (ConvL &cv : net->conv) {
            cv.wf.alloc((size_t)cv.rows * 16 * cv.kp * 2);
            cv.wb.alloc((size_t)cv.rows_b * 16 * cv.kp_b * 2);
        }
        std::vector<float> h(net->nparam, 0.f);
        Rng rng{seed};
        for (const ConvL &cv : net->conv) {
            const double sd = std::sqrt((cv.relu ? 2.0 : 1.0) / (double)cv.ktot);
            for (size_t i = 0; i < (size_t)cv.cout * cv.ktot; i++) h[cv.woff + i] = (float)(sd * rng.normal());
        }
        net->p.alloc(net->nparam * sizeof(float));
        net->gr.alloc(net->nparam * sizeof(float));
        net->m.alloc(net->nparam * sizeof(float));
        net->v.alloc(net->nparam * sizeof(float));
        HIPCHK(hipStreamCreate(&net->stream));
        HIPCHK(hipMemcpy(net->p.p, h.data(), net->nparam * sizeof(float), hipMemcpyHostToDevice));
        HIPCHK(hipMemset(net->m.p, 0, net->nparam * sizeof(float)));
        HIPCHK(hipMemset(net->v.p, 0, net->nparam * sizeof(float)));
        HIPCHK(hipMemset(net->gr.p, 0, net->nparam * sizeof(float)));
        *out = net.release();
    });
}

int srmg_unet_destroy(srmg_unet *n) {
    return guarded([&] {
        if (!n) return;
        if (n->stream) (void)hipStreamSynchronize(n->stream);
        hipStream_t s = n->stream;
        delete n;
        if (s) (void)hipStreamDestroy(s);
    });
}

int srmg_unet_param_count(const srmg_unet *n, int64_t *count) {
    return guarded([&] {
        if (!n || !count) fail("null argument");
        *count = (int64_t)n->nparam;
    });
}

int srmg_unet_get_params(srmg_unet *n, float *host) {
    return guarded([&] {
        checked(n);
        if (!host) fail("null argument");
        HIPCHK(hipStreamSynchronize(n->stream));
        HIPCHK(hipMemcpy(host, n->p.p, n->nparam * sizeof(float), hipMemcpyDeviceToHost));
    });
}

int srmg_unet_set_params(srmg_unet *n, const float *host) {
    return guarded([&] {
        checked(n);
        if (!host) fail("null argument");
        HIPCHK(hipStreamSynchronize(n->stream));
        HIPCHK(hipMemcpy(n->p.p, host, n->nparam * sizeof(float), hipMemcpyHostToDevice));
        HIPCHK(hipMemset(n->m.p, 0, n->nparam * sizeof(float)));
        HIPCHK(hipMemset(n->v.p, 0, n->nparam * sizeof(float)));
        n->steps = 0;
        n->packed = false;
    });
}

int srmg_unet_set_output_scale(srmg_unet *n, double c_out) {
    return guarded([&] {
        checked(n);
        if (!(c_out > 0.0) || !std::isfinite(c_out)) fail("output scale must be positive and finite");
        n->c_out = c_out;
    });
}

int srmg_unet_get_output_scale(const srmg_unet *n, double *c_out) {
    return guarded([&] {
        if (!n || !c_out) fail("null argument");
        *c_out = n->c_out;
    });
}

int srmg_unet_set_problem(srmg_unet *n, const srmg_op *op) {
    return guarded([&] {
        checked(n);
        if (!op) fail("null operator");
        n->has_problem = true;
        n->geometry = op->geometry;
        n->disc = op->disc;
        n->k2 = op->disc ? op->k2 : 0.0;
        std::memcpy(n->bc, op->bc, 27);
    });
}

int srmg_unet_forward(srmg_unet *n, const float *f, float *u, int batch) {
    return guarded([&] {
        checked(n);
        if (!f || !u) fail("null argument");
        check_batch(n, batch);
        ensure_batch(n, batch);
        features<float>(n, n->stream, f, batch);
        run_forward(n, n->stream, batch);
        const int64_t nvox = (int64_t)batch * n->V[0];
        hipLaunchKernelGGL(k_output<float>, dim3(nblocks(nvox)), dim3(TPB), 0, n->stream, n->Y.as<float>(),
                           n->scale.as<double>(), n->c_out, n->V[0], nvox, u);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(n->stream));
    });
}

int srmg_unet_loss_grad(srmg_unet *n, const float *f, const float *u, int batch, double *loss, float *grad) {
    return guarded([&] {
        checked(n);
        if (!f || !u) fail("null argument");
        check_batch(n, batch);
        if (!n->packed) pack(n, n->stream);
        loss_grad(n, f, u, batch);
        HIPCHK(hipGetLastError());
        HIPCHK(hipStreamSynchronize(n->stream));
        if (loss) HIPCHK(hipMemcpy(loss, n->loss.p, sizeof(double), hipMemcpyDeviceToHost));
        if (grad) HIPCHK(hipMemcpy(grad, n->gr.p, n->nparam * sizeof(float), hipMemcpyDeviceToHost));
    });
}

int srmg_unet_train_step(srmg_unet *n, const float *f, const float *u, int batch, float lr, double *loss) {
    return guarded([&] {
        checked(n);
        if (!f || !u) fail("null argument");
        check_batch(n, batch);
        if (!(lr > 0.f)) fail("learning rate must be positive");
        if (!n->packed) pack(n, n->stream);
        loss_grad(n, f, u, batch);
        n->steps++;
        const float b1 = 0.9f, b2 = 0.999f;
        const float c1 = 1.f - std::pow(b1, (float)n->steps), c2 = 1.f - std::pow(b2, (float)n->steps);
        hipLaunchKernelGGL(k_adam, dim3(nblocks((int64_t)n->nparam)), dim3(TPB), 0, n->stream, n->p.as<float>(),
                           n->gr.as<float>(), n->m.as<float>(), n->v.as<float>(), (int64_t)n->nparam, lr, b1, b2,
                           1e-8f, c1, c2);
        pack(n, n->stream);
        HIPCHK(hipGetLastError());
        if (loss) {
            HIPCHK(hipMemcpyAsync(loss, n->loss.p, sizeof(double), hipMemcpyDeviceToHost, n->stream));
            HIPCHK(hipStreamSynchronize(n->stream));
        }
    });
}

int srmg_unet_synchronize(srmg_unet *n) {
    return guarded([&] {
        checked(n);
        HIPCHK(hipStreamSynchronize(n->stream));
    });
}

}  // extern "C"
