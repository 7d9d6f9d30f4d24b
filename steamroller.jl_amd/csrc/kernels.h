// HIP kernels of the multigrid path (gfx950). Every kernel is templated on the
// dimension D, the block side M and the element type T (double or float).
//
// Floating point: this translation unit is compiled with -ffp-contract=off so
// that products and sums round exactly as written; fma() appears only where the
// reference writes muladd (src/multigrid.jl:176-177). Stencil terms are summed
// in the order the reference's @stencil macro emits them (src/laplacian.jl:25-49),
// so the FP64 kernels reproduce the CPU restatement bit for bit.
#pragma once

#include <hip/hip_runtime.h>

#include "layout.h"

namespace srmg {

constexpr int WG = 256;  // work-group size of the elementwise/stencil kernels

template <typename T>
struct LevelArgs {
    int blk0;      // first device block of the level
    int nblk;      // blocks in the level
    T s;           // s_l = s / 4^(l-1)
    T cc;          // stencil centre = diagelm: -2D, or -2D - s_l k2 (Helmholtz)
    T nwc;         // -(omega / diagelm)
    T sg[6];       // ghost = sg[face] * mirror cell (GeneralHomogeneousBoundaryConditions)
    int rdim;      // radial dimension (cylindrical) or -1
    const T *wm;   // (2J-2)/(2J-1) by 1-based global radial index J at this level
    const T *wp;   // 2J/(2J-1)
    // several problems in one launch: (s, cc, nwc) of block blk are
    // pp[3 blk + 0..2] (one load; through a per-block problem index it was two
    // in a row); nullptr when the context holds one problem
    const T *pp;
    // processing order of the level's sibling groups in the column sweeps:
    // work group slot i takes group gord[i]; nullptr: group i
    const int *gord;
};

template <typename T>
struct BP {
    T s, cc, nwc;
};

template <typename T>
__device__ __forceinline__ BP<T> bparams(const LevelArgs<T> &a, int blk) {
    if (a.pp) {
        const T *q = a.pp + 3 * (size_t)blk;
        return {q[0], q[1], q[2]};
    }
    return {a.s, a.cc, a.nwc};
}

template <typename T> __device__ __forceinline__ T fma_t(T a, T b, T c);
template <> __device__ __forceinline__ double fma_t<double>(double a, double b, double c) { return fma(a, b, c); }
template <> __device__ __forceinline__ float fma_t<float>(float a, float b, float c) { return fmaf(a, b, c); }

// f(integral_constant<int, i>) for i = 0 .. N-1, unrolled at compile time
template <int N, int I = 0, class Fn>
__device__ __forceinline__ void static_for(Fn &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>());
        static_for<N, I + 1>(f);
    }
}

// Work-group barrier that orders LDS accesses only: global loads still in
// flight stay in flight across it (__syncthreads would wait for them).
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// a field formed from two while it is read
template <typename T>
struct Diff {
    const T *__restrict__ a, *__restrict__ b;
    __device__ __forceinline__ T operator[](size_t i) const { return a[i] - b[i]; }
};

// Value of cell (c0,c1,c2) + dir e_dim of block blk, crossing the block face if
// needed: same-level neighbour cell, mirror (depth-1 ghost = sign * own cell,
// src/boundary.jl:45-47 with src/blockfield.jl:513-521), or the coarse-fine
// ghost buffer.
// (x: a field's values, or a difference of two fields'.)
template <int D, int M, typename T, class X>
__device__ __forceinline__ T nbv(const X x, const T *__restrict__ ib,
                                 const int *__restrict__ nbr, int blk, int c0, int c1, int c2,
                                 int dim, int dir, const T *sg) {
    using LY = Lay<D, M>;
    int n0 = c0 + (dim == 0 ? dir : 0);
    int n1 = c1 + (dim == 1 ? dir : 0);
    int n2 = c2 + (dim == 2 ? dir : 0);
    int cd = dim == 0 ? n0 : (dim == 1 ? n1 : n2);
    if (cd >= 0 && cd < M) return x[(size_t)blk * LY::V + LY::sidx(n0, n1, n2)];
    int f = 2 * dim + (dir > 0 ? 1 : 0);
    int t = nbr[blk * 2 * D + f];
    if (t >= 0) {
        int w = dir > 0 ? 0 : M - 1;
        if (dim == 0) n0 = w; else if (dim == 1) n1 = w; else n2 = w;
        return x[(size_t)t * LY::V + LY::sidx(n0, n1, n2)];
    }
    if (t == NB_BOUNDARY) return sg[f] * x[(size_t)blk * LY::V + LY::sidx(c0, c1, c2)];
    return ib[(size_t)nb_slot(t) * LY::F + LY::faceidx(dim, c0, c1, c2)];
}

// applystencil(u, s, I, J, disc, geom, Val(:lhs)) for the order-2 operators
// (src/laplacian.jl:78-128, 278-303; src/helmholtz.jl:17-100).
template <int D, int M, typename T>
__device__ __forceinline__ T stencil(const T *__restrict__ x, const T *__restrict__ ib,
                                     const int *__restrict__ nbr, int blk, int c0, int c1, int c2,
                                     T own, const LevelArgs<T> &a, T cc, T wmr, T wpr) {
    T v = T(0);
#pragma unroll
    for (int d = D - 1; d >= 0; d--) {
        T w = (d == a.rdim) ? wmr : T(1);
        v += w * nbv<D, M, T>(x, ib, nbr, blk, c0, c1, c2, d, -1, a.sg);
    }
    v += cc * own;
#pragma unroll
    for (int d = 0; d < D; d++) {
        T w = (d == a.rdim) ? wpr : T(1);
        v += w * nbv<D, M, T>(x, ib, nbr, blk, c0, c1, c2, d, +1, a.sg);
    }
    return v;
}

template <int D, int M, typename T>
__device__ __forceinline__ void radial_weights(const LevelArgs<T> &a, const int *__restrict__ coord,
                                               int blk, int c0, int c1, T &wm, T &wp) {
    wm = T(1);
    wp = T(1);
    if (a.rdim >= 0) {
        int cr = a.rdim == 0 ? c0 : c1;
        int J = M * (coord[blk * D + a.rdim] - 1) + cr + 1;
        wm = a.wm[J];
        wp = a.wp[J];
    }
}

// per-block parameters from the per-(tree, level) ones, blocks' problem
// indices in pix
template <typename T>
__global__ __launch_bounds__(WG) void k_block_params(T *__restrict__ out, const T *__restrict__ pp,
                                                     const int *__restrict__ pix, int nb) {
    const int i = blockIdx.x * WG + threadIdx.x;
    if (i < 3 * nb) out[i] = pp[3 * pix[i / 3] + i % 3];
}

// One colour of gauss_seidel! (src/multigrid.jl:153-180) on every block of a
// level: pass 0 updates the cells with odd global index sum, pass 1 the rest.
// Same-colour cells never read each other, so the update is in place.
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_gs_pass(T *__restrict__ u, const T *__restrict__ b,
                                                const T *__restrict__ ib, const int *__restrict__ nbr,
                                                const int *__restrict__ coord, LevelArgs<T> a, int pass) {
    using LY = Lay<D, M>;
    int gt = blockIdx.x * blockDim.x + threadIdx.x;
    int lb = gt / LY::H;
    if (lb >= a.nblk) return;
    int blk = a.blk0 + lb;
    int q = pass * LY::H + (gt - lb * LY::H);
    int c0, c1, c2;
    LY::decode(q, c0, c1, c2);
    size_t o = (size_t)blk * LY::V + q;
    T own = u[o];
    T wm, wp;
    radial_weights<D, M, T>(a, coord, blk, c0, c1, wm, wp);
    BP<T> bp = bparams(a, blk);
    T Lu = stencil<D, M, T>(u, ib, nbr, blk, c0, c1, c2, own, a, bp.cc, wm, wp);
    T v = fma_t<T>(bp.s, b[o], Lu);
    u[o] = fma_t<T>(bp.nwc, v, own);
}

// residual! over a level (src/multigrid.jl:309-323): r = -(b + L u / s)
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_residual(T *__restrict__ r, const T *__restrict__ u,
                                                 const T *__restrict__ b, const T *__restrict__ ib,
                                                 const int *__restrict__ nbr, const int *__restrict__ coord,
                                                 LevelArgs<T> a) {
    using LY = Lay<D, M>;
    int gt = blockIdx.x * blockDim.x + threadIdx.x;
    int lb = gt / LY::V;
    if (lb >= a.nblk) return;
    int blk = a.blk0 + lb;
    int q = gt - lb * LY::V;
    int c0, c1, c2;
    LY::decode(q, c0, c1, c2);
    size_t o = (size_t)blk * LY::V + q;
    T wm, wp;
    radial_weights<D, M, T>(a, coord, blk, c0, c1, wm, wp);
    BP<T> bp = bparams(a, blk);
    T Lu = stencil<D, M, T>(u, ib, nbr, blk, c0, c1, c2, u[o], a, bp.cc, wm, wp);
    r[o] = -(b[o] + Lu / bp.s);
}

// Linear interpolation weights (src/interp.jl:7-11)
template <int D, typename T> __device__ __forceinline__ T w0() { return D == 2 ? T(0.5) : T(0.25); }
template <typename T> __device__ __forceinline__ T w1() { return T(0.25); }

template <typename T>
struct Bc27 {
    T v[27];
};

// restrict! (src/restrict.jl:5-37): a coarse cell of the parent subblock = mean
// of its 2^D children, summed with the first index fastest. gt: the cell among
// those covered by the level's blocks; its place (index o, block pb, X) and mean f
template <int D, int M, typename T>
__device__ __forceinline__ bool restricted(const T *__restrict__ xf, const int *__restrict__ parent,
                                           const int *__restrict__ sub, int blk0, int nblk, int gt, size_t &o, int &pb,
                                           int &X0, int &X1, int &X2, T &f) {
    using LY = Lay<D, M>;
    constexpr int NS = LY::V / LY::NC;  // coarse cells per subblock
    const int lb = gt / NS;
    if (lb >= nblk) return false;
    const int fb = blk0 + lb, j = gt - lb * NS;
    const int j0 = j % LY::MH, j1 = (j / LY::MH) % LY::MH, j2 = (D == 3) ? j / (LY::MH * LY::MH) : 0;
    f = T(0);
#pragma unroll
    for (int q = 0; q < LY::NC; q++) {
        int i0 = q & 1, i1 = (q >> 1) & 1, i2 = (q >> 2) & 1;
        f += xf[(size_t)fb * LY::V + LY::sidx(2 * j0 + i0, 2 * j1 + i1, D == 3 ? 2 * j2 + i2 : 0)];
    }
    f = f / T(LY::NC);
    pb = parent[fb];
    const int sb = sub[fb];
    X0 = (sb & 1) * LY::MH + j0;
    X1 = ((sb >> 1) & 1) * LY::MH + j1;
    X2 = (D == 3) ? ((sb >> 2) & 1) * LY::MH + j2 : 0;
    o = (size_t)pb * LY::V + LY::sidx(X0, X1, X2);
    return true;
}
template <int D, int M, typename T>
__device__ __forceinline__ void restrict_cell(T *__restrict__ xc, const T *__restrict__ xf,
                                              const int *__restrict__ parent, const int *__restrict__ sub, int blk0,
                                              int nblk, int gt) {
    size_t o;
    int pb, X0, X1, X2;
    T f;
    if (restricted<D, M, T>(xf, parent, sub, blk0, nblk, gt, o, pb, X0, X1, X2, f)) xc[o] = f;
}

// ---- LaplacianDiscretization{D,4}: the 9- and 19-point operators ----
//
// Their stencils reach corner (2D) and edge (3D) ghosts, so the order-4 path
// keeps every block's depth-1 ghosts explicitly: a frame of (M + 2)^D values
// per block (the interior unused), filled as fill_ghost! fills the reference's
// ghost layers (src/connectivity.jl:155-258, with BoxStencil records): the
// copies from same-level neighbours, then the boundary mirrors (which read
// the frame where the mirrored cell is itself a ghost), then the coarse-fine
// interpolations. box[blk * 3^D + k] for the direction k = sum (dir_d + 1) 3^d
// is the same-level neighbour, -(1 + mask) where the direction leaves the
// domain in the dimensions of mask, or -16 - j for coarse-fine slot j
// (coarse block, subblock code).
template <int D, int M>
struct Frame {
    static constexpr int S = M + 2;
    static constexpr int P = D == 3 ? S * S * S : S * S;
    __host__ __device__ static constexpr int at(int c0, int c1, int c2) {
        return D == 3 ? ((c2 + 1) * S + (c1 + 1)) * S + (c0 + 1) : (c1 + 1) * S + (c0 + 1);
    }
};

// the value at cell c of block blk, c at most one cell outside the block
template <int D, int M, typename T>
__device__ __forceinline__ T boxv(const T *__restrict__ x, const T *__restrict__ g, int blk, int c0, int c1,
                                  int c2) {
    using LY = Lay<D, M>;
    const bool in = c0 >= 0 && c0 < M && c1 >= 0 && c1 < M && (D == 2 || (c2 >= 0 && c2 < M));
    return in ? x[(size_t)blk * LY::V + LY::sidx(c0, c1, c2)]
              : g[(size_t)blk * Frame<D, M>::P + Frame<D, M>::at(c0, c1, D == 3 ? c2 : 0)];
}

// the direction of a frame cell (-1, 0, 1 per dimension), its index k, and
// whether it is a ghost
template <int D, int M>
__device__ __forceinline__ bool frame_cell(int q, int *c, int *dir, int &k) {
    constexpr int S = M + 2;
    c[0] = q % S - 1;
    c[1] = (q / S) % S - 1;
    c[2] = D == 3 ? q / (S * S) - 1 : 0;
    bool ghost = false;
    k = 0;
    int m = 1;
#pragma unroll
    for (int d = 0; d < 3; d++) {
        dir[d] = 0;
        if (d < D) {
            dir[d] = c[d] < 0 ? -1 : (c[d] >= M ? 1 : 0);
            ghost |= dir[d] != 0;
            k += (dir[d] + 1) * m;
            m *= 3;
        }
    }
    return ghost;
}

// The value fill_ghost_copy! then fill_ghost_bnd! give ghost cell c of blk (c
// at most one cell outside the block, modified). A ghost facing a same-level
// neighbour is that neighbour's cell. A ghost beyond the domain is a[bnd]
// times the cell mirrored in the dimensions that leave the domain; when other
// dimensions stay outside, the mirrored cell is a ghost of a direction inside
// the domain: a same-level neighbour's cell (read from the neighbour, the value
// the copy writes) or a coarse-fine ghost (read from the frame, as the
// interpolation that refills it comes after both fills). Coarse-fine ghosts
// themselves are read from the frame. row: the block's entries of box.
template <int D, int M, typename T>
__device__ __forceinline__ T ghost_value(const T *__restrict__ x, const T *__restrict__ g,
                                         const int *row, const Bc27<T> &bc, int blk, int *c) {
    using LY = Lay<D, M>;
    constexpr int P = Frame<D, M>::P, NB3 = D == 3 ? 27 : 9;
    int dir[3] = {0, 0, 0}, k = 0, m = 1;
#pragma unroll
    for (int d = 0; d < D; d++) {
        dir[d] = c[d] < 0 ? -1 : (c[d] >= M ? 1 : 0);
        k += (dir[d] + 1) * m;
        m *= 3;
    }
    const int e = row[k];
    if (e >= 0) {
#pragma unroll
        for (int d = 0; d < D; d++) c[d] -= dir[d] * M;
        return x[(size_t)e * LY::V + LY::sidx(c[0], c[1], c[2])];
    }
    if (e < -8) return g[(size_t)blk * P + Frame<D, M>::at(c[0], c[1], D == 3 ? c[2] : 0)];
    const int mask = -1 - e;
    int bi = 0, k2 = 0;
    m = 1;
#pragma unroll
    for (int d = 0; d < D; d++) {
        const bool bd = (mask >> d) & 1;
        bi += ((bd ? dir[d] : 0) + 1) * m;
        if (bd) c[d] = dir[d] < 0 ? -1 - c[d] : 2 * M - 1 - c[d];
        k2 += ((bd ? 0 : dir[d]) + 1) * m;
        m *= 3;
    }
    T v;
    const int e2 = row[k2];
    if (k2 == NB3 / 2) {
        v = x[(size_t)blk * LY::V + LY::sidx(c[0], c[1], c[2])];
    } else if (e2 >= 0) {
#pragma unroll
        for (int d = 0; d < D; d++)
            if (!((mask >> d) & 1)) c[d] -= dir[d] * M;
        v = x[(size_t)e2 * LY::V + LY::sidx(c[0], c[1], c[2])];
    } else {
        v = g[(size_t)blk * P + Frame<D, M>::at(c[0], c[1], D == 3 ? c[2] : 0)];
    }
    return bc.v[bi] * v;
}

// frame cell q of block blk: same-level copy or boundary mirror (coarse-fine
// frame cells are k_frame_interp's)
template <int D, int M, typename T>
__device__ __forceinline__ void frame_copybnd_cell(T *__restrict__ g, const T *__restrict__ x,
                                                   const int *__restrict__ box, int blk, int q, const Bc27<T> &bc) {
    constexpr int P = Frame<D, M>::P, NB3 = D == 3 ? 27 : 9;
    int c[3], dir[3], k;
    if (!frame_cell<D, M>(q, c, dir, k)) return;
    if (box[blk * NB3 + k] < -8) return;  // coarse-fine: k_frame_interp
    g[(size_t)blk * P + q] = ghost_value<D, M, T>(x, g, box + blk * NB3, bc, blk, c);
}

// fill_ghost_copy! then fill_ghost_bnd! in one pass (ghost_value); one pass
// needs no ordering between blocks and gives the bits of the two in order
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_frame_copybnd(T *__restrict__ g, const T *__restrict__ x,
                                                      const int *__restrict__ box, int blk0, int nblk, Bc27<T> bc) {
    constexpr int P = Frame<D, M>::P;
    // 64-bit: a level's nblk * P frame cells can pass 2^31 before its nblk * V cells do
    const int64_t gt = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t lb = gt / P;
    if (lb >= nblk) return;
    frame_copybnd_cell<D, M, T>(g, x, box, blk0 + (int)lb, (int)(gt - lb * P), bc);
}

// reads of cells at most one cell outside a block for the order-4 stencils:
// from the frame as last filled (FrameRead), or live (LiveRead: the values a
// copy-then-boundary fill of the frame would give now)
template <int D, int M, typename T>
struct FrameRead {
    const T *__restrict__ x;
    const T *__restrict__ g;
    __device__ __forceinline__ T operator()(int blk, int c0, int c1, int c2) const {
        return boxv<D, M, T>(x, g, blk, c0, c1, c2);
    }
};
template <int D, int M, typename T>
struct LiveRead {
    const T *__restrict__ x;
    const T *__restrict__ g;
    const int *__restrict__ box;
    const Bc27<T> &bc;
    __device__ __forceinline__ T operator()(int blk, int c0, int c1, int c2) const {
        using LY = Lay<D, M>;
        if (c0 >= 0 && c0 < M && c1 >= 0 && c1 < M && (D == 2 || (c2 >= 0 && c2 < M)))
            return x[(size_t)blk * LY::V + LY::sidx(c0, c1, c2)];
        int c[3] = {c0, c1, D == 3 ? c2 : 0};
        return ghost_value<D, M, T>(x, g, box + blk * (D == 3 ? 27 : 9), bc, blk, c);
    }
};

// fill_ghost_interp! (src/connectivity.jl:251-258, src/interp.jl:23-60): a
// ghost facing a coarse block is the linear interpolation of the coarse cell
// under it with its axis neighbours (coarse ghosts from the coarse frame),
// the offsets towards this block in the dimensions of the direction
template <int D, int M, typename T>
__device__ __forceinline__ T interp_value(const T *__restrict__ g, const T *__restrict__ x, const int2 sl, const int *c,
                                          const int *dir) {
    using LY = Lay<D, M>;
    const int pb = sl.x, sb = sl.y;
    int J[3] = {0, 0, 0}, i[3] = {0, 0, 0};
#pragma unroll
    for (int d = 0; d < D; d++) {
        const int sbd = (sb >> d) & 1;
        if (dir[d] != 0) {
            J[d] = sbd * LY::MH + (dir[d] < 0 ? LY::MH - 1 : 0);
            i[d] = dir[d] < 0 ? 1 : 0;
        } else {
            J[d] = sbd * LY::MH + (c[d] >> 1);
            i[d] = c[d] & 1;
        }
    }
    T f = w0<D, T>() * x[(size_t)pb * LY::V + LY::sidx(J[0], J[1], J[2])];
#pragma unroll
    for (int j = 0; j < D; j++) {
        int K[3] = {J[0], J[1], J[2]};
        K[j] += 2 * i[j] - 1;
        f += w1<T>() * boxv<D, M, T>(x, g, pb, K[0], K[1], K[2]);
    }
    return f;
}

// into g, and into g2 as well unless it is null
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_frame_interp(T *g, T *g2, const T *__restrict__ x,
                                                     const int *__restrict__ box, const int2 *__restrict__ slots,
                                                     int blk0, int nblk) {
    constexpr int P = Frame<D, M>::P, NB3 = D == 3 ? 27 : 9;
    // 64-bit: a level's nblk * P frame cells can pass 2^31 before its nblk * V cells do
    const int64_t gt = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t lb = gt / P;
    if (lb >= nblk) return;
    const int q = (int)(gt - lb * P), blk = blk0 + (int)lb;
    int c[3], dir[3], k;
    if (!frame_cell<D, M>(q, c, dir, k)) return;
    const int e = box[blk * NB3 + k];
    if (e > -16) return;
    const T f = interp_value<D, M, T>(g, x, slots[-16 - e], c, dir);
    g[(size_t)blk * P + q] = f;
    if (g2) g2[(size_t)blk * P + q] = f;
}

// fill_ghost!'s three steps for a 2D level in one launch, a wave pair a block:
// every ghost is read before any is written, since a boundary ghost may mirror
// a coarse-fine one of the same block as it was before the interpolation (no
// other read of this level's frames; the coarse level's are not written here).
// One launch of 3.6 us for k_frame_copybnd's 3.1 and k_frame_interp's 2.7.
template <int M, typename T>
__global__ __launch_bounds__(128) void k_frame_fill2(T *g, const T *__restrict__ x, const T *__restrict__ xc,
                                                     const int *__restrict__ box, const int2 *__restrict__ slots,
                                                     int blk0, Bc27<T> bc) {
    constexpr int S = M + 2, P = Frame<2, M>::P;
    static_assert(4 * (M + 1) <= 128, "a thread for each ghost");
    const int blk = blk0 + blockIdx.x, i = threadIdx.x;
    // the ring: the rows below and above, then the columns
    const int q = i < S ? i : (i < 2 * S ? i + S * (S - 2) : S + (i - 2 * S) / 2 * S + ((i - 2 * S) & 1) * (S - 1));
    const bool in = i < 4 * (M + 1);
    T v = T(0);
    if (in) {
        int c[3], dir[3], k;
        (void)frame_cell<2, M>(q, c, dir, k);
        const int e = box[blk * 9 + k];
        if (e <= -16) v = interp_value<2, M, T>(g, xc, slots[-16 - e], c, dir);
        else v = ghost_value<2, M, T>(x, g, box + blk * 9, bc, blk, c);
    }
    __syncthreads();
    if (in) g[(size_t)blk * P + q] = v;
}

// interp_add_level! (src/interp.jl:102-115) reading the coarse ghosts from
// the frames
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_interp_add4(T *__restrict__ u, const T *__restrict__ u1,
                                                    const T *__restrict__ g1, const int *__restrict__ parent,
                                                    const int *__restrict__ sub, int blk0, int nblk) {
    using LY = Lay<D, M>;
    const int gt = blockIdx.x * blockDim.x + threadIdx.x;
    const int lb = gt / LY::V;
    if (lb >= nblk) return;
    const int fb = blk0 + lb, q = gt - lb * LY::V;
    int x0, x1, x2;
    LY::decode(q, x0, x1, x2);
    const int pb = parent[fb], sb = sub[fb];
    const int J0 = (sb & 1) * LY::MH + (x0 >> 1);
    const int J1 = ((sb >> 1) & 1) * LY::MH + (x1 >> 1);
    const int J2 = (D == 3) ? ((sb >> 2) & 1) * LY::MH + (x2 >> 1) : 0;
    T f = w0<D, T>() * u1[(size_t)pb * LY::V + LY::sidx(J0, J1, J2)];
    f += w1<T>() * boxv<D, M, T>(u1, g1, pb, J0 + 2 * (x0 & 1) - 1, J1, J2);
    f += w1<T>() * boxv<D, M, T>(u1, g1, pb, J0, J1 + 2 * (x1 & 1) - 1, J2);
    if (D == 3) f += w1<T>() * boxv<D, M, T>(u1, g1, pb, J0, J1, J2 + 2 * (x2 & 1) - 1);
    const size_t o = (size_t)fb * LY::V + q;
    u[o] = f + u[o];
}

// applystencil (src/laplacian.jl:133-141, 305-320): the literal's nonzero
// terms in column-major order, then one division by 6
template <int D, int M, typename T, typename A>
__device__ __forceinline__ T stencil4(const A &at, int blk, int c0, int c1, int c2) {
    T v = T(0);
    constexpr int NK = D == 3 ? 1 : 0;
#pragma unroll
    for (int k = -NK; k <= NK; k++)
#pragma unroll
        for (int j = -1; j <= 1; j++)
#pragma unroll
            for (int i = -1; i <= 1; i++) {
                const int n = (i != 0) + (j != 0) + (k != 0);
                const int a = D == 2 ? (n == 0 ? -20 : (n == 1 ? 4 : 1))
                                     : (k == 0 ? (n == 0 ? -24 : (n == 1 ? 2 : 1)) : (n == 1 ? 2 : (n == 2 ? 1 : 0)));
                if (a == 0) continue;
                v += T(a) * at(blk, c0 + i, c1 + j, c2 + k);
            }
    return v / T(6);
}

// LaplacianDiscretization{2,4} x CylindricalGeometry{N+1} (src/laplacian.jl:
// 156-201) at 1-based global radial index i: the 3x3 literal's entries
// (integer ratios rounded once), visited column-major, divided by 6; and its
// diagelm
template <typename T>
struct Cyl4 {
    T lo, hi, pm, pp, cc, dg;
};
template <typename T>
__device__ __forceinline__ Cyl4<T> cyl4(long long i) {
    const long long q = 2 * i - 1;
    Cyl4<T> w;
    w.lo = (T)(2 * (i - 1)) / (T)q;
    w.hi = (T)(2 * i) / (T)q;
    w.pm = (T)(4 * (-2 + 9 * i - 16 * i * i + 8 * i * i * i)) / (T)(q * q * q);
    w.pp = (T)(4 * (1 + i - 8 * i * i + 8 * i * i * i)) / (T)(q * q * q);
    w.cc = (T)(-16 * (1 - 5 * i + 5 * i * i)) / (T)((1 - 2 * i) * (1 - 2 * i));
    w.dg = w.cc / T(6);
    return w;
}
// at(a, b): the value at offset (a, b)
template <typename T, typename A>
__device__ __forceinline__ T stencil4cyl(const A &at, int N, const Cyl4<T> &l) {
    T w[3][3];
    if (N == 0) {
        w[0][0] = l.lo; w[0][1] = l.pm; w[0][2] = l.lo;
        w[1][0] = T(4); w[1][1] = l.cc; w[1][2] = T(4);
        w[2][0] = l.hi; w[2][1] = l.pp; w[2][2] = l.hi;
    } else {
        w[0][0] = l.lo; w[0][1] = T(4); w[0][2] = l.hi;
        w[1][0] = l.pm; w[1][1] = l.cc; w[1][2] = l.pp;
        w[2][0] = l.lo; w[2][1] = T(4); w[2][2] = l.hi;
    }
    T v = T(0);
#pragma unroll
    for (int b = 0; b < 3; b++)
#pragma unroll
        for (int a = 0; a < 3; a++) v += w[a][b] * at(a - 1, b - 1);
    return v / T(6);
}

// the order-4 operator at cell (c0, c1, c2) of blk: Cartesian (rd < 0) or
// cylindrical with radial dimension rd (global radial index from coord)
template <int D, int M, typename T, typename A>
__device__ __forceinline__ T apply4a(const A &at, const int *__restrict__ coord, int blk, int c0, int c1, int c2,
                                     int rd, T &diag) {
    if constexpr (D == 2) {
        if (rd >= 0) {
            const long long i = (long long)(rd == 0 ? c0 : c1) + 1 + (long long)M * (coord[blk * D + rd] - 1);
            const Cyl4<T> w = cyl4<T>(i);
            diag = w.dg;
            return stencil4cyl<T>([&](int x, int y) { return at(blk, c0 + x, c1 + y, 0); }, rd, w);
        }
    }
    diag = D == 2 ? T(-20.0 / 6.0) : T(-4);
    return stencil4<D, M, T>(at, blk, c0, c1, c2);
}
template <int D, int M, typename T>
__device__ __forceinline__ T apply4(const T *__restrict__ x, const T *__restrict__ g,
                                    const int *__restrict__ coord, int blk, int c0, int c1, int c2, int rd,
                                    T &diag) {
    return apply4a<D, M, T>(FrameRead<D, M, T>{x, g}, coord, blk, c0, c1, c2, rd, diag);
}

// the FP32 right-hand side of the order-4 correction equation of a mixed
// precision step: be = b + L4 u / s in FP64, rounded once
template <int D, int M>
__global__ __launch_bounds__(WG) void k_defect4(float *__restrict__ be, const double *__restrict__ u,
                                                const double *__restrict__ b, const double *__restrict__ g,
                                                const int *__restrict__ coord, int rd, int blk0, int nblk,
                                                double s) {
    using LY = Lay<D, M>;
    const int gt = blockIdx.x * blockDim.x + threadIdx.x;
    const int lb = gt / LY::V;
    if (lb >= nblk) return;
    const int blk = blk0 + lb, q = gt - lb * LY::V;
    int c0, c1, c2;
    LY::decode(q, c0, c1, c2);
    const size_t o = (size_t)blk * LY::V + q;
    double c;
    const double Lu = apply4<D, M, double>(u, g, coord, blk, c0, c1, c2, rd, c);
    be[o] = (float)(b[o] + Lu / s);
}

// gauss_seidel!(..., ::FourColors{P1,P2}) (src/multigrid.jl:206-232) over a
// level: colour cells (x = P1, y = P2 mod 2 from the first valid cell; in 3D
// both shifted by the 1-based third index with G = 2 ghost layers, the
// reference's depth), u -= omega (Lu + s b) / diagelm; cells of one colour do
// not read each other
// LIVE: ghosts read live (LiveRead) instead of from the frame, which equals a
// pass that follows a copy-then-boundary fill: the cells one pass reads across
// a block face are of other colours, or, for a boundary mirror, the cell being
// updated itself (read before its write), so none changes during the pass
// (3D; k_gs4_sweep takes 2D levels: a 3D block's halo would be several times
// the block)
template <int M, typename T, bool LIVE>
__global__ __launch_bounds__(WG) void k_gs4_pass(T *__restrict__ u, const T *__restrict__ b,
                                                 const T *__restrict__ g, int blk0, int nblk, T s, T omega, int P1,
                                                 int P2, const int *__restrict__ box, Bc27<T> bc) {
    using LY = Lay<3, M>;
    constexpr int H2 = M / 2, NCC = H2 * H2 * M;
    const int gt = blockIdx.x * blockDim.x + threadIdx.x;
    const int lb = gt / NCC;
    if (lb >= nblk) return;
    const int blk = blk0 + lb, q = gt - lb * NCC, z = q / (H2 * H2);
    const int x0 = 2 * (q % H2) + ((P1 + z + 3) & 1), x1 = 2 * ((q / H2) % H2) + ((P2 + z + 3) & 1);
    const size_t o = (size_t)blk * LY::V + LY::sidx(x0, x1, z);
    T c, Lu;
    if constexpr (LIVE)
        Lu = apply4a<3, M, T>(LiveRead<3, M, T>{u, g, box, bc}, nullptr, blk, x0, x1, z, -1, c);
    else
        Lu = apply4a<3, M, T>(FrameRead<3, M, T>{u, g}, nullptr, blk, x0, x1, z, -1, c);
    u[o] = u[o] - omega * (Lu + s * b[o]) / c;
}

// NS sweeps, with their four colour passes each, of a 2D level in one launch
// and out of place: a work group takes a block with the cells around it that
// its passes depend on (for a sweep one cell to the sides and three above and
// below: the colours' order (0,0), (0,1), (1,0), (1,1) needs no more; for each
// sweep before it two and four more), and runs the passes there, those of the
// neighbours' cells too (325 cells for 256 with M = 16, 565 in the first of
// two sweeps). In place and pass by pass a sweep of 24 blocks took four launches
// of 4.4 us, all of it round trips: the box row, the cells, the divisions for
// the radial weights (here one table for the block). Two
// sweeps of 20 to 32 blocks take 12 to 13 us (one: 8.4; 1.2 us a pass, 60 FP64
// instructions in a chain), where the eight passes took 35; of 1024 blocks 25 us
// for 53.
//
// The tile holds the live ghosts: a boundary ghost is written again with its
// mirror cell, a coarse-fine ghost does not change during a sweep (its value
// depends on its place only, not on the block it is a ghost of). FRAME0: the
// first pass reads the ghosts of every block from its frame as it was last
// filled (LiveRead and FrameRead differ there if the level was not filled just
// before, and where a boundary mirrors a coarse-fine ghost).
template <int M>
constexpr int GS4_THREADS = M == 16 ? 256 : 128;
template <int M, typename T, int NS, bool FRAME0>
__global__ __launch_bounds__(GS4_THREADS<M>) void k_gs4_sweep(T *__restrict__ out, const T *__restrict__ u,
                                                              const T *__restrict__ b, const T *__restrict__ g,
                                                              const int *__restrict__ coord, int rd, int blk0, T s,
                                                              T omega, const int *__restrict__ box, Bc27<T> bc) {
    using LY = Lay<2, M>;
    constexpr int J = NS - 1, NT = GS4_THREADS<M>, P = Frame<2, M>::P, H2 = M / 2;
    constexpr int X0 = -1 - 2 * J, Y0 = -3 - 4 * J, W = M - 2 * X0 + 1, H = M - 2 * Y0 + 1, NR = M - 2 * Y0 - 1;
    constexpr int LW = M == 16 ? 32 : 16, RY = NT / LW, NI = (H + RY - 1) / RY;  // loads: RY rows at a time
    constexpr int CW = LW / 2;                                                   // a pass: CW columns of cells
    static_assert(H2 + 1 + 2 * J <= CW && (H2 + 3 + 4 * J) * CW <= NT, "a colour's cells are one for each thread");
    static_assert(Y0 >= -M && W <= LW && NR <= NT, "a row, and the radial weights, are one for each thread");
    // the iterate and b, the columns of one parity together: a pass reads
    // cells two apart in x
    constexpr int WH = (W + 1) / 2;
    __shared__ T t[2 * WH * H], tb[2 * WH * H];
    const auto at_ = [](int x, int y) { return ((y - Y0) * 2 + ((x - X0) & 1)) * WH + ((x - X0) >> 1); };
    __shared__ Cyl4<T> wr[NR];
    __shared__ int rows[9][9];  // the entries of box of the blocks around (4: this one)
    const int tid = threadIdx.x, blk = blk0 + blockIdx.x;
    if (tid < 9) rows[4][tid] = box[blk * 9 + tid];
    const int rc = rd >= 0 ? coord[blk * 2 + rd] - 1 : 0;
    __syncthreads();
    for (int i = tid; i < 81; i += NT) {
        const int n = i / 9, e = rows[4][n];
        if (n != 4 && e >= 0) rows[n][i - 9 * n] = box[e * 9 + i - 9 * n];
    }
    const auto side = [](int c) { return c < 0 ? 0 : (c >= M ? 2 : 1); };
    // the tile's cells in the blocks around
    const int lx = tid % LW + X0, ly = tid / LW + Y0, sx = side(lx);
    T v[NI], vb[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int y = ly + i * RY, sy = side(y), e = rows[4][sx + 3 * sy];
        v[i] = vb[i] = T(0);
        if (lx < X0 + W && y < Y0 + H && e >= 0) {
            const size_t o = (size_t)e * LY::V + LY::sidx(lx - M * (sx - 1), y - M * (sy - 1), 0);
            v[i] = u[o];
            vb[i] = b[o];
        }
    }
    // the cell of this thread in colour 0, as place in the tile: colour col's
    // is at (col / 2, col) from it, a later sweep's at (2, 4)
    const int px = 2 * (tid % CW) - 2 * J, py = 2 * (tid / CW) - 2 - 4 * J;
    T f0[9];
    if constexpr (FRAME0) {
        const int x = px - M * (side(px) - 1), y = py - M * (side(py) - 1);
        const bool edge = x == 0 || x == M - 1 || y == 0 || y == M - 1;
        const int e = px <= M + 2 * J && py <= M + 2 + 4 * J ? rows[4][side(px) + 3 * side(py)] : -1;
#pragma unroll
        for (int k = 0; k < 9; k++) {
            f0[k] = T(0);
            if (edge && e >= 0 && (side(x + k % 3 - 1) != 1 || side(y + k / 3 - 1) != 1))
                f0[k] = g[(size_t)e * P + Frame<2, M>::at(x + k % 3 - 1, y + k / 3 - 1, 0)];
        }
    }
    if (rd >= 0 && tid < NR) wr[tid] = cyl4<T>((long long)tid + Y0 + 2 + (long long)M * rc);
#pragma unroll
    for (int i = 0; i < NI; i++)
        if (lx < X0 + W && ly + i * RY < Y0 + H) {
            t[at_(lx, ly + i * RY)] = v[i];
            tb[at_(lx, ly + i * RY)] = vb[i];
        }
    __syncthreads();
    // the ghosts among them: each is one of the block next to it in x, in y or
    // in both (ghost_value, the cells taken from the tile)
#pragma unroll 1
    for (int i = 0; i < NI; i++) {
        const int y = ly + i * RY, sy = side(y);
        if (lx >= X0 + W || y >= Y0 + H || rows[4][sx + 3 * sy] >= 0) continue;
        const int ax = lx == -1 || lx == M ? 1 : (lx == 0 ? 0 : (lx == M - 1 ? 2 : sx));
        const int ay = y == -1 || y == M ? 1 : (y == 0 ? 0 : (y == M - 1 ? 2 : sy));
        int n = ax + 3 * sy;
        if (rows[4][n] < 0) n = sx + 3 * ay;
        if (rows[4][n] < 0) n = ax + 3 * ay;
        const int en = rows[4][n];
        if (en < 0) continue;  // no pass reads it
        const int x0 = M * (n % 3 - 1), y0 = M * (n / 3 - 1);
        int c0 = lx - x0, c1 = y - y0, k = side(c0) + 3 * side(c1);
        int bi = 4, e = rows[n][k];
        if (e >= -8) {
            const int mask = -1 - e;
            if (mask & 1) {
                bi += side(c0) - 1;
                k += 1 - side(c0);
                c0 = c0 < 0 ? 0 : M - 1;
            }
            if (mask & 2) {
                bi += 3 * (side(c1) - 1);
                k += 3 * (1 - side(c1));
                c1 = c1 < 0 ? 0 : M - 1;
            }
            e = rows[n][k];
        }
        const T m = e >= 0 ? t[at_(c0 + x0, c1 + y0)] : g[(size_t)en * P + Frame<2, M>::at(c0, c1, 0)];
        t[at_(lx, y)] = bi == 4 ? m : bc.v[bi] * m;
    }
    // the passes in which this thread has a cell, and the domain's faces
    unsigned act = 0;
#pragma unroll
    for (int pass = 0; pass < 4 * NS; pass++) {
        const int col = pass & 3, j = J - (pass >> 2);
        const int x = px + 2 * (J - j) + (col >> 1), y = py + 4 * (J - j) + col;
        const bool in = x <= M - (col >> 1) + 2 * j && y <= M + 2 - col + 4 * j;
        if (in && rows[4][side(x) + 3 * side(y)] >= 0) act |= 1u << pass;
    }
    const auto outside = [&](int k) { return rows[4][k] < 0 && rows[4][k] >= -8; };
    const bool out0 = outside(3), out1 = outside(5), out2 = outside(1), out3 = outside(7);
    __syncthreads();
    const auto run = [&](int pass, auto framed) {
        const int x = px + 2 * (pass >> 2) + ((pass & 3) >> 1), y = py + pass;
        if ((act >> pass) & 1) {
            const int q = at_(x, y), qe = at_(x - 1, y), qo = at_(x + 1, y);
            const auto at = [&](int a, int c) {
                if constexpr (decltype(framed)::value) {
                    const int xa = x - M * (side(x) - 1) + a, yc = y - M * (side(y) - 1) + c;
                    if (side(xa) != 1 || side(yc) != 1) return f0[a + 1 + 3 * (c + 1)];
                }
                return t[(a < 0 ? qe : (a > 0 ? qo : q)) + c * 2 * WH];
            };
            T d, Lu;
            if (rd >= 0) {
                const Cyl4<T> &w = wr[(rd == 0 ? x : y) - Y0 - 1];
                d = w.dg;
                Lu = stencil4cyl<T>(at, rd, w);
            } else {
                d = T(-20.0 / 6.0);
                Lu = stencil4<2, M, T>([&](int, int a, int c, int) { return at(a, c); }, 0, 0, 0, 0);
            }
            const T nv = t[q] - omega * (Lu + s * tb[q]) / d;
            t[q] = nv;
            // its boundary ghosts
            const int gx = x == 0 && out0 ? -1 : (x == M - 1 && out1 ? 1 : 0);
            const int gy = y == 0 && out2 ? -1 : (y == M - 1 && out3 ? 1 : 0);
            if (gx) t[at_(x + gx, y)] = bc.v[gx + 4] * nv;
            if (gy) t[at_(x, y + gy)] = bc.v[3 * gy + 4] * nv;
            if (gx && gy) t[at_(x + gx, y + gy)] = bc.v[3 * gy + gx + 4] * nv;
        }
        __syncthreads();
    };
    if constexpr (FRAME0) run(0, std::true_type{});
#pragma unroll 1
    for (int pass = FRAME0 ? 1 : 0; pass < 4 * NS; pass++) run(pass, std::false_type{});
    for (int i = tid; i < LY::V; i += NT) {
        int c0, c1, c2;
        LY::decode(i, c0, c1, c2);
        out[(size_t)blk * LY::V + i] = t[at_(c0, c1)];
    }
}

// residual! (src/multigrid.jl:309-323) with the order-4 operator
template <int D, int M, typename T>
__device__ __forceinline__ void resid4_cell(T *__restrict__ r, const T *__restrict__ u, const T *__restrict__ b,
                                            const T *__restrict__ g, const int *__restrict__ coord, int rd, int blk,
                                            int q, T s) {
    using LY = Lay<D, M>;
    int c0, c1, c2;
    LY::decode(q, c0, c1, c2);
    const size_t o = (size_t)blk * LY::V + q;
    T c;
    const T Lu = apply4<D, M, T>(u, g, coord, blk, c0, c1, c2, rd, c);
    r[o] = -(b[o] + Lu / s);
}
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_resid4(T *__restrict__ r, const T *__restrict__ u, const T *__restrict__ b,
                                               const T *__restrict__ g, const int *__restrict__ coord, int rd,
                                               int blk0, int nblk, T s) {
    using LY = Lay<D, M>;
    const int gt = blockIdx.x * blockDim.x + threadIdx.x;
    const int lb = gt / LY::V;
    if (lb >= nblk) return;
    resid4_cell<D, M, T>(r, u, b, g, coord, rd, blk0 + lb, gt - lb * LY::V, s);
}

// The steps of an order-4 cycle around its sweeps that do not wait for each
// other share a launch, each with its own work groups: on small levels a step
// is one round trip of 2 to 4 us, whatever it does (a cycle on three levels of
// 20 to 32 blocks: 17 launches between its sweeps instead of 38).
//
// After the sweeps down: refill the copy and boundary ghosts of the level
// (nframe work groups), restrict it.
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k4_refill_restrict(T *__restrict__ g, T *__restrict__ xc, const T *__restrict__ x,
                                                         const int *__restrict__ box, const int *__restrict__ parent,
                                                         const int *__restrict__ sub, int blk0, int nblk, Bc27<T> bc,
                                                         unsigned nframe) {
    using LY = Lay<D, M>;
    constexpr int P = Frame<D, M>::P;
    if (blockIdx.x < nframe) {
        const int64_t gt = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, lb = gt / P;
        if (lb < nblk) frame_copybnd_cell<D, M, T>(g, x, box, blk0 + (int)lb, (int)(gt - lb * P), bc);
        return;
    }
    restrict_cell<D, M, T>(xc, x, parent, sub, blk0, nblk, (int)((blockIdx.x - nframe) * blockDim.x + threadIdx.x));
}
// Then: the level's residual (nres work groups), the copy and boundary ghosts
// of the coarse level (nframe), and its values kept in u1.
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k4_resid_coarse(T *__restrict__ r, const T *__restrict__ u,
                                                      const T *__restrict__ b, const T *g,
                                                      const int *__restrict__ coord, int rd, int blk0, int nblk, T s,
                                                      T *gw, T *__restrict__ u1, const T *__restrict__ uc,
                                                      const int *__restrict__ box, int cblk0, int ncoarse, Bc27<T> bc,
                                                      unsigned nres, unsigned nframe) {
    using LY = Lay<D, M>;
    constexpr int P = Frame<D, M>::P;
    if (blockIdx.x < nres) {
        const int gt = blockIdx.x * blockDim.x + threadIdx.x, lb = gt / LY::V;
        if (lb < nblk) resid4_cell<D, M, T>(r, u, b, g, coord, rd, blk0 + lb, gt - lb * LY::V, s);
    } else if (blockIdx.x < nres + nframe) {
        const int64_t gt = (int64_t)(blockIdx.x - nres) * blockDim.x + threadIdx.x, lb = gt / P;
        if (lb < ncoarse) frame_copybnd_cell<D, M, T>(gw, uc, box, cblk0 + (int)lb, (int)(gt - lb * P), bc);
    } else {
        const size_t i = (size_t)(blockIdx.x - nres - nframe) * blockDim.x + threadIdx.x;
        if (i < (size_t)ncoarse * LY::V) u1[(size_t)cblk0 * LY::V + i] = uc[(size_t)cblk0 * LY::V + i];
    }
}
// Before the correction: u1 = u - u1 on the coarse level's cells (nval work
// groups) and, with coarse-fine ghosts on it, ghosts (ndiff), and the copy and
// boundary ghosts of u's top level after its sweeps.
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k4_diff(T *__restrict__ u1, const T *__restrict__ u, T *__restrict__ g1, T *g,
                                              const int *__restrict__ box, int blk0, int nblk, Bc27<T> bc,
                                              unsigned nval, unsigned ndiff) {
    using LY = Lay<D, M>;
    constexpr int P = Frame<D, M>::P;
    if (blockIdx.x < nval) {
        const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x, o = (size_t)blk0 * LY::V + i;
        if (i < (size_t)nblk * LY::V) u1[o] = u[o] - u1[o];
    } else if (blockIdx.x < nval + ndiff) {
        const size_t i = (size_t)(blockIdx.x - nval) * blockDim.x + threadIdx.x, o = (size_t)blk0 * P + i;
        if (i < (size_t)nblk * P) g1[o] = g[o] - g1[o];
    } else {
        const int64_t gt = (int64_t)(blockIdx.x - nval - ndiff) * blockDim.x + threadIdx.x, lb = gt / P;
        if (lb < nblk) frame_copybnd_cell<D, M, T>(g, u, box, blk0 + (int)lb, (int)(gt - lb * P), bc);
    }
}

// restrict! of the residual, and residual_postrestrict_level!
// (src/multigrid.jl:112-119, 331-344) with the order-4 operator on the coarse
// cells covered by the fine blocks
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_postrestrict4(T *__restrict__ bout, const T *__restrict__ u,
                                                      T *__restrict__ rc, const T *__restrict__ r,
                                                      const T *__restrict__ g, const int *__restrict__ coord, int rd,
                                                      const int *__restrict__ parent, const int *__restrict__ sub,
                                                      int fblk0, int nfine, T s) {
    using LY = Lay<D, M>;
    size_t o;
    int pb, X0, X1, X2;
    T f;
    if (!restricted<D, M, T>(r, parent, sub, fblk0, nfine, blockIdx.x * blockDim.x + threadIdx.x, o, pb, X0, X1, X2, f))
        return;
    rc[o] = f;
    T c;
    const T Lu = apply4<D, M, T>(u, g, coord, pb, X0, X1, X2, rd, c);
    bout[o] = -(f + Lu / s);
}

// rhs! (src/multigrid.jl:363-388) of the compact 4th-order Laplacian
// (LaplacianDiscretization{D,4}, src/laplacian.jl:142-149, 167-175, 187-195,
// 322-337): b1 = (1/12) [0 1 0; 1 8 1; 0 1 0] b in 2D (the radial weights of
// the cylindrical forms on the radial neighbours), the 7-point [1 .. 6 .. 1]
// in 3D; the @stencil order of terms is the order-2 stencil's with centre
// weight 12 - 2D, then one division by 12.
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_rhs4(T *__restrict__ b1, const T *__restrict__ b, const T *__restrict__ ib,
                                             const int *__restrict__ nbr, const int *__restrict__ coord,
                                             LevelArgs<T> a) {
    using LY = Lay<D, M>;
    int gt = blockIdx.x * blockDim.x + threadIdx.x;
    int lb = gt / LY::V;
    if (lb >= a.nblk) return;
    int blk = a.blk0 + lb;
    int q = gt - lb * LY::V;
    int c0, c1, c2;
    LY::decode(q, c0, c1, c2);
    size_t o = (size_t)blk * LY::V + q;
    T wm, wp;
    radial_weights<D, M, T>(a, coord, blk, c0, c1, wm, wp);
    T v = stencil<D, M, T>(b, ib, nbr, blk, c0, c1, c2, b[o], a, T(12 - 2 * D), wm, wp);
    b1[o] = v / T(12);
}

// restrict! over the Child edges of a level
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_restrict(T *__restrict__ xc, const T *__restrict__ xf,
                                                 const int *__restrict__ parent, const int *__restrict__ sub,
                                                 int blk0, int nblk) {
    restrict_cell<D, M, T>(xc, xf, parent, sub, blk0, nblk, blockIdx.x * blockDim.x + threadIdx.x);
}

// residual_postrestrict_level! (src/multigrid.jl:112-119, 331-344): FAS
// right-hand side at every coarse cell covered by a block of this level,
// b = -(r + L_{l-1} u / s_{l-1}); `a` describes the coarse level.
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_postrestrict(T *__restrict__ bout, const T *__restrict__ u,
                                                     const T *__restrict__ r, const T *__restrict__ ib,
                                                     const int *__restrict__ nbr, const int *__restrict__ coord,
                                                     const int *__restrict__ parent, const int *__restrict__ sub,
                                                     int fblk0, int nfine, LevelArgs<T> a) {
    using LY = Lay<D, M>;
    constexpr int NS = LY::V / LY::NC;
    int gt = blockIdx.x * blockDim.x + threadIdx.x;
    int lb = gt / NS;
    if (lb >= nfine) return;
    int fb = fblk0 + lb;
    int j = gt - lb * NS;
    int j0 = j % LY::MH, j1 = (j / LY::MH) % LY::MH, j2 = (D == 3) ? j / (LY::MH * LY::MH) : 0;
    int pb = parent[fb];
    int sb = sub[fb];
    int X0 = (sb & 1) * LY::MH + j0, X1 = ((sb >> 1) & 1) * LY::MH + j1;
    int X2 = (D == 3) ? ((sb >> 2) & 1) * LY::MH + j2 : 0;
    size_t o = (size_t)pb * LY::V + LY::sidx(X0, X1, X2);
    T wm, wp;
    radial_weights<D, M, T>(a, coord, pb, X0, X1, wm, wp);
    BP<T> bp = bparams(a, pb);
    T Lu = stencil<D, M, T>(u, ib, nbr, pb, X0, X1, X2, u[o], a, bp.cc, wm, wp);
    bout[o] = -(r[o] + Lu / bp.s);
}

// copyto! / diffto! over the valid cells of a block range (src/blockfield.jl:557-576)
template <typename T>
__global__ __launch_bounds__(WG) void k_copy(T *__restrict__ dst, const T *__restrict__ src, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = src[i];
}

// storage position of local cell (x, y, z) and its inverse, as Lay<D, M>, for
// sizes known at run time (the host-layout conversions)
__device__ __forceinline__ int rt_sidx(int D, int M, int x, int y, int z) {
    const int V = D == 2 ? M * M : M * M * M;
    return (((x + y + z + D) & 1) ? 0 : V / 2) + (x >> 1) + (M / 2) * (y + M * z);
}

// Host blocks in the pinned ring -> device blocks dev (one work group each): the
// planes of the last dimension from one cell below the valid ones to one above,
// S = M + 2 G cells in the other dimensions, read once and in order, as the bus
// likes it. Valid cells, and the depth-1 ghosts of coarse-fine faces into their
// slabs. A block is shared out over gridDim.y work groups (HOST_IN_CELLS cells
// each): a piece of the ring holds 15 blocks of 16^3 with three ghost layers, and
// with one work group for each its reads over the bus were waited out one after
// the other (699 such blocks 3.3 ms, now 1.25).
constexpr int HOST_IN_CELLS = 1024;
template <typename TH, typename TD>
__global__ __launch_bounds__(WG) void k_host_in(TD *__restrict__ data, TD *__restrict__ ib, const TH *__restrict__ src,
                                                const int *__restrict__ dev, const int *__restrict__ nbr, int D,
                                                int M, int G) {
    const int b = dev[blockIdx.x];
    const int S = M + 2 * G, V = D == 2 ? M * M : M * M * M, F = V / M;
    const int n = (D == 2 ? S : S * S) * (M + 2);
    const TH *p = src + (size_t)blockIdx.x * n;
    for (int i = blockIdx.y * WG + threadIdx.x; i < n; i += gridDim.y * WG) {
        const TH v = p[i];
        const int r = i / S;
        const int x[3] = {i % S - G, D == 2 ? r - 1 : r % S - G, D == 2 ? 0 : r / S - 1};
        int f = -1, out = 0;
        for (int d = 0; d < D; d++)
            if (x[d] < 0 || x[d] >= M) {
                out += x[d] < -1 || x[d] > M ? 2 : 1;
                f = 2 * d + (x[d] < 0 ? 0 : 1);
            }
        if (out > 1) continue;
        if (out == 0) {
            data[(size_t)b * V + rt_sidx(D, M, x[0], x[1], x[2])] = (TD)v;
            continue;
        }
        const int t = nbr[(size_t)b * 2 * D + f], dim = f >> 1;
        const int a = dim == 0 ? x[1] : x[0], c = dim == 2 ? x[1] : x[2];
        if (t <= -2) ib[(size_t)nb_slot(t) * F + a + M * c] = (TD)v;
    }
}

struct Faces6 {
    int8_t s[6];
};

// Device blocks -> boxes of M + 2 g cells per dimension (g = 0 or 1) in the
// pinned ring, in the order of the host's block ids (one work group each, dev the
// device blocks): valid cells and, with g = 1, the face ghosts (copies, +-mirrors, slabs); edges and corners are not
// written.
template <typename TD, typename TH>
__global__ __launch_bounds__(WG) void k_host_out(TH *__restrict__ dst, const TD *__restrict__ data,
                                                 const TD *__restrict__ ib, const int *__restrict__ dev,
                                                 const int *__restrict__ nbr, int D, int M, int g, Faces6 sg) {
    const int b = dev[blockIdx.x];
    const int B = M + 2 * g, n = D == 2 ? B * B : B * B * B, V = D == 2 ? M * M : M * M * M, F = V / M;
    TH *p = dst + (size_t)blockIdx.x * n;
    for (int i = threadIdx.x; i < n; i += WG) {
        int x[3] = {i % B - g, (i / B) % B - g, D == 3 ? i / (B * B) - g : 0};
        int f = -1, out = 0;
        for (int d = 0; d < D; d++)
            if (x[d] < 0 || x[d] >= M) {
                out++;
                f = 2 * d + (x[d] < 0 ? 0 : 1);
            }
        if (out > 1) continue;
        if (out == 0) {
            p[i] = (TH)data[(size_t)b * V + rt_sidx(D, M, x[0], x[1], x[2])];
            continue;
        }
        const int t = nbr[(size_t)b * 2 * D + f], dim = f >> 1;
        if (t <= -2) {
            const int a = dim == 0 ? x[1] : x[0], c = dim == 2 ? x[1] : x[2];
            p[i] = (TH)ib[(size_t)nb_slot(t) * F + a + M * c];
        } else {
            // the neighbour's cell across the face, or the own cell at it
            x[dim] = (t >= 0) == ((f & 1) != 0) ? 0 : M - 1;
            const TH v = (TH)data[(size_t)(t >= 0 ? t : b) * V + rt_sidx(D, M, x[0], x[1], x[2])];
            p[i] = t >= 0 ? v : (TH)sg.s[f] * v;
        }
    }
}

// r = a + b: a stream kernel of the solver's own size, for bandwidth calibration
template <typename T>
__global__ __launch_bounds__(WG) void k_triad(T *__restrict__ r, const T *__restrict__ a, const T *__restrict__ b,
                                              size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) r[i] = a[i] + b[i];
}

// the same with 16-byte loads and nontemporal 16-byte stores per lane (n a
// multiple of 16 / sizeof(T)): the strongest plain stream form, the
// bandwidth ceiling of the calibration
template <typename T>
__global__ __launch_bounds__(WG) void k_triad16(T *__restrict__ r, const T *__restrict__ a, const T *__restrict__ b,
                                                size_t n) {
    constexpr int K = 16 / sizeof(T);
    typedef T V __attribute__((ext_vector_type(K)));
    const size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * K;
    if (i >= n) return;
    const V x = *reinterpret_cast<const V *>(a + i), y = *reinterpret_cast<const V *>(b + i);
    __builtin_nontemporal_store(x + y, reinterpret_cast<V *>(r + i));
}

template <typename T>
__global__ __launch_bounds__(WG) void k_fill(T *__restrict__ dst, T v, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) dst[i] = v;
}


// interp_add_level!(u, u1, child) (src/interp.jl:102-141, 185-193): every
// fine cell += linear interpolation of the parent's correction u1.
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_interp_add(T *__restrict__ u, const T *__restrict__ u1,
                                                   const T *__restrict__ ib1, const int *__restrict__ nbr,
                                                   const int *__restrict__ parent, const int *__restrict__ sub,
                                                   int blk0, int nblk, LevelArgs<T> a) {
    using LY = Lay<D, M>;
    int gt = blockIdx.x * blockDim.x + threadIdx.x;
    int lb = gt / LY::V;
    if (lb >= nblk) return;
    int fb = blk0 + lb;
    int q = gt - lb * LY::V;
    int x0, x1, x2;
    LY::decode(q, x0, x1, x2);
    int pb = parent[fb];
    int sb = sub[fb];
    int J0 = (sb & 1) * LY::MH + (x0 >> 1);
    int J1 = ((sb >> 1) & 1) * LY::MH + (x1 >> 1);
    int J2 = (D == 3) ? ((sb >> 2) & 1) * LY::MH + (x2 >> 1) : 0;
    T f = w0<D, T>() * u1[(size_t)pb * LY::V + LY::sidx(J0, J1, J2)];
    f += w1<T>() * nbv<D, M, T>(u1, ib1, nbr, pb, J0, J1, J2, 0, 2 * (x0 & 1) - 1, a.sg);
    f += w1<T>() * nbv<D, M, T>(u1, ib1, nbr, pb, J0, J1, J2, 1, 2 * (x1 & 1) - 1, a.sg);
    if (D == 3) f += w1<T>() * nbv<D, M, T>(u1, ib1, nbr, pb, J0, J1, J2, 2, 2 * (x2 & 1) - 1, a.sg);
    size_t o = (size_t)fb * LY::V + q;
    u[o] = f + u[o];
}

// applydelta!'s field transfer (src/refinement.jl:339-370; interp! and
// restrict! of src/streamer.jl:191-221) from the old block layout (uo, its
// coarse-fine slabs ibo and neighbour table nbro) into the new one (un).
// Blocks that keep their (level, coordinate): moved to their new position;
// cp[k] = (old block, new block).
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_regrid_copy(T *__restrict__ un, const T *__restrict__ uo,
                                                    const int2 *__restrict__ cp, int n) {
    using LY = Lay<D, M>;
    const size_t gt = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int k = (int)(gt / LY::V);
    if (k >= n) return;
    const int q = (int)(gt - (size_t)k * LY::V);
    const int2 p = cp[k];
    un[(size_t)p.y * LY::V + q] = uo[(size_t)p.x * LY::V + q];
}

// New blocks: interp! (src/interp.jl:23-60, func = _first) from the parent's
// old values and its depth-1 ghosts, in k_interp_add's order of terms;
// ip[k] = (new block, old parent, subblock code).
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_regrid_interp(T *__restrict__ un, const T *__restrict__ uo,
                                                      const T *__restrict__ ibo, const int *__restrict__ nbro,
                                                      const int4 *__restrict__ ip, int n, LevelArgs<T> a) {
    using LY = Lay<D, M>;
    const size_t gt = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int k = (int)(gt / LY::V);
    if (k >= n) return;
    const int q = (int)(gt - (size_t)k * LY::V);
    int x0, x1, x2;
    LY::decode(q, x0, x1, x2);
    const int4 it = ip[k];
    const int pb = it.y, sb = it.z;
    const int J0 = (sb & 1) * LY::MH + (x0 >> 1);
    const int J1 = ((sb >> 1) & 1) * LY::MH + (x1 >> 1);
    const int J2 = (D == 3) ? ((sb >> 2) & 1) * LY::MH + (x2 >> 1) : 0;
    T f = w0<D, T>() * uo[(size_t)pb * LY::V + LY::sidx(J0, J1, J2)];
    f += w1<T>() * nbv<D, M, T>(uo, ibo, nbro, pb, J0, J1, J2, 0, 2 * (x0 & 1) - 1, a.sg);
    f += w1<T>() * nbv<D, M, T>(uo, ibo, nbro, pb, J0, J1, J2, 1, 2 * (x1 & 1) - 1, a.sg);
    if (D == 3) f += w1<T>() * nbv<D, M, T>(uo, ibo, nbro, pb, J0, J1, J2, 2, 2 * (x2 & 1) - 1, a.sg);
    un[(size_t)it.x * LY::V + q] = f;
}

// Removed blocks: restrict! (src/restrict.jl:5-26) into the parent's
// subblock, in k_restrict's order; rp[k] = (old block, new parent, subblock
// code).
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_regrid_restrict(T *__restrict__ un, const T *__restrict__ uo,
                                                        const int4 *__restrict__ rp, int n) {
    using LY = Lay<D, M>;
    constexpr int NS = LY::V / LY::NC;
    const size_t gt = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int k = (int)(gt / NS);
    if (k >= n) return;
    const int j = (int)(gt - (size_t)k * NS);
    const int j0 = j % LY::MH, j1 = (j / LY::MH) % LY::MH, j2 = (D == 3) ? j / (LY::MH * LY::MH) : 0;
    const int4 it = rp[k];
    T f = T(0);
#pragma unroll
    for (int c = 0; c < LY::NC; c++) {
        const int i0 = c & 1, i1 = (c >> 1) & 1, i2 = (c >> 2) & 1;
        f += uo[(size_t)it.x * LY::V + LY::sidx(2 * j0 + i0, 2 * j1 + i1, D == 3 ? 2 * j2 + i2 : 0)];
    }
    const int sb = it.z;
    const int X0 = (sb & 1) * LY::MH + j0, X1 = ((sb >> 1) & 1) * LY::MH + j1;
    const int X2 = (D == 3) ? ((sb >> 2) & 1) * LY::MH + j2 : 0;
    un[(size_t)it.y * LY::V + LY::sidx(X0, X1, X2)] = f / T(LY::NC);
}

// fill_ghost_interp! (src/connectivity.jl:251-258, src/blockfield.jl:416-434)
// for the depth-1 ghost layer: slot k holds the ghost slab of one coarse-fine
// face. The coarse layer adjacent to the face feeds the fine ghost layer next
// to the fine block's valid cells, i.e. child offset 1 on a low face and 0 on a
// high face in the face dimension. `a` describes the coarse level (mirror signs).
template <int D, int M, typename T, class X>
__device__ __forceinline__ void fill_interp_one(int gt, T *__restrict__ ib, const X x,
                                                const int *__restrict__ nbr, const int4 *__restrict__ slots,
                                                int slot0, int nslot, const LevelArgs<T> &a) {
    using LY = Lay<D, M>;
    int ls = gt / LY::F;
    if (ls >= nslot) return;
    int k = slot0 + ls;
    int t = gt - ls * LY::F;
    int4 sl = slots[k];  // (fine, face, coarse, subblock code)
    int dim = sl.y >> 1, dir = (sl.y & 1) ? 1 : -1;
    int pb = sl.z, sb = sl.w;
    int c[3] = {0, 0, 0};
    // tangential coordinates in increasing dimension order
    int ta = t % M, tb = t / M;
    if (dim == 0) { c[1] = ta; c[2] = tb; }
    else if (dim == 1) { c[0] = ta; c[2] = tb; }
    else { c[0] = ta; c[1] = tb; }
    int J[3] = {0, 0, 0}, i[3] = {0, 0, 0};
#pragma unroll
    for (int d = 0; d < D; d++) {
        int sbd = (sb >> d) & 1;
        if (d == dim) {
            J[d] = sbd * LY::MH + (dir < 0 ? LY::MH - 1 : 0);
            i[d] = dir < 0 ? 1 : 0;
        } else {
            J[d] = sbd * LY::MH + (c[d] >> 1);
            i[d] = c[d] & 1;
        }
    }
    T f = w0<D, T>() * x[(size_t)pb * LY::V + LY::sidx(J[0], J[1], J[2])];
#pragma unroll
    for (int j = 0; j < D; j++)
        f += w1<T>() * nbv<D, M, T>(x, ib, nbr, pb, J[0], J[1], J[2], j, 2 * i[j] - 1, a.sg);
    ib[(size_t)k * LY::F + t] = f;
}

template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_fill_interp(T *__restrict__ ib, const T *__restrict__ x,
                                                    const int *__restrict__ nbr, const int4 *__restrict__ slots,
                                                    int slot0, int nslot, LevelArgs<T> a) {
    fill_interp_one<D, M, T>(blockIdx.x * blockDim.x + threadIdx.x, ib, x, nbr, slots, slot0, nslot, a);
}

template <typename T> struct Vec16;
template <> struct Vec16<float> { using V = float4; };
template <> struct Vec16<double> { using V = double2; };

// Two independent steps of the V-cycle ascent in one launch: the first
// nwg_diff work groups form dst = a1 - a2 over n values (16 bytes
// per lane, n a multiple of 16 / sizeof(T), the arrays 16-byte aligned; dst
// may be a2), the rest refresh nslot coarse-fine ghost slabs
// (k_fill_interp). The slabs read another level than the difference writes.
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_diff_fill(T *dst, const T *a1, const T *a2, size_t n, unsigned nwg_diff,
                                                  T *__restrict__ ib, const T *__restrict__ x,
                                                  const int *__restrict__ nbr, const int4 *__restrict__ slots,
                                                  int slot0, int nslot, LevelArgs<T> a) {
    if (blockIdx.x < nwg_diff) {
        using V = typename Vec16<T>::V;
        constexpr int K = sizeof(V) / sizeof(T);
        const size_t i = ((size_t)blockIdx.x * WG + threadIdx.x) * K;
        if (i < n) {
            V p = *reinterpret_cast<const V *>(a1 + i);
            const V q = *reinterpret_cast<const V *>(a2 + i);
            T *pv = reinterpret_cast<T *>(&p);
            const T *qv = reinterpret_cast<const T *>(&q);
#pragma unroll
            for (int k = 0; k < K; k++) pv[k] = pv[k] - qv[k];
            *reinterpret_cast<V *>(dst + i) = p;
        }
    } else {
        fill_interp_one<D, M, T>((blockIdx.x - nwg_diff) * WG + threadIdx.x, ib, x, nbr, slots, slot0, nslot, a);
    }
}

// Sums of the residual partials, one work group per tree: the ranges
// rng[t nr .. (t + 1) nr) (int2: first, count) in order, each thread every
// SUM_NT-th partial with 16 loads in flight, then a halving tree. out is
// host memory that the device can write: no copy follows. (Two launches and a
// copy before: 12 us per norm on one tree, 8 on several.)
// One work group has a pass of SUM_PASS loads in flight and waits them out: on
// one tree of more than SUM_ONE partials the passes are work groups of a launch
// of their own (partial's tail as out), and the pieces' sums one more.
constexpr int SUM_NT = 1024, SUM_PASS = 16 * SUM_NT, SUM_ONE = 2 * SUM_PASS;
__global__ __launch_bounds__(SUM_NT) void k_sum_ranges(const double *partial, const int2 *__restrict__ rng, int nr,
                                                       double *out) {
    __shared__ double red[SUM_NT / 64];
    const int tid = threadIdx.x;
    double acc = 0.0;
    for (int k = 0; k < nr; k++) {
        const int2 r = rng[blockIdx.x * nr + k];
        const int end = r.x + r.y;
        for (int i = r.x + tid; i < end; i += 16 * SUM_NT) {
            double p[16];
#pragma unroll
            for (int j = 0; j < 16; j++) p[j] = i + j * SUM_NT < end ? partial[i + j * SUM_NT] : 0.0;
#pragma unroll
            for (int j = 0; j < 16; j++) acc += p[j];
        }
    }
#pragma unroll
    for (int w = 32; w > 0; w >>= 1) acc += __shfl_down(acc, w, 64);
    if ((tid & 63) == 0) red[tid >> 6] = acc;
    __syncthreads();
    if (tid >= SUM_NT / 64) return;
    acc = red[tid];
#pragma unroll
    for (int w = SUM_NT / 128; w > 0; w >>= 1) acc += __shfl_down(acc, w, SUM_NT / 64);
    if (tid == 0) out[blockIdx.x] = acc;
}

// ---- fused red-black sweep ----

// Work-group -> tile mapping that keeps consecutive tiles (Morton order) on one
// XCD: the hardware hands work group i to XCD i mod 8, so XCD x receives a
// contiguous range of tiles and neighbouring blocks meet in its L2.
__device__ __forceinline__ int xcd_remap(int i, int G) {
    constexpr int NX = 8;
    int x = i % NX, local = i / NX;
    int per = G / NX, rem = G % NX;
    return (x < rem) ? x * (per + 1) + local : rem * (per + 1) + (x - rem) * per + local;
}

// LDS tile of G^D blocks of M^D cells with a depth-1 halo: cells -1 .. G M.
// Rows hold R >= S entries (R > S pads rows against LDS bank conflicts).
// Helpers that work on one block of a tile take a pointer offset to that
// block's origin (the tile index is linear in the coordinates).
template <int D, int M, int G = 1, int R = G * M + 2>
struct Tile {
    static constexpr int S = G * M + 2;
    static_assert(R >= S, "row pitch below the row length");
    static constexpr int SZ = (D == 2) ? R * S : R * S * S;
    __device__ static __forceinline__ int at(int x, int y, int z) {
        return (x + 1) + R * ((y + 1) + (D == 3 ? S * (z + 1) : 0));
    }
    __device__ static __forceinline__ int at3(const int *c) { return at(c[0], c[1], D == 3 ? c[2] : 0); }
    __host__ __device__ static constexpr int stride(int d) { return d == 0 ? 1 : (d == 1 ? R : R * S); }
    // offset of block k of a G = 2 group (k's bit d = upper half along d)
    __device__ static __forceinline__ int origin(int k) {
        return M * ((k & 1) + R * (((k >> 1) & 1) + (D == 3 ? S * ((k >> 2) & 1) : 0)));
    }
};

// Per-block halo table used by the tiled kernels: the block's own 2D face
// entries, then for each face f the neighbour-table entries of the block across
// f on its 2(D-1) side faces (tangential dimensions in increasing order, low
// side first); unused when face f is not a same-level face.
template <int D>
struct Halo {
    static constexpr int ND = 2 * D;
    static constexpr int NS = 2 * (D - 1);
    static constexpr int N = ND + ND * NS;
};

// Stencil of the tile cell at p, all neighbours in the tile. RD is the radial
// dimension (cylindrical geometry) or -1; terms in the reference's order.
template <int D, int M, typename T, int RD, class TL = Tile<D, M>>
__device__ __forceinline__ T tstencil(const T *t, int p, T own, T cc, T wm, T wp) {
    T v = T(0);
#pragma unroll
    for (int d = D - 1; d >= 0; d--) {
        if (d == RD) v += wm * t[p - TL::stride(d)];
        else v += t[p - TL::stride(d)];
    }
    v += cc * own;
#pragma unroll
    for (int d = 0; d < D; d++) {
        if (d == RD) v += wp * t[p + TL::stride(d)];
        else v += t[p + TL::stride(d)];
    }
    return v;
}

// Radial weights in two load round trips, which the kernels below issue with
// the trips they make anyway (the block's coordinate with the interior, the
// weights with the halo) instead of waiting for both before the arithmetic:
// the radial index J of a block's cell 0, then the weights of a cell at J + cr.
// With them and the per-block parameters read directly, the launches of a 2D
// cylindrical forest of 27 trees lose about one microsecond in six.
template <int D, int M, int RD>
__device__ __forceinline__ int rbase(const int *__restrict__ coord, int blk) {
    return RD >= 0 ? M * (coord[blk * D + RD] - 1) + 1 : 0;
}
template <typename T, int RD>
__device__ __forceinline__ void rweights(const LevelArgs<T> &a, int J, T &wm, T &wp) {
    wm = T(1);
    wp = T(1);
    if (RD >= 0) {
        wm = a.wm[J];
        wp = a.wp[J];
    }
}

// Depth-1 halo cell number t of face F (a compile-time face) of block blk:
// its tile position, and its value (neighbour cell, mirror of the facing cell,
// or frozen slab).
template <int D, int M, int F, class TL = Tile<D, M>>
__device__ __forceinline__ int halo_at(int t) {
    constexpr int DIM = F >> 1, DIR = (F & 1) ? 1 : -1;
    int c[3] = {0, 0, 0};
    int ta = t % M, tb = t / M;
    if (DIM == 0) { c[1] = ta; c[2] = tb; }
    else if (DIM == 1) { c[0] = ta; c[2] = tb; }
    else { c[0] = ta; c[1] = tb; }
    c[DIM] = DIR > 0 ? M : -1;
    return TL::at(c[0], c[1], c[2]);
}

template <int D, int M, typename T, int F, class X>
__device__ __forceinline__ T halo_value(int e, int blk, int t, const X x, const T *__restrict__ ib, T sg) {
    using LY = Lay<D, M>;
    constexpr int DIM = F >> 1, DIR = (F & 1) ? 1 : -1;
    int c[3] = {0, 0, 0};
    int ta = t % M, tb = t / M;
    if (DIM == 0) { c[1] = ta; c[2] = tb; }
    else if (DIM == 1) { c[0] = ta; c[2] = tb; }
    else { c[0] = ta; c[1] = tb; }
    if (e >= 0) {
        c[DIM] = DIR > 0 ? 0 : M - 1;
        return x[(size_t)e * LY::V + LY::sidx(c[0], c[1], c[2])];
    } else if (e == NB_BOUNDARY) {
        c[DIM] = DIR > 0 ? M - 1 : 0;
        return sg * x[(size_t)blk * LY::V + LY::sidx(c[0], c[1], c[2])];
    }
    return ib[(size_t)nb_slot(e) * LY::F + t];
}

template <int D, int M, typename T, int F, class TL = Tile<D, M>>
__device__ __forceinline__ void halo_cell(T *tile, int e, int blk, int t, const T *__restrict__ x,
                                          const T *__restrict__ ib, T sg) {
    tile[halo_at<D, M, F, TL>(t)] = halo_value<D, M, T, F>(e, blk, t, x, ib, sg);
}

// face number f known only at run time (uniform per wave where the work
// layout allows it)
#define SRMG_FACE_SWITCH(f, EXPR)                \
    switch (f) {                                 \
        case 0: { constexpr int FF = 0; EXPR; } break; \
        case 1: { constexpr int FF = 1; EXPR; } break; \
        case 2: { constexpr int FF = 2; EXPR; } break; \
        case 3: { constexpr int FF = 3; EXPR; } break; \
        case 4: { constexpr int FF = (D == 3 ? 4 : 3); EXPR; } break; \
        default: { constexpr int FF = (D == 3 ? 5 : 3); EXPR; } break; \
    }

template <int D, int M, typename T, class TL = Tile<D, M>>
__device__ __forceinline__ void halo_switch(T *tl, int e, int f, int blk, int t, const T *__restrict__ x,
                                            const T *__restrict__ ib, const T *sg) {
    SRMG_FACE_SWITCH(f, (halo_cell<D, M, T, FF, TL>(tl, e, blk, t, x, ib, sg[FF])))
}

template <int D, int M, typename T, class X>
__device__ __forceinline__ T halo_value_sw(int f, int e, int blk, int t, const X x, const T *__restrict__ ib,
                                           const T *sg) {
    T v = T(0);
    SRMG_FACE_SWITCH(f, (v = halo_value<D, M, T, FF>(e, blk, t, x, ib, sg[FF])))
    return v;
}

template <int D, int M, class TL>
__device__ __forceinline__ int halo_at_sw(int f, int t) {
    int p = 0;
    SRMG_FACE_SWITCH(f, (p = halo_at<D, M, FF, TL>(t)))
    return p;
}

// Neighbour face-layer cells recomputed by the fused sweep: for the face
// normal to DIM on side dir, the neighbour's first-half-sweep cells of its
// layer facing this block, numbered tq in [0, F/2).
template <int D, int M, typename T, int DIM, class TL = Tile<D, M>>
struct RecFace {
    using LY = Lay<D, M>;
    using HT = Halo<D>;
    static constexpr int DA = DIM == 0 ? 1 : 0;
    static constexpr int DB = DIM == 2 ? 1 : 2;
    static constexpr int NS = 2 * (D - 1);

    __device__ static __forceinline__ void cell(int dir, int tq, int *cB) {
        constexpr int MH = LY::MH;
        int w = dir > 0 ? 0 : M - 1;
        int tb = (D == 3) ? tq / MH : 0;
        cB[0] = cB[1] = cB[2] = 0;
        cB[DIM] = w;
        cB[DA] = 2 * (tq % MH) + ((1 + w + tb + D) & 1);
        if (D == 3) cB[DB] = tb;
    }

    // operands outside the tile: one layer deeper in the neighbour, its
    // right-hand side, and its ghosts across its side faces. ZIN: the field
    // and its ghost slabs are zero (only the right-hand side is read).
    template <bool ZIN = false>
    __device__ static __forceinline__ void prefetch(int dir, int tq, int e, const int *gs, const T *__restrict__ x,
                                                    const T *__restrict__ b, const T *__restrict__ ib, T &rd, T &rb,
                                                    T *rg) {
        int cB[3];
        cell(dir, tq, cB);
        rb = b[(size_t)e * LY::V + LY::sidx(cB[0], cB[1], cB[2])];
        if constexpr (ZIN) {
            rd = T(0);
#pragma unroll
            for (int k = 0; k < NS; k++) rg[k] = T(0);
            return;
        }
        int c2[3] = {cB[0], cB[1], cB[2]};
        c2[DIM] = dir > 0 ? 1 : M - 2;
        rd = x[(size_t)e * LY::V + LY::sidx(c2[0], c2[1], c2[2])];
        // one guarded load per side face: the neighbour's cell (same level)
        // or the frozen slab (coarse-fine); nothing at a domain boundary or
        // off the edge of the face
#pragma unroll
        for (int k = 0; k < NS; k++) {
            const int dd = (k < 2) ? DA : DB;
            const int side = k & 1;
            const int g = gs[k];
            int c3[3] = {cB[0], cB[1], cB[2]};
            c3[dd] = side ? 0 : M - 1;
            const size_t o = g >= 0 ? (size_t)g * LY::V + LY::sidx(c3[0], c3[1], c3[2])
                                    : (size_t)max(nb_slot(g), 0) * LY::F + LY::faceidx(dd, cB[0], cB[1], cB[2]);
            const T *src = g >= 0 ? x : ib;
            rg[k] = T(0);
            if (cB[dd] == (side ? M - 1 : 0) && g != NB_BOUNDARY) rg[k] = src[o];
        }
    }

    // first-half-sweep value of the neighbour cell, written into this block's halo
    // (wm, wp: the radial weights at that cell, radial_index of this block's J)
    template <int RD>
    __device__ static __forceinline__ int radial_index(int dir, int tq, int J) {
        int cB[3];
        cell(dir, tq, cB);
        return RD < 0 ? 0 : J + (DIM == RD ? dir * M : 0) + cB[RD < 0 ? 0 : RD];
    }
    template <int RD>
    __device__ static __forceinline__ void compute(int dir, int tq, const int *gs, T *tile, T wm, T wp,
                                                   const LevelArgs<T> &a, const BP<T> &bp, T rd, T rb, const T *rg) {
        int cB[3];
        cell(dir, tq, cB);
        int ch[3] = {cB[0], cB[1], cB[2]};
        ch[DIM] = dir > 0 ? M : -1;
        const int ph = TL::at(ch[0], ch[1], ch[2]);
        const T xo = tile[ph];
        T nbm[3], nbp[3];
        // across the shared face: this block's cell; one layer deeper: rd
        const int pa = TL::at(DIM == 0 ? (dir > 0 ? M - 1 : 0) : cB[0], DIM == 1 ? (dir > 0 ? M - 1 : 0) : cB[1],
                              DIM == 2 ? (dir > 0 ? M - 1 : 0) : cB[2]);
        if (dir > 0) { nbm[DIM] = tile[pa]; nbp[DIM] = rd; }
        else { nbm[DIM] = rd; nbp[DIM] = tile[pa]; }
        // along the face layer: in the halo; off the edge of the face: the
        // prefetched ghost, or the mirror at a domain boundary (the tile
        // position read for an off-edge cell is inside the tile and unused)
#pragma unroll
        for (int k = 0; k < NS; k++) {
            const int dd = (k < 2) ? DA : DB;
            const int side = k & 1;
            const int cc = cB[dd] + (side ? 1 : -1);
            const T vt = tile[ph + (side ? 1 : -1) * TL::stride(dd)];
            const T vg = (gs[k] == NB_BOUNDARY) ? a.sg[2 * dd + side] * xo : rg[k];
            const T v = (cc >= 0 && cc < M) ? vt : vg;
            if (side) nbp[dd] = v; else nbm[dd] = v;
        }
        T Lx = T(0);
#pragma unroll
        for (int dd = D - 1; dd >= 0; dd--) {
            if (dd == RD) Lx += wm * nbm[dd];
            else Lx += nbm[dd];
        }
        Lx += bp.cc * xo;
#pragma unroll
        for (int dd = 0; dd < D; dd++) {
            if (dd == RD) Lx += wp * nbp[dd];
            else Lx += nbp[dd];
        }
        tile[ph] = fma_t<T>(bp.nwc, fma_t<T>(bp.s, rb, Lx), xo);
    }
};

// One full gauss_seidel_iter! sweep (src/multigrid.jl:250-265: RedBlack{0} on
// all blocks, copy/boundary ghost fill, RedBlack{1}, fill) in one launch.
// Reads ui, writes uo (ping-pong, so neighbours always see the old values).
// Each work group stages BPW blocks with a depth-1 face halo in LDS. The
// second half-sweep needs the neighbours' face-layer cells after the first
// half-sweep; the work group recomputes them from the same inputs with the
// same operations as their owners, so the result is identical to the
// two-launch form. Boundary ghosts mirror the cell they face, and coarse-fine
// ghosts stay frozen during smoothing (src/multigrid.jl:256-263).
// Memory round trips before compute: (interior, b, halo table), then (halo
// cells, recompute operands). Faces are compile-time constants in unrolled
// loops, so work that is uniform per face carries no per-lane selects.
template <int D, int M, typename T, int BPW, int NT, int RD>
__global__ __launch_bounds__(NT) void k_gs_sweep(T *__restrict__ uo, const T *__restrict__ ui,
                                                 const T *__restrict__ b, const T *__restrict__ ib,
                                                 const int *__restrict__ htab, const int *__restrict__ coord,
                                                 LevelArgs<T> a) {
    using LY = Lay<D, M>;
    using TL = Tile<D, M>;
    using HT = Halo<D>;
    constexpr int F = LY::F, V = LY::V, H = LY::H, F2 = F / 2, ND = 2 * D, NS = 2 * (D - 1);
    static_assert((BPW * H) % NT == 0, "cells per colour must be a multiple of the work-group size");
    constexpr int CPT = BPW * H / NT;
    constexpr int NREC = BPW * ND * F2;
    constexpr int RPT = (NREC + NT - 1) / NT;
    constexpr int NHALO = BPW * ND * F;
    __shared__ T tile[BPW * TL::SZ];
    __shared__ int tab[BPW * HT::N];
    __shared__ BP<T> prm[BPW];
    const int lb0 = xcd_remap(blockIdx.x, gridDim.x) * BPW;
    const int tid = threadIdx.x;
    const int nloc = min(BPW, a.nblk - lb0);
    const int blk0 = a.blk0 + lb0;

    // round trip 1: interior cells, own right-hand side, halo tables, parameters
    T ux[CPT][2], bo[CPT], be[CPT];
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        int i = tid + k * NT, lb = i / H, r = i - lb * H;
        ux[k][0] = ux[k][1] = bo[k] = be[k] = T(0);
        if (lb < nloc) {
            size_t o = (size_t)(blk0 + lb) * V + r;
            ux[k][0] = ui[o];
            ux[k][1] = ui[o + H];
            bo[k] = b[o];
            be[k] = b[o + H];
        }
    }
    constexpr int TP = (BPW * HT::N + NT - 1) / NT;
    int tv[TP];
#pragma unroll
    for (int k = 0; k < TP; k++) {
        const int i = tid + k * NT;
        tv[k] = i < nloc * HT::N ? htab[(size_t)blk0 * HT::N + i] : 0;
    }
    BP<T> bpl{};
    if (tid < nloc) bpl = bparams(a, blk0 + tid);
    // radial index of the thread's cells' blocks and of its recompute items' blocks
    int Jc[CPT], Jr[RPT];
#pragma unroll
    for (int k = 0; k < CPT; k++) Jc[k] = rbase<D, M, RD>(coord, blk0 + min((tid + k * NT) / H, nloc - 1));
#pragma unroll
    for (int k = 0; k < RPT; k++) Jr[k] = rbase<D, M, RD>(coord, blk0 + min((tid + k * NT) / (ND * F2), nloc - 1));
#pragma unroll
    for (int k = 0; k < TP; k++) {
        const int i = tid + k * NT;
        if (i < nloc * HT::N) tab[i] = tv[k];
    }
    if (tid < nloc) prm[tid] = bpl;
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        int i = tid + k * NT, lb = i / H, r = i - lb * H;
        if (lb < nloc) {
            int x, y, z;
            LY::decode(r, x, y, z);
            tile[lb * TL::SZ + TL::at(x, y, z)] = ux[k][0];
            LY::decode(H + r, x, y, z);
            tile[lb * TL::SZ + TL::at(x, y, z)] = ux[k][1];
        }
    }
    __syncthreads();

    // round trip 2: halo cells (stored into the tile once every load of the
    // round trip is issued) ...
    constexpr int PH = (NHALO + NT - 1) / NT;
    T hv[PH];
#pragma unroll
    for (int j = 0; j < PH; j++) {
        const int i = tid + NT * j, lb = min(i / (ND * F), BPW - 1), rem = i - lb * (ND * F);
        const int f = min(rem / F, ND - 1), t = rem - f * F;
        hv[j] = T(0);
        if (i < NHALO && lb < nloc) hv[j] = halo_value_sw<D, M, T>(f, tab[lb * HT::N + f], blk0 + lb, t, ui, ib, a.sg);
    }
    // the radial weights of the thread's cells
    T wc[CPT][2][2];
#pragma unroll
    for (int k = 0; k < CPT; k++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            int x, y, z;
            LY::decode(h * H + (tid + k * NT) % H, x, y, z);
            rweights<T, RD>(a, Jc[k] + (RD == 0 ? x : y), wc[k][h][0], wc[k][h][1]);
        }
    // ... and the operands of the recomputed neighbour cells
    T rd[RPT], rb[RPT], rg[RPT][NS], rw[RPT][2];
    int rj[RPT];
#pragma unroll
    for (int k = 0; k < RPT; k++) {
        int j = tid + k * NT;
        rj[k] = -1;
        rd[k] = rb[k] = rw[k][0] = rw[k][1] = T(0);
        if (j >= NREC) continue;
        int lb = j / (ND * F2), rem = j - lb * (ND * F2);
        int f = rem / F2, tq = rem - f * F2;
        if (lb >= nloc) continue;
        const int *tb = tab + lb * HT::N, *gs = tb + HT::ND + f * HT::NS;
        int e = tb[f];
        if (e < 0) continue;
        rj[k] = j;
        int dim = f >> 1, dir = (f & 1) ? 1 : -1;
        const int J = dim == 0 ? RecFace<D, M, T, 0>::template radial_index<RD>(dir, tq, Jr[k])
                               : RecFace<D, M, T, 1>::template radial_index<RD>(dir, tq, Jr[k]);
        rweights<T, RD>(a, J, rw[k][0], rw[k][1]);
        if (dim == 0) RecFace<D, M, T, 0>::prefetch(dir, tq, e, gs, ui, b, ib, rd[k], rb[k], rg[k]);
        else if (dim == 1) RecFace<D, M, T, 1>::prefetch(dir, tq, e, gs, ui, b, ib, rd[k], rb[k], rg[k]);
        else RecFace<D, M, T, (D == 3 ? 2 : 1)>::prefetch(dir, tq, e, gs, ui, b, ib, rd[k], rb[k], rg[k]);
    }
#pragma unroll
    for (int j = 0; j < PH; j++) {
        const int i = tid + NT * j, lb = min(i / (ND * F), BPW - 1), rem = i - lb * (ND * F);
        const int f = min(rem / F, ND - 1), t = rem - f * F;
        if (i < NHALO && lb < nloc) tile[lb * TL::SZ + halo_at_sw<D, M, TL>(f, t)] = hv[j];
    }
    __syncthreads();

    // first half-sweep: cells with odd global index sum
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        int i = tid + k * NT, lb = i / H, r = i - lb * H;
        if (lb < nloc) {
            int x, y, z;
            LY::decode(r, x, y, z);
            int p = lb * TL::SZ + TL::at(x, y, z);
            const BP<T> bp = prm[lb];
            T Lu = tstencil<D, M, T, RD>(tile, p, ux[k][0], bp.cc, wc[k][0][0], wc[k][0][1]);
            ux[k][0] = fma_t<T>(bp.nwc, fma_t<T>(bp.s, bo[k], Lu), ux[k][0]);
            tile[p] = ux[k][0];
        }
    }
    // the same half-sweep on the neighbours' face-layer cells
#pragma unroll
    for (int k = 0; k < RPT; k++) {
        int j = rj[k];
        if (j < 0) continue;
        int lb = j / (ND * F2), rem = j - lb * (ND * F2);
        int f = rem / F2, tq = rem - f * F2;
        const int *tb = tab + lb * HT::N, *gs = tb + HT::ND + f * HT::NS;
        T *tl = tile + lb * TL::SZ;
        int dim = f >> 1, dir = (f & 1) ? 1 : -1;
        const BP<T> bp = prm[lb];
        const T wm = rw[k][0], wp = rw[k][1];
        if (dim == 0)
            RecFace<D, M, T, 0>::template compute<RD>(dir, tq, gs, tl, wm, wp, a, bp, rd[k], rb[k], rg[k]);
        else if (dim == 1)
            RecFace<D, M, T, 1>::template compute<RD>(dir, tq, gs, tl, wm, wp, a, bp, rd[k], rb[k], rg[k]);
        else
            RecFace<D, M, T, (D == 3 ? 2 : 1)>::template compute<RD>(dir, tq, gs, tl, wm, wp, a, bp, rd[k], rb[k],
                                                                     rg[k]);
    }
    __syncthreads();

    // second half-sweep: the remaining cells
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        int i = tid + k * NT, lb = i / H, r = i - lb * H;
        if (lb < nloc) {
            int x, y, z;
            LY::decode(H + r, x, y, z);
            int p = lb * TL::SZ + TL::at(x, y, z);
            const BP<T> bp = prm[lb];
            T Lu = tstencil<D, M, T, RD>(tile, p, ux[k][1], bp.cc, wc[k][1][0], wc[k][1][1]);
            size_t o = (size_t)(blk0 + lb) * V + r;
            uo[o] = ux[k][0];
            uo[o + H] = fma_t<T>(bp.nwc, fma_t<T>(bp.s, be[k], Lu), ux[k][1]);
        }
    }
}

// The blocks around each block of a 2D level, for k_gs_sweep2: in nine[45 blk],
// the same-level block at offset (n % 3 - 1, n / 3 - 1), -1 where there is none
// or -2 beyond the domain (n = 0 .. 8; a diagonal one by way of a face
// neighbour, as values reach this block), then the neighbour-table entries of
// each.
constexpr int NINE = 45;
__global__ __launch_bounds__(WG) void k_nine(int *__restrict__ nine, const int *__restrict__ nbr, int nb) {
    const int64_t gt = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int blk = (int)(gt / NINE), i = (int)(gt - (int64_t)blk * NINE);
    if (blk >= nb) return;
    const int n = i < 9 ? i : (i - 9) / 4, dx = n % 3, dy = n / 3;
    int e = blk;
    if (dx != 1 && dy != 1) {
        const int ex = nbr[(size_t)blk * 4 + (dx >> 1)], ey = nbr[(size_t)blk * 4 + 2 + (dy >> 1)];
        e = ex >= 0 ? nbr[(size_t)ex * 4 + 2 + (dy >> 1)] : (ey >= 0 ? nbr[(size_t)ey * 4 + (dx >> 1)] : -2);
    } else if (dx != 1) {
        e = nbr[(size_t)blk * 4 + (dx >> 1)];
    } else if (dy != 1) {
        e = nbr[(size_t)blk * 4 + 2 + (dy >> 1)];
    }
    if (e < 0) e = e == NB_BOUNDARY ? -2 : -1;
    nine[gt] = i < 9 ? e : (e >= 0 ? nbr[(size_t)e * 4 + (i - 9) % 4] : NB_BOUNDARY);
}

// Two sweeps of a 2D level in one launch: k_gs_sweep's scheme with a deeper
// halo. A work group takes a block with the cells within four steps of it and
// runs the four half-sweeps there, each on the cells within one step less
// (the neighbours' cells by the operations of their owners), so the result is
// that of two launches. On a small level a launch is its round trips and costs
// the same whatever it does; on a large one the two sweeps read the field once.
// Two sweeps of 16 to 256 blocks of 16^2 in FP64: 10.5 -> 4.8 us, of 1,024: 11.2
// -> 6.2, of 4,096: 16.0 -> 12.0, of 16,384: 53.8 -> 33.6 (3.2 TB/s of what one
// pass over u, b and u must move; the halo's arithmetic bounds it).
//
// Ghosts: a boundary ghost is the cell itself times the face's sign. Frozen
// slab values stand in the tile where they are seen, those seen across a y face
// in a second tile, since beyond a concave corner of the level one place is
// two blocks' ghost.
//
// Of a large level it is the index arithmetic that costs: the cells of each
// thread are a table (Gs2Table), and what only blocks at a face of the level
// need is behind a branch on the wave's view of the surroundings.
template <int M>
constexpr int GS2_THREADS = M == 16 ? 256 : 128;
// What thread tid does: cells 0 and 1 of half-sweeps k and k + 2, and cell 2 of
// the ring four steps from the block (read only). Of each: the place co in its
// block and cq in the tile (by row, the columns of one colour together: a
// half-sweep reads the other), the offset cn of its block, the distance cd
// from this one (7: no such cell); of the first two cells the offsets of the
// blocks of the four cells they read.
template <int M>
struct Gs2Table {
    static constexpr int HD = 4, W = M + 2 * HD, WH = W / 2, NX = M / 2 + 3, NRING = 4 * M + 12;
    struct E {
        uint32_t q[4];  // co, cq: 12 bits each (cells 0, 1, 2); co of cell k at 12 k of q[0..1] as 64 bits, cq of q[2..3]
        uint32_t c;     // cn: 4 bits each; cd: 3 bits each from bit 12; x even: bits 24, 25
        uint32_t r;     // 4 bits each: cell k, face f at 4 (4 k + f)
        uint32_t pad[2];
    } e[GS2_THREADS<M>];
    static constexpr int side(int c) { return c < 0 ? 0 : (c >= M ? 2 : 1); }
    static constexpr int over(int c) { return c < 0 ? -c : (c >= M ? c - M + 1 : 0); }
    static constexpr int pos(int x, int y) { return ((y + HD) * 2 + ((x + y) & 1)) * WH + ((x + HD) >> 1); }
    constexpr Gs2Table() : e() {
        static_assert(NX * (M + 6) <= GS2_THREADS<M> && NRING <= GS2_THREADS<M> && W * W < 4096 && HD <= M,
                      "work of each thread");
        for (int t = 0; t < GS2_THREADS<M>; t++) {
            uint64_t co = 0, cq = 0;
            uint32_t c = 0, r = 0;
            for (int k = 0; k < 3; k++) {
                int x = 0, y = t / NX - 3;
                bool in = y < M + 3;
                if (k < 2) {
                    x = 2 * (t % NX) - 3 + ((y + k) & 1);
                    in = in && over(x) + over(y) < HD;
                } else {
                    const int f = t / M, q = t % M, j = t - 4 * M, dx = j % 3 + 1;
                    x = f == 0 ? -HD : (f == 1 ? M - 1 + HD : q);
                    y = f == 2 ? -HD : (f == 3 ? M - 1 + HD : q);
                    if (f >= 4) {
                        x = (j / 3) & 1 ? M - 1 + dx : -dx;
                        y = (j / 3) & 2 ? M - 1 + HD - dx : dx - HD;
                    }
                    in = t < NRING;
                }
                if (!in) {
                    c |= 7u << (12 + 3 * k);
                    continue;
                }
                const int bx = x - M * (side(x) - 1), by = y - M * (side(y) - 1);
                const int odd = (bx + by) & 1;  // Lay<2, M>::sidx
                co |= (uint64_t)((odd ? 0 : M * M / 2) + (bx >> 1) + M / 2 * by) << (12 * k);
                cq |= (uint64_t)pos(x, y) << (12 * k);
                c |= (uint32_t)(side(x) + 3 * side(y)) << (4 * k);
                c |= (uint32_t)(over(x) + over(y)) << (12 + 3 * k);
                if (k == 2) continue;
                if (!(x & 1)) c |= 1u << (24 + k);
                for (int f = 0; f < 4; f++) {
                    const int nx = x + (f == 0 ? -1 : (f == 1 ? 1 : 0)), ny = y + (f == 2 ? -1 : (f == 3 ? 1 : 0));
                    r |= (uint32_t)(side(nx) + 3 * side(ny)) << (4 * (4 * k + f));
                }
            }
            e[t].q[0] = (uint32_t)co;
            e[t].q[1] = (uint32_t)(co >> 32);
            e[t].q[2] = (uint32_t)cq;
            e[t].q[3] = (uint32_t)(cq >> 32);
            e[t].c = c;
            e[t].r = r;
        }
    }
};
template <int M>
__device__ const Gs2Table<M> GS2_TABLE{};

template <int M, typename T, int RD>
__global__ __launch_bounds__(GS2_THREADS<M>) void k_gs_sweep2(T *__restrict__ uo, const T *__restrict__ ui,
                                                              const T *__restrict__ b, const T *__restrict__ ib,
                                                              const int *__restrict__ nine,
                                                              const int *__restrict__ coord, LevelArgs<T> a) {
    using LY = Lay<2, M>;
    using TB = Gs2Table<M>;
    constexpr int HD = TB::HD, W = TB::W, WH = TB::WH;
    __shared__ T t[2 * W * W];  // the tile, then the one seen across y faces
    __shared__ int nn[NINE];
    const int tid = threadIdx.x, blk = a.blk0 + xcd_remap(blockIdx.x, gridDim.x);

    // round trip 1: the block's surroundings and parameters, this thread's cells
    const uint4 q4 = *reinterpret_cast<const uint4 *>(GS2_TABLE<M>.e[tid].q);
    const uint2 q2 = *reinterpret_cast<const uint2 *>(&GS2_TABLE<M>.e[tid].c);
    int nv = 0;
    if (tid < NINE) nv = nine[(size_t)blk * NINE + tid];
    const BP<T> bp = bparams(a, blk);
    const int J = rbase<2, M, RD>(coord, blk);
    const uint64_t qo = q4.x | (uint64_t)q4.y << 32, qq = q4.z | (uint64_t)q4.w << 32;
    int co[3], cq[3], cd[3], e[3];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        co[k] = (int)(qo >> (12 * k)) & 4095;
        cq[k] = (int)(qq >> (12 * k)) & 4095;
        cd[k] = (int)(q2.x >> (12 + 3 * k)) & 7;
    }
    if (tid < NINE) nn[tid] = nv;
    __syncthreads();

    // round trip 2: the cells, the radial weights. miss, dom: the offsets
    // without a block, and beyond the domain
    const int lane = tid & 63, ns = nn[lane < 9 ? lane : 4];
    const unsigned miss = (unsigned)__ballot(ns < 0) & 511u, dom = (unsigned)__ballot(ns == -2) & 511u;
    T v[3], vb[2], wm[2] = {T(1), T(1)}, wp[2] = {T(1), T(1)};
    const int tn[2] = {2 * (tid % TB::NX) - 3, tid / TB::NX - 3};
#pragma unroll
    for (int k = 0; k < 3; k++) {
        v[k] = T(0);
        if (k < 2) vb[k] = T(0);
        e[k] = -1;
        if (cd[k] == 7) continue;
        e[k] = nn[q2.x >> (4 * k) & 15];
        if (e[k] < 0) continue;
        const size_t o = (size_t)e[k] * LY::V + co[k];
        v[k] = ui[o];
        if (k < 2) {
            vb[k] = b[o];
            rweights<T, RD>(a, J + (RD == 0 ? tn[0] + ((tn[1] + k) & 1) : tn[1]), wm[k], wp[k]);
        }
    }
    // the faces of the two cells beyond which there is no block, or no domain
    unsigned fm = 0, fd = 0;
    if (miss) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const unsigned n = q2.y >> (4 * j) & 15;
            fm |= (miss >> n & 1) << j;
            fd |= (dom >> n & 1) << j;
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            if (cd[k] == 7 || e[k] >= 0) continue;
            // a slab cell, seen from the column beside (across its face fx) or the row beside
            const int q = cq[k], h = q % WH, yy = q / (2 * WH), y = yy - HD;
            const int x = 2 * h - HD + ((q / WH + y) & 1);
            const int n = q2.x >> (4 * k) & 15, sx = n % 3, sy = n / 3;
            const int nx = x == 0 ? 0 : (x == -1 || x == M ? 1 : (x == M - 1 ? 2 : 3));
            const int fx = x == 0 || x == M ? 1 : 0;
            const int ny = y == 0 ? 0 : (y == -1 || y == M ? 1 : (y == M - 1 ? 2 : 3));
            const int fy = y == 0 || y == M ? 3 : 2;
            const int g0 = nx < 3 ? nn[9 + 4 * (nx + 3 * sy) + fx] : NB_BOUNDARY;
            const int g1 = ny < 3 ? nn[9 + 4 * (sx + 3 * ny) + fy] : NB_BOUNDARY;
            if (g0 < NB_BOUNDARY) v[k] = ib[(size_t)nb_slot(g0) * LY::F + y - M * (sy - 1)];
            if (g1 < NB_BOUNDARY) t[W * W + q] = ib[(size_t)nb_slot(g1) * LY::F + x - M * (sx - 1)];
        }
    }
#pragma unroll
    for (int k = 0; k < 3; k++)
        if (cd[k] != 7) t[cq[k]] = v[k];
    __syncthreads();
    // where the four cells are: beside, in the other colour's half of the row
    int px[2], ym[2], yp[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int r = cq[k] + (k == 0 ? -WH : WH);
        px[k] = r - (int)(q2.x >> (24 + k) & 1);
        ym[k] = r - 2 * WH + (fm >> (4 * k + 2) & 1 ? W * W : 0);
        yp[k] = r + 2 * WH + (fm >> (4 * k + 3) & 1 ? W * W : 0);
    }
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const int k = p & 1;
        if (e[k] >= 0 && cd[k] < HD - p) {
            const T o = v[k];
            T xa = t[px[k]], xb = t[px[k] + 1], ya = t[ym[k]], yb = t[yp[k]];
            if (dom) {
                if (fd >> (4 * k) & 1) xa = a.sg[0] * o;
                if (fd >> (4 * k) & 2) xb = a.sg[1] * o;
                if (fd >> (4 * k) & 4) ya = a.sg[2] * o;
                if (fd >> (4 * k) & 8) yb = a.sg[3] * o;
            }
            T Lu = T(0);
            if (RD == 1) Lu += wm[k] * ya;
            else Lu += ya;
            if (RD == 0) Lu += wm[k] * xa;
            else Lu += xa;
            Lu += bp.cc * o;
            if (RD == 0) Lu += wp[k] * xb;
            else Lu += xb;
            if (RD == 1) Lu += wp[k] * yb;
            else Lu += yb;
            v[k] = fma_t<T>(bp.nwc, fma_t<T>(bp.s, vb[k], Lu), o);
            if (p < 3) t[cq[k]] = v[k];
        }
        if (p < 3) lds_barrier();
    }
#pragma unroll
    for (int k = 0; k < 2; k++)
        if (cd[k] == 0) uo[(size_t)blk * LY::V + co[k]] = v[k];
}

// k_gs_sweep on sibling groups: the 2^D children of one parent (consecutive
// in the Morton order of a level, always created together) form one
// (2M)^D tile. The faces between siblings need no halo and no recompute; the
// group's exterior faces are handled per block exactly as in k_gs_sweep (own
// halo-table entries, neighbour recompute from the same inputs), so the result
// is bitwise the same. One group per work group.
template <int D, int M, typename T, int NT, int RD>
__global__ __launch_bounds__(NT) void k_gs_sweep_group(T *__restrict__ uo, const T *__restrict__ ui,
                                                       const T *__restrict__ b, const T *__restrict__ ib,
                                                       const int *__restrict__ htab, const int *__restrict__ coord,
                                                       LevelArgs<T> a) {
    using LY = Lay<D, M>;
    using TL = Tile<D, M, 2>;
    using HT = Halo<D>;
    constexpr int NB = 1 << D;
    constexpr int F = LY::F, V = LY::V, H = LY::H, F2 = F / 2, NS = 2 * (D - 1);
    static_assert((NB * H) % NT == 0, "cells per colour must be a multiple of the work-group size");
    constexpr int CPT = NB * H / NT;
    constexpr int NREC = NB * D * F2;  // exterior faces: D per block
    constexpr int RPT = (NREC + NT - 1) / NT;
    constexpr int NHALO = NB * D * F;
    __shared__ T tile[TL::SZ];
    __shared__ int tab[NB * HT::N];
    __shared__ BP<T> prm[NB];
    const int blk0 = a.blk0 + xcd_remap(blockIdx.x, gridDim.x) * NB;
    const int tid = threadIdx.x;

    T ux[CPT][2], bo[CPT], be[CPT];
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        const int i = tid + k * NT, lb = i / H, r = i - lb * H;
        const size_t o = (size_t)(blk0 + lb) * V + r;
        ux[k][0] = ui[o];
        ux[k][1] = ui[o + H];
        bo[k] = b[o];
        be[k] = b[o + H];
    }
    static_assert(NB * HT::N <= NT, "one table entry per thread");
    const int tv = tid < NB * HT::N ? htab[(size_t)blk0 * HT::N + tid] : 0;
    BP<T> bpl{};
    if (tid < NB) bpl = bparams(a, blk0 + tid);
    int Jc[CPT], Jr[RPT];
#pragma unroll
    for (int k = 0; k < CPT; k++) Jc[k] = rbase<D, M, RD>(coord, blk0 + (tid + k * NT) / H);
#pragma unroll
    for (int k = 0; k < RPT; k++) Jr[k] = rbase<D, M, RD>(coord, blk0 + min((tid + k * NT) / (D * F2), NB - 1));
    if (tid < NB * HT::N) tab[tid] = tv;
    if (tid < NB) prm[tid] = bpl;
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        const int i = tid + k * NT, lb = i / H, r = i - lb * H;
        int x, y, z;
        LY::decode(r, x, y, z);
        tile[TL::origin(lb) + TL::at(x, y, z)] = ux[k][0];
        LY::decode(H + r, x, y, z);
        tile[TL::origin(lb) + TL::at(x, y, z)] = ux[k][1];
    }
    __syncthreads();

    // halo of the exterior faces: block lb, dimension d, face side = its bit
    // d (stored into the tile once the recompute operands' loads are issued)
    constexpr int PH = (NHALO + NT - 1) / NT;
    T hv[PH];
#pragma unroll
    for (int j = 0; j < PH; j++) {
        const int i = tid + NT * j, lb = min(i / (D * F), NB - 1), rem = i - lb * (D * F);
        const int d = min(rem / F, D - 1), t = rem - d * F;
        const int f = 2 * d + ((lb >> d) & 1);
        hv[j] = T(0);
        if (i < NHALO) hv[j] = halo_value_sw<D, M, T>(f, tab[lb * HT::N + f], blk0 + lb, t, ui, ib, a.sg);
    }
    T wc[CPT][2][2];
#pragma unroll
    for (int k = 0; k < CPT; k++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            int x, y, z;
            LY::decode(h * H + (tid + k * NT) % H, x, y, z);
            rweights<T, RD>(a, Jc[k] + (RD == 0 ? x : y), wc[k][h][0], wc[k][h][1]);
        }
    T rd[RPT], rb[RPT], rg[RPT][NS], rw[RPT][2];
    int rj[RPT];
#pragma unroll
    for (int k = 0; k < RPT; k++) {
        const int j = tid + k * NT;
        rj[k] = -1;
        rd[k] = rb[k] = rw[k][0] = rw[k][1] = T(0);
        if (j >= NREC) continue;
        const int lb = j / (D * F2), rem = j - lb * (D * F2);
        const int d = rem / F2, tq = rem - d * F2;
        const int f = 2 * d + ((lb >> d) & 1);
        const int *tb = tab + lb * HT::N, *gs = tb + HT::ND + f * HT::NS;
        const int e = tb[f];
        if (e < 0) continue;
        rj[k] = j;
        const int dir = (f & 1) ? 1 : -1;
        const int J = d == 0 ? RecFace<D, M, T, 0, TL>::template radial_index<RD>(dir, tq, Jr[k])
                             : RecFace<D, M, T, 1, TL>::template radial_index<RD>(dir, tq, Jr[k]);
        rweights<T, RD>(a, J, rw[k][0], rw[k][1]);
        if (d == 0) RecFace<D, M, T, 0, TL>::prefetch(dir, tq, e, gs, ui, b, ib, rd[k], rb[k], rg[k]);
        else if (d == 1) RecFace<D, M, T, 1, TL>::prefetch(dir, tq, e, gs, ui, b, ib, rd[k], rb[k], rg[k]);
        else RecFace<D, M, T, (D == 3 ? 2 : 1), TL>::prefetch(dir, tq, e, gs, ui, b, ib, rd[k], rb[k], rg[k]);
    }
#pragma unroll
    for (int j = 0; j < PH; j++) {
        const int i = tid + NT * j, lb = min(i / (D * F), NB - 1), rem = i - lb * (D * F);
        const int d = min(rem / F, D - 1), t = rem - d * F;
        const int f = 2 * d + ((lb >> d) & 1);
        if (i < NHALO) tile[TL::origin(lb) + halo_at_sw<D, M, TL>(f, t)] = hv[j];
    }
    __syncthreads();

    // first half-sweep
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        const int i = tid + k * NT, lb = i / H, r = i - lb * H;
        int x, y, z;
        LY::decode(r, x, y, z);
        const int p = TL::origin(lb) + TL::at(x, y, z);
        const BP<T> bp = prm[lb];
        T Lu = tstencil<D, M, T, RD, TL>(tile, p, ux[k][0], bp.cc, wc[k][0][0], wc[k][0][1]);
        ux[k][0] = fma_t<T>(bp.nwc, fma_t<T>(bp.s, bo[k], Lu), ux[k][0]);
        tile[p] = ux[k][0];
    }
#pragma unroll
    for (int k = 0; k < RPT; k++) {
        const int j = rj[k];
        if (j < 0) continue;
        const int lb = j / (D * F2), rem = j - lb * (D * F2);
        const int d = rem / F2, tq = rem - d * F2;
        const int f = 2 * d + ((lb >> d) & 1);
        const int *tb = tab + lb * HT::N, *gs = tb + HT::ND + f * HT::NS;
        T *tl = tile + TL::origin(lb);
        const int dir = (f & 1) ? 1 : -1;
        const BP<T> bp = prm[lb];
        const T wm = rw[k][0], wp = rw[k][1];
        if (d == 0)
            RecFace<D, M, T, 0, TL>::template compute<RD>(dir, tq, gs, tl, wm, wp, a, bp, rd[k], rb[k], rg[k]);
        else if (d == 1)
            RecFace<D, M, T, 1, TL>::template compute<RD>(dir, tq, gs, tl, wm, wp, a, bp, rd[k], rb[k], rg[k]);
        else
            RecFace<D, M, T, (D == 3 ? 2 : 1), TL>::template compute<RD>(dir, tq, gs, tl, wm, wp, a, bp, rd[k], rb[k],
                                                                         rg[k]);
    }
    __syncthreads();

    // second half-sweep
#pragma unroll
    for (int k = 0; k < CPT; k++) {
        const int i = tid + k * NT, lb = i / H, r = i - lb * H;
        int x, y, z;
        LY::decode(H + r, x, y, z);
        const int p = TL::origin(lb) + TL::at(x, y, z);
        const BP<T> bp = prm[lb];
        T Lu = tstencil<D, M, T, RD, TL>(tile, p, ux[k][1], bp.cc, wc[k][1][0], wc[k][1][1]);
        const size_t o = (size_t)(blk0 + lb) * V + r;
        uo[o] = ux[k][0];
        uo[o + H] = fma_t<T>(bp.nwc, fma_t<T>(bp.s, be[k], Lu), ux[k][1]);
    }
}

// k_gs_sweep_group for D = 3, M = 8 with a column mapping: 256 threads per
// sibling group (16^3 cells), each thread owns one (X, Y) column of the group
// tile and keeps its 16 cells and right-hand sides in registers, so that the
// Z neighbours of a cell come from registers and only the X and Y neighbours
// from the LDS tile. Wave w covers rows Y in [8 (w >> 1), 8 (w >> 1) + 8) and
// the columns with X + Y = w (mod 2): the red cells of all its lanes then sit
// at Z = P (mod 2), P = w & 1, a compile-time constant of the code path the
// wave runs. Tile rows are padded to 24 entries (no bank conflicts in the X
// and Y neighbour reads of a wave). Halo cells, neighbour recompute and the
// order of every sum as in k_gs_sweep_group, so the same bits. Round trips:
// the group's halo-table rows (issued before the interior loads and waited
// for alone), then the halo cells and recompute operands with the interior
// loads still in flight.
template <int D, int M, typename T, int RD>
struct ColSweep {
    static_assert(D == 3 && M == 8 && RD < 0, "column sweep is written for 8^3 Cartesian blocks");
    using LY = Lay<D, M>;
    using TL = Tile<D, M, 2, 24>;
    using HT = Halo<D>;
    static constexpr int NB = 8, V = LY::V, H = LY::H, NG = 2 * M;
    static constexpr int SY = TL::stride(1), SZ = TL::stride(2);
    struct Smem {
        T tile[TL::SZ];
        int tab[NB * HT::N];
        BP<T> prm[NB];
    };

    // offset of cell Z of a column from the column's base in its block (the
    // lower block for Z < 8, the upper one, 4 blocks on, for Z >= 8; storage
    // half 0 holds the red cells)
    template <int P, int Z>
    __device__ static constexpr int zoff() {
        return LY::MH * M * (Z & 7) + (((Z + P) & 1) ? H : 0);
    }

    template <int P>
    __device__ static __forceinline__ void run(Smem &sm, T *__restrict__ uo, const T *__restrict__ ui,
                                               const T *__restrict__ b, const T *__restrict__ ib,
                                               const int *__restrict__ coord, const LevelArgs<T> &a, int blk0,
                                               int w, int lane, int tv, const BP<T> &bpl) {
        const int tid = w * 64 + lane;
        const int Y = 8 * (w >> 1) + (lane >> 3), X = 2 * (lane & 7) + ((Y + P) & 1);
        const int x = X & 7, y = Y & 7, kxy = (X >> 3) | ((Y >> 3) << 1);
        const size_t g0 = (size_t)(blk0 + kxy) * V + (size_t)((x >> 1) + LY::MH * y);
        const T *__restrict__ ul = ui + g0, *__restrict__ uh = ul + 4 * V;
        const T *__restrict__ bl = b + g0, *__restrict__ bh = bl + 4 * V;
        T uc[NG], bc[NG];
        static_for<NG>([&](auto zc) {
            constexpr int Z = decltype(zc)::value;
            uc[Z] = (Z < 8 ? ul : uh)[zoff<P, Z>()];
            bc[Z] = (Z < 8 ? bl : bh)[zoff<P, Z>()];
        });
        if (tid < NB * HT::N) sm.tab[tid] = tv;
        if (tid < NB) sm.prm[tid] = bpl;
        lds_barrier();

        // halo cells of the six group faces: wave w takes the block face w of
        // each (tangential bits of the block from w), lane = cell t of the
        // face; a boundary face's mirror factor is applied at the tile write
        T hv[6], hm[6];
        static_for<6>([&](auto fc) {
            constexpr int F = decltype(fc)::value;
            constexpr int DIM = F >> 1, DA = DIM == 0 ? 1 : 0, DB = DIM == 2 ? 1 : 2;
            const int k = ((F & 1) << DIM) | ((w & 1) << DA) | ((w >> 1) << DB);
            const int e = __builtin_amdgcn_readfirstlane(sm.tab[k * HT::N + F]);
            hv[F] = halo_value<D, M, T, F>(e, blk0 + k, lane, ui, ib, T(1));
            hm[F] = e == NB_BOUNDARY ? a.sg[F] : T(1);
        });
        // recompute operands: for dimension DIM, waves 0-1 the low group face,
        // waves 2-3 the high one; half-wave = block face, tq = lane & 31
        const int rside = w >> 1, rbf = ((w & 1) << 1) | ((lane >> 5) & 1), rtq = lane & 31;
        T rd[3], rb[3], rg[3][4];
        int re[3];
        static_for<3>([&](auto dc) {
            constexpr int DIM = decltype(dc)::value;
            constexpr int DA = DIM == 0 ? 1 : 0, DB = DIM == 2 ? 1 : 2;
            const int k = (rside << DIM) | ((rbf & 1) << DA) | ((rbf >> 1) << DB), f = 2 * DIM + rside;
            const int *tb = sm.tab + k * HT::N;
            re[DIM] = tb[f];
            rd[DIM] = rb[DIM] = T(0);
            if (re[DIM] >= 0)
                RecFace<D, M, T, DIM, TL>::prefetch(rside ? 1 : -1, rtq, re[DIM], tb + HT::ND + f * HT::NS, ui, b, ib,
                                                    rd[DIM], rb[DIM], rg[DIM]);
        });
        // the tile
        const int pc = TL::at(X, Y, 0);
        static_for<NG>([&](auto zc) {
            constexpr int Z = decltype(zc)::value;
            sm.tile[pc + Z * SZ] = uc[Z];
        });
        static_for<6>([&](auto fc) {
            constexpr int F = decltype(fc)::value;
            constexpr int DIM = F >> 1, DA = DIM == 0 ? 1 : 0, DB = DIM == 2 ? 1 : 2;
            const int k = ((F & 1) << DIM) | ((w & 1) << DA) | ((w >> 1) << DB);
            sm.tile[TL::origin(k) + halo_at<D, M, F, TL>(lane)] = hm[F] * hv[F];
        });
        lds_barrier();

        // one cell update of the column (tstencil's order of terms)
        const BP<T> bq[2] = {sm.prm[kxy], sm.prm[kxy | 4]};
        T *const t = sm.tile;
        auto update = [&](auto zc) {
            constexpr int Z = decltype(zc)::value;
            const int p = pc + Z * SZ;
            const BP<T> &bp = bq[Z >> 3];
            const T zm = (Z == 0) ? t[pc - SZ] : uc[Z > 0 ? Z - 1 : 0];
            const T zp = (Z == NG - 1) ? t[pc + NG * SZ] : uc[Z < NG - 1 ? Z + 1 : 0];
            T v = T(0);
            v += zm;
            v += t[p - SY];
            v += t[p - 1];
            v += bp.cc * uc[Z];
            v += t[p + 1];
            v += t[p + SY];
            v += zp;
            uc[Z] = fma_t<T>(bp.nwc, fma_t<T>(bp.s, bc[Z], v), uc[Z]);
        };
        // first half-sweep: red cells
        static_for<NG / 2>([&](auto ic) {
            constexpr int Z = 2 * decltype(ic)::value + P;
            update(std::integral_constant<int, Z>());
            t[pc + Z * SZ] = uc[Z];
        });
        // the neighbours' face-layer cells
        static_for<3>([&](auto dc) {
            constexpr int DIM = decltype(dc)::value;
            constexpr int DA = DIM == 0 ? 1 : 0, DB = DIM == 2 ? 1 : 2;
            const int k = (rside << DIM) | ((rbf & 1) << DA) | ((rbf >> 1) << DB), f = 2 * DIM + rside;
            if (re[DIM] >= 0)
                RecFace<D, M, T, DIM, TL>::template compute<RD>(rside ? 1 : -1, rtq,
                                                                sm.tab + k * HT::N + HT::ND + f * HT::NS,
                                                                t + TL::origin(k), T(1), T(1), a, sm.prm[k], rd[DIM],
                                                                rb[DIM], rg[DIM]);
        });
        lds_barrier();

        // second half-sweep: black cells; then the column goes out
        static_for<NG / 2>([&](auto ic) {
            constexpr int Z = 2 * decltype(ic)::value + 1 - P;
            update(std::integral_constant<int, Z>());
        });
        T *__restrict__ ol = uo + g0, *__restrict__ oh = ol + 4 * V;
        static_for<NG>([&](auto zc) {
            constexpr int Z = decltype(zc)::value;
            (Z < 8 ? ol : oh)[zoff<P, Z>()] = uc[Z];
        });
    }
};

template <int D, int M, typename T, int RD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 5 : 1))) void k_gs_sweep_col(
    T *__restrict__ uo, const T *__restrict__ ui, const T *__restrict__ b, const T *__restrict__ ib,
    const int *__restrict__ htab, const int *__restrict__ coord, LevelArgs<T> a) {
    using CS = ColSweep<D, M, T, RD>;
    using HT = Halo<D>;
    __shared__ typename CS::Smem sm;
    const int blk0 = a.blk0 + xcd_remap(blockIdx.x, gridDim.x) * CS::NB;
    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    // halo-table rows and block parameters of the group, first
    int tv = 0;
    if (tid < CS::NB * HT::N) tv = htab[(size_t)blk0 * HT::N + tid];
    BP<T> bpl{};
    if (tid < CS::NB) bpl = bparams(a, blk0 + tid);
    if (w & 1) CS::template run<1>(sm, uo, ui, b, ib, coord, a, blk0, w, lane, tv, bpl);
    else CS::template run<0>(sm, uo, ui, b, ib, coord, a, blk0, w, lane, tv, bpl);
}

// k_gs_sweep_col with each column split between two threads (512 threads per
// sibling group): wave w covers the columns of wave w & 3 of k_gs_sweep_col in
// the block layer w >> 2 (8 cells each), so a group's work is spread over
// twice as many waves; the Z neighbours across the layers come from the tile.
// For the small levels, whose few groups leave most of the chip idle. The
// same operations on the same values as k_gs_sweep_col (same bits).
template <int D, int M, typename T, int RD>
struct ColSweepZ {
    using CS = ColSweep<D, M, T, RD>;
    using LY = Lay<D, M>;
    using TL = typename CS::TL;
    using HT = Halo<D>;
    static constexpr int NB = 8, V = LY::V, H = LY::H;
    static constexpr int SY = TL::stride(1), SZ = TL::stride(2);
    using Smem = typename CS::Smem;

    template <int DIM, bool ZIN = false>
    __device__ static __forceinline__ void rec_pre(Smem &sm, int q, const T *__restrict__ ui, const T *__restrict__ b,
                                                   const T *__restrict__ ib, int &re, T &rd, T &rb, T *rg) {
        constexpr int DA = DIM == 0 ? 1 : 0, DB = DIM == 2 ? 1 : 2;
        const int rside = q >> 7, rbf = (q >> 5) & 3, rtq = q & 31;
        const int k = (rside << DIM) | ((rbf & 1) << DA) | ((rbf >> 1) << DB), f = 2 * DIM + rside;
        const int *tb = sm.tab + k * HT::N;
        re = tb[f];
        rd = rb = T(0);
        if (re >= 0)
            RecFace<D, M, T, DIM, TL>::template prefetch<ZIN>(rside ? 1 : -1, rtq, re, tb + HT::ND + f * HT::NS, ui,
                                                              b, ib, rd, rb, rg);
    }
    template <int DIM>
    __device__ static __forceinline__ void rec_cmp(Smem &sm, int q, const int *__restrict__ coord,
                                                   const LevelArgs<T> &a, int re, T rd, T rb, const T *rg) {
        constexpr int DA = DIM == 0 ? 1 : 0, DB = DIM == 2 ? 1 : 2;
        const int rside = q >> 7, rbf = (q >> 5) & 3, rtq = q & 31;
        const int k = (rside << DIM) | ((rbf & 1) << DA) | ((rbf >> 1) << DB), f = 2 * DIM + rside;
        if (re >= 0)
            RecFace<D, M, T, DIM, TL>::template compute<RD>(rside ? 1 : -1, rtq,
                                                            sm.tab + k * HT::N + HT::ND + f * HT::NS,
                                                            sm.tile + TL::origin(k), T(1), T(1), a, sm.prm[k], rd, rb,
                                                            rg);
    }

    // VAR bit 0: the column goes out with nontemporal stores; bit 1: the
    // block's own right-hand side is read with nontemporal loads (both keep
    // L2 for the neighbours' face cells, which other work groups re-read);
    // bit 2: the input field and its ghost slabs are zero on this level (the
    // first sweep of a correction solve): nothing of it is read, the sweep
    // gives the bits of the same sweep over zeros
    template <int P, int VAR>
    __device__ static __forceinline__ void run(Smem &sm, T *__restrict__ uo, const T *__restrict__ ui,
                                               const T *__restrict__ b, const T *__restrict__ ib,
                                               const int *__restrict__ coord, const LevelArgs<T> &a, int blk0,
                                               int w, int lane, int tv, const BP<T> &bpl) {
        const int tid = w * 64 + lane;
        const int wc = w & 3, wz = w >> 2;
        const int Y = 8 * (wc >> 1) + (lane >> 3), X = 2 * (lane & 7) + ((Y + P) & 1);
        const int x = X & 7, y = Y & 7, kb = ((X >> 3) | ((Y >> 3) << 1)) | (wz << 2);
        const size_t g0 = (size_t)(blk0 + kb) * V + (size_t)((x >> 1) + LY::MH * y);
        constexpr bool ZIN = (VAR & 4) != 0;
        T uc[M], bc[M];
        static_for<M>([&](auto zc) {
            constexpr int z = decltype(zc)::value;
            uc[z] = ZIN ? T(0) : ui[g0 + CS::template zoff<P, z>()];
            if constexpr (VAR & 2) bc[z] = __builtin_nontemporal_load(&b[g0 + CS::template zoff<P, z>()]);
            else bc[z] = b[g0 + CS::template zoff<P, z>()];
        });
        if (tid < NB * HT::N) sm.tab[tid] = tv;
        if (tid < NB) sm.prm[tid] = bpl;
        lds_barrier();

        // halo cells of the six group faces: wave w takes the (face, block
        // face) pairs 3 w .. 3 w + 2 of the 24 (face uniform per wave), lane =
        // cell t of the face; a boundary face's mirror factor is applied at
        // the tile write
        T hv[3], hm[3];
        int hF[3], hk[3];
#pragma unroll
        for (int j = 0; j < 3; j++) {
            const int pr = 3 * w + j, F = pr >> 2, bf = pr & 3;
            const int DIM = F >> 1, DA = DIM == 0 ? 1 : 0, DB = DIM == 2 ? 1 : 2;
            const int k = ((F & 1) << DIM) | ((bf & 1) << DA) | ((bf >> 1) << DB);
            const int e = __builtin_amdgcn_readfirstlane(sm.tab[k * HT::N + F]);
            hF[j] = F;
            hk[j] = k;
            T v = T(0), m = T(1);
            if constexpr (ZIN) {
                SRMG_FACE_SWITCH(F, (m = e == NB_BOUNDARY ? a.sg[FF] : T(1)));
            } else {
                SRMG_FACE_SWITCH(F, (v = halo_value<D, M, T, FF>(e, blk0 + k, lane, ui, ib, T(1)),
                                     m = e == NB_BOUNDARY ? a.sg[FF] : T(1)));
            }
            hv[j] = v;
            hm[j] = m;
        }
        // recompute operands: waves 0-3 dimensions 0 and 2, waves 4-7 dimension 1
        int re[2];
        T rd[2], rb[2], rg[2][4];
        if (w < 4) {
            rec_pre<0, ZIN>(sm, tid, ui, b, ib, re[0], rd[0], rb[0], rg[0]);
            rec_pre<2, ZIN>(sm, tid, ui, b, ib, re[1], rd[1], rb[1], rg[1]);
        } else {
            rec_pre<1, ZIN>(sm, tid - 256, ui, b, ib, re[0], rd[0], rb[0], rg[0]);
        }
        // the tile
        const int pc = TL::at(X, Y, 8 * wz);
        static_for<M>([&](auto zc) {
            constexpr int z = decltype(zc)::value;
            sm.tile[pc + z * SZ] = uc[z];
        });
#pragma unroll
        for (int j = 0; j < 3; j++)
            sm.tile[TL::origin(hk[j]) + halo_at_sw<D, M, TL>(hF[j], lane)] = hm[j] * hv[j];
        lds_barrier();

        const BP<T> bp = sm.prm[kb];
        T *const t = sm.tile;
        auto update = [&](auto zc) {
            constexpr int z = decltype(zc)::value;
            const int p = pc + z * SZ;
            const T zm = (z == 0) ? t[p - SZ] : uc[z > 0 ? z - 1 : 0];
            const T zp = (z == M - 1) ? t[p + SZ] : uc[z < M - 1 ? z + 1 : 0];
            T v = T(0);
            v += zm;
            v += t[p - SY];
            v += t[p - 1];
            v += bp.cc * uc[z];
            v += t[p + 1];
            v += t[p + SY];
            v += zp;
            uc[z] = fma_t<T>(bp.nwc, fma_t<T>(bp.s, bc[z], v), uc[z]);
        };
        // first half-sweep: red cells (z = P mod 2 in the layer, which starts at an even Z)
        static_for<M / 2>([&](auto ic) {
            constexpr int z = 2 * decltype(ic)::value + P;
            update(std::integral_constant<int, z>());
            t[pc + z * SZ] = uc[z];
        });
        if (w < 4) {
            rec_cmp<0>(sm, tid, coord, a, re[0], rd[0], rb[0], rg[0]);
            rec_cmp<2>(sm, tid, coord, a, re[1], rd[1], rb[1], rg[1]);
        } else {
            rec_cmp<1>(sm, tid - 256, coord, a, re[0], rd[0], rb[0], rg[0]);
        }
        lds_barrier();
        static_for<M / 2>([&](auto ic) {
            constexpr int z = 2 * decltype(ic)::value + 1 - P;
            update(std::integral_constant<int, z>());
        });
        static_for<M>([&](auto zc) {
            constexpr int z = decltype(zc)::value;
            if constexpr (VAR & 1) __builtin_nontemporal_store(uc[z], &uo[g0 + CS::template zoff<P, z>()]);
            else uo[g0 + CS::template zoff<P, z>()] = uc[z];
        });
    }
};

template <int D, int M, typename T, int RD, int VAR = 0>
__global__ __launch_bounds__(512) void k_gs_sweep_colz(T *__restrict__ uo, const T *__restrict__ ui,
                                                       const T *__restrict__ b, const T *__restrict__ ib,
                                                       const int *__restrict__ htab, const int *__restrict__ coord,
                                                       LevelArgs<T> a) {
    using CZ = ColSweepZ<D, M, T, RD>;
    using HT = Halo<D>;
    __shared__ typename CZ::Smem sm;
    int gi = xcd_remap(blockIdx.x, gridDim.x);
    if (a.gord) gi = a.gord[gi];
    const int blk0 = a.blk0 + gi * CZ::NB;
    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    int tv = 0;
    if (tid < CZ::NB * HT::N) tv = htab[(size_t)blk0 * HT::N + tid];
    BP<T> bpl{};
    if (tid < CZ::NB) bpl = bparams(a, blk0 + tid);
    if (w & 1) CZ::template run<1, VAR>(sm, uo, ui, b, ib, coord, a, blk0, w, lane, tv, bpl);
    else CZ::template run<0, VAR>(sm, uo, ui, b, ib, coord, a, blk0, w, lane, tv, bpl);
}

// ---- tiled residual kernels ----

struct NoLoads {
    __device__ __forceinline__ void operator()() const {}
};

// Stage BPW blocks (valid cells + depth-1 face halo) of x in the LDS tile.
// list != nullptr selects the blocks through an index list (leaf blocks).
// Two barriers: after (interior, halo table) and after the halo cells
// (LDSB: barriers that order LDS only, for callers with loads in flight).
// with1 and with2 issue the caller's own loads with the first and the second
// round trip; with2 may also store to LDS what is read after the call.
template <int D, int M, typename T, int BPW, int NT, bool LDSB = false, class W1 = NoLoads, class W2 = NoLoads,
          class X = const T *>
__device__ __forceinline__ void load_tile(T *tile, int *tab, int *blks, const X x, const T *__restrict__ ib, const int *__restrict__ htab,
                                          const int *__restrict__ list, int first, int nloc, const T *sg,
                                          W1 &&with1 = W1(), W2 &&with2 = W2()) {
    using LY = Lay<D, M>;
    using TL = Tile<D, M>;
    using HT = Halo<D>;
    constexpr int F = LY::F, V = LY::V, ND = 2 * D;
    static_assert(BPW * ND <= NT, "one table entry per thread");
    // each phase issues all of its loads before the first tile store (a loop
    // that stores between its loads waits out each load in turn)
    constexpr int PI = (BPW * V + NT - 1) / NT, PH = (BPW * ND * F + NT - 1) / NT;
    const int tid = threadIdx.x;
    auto blk_at = [&](int lb) { return list ? list[first + min(lb, nloc - 1)] : first + min(lb, nloc - 1); };
    static_assert(V % 64 == 0 && NT % 64 == 0, "the cells of a wave are one block's");
    int bl[PI];
#pragma unroll
    for (int j = 0; j < PI; j++) bl[j] = blk_at(__builtin_amdgcn_readfirstlane((tid + NT * j) / V));
    const int bt = blk_at(tid / ND), bs = blk_at(min(tid, BPW - 1));
    T xv[PI];
#pragma unroll
    for (int j = 0; j < PI; j++) {
        const int i = tid + NT * j, lb = min(i / V, BPW - 1);
        xv[j] = (i < nloc * V) ? x[(size_t)bl[j] * V + (i - lb * V)] : T(0);
    }
    const int tv = tid < nloc * ND ? htab[(size_t)bt * HT::N + tid % ND] : 0;
    with1();
    if (tid < BPW) blks[tid] = tid < nloc ? bs : 0;
    if (tid < nloc * ND) tab[tid] = tv;
#pragma unroll
    for (int j = 0; j < PI; j++) {
        const int i = tid + NT * j, lb = min(i / V, BPW - 1);
        if (i < nloc * V) {
            int cx, cy, cz;
            LY::decode(i - lb * V, cx, cy, cz);
            tile[lb * TL::SZ + TL::at(cx, cy, cz)] = xv[j];
        }
    }
    if (LDSB) lds_barrier(); else __syncthreads();
    T hv[PH];
#pragma unroll
    for (int j = 0; j < PH; j++) {
        const int i = tid + NT * j, lb = min(i / (ND * F), BPW - 1), rem = i - lb * (ND * F);
        const int f = min(rem / F, ND - 1), t = rem - f * F;
        hv[j] = T(0);
        if (i < nloc * ND * F) hv[j] = halo_value_sw<D, M, T>(f, tab[lb * ND + f], blks[lb], t, x, ib, sg);
    }
    with2();
#pragma unroll
    for (int j = 0; j < PH; j++) {
        const int i = tid + NT * j, lb = min(i / (ND * F), BPW - 1), rem = i - lb * (ND * F);
        const int f = min(rem / F, ND - 1), t = rem - f * F;
        if (i < nloc * ND * F) tile[lb * TL::SZ + halo_at_sw<D, M, TL>(f, t)] = hv[j];
    }
    if (LDSB) lds_barrier(); else __syncthreads();
}

// k_interp_add on a level of complete sibling groups: the 2^D children of a
// parent are one work group, which stages the parent (with its depth-1 face
// halo: neighbour cells, mirrors, coarse-fine slabs of level l-1) in LDS and
// interpolates every child cell from there. Same operations and order as
// k_interp_add, so the result is bitwise the same.
template <int D, int M, typename T, int NT, class X>
__device__ __forceinline__ void interp_add_group_one(int g, T *__restrict__ u, const X u1,
                                                     const T *__restrict__ ib1, const int *__restrict__ htab,
                                                     const int *__restrict__ parent, int blk0,
                                                     const LevelArgs<T> &ac) {
    using LY = Lay<D, M>;
    using TL = Tile<D, M>;
    constexpr int NB = 1 << D, V = LY::V, MH = LY::MH;
    static_assert((NB * V) % NT == 0, "cells of a group must be a multiple of the work-group size");
    __shared__ T tile[TL::SZ];
    __shared__ int tab[2 * D];
    __shared__ int blks[1];
    const int g0 = blk0 + g * NB;
    const int pb = parent[g0];
    // the children's cells next: their loads stay in flight while the parent is staged
    T uo[NB * V / NT];
#pragma unroll
    for (int k = 0; k < NB * V / NT; k++) uo[k] = u[(size_t)g0 * V + threadIdx.x + k * NT];
    load_tile<D, M, T, 1, NT, true, NoLoads, NoLoads, X>(tile, tab, blks, u1, ib1, htab, nullptr, pb, 1, ac.sg);
#pragma unroll
    for (int k = 0; k < NB * V / NT; k++) {
        const int i = threadIdx.x + k * NT, lb = i / V, q = i - lb * V;
        int x0, x1, x2;
        LY::decode(q, x0, x1, x2);
        const int J0 = (lb & 1) * MH + (x0 >> 1);
        const int J1 = ((lb >> 1) & 1) * MH + (x1 >> 1);
        const int J2 = (D == 3) ? ((lb >> 2) & 1) * MH + (x2 >> 1) : 0;
        const int p = TL::at(J0, J1, J2);
        T f = w0<D, T>() * tile[p];
        f += w1<T>() * tile[p + (2 * (x0 & 1) - 1)];
        f += w1<T>() * tile[p + (2 * (x1 & 1) - 1) * TL::stride(1)];
        if (D == 3) f += w1<T>() * tile[p + (2 * (x2 & 1) - 1) * TL::stride(2)];
        const size_t o = (size_t)(g0 + lb) * V + q;
        u[o] = f + uo[k];
    }
}

template <int D, int M, typename T, int NT>
__global__ __launch_bounds__(NT) void k_interp_add_group(T *__restrict__ u, const T *__restrict__ u1,
                                                         const T *__restrict__ ib1, const int *__restrict__ htab,
                                                         const int *__restrict__ parent, int blk0,
                                                         LevelArgs<T> ac) {
    interp_add_group_one<D, M, T, NT>(blockIdx.x, u, u1, ib1, htab, parent, blk0, ac);
}

// k_interp_add_group on the first ngroups work groups and k_fill_interp of the
// fine level's slabs (from the coarse level of u, already final) on the rest:
// the prolongation writes the fine cells of u, the slab fill writes u's
// fine-level slabs; neither reads what the other writes.
template <int D, int M, typename T, int NT>
__global__ __launch_bounds__(NT) void k_interp_fill_group(T *__restrict__ u, const T *__restrict__ u1,
                                                          const T *__restrict__ ib1, const int *__restrict__ htab,
                                                          const int *__restrict__ parent, int blk0, unsigned ngroups,
                                                          T *__restrict__ ibu, const T *__restrict__ xc,
                                                          const int *__restrict__ nbr, const int4 *__restrict__ slots,
                                                          int slot0, int nslot, LevelArgs<T> ac) {
    if (blockIdx.x < ngroups)
        interp_add_group_one<D, M, T, NT>(blockIdx.x, u, u1, ib1, htab, parent, blk0, ac);
    else
        fill_interp_one<D, M, T>((blockIdx.x - ngroups) * NT + threadIdx.x, ibu, xc, nbr, slots, slot0, nslot, ac);
}

// k_interp_fill_group with the correction u - u1 of the coarse level formed as
// it is read (u1: u there before the correction) instead of by a launch of its
// own (k_diff_fill, 3 to 5 us on a small level and a pass over the coarse level on
// a large one). The work groups past ngroups + nwg_fill fill u1's slabs of the
// fine level with the correction's ghosts, which the next finer level's
// prolongation reads (nslot1: 0 on the finest level).
template <int D, int M, typename T, int NT>
__global__ __launch_bounds__(NT) void k_interp_fill_diff(T *__restrict__ u, const T *__restrict__ uc,
                                                         const T *__restrict__ u1c, T *__restrict__ ib1,
                                                         const int *__restrict__ htab,
                                                         const int *__restrict__ parent, int blk0, unsigned ngroups,
                                                         unsigned nwg_fill, T *__restrict__ ibu,
                                                         const int *__restrict__ nbr, const int4 *__restrict__ slots,
                                                         int slot0, int nslot, int nslot1, LevelArgs<T> ac) {
    const Diff<T> d{uc, u1c};
    if (blockIdx.x < ngroups)
        interp_add_group_one<D, M, T, NT>(blockIdx.x, u, d, ib1, htab, parent, blk0, ac);
    else if (blockIdx.x < ngroups + nwg_fill)
        fill_interp_one<D, M, T>((blockIdx.x - ngroups) * NT + threadIdx.x, ibu, uc, nbr, slots, slot0, nslot, ac);
    else
        fill_interp_one<D, M, T>((blockIdx.x - ngroups - nwg_fill) * NT + threadIdx.x, ib1, d, nbr, slots, slot0,
                                 nslot1, ac);
}

enum { RES_WRITE = 0, RES_NORM = 1, RES_DEFECT = 2 };

// Residual of a level from LDS tiles (src/multigrid.jl:309-323).
//   RES_WRITE:  r = -(b + L u / s) on the blocks [a.blk0, a.blk0 + a.nblk)
//   RES_NORM:   leaf blocks list[0..n), or where list is null the n blocks from
//               a.blk0: partial[k] = wgt * sum of r^2 over block k of them
//   RES_DEFECT: out (float) = b + L u / s = -r on the level's blocks, and
//               partial[k] = wgt * sum of r^2 over block k if it is a leaf (else 0)
// Each block's partial is an LDS tree sum in a fixed order.
// (work group wg of nwg; sm: the work group's LDS)
template <int D, int M, typename T, int BPW, int NT, int MODE>
struct ResidTileLds {
    double red[MODE == RES_WRITE ? 1 : BPW * NT];
    T tile[BPW * Tile<D, M>::SZ];
    BP<T> prm[BPW];
    int tab[BPW * 2 * D], blks[BPW];
};
template <int D, int M, typename T, typename TO, int BPW, int NT, int MODE, int RD>
__device__ __forceinline__ void resid_tile(ResidTileLds<D, M, T, BPW, NT, MODE> &sm, int wg, int nwg,
                                           TO *__restrict__ out, const T *__restrict__ u, const T *__restrict__ b,
                                           const T *__restrict__ ib, const int *__restrict__ htab,
                                           const int *__restrict__ coord, const int *__restrict__ list,
                                           const int *__restrict__ isleaf, int n, const LevelArgs<T> &a, double wgt,
                                           double *__restrict__ partial) {
    using LY = Lay<D, M>;
    using TL = Tile<D, M>;
    constexpr int V = LY::V;
    T *tile = sm.tile;
    int *tab = sm.tab, *blks = sm.blks;
    BP<T> *prm = sm.prm;
    double *red = sm.red;
    const int first = xcd_remap(wg, nwg) * BPW;
    const int nloc = min(BPW, n - first);
    const int *lst = (MODE == RES_NORM) ? list : nullptr;
    const int base = lst ? first : a.blk0 + first;
    // the right-hand sides of the thread's cells, their radial weights and the
    // block parameters come with the tile's two round trips
    constexpr int PER = (BPW * V + NT - 1) / NT;
    T bv[PER], wv[PER][2];
    int Jc[PER];
    bool leafs[PER];
    BP<T> bpl{};
    auto blk_at = [&](int lb) { return lst ? lst[base + min(lb, nloc - 1)] : base + min(lb, nloc - 1); };
    load_tile<D, M, T, BPW, NT>(
        tile, tab, blks, u, ib, htab, lst, base, nloc, a.sg,
        [&] {
            if ((int)threadIdx.x < nloc) bpl = bparams(a, blk_at(threadIdx.x));
#pragma unroll
            for (int j = 0; j < PER; j++) {
                const int i = threadIdx.x + NT * j, lb = min(i / V, BPW - 1);
                const int blk = blk_at(__builtin_amdgcn_readfirstlane(lb));
                bv[j] = (i < nloc * V) ? b[(size_t)blk * V + (i - lb * V)] : T(0);
                Jc[j] = rbase<D, M, RD>(coord, blk);
                leafs[j] = MODE == RES_DEFECT && isleaf[blk];
            }
        },
        [&] {
#pragma unroll
            for (int j = 0; j < PER; j++) {
                int x, y, z;
                LY::decode((threadIdx.x + NT * j) % V, x, y, z);
                rweights<T, RD>(a, Jc[j] + (RD == 0 ? x : y), wv[j][0], wv[j][1]);
            }
            if ((int)threadIdx.x < nloc) prm[threadIdx.x] = bpl;
        });
    double acc[BPW];
#pragma unroll
    for (int lb = 0; lb < BPW; lb++) acc[lb] = 0.0;
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = threadIdx.x + NT * j;
        if (i >= nloc * V) break;
        int lb = i / V, q = i - lb * V;
        int blk = blks[lb];
        int x, y, z;
        LY::decode(q, x, y, z);
        int p = lb * TL::SZ + TL::at(x, y, z);
        const BP<T> bp = prm[lb];
        T Lu = tstencil<D, M, T, RD>(tile, p, tile[p], bp.cc, wv[j][0], wv[j][1]);
        size_t o = (size_t)blk * V + q;
        T rr = -(bv[j] + Lu / bp.s);
        if (MODE == RES_WRITE) out[o] = (TO)rr;
        if (MODE == RES_DEFECT) out[o] = (TO)(bv[j] + Lu / bp.s);
        if (MODE == RES_NORM || leafs[j]) {
#pragma unroll
            for (int k = 0; k < BPW; k++)
                if (k == lb) acc[k] += (double)rr * (double)rr;
        }
    }
    if (MODE != RES_WRITE) {
        // each block's halving tree over the NT threads, all blocks at once:
        // the levels of 64 and more across waves in LDS, the rest inside one
        // wave per block by lane shuffles (the same pairs in the same order)
        static_assert(NT % 64 == 0 && NT >= 128, "whole waves, at least two");
#pragma unroll
        for (int lb = 0; lb < BPW; lb++) red[lb * NT + threadIdx.x] = acc[lb];
        __syncthreads();
        for (int w = NT / 2; w >= 64; w >>= 1) {
            if ((int)threadIdx.x < w) {
#pragma unroll
                for (int lb = 0; lb < BPW; lb++) red[lb * NT + threadIdx.x] += red[lb * NT + threadIdx.x + w];
            }
            __syncthreads();
        }
        const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        for (int lb = wave; lb < BPW; lb += NT / 64) {
            double v = red[lb * NT + lane];
#pragma unroll
            for (int w = 32; w > 0; w >>= 1) {
                const double o = __shfl_down(v, w, 64);
                if (lane < w) v += o;
            }
            if (lane == 0 && lb < nloc) partial[first + lb] = v * wgt;
        }
    }
}

template <int D, int M, typename T, typename TO, int BPW, int NT, int MODE, int RD>
__global__ __launch_bounds__(NT) void k_resid_tile(TO *__restrict__ out, const T *__restrict__ u,
                                                   const T *__restrict__ b, const T *__restrict__ ib,
                                                   const int *__restrict__ htab, const int *__restrict__ coord,
                                                   const int *__restrict__ list, const int *__restrict__ isleaf,
                                                   int n, LevelArgs<T> a, double wgt, double *__restrict__ partial) {
    __shared__ ResidTileLds<D, M, T, BPW, NT, MODE> sm;
    resid_tile<D, M, T, TO, BPW, NT, MODE, RD>(sm, blockIdx.x, gridDim.x, out, u, b, ib, htab, coord, list, isleaf, n, a,
                                               wgt, partial);
}

// Stage sibling group g0 (2^D blocks from device block g0) of u into a
// Tile<D, M, 2> with the halo of the group's exterior faces, its halo table
// entries and block parameters; every load of a phase is issued before the
// phase's first LDS store. Ends with a barrier (which also waits for loads
// the caller issued before the call). with1 and with2: as in load_tile.
template <int D, int M, typename T, int NT, class W1, class W2>
__device__ __forceinline__ void stage_group(T *tile, int *tab, BP<T> *prm, const T *__restrict__ u,
                                            const T *__restrict__ ib, const int *__restrict__ htab,
                                            const LevelArgs<T> &a, int g0, W1 &&with1, W2 &&with2) {
    using LY = Lay<D, M>;
    using TL = Tile<D, M, 2>;
    using HT = Halo<D>;
    constexpr int NB = 1 << D, V = LY::V, F = LY::F;
    constexpr int PU = (NB * V + NT - 1) / NT, PH = (NB * D * F + NT - 1) / NT;
    const int tid = threadIdx.x;
    T uv[PU];
#pragma unroll
    for (int j = 0; j < PU; j++) {
        const int i = tid + NT * j;
        uv[j] = (i < NB * V) ? u[(size_t)g0 * V + i] : T(0);
    }
    static_assert(NB * 2 * D <= NT, "one table entry per thread");
    int tv = 0;
    if (tid < NB * 2 * D) tv = htab[(size_t)(g0 + tid / (2 * D)) * HT::N + tid % (2 * D)];
    BP<T> bpl{};
    if (tid < NB) bpl = bparams(a, g0 + tid);
    with1();
    if (tid < NB * 2 * D) tab[tid] = tv;
    if (tid < NB) prm[tid] = bpl;
#pragma unroll
    for (int j = 0; j < PU; j++) {
        const int i = tid + NT * j, lb = min(i / V, NB - 1), q = i - lb * V;
        if (i < NB * V) {
            int x, y, z;
            LY::decode(q, x, y, z);
            tile[TL::origin(lb) + TL::at(x, y, z)] = uv[j];
        }
    }
    __syncthreads();
    T hv[PH];
#pragma unroll
    for (int j = 0; j < PH; j++) {
        const int i = tid + NT * j, lb = min(i / (D * F), NB - 1), rem = i - lb * (D * F);
        const int d = min(rem / F, D - 1), t = rem - d * F;
        const int f = 2 * d + ((lb >> d) & 1);
        hv[j] = T(0);
        if (i < NB * D * F) hv[j] = halo_value_sw<D, M, T>(f, tab[lb * 2 * D + f], g0 + lb, t, u, ib, a.sg);
    }
    with2();
#pragma unroll
    for (int j = 0; j < PH; j++) {
        const int i = tid + NT * j, lb = min(i / (D * F), NB - 1), rem = i - lb * (D * F);
        const int d = min(rem / F, D - 1), t = rem - d * F;
        const int f = 2 * d + ((lb >> d) & 1);
        if (i < NB * D * F) tile[TL::origin(lb) + halo_at_sw<D, M, TL>(f, t)] = hv[j];
    }
    __syncthreads();
}

// k_resid_tile (RES_WRITE, RES_DEFECT; RES_DEFECT with out == nullptr forms
// only the partials, on a level of leaves in block order those of
// k_resid_tile<RES_NORM>) on a level of complete sibling groups:
// one group of 2^D blocks per work group of NT threads, staged as one
// (2M)^D tile with the halo of the group's exterior faces only. Teams of RT
// threads take one block at a time and visit its cells in the order of
// k_resid_tile<.., 1, RT, ..> (cells t, t + RT, ...; partials as the same
// RT-wide tree sum), so outputs and partials are bitwise the same.
template <int D, int M, typename T, int MODE, int NT>
struct ResidGroupLds {
    double red[MODE == RES_DEFECT ? NT : 1];
    T tile[Tile<D, M, 2>::SZ];
    BP<T> prm[1 << D];
    int tab[(1 << D) * 2 * D];
};
template <int D, int M, typename T, typename TO, int RT, int MODE, int RD, int NT>
__device__ __forceinline__ void resid_group(ResidGroupLds<D, M, T, MODE, NT> &sm, int wg, int nwg,
                                            TO *__restrict__ out, const T *__restrict__ u, const T *__restrict__ b,
                                            const T *__restrict__ ib, const int *__restrict__ htab,
                                            const int *__restrict__ coord, const int *__restrict__ isleaf,
                                            const LevelArgs<T> &a, double wgt, double *__restrict__ partial) {
    using LY = Lay<D, M>;
    using TL = Tile<D, M, 2>;
    constexpr int NB = 1 << D, V = LY::V;
    constexpr int TEAMS = NT / RT;
    static_assert(NB % TEAMS == 0 && RT >= 64, "team layout");
    T *tile = sm.tile;
    int *tab = sm.tab;
    BP<T> *prm = sm.prm;
    double *red = sm.red;
    constexpr int NR = NB / TEAMS, QR = (V + RT - 1) / RT;
    const int gl = xcd_remap(wg, nwg);
    const int g0 = a.blk0 + gl * NB;
    const int tid = threadIdx.x;
    const int team = tid / RT, t = tid - team * RT;
    // the right-hand sides of the thread's cells, in flight during the staging
    T bv[NR][QR];
#pragma unroll
    for (int round = 0; round < NR; round++)
#pragma unroll
        for (int h = 0; h < QR; h++) {
            const int q = t + RT * h;
            bv[round][h] = q < V ? b[(size_t)(g0 + team + round * TEAMS) * V + q] : T(0);
        }
    // their radial weights come with the staging's two round trips
    int Jc[NR];
    T wv[NR][QR][2];
    auto coords = [&] {
#pragma unroll
        for (int round = 0; round < NR; round++) Jc[round] = rbase<D, M, RD>(coord, g0 + team + round * TEAMS);
    };
    auto weights = [&] {
#pragma unroll
        for (int round = 0; round < NR; round++)
#pragma unroll
            for (int h = 0; h < QR; h++) {
                int x, y, z;
                LY::decode((t + RT * h) % V, x, y, z);
                rweights<T, RD>(a, Jc[round] + (RD == 0 ? x : y), wv[round][h][0], wv[round][h][1]);
            }
    };
    bool leafs[NR];
    stage_group<D, M, T, NT>(
        tile, tab, prm, u, ib, htab, a, g0,
        [&] {
            coords();
#pragma unroll
            for (int round = 0; round < NR; round++)
                leafs[round] = (MODE == RES_DEFECT) && isleaf[g0 + team + round * TEAMS];
        },
        weights);
#pragma unroll
    for (int round = 0; round < NR; round++) {
        const int lb = team + round * TEAMS, blk = g0 + lb;
        const BP<T> bp = prm[lb];
        const bool leaf = leafs[round];
        double acc = 0.0;
#pragma unroll
        for (int h = 0; h < QR; h++) {
            const int q = t + RT * h;
            if (q >= V) break;
            int x, y, z;
            LY::decode(q, x, y, z);
            const int p = TL::origin(lb) + TL::at(x, y, z);
            T Lu = tstencil<D, M, T, RD, TL>(tile, p, tile[p], bp.cc, wv[round][h][0], wv[round][h][1]);
            const size_t o = (size_t)blk * V + q;
            T rr = -(bv[round][h] + Lu / bp.s);
            if (MODE == RES_WRITE) out[o] = (TO)rr;
            if (MODE == RES_DEFECT) {
                if (out != nullptr) out[o] = (TO)(bv[round][h] + Lu / bp.s);
                if (leaf) acc += (double)rr * (double)rr;
            }
        }
        if (MODE == RES_DEFECT) {
            // the team's halving tree: levels of 64 and more in LDS, the
            // rest inside the team's first wave by lane shuffles (same pairs)
            red[tid] = acc;
            __syncthreads();
            for (int w = RT / 2; w >= 64; w >>= 1) {
                if (t < w) red[tid] += red[tid + w];
                __syncthreads();
            }
            if (t < 64) {
                double v = red[tid];
#pragma unroll
                for (int w = 32; w > 0; w >>= 1) {
                    const double o = __shfl_down(v, w, 64);
                    if (t < w) v += o;
                }
                if (t == 0) partial[(blk - a.blk0)] = v * wgt;
            }
            __syncthreads();
        }
    }
}

template <int D, int M, typename T, typename TO, int RT, int MODE, int RD, int NT = 1024>
__global__ __launch_bounds__(NT) void k_resid_group(TO *__restrict__ out, const T *__restrict__ u,
                                                      const T *__restrict__ b, const T *__restrict__ ib,
                                                      const int *__restrict__ htab, const int *__restrict__ coord,
                                                      const int *__restrict__ isleaf, LevelArgs<T> a, double wgt,
                                                      double *__restrict__ partial) {
    __shared__ ResidGroupLds<D, M, T, MODE, NT> sm;
    resid_group<D, M, T, TO, RT, MODE, RD, NT>(sm, blockIdx.x, gridDim.x, out, u, b, ib, htab, coord, isleaf, a, wgt,
                                               partial);
}

// The V-cycle descent's residual and restrictions on a level of complete
// sibling groups, in one launch: residual of the group (as k_resid_group,
// kept in LDS instead of written), then on the parent's cells the restricted
// residual rc and the restricted u (into uc and, if u1c is not null, u1c),
// each the sum of the 2^D children in k_restrict's order divided by 2^D. Work
// groups past ngroups copy u -> u1 on the coarse level's leaf blocks (lists
// leaves[0..nleafc)), completing copyto!(u1, u) on that level. Same values
// and operations as residual + restrict(u) + copy + restrict(r).
//
// 2D: the coarse right-hand side of the parent's cells too (k_postrestrict_group
// on its own: 3.3 to 4.8 us of launch and two round trips a level). What it
// needs beyond the parent's cells are the coarse cells around: a covered one is
// the mean of its children (restricted here again, in the same order), a leaf's
// is read, a mirror or a slab as ever. FP64 levels of 504 / 1,976 / 3,872 blocks:
// 5.8 / 7.0 / 9.0 us for 4.7 + 4.1 / 5.9 + 4.2 / 7.5 + 4.8 in two launches.
template <int D, int M, typename T, int RT, int RD, int NT = 1024>
__global__ __launch_bounds__(NT) void k_resid_restrict(const T *__restrict__ u, const T *__restrict__ b,
                                                         const T *__restrict__ ib, const int *__restrict__ htab,
                                                         const int *__restrict__ coord,
                                                         const int *__restrict__ parent, LevelArgs<T> a,
                                                         unsigned ngroups, T *__restrict__ rc, T *__restrict__ uc,
                                                         T *__restrict__ u1c, const T *ucin,
                                                         const int *__restrict__ leaves, int nleafc, T *__restrict__ bc,
                                                         LevelArgs<T> ac) {
    using LY = Lay<D, M>;
    using TL = Tile<D, M, 2>;
    using HT = Halo<D>;
    using TC = Tile<D, M>;
    constexpr int NB = 1 << D, V = LY::V, F = LY::F, MH = LY::MH;
    constexpr int TEAMS = NT / RT;
    static_assert(NB % TEAMS == 0 && RT >= 64, "team layout");
    static_assert(D == 3 || (V <= NT && 4 * M <= NT), "2D: a coarse cell, and one of those around, for each thread");
    const int tid = threadIdx.x;
    if (blockIdx.x >= ngroups) {
        // u1 = u on the coarse level's leaf blocks
        const int64_t i = (int64_t)(blockIdx.x - ngroups) * NT + tid;
        if (i < (int64_t)nleafc * V) {
            const size_t o = (size_t)leaves[i / V] * V + (size_t)(i % V);
            u1c[o] = ucin[o];
        }
        return;
    }
    __shared__ T tile[TL::SZ];
    __shared__ T rt[NB * V];
    __shared__ int tab[NB * 2 * D];
    __shared__ BP<T> prm[NB];
    constexpr int NR = NB / TEAMS, QR = (V + RT - 1) / RT;
    const int gl = xcd_remap(blockIdx.x, ngroups);
    const int g0 = a.blk0 + gl * NB;
    const int team = tid / RT, t = tid - team * RT;
    // the right-hand sides of the thread's cells, in flight during the staging
    T bv[NR][QR];
#pragma unroll
    for (int round = 0; round < NR; round++)
#pragma unroll
        for (int h = 0; h < QR; h++) {
            const int q = t + RT * h;
            bv[round][h] = q < V ? b[(size_t)(g0 + team + round * TEAMS) * V + q] : T(0);
        }
    // their radial weights come with the staging's two round trips
    int Jc[NR];
    T wv[NR][QR][2];
    auto coords = [&] {
#pragma unroll
        for (int round = 0; round < NR; round++) Jc[round] = rbase<D, M, RD>(coord, g0 + team + round * TEAMS);
    };
    auto weights = [&] {
#pragma unroll
        for (int round = 0; round < NR; round++)
#pragma unroll
            for (int h = 0; h < QR; h++) {
                int x, y, z;
                LY::decode((t + RT * h) % V, x, y, z);
                rweights<T, RD>(a, Jc[round] + (RD == 0 ? x : y), wv[round][h][0], wv[round][h][1]);
            }
    };
    int pb = 0;
    // the coarse cell beyond face f, tangential index ct, of the parent
    const int f = tid / M, ct = tid % M, fr0 = f & 1 ? 0 : M - 2;
    T hc = T(0), cw[2] = {T(1), T(1)};
    BP<T> cbp{};
    auto around = [&] {
        if constexpr (D == 2) {
            cbp = bparams(ac, pb);
            if constexpr (RD >= 0) {
                int x, y, z;
                LY::decode(tid % V, x, y, z);
                // the parent's radial index, from its first child's
                const int Jp = M * ((rbase<D, M, RD>(coord, g0) - 1) / M / 2) + 1;
                rweights<T, RD>(ac, Jp + (RD == 0 ? x : y), cw[0], cw[1]);
            }
            if (f >= 4) return;
            // the child on that face
            const int half = ct >= MH, k = f < 2 ? (f & 1) + 2 * half : half + 2 * (f & 1);
            const int e = tab[k * 2 * D + f];
            if (e >= 0) {
                T m = T(0);
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int in = f < 2 ? q & 1 : q >> 1, it = f < 2 ? q >> 1 : q & 1;
                    const int cn = fr0 + in, cf = 2 * (ct - half * MH) + it;
                    m += u[(size_t)e * V + LY::sidx(f < 2 ? cn : cf, f < 2 ? cf : cn, 0)];
                }
                hc = m / T(LY::NC);
            } else if (e != NB_BOUNDARY) {
                const int pe = htab[(size_t)pb * HT::N + f];
                const int cn = f & 1 ? 0 : M - 1;
                hc = pe >= 0 ? ucin[(size_t)pe * V + LY::sidx(f < 2 ? cn : ct, f < 2 ? ct : cn, 0)]
                             : ib[(size_t)max(nb_slot(pe), 0) * F + ct];
            }
        }
    };
    stage_group<D, M, T, NT>(
        tile, tab, prm, u, ib, htab, a, g0,
        [&] {
            coords();
            pb = parent[g0];
        },
        [&] {
            weights();
            around();
        });
#pragma unroll
    for (int round = 0; round < NR; round++) {
        const int lb = team + round * TEAMS;
        const BP<T> bp = prm[lb];
#pragma unroll
        for (int h = 0; h < QR; h++) {
            const int q = t + RT * h;
            if (q >= V) break;
            int x, y, z;
            LY::decode(q, x, y, z);
            const int p = TL::origin(lb) + TL::at(x, y, z);
            T Lu = tstencil<D, M, T, RD, TL>(tile, p, tile[p], bp.cc, wv[round][h][0], wv[round][h][1]);
            rt[lb * V + q] = -(bv[round][h] + Lu / bp.s);
        }
    }
    __syncthreads();
    __shared__ T ctile[D == 2 ? TC::SZ : 1];
    T rcv = T(0);
    // the parent's cells: coarse cell X of sub-block k = (X >= MH per dim)
    for (int i = tid; i < V; i += NT) {
        int X0, X1, X2;
        LY::decode(i, X0, X1, X2);
        const int k = (X0 >= MH ? 1 : 0) | (X1 >= MH ? 2 : 0) | (D == 3 && X2 >= MH ? 4 : 0);
        const int j0 = X0 - (k & 1) * MH, j1 = X1 - ((k >> 1) & 1) * MH, j2 = (D == 3) ? X2 - ((k >> 2) & 1) * MH : 0;
        T fr = T(0), fu = T(0);
#pragma unroll
        for (int q = 0; q < LY::NC; q++) {
            const int i0 = q & 1, i1 = (q >> 1) & 1, i2 = (q >> 2) & 1;
            const int cx = 2 * j0 + i0, cy = 2 * j1 + i1, cz = D == 3 ? 2 * j2 + i2 : 0;
            fr += rt[k * V + LY::sidx(cx, cy, cz)];
            fu += tile[TL::origin(k) + TL::at(cx, cy, cz)];
        }
        const size_t o = (size_t)pb * V + i;
        rc[o] = fr / T(LY::NC);
        const T uv = fu / T(LY::NC);
        uc[o] = uv;
        if (u1c) u1c[o] = uv;
        if constexpr (D == 2) {
            rcv = fr / T(LY::NC);
            ctile[TC::at(X0, X1, 0)] = uv;
        }
    }
    if constexpr (D == 2) {
        __syncthreads();
        if (f < 4) {
            const int cn = f & 1 ? M : -1, in = f & 1 ? M - 1 : 0;
            const int k = (f < 2 ? (f & 1) : (ct >= MH)) + 2 * (f < 2 ? (ct >= MH) : (f & 1));
            if (tab[k * 2 * D + f] == NB_BOUNDARY) hc = ac.sg[f] * ctile[f < 2 ? TC::at(in, ct, 0) : TC::at(ct, in, 0)];
            ctile[f < 2 ? TC::at(cn, ct, 0) : TC::at(ct, cn, 0)] = hc;
        }
        __syncthreads();
        if (tid < V) {
            int X0, X1, X2;
            LY::decode(tid, X0, X1, X2);
            const int p = TC::at(X0, X1, 0);
            const T Lu = tstencil<D, M, T, RD>(ctile, p, ctile[p], cbp.cc, cw[0], cw[1]);
            bc[(size_t)pb * V + tid] = -(rcv + Lu / cbp.s);
        }
    }
}

// k_resid_restrict for D = 3, M = 8 with the column mapping of k_gs_sweep_col:
// 256 threads per sibling group, thread = (X, Y) column of the group with its
// 16 cells and right-hand sides in registers (Z neighbours from registers).
// The residual stays in registers while the parent's u is restricted from
// the u tile; then it takes u's place in the tile, from which the parent's
// residual is restricted (both in k_restrict's order). Same operations as
// k_resid_restrict, so the same bits. Work groups past ngroups copy u to u1
// on the coarse level's leaf blocks (256 cells each).
// Column staging shared by the column residual kernels (3D, 8^3, one sibling
// group of 16^3 cells per 256-thread work group): thread (w, lane) owns the
// (X, Y) column X + Y = w (mod 2) of rows 8 (w >> 1) .. 8 (w >> 1) + 7 (as in
// k_gs_sweep_col); its 16 cells of u and b go to registers, u with the group's
// depth-1 face halo to the LDS tile. tab holds the group's own face entries
// (2D per block, loaded by the caller into tv), prm the block parameters.
template <int D, int M, typename T, int RD>
struct ColStage {
    static_assert(D == 3 && M == 8 && RD < 0, "column kernels are written for 8^3 Cartesian blocks");
    using LY = Lay<D, M>;
    using TL = Tile<D, M, 2>;
    static constexpr int NB = 8, V = LY::V, NG = 2 * M, ND = 2 * D;
    static constexpr int SY = TL::stride(1), SZ = TL::stride(2);

    struct Col {
        int X, Y, x, y, kxy, pc;
        size_t gb;  // the column's base offset in its lower block
    };

    template <int P>
    __device__ static __forceinline__ Col column(int g0, int w, int lane) {
        Col c;
        c.Y = 8 * (w >> 1) + (lane >> 3);
        c.X = 2 * (lane & 7) + ((c.Y + P) & 1);
        c.x = c.X & 7;
        c.y = c.Y & 7;
        c.kxy = (c.X >> 3) | ((c.Y >> 3) << 1);
        c.gb = (size_t)(g0 + c.kxy) * V + (size_t)((c.x >> 1) + LY::MH * c.y);
        c.pc = TL::at(c.X, c.Y, 0);
        return c;
    }

    template <int P>
    __device__ static __forceinline__ void stage(T *tile, int *tab, BP<T> *prm, const Col &c, const T *__restrict__ u,
                                                 const T *__restrict__ b, const T *__restrict__ ib,
                                                 const LevelArgs<T> &a, int g0, int w, int lane, int tv,
                                                 const BP<T> &bpl, T *ux, T *bx) {
        using CS = ColSweep<D, M, T, RD>;
        const int tid = w * 64 + lane;
        const T *__restrict__ ul = u + c.gb, *__restrict__ uh = ul + 4 * V;
        const T *__restrict__ bl = b + c.gb, *__restrict__ bh = bl + 4 * V;
        static_for<NG>([&](auto zc) {
            constexpr int Z = decltype(zc)::value;
            ux[Z] = (Z < 8 ? ul : uh)[CS::template zoff<P, Z>()];
            bx[Z] = (Z < 8 ? bl : bh)[CS::template zoff<P, Z>()];
        });
        if (tid < NB * ND) tab[tid] = tv;
        if (tid < NB) prm[tid] = bpl;
        lds_barrier();
        // halo of the six group faces (wave w: block face w of each; lane: cell)
        T hv[6], hm[6];
        static_for<6>([&](auto fc) {
            constexpr int F = decltype(fc)::value;
            constexpr int DIM = F >> 1, DA = DIM == 0 ? 1 : 0, DB = DIM == 2 ? 1 : 2;
            const int k = ((F & 1) << DIM) | ((w & 1) << DA) | ((w >> 1) << DB);
            const int e = __builtin_amdgcn_readfirstlane(tab[k * ND + F]);
            hv[F] = halo_value<D, M, T, F>(e, g0 + k, lane, u, ib, T(1));
            hm[F] = e == NB_BOUNDARY ? a.sg[F] : T(1);
        });
        static_for<NG>([&](auto zc) {
            constexpr int Z = decltype(zc)::value;
            tile[c.pc + Z * SZ] = ux[Z];
        });
        static_for<6>([&](auto fc) {
            constexpr int F = decltype(fc)::value;
            constexpr int DIM = F >> 1, DA = DIM == 0 ? 1 : 0, DB = DIM == 2 ? 1 : 2;
            const int k = ((F & 1) << DIM) | ((w & 1) << DA) | ((w >> 1) << DB);
            tile[TL::origin(k) + halo_at<D, M, F, TL>(lane)] = hm[F] * hv[F];
        });
        lds_barrier();
    }

    // L u of cell Z of the column (tstencil's order of terms)
    template <int Z>
    __device__ static __forceinline__ T lu(const T *t, const Col &c, const T *ux, T cc) {
        const int p = c.pc + Z * SZ;
        const T zm = (Z == 0) ? t[c.pc - SZ] : ux[Z > 0 ? Z - 1 : 0];
        const T zp = (Z == NG - 1) ? t[c.pc + NG * SZ] : ux[Z < NG - 1 ? Z + 1 : 0];
        T v = T(0);
        v += zm;
        v += t[p - SY];
        v += t[p - 1];
        v += cc * ux[Z];
        v += t[p + 1];
        v += t[p + SY];
        v += zp;
        return v;
    }
};

template <int D, int M, typename T, int RD>
struct ColResid {
    using CT = ColStage<D, M, T, RD>;
    using LY = Lay<D, M>;
    using TL = Tile<D, M, 2>;
    static constexpr int NB = 8, V = LY::V, NG = 2 * M, ND = 2 * D;
    struct Smem {
        T tile[TL::SZ];  // u with its halo; then the residual at the group's cells
        int tab[NB * ND];
        BP<T> prm[NB];
    };

    template <int P>
    __device__ static __forceinline__ void run(Smem &sm, const T *__restrict__ u, const T *__restrict__ b,
                                               const T *__restrict__ ib, const int *__restrict__ parent,
                                               const LevelArgs<T> &a, int g0, int w, int lane, int tv,
                                               const BP<T> &bpl, T *__restrict__ rc, T *__restrict__ uc,
                                               T *__restrict__ u1c) {
        const int tid = w * 64 + lane;
        const typename CT::Col c = CT::template column<P>(g0, w, lane);
        T ux[NG], bx[NG];
        CT::template stage<P>(sm.tile, sm.tab, sm.prm, c, u, b, ib, a, g0, w, lane, tv, bpl, ux, bx);
        // residual r = -(b + L u / s), kept in registers
        const BP<T> bq[2] = {sm.prm[c.kxy], sm.prm[c.kxy | 4]};
        T rr[NG];
        static_for<NG>([&](auto zc) {
            constexpr int Z = decltype(zc)::value;
            const BP<T> &bp = bq[Z >> 3];
            const T v = CT::template lu<Z>(sm.tile, c, ux, bp.cc);
            rr[Z] = -(bx[Z] + v / bp.s);
        });
        // the parent's cells, in storage order: coarse cell (X0, X1, X2) sums
        // group cells (2 X0 + i0, 2 X1 + i1, 2 X2 + i2), q = i0 + 2 i1 + 4 i2;
        // u's sums first, then the residual takes u's place in the tile
        constexpr int PC = V / 256;
        T fu[PC];
#pragma unroll
        for (int h = 0; h < PC; h++) {
            int X0, X1, X2;
            LY::decode(tid + 256 * h, X0, X1, X2);
            fu[h] = T(0);
#pragma unroll
            for (int q = 0; q < LY::NC; q++)
                fu[h] += sm.tile[TL::at(2 * X0 + (q & 1), 2 * X1 + ((q >> 1) & 1), 2 * X2 + ((q >> 2) & 1))];
        }
        lds_barrier();  // every read of u in the tile is done
        static_for<NG>([&](auto zc) {
            constexpr int Z = decltype(zc)::value;
            sm.tile[TL::at(c.X, c.Y, Z)] = rr[Z];
        });
        lds_barrier();
        const int pb = parent[g0];
#pragma unroll
        for (int h = 0; h < PC; h++) {
            const int i = tid + 256 * h;
            int X0, X1, X2;
            LY::decode(i, X0, X1, X2);
            T fr = T(0);
#pragma unroll
            for (int q = 0; q < LY::NC; q++)
                fr += sm.tile[TL::at(2 * X0 + (q & 1), 2 * X1 + ((q >> 1) & 1), 2 * X2 + ((q >> 2) & 1))];
            const size_t o = (size_t)pb * V + i;
            rc[o] = fr / T(LY::NC);
            const T uv = fu[h] / T(LY::NC);
            uc[o] = uv;
            if (u1c) u1c[o] = uv;
        }
    }
};

// k_resid_group<RES_DEFECT> (FP64 in, FP32 out) with the column mapping: out =
// b + L u / s on every cell of the group, and per block the partial
// wgt * sum of r^2 over its cells if it is a leaf (0 otherwise), summed as
// k_resid_group sums it (thread t of 256: cells q = t, t + 256 in that order,
// then the halving tree over t), so the partials are the same bits. With
// out == nullptr only the partials are formed: on a level whose blocks are all
// leaves, in level order, these are the partials of k_resid_tile<RES_NORM>
// (the same per-block order).
template <int D, int M, int RD>
struct ColDefect {
    using T = double;
    using CT = ColStage<D, M, T, RD>;
    using LY = Lay<D, M>;
    using TL = Tile<D, M, 2>;
    static constexpr int NB = 8, V = LY::V, NG = 2 * M, ND = 2 * D;
    static_assert(TL::SZ >= NB * V, "the squares reuse the tile");
    struct Smem {
        T tile[TL::SZ];  // u with its halo; then the squares sq[k V + q] of block k, cell q
        int tab[NB * ND];
        BP<T> prm[NB];
        int leaf[NB];
    };

    template <int P>
    __device__ static __forceinline__ void run(Smem &sm, float *__restrict__ out, const T *__restrict__ u,
                                               const T *__restrict__ b, const T *__restrict__ ib,
                                               const LevelArgs<T> &a, int g0, int w, int lane, int tv,
                                               const BP<T> &bpl, double wgt, double *__restrict__ partial) {
        using CS = ColSweep<D, M, T, RD>;
        const int tid = w * 64 + lane;
        const typename CT::Col c = CT::template column<P>(g0, w, lane);
        T ux[NG], bx[NG];
        CT::template stage<P>(sm.tile, sm.tab, sm.prm, c, u, b, ib, a, g0, w, lane, tv, bpl, ux, bx);
        const BP<T> bq[2] = {sm.prm[c.kxy], sm.prm[c.kxy | 4]};
        const bool lf[2] = {sm.leaf[c.kxy] != 0, sm.leaf[c.kxy | 4] != 0};
        float *__restrict__ ol = out + c.gb, *__restrict__ oh = ol + 4 * V;
        double sq[NG];
        static_for<NG>([&](auto zc) {
            constexpr int Z = decltype(zc)::value;
            const BP<T> &bp = bq[Z >> 3];
            const T v = CT::template lu<Z>(sm.tile, c, ux, bp.cc);
            if (out != nullptr) (Z < 8 ? ol : oh)[CS::template zoff<P, Z>()] = (float)(bx[Z] + v / bp.s);
            const T rr = -(bx[Z] + v / bp.s);
            sq[Z] = lf[Z >> 3] ? (double)rr * (double)rr : 0.0;
        });
        lds_barrier();  // every tile read is done: the squares take its place
        static_for<NG>([&](auto zc) {
            constexpr int Z = decltype(zc)::value;
            const int k = c.kxy | ((Z >> 3) << 2);
            sm.tile[k * V + LY::sidx(c.x, c.y, Z & 7)] = sq[Z];
        });
        lds_barrier();
        // per block: acc_t = (0 + sq[t]) + sq[t + 256], then the halving tree
        for (int k = 0; k < NB; k++) {
            double acc = 0.0;
            acc += sm.tile[k * V + tid];
            acc += sm.tile[k * V + tid + 256];
            sm.tile[k * V + tid] = acc;
        }
        lds_barrier();
        // the tree's levels 128 and 64 across waves in LDS; 32 .. 1 inside
        // wave w for blocks w and w + 4 by lane shuffles (the same pairs)
        for (int wd = 128; wd >= 64; wd >>= 1) {
            for (int i = tid; i < NB * wd; i += 256) {
                const int k = i / wd, t = i - k * wd;
                sm.tile[k * V + t] += sm.tile[k * V + t + wd];
            }
            lds_barrier();
        }
#pragma unroll
        for (int j = 0; j < NB / 4; j++) {
            const int k = w + 4 * j;
            double v = sm.tile[k * V + lane];
#pragma unroll
            for (int wd = 32; wd > 0; wd >>= 1) {
                const double o = __shfl_down(v, wd, 64);
                if (lane < wd) v += o;
            }
            if (lane == 0) partial[g0 + k - a.blk0] = v * wgt;
        }
    }
};

// work group wg of nwg
template <int D, int M, int RD>
__device__ __forceinline__ void defect_col(typename ColDefect<D, M, RD>::Smem &sm, int wg, int nwg,
                                           float *__restrict__ out, const double *__restrict__ u,
                                           const double *__restrict__ b, const double *__restrict__ ib,
                                           const int *__restrict__ htab, const int *__restrict__ isleaf,
                                           const LevelArgs<double> &a, double wgt, double *__restrict__ partial) {
    using CD = ColDefect<D, M, RD>;
    using HT = Halo<D>;
    constexpr int ND = CD::ND;
    const int tid = threadIdx.x;
    const int g0 = a.blk0 + xcd_remap(wg, nwg) * CD::NB;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    int tv = 0;
    if (tid < CD::NB * ND) {
        const int lb = tid / ND;
        tv = htab[(size_t)(g0 + lb) * HT::N + (tid - lb * ND)];
    }
    BP<double> bpl{};
    if (tid < CD::NB) {
        bpl = bparams(a, g0 + tid);
        sm.leaf[tid] = isleaf[g0 + tid];
    }
    if (w & 1) CD::template run<1>(sm, out, u, b, ib, a, g0, w, lane, tv, bpl, wgt, partial);
    else CD::template run<0>(sm, out, u, b, ib, a, g0, w, lane, tv, bpl, wgt, partial);
}

// one level on its own
template <int D, int M, int RD>
__global__ __launch_bounds__(256) void k_defect_col(float *__restrict__ out, const double *__restrict__ u,
                                                    const double *__restrict__ b, const double *__restrict__ ib,
                                                    const int *__restrict__ htab, const int *__restrict__ isleaf,
                                                    LevelArgs<double> a, double wgt, double *__restrict__ partial) {
    __shared__ typename ColDefect<D, M, RD>::Smem sm;
    defect_col<D, M, RD>(sm, blockIdx.x, gridDim.x, out, u, b, ib, htab, isleaf, a, wgt, partial);
}

// ---- residual norms and defects of several levels in one launch ----
//
// A solve's norm needs every level, and a level that does not fill the chip
// costs a launch of 5 to 8 us whatever its size. Each segment is one level
// with the kernel that suits it: resid_tile on its leaves (NORM) or blocks,
// resid_group or defect_col on complete sibling groups. Segments start at
// multiples of eight work groups, so that xcd_remap's places hold.
enum { SEG_TILE = 0, SEG_GROUP = 1, SEG_COL = 2 };
template <typename T>
struct ResidSeg {
    LevelArgs<T> a;
    double wgt;
    int wg0, nwg;  // its work groups
    int kind;
    int n, list0;  // SEG_TILE: blocks, and where its leaves start in the list (NORM;
                   // -1: they are all blocks in their order)
    int p0;        // its first partial
};
constexpr int SEG_MAX = 12;
template <typename T>
struct ResidSegs {
    ResidSeg<T> s[SEG_MAX];
    int n;
};

// COLS: segments of defect_col among them. Its registers and LDS leave 12 waves
// to a CU for 32, which a tile segment pays for: on 9,261 blocks of 8^3 without
// sibling groups 42 us for 22, on 103,823 495 for 237. So large levels without
// groups take a launch without it (TILE_APART; on 2,048 leaves beside 12,608 blocks
// with groups one launch takes 26.0 us, two 26.4). And a work group of it waits out
// the look-up of its segment, with nothing else to run: 110,592 blocks with
// groups took 212 us a norm for 197 in k_defect_col, so a column level of that
// order (COL_APART: where the difference pays for a launch), or one with no other
// beside it, goes there.
constexpr int TILE_APART = 3000, COL_APART = 80000;
template <int D, int M, typename T>
constexpr bool RESID_COLS = D == 3 && M == 8 && sizeof(T) == 8;
template <int D, int M, typename T, typename TO, int BPW, int NT, bool NORM, int RD, bool COLS>
__global__ __launch_bounds__(NT) void k_resid_levels(ResidSegs<T> g, TO *__restrict__ out, const T *__restrict__ u,
                                                     const T *__restrict__ b, const T *__restrict__ ib,
                                                     const int *__restrict__ htab, const int *__restrict__ coord,
                                                     const int *__restrict__ leaves, const int *__restrict__ isleaf,
                                                     double *__restrict__ partial) {
    constexpr bool GROUPS = D == 2 && M == 16 && NT == 256;
    static_assert(!COLS || RD < 0, "columns are Cartesian");
    constexpr int TM = NORM ? RES_NORM : RES_DEFECT;
    using TileLds = ResidTileLds<D, M, T, BPW, NT, TM>;
    using GroupLds = ResidGroupLds<D, M, T, RES_DEFECT, GROUPS ? NT : 1>;
    constexpr size_t tb = sizeof(TileLds), gb = GROUPS ? sizeof(GroupLds) : 0;
    size_t constexpr cb = [] {
        if constexpr (COLS) return sizeof(typename ColDefect<D, M, RD>::Smem);
        else return (size_t)0;
    }();
    __shared__ __align__(16) char sm[tb > gb ? (tb > cb ? tb : cb) : (gb > cb ? gb : cb)];
    int k = 0;
    while (k + 1 < g.n && (int)blockIdx.x >= g.s[k + 1].wg0) k++;
    const ResidSeg<T> &s = g.s[k];
    const int wg = blockIdx.x - s.wg0;
    if (wg >= s.nwg) return;
    if constexpr (GROUPS) {
        if (s.kind == SEG_GROUP) {
            resid_group<D, M, T, TO, NT, RES_DEFECT, RD, NT>(*reinterpret_cast<GroupLds *>(sm), wg, s.nwg, out, u, b, ib,
                                                             htab, coord, isleaf, s.a, s.wgt, partial + s.p0);
            return;
        }
    }
    if constexpr (COLS) {
        if (s.kind == SEG_COL) {
            defect_col<D, M, RD>(*reinterpret_cast<typename ColDefect<D, M, RD>::Smem *>(sm), wg, s.nwg,
                                 (float *)out, u, b, ib, htab, isleaf, s.a, s.wgt, partial + s.p0);
            return;
        }
    }
    resid_tile<D, M, T, TO, BPW, NT, TM, RD>(*reinterpret_cast<TileLds *>(sm), wg, s.nwg, out, u, b, ib, htab, coord,
                                             NORM && s.list0 >= 0 ? leaves + s.list0 : nullptr, isleaf, s.n, s.a,
                                             s.wgt, partial + s.p0);
}

template <int D, int M, typename T, int RD>
__global__ __launch_bounds__(256) void k_resid_restrict_col(const T *__restrict__ u, const T *__restrict__ b,
                                                            const T *__restrict__ ib, const int *__restrict__ htab,
                                                            const int *__restrict__ parent, LevelArgs<T> a,
                                                            unsigned ngroups, T *__restrict__ rc, T *__restrict__ uc,
                                                            T *__restrict__ u1c, const T *__restrict__ ucin,
                                                            const int *__restrict__ leaves, int nleafc) {
    using CR = ColResid<D, M, T, RD>;
    using HT = Halo<D>;
    constexpr int V = CR::V, ND = CR::ND;
    const int tid = threadIdx.x;
    if (blockIdx.x >= ngroups) {
        const int64_t i = (int64_t)(blockIdx.x - ngroups) * 256 + tid;
        if (i < (int64_t)nleafc * V) {
            const size_t o = (size_t)leaves[i / V] * V + (size_t)(i % V);
            u1c[o] = ucin[o];
        }
        return;
    }
    __shared__ typename CR::Smem sm;
    const int g0 = a.blk0 + xcd_remap(blockIdx.x, ngroups) * CR::NB;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    int tv = 0;
    if (tid < CR::NB * ND) {
        const int lb = tid / ND;
        tv = htab[(size_t)(g0 + lb) * HT::N + (tid - lb * ND)];
    }
    BP<T> bpl{};
    if (tid < CR::NB) bpl = bparams(a, g0 + tid);
    if (w & 1) CR::template run<1>(sm, u, b, ib, parent, a, g0, w, lane, tv, bpl, rc, uc, u1c);
    else CR::template run<0>(sm, u, b, ib, parent, a, g0, w, lane, tv, bpl, rc, uc, u1c);
}

// k_postrestrict on a level of complete sibling groups: the parent of group g
// is fully covered, so one work group stages the parent's u (level l-1, with
// its depth-1 halo) in LDS and forms b = -(r + L u / s) on all its cells.
// Same operations as k_postrestrict (the tile stencil equals the gather one).
template <int D, int M, typename T, int RD>
__global__ __launch_bounds__(256) void k_postrestrict_group(T *__restrict__ bout, const T *__restrict__ u,
                                                            const T *__restrict__ r, const T *__restrict__ ib,
                                                            const int *__restrict__ htab,
                                                            const int *__restrict__ coord,
                                                            const int *__restrict__ parent, int fblk0,
                                                            LevelArgs<T> ac) {
    using LY = Lay<D, M>;
    using TL = Tile<D, M>;
    constexpr int NB = 1 << D, V = LY::V;
    constexpr int PER = (V + 255) / 256;
    __shared__ T tile[TL::SZ];
    __shared__ int tab[2 * D];
    __shared__ int blks[1];
    // the parent's r first: its loads stay in flight while the tile is staged
    const int pb = parent[fblk0 + (int)blockIdx.x * NB];
    T rv[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int q = threadIdx.x + 256 * j;
        rv[j] = q < V ? r[(size_t)pb * V + q] : T(0);
    }
    int Jc = 0;
    BP<T> bp{};
    T wv[PER][2];
    load_tile<D, M, T, 1, 256, true>(
        tile, tab, blks, u, ib, htab, nullptr, pb, 1, ac.sg,
        [&] {
            Jc = rbase<D, M, RD>(coord, pb);
            bp = bparams(ac, pb);
        },
        [&] {
#pragma unroll
            for (int j = 0; j < PER; j++) {
                int x, y, z;
                LY::decode((threadIdx.x + 256 * j) % V, x, y, z);
                rweights<T, RD>(ac, Jc + (RD == 0 ? x : y), wv[j][0], wv[j][1]);
            }
        });
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int q = threadIdx.x + 256 * j;
        if (q >= V) break;
        int x, y, z;
        LY::decode(q, x, y, z);
        const int p = TL::at(x, y, z);
        T Lu = tstencil<D, M, T, RD>(tile, p, tile[p], bp.cc, wv[j][0], wv[j][1]);
        bout[(size_t)pb * V + q] = -(rv[j] + Lu / bp.s);
    }
}

// ---- electric field ----

template <typename T>
struct EFieldArgs {
    int blk0;    // first device block of the level
    T hl;        // cell size of the level: h / 2^(l-1)
    T e0[3];     // constant external field
    T sg[6];     // boundary ghost signs of u
    // free boundary (fill_ghost_free!, src/freebc.jl:218-238), 2D only: the
    // ghosts on the +fdim face of the outermost blocks (coordinate fkd along
    // fdim) gain 2 mean(fbb over fp entries); fbb == nullptr: none
    const T *fbb;
    const int *coord;
    int fdim, fkd, fp;
};

// electric_field! (src/multigrid.jl:421-449) with a constant external field
// (src/multigrid.jl:451) on one block per work group: u with its depth-1 halo
// in LDS (the ghosts of the post-solve fills, src/streamer.jl:340-349);
// E_d on the M+1 faces of every line along d, (u[c - e_d] - u[c]) / h_l + e0_d
// (face i is the lower face of cell i), stored as ef[blk][d][i + (M+1) o]
// with o the other coordinates in increasing dimension order; |E| at the cell
// centres, sqrt(sum_d (E_d(lower) + E_d(upper))^2 / 4), in the block layout.
template <int D, int M, typename T>
__global__ __launch_bounds__(256) void k_efield(T *__restrict__ eabs, T *__restrict__ ef, const T *__restrict__ u,
                                                const T *__restrict__ ib, const int *__restrict__ htab,
                                                EFieldArgs<T> ea) {
    using LY = Lay<D, M>;
    using TL = Tile<D, M>;
    constexpr int V = LY::V, NF = (M + 1) * (D == 2 ? M : M * M);
    __shared__ T tile[TL::SZ];
    __shared__ int tab[2 * D];
    __shared__ int blks[1];
    const int blk = ea.blk0 + blockIdx.x;
    load_tile<D, M, T, 1, 256>(tile, tab, blks, u, ib, htab, nullptr, blk, 1, ea.sg);
    if constexpr (D == 2) {
        if (ea.fbb != nullptr && ea.coord[blk * D + ea.fdim] == ea.fkd) {
            const int od = 1 - ea.fdim;
            const int i0 = (ea.coord[blk * D + od] - 1) * M;
            for (int i = threadIdx.x; i < M; i += 256) {
                T sum = T(0);
                for (int j = ea.fp * (i0 + i); j < ea.fp * (i0 + i + 1); j++) sum += ea.fbb[j];
                const T bmean = sum / T(ea.fp);
                int c[3] = {0, 0, 0};
                c[ea.fdim] = M;
                c[od] = i;
                tile[TL::at(c[0], c[1], 0)] += T(2) * bmean;
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int d = 0; d < D; d++) {
        const int da = d == 0 ? 1 : 0, db = d == 2 ? 1 : 2;
        for (int i = threadIdx.x; i < NF; i += 256) {
            const int fi = i % (M + 1), o = i / (M + 1);
            int c[3] = {0, 0, 0};
            c[d] = fi;
            c[da] = o % M;
            if (D == 3) c[db] = o / M;
            const int p = TL::at(c[0], c[1], c[2]);
            ef[((size_t)blk * D + d) * NF + i] = (tile[p - TL::stride(d)] - tile[p]) / ea.hl + ea.e0[d];
        }
    }
    for (int q = threadIdx.x; q < V; q += 256) {
        int x, y, z;
        LY::decode(q, x, y, z);
        const int p = TL::at(x, y, z);
        T f2 = T(0);
#pragma unroll
        for (int d = 0; d < D; d++) {
            const T lo = (tile[p - TL::stride(d)] - tile[p]) / ea.hl + ea.e0[d];
            const T hi = (tile[p] - tile[p + TL::stride(d)]) / ea.hl + ea.e0[d];
            const T t = lo + hi;
            f2 += t * t / T(4);
        }
        eabs[(size_t)blk * V + q] = sqrt(f2);
    }
}

// ---- free boundary conditions (src/freebc.jl, 2D cylindrical) ----

// getouter! (src/freebc.jl:112-142) as a gather: u1[j] = u[src[j]] / hl[j],
// where src names the outermost cell of the finest level covering entry j
__global__ __launch_bounds__(WG) void k_fb_gather(double *__restrict__ u1, const double *__restrict__ u,
                                                  const int64_t *__restrict__ src, const double *__restrict__ hl,
                                                  int64_t n) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) u1[j] = u[src[j]] / hl[j];
}

// y = S x for an n x n sine matrix given transposed (ST[j n + k] = S[k][j]),
// summed in j order; then y_k = fm[k] * y_k (fm != nullptr: am = f .* u1,
// src/freebc.jl:103) or y_k = y_k h / 2^(level-1) / 2 (src/freebc.jl:106)
__global__ __launch_bounds__(WG) void k_fb_dst(const double *__restrict__ ST, const double *__restrict__ x,
                                               double *__restrict__ y, int64_t n, const double *__restrict__ fm,
                                               double h, double lev) {
    const int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    double acc = 0.0;
    for (int64_t j = 0; j < n; j++) acc += ST[j * n + k] * x[j];
    y[k] = fm ? fm[k] * acc : acc * h / lev / 2.0;
}

// setouter! (src/freebc.jl:149-215): cell cells[i] receives, in order, the
// contributions r in [rs[i], rs[i+1]): q += coef[r] (sum of b over
// [bs[r], bs[r] + bl[r]) / bd[r]) / sl[r]
__global__ __launch_bounds__(WG) void k_fb_setouter(double *__restrict__ q, const int64_t *__restrict__ cells,
                                                    const int *__restrict__ rs, const double *__restrict__ coef,
                                                    const int64_t *__restrict__ bs, const int *__restrict__ bl,
                                                    const double *__restrict__ bd, const double *__restrict__ sl,
                                                    const double *__restrict__ b, int ncells) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= ncells) return;
    double v = q[cells[i]];
    for (int r = rs[i]; r < rs[i + 1]; r++) {
        double sum = 0.0;
        for (int64_t j = bs[r]; j < bs[r] + bl[r]; j++) sum += b[j];
        v += coef[r] * (sum / bd[r]) / sl[r];
    }
    q[cells[i]] = v;
}

// resnorm partials of u = 0 (the residual is -b): the same blocks, visiting
// order and tree sums as k_resid_tile<RES_NORM>, so the partials are bitwise
// those of a residual norm of a zero field, without reading one. be (may be
// null) receives (float) b on the visited blocks. list: the leaves of all
// levels, lv.first[l] .. of level l, weighted by 2^(-D l).
struct LeafLevels {
    int n, first[32];
};
template <int D, int M, typename T, int BPW, int NT>
__global__ __launch_bounds__(NT) void k_bnorm(const T *__restrict__ b, const int *__restrict__ list, int n,
                                              LeafLevels lv, double *__restrict__ partial, float *__restrict__ be) {
    constexpr int V = Lay<D, M>::V;
    __shared__ int blks[BPW];
    __shared__ double red[BPW * NT];
    const int first = xcd_remap(blockIdx.x, gridDim.x) * BPW;
    const int nloc = min(BPW, n - first);
    if ((int)threadIdx.x < BPW) blks[threadIdx.x] = ((int)threadIdx.x < nloc) ? list[first + threadIdx.x] : 0;
    __syncthreads();
    // every load of the thread's cells before the first store and sum
    constexpr int PER = (BPW * V + NT - 1) / NT;
    double acc[BPW];
#pragma unroll
    for (int lb = 0; lb < BPW; lb++) acc[lb] = 0.0;
    T bv[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = threadIdx.x + NT * j, lb = min(i / V, BPW - 1);
        bv[j] = (i < nloc * V) ? b[(size_t)blks[lb] * V + (i - lb * V)] : T(0);
    }
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = threadIdx.x + NT * j, lb = min(i / V, BPW - 1);
        if (i >= nloc * V) break;
        if (be) be[(size_t)blks[lb] * V + (i - lb * V)] = (float)bv[j];
        const T rr = -bv[j];
#pragma unroll
        for (int k = 0; k < BPW; k++)
            if (k == lb) acc[k] += (double)rr * (double)rr;
    }
    // the halving tree of every block at once (the same pairs as one block
    // at a time; blocks past nloc are summed and dropped): the levels of 64
    // and more across waves in LDS, the rest inside one wave per block by
    // lane shuffles
    static_assert(NT % 64 == 0 && NT >= 128, "whole waves, at least two");
#pragma unroll
    for (int lb = 0; lb < BPW; lb++) red[lb * NT + threadIdx.x] = acc[lb];
    __syncthreads();
    for (int w = NT / 2; w >= 64; w >>= 1) {
        if ((int)threadIdx.x < w) {
#pragma unroll
            for (int lb = 0; lb < BPW; lb++) red[lb * NT + threadIdx.x] += red[lb * NT + threadIdx.x + w];
        }
        __syncthreads();
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int lb = wave; lb < BPW; lb += NT / 64) {
        double v = red[lb * NT + lane];
#pragma unroll
        for (int w = 32; w > 0; w >>= 1) {
            const double o = __shfl_down(v, w, 64);
            if (lane < w) v += o;
        }
        if (lane == 0 && lb < nloc) {
            int l = 0;
            while (l + 1 < lv.n && first + lb >= lv.first[l + 1]) l++;
            partial[first + lb] = v * ldexp(1.0, -D * l);
        }
    }
}

// ---- exact level-1 solve (FP64) ----

// level-1 valid cells -> uniform grid (column-major, dimension 1 fastest), times c
template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_grid_gather(double *__restrict__ g, const T *__restrict__ x,
                                                    const int *__restrict__ coord, int blk0, int nblk,
                                                    int N0, int N1, int nper, size_t total,
                                                    const double *__restrict__ cs) {
    using LY = Lay<D, M>;
    int gt = blockIdx.x * blockDim.x + threadIdx.x;
    int lb = gt / LY::V;
    if (lb >= nblk) return;
    int blk = blk0 + lb;
    int q = gt - lb * LY::V;
    int c0, c1, c2;
    LY::decode(q, c0, c1, c2);
    int grid = lb / nper;
    size_t gi = (size_t)grid * total + (size_t)(M * (coord[blk * D] - 1) + c0) +
                (size_t)N0 * ((size_t)(M * (coord[blk * D + 1] - 1) + c1) +
                              (D == 3 ? (size_t)N1 * (size_t)(M * (coord[blk * D + 2] - 1) + c2) : 0));
    g[gi] = cs[grid] * (double)x[(size_t)blk * LY::V + q];
}

template <int D, int M, typename T>
__global__ __launch_bounds__(WG) void k_grid_scatter(T *__restrict__ x, const double *__restrict__ g,
                                                     const int *__restrict__ coord, int blk0, int nblk,
                                                     int N0, int N1, int nper, size_t total) {
    using LY = Lay<D, M>;
    int gt = blockIdx.x * blockDim.x + threadIdx.x;
    int lb = gt / LY::V;
    if (lb >= nblk) return;
    int blk = blk0 + lb;
    int q = gt - lb * LY::V;
    int c0, c1, c2;
    LY::decode(q, c0, c1, c2);
    int grid = lb / nper;
    size_t gi = (size_t)grid * total + (size_t)(M * (coord[blk * D] - 1) + c0) +
                (size_t)N0 * ((size_t)(M * (coord[blk * D + 1] - 1) + c1) +
                              (D == 3 ? (size_t)N1 * (size_t)(M * (coord[blk * D + 2] - 1) + c2) : 0));
    x[(size_t)blk * LY::V + q] = (T)g[gi];
}

// Y = A X along one axis of a column-major grid: A is n x n (row-major), the
// grid is viewed as [outer][n][inner] (inner = stride of the axis) and every
// (outer, inner) pair is a column of X. Register-tiled FP64 GEMM: a work
// group computes a 64 x TC tile of Y (rows i, columns) with 256 threads, each
// an RA x 4 sub-tile (RA = TC / 16), over k-chunks of 16 staged in LDS
// (zero-padded past n). Each output is one dot product summed in k order, so
// every TC gives the same bits; narrow tiles give small grids more work groups.
template <int TC>
__global__ __launch_bounds__(256) void k_axis_gemm(const double *__restrict__ A, int n, int inner, int ncol,
                                                   const double *__restrict__ in, double *__restrict__ out) {
    constexpr int TI = 64, TK = 16, RA = TC / 16, TCQ = TC / 4;
    __shared__ double As[TK][TI + 1];
    __shared__ double Xs[TK][TC + 1];
    const int tid = threadIdx.x;
    const int i0 = blockIdx.y * TI, c0 = blockIdx.x * TC;
    const int ti = (tid / TCQ) * RA, tc = (tid % TCQ) * 4;
    double acc[RA][4];
#pragma unroll
    for (int a = 0; a < RA; a++)
#pragma unroll
        for (int q = 0; q < 4; q++) acc[a][q] = 0.0;
    for (int k0 = 0; k0 < n; k0 += TK) {
        // A tile: rows i0..i0+63, columns k0..k0+15
        for (int e = tid; e < TI * TK; e += 256) {
            int ii = e / TK, kk = e - ii * TK;
            int gi = i0 + ii;
            As[kk][ii] = (gi < n && k0 + kk < n) ? A[(size_t)gi * n + k0 + kk] : 0.0;
        }
        // X tile: rows k0..k0+15, columns c0..c0+63
        for (int e = tid; e < TK * TC; e += 256) {
            int kk, cc;
            if (inner == 1) { cc = e / TK; kk = e - cc * TK; }   // k contiguous per column
            else { kk = e / TC; cc = e - kk * TC; }              // columns contiguous
            int col = c0 + cc;
            double v = 0.0;
            if (col < ncol && k0 + kk < n) {
                size_t o = (size_t)(col / inner), j = (size_t)(col % inner);
                v = in[o * (size_t)n * inner + (size_t)(k0 + kk) * inner + j];
            }
            Xs[kk][cc] = v;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < TK; kk++) {
            double av[RA], xv[4];
#pragma unroll
            for (int a = 0; a < RA; a++) av[a] = As[kk][ti + a];
#pragma unroll
            for (int q = 0; q < 4; q++) xv[q] = Xs[kk][tc + q];
#pragma unroll
            for (int a = 0; a < RA; a++)
#pragma unroll
                for (int q = 0; q < 4; q++) acc[a][q] += av[a] * xv[q];
        }
        __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < RA; a++) {
        int gi = i0 + ti + a;
        if (gi >= n) continue;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            int col = c0 + tc + q;
            if (col >= ncol) continue;
            size_t o = (size_t)(col / inner), j = (size_t)(col % inner);
            out[o * (size_t)n * inner + (size_t)gi * inner + j] = acc[a][q];
        }
    }
}

// k_axis_gemm for n <= 64 in one load phase: all of A (n x n) and the n x TC
// column tile of X in LDS behind one barrier, then every thread sums its
// 4 outputs over k = 0 .. n-1 in order (the same bits as k_axis_gemm).
template <int TC>
__global__ __launch_bounds__(256) void k_axis_gemm_small(const double *__restrict__ A, int n, int inner, int ncol,
                                                         const double *__restrict__ in, double *__restrict__ out) {
    constexpr int NMAX = 64, RA = TC / 16, TCQ = TC / 4;
    __shared__ double As[NMAX][NMAX + 1];   // As[k][i] = A[i][k]
    __shared__ double Xs[NMAX][TC + 1];
    const int tid = threadIdx.x;
    const int c0 = blockIdx.x * TC;
    for (int e = tid; e < n * n; e += 256) {
        const int i = e / n, k = e - i * n;
        As[k][i] = A[e];
    }
    for (int e = tid; e < n * TC; e += 256) {
        int kk, cc;
        if (inner == 1) { cc = e / n; kk = e - cc * n; }   // k contiguous per column
        else { kk = e / TC; cc = e - kk * TC; }            // columns contiguous
        const int col = c0 + cc;
        double v = 0.0;
        if (col < ncol) {
            const size_t o = (size_t)(col / inner), j = (size_t)(col % inner);
            v = in[o * (size_t)n * inner + (size_t)kk * inner + j];
        }
        Xs[kk][cc] = v;
    }
    __syncthreads();
    const int ti = (tid / TCQ) * RA, tc = (tid % TCQ) * 4;
    double acc[RA][4];
#pragma unroll
    for (int a = 0; a < RA; a++)
#pragma unroll
        for (int q = 0; q < 4; q++) acc[a][q] = 0.0;
    for (int k = 0; k < n; k++) {
        double av[RA], xv[4];
#pragma unroll
        for (int a = 0; a < RA; a++) av[a] = As[k][ti + a];
#pragma unroll
        for (int q = 0; q < 4; q++) xv[q] = Xs[k][tc + q];
#pragma unroll
        for (int a = 0; a < RA; a++)
#pragma unroll
            for (int q = 0; q < 4; q++) acc[a][q] += av[a] * xv[q];
    }
#pragma unroll
    for (int a = 0; a < RA; a++) {
        const int gi = ti + a;
        if (gi >= n) continue;
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int col = c0 + tc + q;
            if (col >= ncol) continue;
            const size_t o = (size_t)(col / inner), j = (size_t)(col % inner);
            out[o * (size_t)n * inner + (size_t)gi * inner + j] = acc[a][q];
        }
    }
}

// k_axis_gemm for n <= 256 without LDS; each output is the k-ordered sum of
// products of k_axis_gemm (same bits).
// Axis with stride 1 (a column is n contiguous values): thread i computes row
// i of RB consecutive columns (n threads rounded up to whole waves). Row k of
// At (= column k of A) is a coalesced load; X[col][k] is the same for every
// lane (a scalar load).
template <int RB>
__global__ __launch_bounds__(256) void k_axis_gemm_c(const double *__restrict__ At, int n, int ncol,
                                                    const double *__restrict__ in, double *__restrict__ out) {
    const int i = threadIdx.x;
    const int c0 = blockIdx.x * RB;
    if (i >= n) return;
    double acc[RB];
#pragma unroll
    for (int r = 0; r < RB; r++) acc[r] = 0.0;
#pragma unroll 8
    for (int k = 0; k < n; k++) {
        const double a = At[(size_t)k * n + i];
#pragma unroll
        for (int r = 0; r < RB; r++) {
            const int col = min(c0 + r, ncol - 1);
            acc[r] += a * in[(size_t)col * n + k];
        }
    }
#pragma unroll
    for (int r = 0; r < RB; r++)
        if (c0 + r < ncol) out[(size_t)(c0 + r) * n + i] = acc[r];
}

// Axis with a stride (inner) that is a multiple of 64: lane j is one of 64
// consecutive columns (the same outer index), and the work group computes RB
// rows of them. X[o][k][j] is a coalesced load; A[i][k] is the same for every
// lane (a scalar load).
template <int RB>
__global__ __launch_bounds__(64) void k_axis_gemm_r(const double *__restrict__ A, int n, int inner,
                                                    const double *__restrict__ in, double *__restrict__ out) {
    const int col = blockIdx.x * 64 + threadIdx.x;
    const int i0 = blockIdx.y * RB;
    const size_t o = (size_t)(col / inner), jj = (size_t)(col % inner);
    const double *__restrict__ x = in + o * (size_t)n * inner + jj;
    double acc[RB];
#pragma unroll
    for (int r = 0; r < RB; r++) acc[r] = 0.0;
#pragma unroll 8
    for (int k = 0; k < n; k++) {
        const double xv = x[(size_t)k * inner];
#pragma unroll
        for (int r = 0; r < RB; r++) {
            const int i = min(i0 + r, n - 1);
            acc[r] += A[(size_t)i * n + k] * xv;
        }
    }
    double *__restrict__ y = out + o * (size_t)n * inner + jj;
#pragma unroll
    for (int r = 0; r < RB; r++)
        if (i0 + r < n) y[(size_t)(i0 + r) * inner] = acc[r];
}

// k_axis_gemm for 64 < n <= 256 with the whole k range of a 16 x 16 output
// tile in LDS: the tile's 16 rows of A and 16 columns of X are loaded at once
// (every load in flight before the first product), then each thread sums its
// output over k in increasing order from 0.0 (the bits of k_axis_gemm). One
// load round trip per launch instead of one per k chunk or per few k.
constexpr int AXF = 16;  // output rows and columns per work group
__global__ __launch_bounds__(256) void k_axis_gemm_full(const double *__restrict__ A, int n, int inner, int ncol,
                                                        const double *__restrict__ in, double *__restrict__ out) {
    __shared__ double As[AXF * 257];  // As[r][k], row stride n + 1
    __shared__ double Xs[256 * (AXF + 1)];  // Xs[k][c]
    const int tid = threadIdx.x;
    const int i0 = blockIdx.y * AXF, c0 = blockIdx.x * AXF;
    const int sa = n + 1;
    double va[16], vx[16];
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int e = tid + q * 256, r = e / n, k = e - r * n;
        va[q] = (r < AXF && i0 + r < n) ? A[(size_t)(i0 + r) * n + k] : 0.0;
    }
    // X tile: element (k, c) of column c0 + c; consecutive threads take
    // consecutive k for the stride-1 axis and consecutive columns otherwise
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int e = tid + q * 256;
        int k, c;
        if (inner == 1) { c = e / n; k = e - c * n; }
        else { k = e / AXF; c = e - k * AXF; }
        const int col = c0 + c;
        double v = 0.0;
        if (k < n && c < AXF && col < ncol) {
            const size_t o = (size_t)(col / inner), jj = (size_t)(col % inner);
            v = in[(o * (size_t)n + k) * inner + jj];
        }
        vx[q] = v;
    }
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int e = tid + q * 256, r = e / n, k = e - r * n;
        if (r < AXF) As[r * sa + k] = va[q];
    }
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int e = tid + q * 256;
        int k, c;
        if (inner == 1) { c = e / n; k = e - c * n; }
        else { k = e / AXF; c = e - k * AXF; }
        if (k < n && c < AXF) Xs[k * (AXF + 1) + c] = vx[q];
    }
    __syncthreads();
    const int r = tid / AXF, c = tid - r * AXF;
    const int i = i0 + r, col = c0 + c;
    double acc = 0.0;
#pragma unroll 8
    for (int k = 0; k < n; k++) acc += As[r * sa + k] * Xs[k * (AXF + 1) + c];
    if (i < n && col < ncol) {
        const size_t o = (size_t)(col / inner), jj = (size_t)(col % inner);
        out[(o * (size_t)n + i) * inner + jj] = acc;
    }
}

// divide by the eigenvalues of the Kronecker-sum operator; the grid holds
// `ngrid` stacked level-1 grids of `total` points, grid g with shift[g]
// (Helmholtz: -s k^2; Laplacian: 0)
__global__ __launch_bounds__(WG) void k_eig_scale(double *__restrict__ g, const double *__restrict__ l0,
                                                  const double *__restrict__ l1, const double *__restrict__ l2,
                                                  int N0, int N1, int D, const double *__restrict__ shift,
                                                  size_t total, int ngrid) {
    size_t gi = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (gi >= total * ngrid) return;
    size_t gg = gi / total;
    size_t r = gi - gg * total;
    double ev = shift[gg];
    ev += l0[r % N0]; r /= N0;
    ev += l1[r % N1]; r /= N1;
    if (D == 3) ev += l2[r];
    g[gi] /= ev;
}

// ---- level-1 exact solve of 2D grids in four launches ----
//
// Gather and forward x (MODE 0), forward y and the division (1), inverse y (2),
// inverse x and scatter (3), each as k_axis_gemm_full forms an axis (a 16 x 16
// output tile per work group, the whole k range of its operands in LDS, each
// output one sum over k in increasing order), each over the grids of every
// coarse group at once. These launches are bound by latency (two load round
// trips and a chain of n sums), so what they cost is their number: 50 us per
// solve of 128 x 256 as seven launches, 31 us as four; a forest with five
// shapes of level 1 needed 35 launches.
struct L12Group {
    int N0, N1, ntree, nper;           // nper: blocks per tree
    size_t goff;                       // the group's grids in the scratch grids
    const double *Q[2], *P[2], *lam[2], *shift, *cs;
    const int *btab;
};
constexpr int L12_MAX = 8;  // groups per launch
struct L12Args {
    L12Group g[L12_MAX];
};

__host__ __device__ inline int l12_tiles(const L12Group &g, bool axis0) {
    const int n = axis0 ? g.N0 : g.N1, ncol = g.ntree * (axis0 ? g.N1 : g.N0);
    return ((n + AXF - 1) / AXF) * ((ncol + AXF - 1) / AXF);
}

template <int MODE, int M, typename T>
__global__ __launch_bounds__(256) void k_l1_2d(L12Args a, double *__restrict__ out, const double *__restrict__ in,
                                               const T *__restrict__ src, T *__restrict__ dst) {
    using LY = Lay<2, M>;
    constexpr bool AX0 = MODE == 0 || MODE == 3;
    __shared__ double As[AXF * 257];        // As[r][k], row stride n + 1
    __shared__ double Xs[256 * (AXF + 1)];  // Xs[k][c]
    int wg = blockIdx.x, gi = 0;
    while (wg >= l12_tiles(a.g[gi], AX0)) wg -= l12_tiles(a.g[gi++], AX0);
    const L12Group &g = a.g[gi];
    const int tid = threadIdx.x, N0 = g.N0, N1 = g.N1, nb0 = N0 / M;
    const int n = AX0 ? N0 : N1, nother = AX0 ? N1 : N0, ncol = g.ntree * nother;
    const int ti = (n + AXF - 1) / AXF, i0 = wg % ti * AXF, c0 = wg / ti * AXF, sa = n + 1;
    const double *__restrict__ A = MODE == 0 ? g.Q[0] : MODE == 1 ? g.Q[1] : MODE == 2 ? g.P[1] : g.P[0];
    const double *__restrict__ gin = in + g.goff;
    // 16 rows (or columns) of the tile by 16 consecutive k, 16 times: no
    // division per element, 128 contiguous bytes per 16 lanes
    const int hi = tid >> 4, lo = tid & 15;
    // this thread's column of X: along x its k runs over lo + 16 q, along y over hi + 16 q
    const int xc = c0 + (AX0 ? hi : lo), xt = min(xc / nother, g.ntree - 1), xj = xc - xt * nother;
    const bool xok = xc < ncol;
    double va[16], vx[16];
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int k = lo + 16 * q;
        va[q] = (k < n && i0 + hi < n) ? A[(size_t)(i0 + hi) * n + k] : 0.0;
    }
    if constexpr (MODE == 0) {
        const int *tb = g.btab + (size_t)xt * g.nper + (xj / M) * nb0;
        int blk[16];
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int k = lo + 16 * q;
            blk[q] = (xok && k < n) ? tb[k / M] : 0;
        }
        const double cs = g.cs[xt];
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int k = lo + 16 * q;
            vx[q] = (xok && k < n) ? cs * (double)src[(size_t)blk[q] * LY::V + LY::sidx(k % M, xj % M, 0)] : 0.0;
        }
    } else {
#pragma unroll
        for (int q = 0; q < 16; q++) {
            const int k = (AX0 ? lo : hi) + 16 * q;
            vx[q] = 0.0;
            if (xok && k < n) vx[q] = AX0 ? gin[(size_t)xc * N0 + k] : gin[((size_t)xt * N1 + k) * N0 + xj];
        }
    }
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int k = lo + 16 * q;
        if (k < n) As[hi * sa + k] = va[q];
    }
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int k = (AX0 ? lo : hi) + 16 * q;
        if (k < n) Xs[k * (AXF + 1) + (AX0 ? hi : lo)] = vx[q];
    }
    // the output's place, and what it takes besides the sum
    const int r = AX0 ? tid % AXF : tid / AXF, c = AX0 ? tid / AXF : tid % AXF;
    const int i = i0 + r, col = c0 + c, t = col / nother, j = col - t * nother;
    const bool ok = i < n && col < ncol;
    double ev = 1.0;
    int blk = 0;
    if (MODE == 1 && ok) {
        ev = g.shift[t];
        ev += g.lam[0][j];
        ev += g.lam[1][i];
    }
    if (MODE == 3 && ok) blk = g.btab[(size_t)t * g.nper + (j / M) * nb0 + i / M];
    __syncthreads();
    double acc = 0.0;
#pragma unroll 8
    for (int k = 0; k < n; k++) acc += As[r * sa + k] * Xs[k * (AXF + 1) + c];
    if (!ok) return;
    if (MODE == 0) out[g.goff + (size_t)col * N0 + i] = acc;
    if (MODE == 1) out[g.goff + ((size_t)t * N1 + i) * N0 + j] = acc / ev;
    if (MODE == 2) out[g.goff + ((size_t)t * N1 + i) * N0 + j] = acc;
    if (MODE == 3) dst[(size_t)blk * LY::V + LY::sidx(i % M, j % M, 0)] = (T)acc;
}

// ---- level-1 exact solve of 3D grids in three launches ----
//
// For stacked 3D grids [g][z][y][x] (x fastest) whose extents are multiples of
// 8 and at most 64, the transforms of k_axis_gemm (each output one sum over k
// in increasing order, from 0.0, of A[i][k] x[k], no fused multiply-add) in
// the order forward x, y, z; the eigenvalue division of k_eig_scale; inverse
// z, y, x. Each launch keeps a plane or a set of columns in LDS, so the nine
// launches of the axis-by-axis form (gather, three transforms, scale, three
// transforms, scatter) become three with the same bits:
//   k_l1_fwd_xy  plane (g, z), IC output columns: gather, forward x, forward y
//   k_l1_z       CC columns (y, x) of grid g: forward z, divide, inverse z
//   k_l1_inv_yx  plane (g, z), JC output rows: inverse y, inverse x, scatter
// BLK: the input (output) is the level-1 block field, gathered through btab
// (btab[g * nper + (bz * nb1 + by) * nb0 + bx] is the block at block position
// (bx, by, bz) of grid g) and scaled by cs[g]; otherwise a plain grid.

constexpr int L1T = 256;  // threads per work group of the three kernels (four waves)
constexpr int L1S = 65;   // LDS row stride of a staged plane (doubles)

// out[r] = sum over k < K of a(r, k) b(r, k), in increasing k from 0.0 (no
// fused multiply-add), for the R outputs of a thread at once
template <int R, class Fa, class Fb>
__device__ __forceinline__ void l1_dots(double (&out)[R], int K, Fa fa, Fb fb) {
#pragma unroll
    for (int r = 0; r < R; r++) out[r] = 0.0;
#pragma unroll 8
    for (int k = 0; k < K; k++) {
#pragma unroll
        for (int r = 0; r < R; r++) out[r] += fa(r, k) * fb(r, k);
    }
}

// rows of an n x m matrix (m <= 64) staged row by row: wave w takes rows w,
// w + 4, ..., lane = column; every load is issued before the first store
template <class Ld, class St>
__device__ __forceinline__ void l1_rows(int n, int m, Ld ld, St st) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    double v[16];
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int row = w + 4 * r;
        v[r] = (row < n && lane < m) ? ld(row, lane) : 0.0;
    }
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int row = w + 4 * r;
        if (row < n && lane < m) st(row, lane, v[r]);
    }
}

template <int M, typename T, bool BLK, int IC>
__global__ __launch_bounds__(L1T) void k_l1_fwd_xy(double *__restrict__ out, const T *__restrict__ src,
                                                   const double *__restrict__ gin, const int *__restrict__ btab,
                                                   const double *__restrict__ cs, const double *__restrict__ A0t,
                                                   const double *__restrict__ A1t, int N0, int N1, int N2) {
    using LY = Lay<3, M>;
    constexpr int RO = 64 * IC / L1T;  // outputs per thread
    constexpr int KS = L1T / IC;       // rows of a0 loaded per pass
    __shared__ double xs[64 * L1S];    // the plane X[y][x]
    __shared__ double a1[64 * 64];     // a1[k][j] = A1[j][k]
    __shared__ double a0[64 * IC];     // a0[k][il] = A0[i0 + il][k]
    __shared__ double y1[64 * IC];     // Y1[y][il]
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int z = blockIdx.x % N2, g = blockIdx.x / N2, i0 = blockIdx.y * IC;
    const int il = tid % IC, yb = tid / IC;
    double a0r[RO];
#pragma unroll
    for (int r = 0; r < RO; r++) {
        const int k = yb + KS * r;
        a0r[r] = k < N0 ? A0t[(size_t)k * N0 + i0 + il] : 0.0;
    }
    if constexpr (BLK) {
        const int nb0 = N0 / M, nb1 = N1 / M, nper = nb0 * nb1 * (N2 / M);
        const int *tb = btab + (size_t)g * nper + (z / M) * nb0 * nb1;
        const double c = cs[g];
        int blk[16];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int y = w + 4 * r;
            blk[r] = (y < N1 && lane < N0) ? tb[(y / M) * nb0 + lane / M] : 0;
        }
        double v[16];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int y = w + 4 * r;
            v[r] = (y < N1 && lane < N0)
                       ? c * (double)src[(size_t)blk[r] * LY::V + LY::sidx(lane % M, y % M, z % M)]
                       : 0.0;
        }
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int y = w + 4 * r;
            if (y < N1 && lane < N0) xs[y * L1S + lane] = v[r];
        }
    } else {
        const double *p = gin + ((size_t)g * N2 + z) * N1 * N0;
        l1_rows(N1, N0, [&](int y, int x) { return p[(size_t)y * N0 + x]; },
                [&](int y, int x, double v) { xs[y * L1S + x] = v; });
    }
    l1_rows(N1, N1, [&](int k, int j) { return A1t[(size_t)k * N1 + j]; },
            [&](int k, int j, double v) { a1[k * 64 + j] = v; });
#pragma unroll
    for (int r = 0; r < RO; r++) {
        const int k = yb + KS * r;
        if (k < N0) a0[k * IC + il] = a0r[r];
    }
    __syncthreads();
    // Y1[y][il] = sum_k A0[i0 + il][k] X[y][k], y = yb + KS r
    {
        double acc[RO];
        l1_dots(acc, N0, [&](int r, int k) { return a0[k * IC + il]; },
                [&](int r, int k) { return xs[(yb + KS * r) * L1S + k]; });
#pragma unroll
        for (int r = 0; r < RO; r++) y1[(yb + KS * r) * IC + il] = acc[r];
    }
    __syncthreads();
    // Y2[j][il] = sum_k A1[j][k] Y1[k][il], j = yb + KS r
    double acc[RO];
    l1_dots(acc, N1, [&](int r, int k) { return a1[k * 64 + yb + KS * r]; },
            [&](int r, int k) { return y1[k * IC + il]; });
    double *po = out + ((size_t)g * N2 + z) * N1 * N0 + i0 + il;
#pragma unroll
    for (int r = 0; r < RO; r++) {
        const int j = yb + KS * r;
        if (j < N1) po[(size_t)j * N0] = acc[r];
    }
}

// forward z, division by shift[g] + l0[x] + l1[y] + l2[z] (k_eig_scale's sum
// order), inverse z on CC consecutive columns c = y N0 + x of grid g
template <int CC>
__global__ __launch_bounds__(L1T) void k_l1_z(double *__restrict__ out, const double *__restrict__ in,
                                              const double *__restrict__ A2t, const double *__restrict__ B2t,
                                              const double *__restrict__ l0, const double *__restrict__ l1,
                                              const double *__restrict__ l2, const double *__restrict__ shift,
                                              int N0, int N1, int N2) {
    constexpr int RO = 64 * CC / L1T;  // outputs per thread
    constexpr int ZS = L1T / CC;       // z rows per pass
    __shared__ double am[64 * 64];     // am[k][zo] = A2[zo][k]
    __shared__ double bm[64 * 64];     // bm[k][zo] = B2[zo][k]
    __shared__ double ts[64 * CC];     // the columns, Y[z][cc]
    __shared__ double ws[64 * CC];     // the divided forward transform
    const int tid = threadIdx.x;
    const int ncb = N0 * N1 / CC;
    const int g = blockIdx.x / ncb, c0 = (blockIdx.x - g * ncb) * CC;
    const size_t plane = (size_t)N0 * N1;
    const int cc = tid % CC, zb = tid / CC;
    const double *pin = in + (size_t)g * N2 * plane + c0 + cc;
    double tv[RO];
#pragma unroll
    for (int r = 0; r < RO; r++) {
        const int zz = zb + ZS * r;
        tv[r] = zz < N2 ? pin[(size_t)zz * plane] : 0.0;
    }
    const int c = c0 + cc, y = c / N0, x = c - y * N0;
    double ev0 = shift[g];
    ev0 += l0[x];
    ev0 += l1[y];
    double ev[RO];
#pragma unroll
    for (int r = 0; r < RO; r++) {
        const int zo = zb + ZS * r;
        ev[r] = ev0 + (zo < N2 ? l2[zo] : 0.0);
    }
    l1_rows(N2, N2, [&](int k, int zo) { return A2t[(size_t)k * N2 + zo]; },
            [&](int k, int zo, double v) { am[k * 64 + zo] = v; });
    l1_rows(N2, N2, [&](int k, int zo) { return B2t[(size_t)k * N2 + zo]; },
            [&](int k, int zo, double v) { bm[k * 64 + zo] = v; });
#pragma unroll
    for (int r = 0; r < RO; r++) {
        const int zz = zb + ZS * r;
        if (zz < N2) ts[zz * CC + cc] = tv[r];
    }
    __syncthreads();
    {
        double acc[RO];
        l1_dots(acc, N2, [&](int r, int k) { return am[k * 64 + zb + ZS * r]; },
                [&](int r, int k) { return ts[k * CC + cc]; });
#pragma unroll
        for (int r = 0; r < RO; r++) ws[(zb + ZS * r) * CC + cc] = acc[r] / ev[r];
    }
    __syncthreads();
    double acc[RO];
    l1_dots(acc, N2, [&](int r, int k) { return bm[k * 64 + zb + ZS * r]; },
            [&](int r, int k) { return ws[k * CC + cc]; });
    double *po = out + (size_t)g * N2 * plane + c0 + cc;
#pragma unroll
    for (int r = 0; r < RO; r++) {
        const int zo = zb + ZS * r;
        if (zo < N2) po[(size_t)zo * plane] = acc[r];
    }
}

template <int M, typename T, bool BLK, int JC>
__global__ __launch_bounds__(L1T) void k_l1_inv_yx(T *__restrict__ dst, double *__restrict__ gout,
                                                   const double *__restrict__ in, const int *__restrict__ btab,
                                                   const double *__restrict__ B1t, const double *__restrict__ B0t,
                                                   int N0, int N1, int N2) {
    using LY = Lay<3, M>;
    constexpr int RO = JC / 4;       // outputs per thread: rows jl = w + 4 r, column = lane
    constexpr int KS = L1T / JC;     // rows of b1 loaded per pass
    __shared__ double vs[64 * L1S];  // the plane V[y][x]
    __shared__ double b0[64 * 64];   // b0[k][i] = B0[i][k]
    __shared__ double b1[64 * JC];   // b1[k][jl] = B1[j0 + jl][k]
    __shared__ double ts[JC * L1S];  // T[jl][x]
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int z = blockIdx.x % N2, g = blockIdx.x / N2, j0 = blockIdx.y * JC;
    const int jq = tid % JC, kb = tid / JC;
    double b1r[64 / KS];
#pragma unroll
    for (int r = 0; r < 64 / KS; r++) {
        const int k = kb + KS * r;
        b1r[r] = k < N1 ? B1t[(size_t)k * N1 + j0 + jq] : 0.0;
    }
    const double *pin = in + ((size_t)g * N2 + z) * N1 * N0;
    l1_rows(N1, N0, [&](int y, int x) { return pin[(size_t)y * N0 + x]; },
            [&](int y, int x, double v) { vs[y * L1S + x] = v; });
    l1_rows(N0, N0, [&](int k, int i) { return B0t[(size_t)k * N0 + i]; },
            [&](int k, int i, double v) { b0[k * 64 + i] = v; });
#pragma unroll
    for (int r = 0; r < 64 / KS; r++) {
        const int k = kb + KS * r;
        if (k < N1) b1[k * JC + jq] = b1r[r];
    }
    __syncthreads();
    // T[jl][x] = sum_k B1[j0 + jl][k] V[k][x], jl = w + 4 r, x = lane
    {
        double acc[RO];
        l1_dots(acc, N1, [&](int r, int k) { return b1[k * JC + w + 4 * r]; },
                [&](int r, int k) { return vs[k * L1S + lane]; });
#pragma unroll
        for (int r = 0; r < RO; r++) ts[(w + 4 * r) * L1S + lane] = acc[r];
    }
    __syncthreads();
    // U[jl][i] = sum_k B0[i][k] T[jl][k], i = lane
    double acc[RO];
    l1_dots(acc, N0, [&](int r, int k) { return b0[k * 64 + lane]; },
            [&](int r, int k) { return ts[(w + 4 * r) * L1S + k]; });
    if (lane >= N0) return;
    const int nb0 = N0 / M, nb1 = N1 / M, nper = nb0 * nb1 * (N2 / M);
#pragma unroll
    for (int r = 0; r < RO; r++) {
        const int j = j0 + w + 4 * r;
        if constexpr (BLK) {
            const int blk = btab[(size_t)g * nper + ((z / M) * nb1 + j / M) * nb0 + lane / M];
            dst[(size_t)blk * LY::V + LY::sidx(lane % M, j % M, z % M)] = (T)acc[r];
        } else {
            gout[(((size_t)g * N2 + z) * N1 + j) * N0 + lane] = acc[r];
        }
    }
}

// ---- the same for many stacked grids ----
//
// With hundreds of planes the launches are bound by FP64 arithmetic (a product
// and a sum each, 39 T/s on the chip), not by latency, and the split of a plane
// over work groups repeats its loads. Here a work group takes a whole plane
// (or 64 columns along z): lanes along one axis, and per wave eight (four)
// output rows at once, so that one LDS read per lane and k serves eight sums
// and the matrix row, equal for all lanes, comes through scalar loads. A work
// group reads its whole plane before it writes, so a launch may write in place.
// Same sums in the same order as k_l1_fwd_xy, k_l1_z and k_l1_inv_yx.

// rows row0 .. row0 + RB - 1 of A (n x n, row-major, n a multiple of 8) times
// the lane's vector x[k ks], into acc
template <int RB>
__device__ __forceinline__ void l1b_rows(double (&acc)[RB], const double *__restrict__ A, int row0, int n,
                                         const double *x, int ks) {
#pragma unroll
    for (int r = 0; r < RB; r++) acc[r] = 0.0;
    const double *a = A + (size_t)row0 * n;
    for (int k = 0; k < n; k += 8) {
        double xk[8];
#pragma unroll
        for (int i = 0; i < 8; i++) xk[i] = x[(k + i) * ks];
#pragma unroll
        for (int r = 0; r < RB; r++)
#pragma unroll
            for (int i = 0; i < 8; i++) acc[r] += a[(size_t)r * n + k + i] * xk[i];
    }
}

// forward x, then forward y, of plane blockIdx.x
template <int RB>
__global__ __launch_bounds__(L1T) void k_l1b_fwd_xy(double *out, const double *in, const double *__restrict__ A0,
                                                    const double *__restrict__ A1, int N0, int N1) {
    constexpr int RW = 16 / RB;  // row groups per wave
    __shared__ double xs[64 * L1S];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const double *p = in + (size_t)blockIdx.x * N1 * N0;
    l1_rows(N1, N0, [&](int y, int x) { return p[(size_t)y * N0 + x]; },
            [&](int y, int x, double v) { xs[y * L1S + x] = v; });
    __syncthreads();
    double acc[RW][RB];
    // Y1[y][i] = sum_k A0[i][k] X[y][k], lane = y
#pragma unroll
    for (int j = 0; j < RW; j++)
        if ((w + 4 * j) * RB < N0) l1b_rows(acc[j], A0, (w + 4 * j) * RB, N0, xs + lane * L1S, 1);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RW; j++)
        if ((w + 4 * j) * RB < N0)
#pragma unroll
            for (int r = 0; r < RB; r++) xs[lane * L1S + (w + 4 * j) * RB + r] = acc[j][r];
    __syncthreads();
    // Y2[j][i] = sum_k A1[j][k] Y1[k][i], lane = i
    double *po = out + (size_t)blockIdx.x * N1 * N0;
#pragma unroll
    for (int j = 0; j < RW; j++) {
        if ((w + 4 * j) * RB >= N1) continue;
        double v[RB];
        l1b_rows(v, A1, (w + 4 * j) * RB, N1, xs + lane, L1S);
        if (lane < N0)
#pragma unroll
            for (int r = 0; r < RB; r++) po[(size_t)((w + 4 * j) * RB + r) * N0 + lane] = v[r];
    }
}

// forward z, the eigenvalue division, inverse z of 64 columns (y, x)
template <int RB>
__global__ __launch_bounds__(L1T) void k_l1b_z(double *g, const double *__restrict__ A2,
                                               const double *__restrict__ B2, const double *__restrict__ l0,
                                               const double *__restrict__ l1, const double *__restrict__ l2,
                                               const double *__restrict__ shift, int N0, int N1, int N2) {
    constexpr int RW = 16 / RB;
    __shared__ double zs[64 * 64];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ncb = N0 * N1 / 64, gi = blockIdx.x / ncb, c = (blockIdx.x - gi * ncb) * 64 + lane;
    const size_t plane = (size_t)N0 * N1;
    double *p = g + (size_t)gi * N2 * plane + c;
    l1_rows(N2, 64, [&](int z, int) { return p[(size_t)z * plane]; },
            [&](int z, int i, double v) { zs[z * 64 + i] = v; });
    double ev0 = shift[gi];
    ev0 += l0[c % N0];
    ev0 += l1[c / N0];
    __syncthreads();
    double acc[RW][RB];
#pragma unroll
    for (int j = 0; j < RW; j++) {
        if ((w + 4 * j) * RB >= N2) continue;
        l1b_rows(acc[j], A2, (w + 4 * j) * RB, N2, zs + lane, 64);
#pragma unroll
        for (int r = 0; r < RB; r++) acc[j][r] = acc[j][r] / (ev0 + l2[(w + 4 * j) * RB + r]);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RW; j++)
        if ((w + 4 * j) * RB < N2)
#pragma unroll
            for (int r = 0; r < RB; r++) zs[((w + 4 * j) * RB + r) * 64 + lane] = acc[j][r];
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RW; j++) {
        if ((w + 4 * j) * RB >= N2) continue;
        double v[RB];
        l1b_rows(v, B2, (w + 4 * j) * RB, N2, zs + lane, 64);
#pragma unroll
        for (int r = 0; r < RB; r++) p[(size_t)((w + 4 * j) * RB + r) * plane] = v[r];
    }
}

// inverse y, then inverse x, of plane blockIdx.x, in place
template <int RB>
__global__ __launch_bounds__(L1T) void k_l1b_inv_yx(double *g, const double *__restrict__ B1,
                                                    const double *__restrict__ B0, int N0, int N1) {
    constexpr int RW = 16 / RB;
    __shared__ double vs[64 * L1S];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double *p = g + (size_t)blockIdx.x * N1 * N0;
    l1_rows(N1, N0, [&](int y, int x) { return p[(size_t)y * N0 + x]; },
            [&](int y, int x, double v) { vs[y * L1S + x] = v; });
    __syncthreads();
    double acc[RW][RB];
    // T[j][x] = sum_k B1[j][k] V[k][x], lane = x
#pragma unroll
    for (int j = 0; j < RW; j++)
        if ((w + 4 * j) * RB < N1) l1b_rows(acc[j], B1, (w + 4 * j) * RB, N1, vs + lane, L1S);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RW; j++)
        if ((w + 4 * j) * RB < N1)
#pragma unroll
            for (int r = 0; r < RB; r++) vs[((w + 4 * j) * RB + r) * L1S + lane] = acc[j][r];
    __syncthreads();
    // U[j][i] = sum_k B0[i][k] T[j][k], lane = j; back through LDS so that rows
    // leave whole
#pragma unroll
    for (int j = 0; j < RW; j++)
        if ((w + 4 * j) * RB < N0) l1b_rows(acc[j], B0, (w + 4 * j) * RB, N0, vs + lane * L1S, 1);
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RW; j++)
        if ((w + 4 * j) * RB < N0)
#pragma unroll
            for (int r = 0; r < RB; r++) vs[lane * L1S + (w + 4 * j) * RB + r] = acc[j][r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const int y = w + 4 * r;
        if (y < N1 && lane < N0) p[(size_t)y * N0 + lane] = vs[y * L1S + lane];
    }
}

// ---- mixed precision helpers ----

// u += e over n cells (FP64 += FP32)
__global__ __launch_bounds__(WG) void k_add_correction(double *__restrict__ u, const float *__restrict__ e, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) u[i] += (double)e[i];
}

// The end of a mixed-precision outer step on a grouped level, run from the
// finest level down: on every block of sibling group g, u += e if the block is
// a leaf (a covered block already holds the restriction of its children,
// written by the finer level's launch, and u += e there would be overwritten
// anyway) and e = 0; then the parent's cells get the restriction of the
// group's u (k_restrict's order) and e = 0. Work groups past ngroups do
// u += e, e = 0 on the leaf blocks leaves[0..nleafc) of the coarser level
// (used for the coarsest level, which has no parent). The values equal those
// of u += e everywhere followed by restrict! level by level. ZERO: the leaf
// blocks' u is known to be 0 (the first step of a solve from u = 0) and is
// not read: u = 0.0 + e. KEEPE: e is not cleared on the group's own blocks
// (the next correction's first sweep there reads none of it; the parents'
// e is cleared).
template <int D, int M, bool ZERO = false, bool KEEPE = false>
__global__ __launch_bounds__(256) void k_add_restrict(double *__restrict__ u, float *__restrict__ e,
                                                      const int *__restrict__ isleaf, const int *__restrict__ parent,
                                                      int blk0, unsigned ngroups, const int *__restrict__ leaves,
                                                      int nleafc) {
    using LY = Lay<D, M>;
    constexpr int NB = 1 << D, V = LY::V, MH = LY::MH;
    const int tid = threadIdx.x;
    if (blockIdx.x >= ngroups) {
        const int c0 = (int)(blockIdx.x - ngroups) * 256;
        for (int i = c0 + tid; i < c0 + 256 && i < nleafc * V; i += 256) {
            const size_t o = (size_t)leaves[i / V] * V + (size_t)(i % V);
            u[o] = (ZERO ? 0.0 : u[o]) + (double)e[o];
            e[o] = 0.0f;
        }
        return;
    }
    // every load of the thread's cells is issued before the first store
    // (a loop that stores between its loads waits out each load in turn)
    constexpr int PER = NB * V / 256;
    static_assert(NB * V % 256 == 0, "group cells must be a multiple of the work-group size");
    __shared__ double ut[NB * V];
    __shared__ int leaf[NB];
    const int g0 = blk0 + (int)blockIdx.x * NB;
    if (tid < NB) leaf[tid] = isleaf[g0 + tid];
    __syncthreads();
    float ev[PER];
    double uv[PER];
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = tid + 256 * j;
        const size_t o = (size_t)g0 * V + i;
        ev[j] = e[o];
        uv[j] = (ZERO && leaf[i / V]) ? 0.0 : u[o];
    }
#pragma unroll
    for (int j = 0; j < PER; j++) {
        const int i = tid + 256 * j;
        const size_t o = (size_t)g0 * V + i;
        double v = uv[j];
        if (leaf[i / V]) {
            v = (ZERO ? 0.0 : uv[j]) + (double)ev[j];
            u[o] = v;
        }
        if (!KEEPE) e[o] = 0.0f;
        ut[i] = v;
    }
    __syncthreads();
    const int pb = parent[g0];
    for (int i = tid; i < V; i += 256) {
        int X0, X1, X2;
        LY::decode(i, X0, X1, X2);
        const int k = (X0 >= MH ? 1 : 0) | (X1 >= MH ? 2 : 0) | (D == 3 && X2 >= MH ? 4 : 0);
        const int j0 = X0 - (k & 1) * MH, j1 = X1 - ((k >> 1) & 1) * MH, j2 = (D == 3) ? X2 - ((k >> 2) & 1) * MH : 0;
        double f = 0.0;
#pragma unroll
        for (int q = 0; q < LY::NC; q++) {
            const int i0 = q & 1, i1 = (q >> 1) & 1, i2 = (q >> 2) & 1;
            f += ut[k * V + LY::sidx(2 * j0 + i0, 2 * j1 + i1, D == 3 ? 2 * j2 + i2 : 0)];
        }
        const size_t o = (size_t)pb * V + i;
        u[o] = f / double(LY::NC);
        e[o] = 0.0f;
    }
}

}  // namespace srmg
