// adjoint.hip -- tangent-linear and adjoint of one fused RK3 substep (no reference counterpart).
//
// Forward substep s (per field q, cell c):  w' = alpha_s w + dt R(f),  f' = f + beta_s w'.
// Tangent:  dw' = alpha_s dw + dt (J(f) df + dR/dnu dnu + dR/deta deta),  df' = df + beta_s dw'.
// Adjoint:  mu = lw' + beta_s lf',  lw = alpha_s mu,  lf = lf' + dt J(f)^T mu,
//           lnu += dt <mu, dR/dnu>,  leta += dt <mu, dR/deta>.
// J^T mu is computed in two stages: (A) per cell, the adjoint of every derivative quantity
// the right-hand side reads at a neighbour (NG = 47 fields, "derivative adjoints"), together
// with the pointwise parts: lw = alpha mu and lf += dt * (the adjoint of the cell's own value);
// (C) per output field, the transposed stencils applied to the derivative adjoints by a z-marching
// kernel, added to lf (first derivatives are antisymmetric, so their transpose is the negative;
// second, upwind and mixed ones are symmetric). Between them stands (B), the transpose of the forward
// halo copy: (C) reads periodic images.
#include <algorithm>
#include <cstdio>
#include <cstring>

#include "block_stage.h"
#include "kernels.h"
#include "mhd_adjoint.h"

namespace acamd {


template <typename T>
struct AdjArgs {
    SolveArgs<T> s;        // f = s.in (halos filled), coefficients, parameters, alpha, beta
    T* lf;                 // adjoint of f, NF slabs of m^3, updated in place
    T* lw;                 // adjoint of w, updated in place
    T* g;                  // derivative adjoints, NG fields
    long long g_row, g_plane, g_field;  // strides of g (values)
    double* partials;      // 2 per block (nu, eta)
    const T* df_in;        // tangent: df (halos filled)
    T* df_out;             // tangent: df'
    T* dw;                 // tangent: dw, updated in place
    T dnu, deta;
    long long count;       // m^3
};

template <typename T>
__device__ __forceinline__ T d1(const T* __restrict__ f, long long c, long long s, const T* k)
{
    return k[1] * (f[c + s] - f[c - s]) + k[2] * (f[c + 2 * s] - f[c - 2 * s]) +
           k[3] * (f[c + 3 * s] - f[c - 3 * s]);
}
template <typename T>
__device__ __forceinline__ T d2(const T* __restrict__ f, long long c, long long s, const T* k)
{
    return k[0] * f[c] + k[1] * (f[c + s] + f[c - s]) + k[2] * (f[c + 2 * s] + f[c - 2 * s]) +
           k[3] * (f[c + 3 * s] + f[c - 3 * s]);
}
template <typename T>
__device__ __forceinline__ T dm(const T* __restrict__ f, long long c, long long sa, long long sb,
                                const T* k)
{
    T r = T(0);
#pragma unroll
    for (int o = 1; o <= 3; ++o)
        r += k[o] * ((f[c + o * sa + o * sb] + f[c - o * sa - o * sb]) -
                     (f[c + o * sa - o * sb] + f[c - o * sa + o * sb]));
    return r;
}

// All derivative quantities of the eight fields at cell c (field q at base + q * count).
template <typename T, bool UPWD>
__device__ __forceinline__ void gather(const T* const* f, long long c, long long sy, long long sz,
                                       const Coeffs<T>& C, CellDerivs<T>& d, UpwindDirs<T>& up)
{
    const long long st[3] = {1, sy, sz};
    T val[NF], grad[NF][3], lap[NF];
#pragma unroll
    for (int q = 0; q < NF; ++q) {
        val[q] = f[q][c];
#pragma unroll
        for (int ax = 0; ax < 3; ++ax)
            grad[q][ax] = d1(f[q], c, st[ax], C.d1[ax]);
        lap[q] = d2(f[q], c, st[0], C.d2[0]) + d2(f[q], c, st[1], C.d2[1]) + d2(f[q], c, st[2], C.d2[2]);
    }
    d.lr = val[0];
    d.laplr = lap[0];
    d.s = val[7];
    d.laps = lap[7];
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        d.glr[ax] = grad[0][ax];
        d.gs[ax] = grad[7][ax];
        d.u[ax] = val[1 + ax];
        d.lapu[ax] = lap[1 + ax];
        d.lapa[ax] = lap[4 + ax];
#pragma unroll
        for (int bx = 0; bx < 3; ++bx) {
            d.gu[ax][bx] = grad[1 + ax][bx];
            d.ga[ax][bx] = grad[4 + ax][bx];
        }
    }
#pragma unroll
    for (int ax = 0; ax < 3; ++ax) {
        up.ul[ax] = UPWD ? d2(f[0], c, st[ax], C.up[ax]) : T(0);
#pragma unroll
        for (int i = 0; i < 3; ++i)
            up.uu[i][ax] = UPWD ? d2(f[1 + i], c, st[ax], C.up[ax]) : T(0);
    }
#pragma unroll
    for (int v = 0; v < 2; ++v) {
        const T* fx = f[1 + 3 * v];
        const T* fy = f[2 + 3 * v];
        const T* fz = f[3 + 3 * v];
        T* gd = v == 0 ? d.gdu : d.gda;
        gd[0] = d2(fx, c, st[0], C.d2[0]) + dm(fy, c, st[0], st[1], C.mx[0]) + dm(fz, c, st[0], st[2], C.mx[1]);
        gd[1] = dm(fx, c, st[0], st[1], C.mx[0]) + d2(fy, c, st[1], C.d2[1]) + dm(fz, c, st[1], st[2], C.mx[2]);
        gd[2] = dm(fx, c, st[0], st[2], C.mx[1]) + dm(fy, c, st[1], st[2], C.mx[2]) + d2(fz, c, st[2], C.d2[2]);
    }
    combine_upwind(d, up);
}

template <typename T>
__device__ __forceinline__ void cell_index(const SolveArgs<T>& a, bool& active, long long& c)
{
    const int i = threadIdx.x + blockIdx.x * blockDim.x;
    const int j = threadIdx.y + blockIdx.y * blockDim.y;
    const int k = blockIdx.z;
    active = i < a.nx && j < a.ny && k < a.nz;
    c = (long long)(i + R) + (long long)a.mx * (j + R) + a.sz * (k + R);
}

// ---------------------------------------------------------------- tangent
template <typename T, bool UPWD, bool ENTROPY>
__global__ void __launch_bounds__(256) tangent_kernel(AdjArgs<T> A)
{
    const SolveArgs<T>& a = A.s;
    bool active;
    long long c;
    cell_index(a, active, c);
    if (!active)
        return;
    CellDerivs<T> d, dd;
    UpwindDirs<T> up, dup;
    gather<T, UPWD>(a.in, c, a.mx, a.sz, a.C, d, up);
    const T* df[NF];
#pragma unroll
    for (int q = 0; q < NF; ++q)
        df[q] = A.df_in + (long long)q * A.count;
    gather<T, UPWD>(df, c, a.mx, a.sz, a.C, dd, dup);
    T rdot[NF];
    mhd_rhs_jvp<T, UPWD, ENTROPY>(d, up, dd, dup, a.P, A.dnu, A.deta, rdot);
#pragma unroll
    for (int q = 0; q < NF; ++q) {
        const long long o = (long long)q * A.count + c;
        if (q == 7 && !ENTROPY) {
            A.df_out[o] = df[q][c];
            continue;
        }
        T dwn = a.dt * rdot[q];
        if (a.step > 0)
            dwn = a.alpha * A.dw[o] + dwn;
        if (a.step < 2)
            A.dw[o] = dwn;
        A.df_out[o] = df[q][c] + a.beta * dwn;
    }
}

// ---------------------------------------------------------------- adjoint (A): local part
// One cell per thread on blocks of 16 x 4 x 4 cells, where the tiled form does not apply: on grids that its 64 x 4
// columns do not divide, and in FP64 where blocks are the faster form. All stencils read the block's box in LDS. 16 columns are one 64-byte line of the derivative adjoints in FP32. Reading the stencils
// from global memory it took 163 us at 72 x 60 x 50 FP64, now 70; whole adjoint substep 144 x 128 x 112 FP32
// 1206 -> 574 us. Two workgroups share a CU in FP32 (222 VGPRs), one in FP64; their load, stencil and store
// phases overlap only with each other's.
template <typename T, bool UPWD, bool ENTROPY>
__global__ void __launch_bounds__(BX * BY * BZ) adjoint_local_kernel(AdjArgs<T> A)
{
    constexpr int NW = BlockStage<T>::NW, LPS = BlockStage<T>::LPS;
    __shared__ T lds[NF * LPS];
    __shared__ double sh[2][NW];
    const SolveArgs<T>& a = A.s;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int3 o0 = block_origin(a.nx, a.ny);
    stage_block(a, o0, false, lds);
    const int tx = tid % BX, ty = tid / BX % BY, tz = tid / (BX * BY);
    const int i = o0.x + tx, j = o0.y + ty, k = o0.z + tz;
    const bool active = i < a.nx && j < a.ny && k < a.nz;
    const long long c = active ? (long long)(i + R) + (long long)a.mx * (j + R) + a.sz * (k + R) : 0;
    // threads outside the grid carry zeros through the barrier: every carried register is defined
    T lf[NF] = {}, mu[NF] = {};
    if (active) {
#pragma unroll
        for (int q = 0; q < NF; ++q) {
            const long long o = (long long)q * A.count + c;
            lf[q] = A.lf[o];
            mu[q] = A.lw[o] + a.beta * lf[q];
        }
    }
    memory_barrier();
    double pnu = 0.0, peta = 0.0;
    if (active) {
        CellDerivs<T> d, ad;
        UpwindDirs<T> up, aup;
        const T* f[NF];
#pragma unroll
        for (int q = 0; q < NF; ++q)
            f[q] = lds + q * LPS;
        gather<T, UPWD>(f, (tx + R) + BLX * (ty + R) + BLX * BLY * (tz + R), BLX, BLX * BLY, a.C, d, up);
        if (!ENTROPY)
            mu[7] = T(0);
        T anu, aeta;
        mhd_rhs_vjp<T, UPWD, ENTROPY>(d, up, mu, a.P, ad, aup, anu, aeta);
        pnu = (double)a.dt * (double)anu;
        peta = (double)a.dt * (double)aeta;
        T* g = A.g + i + A.g_row * j + A.g_plane * k;
        put_derivative_adjoints<UPWD>(ad, aup, [&](int f, T v) { g[f * A.g_field] = v; });
#pragma unroll
        for (int q = 0; q < NF; ++q) {
            const long long o = (long long)q * A.count + c;
            A.lw[o] = a.alpha * mu[q];
            if (q < 4 || (q == 7 && ENTROPY))
                A.lf[o] = lf[q] + a.dt * value_adjoint(ad, q);
        }
    }
    // block sums of the parameter sensitivities (FP64)
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        pnu += __shfl_xor(pnu, off, 64);
        peta += __shfl_xor(peta, off, 64);
    }
    if (lane == 0) {
        sh[0][wave] = pnu;
        sh[1][wave] = peta;
    }
    __syncthreads();
    if (tid == 0) {
        double s0 = 0.0, s1 = 0.0;
        for (int w = 0; w < NW; ++w) {
            s0 += sh[0][w];
            s1 += sh[1][w];
        }
        A.partials[2 * (long long)blockIdx.x + 0] = s0;
        A.partials[2 * (long long)blockIdx.x + 1] = s1;
    }
}

// Deterministic sum of the (nu, eta) block partials: stage 1 reduces contiguous ranges of partials per
// workgroup, stage 2 (one workgroup) adds the range sums into out. Up to PARAM_DIRECT partials stage 2
// takes them itself: sixteen a thread cost less than a launch (2.3 us of an adjoint substep: 32^3 FP32
// 31.7 -> 29.4 us, 128^3 393 -> 390.5).
constexpr int PARAM_RANGES = 256;
constexpr long long PARAM_DIRECT = 4096;

__device__ __forceinline__ void block_sum2(double& s0, double& s1)
{
    __shared__ double sh[2][4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        s0 += __shfl_xor(s0, off, 64);
        s1 += __shfl_xor(s1, off, 64);
    }
    if ((threadIdx.x & 63) == 0) {
        sh[0][threadIdx.x >> 6] = s0;
        sh[1][threadIdx.x >> 6] = s1;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double t0 = 0.0, t1 = 0.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
            t0 += sh[0][w];
            t1 += sh[1][w];
        }
        s0 = t0;
        s1 = t1;
    }
}

__global__ void __launch_bounds__(256) adjoint_param_stage1(const double* partials, long long nb,
                                                            double* ranges)
{
    const long long per = (nb + PARAM_RANGES - 1) / PARAM_RANGES;
    const long long b0 = per * blockIdx.x;
    const long long b1 = b0 + per < nb ? b0 + per : nb;
    double s0 = 0.0, s1 = 0.0;
    for (long long t = b0 + threadIdx.x; t < b1; t += blockDim.x) {
        s0 += partials[2 * t];
        s1 += partials[2 * t + 1];
    }
    block_sum2(s0, s1);
    if (threadIdx.x == 0) {
        ranges[2 * blockIdx.x] = s0;
        ranges[2 * blockIdx.x + 1] = s1;
    }
}

__global__ void __launch_bounds__(256) adjoint_param_stage2(const double* ranges, int n, double* out)
{
    double s0 = 0.0, s1 = 0.0;
    for (int t = threadIdx.x; t < n; t += blockDim.x) {
        s0 += ranges[2 * t];
        s1 += ranges[2 * t + 1];
    }
    block_sum2(s0, s1);
    if (threadIdx.x == 0) {
        out[0] += s0;
        out[1] += s1;
    }
}

// ---------------------------------------------------------------- adjoint (C): transposed stencils
// A thread owns an (x, y) column and walks a chunk of planes. An output field Q has a chain acc[k] of
// partial sums for planes p - 3 + k (k = 0..6), where p is the plane being read. Reading plane p pushes
//   * its pointwise and in-plane (x / y) contributions into acc[3] (plane p itself);
//   * its z-stencil contributions into acc[3 -+ i]: a value a(p) under the transposed first
//     derivative lands on plane p - i with -d1_i and on p + i with +d1_i; under second
//     derivative, upwind and D2z of grad(div) with the symmetric weights;
//   * the xz / yz mixed parts: D_i G(p) = G(x+i, p) - G(x-i, p) lands on p - i with +c_i and on
//     p + i with -c_i.
// Plane p - 3 is then complete (acc[0]) and its adjoint update is written. The derivative-adjoint
// fields that Q reads with in-plane (x / y) neighbours are DMA'd plane by plane into LDS with their
// radius-3 halo, one plane ahead; fields read only at the column come straight from memory. Halos
// are read from the periodic images, wrapped at any grid size, so the derivative adjoints need no
// halo fill.

// Fields of output Q that are read with in-plane neighbours ("staged"), in slot order: its own
// x / y first derivatives (those that exist), Laplacian and, for lnrho and u with upwinding, the
// x / y upwind operators; then the grad(div) fields G0, G1[, G2] of the vector (G2 only for the
// x and y components).
__host__ __device__ constexpr int own_staged_role(int Q, bool upwd, int slot)
{
    int n = 0;
    for (int role : {ROLE_DX, ROLE_DY, ROLE_LAP, ROLE_UPX, ROLE_UPY}) {
        if ((role == ROLE_UPX || role == ROLE_UPY) && !(upwd && Q < 4))
            continue;
        if (g_index(Q, role) < 0)
            continue;
        if (n == slot)
            return role;
        ++n;
    }
    return -1;
}
__host__ __device__ constexpr int own_staged_count(int Q, bool upwd)
{
    int n = 0;
    while (own_staged_role(Q, upwd, n) >= 0)
        ++n;
    return n;
}
// Slot of an own role among the staged fields of Q, or -1.
__host__ __device__ constexpr int staged_slot(int Q, bool upwd, int role)
{
    for (int sl = 0; sl < own_staged_count(Q, upwd); ++sl)
        if (own_staged_role(Q, upwd, sl) == role)
            return sl;
    return -1;
}
__host__ __device__ constexpr int staged_count(int Q, bool upwd)
{
    const int gd = (Q >= 1 && Q <= 6) ? ((Q - 1) % 3 == 2 ? 2 : 3) : 0;
    return own_staged_count(Q, upwd) + gd;
}
__host__ __device__ constexpr int staged_field(int Q, bool upwd, int slot)
{
    const int no = own_staged_count(Q, upwd);
    if (slot < no)
        return g_index(Q, own_staged_role(Q, upwd, slot));
    return (Q <= 3 ? G_GDU : G_GDA) + (slot - no);
}

// Fields of output Q read only at the column itself, in slot order: its own z first derivative
// (where it exists) and z upwind operator (lnrho and u with upwinding); then G2 of grad(div) for
// the z components.
__host__ __device__ constexpr int own_column_count(int Q, bool upwd)
{
    return (g_index(Q, ROLE_DZ) >= 0 ? 1 : 0) + ((upwd && Q < 4) ? 1 : 0);
}
__host__ __device__ constexpr int column_count(int Q, bool upwd)
{
    return own_column_count(Q, upwd) + ((Q == 3 || Q == 6) ? 1 : 0);
}
__host__ __device__ constexpr int column_field(int Q, bool upwd, int slot)
{
    const bool dz = g_index(Q, ROLE_DZ) >= 0;
    if (dz && slot == 0)
        return g_index(Q, ROLE_DZ);
    if (slot < own_column_count(Q, upwd))
        return g_index(Q, ROLE_UPZ);
    return (Q <= 3 ? G_GDU : G_GDA) + 2;
}

// Column blocks: 64 x 16 in FP32, else 32 x 16 or 16 x 16, whichever loads the fewest LDS cells for the
// grid (the radius-3 halo makes that 1.50, 1.63 and 1.89 per output cell).
constexpr int TY_T = 16;
template <typename T, int TX>
struct TransposeTile {
    static constexpr int LX = TX + 2 * R, LY = TY_T + 2 * R;
    static constexpr int NW = TX * TY_T / 64;
    static constexpr int WPE = (int)sizeof(T) / 4;
    static constexpr int LPW = LX * LY * WPE;
    static constexpr int NR = ((LPW + 63) / 64 + NW - 1) / NW;
    static constexpr int LPS = NR * NW * 64 / WPE;  // padded field-plane stride in LDS (elements)
};
constexpr int most_staged(bool upwd) { return upwd ? 8 : 6; }

__device__ __forceinline__ int wrap_index(int i, int n)
{
    while (i < 0)
        i += n;
    while (i >= n)
        i -= n;
    return i;
}

// Output field Q over one column block and z-chunk [z0, z1). lds0 and lds1 are two arrays, named
// statically by the two plane steps of an iteration: LDS reads of one then need not wait for the DMA
// into the other.
template <typename T, bool UPWD, int Q, int TX>
__device__ __forceinline__ void transpose_block(const AdjArgs<T>& A, T* lds0, T* lds1, int x0, int y0,
                                                int z0, int z1)
{
    using G = TransposeTile<T, TX>;
    constexpr int LX = G::LX, LPS = G::LPS, NR = G::NR, NW = G::NW, WPE = G::WPE;
    constexpr int NS = staged_count(Q, UPWD);
    constexpr int NC = column_count(Q, UPWD);
    static_assert(NS <= most_staged(UPWD), "LDS planes");
    const SolveArgs<T>& a = A.s;
    const int tid = threadIdx.x;
    const int tx = tid % TX, ty = tid / TX;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int sy = a.mx;
    const long long sz = a.sz;
    const Coeffs<T>& C = a.C;
    const bool inside = x0 + tx < a.nx && y0 + ty < a.ny;

    // DMA: every lane moves one dword per round; padding lanes re-read dword 0 of the plane
    unsigned g_off[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        int d = (wave + r * NW) * 64 + lane;
        if (d >= G::LPW)
            d = 0;
        const int e = d / WPE, wd = d - e * WPE;
        const int ly = e / LX, lx = e - ly * LX;
        const int gx = wrap_index(x0 + lx - R, a.nx), gy = wrap_index(y0 + ly - R, a.ny);
        g_off[r] = (unsigned)((gx + (int)A.g_row * gy) * (int)sizeof(T) + 4 * wd);
    }
    // byte offset of interior plane p (z wrapped periodically) within a field of g
    auto plane_b = [&](int p) {
        return A.g_plane * (long long)wrap_index(p, a.nz) * (long long)sizeof(T);
    };
    auto dma_plane = [&](int p, T* dst, long long nb) {
        const char* pb = (const char*)A.g + plane_b(p);
        const int first = opaque_s32(wave * (64 / WPE));
#pragma unroll
        for (int sl = 0; sl < NS; ++sl) {
            const char* src = pb + staged_field(Q, UPWD, sl) * nb;
#pragma unroll
            for (int r = 0; r < NR; ++r)
                __builtin_amdgcn_global_load_lds((const void*)(src + opaque(g_off[r])),
                                                 (lds_ptr_t)(dst + sl * LPS + first + r * NW * (64 / WPE)),
                                                 4, 0, 0);
        }
    };

    const int ctr = (ty + R) * LX + (tx + R);
    // columns past the grid read a column inside it and write nothing
    const int cx = inside ? x0 + tx : 0, cy = inside ? y0 + ty : 0;
    const unsigned colb0 = (unsigned)(((cx + R) + sy * (cy + R)) * (int)sizeof(T));
    const unsigned colg0 = (unsigned)((cx + (int)A.g_row * cy) * (int)sizeof(T));
    T acc[7];
#pragma unroll
    for (int k = 0; k < 7; ++k)
        acc[k] = T(0);
    // column values of the plane being processed, and of the next one (loaded a plane ahead)
    T col[NC], coln[NC];
    // lambda_f of the plane completed in this step (lfc) and in the next one (loaded a plane
    // ahead); the local stage has already added its pointwise part
    T lfc = T(0), lfn = T(0), done = T(0);
    auto load_cols = [&](int p, long long nb, unsigned colb, T* dst) {
        const char* pb = (const char*)A.g + plane_b(p);
#pragma unroll
        for (int c = 0; c < NC; ++c)
            dst[c] = *(const T*)(pb + column_field(Q, UPWD, c) * nb + colb);
    };
    // the output plane of step it is p - 3 = z0 - 2R + it (array plane z0 - R + it)
    auto out_off = [&](int it, long long nb, unsigned colb) {
        return Q * nb + sz * (long long)(z0 - R + it) * (long long)sizeof(T) + colb;
    };

    {
        const long long gb = A.g_field * (long long)sizeof(T);
        dma_plane(z0 - R, lds0, gb);
        load_cols(z0 - R, gb, colg0, col);
    }
    memory_barrier();
    const int np = z1 - z0 + 2 * R;
    auto step = [&](int it, const T* lds, T* next) {
        const int p = z0 - R + it;
        const long long nb = opaque_s64(A.count * (long long)sizeof(T));
        const long long gb = opaque_s64(A.g_field * (long long)sizeof(T));
        const unsigned colb = opaque(colb0);
        if (it + 1 < np) {
            dma_plane(p + 1, next, gb);
            load_cols(p + 1, gb, opaque(colg0), coln);
            if (it + 1 >= 2 * R)
                lfn = *(const T*)((const char*)A.lf + out_off(it + 1, nb, colb));
        }
        // the plane completed in the last step: stored here and not before the barrier, which waits for
        // every store
        if (it > 2 * R && inside)
            *(T*)((char*)A.lf + out_off(it - 1, nb, colb)) = done;
        auto lds_at = [&](int sl, int dx, int dy) -> T { return lds[sl * LPS + ctr + dy * LX + dx]; };
        auto d1x = [&](int sl) {
            return C.d1[0][1] * (lds_at(sl, 1, 0) - lds_at(sl, -1, 0)) +
                   C.d1[0][2] * (lds_at(sl, 2, 0) - lds_at(sl, -2, 0)) +
                   C.d1[0][3] * (lds_at(sl, 3, 0) - lds_at(sl, -3, 0));
        };
        auto d1y = [&](int sl) {
            return C.d1[1][1] * (lds_at(sl, 0, 1) - lds_at(sl, 0, -1)) +
                   C.d1[1][2] * (lds_at(sl, 0, 2) - lds_at(sl, 0, -2)) +
                   C.d1[1][3] * (lds_at(sl, 0, 3) - lds_at(sl, 0, -3));
        };
        auto sym = [&](int sl, int ax, const T* w) {
            const int ex = ax == 0, ey = ax == 1;
            return w[0] * lds_at(sl, 0, 0) + w[1] * (lds_at(sl, ex, ey) + lds_at(sl, -ex, -ey)) +
                   w[2] * (lds_at(sl, 2 * ex, 2 * ey) + lds_at(sl, -2 * ex, -2 * ey)) +
                   w[3] * (lds_at(sl, 3 * ex, 3 * ey) + lds_at(sl, -3 * ex, -3 * ey));
        };
        auto mixed_xy = [&](int sl) {
            T r = T(0);
#pragma unroll
            for (int o = 1; o <= 3; ++o)
                r += C.mx[0][o] * ((lds_at(sl, o, o) + lds_at(sl, -o, -o)) -
                                   (lds_at(sl, o, -o) + lds_at(sl, -o, o)));
            return r;
        };
        auto push_anti = [&](T v) {
#pragma unroll
            for (int o = 1; o <= 3; ++o) {
                acc[3 - o] -= C.d1[2][o] * v;
                acc[3 + o] += C.d1[2][o] * v;
            }
        };
        auto push_sym = [&](T v, const T* w) {
            acc[3] += w[0] * v;
#pragma unroll
            for (int o = 1; o <= 3; ++o) {
                acc[3 - o] += w[o] * v;
                acc[3 + o] += w[o] * v;
            }
        };
        auto push_mixed = [&](int sl, int ax) {
            const int ex = ax == 0, ey = ax == 1;
            const T* w = C.mx[ax == 0 ? 1 : 2];
#pragma unroll
            for (int o = 1; o <= 3; ++o) {
                const T D = w[o] * (lds_at(sl, o * ex, o * ey) - lds_at(sl, -o * ex, -o * ey));
                acc[3 - o] += D;
                acc[3 + o] -= D;
            }
        };

        // own stencils (staged and column slots as listed above)
        {
            constexpr int sx = staged_slot(Q, UPWD, ROLE_DX), sy_ = staged_slot(Q, UPWD, ROLE_DY);
            constexpr int sl = staged_slot(Q, UPWD, ROLE_LAP);
            constexpr int sux = staged_slot(Q, UPWD, ROLE_UPX), suy = staged_slot(Q, UPWD, ROLE_UPY);
            constexpr bool has_dz = g_index(Q, ROLE_DZ) >= 0;
            constexpr int cuz = has_dz ? 1 : 0;  // column slot of the z upwind operator
            T r = sym(sl, 0, C.d2[0]) + sym(sl, 1, C.d2[1]);
            if constexpr (sx >= 0)
                r -= d1x(sx);
            if constexpr (sy_ >= 0)
                r -= d1y(sy_);
            if constexpr (sux >= 0)
                r += sym(sux, 0, C.up[0]) + sym(suy, 1, C.up[1]);
            acc[3] += r;
            if constexpr (has_dz)
                push_anti(col[0]);
            push_sym(lds_at(sl, 0, 0), C.d2[2]);
            if constexpr (sux >= 0)
                push_sym(col[cuz], C.up[2]);
        }
        // grad(div v) parts (staged slots from the own-stencil count: G0, G1[, G2])
        if (Q >= 1 && Q <= 6) {
            constexpr int no = own_staged_count(Q, UPWD);
            const int comp = (Q - 1) % 3;
            if (comp == 0) {
                acc[3] += sym(no + 0, 0, C.d2[0]) + mixed_xy(no + 1);
                push_mixed(no + 2, 0);  // d_xz of G2
            }
            else if (comp == 1) {
                acc[3] += mixed_xy(no + 0) + sym(no + 1, 1, C.d2[1]);
                push_mixed(no + 2, 1);  // d_yz of G2
            }
            else {
                push_mixed(no + 0, 0);  // d_xz of G0
                push_mixed(no + 1, 1);  // d_yz of G1
                push_sym(col[NC - 1], C.d2[2]);
            }
        }

        if (it >= 2 * R)
            done = lfc + a.dt * acc[0];
#pragma unroll
        for (int k = 0; k < 6; ++k)
            acc[k] = acc[k + 1];
        acc[6] = T(0);
#pragma unroll
        for (int c = 0; c < NC; ++c)
            col[c] = coln[c];
        lfc = lfn;
        // plane p + 1 has landed and every wave is done with this one
        memory_barrier();
    };
    for (int it = 0; it < np; it += 2) {
        step(it, lds0, lds1);
        if (it + 1 < np)
            step(it + 1, lds1, lds0);
    }
    if (inside)
        *(T*)((char*)A.lf + out_off(np - 1, A.count * (long long)sizeof(T), colb0)) = done;
}

// All output fields in one launch: a workgroup takes one field of one column block and z-chunk. One
// field has 64 workgroups at 128^3 (64 x 16 columns, 32 planes), a quarter of the CUs; eight launches of
// them took 649 us FP32, this one 213, with 47 + 16 fields read or written at least once (530 MB). From
// 256^3 on, where one field fills the chip, both are bound by the memory (1.4 ms). On grids that 64
// columns do not divide, an unstaged kernel per field and a halo fill of the derivative adjoints took
// 0.85 ms (72 x 60 x 50 FP64); this takes 60 us. The fields of one block follow each other (all blocks of
// one field first) since neighbouring blocks in step share more than the fields of a block do (256^3
// FP32, whole adjoint substep: 2.93 ms against 3.24 with the fields of a block side by side).
template <typename T, bool UPWD, int TX>
__global__ void __launch_bounds__(TX * TY_T) adjoint_transpose_kernel(AdjArgs<T> A, int zchunk, int ntx,
                                                                      int nty, int nq)
{
    using G = TransposeTile<T, TX>;
    __shared__ T lds0[most_staged(UPWD) * G::LPS];
    __shared__ T lds1[most_staged(UPWD) * G::LPS];
    // Consecutive hardware block ids go to different XCDs, so each XCD is handed a contiguous range
    // of blocks, whose y neighbours and whose other fields then share its L2.
    const int ntiles = ntx * nty * ((A.s.nz + zchunk - 1) / zchunk);
    const int per_xcd = (ntiles + 7) >> 3;
    const int slot = (int)blockIdx.x >> 3;
    const int t = ((int)blockIdx.x & 7) * per_xcd + slot % per_xcd;
    if (t >= ntiles)
        return;
    const int x0 = t % ntx * TX, y0 = t / ntx % nty * TY_T, z0 = t / (ntx * nty) * zchunk;
    const int z1 = min(z0 + zchunk, A.s.nz);
    // the fields with the most to read first; ss last, which a run without entropy leaves out
    switch (slot / per_xcd) {
    case 0: transpose_block<T, UPWD, 1, TX>(A, lds0, lds1, x0, y0, z0, z1); break;
    case 1: transpose_block<T, UPWD, 2, TX>(A, lds0, lds1, x0, y0, z0, z1); break;
    case 2: transpose_block<T, UPWD, 3, TX>(A, lds0, lds1, x0, y0, z0, z1); break;
    case 3: transpose_block<T, UPWD, 4, TX>(A, lds0, lds1, x0, y0, z0, z1); break;
    case 4: transpose_block<T, UPWD, 5, TX>(A, lds0, lds1, x0, y0, z0, z1); break;
    case 5: transpose_block<T, UPWD, 6, TX>(A, lds0, lds1, x0, y0, z0, z1); break;
    case 6: transpose_block<T, UPWD, 0, TX>(A, lds0, lds1, x0, y0, z0, z1); break;
    default: transpose_block<T, UPWD, 7, TX>(A, lds0, lds1, x0, y0, z0, z1); break;
    }
}

// ---------------------------------------------------------------- launchers
template <typename T>
static dim3 grid_of(const SolveArgs<T>& a)
{
    return dim3((a.nx + 63) / 64, (a.ny + 3) / 4, a.nz);
}

template <typename T>
void launch_tangent(const AdjArgs<T>& A, bool upwd, bool entropy, hipStream_t s)
{
    const dim3 tpb(64, 4, 1), bpg = grid_of(A.s);
    if (upwd && entropy) hipLaunchKernelGGL((tangent_kernel<T, true, true>), bpg, tpb, 0, s, A);
    else if (upwd) hipLaunchKernelGGL((tangent_kernel<T, true, false>), bpg, tpb, 0, s, A);
    else if (entropy) hipLaunchKernelGGL((tangent_kernel<T, false, true>), bpg, tpb, 0, s, A);
    else hipLaunchKernelGGL((tangent_kernel<T, false, false>), bpg, tpb, 0, s, A);
}

// At least the workgroups of stage (A) in either form.
long long adjoint_num_blocks(int nx, int ny, int nz)
{
    return std::max((long long)((nx + 63) / 64) * ((ny + 3) / 4) * nz, block_count(nx, ny, nz));
}

struct TransposeShape {
    int tx, zchunk;
};

// The column block that loads the fewest cells, the wider of equals; then the z-chunk with the least of
// plane steps (six of them start a chunk up) over all workgroups per CU plus half of one workgroup's,
// which the last ones to finish leave the chip idle for.
static TransposeShape transpose_shape(int realsize, int nx, int ny, int nz, int nq)
{
    TransposeShape best{16, nz};
    long long least = 1ll << 62;
    for (int tx : {64, 32, 16}) {
        const long long cells = (long long)((nx + tx - 1) / tx) * (tx + 2 * R);
        if (cells < least && !(tx == 64 && realsize == 8)) {
            least = cells;
            best.tx = tx;
        }
    }
    // workgroups per CU: LDS holds one of 64 x 16 FP32 and 32 x 16 FP64, two of half their size
    const int per_cu = best.tx * realsize >= 256 ? 1 : (best.tx * realsize >= 128 ? 2 : 4);
    const long long tiles = (long long)((nx + best.tx - 1) / best.tx) * ((ny + TY_T - 1) / TY_T);
    double cost = 1e30;
    for (int nch = 1; nch <= nz; ++nch) {
        const int zc = (nz + nch - 1) / nch;
        const double groups = (double)(tiles * ((nz + zc - 1) / zc) * nq) / (256.0 * per_cu);
        const double c = (std::max(groups, 1.0) + 0.5) * (zc + 2 * R);
        if (c < cost) {
            cost = c;
            best.zchunk = zc;
        }
    }
    return best;
}

template <typename T>
void launch_adjoint(const AdjArgs<T>& A, bool upwd, bool entropy, double* param_grad,
                    hipStream_t s)
{
    // (A) derivative adjoints: the tiled kernel where the grid fits its 64 x 4 tiles, else blocks
    long long nb = 0;
    const AdjLocal<T> xl{A.g, A.g_row, A.g_plane, A.g_field, A.lf, A.lw, A.partials};
    if (!launch_adjoint_local_tiled<T>(A.s, xl, upwd, entropy, s, &nb)) {
        nb = block_count(A.s.nx, A.s.ny, A.s.nz);
        const dim3 bpg((unsigned)nb), tpb(BX * BY * BZ);
        if (upwd && entropy) hipLaunchKernelGGL((adjoint_local_kernel<T, true, true>), bpg, tpb, 0, s, A);
        else if (upwd) hipLaunchKernelGGL((adjoint_local_kernel<T, true, false>), bpg, tpb, 0, s, A);
        else if (entropy) hipLaunchKernelGGL((adjoint_local_kernel<T, false, true>), bpg, tpb, 0, s, A);
        else hipLaunchKernelGGL((adjoint_local_kernel<T, false, false>), bpg, tpb, 0, s, A);
    }
    double* sums = A.partials;
    int nsums = (int)std::min(nb, PARAM_DIRECT);
    if (nb > PARAM_DIRECT) {
        sums = A.partials + 2 * nb;
        nsums = PARAM_RANGES;
        hipLaunchKernelGGL(adjoint_param_stage1, dim3(PARAM_RANGES), dim3(256), 0, s,
                           (const double*)A.partials, nb, sums);
    }
    hipLaunchKernelGGL(adjoint_param_stage2, dim3(1), dim3(256), 0, s, (const double*)sums, nsums, param_grad);
    // (C) transposed stencils. Without the entropy equation ss is not evolved (f'_7 = f_7): its lambda_f
    // passes through and the local stage has set its lambda_w to alpha * 0.
    const int nq = entropy ? NF : NF - 1;
    const TransposeShape sh = transpose_shape((int)sizeof(T), A.s.nx, A.s.ny, A.s.nz, nq);
    const int ntx = (A.s.nx + sh.tx - 1) / sh.tx, nty = (A.s.ny + TY_T - 1) / TY_T;
    const int ntiles = ntx * nty * ((A.s.nz + sh.zchunk - 1) / sh.zchunk);
    const dim3 grid((unsigned)((ntiles + 7) / 8 * 8 * nq)), block(sh.tx * TY_T);
#define AC_TRANSPOSE(TX)                                                                           \
    do {                                                                                           \
        if (upwd) hipLaunchKernelGGL((adjoint_transpose_kernel<T, true, TX>), grid, block, 0, s, A, sh.zchunk, ntx, nty, nq); \
        else hipLaunchKernelGGL((adjoint_transpose_kernel<T, false, TX>), grid, block, 0, s, A, sh.zchunk, ntx, nty, nq);     \
    } while (0)
    if (sh.tx == 16)
        AC_TRANSPOSE(16);
    else if (sh.tx == 32)
        AC_TRANSPOSE(32);
#if !AC_DOUBLE_PRECISION
    else
        AC_TRANSPOSE(64);
#endif
#undef AC_TRANSPOSE
}

int adjoint_num_fields() { return NG; }

template void launch_tangent<AcRealT>(const AdjArgs<AcRealT>&, bool, bool, hipStream_t);
template void launch_adjoint<AcRealT>(const AdjArgs<AcRealT>&, bool, bool, double*, hipStream_t);

}  // namespace acamd

// ------------------------------------------------------------------ C entry points
#include "../../include/astaroth.h"

namespace acamd {
// defined in device.hip
void device_solve_args(Device d, SolveArgs<AcRealT>& a, int step, AcRealT dt);
hipStream_t device_stream(Device d, Stream s);
int device_id(Device d);
AcResult device_substep_states(Device d, hipStream_t s, AcRealT dt, AcRealT* scratch);
void device_out_fields(Device d, const AcRealT** out);
}  // namespace acamd

using namespace acamd;

// Layout of the derivative adjoints in the workspace: no halo, rows on 64-byte lines, so that stage (A)'s
// 47 stores per cell write whole lines (rows at the state's odd pitch share lines with their neighbours).
// Whole adjoint substep FP32: 256^3 2931 -> 2779 us, 128^3 421 -> 403. An odd number of lines per row
// (256^3 3014 us) and a skew between the fields (2827) were slower.
struct AdjLayout {
    long long row, plane, field;  // strides in values
};
static AdjLayout adjoint_layout(const int3 n)
{
    const long long line = 64 / (long long)sizeof(AcReal);
    const long long row = (n.x + line - 1) / line * line;
    return {row, row * n.y, row * n.y * n.z};
}

extern "C" size_t acAdjointWorkspaceBytes(const Device d)
{
    const int3 n = acDeviceGetLocalConfig(d).int3_params[AC_nlocal];
    const size_t g = (size_t)adjoint_layout(n).field * NG * sizeof(AcReal);
    const size_t partials =
        ((size_t)adjoint_num_blocks(n.x, n.y, n.z) + PARAM_RANGES) * 2 * sizeof(double);
    return ((g + 255) / 256) * 256 + partials;
}

extern "C" AcResult acDeviceIntegrateSubstepTangent(const Device d, const Stream stream,
                                                    const int step_number, const AcReal dt,
                                                    const AcReal* df_in, AcReal* df_out,
                                                    AcReal* dw, const double* dparams)
{
    if (step_number < 0 || step_number > 2) {
        fprintf(stderr, "astaroth_amd: acDeviceIntegrateSubstepTangent: step_number must be 0..2\n");
        return AC_FAILURE;
    }
    if (hipSetDevice(device_id(d)) != hipSuccess)
        return AC_FAILURE;
    const AcMeshInfo info = acDeviceGetLocalConfig(d);
    const int3 m = info.int3_params[AC_mlocal];
    AdjArgs<AcReal> A;
    memset(&A, 0, sizeof(A));
    device_solve_args(d, A.s, step_number, dt);
    A.count = (long long)m.x * m.y * m.z;
    A.df_in = df_in;
    A.df_out = df_out;
    A.dw = dw;
    A.dnu = dparams ? (AcReal)dparams[0] : (AcReal)0;
    A.deta = dparams ? (AcReal)dparams[1] : (AcReal)0;
    hipStream_t s = device_stream(d, stream);
    AcReal* ptrs[NF];
    for (int q = 0; q < NF; ++q)
        ptrs[q] = const_cast<AcReal*>(df_in) + (long long)q * A.count;
    launch_periodic_fill<AcReal>(ptrs, NF, A.s.nx, A.s.ny, A.s.nz, s);
    launch_tangent<AcReal>(A, info.bool_params[AC_lupwd] != 0, info.bool_params[AC_lentropy] != 0, s);
    return hipGetLastError() == hipSuccess ? AC_SUCCESS : AC_FAILURE;
}

// The adjoint of substep `step` at the state `f` (null: the current one), halos filled.
static AcResult adjoint_substep(const Device d, hipStream_t s, const int step, const AcReal dt, const AcReal* const* f,
                                AcReal* lam_f, AcReal* lam_w, void* workspace, double* param_grad)
{
    const AcMeshInfo info = acDeviceGetLocalConfig(d);
    const int3 m = info.int3_params[AC_mlocal];
    AdjArgs<AcReal> A;
    memset(&A, 0, sizeof(A));
    device_solve_args(d, A.s, step, dt);
    for (int q = 0; q < NF && f != nullptr; ++q)
        A.s.in[q] = f[q];
    A.count = (long long)m.x * m.y * m.z;
    A.lf = lam_f;
    A.lw = lam_w;
    A.g = (AcReal*)workspace;
    const AdjLayout lay = adjoint_layout(info.int3_params[AC_nlocal]);
    A.g_row = lay.row;
    A.g_plane = lay.plane;
    A.g_field = lay.field;
    const size_t gbytes = ((size_t)lay.field * NG * sizeof(AcReal) + 255) / 256 * 256;
    A.partials = (double*)((char*)workspace + gbytes);
    launch_adjoint<AcReal>(A, info.bool_params[AC_lupwd] != 0, info.bool_params[AC_lentropy] != 0,
                           param_grad, s);
    return hipGetLastError() == hipSuccess ? AC_SUCCESS : AC_FAILURE;
}

extern "C" AcResult acDeviceIntegrateSubstepAdjoint(const Device d, const Stream stream,
                                                    const int step_number, const AcReal dt,
                                                    AcReal* lam_f, AcReal* lam_w, void* workspace,
                                                    double* param_grad)
{
    if (step_number < 0 || step_number > 2) {
        fprintf(stderr, "astaroth_amd: acDeviceIntegrateSubstepAdjoint: step_number must be 0..2\n");
        return AC_FAILURE;
    }
    if (hipSetDevice(device_id(d)) != hipSuccess)
        return AC_FAILURE;
    return adjoint_substep(d, device_stream(d, stream), step_number, dt, nullptr, lam_f, lam_w, workspace, param_grad);
}

extern "C" AcResult acDeviceIntegrateStepAdjoint(const Device d, const Stream stream, const AcReal dt,
                                                 AcReal* scratch, AcReal* lam_f, AcReal* lam_w,
                                                 void* workspace, double* param_grad)
{
    if (hipSetDevice(device_id(d)) != hipSuccess)
        return AC_FAILURE;
    hipStream_t s = device_stream(d, stream);
    if (device_substep_states(d, s, dt, scratch) != AC_SUCCESS)
        return AC_FAILURE;
    const int3 m = acDeviceGetLocalConfig(d).int3_params[AC_mlocal];
    const long long count = (long long)m.x * m.y * m.z;
    const AcReal *second[NF], *third[NF];
    device_out_fields(d, second);
    for (int q = 0; q < NF; ++q)
        third[q] = scratch + q * count;
    const AcReal* const* f[3] = {nullptr, second, third};
    for (int step = 2; step >= 0; --step)
        if (adjoint_substep(d, s, step, dt, f[step], lam_f, lam_w, workspace, param_grad) != AC_SUCCESS)
            return AC_FAILURE;
    return AC_SUCCESS;
}
