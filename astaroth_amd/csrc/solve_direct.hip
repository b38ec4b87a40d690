// solve_direct.hip -- one cell per thread fused RK3 substep. This is the simple, obviously-correct solve
// kernel: it is the parity anchor for the marching kernels, the fallback for what they do not cover
// (fields that are not one slab), and the kernel of FP32 gradients on grids that 64 columns do not
// divide. STAGED: a block's stencils are read from LDS (block_stage.h); else from global memory, the
// same arithmetic. Three substeps and fills, staged against not: 144 x 128 x 112 FP32 0.47 against 0.88 ms,
// 100 x 75 x 50 0.147 / 0.189, 48^3 0.056 / 0.076, 40^3 0.058 / 0.058, 32^3 0.0386 / 0.0355 (latency: 128
// blocks on 256 CUs); FP64 100 x 90 x 75 0.445 / 1.12 ms, 16^3 0.047 / 0.074, so FP64 always stages.
// Semantics: ref acc-runtime/samples/mhd_modular/mhdsolver.ac:586-636 fused into one pass (ref
// twopass_solve_intermediate + twopass_solve_final).
#include <type_traits>

#include "block_stage.h"
#include "kernels.h"
#include "mhd_common.h"

namespace acamd {

template <typename T, typename I>
__device__ __forceinline__ T der1(const T* __restrict__ f, I c, I s, const T* k)
{
    return k[1] * (f[c + s] - f[c - s]) + k[2] * (f[c + 2 * s] - f[c - 2 * s]) +
           k[3] * (f[c + 3 * s] - f[c - 3 * s]);
}
// Second (and upwind) derivative. CF: the cancellation-free form of the precise 32-bit mode,
// sum_o k_o ((f_o - f_0) + (f_-o - f_0)), whose weights sum to zero like the sum form's, so the
// centre weight drops out; differences of neighbouring values are exact in FP32.
template <bool CF, typename T, typename I>
__device__ __forceinline__ T der2(const T* __restrict__ f, I c, I s, const T* k)
{
    if constexpr (CF) {
        const T f0 = f[c];
        return k[1] * ((f[c + s] - f0) + (f[c - s] - f0)) +
               k[2] * ((f[c + 2 * s] - f0) + (f[c - 2 * s] - f0)) +
               k[3] * ((f[c + 3 * s] - f0) + (f[c - 3 * s] - f0));
    }
    return k[0] * f[c] + k[1] * (f[c + s] + f[c - s]) + k[2] * (f[c + 2 * s] + f[c - 2 * s]) +
           k[3] * (f[c + 3 * s] + f[c - 3 * s]);
}
// Mixed derivative; CF pairs the corners as (f(o,o) - f(o,-o)) - (f(-o,o) - f(-o,-o)).
template <bool CF, typename T, typename I>
__device__ __forceinline__ T derm(const T* __restrict__ f, I c, I sa, I sb, const T* k)
{
    T r = T(0);
#pragma unroll
    for (int o = 1; o <= 3; ++o) {
        if constexpr (CF)
            r += k[o] * ((f[c + o * sa + o * sb] - f[c + o * sa - o * sb]) -
                         (f[c - o * sa + o * sb] - f[c - o * sa - o * sb]));
        else
            r += k[o] * ((f[c + o * sa + o * sb] + f[c - o * sa - o * sb]) -
                         (f[c + o * sa - o * sb] + f[c - o * sa + o * sb]));
    }
    return r;
}

// The values are computed here: the compiler otherwise reads the LDS values of many stencils ahead of
// their sums and spills (57 registers in FP32, 162 in FP64).
template <typename T>
__device__ __forceinline__ void keep_here(T& a, T& b, T& c, T& d)
{
    asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
}

constexpr int ROW = BX * BZ;

// ROWS: a workgroup takes rows of 64 cells instead of a 16 x 4 x 4 block.
template <typename T, bool UPWD, bool ENTROPY, int KB, bool STAGED, bool ROWS>
__global__ void __launch_bounds__(BX * BY * BZ, (sizeof(T) == 4 && STAGED ? 2 : 1)) solve_direct_kernel(SolveArgs<T> a)
{
    __shared__ T lds[STAGED ? NF * BlockStage<T>::LPS : 1];
    constexpr int UX = ROWS ? ROW : BX, UY = BY, UZ = ROWS ? 1 : BZ;
    static_assert(!(STAGED && ROWS) && UX * UY * UZ == BX * BY * BZ, "one thread per cell");
    int3 o;
    if constexpr (!ROWS) {
        o = block_origin(a.nx, a.ny);
        if constexpr (STAGED)
            stage_block(a, o, a.wrap != 0, lds);
    }
    else {
        const int nbx = (a.nx + UX - 1) / UX, nby = (a.ny + UY - 1) / UY, b = (int)blockIdx.x;
        o = make_int3(b % nbx * UX, b / nbx % nby * UY, b / (nbx * nby));
    }
    const int tid = threadIdx.x;
    const int tx = tid % UX, ty = tid / UX % UY, tz = tid / (UX * UY);
    const int i = o.x + tx, j = o.y + ty, k = o.z + tz;
    const bool active = i < a.nx && j < a.ny && k < a.nz;
    // the precise mode (32-bit compensation records, FP32)
    constexpr bool CF = sizeof(T) == 4 && KB == 32;
    double u2 = 0.0;  // max |u_new|^2 (the courant timestep mode)
    const T dt = solve_dt(a);
    if constexpr (STAGED)
        memory_barrier();
    if (active) {
        const long long c = (long long)(i + R) + (long long)a.mx * (j + R) + a.sz * (k + R);
        // cell and strides where the stencils are read: in the staged box, or in the arrays
        using I = std::conditional_t<STAGED, int, long long>;
        const I sx = 1, sy = STAGED ? (I)BLX : (I)a.mx, sz = STAGED ? (I)(BLX * BLY) : (I)a.sz;
        const I l = STAGED ? (I)((tx + R) + BLX * (ty + R) + BLX * BLY * (tz + R)) : (I)c;
        const I st[3] = {sx, sy, sz};
        const T* in[NF];
#pragma unroll
        for (int q = 0; q < NF; ++q)
            in[q] = STAGED ? lds + q * BlockStage<T>::LPS : a.in[q];
        const Coeffs<T>& C = a.C;

        CellDerivs<T> d;
        T grad[NF][3], lap[NF], upw[4][3];
#pragma unroll
        for (int q = 0; q < NF; ++q) {
            const T* f = in[q];
#pragma unroll
            for (int ax = 0; ax < 3; ++ax)
                grad[q][ax] = der1(f, l, st[ax], C.d1[ax]);
            lap[q] = der2<CF>(f, l, sx, C.d2[0]) + der2<CF>(f, l, sy, C.d2[1]) + der2<CF>(f, l, sz, C.d2[2]);
            if constexpr (STAGED)
                keep_here(grad[q][0], grad[q][1], grad[q][2], lap[q]);
        }
        if (UPWD) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
#pragma unroll
                for (int ax = 0; ax < 3; ++ax)
                    upw[q][ax] = der2<CF>(in[q], l, st[ax], C.up[ax]);
                if constexpr (STAGED)
                    keep_here(upw[q][0], upw[q][1], upw[q][2], lap[q]);
            }
        }
        T val[NF];
#pragma unroll
        for (int q = 0; q < NF; ++q)
            val[q] = in[q][l];

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
        if (UPWD) {
            const T au[3] = {ac_abs(val[1]), ac_abs(val[2]), ac_abs(val[3])};
            d.upl = au[0] * upw[0][0] + au[1] * upw[0][1] + au[2] * upw[0][2];
#pragma unroll
            for (int q = 0; q < 3; ++q)
                d.upu[q] = upw[1 + q][0] * au[0] + upw[1 + q][1] * au[1] + upw[1 + q][2] * au[2];
        }
        else {
            d.upl = T(0);
            d.upu[0] = d.upu[1] = d.upu[2] = T(0);
        }
        // grad div: second derivatives on the diagonal, mixed derivatives off it
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const T* fx = in[1 + 3 * v];
            const T* fy = in[2 + 3 * v];
            const T* fz = in[3 + 3 * v];
            T* gd = v == 0 ? d.gdu : d.gda;
            gd[0] = der2<CF>(fx, l, sx, C.d2[0]) + derm<CF>(fy, l, sx, sy, C.mx[0]) +
                    derm<CF>(fz, l, sx, sz, C.mx[1]);
            gd[1] = derm<CF>(fx, l, sx, sy, C.mx[0]) + der2<CF>(fy, l, sy, C.d2[1]) +
                    derm<CF>(fz, l, sy, sz, C.mx[2]);
            gd[2] = derm<CF>(fx, l, sx, sz, C.mx[1]) + derm<CF>(fy, l, sy, sz, C.mx[2]) +
                    der2<CF>(fz, l, sz, C.d2[2]);
            if constexpr (STAGED)
                keep_here(gd[0], gd[1], gd[2], lap[3 * v + 1]);
        }

        T rhs[NF];
        mhd_rhs<T, UPWD, ENTROPY, CF>(d, a.P, rhs);

        T fnew[NF];
#pragma unroll
        for (int q = 0; q < NF; ++q) {
            if (q == 7 && !ENTROPY) {
                fnew[q] = val[q];
                a.out[q][c] = val[q];
                continue;
            }
            rk_update<T, KB>(a, q, c, val[q], rhs[q], dt, &fnew[q]);
            a.out[q][c] = fnew[q];
        }
        u2 = (double)fnew[1] * (double)fnew[1] + (double)fnew[2] * (double)fnew[2] +
             (double)fnew[3] * (double)fnew[3];
    }
    if (a.step == 2) {
        if (a.umax2_next != nullptr)
            wave_max_to_global(u2, a.umax2_next);
        if (a.time_acc != nullptr && blockIdx.x == 0 && tid == 0)
            *a.time_acc += (double)dt;
    }
}

// FP32 grids of at most one block per CU read the stencils straight from the caches.
template <typename T>
static bool staged(const SolveArgs<T>& a)
{
    return sizeof(T) == 8 || block_count(a.nx, a.ny, a.nz) > 256;
}

template <typename T>
bool direct_reads_periodic(const SolveArgs<T>& a)
{
    return staged(a) && a.nx >= R && a.ny >= R && a.nz >= R;
}

template <typename T, bool UPWD, bool ENTROPY, int KB>
static void launch_direct(const SolveArgs<T>& a, hipStream_t stream)
{
    const dim3 bpg((unsigned)block_count(a.nx, a.ny, a.nz)), tpb(BX * BY * BZ);
    if constexpr (sizeof(T) == 4) {
        if (!staged(a)) {
            // Rows, whose loads are wider, unless they make twice the workgroups (a step, rows / blocks: 300 x 5 x 7 37.0 /
            // 41.4 us, 33 x 33 x 20 35.6 / 40.9, 24 x 20 x 18 34.0 / 36.0; 32^3 35.0 / 34.6, 8^3 45 / 33, 7 x 5 x 300 90 / 47)
            const long long rows = (long long)((a.nx + ROW - 1) / ROW) * ((a.ny + BY - 1) / BY) * a.nz;
            if (rows < 2 * block_count(a.nx, a.ny, a.nz))
                hipLaunchKernelGGL((solve_direct_kernel<T, UPWD, ENTROPY, KB, false, true>), dim3((unsigned)rows), tpb, 0, stream, a);
            else
                hipLaunchKernelGGL((solve_direct_kernel<T, UPWD, ENTROPY, KB, false, false>), bpg, tpb, 0, stream, a);
            return;
        }
    }
    hipLaunchKernelGGL((solve_direct_kernel<T, UPWD, ENTROPY, KB, true, false>), bpg, tpb, 0, stream, a);
}

template <typename T>
void launch_solve_direct(const SolveArgs<T>& a, bool upwd, bool entropy, int kb, hipStream_t s)
{
#define AC_DISPATCH_KB(U, E)                                                          \
    do {                                                                             \
        if (kb == 0) launch_direct<T, U, E, 0>(a, s);                                \
        else if (kb == 8) launch_direct<T, U, E, (sizeof(T) == 4 ? 8 : 0)>(a, s);    \
        else if (kb == 16) launch_direct<T, U, E, (sizeof(T) == 4 ? 16 : 0)>(a, s);  \
        else launch_direct<T, U, E, (sizeof(T) == 4 ? 32 : 0)>(a, s);                \
    } while (0)
    if (upwd && entropy) AC_DISPATCH_KB(true, true);
    else if (upwd) AC_DISPATCH_KB(true, false);
    else if (entropy) AC_DISPATCH_KB(false, true);
    else AC_DISPATCH_KB(false, false);
#undef AC_DISPATCH_KB
}

template void launch_solve_direct<AcRealT>(const SolveArgs<AcRealT>&, bool, bool, int, hipStream_t);
template bool direct_reads_periodic<AcRealT>(const SolveArgs<AcRealT>&);

}  // namespace acamd
