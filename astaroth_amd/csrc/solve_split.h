// solve_split.h -- the role-split fused RK3 substep kernel for gfx950 (instantiated per precision
// and tile in solve_split_*.hip).
//
// Same semantics as solve_direct.hip (ref acc-runtime/samples/mhd_modular/mhdsolver.ac:586-636 in
// one fused pass), on any grid. A workgroup owns a TX x TY column block and marches a z-chunk, with
// one xy plane of all eight fields (radius-3 halo) in LDS per step, brought there by global -> LDS
// DMA into three plane buffers in rotation. Its threads come in two roles of TX * TY each, one column per thread and role:
//   hydro     lnrho, u: derivatives, right-hand sides (less the magnetic thread's force) and updates;
//   magnetic  A, ss: derivatives, right-hand sides and updates; the Lorentz force, the entropy part
//             of the pressure force and the exponentials of the cell.
// The two threads of a column hand each other the dozen values the other needs through LDS.
// Holding one half of a column's carried state each (about 90 values instead of 170), the threads
// fit a register budget at which twice as many waves are resident, which is what the z-march needs:
// in FP32 it is bound by VALU issue, and with two waves per SIMD the VALU idles whenever both wait. In FP64, at one
// wave per SIMD, it is bound by that wave's waits: 256^3 issues vector instructions in 27-36% of its cycles.
//
// One barrier per plane step. Before it, with plane p = z + 3 just landed: chain pushes, in-plane
// derivatives of plane p, and all of output plane z that needs no exchange value (those are
// double-buffered by step parity, so a wave one step ahead writes the other slot). After it: the
// updates and stores of plane z, the loads of the next output's w and compensation, and last the DMA of
// plane p + 3 into the buffer just released. The wait before a barrier counts on that order: it leaves only the
// newest operations in flight, which are the DMA of plane p + 2 issued at the end of the step before, so plane
// p + 1 has landed.
#pragma once

#include "kernels.h"

namespace acamd {

// Sum_o k_o-weighted neighbour sums of a symmetric stencil from S[o] = f(+o) + f(-o) (or, CF,
// f(+o) + f(-o) - 2 f(0), where the centre weight drops out).
template <bool CF, typename T>
__device__ __forceinline__ T sym3(const T* k, T f0, const T* S)
{
    if constexpr (CF)
        return k[1] * S[1] + k[2] * S[2] + k[3] * S[3];
    else
        return k[0] * f0 + k[1] * S[1] + k[2] * S[2] + k[3] * S[3];
}
template <bool CF, typename T>
__device__ __forceinline__ T pair_sum(T p, T m, T f0)
{
    if constexpr (CF)
        return (p - f0) + (m - f0);
    else
        return p + m;
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// A role's half of a cell's compensation record (NF entries of KB bits): hydro holds the entries of
// fields 0..3, magnetic those of 4..7; 4, 8 or 16 bytes, moved in one access.
template <int KB, int ROLE>
struct CompPart {
    uint32_t w[KB > 0 ? KB / 8 : 1];
};
typedef __attribute__((address_space(1))) uint32_t gu32;
typedef __attribute__((address_space(1))) u32x2 gu64;
typedef __attribute__((address_space(1))) u32x4 gu128;
template <int KB, int ROLE>
__device__ __forceinline__ CompPart<KB, ROLE> comp_part_load(const char* base, unsigned off)
{
    CompPart<KB, ROLE> c{};
    const gchar* p = sbase(base) + (off + ROLE * (KB / 2));
    if constexpr (KB == 8) {
        c.w[0] = *(const gu32*)p;
    }
    else if constexpr (KB == 16) {
        const u32x2 v = *(const gu64*)p;
        c.w[0] = v.x;
        c.w[1] = v.y;
    }
    else if constexpr (KB == 32) {
        const u32x4 v = *(const gu128*)p;
        c.w[0] = v.x;
        c.w[1] = v.y;
        c.w[2] = v.z;
        c.w[3] = v.w;
    }
    return c;
}
// Raw (sign-extended) entry of the role's field i.
template <int KB, int ROLE>
__device__ __forceinline__ int comp_part_get(const CompPart<KB, ROLE>& c, int i)
{
    if constexpr (KB == 8)
        return (int)(c.w[0] << (24 - 8 * i)) >> 24;
    else if constexpr (KB == 16)
        return (int)(c.w[i >> 1] << (16 - 16 * (i & 1))) >> 16;
    else if constexpr (KB == 32)
        return (int)c.w[i];
    else
        return 0;
}
template <int KB, int ROLE>
__device__ __forceinline__ void comp_part_store(char* base, unsigned off, const int* raw)
{
    gchar* p = sbase(base) + (off + ROLE * (KB / 2));
    const uint32_t r0 = (uint32_t)raw[0], r1 = (uint32_t)raw[1], r2 = (uint32_t)raw[2],
                   r3 = (uint32_t)raw[3];
    if constexpr (KB == 8)
        *(gu32*)p = (r0 & 0xffu) | ((r1 & 0xffu) << 8) | ((r2 & 0xffu) << 16) | (r3 << 24);
    else if constexpr (KB == 16)
        *(gu64*)p = u32x2{(r0 & 0xffffu) | (r1 << 16), (r2 & 0xffffu) | (r3 << 16)};
    else if constexpr (KB == 32)
        *(gu128*)p = u32x4{r0, r1, r2, r3};
}

// Exchange values of an output cell in LDS: hydro -> magnetic u, grad lnrho, lap lnrho and the viscous
// heating per mass; magnetic -> hydro the part of the momentum equation it holds (entropy pressure
// gradient less Lorentz force per mass) and cs^2. Without entropy only u and the force.
enum { X_F = 0, X_U = 3, X_CS2 = 6, X_GLR = 7, X_LAPLR = 10, X_VISC = 11 };

// End of a plane step: this wave's exchange values are in LDS and all its memory operations but the
// newest NEWEST (the DMA issued last) are done; then the workgroup barrier. The bare barrier, since
// the fence of __syncthreads waits for the DMA too; the clobbers keep every access on its side.
template <int NEWEST>
__device__ __forceinline__ void step_barrier(bool dma_in_flight)
{
    static_assert(NEWEST < 64, "vmcnt has six bits");
    asm volatile("" ::: "memory");
    if (dma_in_flight)
        __builtin_amdgcn_s_waitcnt((NEWEST & 15) | (7 << 4) | ((NEWEST >> 4) << 14));
    else
        __builtin_amdgcn_s_waitcnt(7 << 4);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The kernel's first argument (at the start of the kernel argument segment) through a pointer the
// optimiser does not follow across plane steps. FP64 reads its stencil constants through it: they are
// then loaded again each step (scalar loads, cached) instead of held, two scalar registers each, and
// spilled across the unrolled loop.
template <typename S>
__device__ __forceinline__ const S* step_args()
{
    typedef const __attribute__((address_space(4))) S karg;
    return (const S*)(karg*)opaque_s64((long long)__builtin_amdgcn_kernarg_segment_ptr());
}

template <int V>
struct IntC {
    static constexpr int value = V;
};

template <typename T, int TX, int TY>
struct SplitGeom {
    static constexpr int LX = TX + 2 * R, LY = TY + 2 * R, LP = LX * LY;
    static constexpr int NT = TX * TY;                // threads per role
    static constexpr int NW = NT / 64;                // waves per role
    static constexpr int WPE = (int)sizeof(T) / 4;    // dwords per value
    static constexpr int LPW = LP * WPE;              // dwords per field-plane
    static constexpr int NCHUNK = (LPW + 63) / 64;    // wave-wide DMA chunks (one dword per lane)
    static constexpr int NR = (NCHUNK + NW - 1) / NW; // chunks per wave: role r loads fields 4r..4r+3
    static constexpr int LPS = NR * NW * 64 / WPE;    // LDS stride of a field-plane (values)
};

// FP32: two waves per SIMD (one workgroup of 256 columns per CU, or two of 128); FP64: one, with twice
// the registers (its planes leave no LDS for a second workgroup of 128 columns).
template <typename T, bool UPWD, bool ENTROPY, int KB, int TX, int TY, int STEP>
__global__ void __launch_bounds__(2 * TX* TY, (sizeof(T) == 4 ? 2 : 1))
    solve_split_kernel(SolveArgs<T> a, int zchunk, int ntx, int nty, int nchunks)
{
    typedef SplitGeom<T, TX, TY> G;
    constexpr int LX = G::LX, NT = G::NT, NW = G::NW, NR = G::NR, LPS = G::LPS, WPE = G::WPE;
    constexpr int NX = ENTROPY ? 12 : 6;
    // the precise 32-bit mode: cancellation-free second, upwind and mixed derivatives
    constexpr bool CF = sizeof(T) == 4 && KB == 32;
    static_assert(NT % 64 == 0, "a role must be whole waves");
    // Three plane buffers as three variables, each named statically in its step of the plane loop
    // (unrolled by three): the compiler then knows that a read of one does not touch what the DMA
    // in flight writes, and puts no wait for the DMA before it.
    __shared__ T lds0[NF * LPS];
    __shared__ T lds1[NF * LPS];
    __shared__ T lds2[NF * LPS];
    __shared__ T xch[2][NX][NT];
    __shared__ double wmax[STEP == 2 ? NW : 1];

    // XCD-aware numbering: workgroup b runs on XCD b % 8; each XCD gets a contiguous range of
    // tiles (x fastest, then y, then chunk), whose halo rows then share its L2
    const int nblocks = ntx * nty * nchunks;
    int bid = blockIdx.x;
    if ((nblocks & 7) == 0)
        bid = (bid & 7) * (nblocks >> 3) + (bid >> 3);
    const int tile_x = bid % ntx;
    const int rest = bid / ntx;
    const int tile_y = rest % nty;
    const int chunk = rest / nty;

    if (STEP == 0 && blockIdx.x == 0 && threadIdx.x == 0) {
        // the maxima that substep 2 of this step reduces into, and the call's time at its first step
        if (a.umax2_next != nullptr)
            a.umax2_next[0] = a.umax2_next[1] = 0;
        if (a.time_acc != nullptr)
            *a.time_acc = 0.0;
    }
    const int wave_all = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int role = wave_all >= NW ? 1 : 0;
    const int wave = wave_all - role * NW;
    const int lane = threadIdx.x & 63;
    const int tid = wave * 64 + lane;  // column within the tile
    const int tx = tid % TX, ty = tid / TX;
    const int x0 = tile_x * TX, y0 = tile_y * TY, z0 = chunk * zchunk;
    const int zc = min(zchunk, a.nz - z0);
    const int gx = x0 + tx, gy = y0 + ty;
    const bool inside = gx < a.nx && gy < a.ny;
    const int sy = a.mx;

    // DMA source of this lane: chunk j = wave + r NW covers dwords [64 j, 64 j + 64) of a
    // field-plane. Halo values come from the periodic image (wrap) or from the stored halo; lanes
    // past the plane or past the array (ragged edge tiles) re-read a valid address, unused.
    unsigned g_off[NR];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
        int d = (wave + r * NW) * 64 + lane;
        if (d >= G::LPW)
            d = 0;
        const int e = d / WPE, wd = d - e * WPE;
        const int ly = e / LX, lx = e - ly * LX;
        int hx = x0 + lx, hy = y0 + ly;
        if (a.wrap) {
            hx += hx < R ? a.nx : (hx >= a.nx + R ? -a.nx : 0);
            hy += hy < R ? a.ny : (hy >= a.ny + R ? -a.ny : 0);
        }
        hx = min(hx, a.mx - 1);
        hy = min(hy, a.my - 1);
        g_off[r] = (unsigned)((hx + sy * hy) * (int)sizeof(T) + 4 * wd);
    }
    // DMA of interior plane p (array plane p + R) of this role's fields into buffer dst
    auto dma_plane = [&](T* buf, int p, long long fsb, const SolveArgs<T>& K) __attribute__((always_inline)) {
        if (K.wrap)
            p += p < 0 ? K.nz : (p >= K.nz ? -K.nz : 0);
        const char* src0 = (const char*)K.in[0] + K.sz * (long long)(p + R) * (long long)sizeof(T) +
                           4 * role * fsb;
        unsigned go[NR];
#pragma unroll
        for (int r = 0; r < NR; ++r)
            go[r] = opaque(g_off[r]);
        const int first = opaque_s32(__builtin_amdgcn_readfirstlane(4 * role * LPS + wave * (64 / WPE)));
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            if (!ENTROPY && f == 3 && role == 1)
                break;  // ss is only copied
            const char* src = src0 + f * fsb;
#pragma unroll
            for (int r = 0; r < NR; ++r)
                __builtin_amdgcn_global_load_lds(
                    (const void*)(src + go[r]),
                    (lds_ptr_t)(buf + (first + f * LPS + r * NW * (64 / WPE))), 4, 0, 0);
        }
    };

    const T dt = solve_dt(a);
    const int ctr = (ty + R) * LX + (tx + R);
    // in-plane offset of the column; threads outside the interior use its last row / column, so
    // their loads stay in bounds
    const unsigned ioff = (unsigned)((min(gx, a.nx - 1) + R) + sy * (min(gy, a.ny - 1) + R));
    // max |u_new|^2, NaN while there is no number in it: the timestep of a state whose velocity is NaN all over
    // is NaN, as with the direct kernel
    double u2max = __builtin_nan("");

    const int niter = zc + 2 * R;
    {
        const long long fsb = a.fstride * (long long)sizeof(T);
        dma_plane(lds0, z0 - R, fsb, a);
        dma_plane(lds1, z0 - R + 1, fsb, a);
        dma_plane(lds2, z0 - R + 2, fsb, a);
    }
    plane_barrier();

    if (role == 0) {
        // ================================================================ hydro
        constexpr int NQ = 4;
        T q[NQ][9], ch[3][9];  // windows of 7: step PH of the loop uses entries PH .. PH + 6
        // ch: chains of (nu / 3 + zeta) grad(div u) and, from the plane's own step on, the in-plane
        // part of the momentum right-hand side.
        // In-plane terms of planes p - 3 .. p - 1: d_x, d_y and lap of lnrho, d_x, d_y of u, and the
        // in-plane part of the continuity right-hand side
        struct Pl {
            T lr_dx, lr_dy, lr_lap, cont, u_dx[3], u_dy[3];
        } dly[3] = {};  // of plane p - 3 + k: entry (PH + k) % 3
#pragma unroll
        for (int f = 0; f < NQ; ++f)
#pragma unroll
            for (int i = 0; i < 9; ++i)
                q[f][i] = T(0);
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int i = 0; i < 9; ++i)
                ch[c][i] = T(0);
        // w and the compensation of the next output cell, loaded a step ahead
        T wpre[NQ];
        CompPart<KB, 0> crec{};
#pragma unroll
        for (int f = 0; f < NQ; ++f)
            wpre[f] = T(0);
        auto prefetch = [&](int it, long long fsb, unsigned iob, const SolveArgs<T>& K) __attribute__((always_inline)) {
            const long long pob = K.sz * (long long)(z0 - R + it) * (long long)sizeof(T);
            if (STEP > 0) {
#pragma unroll
                for (int f = 0; f < NQ; ++f)
                    wpre[f] = ld_g<T>(sbase((char*)K.w[0] + (f * fsb + pob)), iob);
            }
            if (KB > 0)
                crec = comp_part_load<KB, 0>((char*)K.comp[0] + pob / (long long)sizeof(T) * (NF * KB / 8),
                                             iob / (unsigned)sizeof(T) * (unsigned)(NF * KB / 8));
        };
        auto step = [&](auto phase, T* buf, int it) __attribute__((always_inline)) {
            constexpr int PH = decltype(phase)::value;
            const bool has_out = it >= 2 * R;
            const SolveArgs<T>& K = *step_args<SolveArgs<T>>();
            const SolveArgs<T>& A = sizeof(T) == 8 ? K : a;
            const Coeffs<T>& C = A.C;
            const PhysParams<T>& P = A.P;
            const int p = z0 - R + it;
            const int cur = it & 1;
            const unsigned iob = opaque(ioff * (unsigned)sizeof(T));
            const long long fsb = opaque_s64(K.fstride * (long long)sizeof(T));
            const long long pob = K.sz * (long long)p * (long long)sizeof(T);  // array plane p - 3 + R
            const T* const L = buf + ctr;
            auto at = [&](int f, int dx, int dy) __attribute__((always_inline)) -> T {
                return L[f * LPS + dy * LX + dx];
            };
#pragma unroll
            for (int f = 0; f < NQ; ++f)
                q[f][PH + 6] = at(f, 0, 0);

            Pl nv = dly[PH];
            // z-chains of grad(div u): plane p adds +c_i D(p) to plane p - i, -c_i D(p) to p + i
            {
                T dxz = T(0), dyz = T(0), dxx = T(0), dyy = T(0);
#pragma unroll
                for (int i = 1; i <= 3; ++i) {
                    const T Dxz = at(3, i, 0) - at(3, -i, 0);
                    const T Dyz = at(3, 0, i) - at(3, 0, -i);
                    const T Dxx = at(1, i, 0) - at(1, -i, 0);
                    const T Dyy = at(2, 0, i) - at(2, 0, -i);
                    const T kx = A.mxv[1][i], ky = A.mxv[2][i];
                    const T ez = kx * Dxx + ky * Dyy;
                    ch[0][PH + 3 - i] = ac_fma(kx, Dxz, ch[0][PH + 3 - i]);
                    ch[0][PH + 3 + i] = ac_fma(-kx, Dxz, ch[0][PH + 3 + i]);
                    ch[1][PH + 3 - i] = ac_fma(ky, Dyz, ch[1][PH + 3 - i]);
                    ch[1][PH + 3 + i] = ac_fma(-ky, Dyz, ch[1][PH + 3 + i]);
                    ch[2][PH + 3 - i] += ez;
                    ch[2][PH + 3 + i] -= ez;
                    dxz += C.d1[0][i] * Dxz;
                    dyz += C.d1[1][i] * Dyz;
                    dxx += C.d1[0][i] * Dxx;
                    dyy += C.d1[1][i] * Dyy;
                }
                nv.u_dx[2] = dxz;
                nv.u_dy[2] = dyz;
                nv.u_dx[0] = dxx;
                nv.u_dy[1] = dyy;
            }

            // output plane: everything but the magnetic thread's force and cs^2
            T rhs[NQ] = {}, glr[3] = {};
            if (has_out) {
                const Pl& o = dly[PH];
                T dz[NQ], dzz[NQ], upz[NQ];
#pragma unroll
                for (int f = 0; f < NQ; ++f) {
                    T D[4], S[4];
#pragma unroll
                    for (int i = 1; i <= 3; ++i) {
                        D[i] = q[f][PH + 3 + i] - q[f][PH + 3 - i];
                        S[i] = pair_sum<CF>(q[f][PH + 3 + i], q[f][PH + 3 - i], q[f][PH + 3]);
                    }
                    dz[f] = C.d1[2][1] * D[1] + C.d1[2][2] * D[2] + C.d1[2][3] * D[3];
                    dzz[f] = sym3<CF>(C.d2[2], q[f][PH + 3], S);
                    upz[f] = UPWD ? sym3<CF>(C.up[2], q[f][PH + 3], S) : T(0);
                }
                const T uz = q[3][PH + 3];
                const T auz = ac_abs(uz);
                rhs[0] = (o.cont - uz * dz[0]) - dz[3];
                if (UPWD)
                    rhs[0] += auz * upz[0];
                const T third = T(1) / T(3);
                glr[0] = o.lr_dx;
                glr[1] = o.lr_dy;
                glr[2] = dz[0];
                const T divu = o.u_dx[0] + o.u_dy[1] + dz[3];
                // twice the traceless rate of strain (ref operators.h:145-161)
                const T d3 = third * divu;
                const T D00 = T(2) * (o.u_dx[0] - d3), D11 = T(2) * (o.u_dy[1] - d3),
                        D22 = T(2) * (dz[3] - d3);
                const T D01 = o.u_dy[0] + o.u_dx[1], D02 = dz[1] + o.u_dx[2], D12 = dz[2] + o.u_dy[2];
                const T Drow[3][3] = {{D00, D01, D02}, {D01, D11, D12}, {D02, D12, D22}};
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    T m = ch[i][PH] - dz[1 + i] * uz;
                    if (UPWD)
                        m += auz * upz[1 + i];
                    const T Dg = Drow[i][0] * glr[0] + Drow[i][1] * glr[1] + Drow[i][2] * glr[2];
                    m += P.nu * (dzz[1 + i] + Dg);
                    if (i == 2)
                        m += P.nu_third_zeta * dzz[3];
                    rhs[1 + i] = m;
                    xch[cur][X_U + i][tid] = q[1 + i][PH + 3];
                }
                if constexpr (ENTROPY) {
                    // 2 nu S:S + zeta (div u)^2 with D = 2 S
                    const T SS2 = T(0.5) * (D00 * D00 + D11 * D11 + D22 * D22) +
                                  (D01 * D01 + D02 * D02 + D12 * D12);
                    xch[cur][X_VISC][tid] = P.nu * SS2 + P.zeta * divu * divu;
                    xch[cur][X_LAPLR][tid] = o.lr_lap + dzz[0];
#pragma unroll
                    for (int i = 0; i < 3; ++i)
                        xch[cur][X_GLR + i][tid] = glr[i];
                }
            }

            // in-plane derivatives of plane p where it is itself output
            if (it >= R && it < zc + R) {
                const T ux = q[1][PH + 6], uy = q[2][PH + 6];
                const T aux = ac_abs(ux), auy = ac_abs(uy);
                T mom[3];
#pragma unroll
                for (int f = 0; f < NQ; ++f) {
                    const T c0 = q[f][PH + 6];
                    T Dx[4], Dy[4], Sx[4], Sy[4];
#pragma unroll
                    for (int i = 1; i <= 3; ++i) {
                        const T xp = at(f, i, 0), xm = at(f, -i, 0);
                        const T yp = at(f, 0, i), ym = at(f, 0, -i);
                        Dx[i] = xp - xm;
                        Dy[i] = yp - ym;
                        Sx[i] = pair_sum<CF>(xp, xm, c0);
                        Sy[i] = pair_sum<CF>(yp, ym, c0);
                    }
                    const T dxx = sym3<CF>(C.d2[0], c0, Sx), dyy = sym3<CF>(C.d2[1], c0, Sy);
                    T up = T(0);
                    if (UPWD)
                        up = aux * sym3<CF>(C.up[0], c0, Sx) + auy * sym3<CF>(C.up[1], c0, Sy);
                    if (f == 0 || f == 2) {
                        const T dx = C.d1[0][1] * Dx[1] + C.d1[0][2] * Dx[2] + C.d1[0][3] * Dx[3];
                        if (f == 0)
                            nv.lr_dx = dx;
                        else
                            nv.u_dx[1] = dx;
                    }
                    if (f == 0 || f == 1) {
                        const T dy = C.d1[1][1] * Dy[1] + C.d1[1][2] * Dy[2] + C.d1[1][3] * Dy[3];
                        if (f == 0)
                            nv.lr_dy = dy;
                        else
                            nv.u_dy[0] = dy;
                    }
                    if (f == 0) {
                        nv.lr_lap = dxx + dyy;
                        nv.cont = up;
                    }
                    else {
                        T m = P.nu * (dxx + dyy) + up;
                        if (f == 1) m += P.nu_third_zeta * dxx;
                        if (f == 2) m += P.nu_third_zeta * dyy;
                        mom[f - 1] = m;
                    }
                }
                nv.cont -= ux * nv.lr_dx + uy * nv.lr_dy + (nv.u_dx[0] + nv.u_dy[1]);
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    ch[i][PH + 3] += mom[i] - (nv.u_dx[i] * ux + nv.u_dy[i] * uy);
                T mxx = T(0), myy = T(0);  // d_xy u_x, d_xy u_y
#pragma unroll
                for (int i = 1; i <= 3; ++i) {
                    if constexpr (CF) {
                        mxx += A.mxv[0][i] * ((at(1, i, i) - at(1, i, -i)) - (at(1, -i, i) - at(1, -i, -i)));
                        myy += A.mxv[0][i] * ((at(2, i, i) - at(2, i, -i)) - (at(2, -i, i) - at(2, -i, -i)));
                    }
                    else {
                        mxx += A.mxv[0][i] * ((at(1, i, i) + at(1, -i, -i)) - (at(1, i, -i) + at(1, -i, i)));
                        myy += A.mxv[0][i] * ((at(2, i, i) + at(2, -i, -i)) - (at(2, i, -i) + at(2, -i, i)));
                    }
                }
                ch[0][PH + 3] += myy;
                ch[1][PH + 3] += mxx;
            }

            dly[PH] = nv;
            // plane p + 1 has landed (issued two steps ago; plane p + 2 may be in flight) and every
            // wave is done with this buffer
            step_barrier<4 * NR>(it + 2 < niter);

            if (has_out) {
                const T cs2 = ENTROPY ? xch[cur][ENTROPY ? X_CS2 : 0][tid] : P.cs2_sound;
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    rhs[1 + i] = (rhs[1 + i] - cs2 * glr[i]) - xch[cur][X_F + i][tid];
                if (inside) {
                    T fnew[NQ];
                    int craw[4];
#pragma unroll
                    for (int f = 0; f < NQ; ++f) {
                        const long long fo = f * fsb + pob;
                        fnew[f] = rk_update_pre<T, KB>(sbase((char*)K.w[0] + fo), sbase((char*)K.out[0] + fo), iob, STEP,
                                                       a.alpha, a.beta, q[f][PH + 3], rhs[f], dt, wpre[f],
                                                       comp_part_get<KB, 0>(crec, f), &craw[f]);
                    }
                    if (KB > 0)
                        comp_part_store<KB, 0>((char*)K.comp[0] + pob / (long long)sizeof(T) * (NF * KB / 8),
                                               iob / (unsigned)sizeof(T) * (unsigned)(NF * KB / 8),
                                               craw);
                    if (STEP == 2)
                        u2max = fmax(u2max, (double)fnew[1] * (double)fnew[1] +
                                                (double)fnew[2] * (double)fnew[2] +
                                                (double)fnew[3] * (double)fnew[3]);
                }
            }
            if (it + 1 >= 2 * R && it + 1 < niter)
                prefetch(it + 1, fsb, iob, K);
            if (it + 3 < niter)
                dma_plane(buf, p + 3, fsb, K);
        };
        // back to phase 0: the six newest entries move to the front, the rest start at zero
        auto rewind = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int f = 0; f < NQ; ++f)
#pragma unroll
                for (int i = 0; i < 6; ++i)
                    q[f][i] = q[f][i + 3];
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int i = 0; i < 9; ++i)
                    ch[c][i] = i < 6 ? ch[c][i + 3] : T(0);
        };
        for (int it = 0; it < niter; it += 3) {
            step(IntC<0>{}, lds0, it);
            if (it + 1 >= niter)
                break;
            step(IntC<1>{}, lds1, it + 1);
            if (it + 2 >= niter)
                break;
            step(IntC<2>{}, lds2, it + 2);
            rewind();
        }
        if (STEP == 2) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1)
                u2max = fmax(u2max, __shfl_xor(u2max, off, 64));
            if (lane == 0)
                wmax[wave] = u2max;
            if (a.time_acc != nullptr && blockIdx.x == 0 && tid == 0)
                *a.time_acc += (double)dt;
        }
    }
    else {
        // ================================================================ magnetic
        constexpr int NQ = ENTROPY ? 4 : 3;
        T q[NQ][9], ch[3][9];  // windows of 7: step PH of the loop uses entries PH .. PH + 6
        T lrq[6] = {};  // lnrho of the column, planes p - 3 .. p (a window of 4)
        struct Pl {
            T ax_dy, ay_dx, az_dx, az_dy, lap[3], s_dx, s_dy, s_lap;
        } dly[3] = {};  // of plane p - 3 + k: entry (PH + k) % 3
#pragma unroll
        for (int f = 0; f < NQ; ++f)
#pragma unroll
            for (int i = 0; i < 9; ++i)
                q[f][i] = T(0);
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int i = 0; i < 9; ++i)
                ch[c][i] = T(0);
        // w and the compensation of the next output cell, loaded a step ahead
        T wpre[NQ];
        T spre = T(0);
        CompPart<KB, 1> crec{};
#pragma unroll
        for (int f = 0; f < NQ; ++f)
            wpre[f] = T(0);
        auto prefetch = [&](int it, long long fsb, unsigned iob, const SolveArgs<T>& K) __attribute__((always_inline)) {
            const long long pob = K.sz * (long long)(z0 - R + it) * (long long)sizeof(T);
            if (STEP > 0) {
#pragma unroll
                for (int f = 0; f < NQ; ++f)
                    wpre[f] = ld_g<T>(sbase((char*)K.w[0] + ((4 + f) * fsb + pob)), iob);
            }
            if (!ENTROPY)
                spre = ld_g<T>(sbase((const char*)K.in[0] + (7 * fsb + pob)), iob);
            if (KB > 0)
                crec = comp_part_load<KB, 1>((char*)K.comp[0] + pob / (long long)sizeof(T) * (NF * KB / 8),
                                             iob / (unsigned)sizeof(T) * (unsigned)(NF * KB / 8));
        };
        auto step = [&](auto phase, T* buf, int it) __attribute__((always_inline)) {
            constexpr int PH = decltype(phase)::value;
            const bool has_out = it >= 2 * R;
            const SolveArgs<T>& K = *step_args<SolveArgs<T>>();
            const SolveArgs<T>& A = sizeof(T) == 8 ? K : a;
            const Coeffs<T>& C = A.C;
            const PhysParams<T>& P = A.P;
            const int p = z0 - R + it;
            const int cur = it & 1;
            const unsigned iob = opaque(ioff * (unsigned)sizeof(T));
            const long long fsb = opaque_s64(K.fstride * (long long)sizeof(T));
            const long long pob = K.sz * (long long)p * (long long)sizeof(T);  // array plane p - 3 + R
            const T* const L = buf + (4 * LPS + ctr);
            auto at = [&](int f, int dx, int dy) __attribute__((always_inline)) -> T {
                return L[f * LPS + dy * LX + dx];
            };
#pragma unroll
            for (int f = 0; f < NQ; ++f)
                q[f][PH + 6] = at(f, 0, 0);
            lrq[PH + 3] = buf[ctr];

            Pl nv = dly[PH];
            // z-chains of grad(div A)
            {
                T dxz = T(0), dyz = T(0);
#pragma unroll
                for (int i = 1; i <= 3; ++i) {
                    const T Dxz = at(2, i, 0) - at(2, -i, 0);
                    const T Dyz = at(2, 0, i) - at(2, 0, -i);
                    const T Dxx = at(0, i, 0) - at(0, -i, 0);
                    const T Dyy = at(1, 0, i) - at(1, 0, -i);
                    const T kx = C.mx[1][i], ky = C.mx[2][i];
                    const T ez = kx * Dxx + ky * Dyy;
                    ch[0][PH + 3 - i] = ac_fma(kx, Dxz, ch[0][PH + 3 - i]);
                    ch[0][PH + 3 + i] = ac_fma(-kx, Dxz, ch[0][PH + 3 + i]);
                    ch[1][PH + 3 - i] = ac_fma(ky, Dyz, ch[1][PH + 3 - i]);
                    ch[1][PH + 3 + i] = ac_fma(-ky, Dyz, ch[1][PH + 3 + i]);
                    ch[2][PH + 3 - i] += ez;
                    ch[2][PH + 3 + i] -= ez;
                    dxz += C.d1[0][i] * Dxz;
                    dyz += C.d1[1][i] * Dyz;
                }
                nv.az_dx = dxz;
                nv.az_dy = dyz;
            }

            // output plane: B, curl B, the force and cs^2 for the hydro thread. The chains hold
            // grad(div A) less the second derivative that the Laplacian of the same component
            // repeats.
            T B[3] = {}, lapA[3] = {}, gs[3] = {}, laps = T(0), heat_j = T(0), heat_u = T(0), kir = T(0);
            if (has_out) {
                const Pl& o = dly[PH];
                T dz[NQ], dzz[NQ];
#pragma unroll
                for (int f = 0; f < NQ; ++f) {
                    T D[4], S[4];
#pragma unroll
                    for (int i = 1; i <= 3; ++i) {
                        D[i] = q[f][PH + 3 + i] - q[f][PH + 3 - i];
                        S[i] = pair_sum<CF>(q[f][PH + 3 + i], q[f][PH + 3 - i], q[f][PH + 3]);
                    }
                    dz[f] = C.d1[2][1] * D[1] + C.d1[2][2] * D[2] + C.d1[2][3] * D[3];
                    dzz[f] = sym3<CF>(C.d2[2], q[f][PH + 3], S);
                }
                B[0] = o.az_dy - dz[1];
                B[1] = dz[0] - o.az_dx;
                B[2] = o.ay_dx - o.ax_dy;
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    lapA[i] = o.lap[i] + dzz[i];
                const T j0 = P.inv_mu0 * (ch[0][PH] - dzz[0]);
                const T j1 = P.inv_mu0 * (ch[1][PH] - dzz[1]);
                const T j2 = P.inv_mu0 * (ch[2][PH] - o.lap[2]);
                const T lr = lrq[PH];
                const T rho = ac_exp(lr);
                const T inv_rho = CF ? T(1) / rho : ac_rcp(rho);
                T f[3] = {inv_rho * (j2 * B[1] - j1 * B[2]), inv_rho * (j0 * B[2] - j2 * B[0]),
                          inv_rho * (j1 * B[0] - j0 * B[1])};
                if constexpr (ENTROPY) {
                    gs[0] = o.s_dx;
                    gs[1] = o.s_dy;
                    gs[2] = dz[3];
                    laps = o.s_lap + dzz[3];
                    const T lnT_rel = P.gamma_inv_cp * q[3][PH + 3] + P.gm1 * (lr - P.lnrho0);
                    const T cs2 = P.cs2_sound * ac_exp(lnT_rel);
                    const T cs2_cp = cs2 * P.inv_cp;
#pragma unroll
                    for (int i = 0; i < 3; ++i)
                        f[i] += cs2_cp * gs[i];
                    xch[cur][X_CS2][tid] = cs2;
                    T inv_pT;
                    if constexpr (sizeof(T) == 4 && !CF)
                        inv_pT = inv_rho * P.pT_scale * ac_rcp(cs2);
                    else
                        inv_pT = ac_exp(-(lr + lnT_rel + P.lnT0));
                    heat_j = inv_pT * (P.eta_mu0 * (j0 * j0 + j1 * j1 + j2 * j2));
                    heat_u = inv_pT * rho;
                    kir = P.K * inv_rho;
                }
#pragma unroll
                for (int i = 0; i < 3; ++i)
                    xch[cur][X_F + i][tid] = f[i];
            }

            if (it >= R && it < zc + R) {
#pragma unroll
                for (int f = 0; f < NQ; ++f) {
                    const T c0 = q[f][PH + 6];
                    T Dx[4], Dy[4], Sx[4], Sy[4];
#pragma unroll
                    for (int i = 1; i <= 3; ++i) {
                        const T xp = at(f, i, 0), xm = at(f, -i, 0);
                        const T yp = at(f, 0, i), ym = at(f, 0, -i);
                        Dx[i] = xp - xm;
                        Dy[i] = yp - ym;
                        Sx[i] = pair_sum<CF>(xp, xm, c0);
                        Sy[i] = pair_sum<CF>(yp, ym, c0);
                    }
                    const T dxx = sym3<CF>(C.d2[0], c0, Sx), dyy = sym3<CF>(C.d2[1], c0, Sy);
                    if (f == 1 || f == 3) {
                        const T dx = C.d1[0][1] * Dx[1] + C.d1[0][2] * Dx[2] + C.d1[0][3] * Dx[3];
                        if (f == 1)
                            nv.ay_dx = dx;
                        else
                            nv.s_dx = dx;
                    }
                    if (f == 0 || f == 3) {
                        const T dy = C.d1[1][1] * Dy[1] + C.d1[1][2] * Dy[2] + C.d1[1][3] * Dy[3];
                        if (f == 0)
                            nv.ax_dy = dy;
                        else
                            nv.s_dy = dy;
                    }
                    if (f < 3)
                        nv.lap[f] = dxx + dyy;
                    else
                        nv.s_lap = dxx + dyy;
                    if (f == 0) ch[0][PH + 3] -= dyy;
                    if (f == 1) ch[1][PH + 3] -= dxx;
                }
                T mxx = T(0), myy = T(0);
#pragma unroll
                for (int i = 1; i <= 3; ++i) {
                    if constexpr (CF) {
                        mxx += C.mx[0][i] * ((at(0, i, i) - at(0, i, -i)) - (at(0, -i, i) - at(0, -i, -i)));
                        myy += C.mx[0][i] * ((at(1, i, i) - at(1, i, -i)) - (at(1, -i, i) - at(1, -i, -i)));
                    }
                    else {
                        mxx += C.mx[0][i] * ((at(0, i, i) + at(0, -i, -i)) - (at(0, i, -i) + at(0, -i, i)));
                        myy += C.mx[0][i] * ((at(1, i, i) + at(1, -i, -i)) - (at(1, i, -i) + at(1, -i, i)));
                    }
                }
                ch[0][PH + 3] += myy;
                ch[1][PH + 3] += mxx;
            }

            dly[PH] = nv;
            // plane p + 1 has landed (issued two steps ago; plane p + 2 may be in flight) and every
            // wave is done with this buffer
            step_barrier<NQ * NR>(it + 2 < niter);

            if (has_out) {
                const T ux = xch[cur][X_U + 0][tid], uy = xch[cur][X_U + 1][tid],
                        uz = xch[cur][X_U + 2][tid];
                T rhs[4] = {(uy * B[2] - uz * B[1]) + P.eta * lapA[0],
                            (uz * B[0] - ux * B[2]) + P.eta * lapA[1],
                            (ux * B[1] - uy * B[0]) + P.eta * lapA[2], T(0)};
                if constexpr (ENTROPY) {
                    T st = P.gamma_inv_cp * laps + P.gm1 * xch[cur][X_LAPLR][tid];
#pragma unroll
                    for (int i = 0; i < 3; ++i) {
                        const T g = xch[cur][X_GLR + i][tid];
                        const T second = P.gamma_inv_cp * gs[i] + P.gm1 * g;
                        const T thirdv = P.gamma * (P.inv_cp * gs[i] + g) - g;
                        st += second * thirdv;
                    }
                    rhs[3] = -(ux * gs[0] + uy * gs[1] + uz * gs[2]) +
                             (heat_j + heat_u * xch[cur][X_VISC][tid]) + kir * st;
                }
                if (inside) {
                    int craw[4];
#pragma unroll
                    for (int f = 0; f < NQ; ++f) {
                        const long long fo = (4 + f) * fsb + pob;
                        rk_update_pre<T, KB>(sbase((char*)K.w[0] + fo), sbase((char*)K.out[0] + fo), iob, STEP, a.alpha,
                                             a.beta, q[f][PH + 3], rhs[f], dt, wpre[f],
                                             comp_part_get<KB, 1>(crec, f), &craw[f]);
                    }
                    if (!ENTROPY) {
                        st_b(sbase((char*)K.out[0] + (7 * fsb + pob)), iob, spre);
                        craw[3] = comp_part_get<KB, 1>(crec, 3);  // ss keeps its entry
                    }
                    if (KB > 0)
                        comp_part_store<KB, 1>((char*)K.comp[0] + pob / (long long)sizeof(T) * (NF * KB / 8),
                                               iob / (unsigned)sizeof(T) * (unsigned)(NF * KB / 8), craw);
                }
            }
            if (it + 1 >= 2 * R && it + 1 < niter)
                prefetch(it + 1, fsb, iob, K);
            if (it + 3 < niter)
                dma_plane(buf, p + 3, fsb, K);
        };
        // back to phase 0: the six newest entries move to the front, the rest start at zero
        auto rewind = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int f = 0; f < NQ; ++f)
#pragma unroll
                for (int i = 0; i < 6; ++i)
                    q[f][i] = q[f][i + 3];
#pragma unroll
            for (int c = 0; c < 3; ++c)
#pragma unroll
                for (int i = 0; i < 9; ++i)
                    ch[c][i] = i < 6 ? ch[c][i + 3] : T(0);
#pragma unroll
            for (int i = 0; i < 3; ++i)
                lrq[i] = lrq[i + 3];
        };
        for (int it = 0; it < niter; it += 3) {
            step(IntC<0>{}, lds0, it);
            if (it + 1 >= niter)
                break;
            step(IntC<1>{}, lds1, it + 1);
            if (it + 2 >= niter)
                break;
            step(IntC<2>{}, lds2, it + 2);
            rewind();
        }
    }
    if (STEP == 2) {
        // One atomic per workgroup, since they meet on one address: with one per wave a step took 32.1 against
        // 30.3 us at 32^3, 57.0 / 54.8 at 64^3, 234 / 230 at 128^3 (FP32).
        __syncthreads();
        if (a.umax2_next != nullptr && threadIdx.x == 0) {
            double m = wmax[0];
            for (int w = 1; w < NW; ++w)
                m = fmax(m, wmax[w]);
            atomic_max_nonneg(a.umax2_next, m);
        }
    }
}

// Launches the kernels of one column block (any grid; one instantiation per switch and substep).
template <typename T, int TX, int TY>
void launch_split_tile(const SolveArgs<T>& a, bool upwd, bool entropy, int kb, int zchunk,
                       hipStream_t st);

#ifdef AC_SPLIT_INSTANTIATE
template <typename T, int TX, int TY, bool U, bool E, int KB>
static void launch_split_kb(const SolveArgs<T>& a, int zchunk, hipStream_t st)
{
    const int ntx = (a.nx + TX - 1) / TX, nty = (a.ny + TY - 1) / TY;
    const int nch = (a.nz + zchunk - 1) / zchunk;
    const dim3 bpg((unsigned)(ntx * nty * nch)), tpb(2 * TX * TY);
    if (a.step == 0)
        hipLaunchKernelGGL((solve_split_kernel<T, U, E, KB, TX, TY, 0>), bpg, tpb, 0, st, a, zchunk, ntx, nty, nch);
    else if (a.step == 1)
        hipLaunchKernelGGL((solve_split_kernel<T, U, E, KB, TX, TY, 1>), bpg, tpb, 0, st, a, zchunk, ntx, nty, nch);
    else
        hipLaunchKernelGGL((solve_split_kernel<T, U, E, KB, TX, TY, 2>), bpg, tpb, 0, st, a, zchunk, ntx, nty, nch);
}

template <typename T, int TX, int TY>
void launch_split_tile(const SolveArgs<T>& a, bool upwd, bool entropy, int kb, int zc, hipStream_t st)
{
#define AC_SPLIT_KB(U, E)                                                                       \
    do {                                                                                        \
        if (kb == 0) launch_split_kb<T, TX, TY, U, E, 0>(a, zc, st);                            \
        else if (kb == 8) launch_split_kb<T, TX, TY, U, E, (sizeof(T) == 4 ? 8 : 0)>(a, zc, st);\
        else if (kb == 16) launch_split_kb<T, TX, TY, U, E, (sizeof(T) == 4 ? 16 : 0)>(a, zc, st); \
        else launch_split_kb<T, TX, TY, U, E, (sizeof(T) == 4 ? 32 : 0)>(a, zc, st);            \
    } while (0)
    if (upwd && entropy) AC_SPLIT_KB(true, true);
    else if (upwd) AC_SPLIT_KB(true, false);
    else if (entropy) AC_SPLIT_KB(false, true);
    else AC_SPLIT_KB(false, false);
#undef AC_SPLIT_KB
}
#endif

}  // namespace acamd
