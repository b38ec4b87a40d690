// aux_kernels.hip -- periodic halo fill (one launch for all fields), FP64-accumulating
// reductions, one-pass diagnostics and small utility kernels.
//
// Periodic fill: ref acc-runtime/built-in/kernels.h:17-41 (BOUNDCOND_PERIODIC_DEVICE) launched
// per field over the whole m^3 volume by ref src/core/device.cc:1009-1017. Here one launch
// enumerates only the m^3 - n^3 halo cells of every field; the source is always an interior
// cell, so the fill has no read/write hazards.
// Reductions: ref src/core/kernels/reductions.cu:98-219 (map kernel into an n^3 scratchpad, then
// hipcub DeviceReduce). Here the map is fused into a single pass with FP64 accumulation and a
// deterministic two-stage tree (fixed grid, fixed order).
#include <algorithm>
#include <cstdio>
#include <cstdlib>

#include "kernels.h"

namespace acamd {

constexpr int RED_TPB = 256;
constexpr int RED_MAX_BLOCKS = 1024;

// ---------------------------------------------------------------- periodic fill
template <typename T>
struct FillArgs {
    T* f[NF];
    int nx, ny, nz, mx, my;
    unsigned halo_count;  // per field (< 2^32: checked at launch)
    int wide;             // every extent >= R: a halo cell's image is one period away
};

// One thread per halo cell and field. The cell enumeration (two z slabs of 3 full planes, then
// per interior plane 3 + 3 full rows and 3 + 3 cells at the ends of each interior row) is
// inverted with 32-bit divisions, and the image is the cell one period away (wrapped with a
// true modulo only on grids narrower than the halo), so the kernel is bound by its memory
// traffic rather than by 64-bit integer division.
template <typename T>
__global__ void __launch_bounds__(256) periodic_fill_kernel(FillArgs<T> a)
{
    const unsigned t0 = blockIdx.x * blockDim.x + threadIdx.x;
    if (t0 >= a.halo_count)
        return;
    T* __restrict__ f = a.f[blockIdx.y];
    const unsigned mx = (unsigned)a.mx, plane = mx * (unsigned)a.my;
    int i, j, k;
    unsigned t = t0;
    if (t < 6u * plane) {
        const unsigned kk = t / plane;
        const unsigned r = t - kk * plane;
        k = kk < 3u ? (int)kk : a.nz + (int)kk;  // planes 0..2, then nz + 3 .. nz + 5
        j = (int)(r / mx);
        i = (int)(r - (unsigned)j * mx);
    }
    else {
        t -= 6u * plane;
        const unsigned per = 6u * mx + 6u * (unsigned)a.ny;
        const unsigned kk = t / per;
        unsigned r = t - kk * per;
        k = R + (int)kk;
        if (r < 6u * mx) {
            const unsigned jj = r / mx;
            j = jj < 3u ? (int)jj : a.ny + (int)jj;  // rows 0..2, then ny + 3 .. ny + 5
            i = (int)(r - jj * mx);
        }
        else {
            r -= 6u * mx;
            const unsigned row = r / 6u;
            const int cc = (int)(r - row * 6u);
            j = R + (int)row;
            i = cc < 3 ? cc : a.nx + cc;
        }
    }
    int is, js, ks;
    if (a.wide) {
        is = i < R ? i + a.nx : (i >= a.nx + R ? i - a.nx : i);
        js = j < R ? j + a.ny : (j >= a.ny + R ? j - a.ny : j);
        ks = k < R ? k + a.nz : (k >= a.nz + R ? k - a.nz : k);
    }
    else {  // proper modulo: an extent smaller than the halo width wraps more than once
        is = ((i - R) % a.nx + a.nx) % a.nx + R;
        js = ((j - R) % a.ny + a.ny) % a.ny + R;
        ks = ((k - R) % a.nz + a.nz) % a.nz + R;
    }
    const long long pl = (long long)plane;
    const long long dst = (long long)i + (long long)a.mx * j + pl * k;
    const long long src = (long long)is + (long long)a.mx * js + pl * ks;
    f[dst] = f[src];
}

template <typename T>
void launch_periodic_fill(T* const* fields, int nfields, int nx, int ny, int nz, hipStream_t s)
{
    FillArgs<T> a;
    for (int q = 0; q < NF; ++q)
        a.f[q] = q < nfields ? fields[q] : nullptr;
    a.nx = nx;
    a.ny = ny;
    a.nz = nz;
    a.mx = nx + 2 * R;
    a.my = ny + 2 * R;
    const long long hc = 6LL * a.mx * a.my + (long long)nz * (6LL * a.mx + 6LL * ny);
    if (hc >= (1LL << 32) || 6LL * a.mx * a.my >= (1LL << 32)) {
        fprintf(stderr, "astaroth_amd: periodic fill: %lld halo cells per field exceed 2^32\n", hc);
        abort();
    }
    a.halo_count = (unsigned)hc;
    a.wide = nx >= R && ny >= R && nz >= R;
    const dim3 tpb(256, 1, 1);
    const dim3 bpg((unsigned)((a.halo_count + 255) / 256), (unsigned)nfields, 1);
    hipLaunchKernelGGL(periodic_fill_kernel<T>, bpg, tpb, 0, s, a);
}

// ---------------------------------------------------------------- reductions
__device__ __forceinline__ double red_init(int op)
{
    return op == 1 ? INFINITY : (op == 2 ? -INFINITY : 0.0);
}
__device__ __forceinline__ double red_combine(int op, double a, double b)
{
    return op == 1 ? fmin(a, b) : (op == 2 ? fmax(a, b) : a + b);
}

// The mapped value of one cell from the values of its arrays, and how many of them a map reads.
template <typename T>
__device__ __forceinline__ double red_map(int map, const T* v)
{
    switch (map) {
    case 1: return (double)v[0];
    case 2: { const double x = v[0]; return x * x; }
    case 3: { const double e = exp((double)v[0]); return e * e; }
    case 4: {
        const double x = v[0], y = v[1], z = v[2];
        return sqrt(x * x + y * y + z * z);
    }
    case 5: {
        const double x = v[0], y = v[1], z = v[2];
        return x * x + y * y + z * z;
    }
    case 6: {
        const double x = exp((double)v[0]), y = exp((double)v[1]),
                     z = exp((double)v[2]);
        return x * x + y * y + z * z;
    }
    case 7: {
        const double x = v[0], y = v[1], z = v[2];
        return sqrt(x * x + y * y + z * z) / sqrt(exp((double)v[3]));
    }
    case 8: {
        const double x = v[0], y = v[1], z = v[2];
        return (x * x + y * y + z * z) / exp((double)v[3]);
    }
    default: return 0.0;
    }
}
static int red_arrays(int map) { return map < 1 || map > 8 ? 0 : (map <= 3 ? 1 : (map <= 6 ? 3 : 4)); }

// The interior cells t, t + step, t + 2 step, ... (x fastest) as indices in an m^3 array. The two
// divisions of each number are taken once, and the steps add (di, dj, dk) with carries. I is 32-bit
// unsigned when the interior has fewer than 2^31 cells and the array fewer than 2^32 (every grid up
// to about 1600^3; use_index32 below), 64-bit otherwise; either visits the same cells in the same order.
template <typename I>
struct CellWalk {
    I i, j, k, di, dj, dk, nx, ny, mx, sz;
    __device__ __forceinline__ CellWalk(I t, I step, int nx_, int ny_, int mx_, int my_)
        : nx((I)nx_), ny((I)ny_), mx((I)mx_), sz((I)mx_ * (I)my_)
    {
        i = t % nx;
        j = t / nx % ny;
        k = t / nx / ny;
        di = step % nx;
        dj = step / nx % ny;
        dk = step / nx / ny;
    }
    __device__ __forceinline__ I cell() const { return (i + R) + mx * (j + R) + sz * (k + R); }
    __device__ __forceinline__ void advance()
    {
        i += di;
        j += dj;
        k += dk;
        if (i >= nx) {
            i -= nx;
            ++j;
        }
        if (j >= ny) {
            j -= ny;
            ++k;
        }
    }
};

static bool use_index32(int nx, int ny, int nz)
{
    const long long n = (long long)nx * ny * nz;
    const long long m = (long long)(nx + 2 * R) * (ny + 2 * R) * (nz + 2 * R);
    return n < (1ll << 31) && m < (1ll << 32);
}

// The halo cells inside a box [x0, x1) x [y0, y1) x [z0, z1) of the m^3 array (a sub-volume fill,
// ref src/core/device.cc:998-1017 with the BOUNDCOND_PERIODIC_DEVICE kernel of
// acc-runtime/built-in/kernels.h:17-41, which skips the interior): one thread per box cell and
// field; interior cells are left alone, halo cells take their periodic image.
template <typename T>
struct FillBoxArgs {
    T* f[NF];
    int nx, ny, nz, mx, my;
    int x0, y0, z0, bx, by;
    unsigned count;  // box cells per field
};

template <typename T>
__global__ void __launch_bounds__(256) periodic_fill_box_kernel(FillBoxArgs<T> a)
{
    const unsigned t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.count)
        return;
    const unsigned bx = (unsigned)a.bx, by = (unsigned)a.by;
    const unsigned r = t / bx;
    const int i = a.x0 + (int)(t - r * bx);
    const int j = a.y0 + (int)(r % by);
    const int k = a.z0 + (int)(r / by);
    const bool inside = i >= R && i < a.nx + R && j >= R && j < a.ny + R && k >= R && k < a.nz + R;
    if (inside)
        return;
    const int is = ((i - R) % a.nx + a.nx) % a.nx + R;
    const int js = ((j - R) % a.ny + a.ny) % a.ny + R;
    const int ks = ((k - R) % a.nz + a.nz) % a.nz + R;
    T* __restrict__ f = a.f[blockIdx.y];
    const long long pl = (long long)a.mx * a.my;
    f[(long long)i + (long long)a.mx * j + pl * k] = f[(long long)is + (long long)a.mx * js + pl * ks];
}

template <typename T>
void launch_periodic_fill_box(T* const* fields, int nfields, int nx, int ny, int nz, const int* lo,
                              const int* hi, hipStream_t s)
{
    FillBoxArgs<T> a;
    for (int q = 0; q < NF; ++q)
        a.f[q] = q < nfields ? fields[q] : nullptr;
    a.nx = nx;
    a.ny = ny;
    a.nz = nz;
    a.mx = nx + 2 * R;
    a.my = ny + 2 * R;
    a.x0 = lo[0];
    a.y0 = lo[1];
    a.z0 = lo[2];
    a.bx = hi[0] - lo[0];
    a.by = hi[1] - lo[1];
    const long long cnt = (long long)a.bx * a.by * (hi[2] - lo[2]);
    if (cnt <= 0)
        return;
    a.count = (unsigned)cnt;  // a box of an m^3 array the caller checked (< 2^32 cells)
    const dim3 tpb(256, 1, 1);
    const dim3 bpg((unsigned)((cnt + 255) / 256), (unsigned)nfields, 1);
    hipLaunchKernelGGL(periodic_fill_box_kernel<T>, bpg, tpb, 0, s, a);
}

template <typename T>
struct RedArgs {
    const T* bufs[4];
    int map, op;
    int nx, ny, nz, mx, my;
    double* partials;
};

__device__ __forceinline__ double block_reduce(int op, double v, double* sh)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        v = red_combine(op, v, __shfl_xor(v, off, 64));
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0)
        sh[wid] = v;
    __syncthreads();
    double r = red_init(op);
    if (threadIdx.x == 0) {
        const int nw = (blockDim.x + 63) >> 6;
        for (int q = 0; q < nw; ++q)
            r = red_combine(op, r, sh[q]);
    }
    return r;
}

// NA arrays are read. The values of eight (one array) or four cells are loaded before the first is
// used, so that enough loads are in flight to reach the memory's rate; they are combined in the
// order of the cells (256^3 FP32: one array 45 -> 24 us, three 52 -> 40, 5.0 TB/s).
template <typename T, typename I, int NA>
__global__ void __launch_bounds__(RED_TPB) reduce_stage1(RedArgs<T> a)
{
    __shared__ double sh[RED_TPB / 64];
    constexpr int U = NA == 1 ? 8 : 4;
    const I n = (I)a.nx * (I)a.ny * (I)a.nz, step = (I)gridDim.x * blockDim.x;
    I t = (I)blockIdx.x * blockDim.x + threadIdx.x;
    CellWalk<I> w(t, step, a.nx, a.ny, a.mx, a.my);
    double acc = red_init(a.op);
    while (t < n) {
        T v[U][NA > 0 ? NA : 1];
        int cnt = 0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (t < n) {
                const I c = w.cell();
#pragma unroll
                for (int q = 0; q < NA; ++q)
                    v[u][q] = a.bufs[q][c];
                ++cnt;
            }
            w.advance();
            t += step;
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (u < cnt)
                acc = red_combine(a.op, acc, red_map(a.map, v[u]));
    }
    const double r = block_reduce(a.op, acc, sh);
    if (threadIdx.x == 0)
        a.partials[blockIdx.x] = r;
}

__global__ void __launch_bounds__(RED_TPB) reduce_stage2(const double* partials, int np, int op,
                                                         double* out)
{
    __shared__ double sh[RED_TPB / 64];
    double acc = red_init(op);
    for (int t = threadIdx.x; t < np; t += blockDim.x)
        acc = red_combine(op, acc, partials[t]);
    const double r = block_reduce(op, acc, sh);
    if (threadIdx.x == 0)
        *out = r;
}

int reduce_num_partials(int nx, int ny, int nz)
{
    const long long n = (long long)nx * ny * nz;
    long long b = (n + RED_TPB - 1) / RED_TPB;
    if (b > RED_MAX_BLOCKS)
        b = RED_MAX_BLOCKS;
    if (b < 1)
        b = 1;
    return (int)b;
}

template <typename T>
void launch_reduce(const T* const* bufs, int map, int op, int nx, int ny, int nz, double* partials,
                   int max_partials, double* result_dev, hipStream_t s)
{
    RedArgs<T> a;
    for (int q = 0; q < 4; ++q)
        a.bufs[q] = bufs[q];
    a.map = map;
    a.op = op;
    a.nx = nx;
    a.ny = ny;
    a.nz = nz;
    a.mx = nx + 2 * R;
    a.my = ny + 2 * R;
    a.partials = partials;
    int nb = reduce_num_partials(nx, ny, nz);
    if (nb > max_partials)
        nb = max_partials;
#define AC_REDUCE(NA)                                                                               \
    do {                                                                                           \
        if (use_index32(nx, ny, nz))                                                               \
            hipLaunchKernelGGL((reduce_stage1<T, unsigned, NA>), dim3(nb), dim3(RED_TPB), 0, s, a); \
        else                                                                                       \
            hipLaunchKernelGGL((reduce_stage1<T, unsigned long long, NA>), dim3(nb), dim3(RED_TPB), 0, s, a); \
    } while (0)
    switch (red_arrays(map)) {
    case 1: AC_REDUCE(1); break;
    case 3: AC_REDUCE(3); break;
    case 4: AC_REDUCE(4); break;
    default: AC_REDUCE(0); break;
    }
#undef AC_REDUCE
    hipLaunchKernelGGL(reduce_stage2, dim3(1), dim3(RED_TPB), 0, s, (const double*)partials, nb,
                       op, result_dev);
}

// ---------------------------------------------------------------- marching along z with curl A
// Kernels that read curl A take 256 columns (numbered x fastest, so no lane is lost to ragged rows) and
// march them through zchunk planes. The z neighbours of A_x and A_y stay in registers, which leaves 26 of
// the 36 neighbour loads of a cell. Items (256 columns of one chunk) go to the XCDs in contiguous
// ranges, workgroup b running on XCD b % 8, so that a row read as a neighbour is in the L2 of the XCD
// that owns it. Diagnostics 256^3 FP32: 360 us a cell at a time with two divisions for its index and a
// barrier pair per accumulator at the end; 231 without those and with the ranges; 195 marching (the eight
// fields read once at 4 TB/s: 134). Reference maxima 128^3 FP32: 376, 32, 28 us.
struct MarchShape {
    int zchunk, blocks;
};
static MarchShape march_shape(int realsize, int nx, int ny, int nz)
{
    const long long cols = ((long long)nx * ny + RED_TPB - 1) / RED_TPB;
    // about 1024 items, of at least four planes (six more are loaded to start a chunk), or of fewer where that makes
    // less than 96 items: a small grid waits for the march of one item, not for its memory. Up to 128 items then, since
    // their atomics meet on one address (reference timestep's maxima FP64 with four planes / as here / up to 320 items:
    // 16^3 9.5 / 7.1 / 7.1 us, 24 x 20 x 18 10.1 / 7.2 / 7.3, 40^3 10.6 / 9.0 / 10.3, 7 x 5 x 300 13.5 / 9.9 / 12.4)
    long long nch = std::max(1ll, std::min(RED_MAX_BLOCKS / cols, (long long)(nz + 3) / 4));
    if (cols * nch < 96)
        nch = std::max(nch, std::min((long long)nz, 128 / cols));
    // Chunks of 64 planes and more are split further where the last round of workgroups leaves much of the chip idle (a
    // CU holds two in FP64, three in FP32): rounds times planes marched, six of them to start a chunk (diagnostics, one
    // or two chunks / split: 384^3 FP64 2675 / 1779 us, 320^3 1297 / 1065, 400 x 400 x 128 929 / 685; 384^3 FP32
    // 826 / 677). Multiples of 512 items lie evenly on the CUs (256^3 FP32, 1024 items: 207 us, split 216).
    const long long slots = realsize == 8 ? 512 : 768;
    const auto rounds = [&](long long c) {
        const long long planes = (nz + c - 1) / c;
        return (cols * ((nz + planes - 1) / planes) + slots - 1) / slots * (planes + 6);
    };
    long long split = nch;
    for (long long c = nch + 1; c <= 16 && nz / c >= 16; ++c)
        if (rounds(c) < rounds(split))
            split = c;
    if (nz / nch >= 64 && cols * nch % 512 != 0 && 10 * rounds(split) <= 9 * rounds(nch))
        nch = split;
    const int zc = (int)((nz + nch - 1) / nch);
    const long long items = cols * ((nz + zc - 1) / zc);
    return {zc, (int)std::min<long long>(items, RED_MAX_BLOCKS)};
}

// Calls f(c, g) for every interior cell c of this workgroup, g[q][ax] = d A_q / d x_ax for q != ax.
template <typename T, typename I, typename F>
__device__ __forceinline__ void march_curl(const T* const* A, const Coeffs<T>& C, int nx, int ny, int nz, int mx,
                                           int my, int zchunk, F&& f)
{
    const long long cols = ((long long)nx * ny + RED_TPB - 1) / RED_TPB;
    const long long items = cols * ((nz + zchunk - 1) / zchunk);
    long long first = blockIdx.x, last = items, step = gridDim.x;
    if (gridDim.x % 8 == 0) {
        const int xcd = blockIdx.x & 7;
        first = items * xcd / 8 + (blockIdx.x >> 3);
        last = items * (xcd + 1) / 8;
        step = gridDim.x >> 3;
    }
    const I sy = (I)mx, sz = (I)mx * (I)my;
    const T* __restrict__ ax = A[0];
    const T* __restrict__ ay = A[1];
    const T* __restrict__ az = A[2];
    auto d1 = [](const T* kk, T p1, T m1, T p2, T m2, T p3, T m3) {
        return kk[1] * (p1 - m1) + kk[2] * (p2 - m2) + kk[3] * (p3 - m3);
    };
    for (long long item = first; item < last; item += step) {
        const long long col = item % cols * RED_TPB + threadIdx.x;
        const int z0 = (int)(item / cols) * zchunk;
        if (col >= (long long)nx * ny)
            continue;
        const int z1 = min(z0 + zchunk, nz);
        I c = (I)((unsigned)col % (unsigned)nx + R) + sy * (I)((unsigned)col / (unsigned)nx + R) + sz * (I)(z0 + R);
        T qx[7], qy[7];
#pragma unroll
        for (int o = 0; o < 6; ++o) {
            qx[o] = ax[c + o * sz - 3 * sz];
            qy[o] = ay[c + o * sz - 3 * sz];
        }
        for (int k = z0; k < z1; ++k) {
            qx[6] = ax[c + 3 * sz];
            qy[6] = ay[c + 3 * sz];
            T g[3][3];
            auto along = [&](const T* p, I s, const T* kk) {
                return d1(kk, p[c + s], p[c - s], p[c + 2 * s], p[c - 2 * s], p[c + 3 * s], p[c - 3 * s]);
            };
            g[0][1] = along(ax, sy, C.d1[1]);
            g[1][0] = along(ay, 1, C.d1[0]);
            g[2][0] = along(az, 1, C.d1[0]);
            g[2][1] = along(az, sy, C.d1[1]);
            g[0][2] = d1(C.d1[2], qx[4], qx[2], qx[5], qx[1], qx[6], qx[0]);
            g[1][2] = d1(C.d1[2], qy[4], qy[2], qy[5], qy[1], qy[6], qy[0]);
            f(c, g);
#pragma unroll
            for (int o = 0; o < 6; ++o) {
                qx[o] = qx[o + 1];
                qy[o] = qy[o + 1];
            }
            c += sz;
        }
    }
}

// ---------------------------------------------------------------- diagnostics

template <typename T>
struct DiagArgs {
    const T* f[NF];
    Coeffs<T> C;
    int nx, ny, nz, mx, my, zchunk;
    double* partials;  // DIAG_SLOTS * gridDim.x
};

__device__ __forceinline__ int diag_op(int slot)
{
    // [min x8][max x8][sum sq x8] then, for |u|^2, |B|^2 and vA^2 = |B|^2 / rho: [sum][max][min]
    if (slot < NF)
        return 1;
    if (slot < 2 * NF)
        return 2;
    if (slot < 3 * NF)
        return 3;
    const int r = (slot - 3 * NF) % 3;
    return r == 0 ? 3 : (r == 1 ? 2 : 1);
}

// Minima and maxima of the fields are kept in T, which holds them exactly. The 33 accumulators are
// reduced per wave and exchanged through LDS once.
template <typename T, typename I>
__global__ void __launch_bounds__(RED_TPB) diagnostics_stage1(DiagArgs<T> a)
{
    __shared__ double sh[DIAG_SLOTS][RED_TPB / 64];
    T lo[NF], hi[NF];
    double sq[NF], acc[DIAG_SLOTS - 3 * NF];
#pragma unroll
    for (int q = 0; q < NF; ++q) {
        lo[q] = (T)INFINITY;
        hi[q] = (T)-INFINITY;
        sq[q] = 0.0;
    }
#pragma unroll
    for (int q = 3 * NF; q < DIAG_SLOTS; ++q)
        acc[q - 3 * NF] = red_init(diag_op(q));
    march_curl<T, I>(a.f + 4, a.C, a.nx, a.ny, a.nz, a.mx, a.my, a.zchunk, [&](I c, const T g[3][3]) {
        T v[NF];
#pragma unroll
        for (int q = 0; q < NF; ++q) {
            v[q] = a.f[q][c];
            lo[q] = fmin(lo[q], v[q]);
            hi[q] = fmax(hi[q], v[q]);
            sq[q] += (double)v[q] * (double)v[q];
        }
        const double ux = v[1], uy = v[2], uz = v[3];
        const double u2 = ux * ux + uy * uy + uz * uz;
        acc[0] += u2;
        acc[1] = fmax(acc[1], u2);
        acc[2] = fmin(acc[2], u2);
        const double bx = (double)g[2][1] - (double)g[1][2], by = (double)g[0][2] - (double)g[2][0],
                     bz = (double)g[1][0] - (double)g[0][1];
        const double b2 = bx * bx + by * by + bz * bz;
        acc[3] += b2;
        acc[4] = fmax(acc[4], b2);
        acc[5] = fmin(acc[5], b2);
        // Alfven speed |B| / sqrt(rho), rho = exp(lnrho) (ref acc-runtime/stdlib/map.h:121-134)
        const double va2 = b2 / exp((double)v[0]);
        acc[6] += va2;
        acc[7] = fmax(acc[7], va2);
        acc[8] = fmin(acc[8], va2);
    });
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < DIAG_SLOTS; ++q) {
        double r;
        if (q < 2 * NF) {
            T m = q < NF ? lo[q % NF] : hi[q % NF];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1)
                m = q < NF ? fmin(m, __shfl_xor(m, off, 64)) : fmax(m, __shfl_xor(m, off, 64));
            r = m;
        }
        else {
            r = q < 3 * NF ? sq[q % NF] : acc[q < 3 * NF ? 0 : q - 3 * NF];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1)
                r = red_combine(diag_op(q), r, __shfl_xor(r, off, 64));
        }
        if (lane == 0)
            sh[q][wid] = r;
    }
    __syncthreads();
    const int q = threadIdx.x;
    if (q < DIAG_SLOTS) {
        double r = red_init(diag_op(q));
        for (int k = 0; k < RED_TPB / 64; ++k)
            r = red_combine(diag_op(q), r, sh[q][k]);
        a.partials[(long long)q * gridDim.x + blockIdx.x] = r;
    }
}

// One workgroup per slot (one for all slots in turn took 79 us at 256^3, this 4).
__global__ void __launch_bounds__(RED_TPB) diagnostics_stage2(const double* partials, int np, double* out)
{
    __shared__ double sh[RED_TPB / 64];
    const int q = blockIdx.x, op = diag_op(q);
    double acc = red_init(op);
    for (int t = threadIdx.x; t < np; t += blockDim.x)
        acc = red_combine(op, acc, partials[(long long)q * np + t]);
    const double r = block_reduce(op, acc, sh);
    if (threadIdx.x == 0)
        out[q] = r;
}

template <typename T>
void launch_diagnostics(const T* const* fields, const Coeffs<T>& C, int nx, int ny, int nz,
                        double* partials, int max_partials, double* out_dev, hipStream_t s)
{
    DiagArgs<T> a;
    for (int q = 0; q < NF; ++q)
        a.f[q] = fields[q];
    a.C = C;
    a.nx = nx;
    a.ny = ny;
    a.nz = nz;
    a.mx = nx + 2 * R;
    a.my = ny + 2 * R;
    a.partials = partials;
    const MarchShape shape = march_shape((int)sizeof(T), nx, ny, nz);
    a.zchunk = shape.zchunk;
    const int nb = std::min(shape.blocks, max_partials / DIAG_SLOTS);
    if (use_index32(nx, ny, nz))
        hipLaunchKernelGGL((diagnostics_stage1<T, unsigned>), dim3(nb), dim3(RED_TPB), 0, s, a);
    else
        hipLaunchKernelGGL((diagnostics_stage1<T, unsigned long long>), dim3(nb), dim3(RED_TPB), 0,
                           s, a);
    hipLaunchKernelGGL(diagnostics_stage2, dim3(DIAG_SLOTS), dim3(RED_TPB), 0, s, (const double*)partials,
                       nb, out_dev);
}

// ---------------------------------------------------------------- max |u|^2
// Block-level max of a non-negative double, one atomic per workgroup at most (two per wave were most of
// the 376 us that the reference timestep's maxima took at 128^3). NaNs are passed over where there are numbers.
__device__ __forceinline__ void block_max_to_global(double v, unsigned long long* dst)
{
    __shared__ double sh[RED_TPB / 64];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
        v = fmax(v, __shfl_xor(v, off, 64));
    __syncthreads();
    if ((threadIdx.x & 63) == 0)
        sh[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < RED_TPB / 64; ++w)
            v = fmax(v, sh[w]);
        atomic_max_nonneg(dst, v);
    }
}

template <typename T>
struct UmaxArgs {
    const T* u[3];
    int nx, ny, nz, mx, my;
    unsigned long long* umax2;
};

template <typename T, typename I>
__global__ void __launch_bounds__(RED_TPB) umax2_kernel(UmaxArgs<T> a)
{
    const I n = (I)a.nx * (I)a.ny * (I)a.nz, step = (I)gridDim.x * blockDim.x;
    I t = (I)blockIdx.x * blockDim.x + threadIdx.x;
    double m = 0.0;
    for (CellWalk<I> w(t, step, a.nx, a.ny, a.mx, a.my); t < n; t += step, w.advance()) {
        const I c = w.cell();
        const double x = a.u[0][c], y = a.u[1][c], z = a.u[2][c];
        m = fmax(m, x * x + y * y + z * z);
    }
    block_max_to_global(m, a.umax2);
}

template <typename T>
void launch_umax2(const T* const* uu, int nx, int ny, int nz, unsigned long long* umax2,
                  hipStream_t s)
{
    UmaxArgs<T> a;
    for (int q = 0; q < 3; ++q)
        a.u[q] = uu[q];
    a.nx = nx;
    a.ny = ny;
    a.nz = nz;
    a.mx = nx + 2 * R;
    a.my = ny + 2 * R;
    a.umax2 = umax2;
    const int nb = reduce_num_partials(nx, ny, nz);
    if (use_index32(nx, ny, nz))
        hipLaunchKernelGGL((umax2_kernel<T, unsigned>), dim3(nb), dim3(RED_TPB), 0, s, a);
    else
        hipLaunchKernelGGL((umax2_kernel<T, unsigned long long>), dim3(nb), dim3(RED_TPB), 0, s, a);
}

// ---------------------------------------------------------------- reference timestep inputs
// The (x, y) pair of cfl_cell for the current state (modes 1 and 2): |u|^2 and the Alfven speed
// squared |curl A|^2 / exp(lnrho), or (|u| + sqrt(cs^2 + vA^2))^2; maxima over interior cells.
template <typename T>
struct CflArgs {
    const T* f[NF];
    Coeffs<T> C;
    int nx, ny, nz, mx, my, zchunk;
    int mode;
    double cs2;
    unsigned long long* out;  // pair
};

template <typename T, typename I>
__global__ void __launch_bounds__(RED_TPB) cfl_state_kernel(CflArgs<T> a)
{
    double mx_ = 0.0, my_ = 0.0;
    march_curl<T, I>(a.f + 4, a.C, a.nx, a.ny, a.nz, a.mx, a.my, a.zchunk, [&](I c, const T g[3][3]) {
        CellDerivs<T> d;
        d.lr = a.f[0][c];
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            d.u[q] = a.f[1 + q][c];
#pragma unroll
            for (int ax = 0; ax < 3; ++ax)
                d.ga[q][ax] = ax == q ? T(0) : g[q][ax];
        }
        double x, y;
        cfl_cell<T>(a.mode, a.cs2, d, x, y);
        mx_ = fmax(mx_, x);
        my_ = fmax(my_, y);
    });
    block_max_to_global(mx_, a.out);
    if (a.mode == 1)
        block_max_to_global(my_, a.out + 1);
}

template <typename T>
void launch_cfl_state(const T* const* fields, const Coeffs<T>& C, int nx, int ny, int nz, int mode,
                      double cs2, unsigned long long* out, hipStream_t s)
{
    CflArgs<T> a;
    for (int q = 0; q < NF; ++q)
        a.f[q] = fields[q];
    a.C = C;
    a.nx = nx;
    a.ny = ny;
    a.nz = nz;
    a.mx = nx + 2 * R;
    a.my = ny + 2 * R;
    a.mode = mode;
    a.cs2 = cs2;
    a.out = out;
    const MarchShape shape = march_shape((int)sizeof(T), nx, ny, nz);
    a.zchunk = shape.zchunk;
    const int nb = shape.blocks;
    if (use_index32(nx, ny, nz))
        hipLaunchKernelGGL((cfl_state_kernel<T, unsigned>), dim3(nb), dim3(RED_TPB), 0, s, a);
    else
        hipLaunchKernelGGL((cfl_state_kernel<T, unsigned long long>), dim3(nb), dim3(RED_TPB), 0, s,
                           a);
}

template void launch_cfl_state<AcRealT>(const AcRealT* const*, const Coeffs<AcRealT>&, int, int, int,
                                         int, double, unsigned long long*, hipStream_t);

// ---------------------------------------------------------------- compensation records
template <typename E>
__global__ void zero_comp_field_kernel(E* first, size_t count)
{
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < count;
         t += (size_t)gridDim.x * blockDim.x)
        first[t * NF] = E(0);
}

void launch_zero_comp_field(void* slab, size_t count, int kahan_bits, int q, hipStream_t s)
{
    size_t nb = (count + 255) / 256;
    if (nb > 65536)
        nb = 65536;
    char* first = (char*)slab + (size_t)q * (kahan_bits / 8);
    if (kahan_bits == 8)
        hipLaunchKernelGGL(zero_comp_field_kernel<int8_t>, dim3((unsigned)nb), dim3(256), 0, s,
                           (int8_t*)first, count);
    else if (kahan_bits == 16)
        hipLaunchKernelGGL(zero_comp_field_kernel<int16_t>, dim3((unsigned)nb), dim3(256), 0, s,
                           (int16_t*)first, count);
    else if (kahan_bits == 32)
        hipLaunchKernelGGL(zero_comp_field_kernel<float>, dim3((unsigned)nb), dim3(256), 0, s,
                           (float*)first, count);
}

// ---------------------------------------------------------------- helical forcing
// ref mhdsolver.ac:286-331 (helical_forcing, forcing) and :614-631 (added to u after the final
// update of substep 2). The geometry and the mode are evaluated in FP64, the force is rounded to
// AcReal and added to the stored u in AcReal, as the reference adds forcing_step to rk3_final.
// A workgroup marches its 64 x 4 columns through zchunk planes, so the phase and the x and y parts of
// k . y, with their FP64 divisions and sines, are taken once per column, and max |u|^2 makes one atomic
// per workgroup (128^3 FP32: 23 -> 18 us; u alone, read and written, is 50 MB).
template <typename T>
__global__ void __launch_bounds__(RED_TPB) forcing_kernel(ForcingArgs<T> a, int zchunk)
{
    const int i = (int)(threadIdx.x & 63) + blockIdx.x * 64;
    const int j = (int)(threadIdx.x >> 6) + blockIdx.y * (RED_TPB / 64);
    const int k0 = blockIdx.z * zchunk;
    const int k1 = i < a.nx && j < a.ny ? min(k0 + zchunk, a.nz) : k0;
    const double dt = (double)solve_dt(a.s);
    const double t0 = a.time_acc ? a.t_base + (*a.time_acc - dt) : a.t_base;
    const bool on = t0 > a.switch_time;
    double u2 = __builtin_nan("");  // no cell yet: an all-NaN velocity gives a NaN timestep
    // y = 2 pi xx / (ds ngrid), xx = (global index - nmin) ds
    auto part = [&](int d, int g, int ng) {
        return a.k[d] * (2.0 * M_PI * (((double)g * a.ds[d]) / (a.ds[d] * (double)ng)));
    };
    const double kxy = (0.0 + part(0, a.gx0 + i, a.ngx)) + part(1, a.gy0 + j, a.ngy);
    double sp, cp;
    sincos(a.phase, &sp, &cp);
    const double amp = sqrt(dt) * a.nn;
    for (int k = k0; k < k1; ++k) {
        const long long c = (long long)(i + R) + (long long)a.mx * (j + R) + a.sz * (k + R);
        T u[3] = {a.uu[0][c], a.uu[1][c], a.uu[2][c]};
        if (on) {
            double sk, ck;
            sincos(kxy + part(2, a.gz0 + k, a.ngz), &sk, &ck);
            const double re = ck * cp - sk * sp;
            const double im = ck * sp + sk * cp;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                u[d] = u[d] + (T)(amp * (a.fre[d] * re - a.fim[d] * im));
                a.uu[d][c] = u[d];
            }
        }
        u2 = fmax(u2, (double)u[0] * (double)u[0] + (double)u[1] * (double)u[1] + (double)u[2] * (double)u[2]);
    }
    if (a.umax2_next != nullptr)
        block_max_to_global(u2, a.umax2_next);
}

template <typename T>
void launch_forcing(const ForcingArgs<T>& a, hipStream_t s)
{
    // planes per workgroup: up to 8 where that leaves four workgroups for each CU
    const long long columns = (long long)((a.nx + 63) / 64) * ((a.ny + 3) / 4);
    const int zc = (int)std::max(1ll, std::min(8ll, columns * a.nz / 1024));
    const dim3 bpg((unsigned)((a.nx + 63) / 64), (unsigned)((a.ny + 3) / 4), (unsigned)((a.nz + zc - 1) / zc));
    hipLaunchKernelGGL((forcing_kernel<T>), bpg, dim3(RED_TPB), 0, s, a, zc);
}

template void launch_forcing<AcRealT>(const ForcingArgs<AcRealT>&, hipStream_t);

// ---------------------------------------------------------------- fills
template <typename T>
__global__ void fill_kernel(T* dst, size_t n, T v)
{
    for (size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x; t < n;
         t += (size_t)gridDim.x * blockDim.x)
        dst[t] = v;
}

template <typename T>
void launch_fill(T* dst, size_t n, T v, hipStream_t s)
{
    if (n == 0)
        return;
    size_t nb = (n + 255) / 256;
    if (nb > 65536)
        nb = 65536;
    hipLaunchKernelGGL(fill_kernel<T>, dim3((unsigned)nb), dim3(256), 0, s, dst, n, v);
}

void launch_zero_bytes(void* dst, size_t nbytes, hipStream_t s)
{
    // Word fill for the aligned body, byte fill for a tail (slabs are 256-byte aligned).
    const size_t words = nbytes / 4;
    launch_fill<unsigned>((unsigned*)dst, words, 0u, s);
    const size_t tail = nbytes - words * 4;
    if (tail)
        launch_fill<unsigned char>((unsigned char*)dst + words * 4, tail, (unsigned char)0, s);
}

template void launch_periodic_fill<AcRealT>(AcRealT* const*, int, int, int, int, hipStream_t);
template void launch_periodic_fill_box<AcRealT>(AcRealT* const*, int, int, int, int, const int*,
                                                  const int*, hipStream_t);
template void launch_reduce<AcRealT>(const AcRealT* const*, int, int, int, int, int, double*, int,
                                     double*, hipStream_t);
template void launch_diagnostics<AcRealT>(const AcRealT* const*, const Coeffs<AcRealT>&, int, int,
                                          int, double*, int, double*, hipStream_t);
template void launch_umax2<AcRealT>(const AcRealT* const*, int, int, int, unsigned long long*,
                                    hipStream_t);
template void launch_fill<AcRealT>(AcRealT*, size_t, AcRealT, hipStream_t);

}  // namespace acamd
