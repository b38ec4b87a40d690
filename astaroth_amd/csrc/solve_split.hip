// solve_split.hip -- shapes, selection and dispatch of the role-split solve kernel (solve_split.h); the
// kernels of each column block are compiled in solve_split_a.hip, _b.hip and _c.hip.
#include <algorithm>

#include "solve_split.h"

namespace acamd {

// Column blocks (tx, ty) and how many of their workgroups share a CU, which their plane buffers and
// exchange in LDS bound (98 KB for the 256 columns of 64 x 4 in FP32 and the 128 columns in FP64, 49 KB
// for 128 columns in FP32). Rows of 32 leave every memory line they write shared with the next block, so
// 64 x 4 is the better one wherever it has long enough chunks (256^3 FP32: 0.593 against 0.76 ms a
// launch); small and narrow grids fill the CUs only with the 128-column blocks (64^3 FP32: 15.6 against
// 17.9 us), and 16 x 8 wastes the fewest columns (100 x 90 x 75 FP64: 0.077 ms against 0.092 with 32 x 4).
struct SplitTile {
    int tx, ty, per_cu;
};
static const SplitTile kSplitTiles[] = {
#if AC_DOUBLE_PRECISION
    {32, 4, 1}, {16, 8, 1},
#else
    {64, 4, 1}, {32, 4, 2}, {16, 8, 2},
#endif
};
constexpr int kCUs = 256;

static long long split_tiles(int tx, int ty, int nx, int ny)
{
    return (long long)((nx + tx - 1) / tx) * ((ny + ty - 1) / ty);
}

bool split_shape_fits(TiledShape s, int nx, int ny, int nz)
{
    bool known = false;
    for (const SplitTile& k : kSplitTiles)
        known = known || (k.tx == s.tx && k.ty == s.ty);
    if (s.kind != 2 || !known || s.zchunk <= 0 || s.zchunk > nz)
        return false;
    // 32-bit block numbers, and 32-bit in-plane byte offsets of values and compensation records
    return split_tiles(s.tx, s.ty, nx, ny) * ((nz + s.zchunk - 1) / s.zchunk) < (1ll << 31) &&
           (long long)(nx + 2 * R) * (ny + 2 * R) * (NF * 4) < (1ll << 32);
}

// One z-chunk per column block. Its cost is rounds of workgroups over the CUs times plane steps per chunk
// (six of them start a chunk up); where two workgroups share a CU, a round that has only one on each
// takes 0.8 of the time of a full one (128 columns FP32: 1.45 against 1.8 us per plane step, measured
// at 32^3 to 128^3). Half or twice the planes of the cheapest split cost 2-50% (128^3 FP32, 64 x 4:
// 0.079 ms with 32 planes, 0.096 with 16, 0.14 with 64). Among splits within 7% of the cheapest
// the shortest chunk of 64 planes or more is taken: more and shorter rounds keep neighbouring blocks
// close and even out when other streams share the chip (a step, launches of three streams / of one: 512^3
// FP32 16-bit 17.0 / 17.0 ms with 86 planes, 20.4 / 17.0 with 171, 17.7 / 17.6 with 32; 256^3 FP64 4.47 / 4.25
// with 64, 4.75 / 4.17 with 128, 4.98 / 4.21 with 256).
// Blocks that cover 30% more columns than the best one are left out. So are narrower blocks where a wider
// one covers as few columns and has at least 16 planes to a chunk: at 128^3 FP32 32 x 4 is faster
// alone than 64 x 4 (0.0705 against 0.079 ms), but it loses that where streams share the chip (0.088
// against 0.085 ms), and from 192^3 on it loses both ways; at 256^3 FP64 16 x 8 and 32 x 4 come out even
// alone, and 16 x 8 takes 5.1 against 4.98 ms a step with three streams.
int split_candidates(int nx, int ny, int nz, TiledShape* out, int max_out)
{
    long long least = 1ll << 62;
    for (const SplitTile& k : kSplitTiles)
        least = std::min(least, split_tiles(k.tx, k.ty, nx, ny) * k.tx * k.ty);
    int n = 0;
    for (const SplitTile& k : kSplitTiles) {
        const long long tiles = split_tiles(k.tx, k.ty, nx, ny), slots = (long long)kCUs * k.per_cu;
        if (100 * tiles * k.tx * k.ty > 130 * least || n >= max_out)
            continue;
        const auto cost = [&](int zc) {
            const long long blocks = tiles * ((nz + zc - 1) / zc), rest = blocks % slots;
            const double last = rest == 0 ? 0.0 : (rest <= kCUs && k.per_cu > 1 ? 0.8 : 1.0);
            return ((double)(blocks / slots) + last) * (zc + 2 * R);
        };
        TiledShape s{k.tx, k.ty, nz, 2};
        for (int nch = 1; nch <= nz; ++nch)
            if (cost((nz + nch - 1) / nch) < cost(s.zchunk))
                s.zchunk = (nz + nch - 1) / nch;
        const double least_cost = cost(s.zchunk);
        for (int nch = 1; (nz + nch - 1) / nch >= 64; ++nch)
            if (cost((nz + nch - 1) / nch) <= 1.07 * least_cost)
                s.zchunk = std::min(s.zchunk, (nz + nch - 1) / nch);
        if (split_shape_fits(s, nx, ny, nz))
            out[n++] = s;
        if (n > 0 && tiles * k.tx * k.ty == least && s.zchunk >= 16)
            break;
    }
    return n;
}

// The kernel addresses field f of every role as slab + f * fstride.
template <typename T>
static bool uniform_slabs(const SolveArgs<T>& a, int kb)
{
    for (int q = 0; q < NF; ++q) {
        const long long o = q * a.fstride;
        if (a.in[q] != a.in[0] + o || a.out[q] != a.out[0] + o || a.w[q] != a.w[0] + o)
            return false;
        if (kb > 0 && (const char*)a.comp[q] != (const char*)a.comp[0] + q * (kb / 8))
            return false;
    }
    return true;
}

template <typename T>
bool split_reads_periodic(const SolveArgs<T>& a, int kb, TiledShape s)
{
    return split_shape_fits(s, a.nx, a.ny, a.nz) && uniform_slabs(a, kb) && a.nx >= R &&
           a.ny >= R && a.nz >= R;
}

template <typename T>
bool launch_solve_split(const SolveArgs<T>& a, bool upwd, bool entropy, int kb, TiledShape s,
                        hipStream_t st)
{
    if (!split_shape_fits(s, a.nx, a.ny, a.nz) || !uniform_slabs(a, kb) ||
        (a.wrap && !split_reads_periodic(a, kb, s)))
        return false;
#if AC_DOUBLE_PRECISION
    if (s.tx == 32)
        launch_split_tile<T, 32, 4>(a, upwd, entropy, kb, s.zchunk, st);
    else
        launch_split_tile<T, 16, 8>(a, upwd, entropy, kb, s.zchunk, st);
#else
    if (s.tx == 64)
        launch_split_tile<T, 64, 4>(a, upwd, entropy, kb, s.zchunk, st);
    else if (s.tx == 32)
        launch_split_tile<T, 32, 4>(a, upwd, entropy, kb, s.zchunk, st);
    else
        launch_split_tile<T, 16, 8>(a, upwd, entropy, kb, s.zchunk, st);
#endif
    return true;
}

template bool launch_solve_split<AcRealT>(const SolveArgs<AcRealT>&, bool, bool, int, TiledShape, hipStream_t);
template bool split_reads_periodic<AcRealT>(const SolveArgs<AcRealT>&, int, TiledShape);

}  // namespace acamd
