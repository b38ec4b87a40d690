// block_stage.h -- staging of a 16 x 4 x 4 block of the state, with its radius-3 halo, in LDS: the eight
// fields' boxes of 22 x 10 x 10 cells by global -> LDS DMA (one dword per lane). Used by the kernels that
// take one cell per thread and read its whole stencil (69 loads per cell, mostly from L2, in place of
// about 230 from global memory).
#pragma once

#include "kernels.h"
#include "mhd_common.h"

namespace acamd {

constexpr int BX = 16, BY = 4, BZ = 4;
constexpr int BLX = BX + 2 * R, BLY = BY + 2 * R, BLZ = BZ + 2 * R;

template <typename T>
struct BlockStage {
    static constexpr int NW = BX * BY * BZ / 64;
    static constexpr int WPE = (int)sizeof(T) / 4;
    static constexpr int BOX = BLX * BLY * BLZ * WPE;              // dwords of a field's box
    static constexpr int NR = ((BOX + 63) / 64 + NW - 1) / NW;     // DMA rounds per wave
    static constexpr int LPS = NR * NW * 64 / WPE;                 // padded field stride in LDS (values)
};

inline long long block_count(int nx, int ny, int nz)
{
    return (long long)((nx + BX - 1) / BX) * ((ny + BY - 1) / BY) * ((nz + BZ - 1) / BZ);
}

// First cell of this workgroup's block. Workgroup b runs on XCD b % 8; each XCD takes a contiguous range
// of blocks, whose neighbours then share its L2.
__device__ __forceinline__ int3 block_origin(int nx, int ny)
{
    const int nb = (int)gridDim.x;
    const int bid = (nb & 7) == 0 ? ((int)blockIdx.x & 7) * (nb >> 3) + ((int)blockIdx.x >> 3) : (int)blockIdx.x;
    const int nbx = (nx + BX - 1) / BX, nby = (ny + BY - 1) / BY;
    return make_int3(bid % nbx * BX, bid / nbx % nby * BY, bid / (nbx * nby) * BZ);
}

// Issues the DMA of the block at o into lds (NF fields, BlockStage::LPS values apart); the caller waits
// for it. wrap: halo cells come from their periodic images in the interior (every extent >= R), else as
// stored. Cells past the array (blocks at the upper edges) are unused and read its last cell.
template <typename T>
__device__ __forceinline__ void stage_block(const SolveArgs<T>& a, int3 o, bool wrap, T* lds)
{
    using S = BlockStage<T>;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
#pragma unroll
    for (int r = 0; r < S::NR; ++r) {
        int d = (wave + r * S::NW) * 64 + lane;
        if (d >= S::BOX)
            d = 0;  // padding lanes re-read dword 0 of the box
        const int e = d / S::WPE, wd = d - e * S::WPE;
        int z = o.z + e / (BLX * BLY), y = o.y + e / BLX % BLY, x = o.x + e % BLX;
        if (wrap) {
            x += x < R ? a.nx : (x >= a.nx + R ? -a.nx : 0);
            y += y < R ? a.ny : (y >= a.ny + R ? -a.ny : 0);
            z += z < R ? a.nz : (z >= a.nz + R ? -a.nz : 0);
        }
        const long long src = min(x, a.mx - 1) + (long long)a.mx * min(y, a.my - 1) + a.sz * min(z, a.mz - 1);
#pragma unroll
        for (int q = 0; q < NF; ++q)
            __builtin_amdgcn_global_load_lds((const void*)((const char*)(a.in[q] + src) + 4 * wd),
                                             (lds_ptr_t)(lds + q * S::LPS + (wave + r * S::NW) * (64 / S::WPE)),
                                             4, 0, 0);
    }
}

// This wave's memory operations and LDS reads are done, then the workgroup barrier.
__device__ __forceinline__ void memory_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

}  // namespace acamd
