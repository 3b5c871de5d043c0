// Launch plumbing shared by the GEMM variant tables.
#pragma once
#include "gemm_kernels.hpp"

namespace icl {

// Tiles of C that a launch covers.
inline long gemm_tiles(const GemmArgs* g, int bm, int bn)
{
    return g->write_tri != ICL_TRI_NONE ? tri_tile_count(g->M, g->N, g->write_tri, bm, bn)
                                        : (long)((g->M + bm - 1) / bm) * ((g->N + bn - 1) / bn);
}

// Launches `kern(arg)` over `blocks` workgroups of NT threads. Kernels that need more
// than 64 KiB of LDS get the dynamic-LDS limit raised once per instantiation.
template <int NT, size_t LDS, typename Kern, typename Arg>
inline hipError_t launch_blocks(Kern kern, long blocks, hipStream_t s, const Arg& arg)
{
    if constexpr (LDS > 65536) {
        static const hipError_t attr =
            hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                static_cast<int>(LDS));
        if (attr != hipSuccess) return attr;
    }
    if (blocks <= 0) return hipSuccess;
    if (blocks > 0x7fffffffL) return hipErrorInvalidValue;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(NT), LDS, s, arg);
    return hipGetLastError();
}

// Launches `kern(arg)` over the tiles of C.
template <int BM, int BN, int NT, size_t LDS, typename Kern, typename Arg>
inline hipError_t launch_gemm(Kern kern, const GemmArgs* g, hipStream_t s, const Arg& arg)
{
    return launch_blocks<NT, LDS>(kern, gemm_tiles(g, BM, BN), s, arg);
}

template <int BM, int BN, int NT, size_t LDS, typename Kern>
inline hipError_t launch_gemm(Kern kern, const GemmArgs* g, hipStream_t s)
{
    return launch_gemm<BM, BN, NT, LDS>(kern, g, s, *g);
}

} // namespace icl
