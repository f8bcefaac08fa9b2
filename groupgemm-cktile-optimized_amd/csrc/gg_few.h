// Few-row kernels: forward and dgrad (gg_few.hip) and wgrad (gg_wfew.hip) of groups with few rows,
// 16-bit and fp8. Host-side interface for the C ABI layer.
#pragma once

#include "gg_kernel.h"

namespace gg {

// Operand formats (A x B) of the few-row kernel.
enum FewFormat : int { kFewBF16 = 0, kFewF16 = 1, kFewE4M3 = 2, kFewE5M2 = 3, kFewE5M2xE4M3 = 4 };

// An instance: tiles of tile_m x tile_n, `waves` waves per workgroup that split the contraction,
// a ring of `stages` chunks per wave; per_cu workgroups fit a CU (LDS), chunk_us is the time of one
// 128-byte chunk of a wave in a launch that does not fill the GPU (MI355X).
struct FewInstance {
    int    tile_m, tile_n, waves, stages, per_cu;
    double chunk_us;
};
constexpr FewInstance kFewInstances[] = {
    {16, 64, 4, 2, 2, 0.38},
    {16, 16, 8, 2, 2, 0.43},
    {32, 64, 4, 1, 3, 0.73},
    {32, 32, 4, 2, 2, 0.31},
    {64, 64, 4, 1, 2, 1.06},
};
constexpr int kFewInstanceCount = static_cast<int>(sizeof(kFewInstances) / sizeof(kFewInstances[0]));

// Enqueue a few-row launch: `grid` workgroups walk the tiles of args (tile_m, tile_n and n_tiles of
// the instance; the group table in args.groups with total_tiles, or d_total's count, or built in
// the kernel from d_lens). mn: B is stored contraction-major (dgrad's w).
hipError_t launch_few_gemm(const KernelArgs &args, int format, bool mn, int instance, int grid, hipStream_t stream);

// The 128 x 128 wgrad kernel (gg_wfew.hip): one workgroup per tile, `grid` of at least
// args.total_tiles of them (group by group: ceil(m_out / 128) x ceil(n / 128) each).
constexpr int kWgradFewTile = 128, kWgradFewThreads = 256;
hipError_t launch_wgrad_few(const KernelArgs &args, int format, int grid, hipStream_t stream);

} // namespace gg
