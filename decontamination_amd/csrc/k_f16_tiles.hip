// Serving forms of the 16-bit BMU search and its fallback: tiles of different requests and models share a launch.
#include "bmu_f16.hpp"

namespace {

// Serving form: one workgroup per tile; tiles of different requests and models share one launch. NW waves of G groups.
template <int DP, int NW, int G, int MODE, bool NEED_C2>
__global__ __launch_bounds__(NW * WAVE, 4) void bmu_f16_tiles_kernel(const BmuModelDev *__restrict__ models,
                                                                         const BmuTile *__restrict__ tiles,
                                                                         int64_t *__restrict__ fb_list,
                                                                         unsigned int *__restrict__ fb_count)
{
    static_assert(NW * G * 32 == SOM_TILE_ROWS, "a tile per workgroup");
    __shared__ F16Smem<DP / 16, NW, G> sm;
    const BmuTile T = tiles[blockIdx.x];
    if (T.n <= 0) return;  // uniform over the workgroup
    const BmuModelDev Md = models[T.model];
    // the descriptors' pointers are generic to the compiler: global_* accesses instead of flat ones
    bmu_f16_run<DP, f16_max_nk(DP), NW, G, MODE, NEED_C2, true, float>(Md, T.x, T.n, T.row0, T.default_index, T.c1, T.c2, T.d1, fb_list,
                                                   fb_count, (int64_t)blockIdx.x << FB_TILE_SHIFT, sm, nullptr, nullptr);
}

// Fallback of the serving form: one workgroup per (tile, row) entry of the list (entries of one launch
// may belong to different models).
template <int DP, int MODE>
__global__ __launch_bounds__(FB_THREADS) void bmu_exact_tiles_kernel(const BmuModelDev *__restrict__ models,
                                                                     const BmuTile *__restrict__ tiles,
                                                                     const int64_t *__restrict__ list,
                                                                     const unsigned int *__restrict__ list_count)
{
    __shared__ Top2Slot red[FB_THREADS / WAVE];
    const int64_t total = (int64_t)(*list_count);
    for (int64_t t = blockIdx.x; t < total; t += gridDim.x) {
        const int64_t e = list[t];
        const BmuTile T = tiles[e >> FB_TILE_SHIFT];
        const int64_t i = e & ((1ll << FB_TILE_SHIFT) - 1);
        const BmuModelDev Md = models[T.model];
        const Top2 tp = group_exact_top2<DP, MODE, float>(T.x + i * Md.dim, Md.dim, Md, red);
        if (threadIdx.x == 0) {
            ((gptr<int32_t>)T.c1)[i] = tp.i1 >= 0 ? tp.i1 : T.default_index;
            if (T.c2) ((gptr<int32_t>)T.c2)[i] = tp.i2;
            if (T.d1) ((gptr<double>)T.d1)[i] = tp.i1 >= 0 ? tp.d1 : __builtin_nan("");
        }
    }
}

constexpr int TILES_FEW = 256;  // one tile per CU

}  // namespace

int somhip_launch_bmu_tiles(hipStream_t st, int dpad, int arithmetic, int need_c2, const BmuModelDev *models,
                            const BmuTile *tiles, int grid, int64_t *fb_list, unsigned int *fb_count)
{
    if (grid <= 0) return SOMHIP_OK;
    if (dpad != 16 && dpad != 32) {
        somhip_set_error("serving supports dim <= 32");
        return SOMHIP_ERR_UNSUPPORTED;
    }
    // Launches that leave CUs with one tile take it in 16 waves of one group, which hide each other's latency: 250,000 rows of requests to a
    // 64x64 map of 32 dims and a 32x32 one took 172 and 55 us a launch in 8 waves of two groups, 140 and 48 us so.
    // Fuller ones keep 8 waves of two groups, which read each fragment once for both.
    const bool few = grid <= TILES_FEW;
    dim3 g((unsigned)grid);
    const int fb_grid = std::max(1, std::min(grid, 1024));
#define SOM_TL(D, MO, C)                                                                                  \
    do {                                                                                                  \
        if (few)                                                                                          \
            hipLaunchKernelGGL((bmu_f16_tiles_kernel<D, 2 * NW_F16, 1, MO, C>), g, dim3(2 * NW_F16 * WAVE), 0, st, models, \
                               tiles, fb_list, fb_count);                                                 \
        else                                                                                              \
            hipLaunchKernelGGL((bmu_f16_tiles_kernel<D, NW_F16, G_F16, MO, C>), g, dim3(NW_F16 * WAVE), 0, st, models, \
                               tiles, fb_list, fb_count);                                                 \
        hipLaunchKernelGGL((bmu_exact_tiles_kernel<D, MO>), dim3(fb_grid), dim3(256), 0, st, models,       \
                           tiles, fb_list, fb_count);                                                    \
    } while (0)
#define SOM_TL2(D)                                                                                        \
    do {                                                                                                  \
        if (arithmetic == SOMHIP_RERANK_FP64) {                                                           \
            if (need_c2) SOM_TL(D, SOMHIP_RERANK_FP64, true); else SOM_TL(D, SOMHIP_RERANK_FP64, false);  \
        } else {                                                                                          \
            if (need_c2) SOM_TL(D, SOMHIP_RERANK_REF32, true); else SOM_TL(D, SOMHIP_RERANK_REF32, false); \
        }                                                                                                 \
    } while (0)
    if (dpad == 16) SOM_TL2(16);
    else SOM_TL2(32);
#undef SOM_TL2
#undef SOM_TL
    SOM_HIP_TRY(hipGetLastError());
    return SOMHIP_OK;
}
