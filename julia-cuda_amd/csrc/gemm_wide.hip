// The wide throughput GEMM kernel (gemm_wide.h) and its launcher.
#include <algorithm>
#include <stdexcept>
#include <string>

#include "gemm_wide.h"

namespace jh {

// Dynamic LDS: Wide<BM>::LDS_BYTES, one block a CU. The grid is at most a block a CU and each block
// runs its tasks in one stream of stage copies.
template <int BM, int EPI, bool SPLIT>
__global__ __launch_bounds__(Wide<BM>::THREADS, 2) void gemm_wide(GemmParams p) {
    extern __shared__ __attribute__((aligned(16))) char lds_dyn[];
    gemm_wide_run<BM, EPI, false, false, SPLIT>(p, blockIdx.x, gridDim.x, lds_dyn);
}

// The tile height of an unsplit m x n GEMM on `cus` CUs: the rounds of tiles over the CUs, times a
// tile's time, which grows as its rows plus about 53 (a tile's measured times at 18752 x 2304 x 768,
// K loop and epilogue: 13.4 us at 160 rows, 15.2 at 192, 17.4 at 224, 19.3 at 256). Measured against
// the other heights (us): qkv at 18752 rows 224 (66.4; 256: 71, 192: 70, 160: 78), at 8192 rows 160
// (33.7; 192: 36.2, 224: 39.6, 256: 42), at 4096 rows 160 (18.5; 192: 20.2, 224: 20.9); wo at
// 18752 rows 224 (29.1; 256: 30.1, 160: 36.5).
int wide_height(int m, int n, int cus) {
    int best = 256;
    long best_cost = -1;
    for (int h : {256, 224, 192, 160}) {
        const long tiles = (long)(n / WIDE_BN) * ((m + h - 1) / h);
        const long cost = (tiles + cus - 1) / cus * (h + 53);
        if (best_cost < 0 || cost < best_cost) best_cost = cost, best = h;
    }
    return best;
}

template <int BM, int EPI, bool SPLIT>
static void launch_wide(const GemmParams& p, hipStream_t st) {
    using C = Wide<BM>;
    static const bool lds_ok =  // once per instantiation, before its first launch
        hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_wide<BM, EPI, SPLIT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS_BYTES) == hipSuccess;
    if (!lds_ok) throw std::runtime_error("gemm: the wide throughput kernel cannot have its LDS");
    const int grid = std::min(p.tiles_n * p.tiles_m * p.splits, device_cus());
    hipLaunchKernelGGL((gemm_wide<BM, EPI, SPLIT>), dim3(grid), dim3(C::THREADS), (C::LDS_BYTES), st, p);
}

template <int EPI>
static void launch_height(const GemmParams& p, int bm, hipStream_t st) {
    if (p.splits > 1) {
        if (bm == 192) launch_wide<192, EPI, true>(p, st);
        else launch_wide<256, EPI, true>(p, st);
        return;
    }
    switch (bm) {
        case 160: launch_wide<160, EPI, false>(p, st); break;
        case 192: launch_wide<192, EPI, false>(p, st); break;
        case 224: launch_wide<224, EPI, false>(p, st); break;
        default: launch_wide<256, EPI, false>(p, st); break;
    }
}

void gemm_wide_launch(const GemmParams& p, int epi, int bm, hipStream_t st) {
    switch (epi) {
        case EPI_K_ROPE: launch_height<EPI_K_ROPE>(p, bm, st); break;
        case EPI_K_LNROPE: launch_height<EPI_K_LNROPE>(p, bm, st); break;
        case EPI_K_LNGEGLU: launch_height<EPI_K_LNGEGLU>(p, bm, st); break;
        case EPI_K_RESSTATS: launch_height<EPI_K_RESSTATS>(p, bm, st); break;
        case EPI_K_LNBIAS: launch_height<EPI_K_LNBIAS>(p, bm, st); break;
        case EPI_K_LNBIASRELU: launch_height<EPI_K_LNBIASRELU>(p, bm, st); break;
        case EPI_K_LNBIASGELU: launch_height<EPI_K_LNBIASGELU>(p, bm, st); break;
        case EPI_K_BIASRESSTATS: launch_height<EPI_K_BIASRESSTATS>(p, bm, st); break;
        case 0: launch_height<0>(p, bm, st); break;
        default: throw std::runtime_error("gemm: no wide kernel for epilogue " + std::to_string(epi));
    }
}

}  // namespace jh
