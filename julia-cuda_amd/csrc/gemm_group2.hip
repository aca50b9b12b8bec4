// The grouped latency GEMM (gemm_group.h) on tiles of two column groups, and of half a one.
#include "gemm_group.h"

namespace jh {

static bool group2_takes(int bm, int k) {
    const int kl = group_lines(k);
    return k >= 256 && bm >= group2_rows_min(kl) && bm <= group_rows_max(kl) && bm <= GROUP2_ROWS_MAX &&
           group_lds_bytes(bm, k) <= GROUP_LDS_MAX;
}

// The smallest such tile whose grid is at most a block a CU (0: none), where gemm_group_height has
// none. Against 128 x 128 tiles on part of the CUs (MI355X, us, those / this): qkv at 896 rows 10.3 /
// 8.4 on 64-row tiles, wo at 2048 and 2600 rows 9.4 / 7.9 and 9.6 / 8.1; wo_mlp (K = 1152) at 1500
// rows 12.8 / 8.8 on 48-row tiles, at 2048 and 2600 rows 15.9 / 10.5 and 16.7 / 13.0 on 64. 80- and
// 96-row tiles were level or slower (qkv at 1024 rows 10.3 / 10.0 / 10.7), as was every one at K = 384.
int gemm_group2_height(int m, int n, int k, int cus, int epi) {
    if (n % 128 || (epi & (EPI_GATHER | EPI_SCORE)) || ((epi & EPI_LN) && k > GEMM_BIG_LN_MAX_K)) return 0;
    for (int h : {32, 48, 64})
        if (group2_takes(h, k) && (long)(n / 128) * (((long)m + h - 1) / h) <= cus) return h;
    return 0;
}

// Tiles of 16 rows x 32 columns where that grid is at most a block a CU: a CU then takes in half of
// w's 64 columns (MI355X, us, 16 x 64 tiles / this: the scorer's lin1 on 6 rows 4.1 / 3.6, linear1 on 80
// rows 3.9 / 3.5, qkv on 48 rows 3.95 / 3.4, at d = 384 on 100 rows 4.0 / 3.2). Not with output
// statistics (a group's are one block's) or the score.
bool gemm_group0_takes(int m, int n, int k, int cus, int epi) {
    return k >= 256 && group_rows_max(group_lines(k)) && !(epi & (EPI_STATS | EPI_SCORE | EPI_GATHER)) &&
           (long)(n / 32) * (((long)m + 15) / 16) <= cus;
}

void gemm_group0_launch(const GemmParams& p, int epi, hipStream_t st) {
    switch (epi) {
        case EPI_K_ROPE: launch_group0_epi<EPI_K_ROPE>(p, st); break;
        case EPI_K_LNROPE: launch_group0_epi<EPI_K_LNROPE>(p, st); break;
        case EPI_K_LNGEGLU: launch_group0_epi<EPI_K_LNGEGLU>(p, st); break;
        case EPI_K_LNBIAS: launch_group0_epi<EPI_K_LNBIAS>(p, st); break;
        case EPI_K_LNBIASRELU: launch_group0_epi<EPI_K_LNBIASRELU>(p, st); break;
        case EPI_K_LNBIASGELU: launch_group0_epi<EPI_K_LNBIASGELU>(p, st); break;
        case 0: launch_group0_epi<0>(p, st); break;
        default: throw std::runtime_error("gemm: no half-group kernel for epilogue " + std::to_string(epi));
    }
}

void gemm_group2_launch(const GemmParams& p, int epi, int bm, hipStream_t st) {
    switch (epi) {
        case EPI_K_ROPE: launch_group2_epi<EPI_K_ROPE>(p, bm, st); break;
        case EPI_K_LNROPE: launch_group2_epi<EPI_K_LNROPE>(p, bm, st); break;
        case EPI_K_LNGEGLU: launch_group2_epi<EPI_K_LNGEGLU>(p, bm, st); break;
        case EPI_K_RESSTATS: launch_group2_epi<EPI_K_RESSTATS>(p, bm, st); break;
        case EPI_K_LNBIAS: launch_group2_epi<EPI_K_LNBIAS>(p, bm, st); break;
        case EPI_K_LNBIASRELU: launch_group2_epi<EPI_K_LNBIASRELU>(p, bm, st); break;
        case EPI_K_LNBIASGELU: launch_group2_epi<EPI_K_LNBIASGELU>(p, bm, st); break;
        case EPI_K_BIASRESSTATS: launch_group2_epi<EPI_K_BIASRESSTATS>(p, bm, st); break;
        case 0: launch_group2_epi<0>(p, bm, st); break;
        default: throw std::runtime_error("gemm: no two-group kernel for epilogue " + std::to_string(epi));
    }
}

}  // namespace jh
