// The grouped latency GEMM (gemm_group.h): which GEMMs take it, and the encoder's epilogues.
#include "gemm_group.h"

namespace jh {

bool gemm_group_takes(int bm, int k) {
    return k >= 256 && bm <= group_rows_max(group_lines(k)) && group_lds_bytes(bm, k) <= GROUP_LDS_MAX;
}

int gemm_group_instance(int k) { return group_lines(k); }

// The smallest tile height whose grid is at most a block a CU (0: none). A CU's intake sets the time,
// so the shortest tiles win wherever they fit (wo at 293 rows: 16-row tiles 3.86 us, 32 4.21, 48
// 4.80, 64 5.30; wo_mlp 4.46, 5.02, 5.90, 6.62), and the tallest that fit still beat two latency tiles
// on some CUs (wi at 512 rows 6.66 against 9.64) and 128 x 128 tiles on part of the CUs (wo at 1024
// rows 96-row tiles 6.7; 128 x 128 10.7).
int gemm_group_height(int m, int n, int k, int cus) {
    for (int h : {16, 32, 48, 64, 80, 96, 128})
        if (gemm_group_takes(h, k) && (long)(n / 64) * (((long)m + h - 1) / h) <= cus) return h;
    return 0;
}

void gemm_group_launch(const GemmParams& p, int epi, int bm, hipStream_t st) {
    switch (epi) {
        case EPI_K_ROPE: launch_group_epi<EPI_K_ROPE>(p, bm, st); break;
        case EPI_K_LNROPE: launch_group_epi<EPI_K_LNROPE>(p, bm, st); break;
        case EPI_K_LNGEGLU: launch_group_epi<EPI_K_LNGEGLU>(p, bm, st); break;
        case EPI_K_RESSTATS: launch_group_epi<EPI_K_RESSTATS>(p, bm, st); break;
        case 0: launch_group_epi<0>(p, bm, st); break;
        default: gemm_group_launch_head(p, epi, bm, st);
    }
}

}  // namespace jh
