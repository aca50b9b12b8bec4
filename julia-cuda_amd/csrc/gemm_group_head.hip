// The grouped latency GEMM (gemm_group.h): the head's epilogues.
#include "gemm_group.h"

namespace jh {

void gemm_group_launch_head(const GemmParams& p, int epi, int bm, hipStream_t st) {
    switch (epi) {
        case EPI_K_LNBIAS: launch_group_epi<EPI_K_LNBIAS>(p, bm, st); break;
        case EPI_K_LNBIASRELU: launch_group_epi<EPI_K_LNBIASRELU>(p, bm, st); break;
        case EPI_K_LNBIASGELU: launch_group_epi<EPI_K_LNBIASGELU>(p, bm, st); break;
        case EPI_K_BIASRESSTATS: launch_group_epi<EPI_K_BIASRESSTATS>(p, bm, st); break;
        case EPI_K_BIASRESSTATS | EPI_GATHER: launch_group_epi<EPI_K_BIASRESSTATS | EPI_GATHER>(p, bm, st); break;
        case EPI_K_LNBIASGELU_SCORE: launch_group_epi<EPI_K_LNBIASGELU_SCORE>(p, bm, st); break;
        case EPI_K_LNBIASGELU_SCORE | EPI_GATHER:
            launch_group_epi<EPI_K_LNBIASGELU_SCORE | EPI_GATHER>(p, bm, st);
            break;
        default: throw std::runtime_error("gemm: no grouped kernel for epilogue " + std::to_string(epi));
    }
}

}  // namespace jh
