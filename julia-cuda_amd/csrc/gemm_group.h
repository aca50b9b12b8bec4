// One output tile of the grouped latency GEMM (BM rows x 64 columns, or 128, or 32), for grids of at most a
// block a CU: eight waves in four K groups of two column halves.
//
// Bound by a launch and a first round trip (~2.5 us), then by how fast a CU takes in its operands: a
// 48-row tile at K = 768 asks for 1344 lines of 128 bytes, about 2 ns each.
//
// a's rows of the tile go into LDS once, whole: K is cut on its 128-byte lines, group g taking lines
// [g N / 4, (g + 1) N / 4) of the N = K / 64, copied by its two waves (half the rows each) as 8 rows x
// one line a copy, ahead of any other load of the tile. Each wave's fragments of w (its K range's 32
// columns) follow, straight into registers, all in flight at once. A CU takes in its operands in the
// order they were asked for, so w's arrival covers the block's barrier on a and the fragment reads.
// The four partial tiles are summed through LDS, in a's space, in group order.
//
// Eight K groups of one wave each (64 columns wide, a copied per wave) asked for a third more lines of
// a where a wave's K range is no whole number of them (K = 768: 16 copies a row for 12 lines), left
// eight partials to sum, and their LDS kept tiles at 64 rows, so that longer inputs ran two tiles a
// CU or 128 x 128 tiles on half the CUs. Measured (MI355X, us a launch, that against this): 293 rows
// qkv 5.67 / 5.15, wi 5.74 / 5.29, wo 4.01 / 3.86, wo_mlp 4.66 / 4.46; 400 rows qkv 6.37 / 5.68; 512
// rows wi 9.64 / 6.66 (80-row tiles), wo_mlp 5.43 / 5.10; 650 rows qkv 9.97 / 7.20 (96-row tiles);
// 1024 rows wo 5.90 / 5.48, wo_mlp 9.17 / 6.75. No gain: the fragments of every step read ahead of
// the MFMAs (qkv 5.33), a group's two waves on one SIMD or adjacent (5.29).
#pragma once

#include <stdexcept>
#include <string>

#include "gemm_tile.h"

namespace jh {

// Dynamic LDS bytes for K: a's rows, or the four partials (rows padded to 68 floats) and a word for
// the score's arrival.
__host__ __device__ constexpr int group_lds_bytes(int bm, int k) {
    return bm * k * 2 > 4 * bm * 68 * 4 + 16 ? bm * k * 2 : 4 * bm * 68 * 4 + 16;
}
constexpr int GROUP_LDS_MAX = 160 * 1024;

// The K lines of the widest group (the instance that runs K), and the highest tile each instance has
// (by a's LDS at its largest K).
constexpr int group_lines(int k) { return (k >> 6) <= 8 ? 2 : ((k >> 6) + 3) / 4; }
constexpr int group_rows_max(int kl) { return kl == 2 ? 128 : kl == 3 ? 96 : kl <= 5 ? 64 : kl == 6 ? 48 : 0; }
// The lowest tile of 128 columns: past what the highest of 64 columns covers.
constexpr int group2_rows_min(int kl) { return kl == 2 ? 256 : kl == 3 ? 64 : kl <= 5 ? 48 : 32; }
constexpr int GROUP2_ROWS_MAX = 64;  // (past it the sum and the epilogue take what the K loop gains)

// Task `task` of tiles_n * tiles_m (XCD-mapped); KL: the K lines of the widest group; NC: the tile's
// 64-column groups, 0: half of one, columns 16 h .. + 15 and 32 + 16 h .. + 15 (the RoPE and GeGLU pairs
// x, x + 32 whole; not the statistics of a group's output, nor the score's partials).
template <int BM, int EPI, int KL, int NC>
__device__ __forceinline__ void gemm_group_tile(const GemmParams& p, int task, char* lds) {
    constexpr int MI = BM / 16, RB = BM / 16;  // 16-row fragments; a wave's copies a line
    constexpr int FJ = NC ? 2 * NC : 1;        // a wave's 16-column fragments
    constexpr int CG = NC ? NC : 1;            // the tile's column groups, whole or in part
    static_assert(NC || !(EPI & (EPI_STATS | EPI_SCORE)), "half a column group");
    constexpr int D = NC <= 1 || 2 * KL < 6 ? 2 * KL : 6;  // K steps of w in flight
    constexpr int NPASS = (BM + 63) / 64;
    const int L = xcd_task(task, p.tiles_n * p.tiles_m);
    const int by = L % p.tiles_m, bt = L / p.tiles_m;
    const int bx = NC ? bt : bt >> 1, hb = bt & 1;  // (hb: the half, with NC = 0)
    const int tid = threadIdx.x, l = tid & 63, r16 = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform
    const int kg = w & 3, ch = w >> 2;
    const int NL = p.k >> 6, l0 = kg * NL >> 2, nl = ((kg + 1) * NL >> 2) - l0;  // KL or KL - 1 lines

    // Copy (line, rb): rows 8 rb .. 8 rb + 7 of the line at LDS (line (BM / 8) + rb) 1024; lane l's 16
    // bytes are row l / 8, chunk (l % 8) ^ sw(row), sw(r) = (r % 8) ^ ((r / 8) % 2): the 16 rows one
    // fragment read takes cover the 64 banks.
    uint32_t aoff[RB];
    {
        const int a_rows = (EPI & EPI_GATHER) ? p.src_m : p.m;
        const auto ar = buffer_rsrc(p.a, (uint32_t)((size_t)a_rows * p.k * 2));
#pragma unroll
        for (int q = 0; q < RB; q++) {
            const int r = 8 * (ch * RB + q) + (l >> 3);
            const int row = min(by * BM + r, p.m - 1);  // rows past m: read, never stored
            aoff[q] = ((uint32_t)src_row<EPI>(p, row) * (uint32_t)p.k +
                       (uint32_t)(l0 * 64 + ((l & 7) ^ (r & 7) ^ ((r >> 3) & 1)) * 8)) * 2u;
        }
        char* dst = lds + (l0 * (BM / 8) + ch * RB) * 1024;
#pragma unroll
        for (int li = 0; li < KL; li++) {
            if (li < KL - 1 || nl == KL) {  // (wave-uniform)
#pragma unroll
                for (int q = 0; q < RB; q++)
                    lds_bdma16<false>(ar, aoff[q], dst + (li * (BM / 8) + q) * 1024, (uint32_t)li * 128u);
            }
        }
    }

    __builtin_amdgcn_sched_barrier(0);  // (the wait below counts w's loads as issued after the copies)

    // The epilogue's other inputs, in flight with the operands.
    const int c0 = (tid & 7) * 4;
    EpiCol ec;
    EpiRow er[NPASS];
    epi_load_col<EPI>(p, CG * bx, c0, ec);
#pragma unroll
    for (int ps = 0; ps < NPASS; ps++) epi_load_row<EPI, false>(p, by * BM + ps * 64 + (tid >> 3), CG * bx, c0, er[ps]);

    // w in fragment order: unit u's fragment j of column group c is 512 values at ((c U + u) 4 + j) 512,
    // lane l's 8 of them at 8 l. Through a descriptor over the group's units: a step past them reads
    // zeros without touching memory.
    half8 fw[D][FJ];
    const int wg = NC == 2 ? 2 * bx + ch : bx, j0 = NC == 2 ? 0 : NC == 1 ? 2 * ch : hb + 2 * ch;
    const auto wr = buffer_rsrc((const f16*)p.w + ((size_t)wg * 2 * NL + 2 * l0) * 2048, (uint32_t)nl * 8192);
    auto load_w = [&](int s) {
#pragma unroll
        for (int j = 0; j < FJ; j++)
            fw[s % D][j] = bload16<false>(wr, (uint32_t)s * 4096 + (j0 + j) * 1024 + l * 16);
    };
#pragma unroll
    for (int s = 0; s < D; s++) load_w(s);
#pragma unroll
    for (int q = 0; q < RB; q++) asm volatile("" ::"v"(aoff[q]));  // (not w's registers: no wait for the copies)
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt<D * FJ>();  // the copies, which went out before w's loads
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    // (The RoPE table rows wait for the positions: after the copies' wait, see gemm_tile.h.)
#pragma unroll
    for (int ps = 0; ps < NPASS; ps++) epi_load_rope<EPI>(p, by * BM + ps * 64 + (tid >> 3), c0, er[ps]);
    __builtin_amdgcn_sched_barrier(0);

    floatx4 acc[MI][FJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < FJ; j++) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    const int sw = (r16 & 7) ^ (r16 >> 3);
    const char* ab = lds + l0 * (BM / 8) * 1024 + (r16 >> 3) * 1024 + (r16 & 7) * 128;
#pragma unroll
    for (int s = 0; s < 2 * KL; s++) {
        if (s < 2 * KL - 2 || nl == KL) {  // (wave-uniform)
            half8 fa[MI];
#pragma unroll
            for (int i = 0; i < MI; i++)
                fa[i] = *(const half8*)(ab + ((s >> 1) * (BM / 8) + 2 * i) * 1024 + 16 * ((4 * (s & 1) + g) ^ sw));
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < FJ; j++) acc[i][j] = mfma16(fw[s % D][j], fa[i], acc[i][j]);
        }
        if (s + D < 2 * KL) load_w(s + D);
    }
    EpiCol ec1;  // the second column group's inputs
    EpiRow er1[NPASS];
    if constexpr (NC == 2) {
        epi_load_col<EPI>(p, 2 * bx + 1, c0, ec1);
#pragma unroll
        for (int ps = 0; ps < NPASS; ps++) {
            er1[ps] = er[ps];
            epi_load_res<EPI, false>(p, by * BM + ps * 64 + (tid >> 3), 2 * bx + 1, c0, er1[ps]);
        }
    }
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();  // every wave has read its rows of a: the partials take their space

    // acc[i][j] lane: row 16 i + r16, columns 16 (j0 + j) + 4 g + e of its column group. The groups one
    // after the other: partials, sum, epilogue.
    float* red = (float*)lds;  // [K group][row][68]
#pragma unroll
    for (int cg = 0; cg < CG; cg++) {
        if (CG == 1 || ch == cg) {
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < FJ; j++)
                    *(floatx4*)&red[(kg * BM + 16 * i + r16) * 68 + 16 * (j0 + j) + 4 * g] = acc[i][j];
        }
        __syncthreads();
        float v[NPASS][8];
#pragma unroll
        for (int ps = 0; ps < NPASS; ps++) {
            const int r = ps * 64 + (tid >> 3);
#pragma unroll
            for (int e = 0; e < 8; e++) v[ps][e] = 0.0f;
            if (r < BM) {
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const float4 lo = *(const float4*)&red[(k * BM + r) * 68 + c0];
                    const float4 hi = *(const float4*)&red[(k * BM + r) * 68 + 32 + c0];
                    v[ps][0] += lo.x, v[ps][1] += lo.y, v[ps][2] += lo.z, v[ps][3] += lo.w;
                    v[ps][4] += hi.x, v[ps][5] += hi.y, v[ps][6] += hi.z, v[ps][7] += hi.w;
                }
            }
        }
        if (cg + 1 < CG) __syncthreads();
        finish<NPASS, EPI, false, 512>(p, v, bx * p.tiles_m + by, 0, by * BM, CG * bx + cg, BM,
                                       (uint32_t*)(lds + 4 * BM * 68 * 4), cg ? ec1 : ec, cg ? er1 : er,
                                       NC || (c0 >> 4) == hb);
    }
}

// ---- the kernel and its launcher, instantiated by the .hip files that include this -------------

// Dynamic LDS: group_lds_bytes(BM, k), one block a CU.
template <int BM, int EPI, int KL, int NC>
__global__ __launch_bounds__(512, 1) void gemm_group(GemmParams p) {
    extern __shared__ __attribute__((aligned(16))) char lds_dyn[];
    gemm_group_tile<BM, EPI, KL, NC>(p, blockIdx.x, lds_dyn);
}

template <int BM, int EPI, int KL, int NC>
void launch_group(const GemmParams& p, hipStream_t st) {
    static const bool lds_ok =  // once per instantiation, before its first launch
        hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_group<BM, EPI, KL, NC>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, GROUP_LDS_MAX) == hipSuccess;
    if (!lds_ok) throw std::runtime_error("gemm: the grouped latency kernel cannot have its LDS");
    hipLaunchKernelGGL((gemm_group<BM, EPI, KL, NC>), dim3(p.tiles_n * p.tiles_m), dim3(512), group_lds_bytes(BM, p.k),
                       st, p);
}

template <int BM, int EPI, int NC, int KL = 2>
void launch_group_lines(const GemmParams& p, hipStream_t st) {
    if constexpr (NC == 2 && BM < group2_rows_min(KL)) {
        if (group_lines(p.k) != KL) launch_group_lines<BM, EPI, NC, KL + 1>(p, st);
        else throw std::runtime_error("gemm: no grouped kernel for k = " + std::to_string(p.k));
    } else if constexpr (BM <= group_rows_max(KL)) {
        if (group_lines(p.k) == KL) launch_group<BM, EPI, KL, NC>(p, st);
        else launch_group_lines<BM, EPI, NC, KL + 1>(p, st);
    } else {
        throw std::runtime_error("gemm: no grouped kernel for k = " + std::to_string(p.k));
    }
}

template <int EPI>
void launch_group_epi(const GemmParams& p, int bm, hipStream_t st) {
    switch (bm) {
        case 16: launch_group_lines<16, EPI, 1>(p, st); return;
        case 32: launch_group_lines<32, EPI, 1>(p, st); return;
        case 48: launch_group_lines<48, EPI, 1>(p, st); return;
        case 64: launch_group_lines<64, EPI, 1>(p, st); return;
    }
    if constexpr (!(EPI & (EPI_GATHER | EPI_SCORE))) {  // (gathered rows and the score: up to 64 rows)
        switch (bm) {
            case 80: launch_group_lines<80, EPI, 1>(p, st); return;
            case 96: launch_group_lines<96, EPI, 1>(p, st); return;
            case 128: launch_group_lines<128, EPI, 1>(p, st); return;
        }
    }
    throw std::runtime_error("gemm: no grouped kernel of " + std::to_string(bm) + " rows");
}

template <int EPI>
void launch_group2_epi(const GemmParams& p, int bm, hipStream_t st) {
    switch (bm) {
        case 32: launch_group_lines<32, EPI, 2>(p, st); break;
        case 48: launch_group_lines<48, EPI, 2>(p, st); break;
        default: launch_group_lines<64, EPI, 2>(p, st); break;
    }
}

template <int EPI>
void launch_group0_epi(const GemmParams& p, hipStream_t st) {
    launch_group_lines<16, EPI, 0>(p, st);
}

void gemm_group_launch_head(const GemmParams& p, int epi, int bm, hipStream_t st);

}  // namespace jh
