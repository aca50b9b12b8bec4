// One output tile of the latency GEMM (BM = 16/32/48/64 rows x 64 columns), as a device function:
// the body of the per-GEMM `gemm_lat` kernels and a task of the persistent layer kernel, which
// pass their own LDS. See gemm.hip for the design.
#pragma once

#include <type_traits>

#include "device.h"

namespace jh {

// The LDS floats of one wave of a BM-row latency tile: its partial BM x 64 tile (rows padded to 68
// floats).
template <int BM>
constexpr int lat_slot_floats() { return BM * 68; }
// LDS floats gemm_lat_tile<BM> needs with NW waves.
template <int BM, int NW = 4>
constexpr int lat_lds_floats() { return NW * lat_slot_floats<BM>(); }

// Rows of one epilogue pass of a four-wave latency tile (256 threads, 8 a row): the unit in which
// a K split's partial tile is stored (gemm_ws_floats sizes the scratch by it). Only four-wave
// tiles take a K split.
constexpr int LAT_SPLIT_PASS_ROWS = 32;

// Shared tail: each thread's 8 values (K fully summed within the block) -> the split-K
// reduction when the grid splits K -> the epilogue. Thread t of NT owns row (pass * NT / 8 +
// t / 8) of the tile and columns c0 = 4 (t % 8), c0 + 32 of 64-column group `grp`.
//
// cols: whether the thread's columns are the tile's (the grouped kernel's tiles of half a group).
//
// Split-K (kernels/src/gemm.rs:355-433): every block writes its partial to the scratch
// (device-coherent stores), waits for them to complete, then counts its arrival; the last of the
// tile's splits (which resets the counter) invalidates its caches and sums all partials in split
// order, so the result does not depend on arrival order.
template <int NPASS, int EPI, bool XG = false, int NT = 256>
__device__ __forceinline__ void finish(const GemmParams& p, float (&v)[NPASS][8], int tile_id,
                                       int z, int row0, int grp, int rows_in_tile,
                                       uint32_t* s_last, const EpiCol& ec,
                                       const EpiRow (&er)[NPASS], bool cols = true) {
    const int tid = threadIdx.x;
    if (p.splits > 1) {
        // [tile][split][pass][half][thread] float4s: coalesced stores and loads.
        // (one buffer descriptor over the tile's partials: 16-byte coherent stores and loads)
        const auto part = buffer_rsrc(p.ws + (size_t)(tile_id * p.splits) * NPASS * 2 * NT * 4,
                                      p.splits * NPASS * 2 * NT * 16);
        const uint32_t mine = (uint32_t)z * NPASS * 2 * NT * 16;
#pragma unroll
        for (int ps = 0; ps < NPASS; ps++)
#pragma unroll
            for (int h = 0; h < 2; h++)
                bstore16f(part, mine + ((ps * 2 + h) * NT + tid) * 16,
                          make_float4(v[ps][4 * h], v[ps][4 * h + 1], v[ps][4 * h + 2], v[ps][4 * h + 3]));
        release_wait();
        __syncthreads();
        if (tid == 0) {
            const uint32_t old = atomic_add_agent(p.counters + tile_id, 1u);
            const uint32_t last = old == (uint32_t)(p.splits - 1);
            if (last) atomic_store_agent(p.counters + tile_id, 0u);
            *s_last = last;
        }
        __syncthreads();
        const uint32_t last = *s_last;
        __syncthreads();  // every thread has read s_last before anyone can write it again
        if (last == 0) return;
#pragma unroll
        for (int ps = 0; ps < NPASS; ps++)
#pragma unroll
            for (int e = 0; e < 8; e++) v[ps][e] = 0.0f;
        for (int zz = 0; zz < p.splits; zz++) {
            const uint32_t src = (uint32_t)zz * NPASS * 2 * NT * 16;
#pragma unroll
            for (int ps = 0; ps < NPASS; ps++)
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const float4 q = bload16f(part, src + ((ps * 2 + h) * NT + tid) * 16);
                    v[ps][4 * h] += q.x;
                    v[ps][4 * h + 1] += q.y;
                    v[ps][4 * h + 2] += q.z;
                    v[ps][4 * h + 3] += q.w;
                }
        }
    }
    const int c0 = (tid & 7) * 4;
#pragma unroll
    for (int ps = 0; ps < NPASS; ps++) {
        const int r = ps * (NT / 8) + (tid >> 3);
        const int row = row0 + r;
        epi_apply<EPI, XG>(p, row, grp, c0, v[ps], cols && r < rows_in_tile && row < p.m, ec, er[ps]);
    }
    if (EPI & EPI_SCORE) {
        // Every tile's partials are stored (device-coherent) before its arrival counts; the last
        // tile to arrive (which resets the counter) sums each row's partials in column order.
        release_wait();
        __syncthreads();
        if (tid == 0) {
            const uint32_t old = atomic_add_agent(p.counters, 1u);
            const uint32_t last = old == (uint32_t)(p.tiles_n * p.tiles_m - 1);
            if (last) atomic_store_agent(p.counters, 0u);
            *s_last = last;
        }
        __syncthreads();
        const uint32_t last = *s_last;
        __syncthreads();  // every thread has read s_last before anyone can write it again
        if (last) {
            for (int r = tid; r < p.m; r += NT) {
                float acc = 0.0f;
                for (int t = 0; t < p.tiles_n; t++) acc += xload32(p.ws + (size_t)r * p.tiles_n + t);
                p.logits[r] = acc + p.score_b;
            }
        }
    }
}

// Task `task` (of tiles_n * tiles_m * splits; XCD-mapped) of c = epilogue(a . w^T). The NW
// waves split the tile's K steps between them; `red` is lat_lds_floats<BM, NW>() floats of LDS.
// Every thread of the block calls it; it ends with a block barrier, so the caller may reuse
// `red` right after. Eight waves (NW = 8: a block with its CU to itself) take a CU's operand loads at
// a higher rate than four.
template <int BM, int EPI, bool XG = false, int NW = 4>
__device__ __forceinline__ void gemm_lat_tile(const GemmParams& p, int task, float* red,
                                              uint32_t* s_last, uint64_t* sub = nullptr) {
    auto mark = [&](int i) {  // profiling: thread 0's view of the task's stages
        if (sub && threadIdx.x == 0) sub[i] = wall_clock64();
    };
    mark(0);
    constexpr int MI = BM / 16;
    constexpr int RPP = 8 * NW;                     // tile rows a pass of the epilogue
    constexpr int NPASS = (BM + RPP - 1) / RPP;
    constexpr int SLOT = lat_slot_floats<BM>();  // a wave's LDS floats
    static_assert(NW != 4 || RPP == LAT_SPLIT_PASS_ROWS, "split partials are sized by 32-row passes");
    const int T = p.tiles_n * p.tiles_m * p.splits;
    const int L = xcd_task(task, T);
    const int z = L % p.splits, t2 = L / p.splits;
    const int by = t2 % p.tiles_m, bx = t2 / p.tiles_m;
    const int tid = threadIdx.x, l = tid & 63, r16 = l & 15, g = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: scalar branches

    // This block's K steps (32 wide), then this wave's share of them.
    const int U = p.k >> 5;
    const int ub = z * U / p.splits, ue = (z + 1) * U / p.splits, nu = ue - ub;
    const int u0 = ub + w * nu / NW, u1 = ub + (w + 1) * nu / NW;
    const f16* ap[MI];
#pragma unroll
    for (int i = 0; i < MI; i++) {
        const int row = min(by * BM + 16 * i + r16, p.m - 1);  // rows past m: read, never stored
        ap[i] = (const f16*)p.a + (size_t)src_row<EPI>(p, row) * p.k + 8 * g;
    }
    // The epilogue's other inputs, in flight with the first operand loads.
    const int c0 = (tid & 7) * 4;
    EpiCol ec;
    EpiRow er[NPASS];
    epi_load_col<EPI>(p, bx, c0, ec);
#pragma unroll
    for (int ps = 0; ps < NPASS; ps++) epi_load_row<EPI, XG>(p, by * BM + ps * RPP + (tid >> 3), bx, c0, er[ps]);

    floatx4 acc[MI][4];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    // The wave's K steps in chunks of UC, two chunks in flight: chunk c + 1's fragments load
    // while chunk c's MFMAs run, so a wave pays one round trip to memory however many chunks its
    // K range takes. The a operand (an activation) comes through the coherent path when XG.
    //
    // The loads are unconditional within a chunk (a step past the wave's range re-reads its last
    // step, and its a fragment is masked to zero without a branch): a guarded load becomes a
    // branch, and the compiler drains every outstanding load at each divergent branch, which would
    // serialise the steps. The chunk guards depend on the wave index only (scalar branches).
    // UC K steps a chunk (2 x UC x (MI + 4) x 4 VGPRs of fragments): four, three or two; five for
    // 16-row tiles whose waves have more than eight K steps (K = 1152), which then take one round
    // trip instead of two.
    auto kloop = [&](auto uc_) {
        constexpr int UC = decltype(uc_)::value;
        half8 fa0[UC][MI], fw0[UC][4], fa1[UC][MI], fw1[UC][4];
        // w in fragment order: unit uu's fragment j is 512 values at ((bx U + uu) 4 + j) 512,
        // and lane l's 8 of them at l * 8 (W rows bx 64 + 16 j + l % 16, K 32 uu + 8 (l / 16) +
        // e); read through a buffer descriptor over exactly the wave's K steps: a slot past them
        // reads zeros without touching memory (a clamped re-read would still cost its bytes).
        const auto wr = buffer_rsrc((const f16*)p.w + ((size_t)bx * U + u0) * 2048,
                                    (uint32_t)(u1 - u0) * 4096);
        auto load = [&](half8 (&fa)[UC][MI], half8 (&fw)[UC][4], int u) {
#pragma unroll
            for (int s = 0; s < UC; s++) {
                const int uu = min(u + s, u1 - 1);
#pragma unroll
                for (int j = 0; j < 4; j++)
                    fw[s][j] = bload16<false>(wr, (uint32_t)(u + s - u0) * 4096 + j * 1024 + l * 16);
#pragma unroll
                for (int i = 0; i < MI; i++) fa[s][i] = load16h<XG>(ap[i] + uu * 32);
            }
        };
        auto compute = [&](const half8 (&fa)[UC][MI], const half8 (&fw)[UC][4], int u) {
#pragma unroll
            for (int s = 0; s < UC; s++) {
                const uint32_t keep = u + s < u1 ? 0xffffffffu : 0u;
#pragma unroll
                for (int i = 0; i < MI; i++) {
                    const half8 a = mask16(fa[s][i], keep);
#pragma unroll
                    for (int j = 0; j < 4; j++) acc[i][j] = mfma16(fw[s][j], a, acc[i][j]);
                }
            }
        };
        // (Scheduling fences keep the compiler from interleaving the MFMAs into the loads, where
        // it would reuse the fragment registers and wait for each step's loads before the next.)
        // The first two chunks unconditionally (every wave has a K step: the host checks; a slot
        // past the wave's range re-reads its last a step and reads zeros of w), so that the
        // compiler knows where the position loads stand in the load order when the table loads
        // wait for them.
        load(fa0, fw0, u0);
        load(fa1, fw1, u0 + UC);
        // The RoPE table rows after the operand loads: they wait for the positions, and issued
        // first that wait would hold back the operand loads by a round trip.
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ps = 0; ps < NPASS; ps++) epi_load_rope<EPI>(p, by * BM + ps * RPP + (tid >> 3), c0, er[ps]);
        for (int u = u0; u < u1; u += 2 * UC) {
            __builtin_amdgcn_sched_barrier(0);
            compute(fa0, fw0, u);
            __builtin_amdgcn_sched_barrier(0);
            if (u + 2 * UC < u1) load(fa0, fw0, u + 2 * UC);
            __builtin_amdgcn_sched_barrier(0);
            if (u + UC < u1) compute(fa1, fw1, u + UC);
            __builtin_amdgcn_sched_barrier(0);
            if (u + 3 * UC < u1) load(fa1, fw1, u + 3 * UC);
        }
    };
    if (MI == 1 && u1 - u0 > 8)
        kloop(std::integral_constant<int, 5>{});
    else
        kloop(std::integral_constant<int, MI == 1 ? 4 : (MI == 2 ? 3 : 2)>{});

    mark(1);
    // acc[i][j] lane: row 16 i + r16, columns 16 j + 4 g + e of the tile. Wave w's partial at
    // red[w][row][col] (rows of 68 floats).
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
            *(floatx4*)&red[w * SLOT + (16 * i + r16) * 68 + 16 * j + 4 * g] = acc[i][j];
    __syncthreads();
    float v[NPASS][8];  // the partials summed in wave order
#pragma unroll
    for (int ps = 0; ps < NPASS; ps++) {
        const int r = ps * RPP + (tid >> 3);
#pragma unroll
        for (int e = 0; e < 8; e++) v[ps][e] = 0.0f;
        if (r < BM) {
#pragma unroll
            for (int ww = 0; ww < NW; ww++) {
                const float4 lo = *(const float4*)&red[ww * SLOT + r * 68 + c0];
                const float4 hi = *(const float4*)&red[ww * SLOT + r * 68 + 32 + c0];
                v[ps][0] += lo.x, v[ps][1] += lo.y, v[ps][2] += lo.z, v[ps][3] += lo.w;
                v[ps][4] += hi.x, v[ps][5] += hi.y, v[ps][6] += hi.z, v[ps][7] += hi.w;
            }
        }
    }
    __syncthreads();  // red is free again
    mark(2);
    finish<NPASS, EPI, XG, 64 * NW>(p, v, bx * p.tiles_m + by, z, by * BM, bx, BM, s_last, ec, er);
    mark(3);
}

// ---- the persistent kernel's tile: weights staged in LDS --------------------------------------
// The weight tile of a task (64 columns x one split's K units, fragment order) is one contiguous
// run of the packed matrix, nu * 4 KB. The persistent kernel copies it into LDS with direct
// global -> LDS loads, if it can before the barrier that precedes the task's phase (the weights
// do not depend on the previous phase), so that after the barrier only the activation loads
// stand between the block and its MFMAs.

struct WTile {
    int bx, ub, nu;  // 64-column group, first K unit, units
};

__device__ __forceinline__ WTile w_tile_of(const GemmParams& p, int task) {
    const int T = p.tiles_n * p.tiles_m * p.splits;
    const int L = xcd_task(task, T);
    const int z = L % p.splits, bx = (L / p.splits) / p.tiles_m;
    const int U = p.k >> 5;
    const int ub = z * U / p.splits;
    return WTile{bx, ub, (z + 1) * U / p.splits - ub};
}

// LDS bytes of the weight tile for splits of a k-wide GEMM (the largest split).
__host__ __device__ constexpr int w_tile_bytes(int k, int splits) {
    return ((k / 32 + splits - 1) / splits) * 4096;
}

// Waves [w_first, 4) copy task's weight tile to `lds` (1 KB per wave load). (Global copies: the
// same copies through a buffer descriptor made the whole-model launch 13-19% slower, the
// prefetch no longer overlapping what runs before the tile's wait.)
__device__ __forceinline__ void w_tile_fetch(const GemmParams& p, WTile t, f16* lds, int w_first) {
    const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
    if (w < w_first) return;
    const f16* src = (const f16*)p.w + (size_t)(t.bx * (p.k >> 5) + t.ub) * 2048 + l * 8;
    for (int c = w - w_first; c < 4 * t.nu; c += 4 - w_first) lds_dma16(src + (size_t)c * 512, lds + c * 512);
}

// LDS floats the cross-wave reduction of a BM-row tile needs (aliases the weight tile).
template <int BM>
constexpr int w_red_floats() { return 4 * BM * 68; }

// Task `task` of c = epilogue(a . w^T) in the persistent kernel. The weight tile is in `lds`
// already (w_ready: its loads were issued earlier by this block, maybe still in flight) or is
// fetched here. a is read with 16-byte buffer loads, rows past m reading zeros: device-coherent
// when AX (a buffer other blocks write more than once per launch, or several blocks write parts
// of one line), else through the caches (a buffer written once per launch, each 128-byte line by
// one block: no L2 can hold a stale copy). The statistics are read device-coherent, the residual
// (a write-once buffer) through the caches; the outputs are stored device-coherent. The four
// waves split the tile's K units; their partial tiles are summed through LDS, in the weight
// tile's space. Every thread calls this; it ends with a block barrier after the last LDS access.
template <int BM, int EPI, bool AX>
__device__ __forceinline__ void gemm_w_tile(const GemmParams& p, int task, char* lds, bool w_ready,
                                            uint32_t* s_last, uint64_t* sub = nullptr) {
    auto mark = [&](int i) {  // profiling: thread 0's view of the task's stages
        if (sub && threadIdx.x == 0) sub[i] = wall_clock64();
    };
    constexpr int MI = BM / 16;
    constexpr int NPASS = (BM + LAT_SPLIT_PASS_ROWS - 1) / LAT_SPLIT_PASS_ROWS;
    constexpr int UMAX = MI >= 3 ? 6 : 9;  // a fragments one wave holds: 72-96 or 36-72 VGPRs
    const int T = p.tiles_n * p.tiles_m * p.splits;
    const int L = xcd_task(task, T);
    const int z = L % p.splits, t2 = L / p.splits;
    const int by = t2 % p.tiles_m, bx = t2 / p.tiles_m;
    const int tid = threadIdx.x, w = tid >> 6, l = tid & 63, r16 = l & 15, g = l >> 4;
    const int U = p.k >> 5;
    const int ub = z * U / p.splits, nu = (z + 1) * U / p.splits - ub;
    const int u0 = w * nu / 4, u1 = (w + 1) * nu / 4;  // this wave's units, relative to ub
    f16* wl = (f16*)lds;
    if (!w_ready) w_tile_fetch(p, WTile{bx, ub, nu}, wl, 0);

    const int c0 = (tid & 7) * 4;
    EpiCol ec;
    EpiRow er[NPASS];
    epi_load_col<EPI>(p, bx, c0, ec);
#pragma unroll
    for (int ps = 0; ps < NPASS; ps++) epi_load_row<EPI, true, false>(p, by * BM + ps * 32 + (tid >> 3), bx, c0, er[ps]);
#pragma unroll
    for (int ps = 0; ps < NPASS; ps++) epi_load_rope<EPI>(p, by * BM + ps * 32 + (tid >> 3), c0, er[ps]);

    const __amdgpu_buffer_rsrc_t ra = buffer_rsrc(p.a, (uint32_t)p.m * (uint32_t)p.k * 2u);
    uint32_t aoff[MI];
#pragma unroll
    for (int i = 0; i < MI; i++)
        aoff[i] = ((uint32_t)(by * BM + 16 * i + r16) * (uint32_t)p.k + (uint32_t)(ub + u0) * 32u + 8u * g) * 2u;

    floatx4 acc[MI][4];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    half8 fa[UMAX][MI];
    auto load_a = [&](int u) {
#pragma unroll
        for (int s = 0; s < UMAX; s++) {
            const uint32_t du = (uint32_t)(min(u + s, u1 - 1) - u0) * 64u;
#pragma unroll
            for (int i = 0; i < MI; i++) fa[s][i] = bload16<AX>(ra, aoff[i] + du);
        }
    };
    // The weight fragments of unit s + 1 are read from LDS while unit s's MFMAs run (the reads
    // are unconditional, clamped to the wave's last unit; only the MFMAs are skipped).
    auto mma = [&](int u) {
        half8 fw[2][4];
        auto rd = [&](half8 (&f)[4], int uu) {
#pragma unroll
            for (int j = 0; j < 4; j++) f[j] = *(const half8*)(wl + (uu * 4 + j) * 512 + l * 8);
        };
        rd(fw[0], u);
#pragma unroll
        for (int s = 0; s < UMAX; s++) {
            if (s + 1 < UMAX) rd(fw[(s + 1) & 1], min(u + s + 1, u1 - 1));
            if (u + s < u1) {  // wave-uniform
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) acc[i][j] = mfma16(fw[s & 1][j], fa[s][i], acc[i][j]);
            }
        }
    };
    if (u0 < u1) load_a(u0);
    __builtin_amdgcn_s_waitcnt(0);  // the weight tile's loads (and the first a chunk) are done
    __syncthreads();                // ... for every wave: the whole tile is in LDS
    mark(0);
    for (int u = u0; u < u1; u += UMAX) {
        if (u != u0) load_a(u);
        mma(u);
    }
    __syncthreads();  // every wave is done with the weight tile: the reduction reuses its space
    mark(1);

    float* red = (float*)lds;
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
            *(floatx4*)&red[(w * BM + 16 * i + r16) * 68 + 16 * j + 4 * g] = acc[i][j];
    __syncthreads();
    float v[NPASS][8];
#pragma unroll
    for (int ps = 0; ps < NPASS; ps++) {
        const int r = ps * 32 + (tid >> 3);
#pragma unroll
        for (int e = 0; e < 8; e++) v[ps][e] = 0.0f;
        if (r < BM) {
#pragma unroll
            for (int ww = 0; ww < 4; ww++) {
                const float4 lo = *(const float4*)&red[(ww * BM + r) * 68 + c0];
                const float4 hi = *(const float4*)&red[(ww * BM + r) * 68 + 32 + c0];
                v[ps][0] += lo.x, v[ps][1] += lo.y, v[ps][2] += lo.z, v[ps][3] += lo.w;
                v[ps][4] += hi.x, v[ps][5] += hi.y, v[ps][6] += hi.z, v[ps][7] += hi.w;
            }
        }
    }
    __syncthreads();  // LDS is free again
    mark(2);
    finish<NPASS, EPI, true>(p, v, bx * p.tiles_m + by, z, by * BM, bx, BM, s_last, ec, er);
    if (sub) {
        release_wait();
        mark(3);
    }
}

}  // namespace jh
