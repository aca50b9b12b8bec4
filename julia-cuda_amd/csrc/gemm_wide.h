// The wide throughput GEMM's tiles (BM x 256, BM = 160, 192, 224 or 256), as a device function that
// runs a block's tasks one after another: the body of the `gemm_wide` kernel for large M and of
// the persistent kernel's large-batch phases. c = epilogue(a . w^T) with the epilogues of the
// latency tile (device.h), applied straight from the accumulators.
//
// Eight waves (two a SIMD) in a 2 x 4 grid each own a (BM / 2) x 64 block of outputs, computed with
// MFMA 16 x 16 x 32, w as the MFMA's A operand: lane l of fragment (i, j) holds output row
// 16 i + l % 16 and columns 16 j + 4 (l / 16) + e, e < 4.
//
// What bounds it, and what follows from it (MI355X, qkv's 18752 x 2304 x 768, random operands):
//  - Power. With every CU busy the clock falls to about 1.75 GHz on random operands (2.4 on
//    zeros, the same K loop: 16.6 against 12.4 us a 256-row tile), so what counts is energy a
//    flop. In a loop of MFMAs alone 16 x 16 x 32 reaches 1.88 PFLOP/s, 32 x 32 x 16 1.60.
//  - Line requests. A stage is 64 wide, so that a copy of a takes whole 128-byte lines (8 rows
//    x 128 bytes); 32-wide stages asked for every line of a twice. Both together, the tile
//    without its epilogue: 58.5 -> 52 us.
//  - The LDS: a stage's 24 to 32 KB of a and 32 KB of w are written once and read 4 and 2 times,
//    as long as the MFMAs take (a 256-row stage: 2048 clocks each at 128 bytes a clock). Four
//    waves of 128 x 128 read a third less but, one a SIMD, wait for each barrier and read
//    themselves: 57.5 us against 52.
//  - What the MFMAs wait for at a tile's ends. The stream of stage copies runs on over the
//    tasks: the next task's first stage (and half of its second) is copied under this task's
//    last stages and epilogue. The epilogue takes its loads before its first store (vector memory
//    completes in order: a load behind a store waits for the store's write-through) and uses no
//    branch, no 64-bit address and no slow multiply a store (buffer descriptors over the tile's
//    rows: rows past m read as zeros, their stores are dropped). qkv 75 -> 66 us in all.
//  - Rounds. Any multiple of 32 rows up to 256 makes a tile, so the pick takes the height whose
//    rounds over the CUs leave the least to do (wide_height in gemm_wide.hip).
//
// The K loop: two LDS stages of 64 K. A stage's two K-32 steps run row by row (4 MFMAs a 16-row
// fragment); a row's fragment of the next step is read once the row's MFMAs are issued. In the
// middle of the second step stands the stage's one barrier: every wave has read all of this
// stage (its reads were issued in the first step) and every wave's copies of the next stage have
// landed. After it this stage's space takes the first half of stage s + 2's copies, one a row,
// and the next step's fragments are read from stage s + 1; the other half of the copies goes out
// in the next stage's first rows (a burst of copies stalls the issuing wave: 8 in four rows 56 us,
// one a row over eight rows 52).
//  - a's stage: rows of 128 bytes; copy I takes rows 8 I .. 8 I + 7, lane l into LDS chunk 64 I + l =
//    chunk l % 8 of row r = 8 I + l / 8, which holds a's 16-byte chunk (l % 8) ^ ((r / 2) % 8): the
//    16 rows one fragment read takes cover the 64 banks.
//  - w's stage: 4 column groups x 2 units of the fragment-ordered matrix (64 columns x 32 K, 4 KB
//    each), copied as they are.
#pragma once

#include "gemm_tile.h"

namespace jh {

constexpr int WIDE_BN = 256;  // columns of a tile

template <int BM>
struct Wide {
    static_assert(BM % 32 == 0 && BM >= 64 && BM <= 256, "tile height");
    static constexpr int BN = WIDE_BN;
    static constexpr int BK = 64;
    static constexpr int WAVES_M = 2, WAVES_N = BN / 64;
    static constexpr int NWAVES = WAVES_M * WAVES_N, THREADS = 64 * NWAVES;
    static constexpr int WM = BM / WAVES_M;           // a wave's block: WM x 64
    static constexpr int MI = WM / 16, NJ = 4;        // its 16 x 16 fragments
    // a's rows in a stage: whole copies for every wave (160 rows take the space of 192, 224 of
    // 256; the copies past the tile's rows read nothing and write zeros).
    static constexpr int A_ROWS = (BM + 8 * NWAVES - 1) / (8 * NWAVES) * 8 * NWAVES;
    static constexpr int A_BYTES = A_ROWS * BK * 2, W_BYTES = BN * BK * 2;
    static constexpr int STAGE = A_BYTES + W_BYTES;   // bytes per stage
    static constexpr int A_LOADS = A_BYTES / 1024 / NWAVES, W_LOADS = W_BYTES / 1024 / NWAVES;
    static constexpr int LOADS = A_LOADS + W_LOADS;   // 1 KB copies a wave and stage
    static_assert(A_LOADS * NWAVES * 1024 == A_BYTES && W_LOADS * NWAVES * 1024 == W_BYTES, "copies");
    static constexpr int EARLY = LOADS / 2;  // a stage's copies issued one step earlier (below)
    static constexpr int BAR = MI / 2;       // the row of a stage's second step where the barrier stands
    // After the stages: per wave the f16 staging of 16 output rows (padded), then colsum and bias
    // of its columns; per row LayerNorm mean and rstd, RoPE position.
    static constexpr int PADH = 64 + 8;
    static constexpr int STAGING = 2 * STAGE;
    static constexpr int COLS = STAGING + NWAVES * 16 * PADH * 2;
    static constexpr int ROWS = COLS + NWAVES * 2 * 64 * 4;
    static constexpr int POSR = ROWS + BM * 8;
    static constexpr int FLAG = POSR + BM * 4;  // split-K: whether this block is a tile's last
    static constexpr int LDS_BYTES = FLAG + 16;
    static_assert(BM * 256 <= STAGE, "a tile's RoPE table rows in a stage's space");
    static_assert(THREADS >= 2 * BM, "two threads a row for the row statistics");
};

// LayerNorm statistics slots one thread reads (two threads split a row's K / 64 slots): the
// wide tiles take LayerNorm epilogues for K <= 64 * 2 * WIDE_LN_SLOTS.
constexpr int WIDE_LN_SLOTS = 8;

// Tasks first, first + stride, ... of tiles_n * tiles_m (x splits with SPLIT; XCD-mapped: an XCD
// takes a contiguous range of tasks, in the grouped order below) by a block of 512 threads. Every
// thread calls it; it ends with a block barrier, the outputs' stores still in flight. AX: a is read
// device-coherent; XG: the input statistics are. The outputs and output statistics are stored
// device-coherent on every path (written through the L2: a kernel's end then has no dirty lines of
// them to write back; plain stores 18.9 -> 21.2 us for qkv at 4096 rows, 66.7 -> 68.2 at 18752).
// The residual is read through the caches. SPLIT: p.splits K splits a tile.
template <int BM, int EPI, bool AX, bool XG, bool SPLIT = false>
__device__ __forceinline__ void gemm_wide_run(const GemmParams& p, int first, int stride, char* lds,
                                             uint64_t* sub = nullptr) {
    auto mark = [&](int i) {  // profiling: thread 0's view of the first task's stages
        if (sub && threadIdx.x == 0) sub[i] = wall_clock64();
    };
    using C = Wide<BM>;
    constexpr int BN = C::BN;
    constexpr int MI = C::MI, NJ = C::NJ;
    constexpr bool LN = (EPI & EPI_LN) != 0, BIAS = (EPI & EPI_BIAS) != 0, ROPE = (EPI & EPI_ROPE) != 0;
    constexpr bool GEGLU = (EPI & EPI_GEGLU) != 0, RES = (EPI & EPI_RES) && !GEGLU;
    constexpr bool KEEP = !ROPE;  // the epilogue does not use the stages' space
    const int S = SPLIT ? p.splits : 1;
    const int T = p.tiles_n * p.tiles_m * S;
    if (first >= T) return;
    const int tid = threadIdx.x, l = tid & 63, r16 = l & 15, g4 = l >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: scalar branches
    const int wm = w / C::WAVES_N, wn = w % C::WAVES_N;
    const int U = p.k >> 6;  // K stages

    struct Tile {
        int bx, by, t2, z, k0, nk;  // column and row block, tile, K split, its first stage and stages
    };
    auto tile_of = [&](int task) {
        Tile t;
        const int L = xcd_task(task, T);
        t.z = L % S, t.t2 = L / S;
        const int G = max(1, (2 << 20) / (BM * p.k * 2));
        const int gsz = G * p.tiles_n, grp0 = t.t2 / gsz * G, in = t.t2 % gsz;
        const int rows_g = min(G, p.tiles_m - grp0);
        t.bx = in / rows_g, t.by = grp0 + in % rows_g;
        t.k0 = t.z * U / S, t.nk = (t.z + 1) * U / S - t.k0;
        return t;
    };

    // ---- stage copies ---------------------------------------------------------------------------
    uint32_t aoff[C::A_LOADS];
#pragma unroll
    for (int q = 0; q < C::A_LOADS; q++) {
        const int r = 8 * (w + C::NWAVES * q) + (l >> 3);
        aoff[q] = (uint32_t)(r * p.k + ((l & 7) ^ ((r >> 1) & 7)) * 8) * 2u;
    }
    const uint32_t woff = l * 16;
    struct Src {
        __amdgpu_buffer_rsrc_t a, w;
        uint32_t ka, kw;
    };
    auto src_of = [&](const Tile& t, int s, bool ok) {
        const size_t arow = (size_t)t.by * BM;
        const uint32_t ab = (uint32_t)__builtin_amdgcn_readfirstlane(min(p.m - (int)arow, BM) * p.k * 2);
        const uint32_t wb = (uint32_t)((BN / 64) * U * 8192);
        return Src{buffer_rsrc(p.a + arow * p.k, ok ? ab : 0u),
                   buffer_rsrc(p.w + (size_t)t.bx * (BN / 64) * U * 4096, ok ? wb : 0u),
                   (uint32_t)(t.k0 + s) * 128u, (uint32_t)(t.k0 + s) * 8192u};
    };
    auto issue = [&](const Src& f, char* st, int q) {
        if (q < C::A_LOADS) {
            lds_bdma16<AX>(f.a, aoff[q], st + (w + C::NWAVES * q) * 1024, f.ka);
        } else {
            const int J = w + C::NWAVES * (q - C::A_LOADS);
            lds_bdma16<false>(f.w, woff, st + C::A_BYTES + J * 1024,
                              f.kw + (uint32_t)((J >> 3) * U * 8192 + (J & 7) * 1024));
        }
    };

    // ---- fragments ------------------------------------------------------------------------------
    const int arow = wm * C::WM + r16;
    const int la0 = arow * 128 + ((g4 ^ ((arow >> 1) & 7)) << 4);
    const int la1 = arow * 128 + (((4 + g4) ^ ((arow >> 1) & 7)) << 4);
    const int lw = C::A_BYTES + wn * 8192 + l * 16;
    half8 fa[2][MI], fw[2][NJ];
    auto rda = [&](const char* st, int t, int i) { fa[t][i] = *(const half8*)(st + (t ? la1 : la0) + 2048 * i); };
    auto rdw = [&](const char* st, int t, int j) { fw[t][j] = *(const half8*)(st + lw + t * 4096 + j * 1024); };

    // ---- the epilogue's per-tile inputs ------------------------------------------------------------
    const int slots = p.k >> 6;
    float* const wcols = (float*)(lds + C::COLS) + w * 2 * 64;
    struct Inputs {
        float2 sl[WIDE_LN_SLOTS];
        float cs, bs;
    };
    [[maybe_unused]] const auto sbuf = buffer_rsrc(p.stats_in, (uint32_t)p.m * (uint32_t)slots * 8u);
    // (the thread index afresh: what is derived from it is not kept in registers through the K loop)
    auto fresh_tid = [&] {
        int x = threadIdx.x;
        asm volatile("" : "+v"(x));
        return x;
    };
    auto load_inputs = [&](const Tile& t, Inputs& in) {
        const int tid = fresh_tid(), l = tid & 63;
        const uint32_t col = (uint32_t)(t.bx * BN + wn * 64 + l) * 4u;
        if (LN) in.cs = bload4(buffer_rsrc(p.colsum, (uint32_t)p.n * 4u), col);
        if (BIAS) in.bs = bload4(buffer_rsrc(p.bias, (uint32_t)p.n * 4u), col);
        if (LN) {
            const int r = min(t.by * BM + min(tid >> 1, BM - 1), p.m - 1);
            const uint32_t so = ((uint32_t)r * slots + (tid & 1)) * 8u;
#pragma unroll
            for (int u = 0; u < WIDE_LN_SLOTS; u++) in.sl[u] = bload8<XG>(sbuf, so + 16 * u);
        }
    };
    auto load_pos = [&](const Tile& t) {
        const int tid = fresh_tid();
        // (without positions an empty descriptor: zero, and the row is the position)
        const int r = min(t.by * BM + min(tid >> 1, BM - 1), p.m - 1);
        return __builtin_bit_cast(int, bload4(buffer_rsrc(p.pos, p.pos ? (uint32_t)p.m * 4u : 0u), (uint32_t)r * 4u));
    };
    auto put_pos = [&](const Tile& t, int v) {
        const int tid = fresh_tid();
        if ((tid & 1) == 0 && tid < 2 * BM) {
            const int at = p.pos ? v : t.by * BM + (tid >> 1);
            ((int*)(lds + C::POSR))[tid >> 1] = min(max(at, 0), p.rope_rows - 1);
        }
    };
    auto put_inputs = [&](const Inputs& in) {
        const int tid = fresh_tid(), l = tid & 63;
        if (LN) wcols[l] = in.cs;
        if (BIAS) wcols[64 + l] = in.bs;
        if (LN) {
            float s = 0.0f, q = 0.0f;
#pragma unroll
            for (int u = 0; u < WIDE_LN_SLOTS; u++) {
                const bool ok = 2 * u + (tid & 1) < slots;
                s += ok ? in.sl[u].x : 0.0f;
                q += ok ? in.sl[u].y : 0.0f;
            }
            s = group_sum<2>(s);
            q = group_sum<2>(q);
            const float mean = s / (float)p.k;
            const float var = fmaxf(q / (float)p.k - mean * mean, 0.0f);
            if ((tid & 1) == 0 && tid < 2 * BM)
                ((float2*)(lds + C::ROWS))[tid >> 1] = make_float2(mean, 1.0f / sqrtf(var + p.eps));
        }
    };

    mark(0);
    Tile t = tile_of(first);
    int pos = 0;  // the task's first stage in the block's stream
    {
        const bool two = t.nk > 1;  // (a one-stage task: the next task's first stage follows, below)
        const Src f0 = src_of(t, 0, true), f1 = src_of(t, two ? 1 : 0, two);
#pragma unroll
        for (int q = 0; q < C::LOADS; q++) issue(f0, lds, q);
#pragma unroll
        for (int q = 0; q < C::EARLY; q++) issue(f1, lds + C::STAGE, q);
        wait_vmcnt<C::EARLY>();
    }
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();

    for (int task = first;;) {
        const bool more = task + stride < T;
        const Tile tn = more ? tile_of(task + stride) : t;
        const Src n0 = src_of(tn, 0, more);  // the next task's first stages (no copies without one)
        const Src n1 = src_of(tn, tn.nk > 1 ? 1 : 0, more && tn.nk > 1);
        auto after = [&](int s) { return s < t.nk ? src_of(t, s, true) : n0; };
        auto at = [&](int x) { return lds + (x & 1) * C::STAGE; };  // stage x of the block's stream
        // The first half of the copies of the stage after this task's first: out already for the
        // block's first task, and where the epilogue before left the space alone.
        if (t.nk == 1 || (!KEEP && task != first)) {
            const Src f = after(1);
#pragma unroll
            for (int q = 0; q < C::EARLY; q++) issue(f, at(pos + 1), q);
        }
        floatx4 acc[MI][NJ];
#pragma unroll
        for (int j = 0; j < NJ; j++) rdw(at(pos), 0, j);
#pragma unroll
        for (int i = 0; i < MI; i++) rda(at(pos), 0, i);
#pragma unroll
        for (int i = 0; i < MI; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        const int rpos = ROPE ? load_pos(t) : 0;
        Inputs in;
        mark(1);

        constexpr int TCOPIES = ROPE ? BM / 4 / C::NWAVES : 0;  // RoPE table copies a wave
        const bool roped = ROPE && t.bx * BN < p.rope_cols;
        auto body = [&](int s, auto last_) {
            constexpr bool LAST = decltype(last_)::value;
            const Src f1 = after(s + 1), f2 = LAST ? n1 : after(s + 2);
            char* const st = at(pos + s);
            char* const sn = at(pos + s + 1);
#pragma unroll
            for (int i = 0; i < MI; i++) {
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int j = 0; j < NJ; j++) acc[i][j] = mfma16(fw[0][j], fa[0][i], acc[i][j]);
                __builtin_amdgcn_sched_barrier(0);
                if (i == 0)
#pragma unroll
                    for (int j = 0; j < NJ; j++) rdw(st, 1, j);
                rda(st, 1, i);
                if (ROPE && LAST && i == 0) put_pos(t, rpos);
                constexpr int N0 = C::LOADS - C::EARLY, R0 = MI / 2;
#pragma unroll
                for (int q = i * N0 / R0; q < (i + 1) * N0 / R0 && q < N0; q++) issue(f1, sn, C::EARLY + q);
            }
#pragma unroll
            for (int i = 0; i < MI; i++) {
                __builtin_amdgcn_sched_barrier(0);
                if (i == C::BAR) {
                    if (!LAST) wait_vmcnt<0>();
                    wait_lgkm0();
                    __builtin_amdgcn_s_barrier();
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int j = 0; j < NJ; j++) acc[i][j] = mfma16(fw[1][j], fa[1][i], acc[i][j]);
                __builtin_amdgcn_sched_barrier(0);
                if (LAST && !ROPE && i == 0) load_inputs(t, in);
                if (i >= C::BAR) {
                    // The rows after the barrier: the next stage's fragments between all but the
                    // last of them (which covers their latency), the copies between all.
                    constexpr int ROWS = MI - C::BAR, RD = ROWS > 1 ? ROWS - 1 : 1, NRD = NJ + MI;
                    const int x = i - C::BAR;
                    if (!LAST) {
#pragma unroll
                        for (int r = x * NRD / RD; r < (x + 1) * NRD / RD && r < NRD; r++) {
                            if (r < NJ) rdw(sn, 0, r);
                            else rda(sn, 0, r - NJ);
                        }
                    }
                    if (!LAST || KEEP) {
#pragma unroll
                        for (int q = x * C::EARLY / ROWS; q < (x + 1) * C::EARLY / ROWS; q++) issue(f2, st, q);
                    }
                }
                // The tile's RoPE table rows, as whole lines into the space of this stage: copy I
                // takes rows 4 I .. 4 I + 3, the 16-byte chunk c of row r at chunk c ^ (r % 16), so
                // that the 16 rows one read takes cover the 64 banks. (All positions are read before
                // the first copy: a copy between them would make the next read wait for it.)
                if (LAST && ROPE && i == C::BAR && roped) {
                    const int l = fresh_tid() & 63;
                    const auto tbuf = buffer_rsrc(p.rope, (uint32_t)p.rope_rows * 256u);
                    const int* rows_pos = (const int*)(lds + C::POSR);
                    uint32_t toff[TCOPIES ? TCOPIES : 1];
#pragma unroll
                    for (int q = 0; q < TCOPIES; q++) {
                        const int rr = 4 * (w + C::NWAVES * q) + (l >> 4), c = (l & 15) ^ (rr & 15);
                        toff[q] = (uint32_t)rows_pos[rr] * 256u + c * 16;
                    }
#pragma unroll
                    for (int q = 0; q < TCOPIES; q++) lds_bdma16<false>(tbuf, toff[q], st + (w + C::NWAVES * q) * 1024);
                }
                if (LAST && ROPE && i == C::BAR) load_inputs(t, in);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        int s = 0;
        for (; s + 1 < t.nk; s++) body(s, std::false_type{});
        body(s, std::true_type{});
        char* const st = at(pos + s);  // the last stage's space: the RoPE table rows
        mark(2);

        // ---- the epilogue ---------------------------------------------------------------------------
        // This wave's copies of the next task's first stage (its second's may be in flight) and of
        // the RoPE table rows have landed, before the stores go out behind them.
        if (ROPE) wait_vmcnt<0>(); else wait_vmcnt<C::EARLY>();
        put_inputs(in);
        wait_lgkm0();
        if (ROPE || LN) __builtin_amdgcn_s_barrier();
        // Split-K (kernels/src/gemm.rs:355-433), as the latency tile's (finish in gemm_tile.h): every
        // split stores its accumulators to the scratch ([tile][split][float4 v][thread], coherent
        // stores), waits for them, then counts its arrival; the tile's last arriver (which resets
        // the counter) sums every split's partial in split order, so the result does not depend on
        // arrival order, and runs the epilogue.
        bool fin = true;
        if (SPLIT && S > 1) {
            constexpr int NV = MI * NJ;  // float4s a lane
            const int tid = fresh_tid();
            const auto part = buffer_rsrc(p.ws + (size_t)t.t2 * S * NV * C::THREADS * 4, S * NV * C::THREADS * 16);
            const uint32_t mine = (uint32_t)t.z * NV * C::THREADS * 16;
#pragma unroll
            for (int i = 0; i < MI; i++)
#pragma unroll
                for (int j = 0; j < NJ; j++)
                    bstore16f(part, mine + ((i * NJ + j) * C::THREADS + tid) * 16,
                              make_float4(acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]));
            release_wait();
            __syncthreads();
            uint32_t* s_last = (uint32_t*)(lds + C::FLAG);
            if (tid == 0) {
                const uint32_t old = atomic_add_agent(p.counters + t.t2, 1u);
                const uint32_t last = old == (uint32_t)(S - 1);
                if (last) atomic_store_agent(p.counters + t.t2, 0u);
                *s_last = last;
            }
            __syncthreads();
            fin = *s_last != 0;
            if (fin) {
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int j = 0; j < NJ; j++) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
                for (int zz = 0; zz < S; zz++) {
                    const uint32_t src = (uint32_t)zz * NV * C::THREADS * 16;
#pragma unroll
                    for (int i = 0; i < MI; i++)
#pragma unroll
                        for (int j = 0; j < NJ; j++) {
                            const float4 v4 = bload16f(part, src + ((i * NJ + j) * C::THREADS + tid) * 16);
                            acc[i][j][0] += v4.x, acc[i][j][1] += v4.y, acc[i][j][2] += v4.z, acc[i][j][3] += v4.w;
                        }
                }
            }
        }
        if (fin) {
            const int l = fresh_tid() & 63, r16 = l & 15, g4 = l >> 4;
            constexpr int WO = GEGLU ? 32 : 64;                 // output columns of the wave
            constexpr int LPR = WO / 8, RPP = 64 / LPR, NPASS = 16 / RPP;  // lanes a row, rows and passes
            constexpr int PADH = WO + 8;
            const int ncol = GEGLU ? (p.n >> 1) : p.n;
            const int g = (t.bx * BN + wn * 64) >> 6;           // the wave's 64-column group
            const int col0 = g * WO;
            const int row0 = t.by * BM + wm * C::WM;
            // Descriptors over the tile's rows from the wave's first: rows past m read as zeros and
            // are not stored (the range check drops them).
            const int rows = __builtin_amdgcn_readfirstlane(max(0, min(p.m - row0, C::WM)));
            const auto cbuf = buffer_rsrc((f16*)p.c + (size_t)min(row0, p.m) * ncol, (uint32_t)rows * ncol * 2u);
            [[maybe_unused]] const auto rbuf = buffer_rsrc((const f16*)(RES && p.res ? p.res : p.c) + (size_t)min(row0, p.m) * ncol,
                                                           (uint32_t)rows * ncol * 2u);
            [[maybe_unused]] const auto obuf = buffer_rsrc(p.stats_out + (size_t)min(row0, p.m) * (p.n >> 6) * 2,
                                                           (uint32_t)rows * (p.n >> 6) * 8u);
            f16* const sgh = (f16*)(lds + C::STAGING) + w * 16 * C::PADH;
            const float2* rows_ms = (const float2*)(lds + C::ROWS) + wm * C::WM + r16;
            const int cl = 8 * (l % LPR), rl0 = l / LPR;
            const uint32_t vo = (uint32_t)(rl0 * ncol + col0 + cl) * 2u, rstep = (uint32_t)ncol * 2u;
            // The residual in rows of 16 bytes a lane, all of it before the first store (it goes
            // through the staging into the accumulators' layout; loading it there as 8-byte pieces
            // asked for every line four times: 19.3 against 16.5 us for wo at 4096 rows, 160-row tiles).
            half8 rin[RES ? MI : 1][NPASS];
            if (RES) {
#pragma unroll
                for (int i = 0; i < MI; i++)
#pragma unroll
                    for (int ps = 0; ps < NPASS; ps++) rin[i][ps] = bload16<false>(rbuf, vo + (16 * i + ps * RPP) * rstep);
            }
            float4 cs[NJ], bs[NJ];
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                if (LN) cs[j] = *(const float4*)(wcols + 16 * j + 4 * g4);
                if (BIAS) bs[j] = *(const float4*)(wcols + 64 + 16 * j + 4 * g4);
            }
            // 16 rows at a time: the column-wise part (LayerNorm, bias, ReLU / GELU, RoPE, GeGLU) on
            // the accumulators, where a lane holds the RoPE and GeGLU pairs (x, x + 32); the residual;
            // f16 through the wave's own LDS rows (LDS operations of one wave complete in order) into
            // 8 consecutive columns a lane for the output statistics (8 lanes a 64-column group) and
            // 16-byte stores.
            auto rows16 = [&](auto roped_) {
                constexpr bool ROPED = decltype(roped_)::value;
#pragma unroll
                for (int i = 0; i < MI; i++) {
                    __builtin_amdgcn_sched_barrier(0);
                    float v[NJ][4];  // row 16 i + r16, columns 16 j + 4 g4 + e of the wave's block
                    float4 tt[2][2];
                    if (ROPED) {
                        const int tr = wm * C::WM + 16 * i + r16;
                        const char* trow = st + tr * 256;
#pragma unroll
                        for (int j = 0; j < 2; j++) {
                            const int ca = 8 * j + 2 * g4;  // dimensions 16 j + 4 g4 .. + 3
                            tt[j][0] = *(const float4*)(trow + ((ca ^ r16) << 4));
                            tt[j][1] = *(const float4*)(trow + (((ca + 1) ^ r16) << 4));
                        }
                    }
#pragma unroll
                    for (int j = 0; j < NJ; j++)
#pragma unroll
                        for (int e = 0; e < 4; e++) v[j][e] = acc[i][j][e];
                    if (LN) {
                        const float2 ms = rows_ms[16 * i];
#pragma unroll
                        for (int j = 0; j < NJ; j++) {
                            const float cc[4] = {cs[j].x, cs[j].y, cs[j].z, cs[j].w};
#pragma unroll
                            for (int e = 0; e < 4; e++) v[j][e] = ms.y * (v[j][e] - ms.x * cc[e]);
                        }
                    }
                    if (BIAS) {
#pragma unroll
                        for (int j = 0; j < NJ; j++) {
                            const float bb[4] = {bs[j].x, bs[j].y, bs[j].z, bs[j].w};
#pragma unroll
                            for (int e = 0; e < 4; e++) v[j][e] += bb[e];
                        }
                    }
                    if (EPI & EPI_RELU) {
#pragma unroll
                        for (int j = 0; j < NJ; j++)
#pragma unroll
                            for (int e = 0; e < 4; e++) v[j][e] = fmaxf(v[j][e], 0.0f);
                    }
                    if (EPI & EPI_GELU) {
#pragma unroll
                        for (int j = 0; j < NJ; j++)
#pragma unroll
                            for (int e = 0; e < 4; e++) v[j][e] = gelu(v[j][e]);
                    }
                    if (ROPED) {
#pragma unroll
                        for (int j = 0; j < 2; j++) {
                            const float4 t0 = tt[j][0], t1 = tt[j][1];
                            const float co[4] = {t0.x, t0.z, t1.x, t1.z}, sn_[4] = {t0.y, t0.w, t1.y, t1.w};
#pragma unroll
                            for (int e = 0; e < 4; e++) {
                                const float x1 = v[j][e], x2 = v[j + 2][e];
                                v[j][e] = x1 * co[e] - x2 * sn_[e];
                                v[j + 2][e] = x2 * co[e] + x1 * sn_[e];
                            }
                        }
                    }
                    if (GEGLU) {
#pragma unroll
                        for (int j = 0; j < 2; j++) {
                            half4 o;
#pragma unroll
                            for (int e = 0; e < 4; e++) o[e] = (f16)(gelu(v[j][e]) * v[j + 2][e]);
                            *(half4*)(sgh + r16 * PADH + 16 * j + 4 * g4) = o;
                        }
                    } else {
                        if (RES) {
#pragma unroll
                            for (int ps = 0; ps < NPASS; ps++) *(half8*)(sgh + (ps * RPP + rl0) * PADH + cl) = rin[i][ps];
#pragma unroll
                            for (int j = 0; j < NJ; j++) {
                                const half4 x = *(const half4*)(sgh + r16 * PADH + 16 * j + 4 * g4);
#pragma unroll
                                for (int e = 0; e < 4; e++) v[j][e] += (float)x[e];
                            }
                        }
#pragma unroll
                        for (int j = 0; j < NJ; j++) {
                            half4 o;
#pragma unroll
                            for (int e = 0; e < 4; e++) o[e] = (f16)v[j][e];
                            *(half4*)(sgh + r16 * PADH + 16 * j + 4 * g4) = o;
                        }
                    }
#pragma unroll
                    for (int ps = 0; ps < NPASS; ps++) {
                        const int rl = ps * RPP + rl0;
                        const half8 o = *(const half8*)(sgh + rl * PADH + cl);
                        bstore16<true>(cbuf, vo + (16 * i + ps * RPP) * rstep, o);
                        if (EPI & EPI_STATS) {
                            float a = 0.0f, b = 0.0f;
#pragma unroll
                            for (int e = 0; e < 8; e++) {
                                const float x = (float)o[e];
                                a += x, b += x * x;
                            }
                            a = group_sum<8>(a);
                            b = group_sum<8>(b);
                            if ((l & 7) == 0)
                                bstore8(obuf, (uint32_t)((16 * i + rl) * (p.n >> 6) + g) * 8u, make_float2(a, b));
                        }
                    }
                }
            };
            if (ROPE && roped) rows16(std::integral_constant<bool, ROPE>{});
            else rows16(std::false_type{});
        }
        if (task == first) mark(3);
        if (!more) break;
        wait_lgkm0();
        __builtin_amdgcn_s_barrier();
        task += stride;
        pos += t.nk;
        t = tn;
        sub = nullptr;
    }
    wait_lgkm0();
    __builtin_amdgcn_s_barrier();
}

}  // namespace jh
