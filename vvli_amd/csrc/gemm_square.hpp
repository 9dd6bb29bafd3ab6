// gemm_square.hpp -- the 128 x 128 tile of the prefill GEMM, for launches whose
// larger tiles would leave CUs idle (included by prefill.hip, which holds the
// shared pieces).
#pragma once

// One block of 8 waves per CU: 2 over rows x 2 over columns (64 x 64 per wave,
// 4 x 4 MFMA tiles) x 2 over the K steps of 32 in a stage of 64; the two K
// halves meet in LDS at the end, each half finishing half of the rows.
//
// Why this split: waves of 64 x 64 move the fewest fragments a product
// (48 KiB out of LDS and 24 into it for 512 cycles of MFMA per SIMD, as much
// per product as the 128 x 256 tile), and the K halves keep two waves on each
// SIMD, which four waves alone (one per SIMD) do not. Counters: matrix cores
// busy 31 % of the cycles at 512 x 8192 x 2048 (one round of tiles: 43 us, 791
// TFLOP/s with hi and lo), 42 % at 2048 x 2048 x 8192 and x 2048; no bank
// conflicts.
//
// Stage (48 KiB): [A hi 16 KiB | A lo 16 KiB | W 16 KiB], rows of 128 bytes,
// 16-byte chunk c of row r at position c ^ (r & 7); three stages. A stage's
// fragments are read during the step before, so its slot is refilled one
// barrier later with the stage three on.
constexpr int kSqM = 128, kSqN = 128, kSqK = 64;
constexpr int kSqOp = kSqM * kSqK * 2;  // bytes of one plane tile (A hi, A lo or W)
constexpr int kSqStage = 3 * kSqOp;
constexpr int kSqLds = 3 * kSqStage;
constexpr int kSqDma = kSqStage / 1024 / (kGemmThreads / 64);  // 1 KiB copies per wave per stage
static_assert(kSqDma == 6, "the waits count stages of 6 copies");
static_assert(kSqOp + 3 * 2048 < 65536 && 8 * 8 * 1024 <= kSqLds, "fragment offsets and the exchange fit");

template <int MODE>
__device__ __forceinline__ void square_store(const GemmArgs& g, const f32x4 (&acc)[2][4], uint32_t row0, uint32_t n0,
                                             uint32_t wn, int lane) {
    const uint32_t fr = lane & 15, rq = 4 * (static_cast<uint32_t>(lane) >> 4);
    const bool split = gridDim.z > 1;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int jr = 0; jr < 4; ++jr) {
            const uint32_t row = row0 + i * 16 + rq + jr;
            if (row >= g.M) continue;
            float* orow = g.out + static_cast<size_t>(row) * g.ldo;
            if (MODE == kGemmGateUp) {
#pragma unroll
                for (int j = 0; j < 4; j += 2) {
                    const uint32_t n = n0 / 2 + (wn * 2 + j / 2) * 16 + fr;
                    if (g.out_hl) {
                        const uint32_t kpo = gemm_kp(g.N);
                        if (n >= kpo) continue;
                        const float v = n < g.N ? silu_mul(acc[i][j][jr], acc[i][j + 1][jr]) : 0.f;
                        const uint16_t h = to_bf16_rne(v);
                        uint16_t* o = g.out_hl + static_cast<size_t>(row) * kpo + n;
                        o[0] = h;
                        o[g.out_plane] = to_bf16_rne(v - from_bf16(h));
                    } else if (n < g.N) {
                        orow[n] = silu_mul(acc[i][j][jr], acc[i][j + 1][jr]);
                    }
                }
                continue;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t n = n0 + wn * 64 + j * 16 + fr;
                if (n >= g.N) continue;
                float v = acc[i][j][jr];
                if (MODE == kGemmPlain && blockIdx.z == 0) {
                    const uint16_t* b = n < g.seg_end[0] ? g.bias[0] : n < g.seg_end[1] ? g.bias[1] : g.bias[2];
                    const uint32_t bi = n < g.seg_end[0] ? n : n < g.seg_end[1] ? n - g.seg_end[0] : n - g.seg_end[1];
                    if (b) v = __fadd_rn(v, from_bf16(b[bi]));
                }
                if (split) part_row(g, row)[n] = v;
                else orow[n] = MODE == kGemmResid ? __fadd_rn(orow[n], v) : v;  // addInto (src/llm.zig:1389-1396)
            }
        }
    }
}

template <int MODE>
__global__ __launch_bounds__(kGemmThreads) void gemm_square_kernel(GemmArgs g) {
    extern __shared__ __attribute__((aligned(1024))) char gemm_smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = (wave >> 1) & 1, wk = wave >> 2;
    const uint32_t cols = MODE == kGemmGateUp ? 2 * g.N : g.N;
    const uint32_t tn = (cols + kSqN - 1) / kSqN, tm = (g.M + kSqM - 1) / kSqM;
    uint32_t m0, n0;
    {  // the XCD-aware order of the 128 x 256 tile
        const uint32_t ntile = gridDim.x;
        const uint32_t xcd = blockIdx.x % 8, per = ntile / 8, rem = ntile % 8;
        const uint32_t u = xcd * per + min(xcd, rem) + blockIdx.x / 8;
        const uint32_t panel = u / (tm * 8), pw = min(8u, tn - 8 * panel), within = u - panel * tm * 8;
        m0 = (within / pw) * kSqM;
        n0 = (8 * panel + within % pw) * kSqN;
    }
    const uint32_t nk_all = (g.K + kSqK - 1) / kSqK, per_split = (nk_all + gridDim.z - 1) / gridDim.z;
    const uint32_t kt0 = blockIdx.z * per_split;
    const int nk = kt0 < nk_all ? static_cast<int>(min(per_split, nk_all - kt0)) : 0;
    if (nk == 0) return;  // uniform (the launcher gives every split K steps)

    // Copies: wave w fetches rows 16w .. 16w + 15 of A hi, A lo and W, 8 rows a
    // copy; lane l row l / 8, chunk (l & 7) ^ (l / 8). Rows past M or N read
    // row 0 (never written), lanes past K zeros.
    const uint16_t* zeros = slab_zeros;
    // Held in registers: fetched before every copy, its wait drained the
    // fragment reads (512 x 8192 x 2048 with its split pass, on a box 10 % slower
    // than others, 49.9 -> 48.9 us).
    asm volatile("" : "+s"(zeros));
    const uint32_t kp = gemm_kp(g.K);
    const size_t plane = g.a_plane ? g.a_plane : static_cast<size_t>(g.M) * kp;
    const uint32_t chunk = ((static_cast<uint32_t>(lane) & 7u) ^ (static_cast<uint32_t>(lane) >> 3)) * 8;
    const uint16_t *srcA[2], *srcW[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t row = wave * 16 + i * 8 + lane / 8;
        srcA[i] = g.a_hl + static_cast<size_t>(m0 + row < g.M ? m0 + row : 0) * kp + chunk;
        bool valid;
        srcW[i] = gemm_w_row<MODE>(g, n0, static_cast<int>(row), 0, valid) + chunk;
    }
    auto issue_one = [&](int kt, int c) {  // c: 0, 1 A hi; 2, 3 A lo; 4, 5 W
        const uint32_t k = (kt0 + kt) * kSqK;
        char* dst = gemm_smem + kt % 3 * kSqStage + (c >> 1) * kSqOp + (wave * 2 + (c & 1)) * 1024;
        const uint16_t* p = c < 4 ? srcA[c & 1] + (c >= 2 ? plane : 0) + k : srcW[c & 1] + k;
        gemm_dma16(k + chunk < g.K ? p : zeros, dst);
    };
    const uint32_t lds0 = gemm_lds_addr(gemm_smem);
    const uint32_t fpos = (lane & 15) * 128 + (((wk * 4 + (static_cast<uint32_t>(lane) >> 4)) ^ (lane & 7u)) << 4);
    const uint32_t fa = lds0 + wm * 64 * 128 + fpos, fb = lds0 + 2 * kSqOp + wn * 64 * 128 + fpos;
    f32x4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 fh[2][4], fl[2][4], fw[2][4];
    constexpr int kKeep = (7 << 4) | (15 << 8);  // expcnt, lgkmcnt: no wait
#define SQ_READ(x, q, so)                                  \
    fh[x][q] = wide_lds_read<(q) * 2048>(fa + (so)),       \
    fl[x][q] = wide_lds_read<kSqOp + (q) * 2048>(fa + (so)), \
    fw[x][q] = wide_lds_read<(q) * 2048>(fb + (so))
    for (int s0 = 0; s0 < 3; ++s0)
        if (s0 < nk)
#pragma unroll
            for (int c = 0; c < kSqDma; ++c) issue_one(s0, c);
    if (nk > 2) __builtin_amdgcn_s_waitcnt(12 | kKeep);
    else if (nk > 1) __builtin_amdgcn_s_waitcnt(6 | kKeep);
    else __builtin_amdgcn_s_waitcnt(0 | kKeep);
    gemm_barrier();
    SQ_READ(0, 0, 0), SQ_READ(0, 1, 0), SQ_READ(0, 2, 0), SQ_READ(0, 3, 0);
    gemm_lds_wait(fh[0], fl[0], fw[0]);
    // Step kt: stage kt + 1 has landed and every wave holds stage kt's
    // fragments, so its slot takes stage kt + 3 while stage kt + 1's fragments
    // are read, between four groups of 8 products.
    auto step = [&](int kt, const int cur) {
        const bool next = kt + 1 < nk, more = kt + 3 < nk;
        if (next) {
            if (kt + 2 < nk) __builtin_amdgcn_s_waitcnt(6 | kKeep);
            else __builtin_amdgcn_s_waitcnt(0 | kKeep);
        }
        gemm_barrier();
        const uint32_t so = (kt + 1) % 3 * kSqStage;
#define SQ_GROUP(q, frag)                                                                                          \
    _Pragma("unroll") for (int i = ((q)&1) * 2; i < ((q)&1) * 2 + 2; ++i) _Pragma("unroll") for (int j = 0; j < 4; ++j) \
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag[cur][i], fw[cur][j], acc[i][j], 0, 0, 0);         \
    __builtin_amdgcn_sched_barrier(0);                                                                             \
    if (next) { SQ_READ(cur ^ 1, q, so); }                                                                         \
    if (more) {                                                                                                    \
        issue_one(kt + 3, q);                                                                                      \
        if ((q) >= 2) issue_one(kt + 3, (q) + 2);                                                                  \
    }                                                                                                              \
    __builtin_amdgcn_sched_barrier(0)
        SQ_GROUP(0, fh);
        SQ_GROUP(1, fh);
        SQ_GROUP(2, fl);
        SQ_GROUP(3, fl);
        if (next) gemm_lds_wait(fh[cur ^ 1], fl[cur ^ 1], fw[cur ^ 1]);
    };
    for (int kt = 0; kt < nk; kt += 2) {
        step(kt, 0);
        if (kt + 1 < nk) step(kt + 1, 1);
    }
#undef SQ_GROUP
#undef SQ_READ
    // The K halves trade sums: half 0 finishes rows 0-31 of the wave tile,
    // half 1 rows 32-63.
    f32x4* xs = reinterpret_cast<f32x4*>(gemm_smem) + lane;
    const int tile = wave & 3;
    __syncthreads();  // all fragments are read
    auto finish = [&](const int keep) {
        const int give = 2 - keep;  // first row tile of the other half's rows
#pragma unroll
        for (int t = 0; t < 8; ++t) xs[((wk * 4 + tile) * 8 + t) * 64] = acc[give + t / 4][t % 4];
        __syncthreads();
        f32x4 r[2][4];
#pragma unroll
        for (int t = 0; t < 8; ++t) r[t / 4][t % 4] = acc[keep + t / 4][t % 4] + xs[(((wk ^ 1) * 4 + tile) * 8 + t) * 64];
        square_store<MODE>(g, r, m0 + wm * 64 + keep * 16, n0, wn, lane);
    };
    if (wk == 0) finish(0);
    else finish(2);
}
