// gemm_wide.hpp -- the 256 x 256 tile of the prefill GEMM (included by
// prefill.hip, which holds the shared pieces and the 128 x 256 tile).
#pragma once

// One block of 8 waves (4 over rows x 2 over columns, 64 x 128 per wave: 4 x 8
// MFMA tiles of 16 x 16) per CU, K steps of 32, no K split.
//
// Why this tile: at 128 x 256 a K step moves 96 KiB of fragments out of LDS
// and 32 KiB into it for 1024 cycles of MFMA per SIMD. Here it is 128 + 48 KiB
// for 2048 cycles: two thirds of it, and 27 % less copied per product. Two waves
// per SIMD stay (128 accumulators + 96 fragment registers + addresses: 251 of
// 256), since one wave per SIMD hides too little of the LDS latency.
// Measured (gate/up at 2048 rows of 2048 x 8192, split activations counted
// twice): 264 -> 217 us, 1040 -> 1265 TFLOP/s on the matrix cores; a large
// bf16 product of the library's reaches 1347 on the same card. Counters there:
// matrix cores busy 59 % of the cycles (43 % on 128 x 256), no bank conflicts,
// the clock at 2.1 GHz where lighter kernels run at 2.4.
//
// Stage (48 KiB): [A hi 16 KiB | A lo 16 KiB | W 16 KiB], rows of 64 bytes
// swizzled as in the 128 x 256 tile; three stages (144 KiB). A wave holds all
// A fragments of a step and half of its W fragments: during the first half of
// the products the other W fragments arrive, during the second half the next
// step's A (second register set) and first W fragments. The stage a step read
// is free once every wave has its second W half, so the one barrier sits
// between the halves and the copies of step kt + 3 follow it.
constexpr int kWM = 256, kWN = 256;
constexpr int kWideOp = kWM * kBK * 2;  // bytes of one plane tile (A hi, A lo or W)
constexpr int kWideStage = 3 * kWideOp;
constexpr int kWideStages = 3;
constexpr int kWideLds = kWideStages * kWideStage;
constexpr int kWideDma = kWideStage / 1024 / (kGemmThreads / 64);  // 1 KiB copies per wave per stage
static_assert(kWideDma == 6, "wide_wait_vm counts in stages of 6 copies");

template <int OFF>
__device__ __forceinline__ bf16x8 wide_lds_read(uint32_t addr) {
    bf16x8 v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(v) : "v"(addr), "n"(OFF));
    return v;
}
__device__ __forceinline__ void wide_wait4(bf16x8 (&a)[4]) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]));
}

template <int MODE>
__global__ __launch_bounds__(kGemmThreads) void gemm_wide_kernel(GemmArgs g) {
    extern __shared__ __attribute__((aligned(1024))) char gemm_smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const uint32_t cols = MODE == kGemmGateUp ? 2 * g.N : g.N;
    const uint32_t tn = (cols + kWN - 1) / kWN;
    uint32_t m0, n0;
    {
        const uint32_t tm = (g.M + kWM - 1) / kWM;
        const uint32_t ntile = gridDim.x;
        const uint32_t xcd = blockIdx.x % 8, per = ntile / 8, rem = ntile % 8;
        const uint32_t u = xcd * per + min(xcd, rem) + blockIdx.x / 8;
        const uint32_t panel = u / (tm * 8), pw = min(8u, tn - 8 * panel), within = u - panel * tm * 8;
        m0 = (within / pw) * kWM;
        n0 = (8 * panel + within % pw) * kWN;
    }
    const int nk = static_cast<int>((g.K + kBK - 1) / kBK);

    f32x4 acc[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Copies: wave w issues the 1 KiB copies of 16-row groups 2w and 2w + 1 of
    // A hi, A lo and W; lane l fetches row 16 grp + l/4, chunk (l & 3) ^ swz.
    // Rows past M or N read row 0 (their outputs are never written); past K, A
    // reads its zero tail and W 8 zeros of that tail.
    const uint32_t kp = gemm_kp(g.K);
    const uint16_t* zeros = g.a_hl + (kp - 8);
    const size_t plane = g.a_plane ? g.a_plane : static_cast<size_t>(g.M) * kp;
    const uint16_t *srcA[2], *srcW[2];
    const uint32_t chunk = (static_cast<uint32_t>(lane & 3) ^ gemm_swz(lane / 4)) * 8;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t row = (wave * 2 + i) * 16 + lane / 4;
        const uint32_t gm = m0 + row < g.M ? m0 + row : 0;
        srcA[i] = g.a_hl + static_cast<size_t>(gm) * kp + chunk;
        bool valid;
        srcW[i] = gemm_w_row<MODE>(g, n0, static_cast<int>(row), 0, valid) + chunk;
    }
    auto issue_one = [&](int kt, uint32_t so, int c) {  // c: 0, 1 A hi; 2, 3 A lo; 4, 5 W
        const uint32_t k = kt * kBK;
        char* dst = gemm_smem + so + (c >> 1) * kWideOp + (wave * 2 + (c & 1)) * 1024;
        if (c < 4) gemm_dma16(srcA[c & 1] + (c >= 2 ? plane : 0) + k, dst);
        else gemm_dma16(k + chunk >= g.K ? zeros : srcW[c & 1] + k, dst);
    };
    auto issue = [&](int kt, uint32_t so) {
#pragma unroll
        for (int c = 0; c < kWideDma; ++c) issue_one(kt, so, c);
    };
    const uint32_t lds0 = gemm_lds_addr(gemm_smem);
    const uint32_t fpos = (lane & 15) * 64 + (((static_cast<uint32_t>(lane) >> 4) ^ gemm_swz(lane & 15)) << 4);
    const uint32_t fa = lds0 + wm * 64 * 64 + fpos, fb = lds0 + 2 * kWideOp + wn * 128 * 64 + fpos;
    bf16x8 ah[2][4], al[2][4], w0[4], w1[4];

#define WIDE_READ4(dst, base, off)                                                       \
    dst[0] = wide_lds_read<(off)>(base), dst[1] = wide_lds_read<(off) + 1024>(base),      \
    dst[2] = wide_lds_read<(off) + 2048>(base), dst[3] = wide_lds_read<(off) + 3072>(base)

    auto wait_vm = [&](bool one_more) {
        constexpr int kKeep = (7 << 4) | (15 << 8);
        if (one_more) __builtin_amdgcn_s_waitcnt(6 | kKeep);
        else __builtin_amdgcn_s_waitcnt(0 | kKeep);
    };
    for (int s0 = 0; s0 < kWideStages; ++s0)
        if (s0 < nk) issue(s0, s0 * kWideStage);
    if (nk > 2) __builtin_amdgcn_s_waitcnt(12 | (7 << 4) | (15 << 8));
    else wait_vm(nk > 1);
    gemm_barrier();
    WIDE_READ4(ah[0], fa, 0);
    WIDE_READ4(al[0], fa, kWideOp);
    WIDE_READ4(w0, fb, 0);
    wide_wait4(ah[0]);
    wide_wait4(al[0]);
    wide_wait4(w0);

#define WIDE_MFMA(frag, i, wf, jo)                                                                              \
    _Pragma("unroll") for (int j = 0; j < 4; ++j) acc[i][jo + j] =                                              \
        __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag[i], wf[j], acc[i][jo + j], 0, 0, 0)

    uint32_t so = 0;  // stage of step kt
    auto step = [&](int kt, const int cur) {
        const bool next = kt + 1 < nk, more = kt + kWideStages < nk;
        const uint32_t sn = so + kWideStage == kWideLds ? 0 : so + kWideStage;
        const uint32_t fbs = fb + so;
        // First half: columns 0-63 of the wave; the second half's W fragments arrive.
        WIDE_MFMA(ah[cur], 0, w0, 0);
        __builtin_amdgcn_sched_barrier(0);
        WIDE_READ4(w1, fbs, 4096);
        __builtin_amdgcn_sched_barrier(0);
        WIDE_MFMA(ah[cur], 1, w0, 0);
        WIDE_MFMA(ah[cur], 2, w0, 0);
        WIDE_MFMA(ah[cur], 3, w0, 0);
        WIDE_MFMA(al[cur], 0, w0, 0);
        WIDE_MFMA(al[cur], 1, w0, 0);
        __builtin_amdgcn_sched_barrier(0);
        wide_wait4(w1);
        if (next) wait_vm(kt + 2 < nk);
        gemm_barrier();
        __builtin_amdgcn_sched_barrier(0);
        WIDE_MFMA(al[cur], 2, w0, 0);
        WIDE_MFMA(al[cur], 3, w0, 0);
        __builtin_amdgcn_sched_barrier(0);
        // Second half: the next step's A and first W fragments, and the copies
        // of step kt + 3 into the stage just read.
        const uint32_t fan = fa + sn, fbn = fb + sn;
        WIDE_MFMA(ah[cur], 0, w1, 4);
        __builtin_amdgcn_sched_barrier(0);
        if (next) { WIDE_READ4(ah[cur ^ 1], fan, 0); }
        if (more) issue_one(kt + kWideStages, so, 0), issue_one(kt + kWideStages, so, 1);
        __builtin_amdgcn_sched_barrier(0);
        WIDE_MFMA(ah[cur], 1, w1, 4);
        WIDE_MFMA(ah[cur], 2, w1, 4);
        __builtin_amdgcn_sched_barrier(0);
        if (next) { WIDE_READ4(w0, fbn, 0); }
        if (more) issue_one(kt + kWideStages, so, 2), issue_one(kt + kWideStages, so, 3);
        __builtin_amdgcn_sched_barrier(0);
        WIDE_MFMA(ah[cur], 3, w1, 4);
        WIDE_MFMA(al[cur], 0, w1, 4);
        __builtin_amdgcn_sched_barrier(0);
        if (next) { WIDE_READ4(al[cur ^ 1], fan, kWideOp); }
        if (more) issue_one(kt + kWideStages, so, 4), issue_one(kt + kWideStages, so, 5);
        __builtin_amdgcn_sched_barrier(0);
        WIDE_MFMA(al[cur], 1, w1, 4);
        WIDE_MFMA(al[cur], 2, w1, 4);
        WIDE_MFMA(al[cur], 3, w1, 4);
        __builtin_amdgcn_sched_barrier(0);
        if (next) {
            wide_wait4(ah[cur ^ 1]);
            wide_wait4(w0);
            wide_wait4(al[cur ^ 1]);
        }
        so = sn;
    };
    for (int kt = 0; kt < nk; kt += 2) {
        step(kt, 0);
        if (kt + 1 < nk) step(kt + 1, 1);
    }
#undef WIDE_MFMA
#undef WIDE_READ4

    const int fr = lane & 15, rq = 4 * (lane >> 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int jr = 0; jr < 4; ++jr) {
            const uint32_t row = m0 + wm * 64 + i * 16 + rq + jr;
            if (row >= g.M) continue;
            float* orow = g.out + static_cast<size_t>(row) * g.ldo;
            if (MODE == kGemmGateUp) {
#pragma unroll
                for (int j = 0; j < 8; j += 2) {
                    const uint32_t n = n0 / 2 + (wn * 4 + j / 2) * 16 + fr;
                    if (g.out_hl) {
                        const uint32_t kpo = gemm_kp(g.N);
                        if (n < kpo) {
                            const float v = n < g.N ? silu_mul(acc[i][j][jr], acc[i][j + 1][jr]) : 0.f;
                            const uint16_t h = to_bf16_rne(v);
                            uint16_t* o = g.out_hl + static_cast<size_t>(row) * kpo + n;
                            o[0] = h;
                            o[g.out_plane] = to_bf16_rne(v - from_bf16(h));
                        }
                    } else if (n < g.N) {
                        orow[n] = silu_mul(acc[i][j][jr], acc[i][j + 1][jr]);
                    }
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const uint32_t n = n0 + wn * 128 + j * 16 + fr;
                    if (n >= g.N) continue;
                    float v = acc[i][j][jr];
                    if (MODE == kGemmResid) {
                        orow[n] = __fadd_rn(orow[n], v);
                    } else {
                        const uint16_t* b = n < g.seg_end[0] ? g.bias[0] : n < g.seg_end[1] ? g.bias[1] : g.bias[2];
                        if (b) {
                            const uint32_t bi = n < g.seg_end[0] ? n : n < g.seg_end[1] ? n - g.seg_end[0]
                                                                                        : n - g.seg_end[1];
                            v = __fadd_rn(v, from_bf16(b[bi]));
                        }
                        orow[n] = v;
                    }
                }
            }
        }
    }
}
