// gemm_slab.hpp -- the prefill / linear GEMM for few rows (M <= 128), bound by
// the W stream (included by prefill.hip, which holds the shared pieces).
#pragma once

// A work item is 64 rows of W times a K range (a split) for all MT * 16 rows
// of A. Blocks of 8 waves, one per CU, take items grid-stride and stream them
// in K chunks of KC through ST stages [A | W 64 x KC]; the chunk stream runs on
// across items, so the copies never drain between two items. A: the hi and lo
// planes (MT * 16 rows of KC bf16 each), or with F32A the f32 rows
// themselves (the same bytes), split into hi / lo in registers as they are
// read. Every copy of a row is KC * 2 (F32A: KC * 4) contiguous bytes; 16-byte
// chunk c of row r sits at position c ^ (r & 15) (128-byte rows: c ^ (r & 7)),
// conflict-free for the fragment reads. W is read once and past the caches
// (nontemporal: 128256 x 2048 at 16 rows 109 -> 100 us); an item's chunks are
// taken from a start that differs from block to block, since all blocks
// reading the same columns of rows a power of two apart meet in few memory
// channels (100 -> 96 us, at 5 rows 92 -> 84, the rate of the one-row GEMV).
// Waves: WM over rows x WN over columns x WK over the K steps of a chunk; the
// WK partial sums meet in LDS in order. One wave column (WN = 1) splits each
// f32 fragment once: 128256 x 2048 at 64 rows 176 -> 157 us.
// What bounds it (variants that leave out one side, 128256 x 2048): at 16 rows
// the W stream (89 us, without A traffic 86, without products 87); at 64 rows
// the work per chunk (157 us; the products and the split alone cost 37).
constexpr int kSlabN = 64;
constexpr int kSlabThreads = 512;
constexpr int kSlabCpolNt = 2;  // cache policy of the W copies: nontemporal

template <int MT, int KC, int ST, int WM, int WN>
struct SlabShape {
    static constexpr int WK = 8 / (WM * WN);
    static constexpr int ABytes = MT * 16 * KC * 4;  // hi + lo planes, or f32 rows
    static constexpr int WBytes = kSlabN * KC * 2;
    static constexpr int Stage = ABytes + WBytes;
    static constexpr int Dma = Stage / 1024 / 8;  // 1 KiB copies per wave per chunk
    static constexpr int Red = (WK - 1) * MT * 16 * kSlabN * 4;
    static constexpr int Lds = ST * Stage + Red;
    static_assert(Stage % 8192 == 0 && Lds <= 160 * 1024, "stages fit");
    static_assert((KC / 32) % WK == 0, "whole K steps per wave");
};

__device__ __align__(16) uint16_t slab_zeros[8];  // what lanes past K copy

template <int OFF = 0>
__device__ __forceinline__ f32x4 slab_read(uint32_t addr) {
    f32x4 v;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(v) : "v"(addr), "n"(OFF));
    return v;
}
__device__ __forceinline__ void slab_write(uint32_t addr, f32x4 v) {
    asm volatile("ds_write_b128 %0, %1" : : "v"(addr), "v"(v));
}
// Nothing that uses v can be scheduled before the wait in front of this.
template <int N>
__device__ __forceinline__ void slab_tie(f32x4 (&v)[N]) {
#pragma unroll
    for (int i = 0; i < N; ++i) asm volatile("" : "+v"(v[i]));
}
template <int N>
__device__ __forceinline__ void slab_wait(f32x4 (&v)[N]) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::);
    slab_tie(v);
}

// Two f32 quads -> hi = bf16(x), lo = bf16(x - hi), round to nearest even.
__device__ __forceinline__ void slab_split(f32x4 a, f32x4 b, bf16x8& hi, bf16x8& lo) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float x = e < 4 ? a[e] : b[e - 4];
        const __bf16 h = static_cast<__bf16>(x);
        hi[e] = h;
        lo[e] = static_cast<__bf16>(x - static_cast<float>(h));
    }
}

// Grouped launches (rows of a mixture's experts): an item is 64 rows of an
// expert's W for one entry of the tile table, columns fastest, so that the
// blocks stream one expert after another. The table moves to LDS at the start:
// read from memory, an entry would wait behind the copies in flight.
constexpr uint32_t kSlabTable = 512;  // entries of 8 bytes: first row; expert, rows

template <int MODE, int MT, int KC, int ST, int WM, int WN, bool F32A, bool GROUPED>
__global__ __launch_bounds__(kSlabThreads) void gemm_slab_kernel(GemmArgs g, uint32_t tiles, uint32_t splits) {
    using S = SlabShape<MT, KC, ST, WM, WN>;
    constexpr int WK = S::WK, MW = MT / WM, NW = 4 / WN;  // MFMA tiles of a wave: MW x NW
    constexpr int Steps = KC / 32 / WK;           // K steps of a wave per chunk
    constexpr int ARow = F32A ? KC * 4 : KC * 2;  // bytes of an A row in LDS
    constexpr int ALanes = ARow / 16, WLanes = KC * 2 / 16;
    constexpr int ACopies = S::ABytes / 1024, WCopies = S::WBytes / 1024;
    constexpr int PA = ACopies / 8, PW = WCopies / 8;  // copies of a wave
    static_assert(ACopies % 8 == 0 && WCopies % 8 == 0 && PA + PW == S::Dma, "whole copies per wave");
    extern __shared__ __attribute__((aligned(1024))) char gemm_smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wave % WN, wm = wave / WN % WM, wk = wave / (WN * WM);
    uint32_t items = tiles * splits;
    const uint32_t table = gemm_lds_addr(gemm_smem) + S::Lds;
    if (GROUPED) {
        const uint32_t count = min(g.tiles[0].x, kSlabTable);
        uint2* tab = reinterpret_cast<uint2*>(gemm_smem + S::Lds);
        for (uint32_t t = tid; t < count; t += kSlabThreads) {
            const uint4 td = g.tiles[1 + t];
            tab[t] = make_uint2(td.y, td.x << 16 | (td.z - td.y));
        }
        items = tiles * static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(count));
        __syncthreads();
    }
    // Item i of a grouped launch: first row, rows, expert.
    struct Group {
        uint32_t m0, rows, expert;
    };
    auto group = [&](uint32_t i) {
        if (!GROUPED) return Group{0, g.M, 0};
        vvli_u32x2 v;
        asm volatile("ds_read_b64 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=&v"(v) : "v"(table + i / tiles * 8));
        const uint32_t y = __builtin_amdgcn_readfirstlane(v.y);
        return Group{static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(v.x)), y & 0xffffu, y >> 16};
    };
    const uint32_t nch = (g.K + KC - 1) / KC, per = (nch + splits - 1) / splits;
    const uint32_t kp = gemm_kp(g.K);
    const size_t plane = g.a_plane ? g.a_plane : static_cast<size_t>(g.M) * kp;

    // Copy sources. A: the 16-byte chunk of each copy is fixed, the row too
    // unless the launch is grouped.
    const char* srcA[PA];
    uint32_t kA[PA];
    auto set_a = [&](uint32_t m0, uint32_t rows) {
#pragma unroll
    for (int i = 0; i < PA; ++i) {
        constexpr int Rows = 64 / ALanes;  // rows per copy
        const uint32_t q = wave * PA + i;
        const uint32_t lr = q * Rows + lane / ALanes;  // row within the A stage (planes: hi rows, then lo rows)
        const uint32_t r = F32A ? lr : lr % (MT * 16);
        const uint32_t c = (lane % ALanes) ^ (r & (ALanes >= 16 ? 15u : 7u));
        const uint32_t m = m0 + min(r, rows - 1);  // rows past the end repeat the last (never written)
        if (F32A) {
            kA[i] = c * 4;
            srcA[i] = reinterpret_cast<const char*>(g.a + static_cast<size_t>(m) * g.lda + kA[i]);
        } else {
            kA[i] = c * 8;
            srcA[i] = reinterpret_cast<const char*>(g.a_hl + (lr >= MT * 16 ? plane : 0) + static_cast<size_t>(m) * kp +
                                                    kA[i]);
        }
    }
    };
    if (!GROUPED) set_a(0, g.M);
    const char* srcW[PW];
    uint32_t kW[PW];
    constexpr int WRows = 64 / WLanes;
    const uint32_t wrow0 = wave * PW * WRows + lane / WLanes;
    auto set_w = [&](uint32_t n0, size_t eoff) {
#pragma unroll
        for (int i = 0; i < PW; ++i) {
            const uint32_t row = wrow0 + i * WRows;
            kW[i] = ((lane % WLanes) ^ (row & (WLanes >= 16 ? 15u : 7u))) * 8;
            bool valid;
            srcW[i] = reinterpret_cast<const char*>(gemm_w_row<MODE>(g, n0, static_cast<int>(row), eoff, valid) + kW[i]);
        }
    };
    // Issue side: the next chunk to copy.
    uint32_t ii = blockIdx.x, ib = 0, il = 0, iat = 0, ileft = 0, ist = 0;
    auto issue_open = [&]() {  // item ii: its K chunks [ib, ib + il) and W rows
        const uint32_t z = ii % splits;
        ib = z * per, il = min(per, nch - ib);
        iat = (ii / splits / 8) % il, ileft = il;
        if (GROUPED) {
            const Group gr = group(ii);
            set_a(gr.m0, gr.rows);
            set_w(ii % tiles * kSlabN, static_cast<size_t>(gr.expert) * g.w_expert);
            return;
        }
        set_w(ii / splits * kSlabN, 0);
    };
    auto issue = [&]() {
        if (ii >= items) return;  // uniform
        if (ileft == 0) issue_open();
        const uint32_t k0 = (ib + iat) * KC;
        char* st = gemm_smem + ist * S::Stage;
#pragma unroll
        for (int i = 0; i < PW; ++i) {
            const char* p = k0 + kW[i] < g.K ? srcW[i] + static_cast<size_t>(k0) * 2 : reinterpret_cast<const char*>(slab_zeros);
            __builtin_amdgcn_global_load_lds(p, (lds_void_t*)(st + S::ABytes + (wave * PW + i) * 1024), 16, 0, kSlabCpolNt);
        }
#pragma unroll
        for (int i = 0; i < PA; ++i) {
            const char* p = k0 + kA[i] < g.K ? srcA[i] + static_cast<size_t>(k0) * (F32A ? 4 : 2)
                                             : reinterpret_cast<const char*>(slab_zeros);
            gemm_dma16(p, st + (wave * PA + i) * 1024);
        }
        ist = ist + 1 == ST ? 0 : ist + 1;
        iat = iat + 1 == il ? 0 : iat + 1;
        if (--ileft == 0) ii += gridDim.x;
    };
    // Chunks this block computes in all, and how many are issued ahead.
    uint32_t total = 0;
    for (uint32_t it = blockIdx.x; it < items; it += gridDim.x) {
        const uint32_t b = it % splits * per;
        total += min(per, nch - b);
    }
#pragma unroll
    for (int s = 0; s < ST - 1; ++s) issue();

    const uint32_t lds0 = gemm_lds_addr(gemm_smem);
    const uint32_t fr = lane & 15, fq = static_cast<uint32_t>(lane) >> 4;
    f32x4 acc[MW][NW];
#pragma unroll
    for (int i = 0; i < MW; ++i)
#pragma unroll
        for (int j = 0; j < NW; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    uint32_t ci = blockIdx.x, cc = 0, cn = 0, cst = 0;  // compute side
    for (uint32_t t = 0; t < total; ++t) {
        if (cc == cn) {
            const uint32_t b = ci % splits * per;
            cc = b, cn = min(b + per, nch);
        }
        {  // this wave's copies of chunk t landed; newer chunks stay in flight
            constexpr int kKeep = (7 << 4) | (15 << 8);
            const uint32_t newer = min(static_cast<uint32_t>(ST - 2), total - 1 - t);
#define SLAB_VM(n) __builtin_amdgcn_s_waitcnt((((n)*S::Dma) & 15) | ((((n)*S::Dma) >> 4) << 14) | kKeep)
            if (newer == 0) SLAB_VM(0);
            else if (newer == 1) SLAB_VM(1);
            else if (newer == 2) SLAB_VM(2);
            else if (newer == 3) SLAB_VM(3);
            else SLAB_VM(4);
#undef SLAB_VM
            static_assert(ST - 2 <= 4, "counted waits");
        }
        gemm_barrier();  // everyone's copies landed; the stage of chunk t - 1 is no longer read
        const uint32_t sb = lds0 + cst * S::Stage;
        cst = cst + 1 == ST ? 0 : cst + 1;
        // All fragments of the chunk are asked for before the next copies go
        // out; the products of step s wait for their own reads only.
        f32x4 fa[Steps][MW][2], fw[Steps][NW];
#pragma unroll
        for (int s = 0; s < Steps; ++s) {
            const uint32_t ks = wk * Steps + s;
            const uint32_t cw = ks * 4 + fq;
            const uint32_t wa =
                sb + S::ABytes + (wn * NW * 16 + fr) * (KC * 2) + ((cw ^ (fr & (WLanes >= 16 ? 15u : 7u))) << 4);
#pragma unroll
            for (int j = 0; j < NW; ++j) fw[s][j] = slab_read(wa + j * (16 * KC * 2));
#pragma unroll
            for (int i = 0; i < MW; ++i) {
                const uint32_t row = (wm * MW + i) * 16 + fr;
                if (F32A) {
                    const uint32_t c0 = ks * 8 + fq * 2;
                    fa[s][i][0] = slab_read(sb + row * ARow + ((c0 ^ (fr & 15u)) << 4));
                    fa[s][i][1] = slab_read(sb + row * ARow + (((c0 + 1) ^ (fr & 15u)) << 4));
                } else {
                    const uint32_t a = sb + row * ARow + ((cw ^ (fr & (ALanes >= 16 ? 15u : 7u))) << 4);
                    fa[s][i][0] = slab_read<0>(a);
                    fa[s][i][1] = slab_read<MT * 16 * ARow>(a);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        issue();
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < Steps; ++s) {
            // (LDS reads return in order: the later steps' reads may be out)
            if (s + 1 < Steps) asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"((Steps - 1) * (NW + 2 * MW) > 15 ? 15 : (Steps - 1) * (NW + 2 * MW)));
            else asm volatile("s_waitcnt lgkmcnt(0)" ::);
            slab_tie(fw[s]);
#pragma unroll
            for (int i = 0; i < MW; ++i) slab_tie(fa[s][i]);
#pragma unroll
            for (int i = 0; i < MW; ++i) {
                bf16x8 hi, lo;
                if (F32A) slab_split(fa[s][i][0], fa[s][i][1], hi, lo);
                else hi = __builtin_bit_cast(bf16x8, fa[s][i][0]), lo = __builtin_bit_cast(bf16x8, fa[s][i][1]);
#pragma unroll
                for (int j = 0; j < NW; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hi, __builtin_bit_cast(bf16x8, fw[s][j]), acc[i][j], 0, 0, 0);
#pragma unroll
                for (int j = 0; j < NW; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(lo, __builtin_bit_cast(bf16x8, fw[s][j]), acc[i][j], 0, 0, 0);
            }
        }
        static_assert(Steps <= 2, "counted waits for at most two steps");
        if (++cc != cn) continue;
        // Item done: the WK partial sums in LDS, then the epilogue.
        const uint32_t n0 = (GROUPED ? ci % tiles : ci / splits) * kSlabN, z = GROUPED ? 0 : ci % splits;
        const Group gr = group(ci);
        const uint32_t red = lds0 + ST * S::Stage + (wm * WN + wn) * (MW * NW * 1024) + lane * 16;
        constexpr uint32_t kRedK = WM * WN * MW * NW * 1024;  // bytes of one K group's sums
        if (wk > 0) {
            // An MFMA result read by inline asm: the wait states by hand.
#pragma unroll
            for (int i = 0; i < MW; ++i)
#pragma unroll
                for (int j = 0; j < NW; ++j) asm volatile("s_nop 15" : "+v"(acc[i][j]));
            asm volatile("s_nop 15\n\ts_nop 15" ::);
#pragma unroll
            for (int i = 0; i < MW; ++i)
#pragma unroll
                for (int j = 0; j < NW; ++j) slab_write(red + (wk - 1) * kRedK + (i * NW + j) * 1024, acc[i][j]);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        }
        if (WK > 1) gemm_barrier();
        if (wk == 0) {
#pragma unroll
            for (int w = 0; w < WK - 1; ++w) {
                f32x4 p[MW * NW];
#pragma unroll
                for (int i = 0; i < MW * NW; ++i) p[i] = slab_read(red + w * kRedK + i * 1024);
                slab_wait(p);
#pragma unroll
                for (int i = 0; i < MW * NW; ++i) acc[i / NW][i % NW] += p[i];
            }
#pragma unroll
            for (int i = 0; i < MW; ++i) {
#pragma unroll
                for (int jr = 0; jr < 4; ++jr) {
                    const uint32_t lrow = (wm * MW + i) * 16 + 4 * fq + jr, row = gr.m0 + lrow;
                    if (lrow >= gr.rows) continue;
                    if (MODE == kGemmGateUp) {
                        const uint32_t kpo = gemm_kp(g.N);
#pragma unroll
                        for (int j = 0; j < NW; j += 2) {
                            const uint32_t n = n0 / 2 + (wn * NW + j) * 8 + fr;
                            if (g.out_hl) {
                                if (n < kpo) {
                                    const float v = n < g.N ? silu_mul(acc[i][j][jr], acc[i][j + 1][jr]) : 0.f;
                                    uint16_t* o = g.out_hl + static_cast<size_t>(row) * kpo + n;
                                    const uint16_t h = to_bf16_rne(v);
                                    o[0] = h;
                                    o[g.out_plane] = to_bf16_rne(v - from_bf16(h));
                                }
                            } else if (n < g.N) {
                                g.out[static_cast<size_t>(row) * g.ldo + n] = silu_mul(acc[i][j][jr], acc[i][j + 1][jr]);
                            }
                        }
                        continue;
                    }
#pragma unroll
                    for (int j = 0; j < NW; ++j) {
                        const uint32_t n = n0 + (wn * NW + j) * 16 + fr;
                        if (n >= g.N) continue;
                        float v = acc[i][j][jr];
                        if (MODE == kGemmPlain && z == 0) {
                            const uint16_t* b = n < g.seg_end[0] ? g.bias[0] : n < g.seg_end[1] ? g.bias[1] : g.bias[2];
                            const uint32_t bi = n < g.seg_end[0] ? n : n < g.seg_end[1] ? n - g.seg_end[0] : n - g.seg_end[1];
                            if (b) v = __fadd_rn(v, from_bf16(b[bi]));
                        }
                        float* orow = g.out + static_cast<size_t>(row) * g.ldo;
                        if (splits > 1) g.part[(static_cast<size_t>(z) * g.M + row) * g.N + n] = v;
                        else if (MODE == kGemmResid) orow[n] = __fadd_rn(orow[n], v);
                        else orow[n] = v;
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < MW; ++i)
#pragma unroll
            for (int j = 0; j < NW; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        ci += gridDim.x;
        cc = cn = 0;
    }
}

// out[i] = sum over the splits of part[z * n + i], in split order.
__global__ __launch_bounds__(256) void slab_reduce_kernel(const float* __restrict__ part, float* __restrict__ out,
                                                          uint32_t n, uint32_t splits) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float q[8];
#pragma unroll
    for (uint32_t z = 0; z < 8; ++z) q[z] = z < splits ? part[static_cast<size_t>(z) * n + i] : 0.f;
    float v = q[0];
#pragma unroll
    for (uint32_t z = 1; z < 8; ++z)
        if (z < splits) v += q[z];
    out[i] = v;
}
