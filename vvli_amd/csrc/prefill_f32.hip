// prefill_f32.hip -- batched prompt processing for f32 weights: what
// prefill.hip does for bf16 ones, with every product in f32
// (v_mfma_f32_16x16x4_f32), so that a prompt keeps the precision of the token
// loop (src/generator.zig:243-251, src/llm.zig:702-766). The RoPE / KV pass is
// shared; the norm, the matrix products and the attention are here.
//
// The token loop reads all weights once per token: Qwen2.5-0.5B's layers at 48
// rows (four of them, 240 MB) took 10.05 ms, 209 us a token; here 326 us. What
// bounds them now is latency: eight launches a layer of 3.7 to 22 us (gate/up
// 22, down 13, o_proj and q|k|v 6 each; gate/up's bytes and products take 6),
// with two of a block's load groups in flight. Counters: gate/up's matrix cores
// are busy 19 % of the cycles, down's 13 %, the others' under 5 %.
#include <algorithm>
#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"

namespace vvli {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// out[M][N] = A[M][K] . W[N][K]^T.
//
// A block owns MT x 16 rows of A and NT x 16 rows of W over a K range; its
// four waves take a quarter of that range each and their sums meet in LDS, in
// wave order. Operands go from the caches straight into registers: the f32
// MFMA takes 32 cycles for 16 x 16 x 4, so a wave's loads (16 bytes per lane,
// 64 bytes of 16 rows per instruction) come to at most 24 bytes per cycle and
// CU, and LDS would only add a hop. Lane l holds k = 4 (l / 16) .. + 3 of row
// l % 16; MFMA j multiplies component j, which orders the k of a 16-wide step
// differently in A and W alike. Two register buffers of U steps each: the
// loads of one are in flight while the other is multiplied.
//
// Sums: chains of 8 products, two of which make a step's sum, the steps added
// up in order, then the waves and splits: about as many roundings on a
// product's way as in the GEMV's per-lane sums and tree. (With chains of 32
// the prompts of 9 to 100 rows were 5 % further off their 64-bit results.)
// ---------------------------------------------------------------------------
constexpr int kF32Threads = 256, kF32Waves = 4;

__device__ __forceinline__ const float* f32_w_row(const F32GemmArgs& g, uint32_t n) {
    const uint32_t nn = n < g.N ? n : 0;  // rows past N read row 0 (never written)
    if (nn < g.seg_end[0]) return g.w[0] + static_cast<size_t>(nn) * g.K;
    if (nn < g.seg_end[1]) return g.w[1] + static_cast<size_t>(nn - g.seg_end[0]) * g.K;
    return g.w[2] + static_cast<size_t>(nn - g.seg_end[1]) * g.K;
}

template <int MODE, int MT, int NT, int U>
__global__ __launch_bounds__(kF32Threads, 2) void gemm_f32_kernel(F32GemmArgs g, uint32_t tm, uint32_t tn) {
    // GateUp: the W rows of a 16-column tile are 8 gate rows and their 8 up rows.
    constexpr int NOut = MODE == kGemmGateUp ? NT * 8 : NT * 16;  // output columns of a block
    __shared__ f32x4 red[kF32Waves][MT * NT][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Consecutive blocks go to the 8 XCDs in turn: each XCD walks a contiguous
    // run of tiles, rows fastest, so a W tile is read through one L2.
    const uint32_t ntile = tm * tn, xcd = blockIdx.x % 8, rem = ntile % 8;
    const uint32_t u = xcd * (ntile / 8) + min(xcd, rem) + blockIdx.x / 8;
    const uint32_t m0 = u % tm * (MT * 16), n0 = u / tm * NOut;
    const uint32_t fr = lane & 15, fq = static_cast<uint32_t>(lane) >> 4;

    // K steps of 16: this block's split, then this wave's share.
    const uint32_t nk = (g.K + 15) / 16, per = (nk + gridDim.z - 1) / gridDim.z;
    const uint32_t b0 = min(nk, blockIdx.z * per), b1 = min(nk, b0 + per);
    const uint32_t wper = (b1 - b0 + kF32Waves - 1) / kF32Waves;
    const uint32_t s0 = min(b1, b0 + wave * wper), s1 = min(b1, s0 + wper);

    const float* pa[MT];
    const float* pw[NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
        pa[i] = g.a + static_cast<size_t>(min(m0 + i * 16 + fr, g.M - 1)) * g.lda;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        if (MODE == kGemmGateUp) {
            const uint32_t n = n0 + j * 8 + (fr & 7);
            pw[j] = (fr < 8 ? g.w[0] : g.w_up) + static_cast<size_t>(n < g.N ? n : 0) * g.K;
        } else pw[j] = f32_w_row(g, n0 + j * 16 + fr);
    }
    f32x4 sum[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    struct Buf {
        f32x4 a[U][MT], w[U][NT];
    };
    // Steps past the end load the row's start (K >= 4) and count as zeros.
    auto load = [&](Buf& b, uint32_t st) {
#pragma unroll
        for (int x = 0; x < U; ++x) {
            const uint32_t k = (st + x) * 16 + fq * 4;
            const uint32_t kk = st + x < s1 && k < g.K ? k : 0;
#pragma unroll
            for (int j = 0; j < NT; ++j)
                b.w[x][j] = *as_global(reinterpret_cast<const f32x4*>(pw[j] + kk));
#pragma unroll
            for (int i = 0; i < MT; ++i)
                b.a[x][i] = *as_global(reinterpret_cast<const f32x4*>(pa[i] + kk));
        }
    };
    auto multiply = [&](Buf& b, uint32_t st) {
        if (st + U > s1 || (st + U) * 16 > g.K) {  // uniform: the last group
#pragma unroll
            for (int x = 0; x < U; ++x)
                if (st + x >= s1 || (st + x) * 16 + fq * 4 >= g.K) {
#pragma unroll
                    for (int j = 0; j < NT; ++j) b.w[x][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int i = 0; i < MT; ++i) b.a[x][i] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
        }
#pragma unroll
        for (int x = 0; x < U; ++x) {
            f32x4 acc[2][MT][NT];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int i = 0; i < MT; ++i)
#pragma unroll
                        for (int j = 0; j < NT; ++j)
                            acc[h][i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                                b.a[x][i][2 * h + e], b.w[x][j][2 * h + e], e ? acc[h][i][j] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) sum[i][j] += acc[0][i][j] + acc[1][i][j];
        }
    };
    Buf b0r, b1r;
    if (s0 < s1) {
        load(b0r, s0);
        for (uint32_t st = s0; st < s1; st += 2 * U) {
            if (st + U < s1) load(b1r, st + U);
            multiply(b0r, st);
            if (st + U >= s1) break;
            if (st + 2 * U < s1) load(b0r, st + 2 * U);
            multiply(b1r, st + U);
        }
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) red[wave][i * NT + j][lane] = sum[i][j];
    __syncthreads();
    const bool split = gridDim.z > 1;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            if ((i * NT + j) % kF32Waves != wave) continue;
            f32x4 v = red[0][i * NT + j][lane];
#pragma unroll
            for (int w = 1; w < kF32Waves; ++w) v += red[w][i * NT + j][lane];
            if (MODE == kGemmGateUp) {  // the up sums sit eight lanes on
                const int up_lane = (lane & ~15) + 8 + (lane & 7);
                f32x4 up = red[0][i * NT + j][up_lane];
#pragma unroll
                for (int w = 1; w < kF32Waves; ++w) up += red[w][i * NT + j][up_lane];
                const uint32_t n = n0 + j * 8 + fr;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t row = m0 + i * 16 + 4 * fq + e;
                    if (fr < 8 && row < g.M && n < g.N)  // siluMulInto, src/llm.zig:1382-1387
                        g.out[static_cast<size_t>(row) * g.ldo + n] =
                            __fmul_rn(__fdiv_rn(v[e], __fadd_rn(1.0f, expf(-v[e]))), up[e]);
                }
                continue;
            }
            const uint32_t n = n0 + j * 16 + fr;
            if (n >= g.N) continue;
            float bias = 0.f;
            if (MODE == kGemmPlain && blockIdx.z == 0) {
                const int s = n < g.seg_end[0] ? 0 : n < g.seg_end[1] ? 1 : 2;
                if (g.bias[s]) bias = g.bias[s][n - (s ? g.seg_end[s - 1] : 0)];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t row = m0 + i * 16 + 4 * fq + e;
                if (row >= g.M) continue;
                float* o = g.out + static_cast<size_t>(row) * g.ldo + n;
                const float r = MODE == kGemmPlain ? __fadd_rn(v[e], bias) : v[e];
                if (split) g.part[(static_cast<size_t>(blockIdx.z) * g.M + row) * g.N + n] = r;
                else *o = MODE == kGemmResid ? __fadd_rn(*o, r) : r;  // addInto, src/llm.zig:1389-1396
            }
        }
    }
}

// y_r = (x_r * w) * s_r, s_r = 1 / sqrt(mean(x_r^2) + eps) (rmsNormInto,
// src/llm.zig:1287-1300), a block per row, after adding the K-split partial
// sums of the product that made x (split order, written back).
constexpr int kNormThreads = 256;
__global__ __launch_bounds__(kNormThreads) void row_norm_f32_kernel(float* __restrict__ x, uint32_t n, uint32_t rows,
                                                                    float eps, const float* __restrict__ w,
                                                                    const float* __restrict__ part, uint32_t splits,
                                                                    float* __restrict__ y) {
    __shared__ float red[kNormThreads / 64];
    const size_t at = static_cast<size_t>(blockIdx.x) * n;
    float ss = 0.f;
    for (uint32_t k = threadIdx.x * 4; k < n; k += kNormThreads * 4) {
        float4 v = *reinterpret_cast<const float4*>(x + at + k);
        if (part) {
            v = add_parts(v, part + at + k, static_cast<size_t>(rows) * n, splits);
            *reinterpret_cast<float4*>(x + at + k) = v;
        }
        ss = fmaf(v.x, v.x, ss), ss = fmaf(v.y, v.y, ss), ss = fmaf(v.z, v.z, ss), ss = fmaf(v.w, v.w, ss);
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < kNormThreads / 64; ++i) t += red[i];
    const float s = 1.0f / sqrtf(t / static_cast<float>(n) + eps);
    for (uint32_t k = threadIdx.x * 4; k < n; k += kNormThreads * 4) {  // (this thread's own x)
        const float4 v = *reinterpret_cast<const float4*>(x + at + k);
        const float4 c = *reinterpret_cast<const float4*>(w + k);
        *reinterpret_cast<float4*>(y + at + k) =
            make_float4(__fmul_rn(__fmul_rn(v.x, c.x), s), __fmul_rn(__fmul_rn(v.y, c.y), s),
                        __fmul_rn(__fmul_rn(v.z, c.z), s), __fmul_rn(__fmul_rn(v.w, c.w), s));
    }
}

__global__ __launch_bounds__(256) void embed_rows_f32_kernel(const float* __restrict__ embed,
                                                             const uint32_t* __restrict__ tokens, uint32_t n,
                                                             float* __restrict__ x) {
    const uint32_t i = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (i < n)
        *reinterpret_cast<float4*>(x + static_cast<size_t>(blockIdx.y) * n + i) =
            *reinterpret_cast<const float4*>(embed + static_cast<size_t>(tokens[blockIdx.y]) * n + i);
}

// ---------------------------------------------------------------------------
// Causal GQA attention over the f32 cache rows (computeAttentionInto,
// src/llm.zig:1302-1335). A block owns 16 query vectors of a kv head ((row,
// q head) pairs, rows slowest); its four waves take the key chunks of 16 in
// turn, each with its own running max, sum and output, which meet in LDS in
// wave order. Products transposed, as in prefill.hip: S^T = K . Q^T gives lane
// l the scores of keys 4 (l / 16) + j of vector l % 16, which are its operand
// of O^T += V^T . P^T. K and V come from the caches; the next chunk's are
// loaded while this one is multiplied. A hidden key has weight 0, which its V
// must not turn into NaN (a later row's V may be anything): the chunks with
// hidden keys, which come last, take V's values that are not finite out of the
// products and add them for the vectors that see them. (In a loop of their own:
// the check in the loop over all chunks cost 5 % behind 16000 rows.)
// ---------------------------------------------------------------------------
template <int HD>
__global__ __launch_bounds__(kF32Threads) void attn_f32_kernel(PrefillAttnArgs a) {
    constexpr int DT = HD / 16;  // 16-dim tiles
    __shared__ f32x4 so[kF32Waves][DT][64];
    __shared__ float sm[kF32Waves][16], sl[kF32Waves][16];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t fr = lane & 15, fq = static_cast<uint32_t>(lane) >> 4;
    const uint32_t G = a.heads / a.kv_heads, nvec = a.rows * G;
    const uint32_t groups = (nvec + 15) / 16;
    const uint32_t kvh = blockIdx.x % a.kv_heads, v0 = (groups - 1 - blockIdx.x / a.kv_heads) * 16;  // longest first
    const uint32_t vec = min(v0 + fr, nvec - 1);
    const uint32_t row = vec / G, head = kvh * G + vec % G, pos = a.start + row;
    const uint32_t keys = a.start + min(v0 + 15, nvec - 1) / G + 1;  // keys of the block's last vector
    const uint32_t chunks = (keys + 15) / 16;
    const uint32_t first_pos = a.start + v0 / G;  // position of the block's first vector

    f32x4 q[DT], o[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d) {
        q[d] = *as_global(reinterpret_cast<const f32x4*>(a.q + static_cast<size_t>(row) * a.ldq + head * HD + d * 16 + fq * 4));
        o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    float m = -INFINITY, l = 0.f;
    const float* kb = a.kcache + kvh * HD + fq * 4;
    const float* vb = a.vcache + kvh * HD + fr;
    f32x4 k[DT];
    float v[4][DT];
    // Keys past the last read it again; their scores are -inf.
    auto load_k = [&](uint32_t c) {
        const float* p = kb + static_cast<size_t>(min(c * 16 + fr, keys - 1)) * a.kvdim;
#pragma unroll
        for (int d = 0; d < DT; ++d) k[d] = *as_global(reinterpret_cast<const f32x4*>(p + d * 16));
    };
    auto load_v = [&](uint32_t c) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float* p = vb + static_cast<size_t>(min(c * 16 + fq * 4 + j, keys - 1)) * a.kvdim;
#pragma unroll
            for (int d = 0; d < DT; ++d) v[j][d] = *as_global(p + d * 16);
        }
    };
    auto chunk = [&](uint32_t c, auto hidden) {  // hidden: keys that some vector must not see
        constexpr bool Hidden = decltype(hidden)::value;
        load_v(c);
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d = 0; d < DT; ++d) {  // chains of 16 products
            f32x4 h = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e) h = __builtin_amdgcn_mfma_f32_16x16x4f32(k[d][e], q[d][e], h, 0, 0, 0);
            s += h;
        }
        if (c + kF32Waves < chunks) load_k(c + kF32Waves);
        float mx = -INFINITY;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            s[j] = !Hidden || c * 16 + fq * 4 + j <= pos ? __fmul_rn(s[j], a.scale) : -INFINITY;
            mx = fmaxf(mx, s[j]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float mn = fmaxf(m, mx);
        const float ms = mn == -INFINITY ? 0.f : mn;  // every key so far is hidden: p = 0, corr = 0
        const float corr = expf(m - ms);
        float p[4];
        float add = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) p[j] = expf(s[j] - ms), add += p[j];
        l = l * corr + add;
        m = mn;
        bool strange = false;
        if (Hidden) {
            float t = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int d = 0; d < DT; ++d) t = fmaf(v[j][d], 0.f, t);  // NaN if one is not finite
            strange = __any(t != 0.f);
            if (strange)
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int d = 0; d < DT; ++d) v[j][d] = fabsf(v[j][d]) < INFINITY ? v[j][d] : 0.f;
        }
        f32x4 add_o[DT];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int d = 0; d < DT; ++d)
                add_o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[j][d], p[j], j ? add_o[d] : f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        if (strange) {  // p[i % 4] of key i sits in the lanes of group i / 4
#pragma unroll 1
            for (uint32_t i = 0; i < 16; ++i) {
                const float pi = i & 2 ? (i & 1 ? p[3] : p[2]) : (i & 1 ? p[1] : p[0]);
                const float pk = __shfl(pi, (i / 4) * 16 + fr, 64);
                const uint32_t key = c * 16 + i;
                const float* vp = a.vcache + static_cast<size_t>(min(key, keys - 1)) * a.kvdim + kvh * HD + fq * 4;
#pragma unroll
                for (int d = 0; d < DT; ++d) {
                    const f32x4 x = *as_global(reinterpret_cast<const f32x4*>(vp + d * 16));
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (key <= pos && !(fabsf(x[e]) < INFINITY)) add_o[d][e] = fmaf(pk, x[e], add_o[d][e]);
                    __builtin_amdgcn_sched_barrier(0);  // (few registers for a rare path)
                }
            }
        }
#pragma unroll
        for (int d = 0; d < DT; ++d) o[d] = o[d] * corr + add_o[d];
    };
    uint32_t c = wave;
    if (c < chunks) load_k(c);
    for (; c < chunks && c * 16 + 15 <= first_pos; c += kF32Waves) chunk(c, std::false_type{});
    for (; c < chunks; c += kF32Waves) chunk(c, std::true_type{});
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (fq == 0) sm[wave][fr] = m, sl[wave][fr] = l;
#pragma unroll
    for (int d = 0; d < DT; ++d) so[wave][d][lane] = o[d];
    __syncthreads();
    float M = -INFINITY;  // finite: wave 0 saw key 0
#pragma unroll
    for (int w = 0; w < kF32Waves; ++w) M = fmaxf(M, sm[w][fr]);
    float L = 0.f, wt[kF32Waves];
#pragma unroll
    for (int w = 0; w < kF32Waves; ++w) {
        wt[w] = expf(sm[w][fr] - M);
        L += sl[w][fr] * wt[w];
    }
    const float inv = 1.0f / L;
    for (int d = wave; d < DT; d += kF32Waves) {
        f32x4 r = so[0][d][lane] * wt[0];
#pragma unroll
        for (int w = 1; w < kF32Waves; ++w) r += so[w][d][lane] * wt[w];
        if (v0 + fr >= nvec) continue;
        r *= inv;
        if (a.out_hl) {  // split planes of o_proj's A: hi = bf16(x), lo = bf16(x - hi)
            bf16x4 hi, lo;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                hi[e] = static_cast<__bf16>(r[e]);
                lo[e] = static_cast<__bf16>(r[e] - static_cast<float>(hi[e]));
            }
            uint16_t* hp = a.out_hl + static_cast<size_t>(row) * (a.heads * HD) + head * HD + d * 16 + fq * 4;
            *reinterpret_cast<bf16x4*>(hp) = hi;
            *reinterpret_cast<bf16x4*>(hp + a.out_plane) = lo;
        } else {
            *reinterpret_cast<f32x4*>(a.out + static_cast<size_t>(row) * a.ldo + head * HD + d * 16 + fq * 4) = r;
        }
    }
}

template <int MODE, int MT, int NT, int U>
hipError_t launch_t(const F32GemmArgs& g, uint32_t splits, hipStream_t s) {
    const uint32_t nout = MODE == kGemmGateUp ? NT * 8 : NT * 16;
    const uint32_t tm = (g.M + MT * 16 - 1) / (MT * 16), tn = (g.N + nout - 1) / nout;
    return vlaunch(gemm_f32_kernel<MODE, MT, NT, U>, dim3(tm * tn, 1, splits), dim3(kF32Threads), 0, s, g, tm, tn);
}

// Tiles and steps in flight: one 16-column tile of W a block up to 64 rows (two
// where gate and up share a block), few steps a buffer so that several blocks
// share a CU. 48 rows through four Qwen2.5-0.5B layers 375 -> 326 us against
// four steps and at least eight a wave.
template <int MODE>
hipError_t launch_mode(const F32GemmArgs& g, uint32_t splits, hipStream_t s) {
    constexpr int NT = MODE == kGemmGateUp ? 2 : 1;
    if (g.M <= 16) return launch_t<MODE, 1, NT, 2>(g, splits, s);
    if (g.M <= 32) return launch_t<MODE, 2, NT, 2>(g, splits, s);
    if (g.M <= 48) return launch_t<MODE, 3, NT, 1>(g, splits, s);
    if (g.M <= 64) return launch_t<MODE, 4, NT, 1>(g, splits, s);
    return launch_t<MODE, 4, 2, 1>(g, splits, s);
}

}  // namespace

// K splits (Plain and Resid, with `part`): up to two blocks per CU, each wave
// of a split at least 2 K steps, at most kMaxPartSplits.
uint32_t gemm_f32_splits(int mode, const F32GemmArgs& g) {
    if (mode == kGemmGateUp || !g.part) return 1;
    const uint32_t mt = g.M <= 16 ? 1 : g.M <= 32 ? 2 : g.M <= 48 ? 3 : 4, nt = g.M <= 64 ? 1 : 2;
    const uint32_t tiles = ((g.M + mt * 16 - 1) / (mt * 16)) * ((g.N + nt * 16 - 1) / (nt * 16));
    const uint32_t nk = (g.K + 15) / 16;
    uint32_t splits = std::max(1u, std::min({512u / std::max(1u, tiles), nk / (kF32Waves * 2), kMaxPartSplits}));
    while (splits > 1 && static_cast<size_t>(splits) * g.M * g.N > gemm_part_elems()) --splits;
    const uint32_t per = (nk + splits - 1) / splits;
    return (nk + per - 1) / per;  // every split gets K steps
}

hipError_t launch_gemm_f32(int mode, const F32GemmArgs& g, hipStream_t s) {
    if (g.M == 0 || g.N == 0) return hipSuccess;
    if (!g.a || !g.out || g.K == 0 || g.K % 4 != 0 || g.lda % 4 != 0 || !g.w[0] || g.seg_end[2] != g.N ||
        (mode == kGemmGateUp && !g.w_up))
        return hipErrorInvalidValue;
    const uint32_t splits = gemm_f32_splits(mode, g);
    switch (mode) {
        case kGemmPlain: return launch_mode<kGemmPlain>(g, splits, s);
        case kGemmResid: return launch_mode<kGemmResid>(g, splits, s);
        case kGemmGateUp: return launch_mode<kGemmGateUp>(g, splits, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_row_norm_f32(float* x, uint32_t n, uint32_t rows, float eps, const float* w, const float* part,
                               uint32_t splits, float* y, hipStream_t s) {
    if (n % 4 != 0 || !w || !y || (part && splits > kMaxPartSplits)) return hipErrorInvalidValue;
    return vlaunch(row_norm_f32_kernel, dim3(rows), dim3(kNormThreads), 0, s, x, n, rows, eps, w,
                   splits > 1 ? part : nullptr, splits, y);
}

hipError_t launch_embed_rows_f32(const float* embed, const uint32_t* tokens, uint32_t rows, uint32_t n, float* x,
                                 hipStream_t s) {
    if (n % 4 != 0) return hipErrorInvalidValue;
    return vlaunch(embed_rows_f32_kernel, dim3((n / 4 + 255) / 256, rows), dim3(256), 0, s, embed, tokens, n, x);
}

// Whether bf16 prompts take it: the MFMA attention of prefill.hip does three
// bf16 products for each f32 one here, about five times as fast, but wants its
// K/V tile images written first (a pass over the earlier rows, scattered
// stores for the new ones) and runs 64 vectors a block. Whole prompts, us a
// layer, that / this: 1B shape 45 rows after 200 94 / 88, 64 after 2000 138 /
// 119, 256 after 500 160 / 157, 400 201 / 198, 512 210 / 212; Qwen2.5-0.5B 32
// rows 63 / 60, 400 after 300 135 / 128, 700 141 / 141; OLMoE 256 391 / 380.
// Few rows behind a long cache, where this one has few blocks and that one packs
// the whole cache first (its best form): 1B shape 4 rows after 32000 702 / 598,
// 16 after 8000 230 / 193, 64 after 2000 134 / 117; Qwen2.5-7B 2 after 32000
// 1178 / 969, 8 after 10000 470 / 404; Qwen2.5-0.5B 64 after 4000 149 / 128.
bool attn_f32_short(uint32_t rows, uint32_t start, uint32_t heads, uint32_t hd) {
    const float pairs = static_cast<float>(heads) * rows * (start + 0.5f * rows) * (hd / 64.f);
    return pairs <= (start ? 6e6f : 3e6f);
}

hipError_t launch_attn_f32(const PrefillAttnArgs& a, uint32_t hd, hipStream_t s) {
    if (a.rows == 0) return hipSuccess;
    if (a.kv_heads == 0 || a.heads % a.kv_heads != 0 ||
        (a.out_hl && (a.out_plane < static_cast<size_t>(a.rows) * a.heads * hd)))
        return hipErrorInvalidValue;
    const uint32_t G = a.heads / a.kv_heads;
    const dim3 grid((a.rows * G + 15) / 16 * a.kv_heads);
    switch (hd) {
        case 32: return vlaunch(attn_f32_kernel<32>, grid, dim3(kF32Threads), 0, s, a);
        case 64: return vlaunch(attn_f32_kernel<64>, grid, dim3(kF32Threads), 0, s, a);
        case 128: return vlaunch(attn_f32_kernel<128>, grid, dim3(kF32Threads), 0, s, a);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace vvli
