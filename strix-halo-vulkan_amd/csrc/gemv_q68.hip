// Q6_K and Q8_0 projections of 2048 columns, up to sixteen activation rows a launch: y[t] = W pro(x[t]) (+ residual[t]).
//
// Bound by HBM: the vocabulary projection of a mixed checkpoint is 255 MB of Q6_K or 330 MB of Q8_0 a token.  What kept it
// from HBM's rate was the way the bytes were fetched (lanes 26 or 34 bytes apart, in pieces of two bytes) and four rows a launch.
// Here the weights of sixteen rows, which lie one after another, go to LDS as one flat run of 16-byte pieces (DMA, two or
// three such tiles ahead of the one in use, one block a compute unit walking the matrix), and the products run on the matrix
// cores: a wave owns 256 of the columns, holds the activations of those in registers for the whole launch and takes its
// sixteen rows' bytes of a tile from LDS.
//   weights      whole numbers q - 32 or q, exact in binary16; the group's scale goes onto the accumulator, the super-block's d
//                onto the sum of its groups
//   activations  scaled by a power of two that brings the row's largest to 2^14 .. 2^15, in three binary16 parts: all 24 bits of
//                anything down to 2^-16 of the largest, and no less of smaller ones than 2^-39 of the largest (error against
//                float64 of 4096 x 2048: 1.0e-7 to 1.4e-7; lane by lane in float32, on the same rows, 1.0e-7 to 1.5e-7).
//                An infinity is all in the first part
//   sums         float32; the waves' columns meet in LDS, in wave order, while the next tile is multiplied
// 151936 x 2048 with the norm folded in, us, before -> now, of 1 / 2 / 8 / 14 rows: Q6_K 123 207 763 1342 -> 59 58 67 67,
// Q8_0 92 153 640 1117 -> 59 61 63 69.  The bytes alone take 41 and 53; forming Q6_K's weights and multiplying them adds what it
// does because vector and matrix instructions take turns on this path (without the products 42).
#include <algorithm>
#include <atomic>
#include <type_traits>

#include "group_dot.hpp"
#include "shv_internal.hpp"

namespace {

using namespace shv;
using namespace shv_any;

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float4_t __attribute__((ext_vector_type(4)));

constexpr int kW = 8;        // waves a block
constexpr int kTokens = 16;  // activation rows a launch

// D: tiles in LDS.
template <int TYPE>
struct Shape {
    static constexpr int K = 256 * kW;
    static constexpr int ROW = TYPE == SHV_GGML_Q6_K ? K / 256 * 210 : K / 32 * 34;  // bytes of a row: whole 16-byte pieces
    // a Q8_0 row of LDS ends in a spare piece: 2176 bytes would put every second row's dwords into the same banks
    static constexpr int PIECES = ROW / 16 + (TYPE == SHV_GGML_Q8_0 ? 1 : 0), PITCH = PIECES * 16;
    static constexpr int ASKS = (16 * PIECES + 63) / 64, SLOT = ASKS * 1024;  // 1 KB pieces of a tile
    static constexpr int PER = (ASKS + kW - 1) / kW;                          // of a wave, at most
    static constexpr int D = 4 * SLOT <= 120 * 1024 ? 4 : 3 * SLOT <= 120 * 1024 ? 3 : 2;
    static constexpr int PART = kW * 16 * kTokens * 4;
    static constexpr size_t LDS = static_cast<size_t>(D) * SLOT + 2 * PART + kTokens * 4;
    static_assert(ROW % 16 == 0 && LDS <= 160 * 1024, "rows of whole pieces, a block's LDS");
};

// bytes 0..3 of v as the halves 1024 + byte, minus `bias`
__device__ __forceinline__ half4_t bytes_to_halves(uint32_t v, _Float16 bias) {
    const half2_t b2 = {bias, bias};
    const half2_t lo = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)) - b2;
    const half2_t hi = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)) - b2;
    return half4_t{lo[0], lo[1], hi[0], hi[1]};
}

// A lane's bytes of a tile: of the wave's super-block of row n, the columns the lane kb of the products takes.
template <int TYPE>
struct Raw;
template <>
struct Raw<SHV_GGML_Q6_K> {
    // a super-block starts at 210 wave, an odd one two bytes past a dword: dwords as they lie, two for one of the block's
    uint32_t v[12][2], s[5];
    int sh;
    static __device__ __forceinline__ int offset(int wave) { return wave * 210 & ~3; }
    // dword i of 12: the low bits, 16 levels a step; from the ninth the high ones
    __device__ __forceinline__ void load(const char *b, int i, int kb) {
        const uint32_t *q = reinterpret_cast<const uint32_t *>(b + 16 * i + 4 * kb);
        v[i][0] = q[0];
        v[i][1] = q[1];
    }
    __device__ __forceinline__ void load_scales(const char *b) {
#pragma unroll
        for (int i = 0; i < 5; i++) s[i] = reinterpret_cast<const uint32_t *>(b + 192)[i];  // and the block's behind them
    }
    __device__ __forceinline__ void load(const char *b, int wave, int kb, int) {
        sh = (wave & 1) * 16;
#pragma unroll
        for (int i = 0; i < 12; i++) load(b, i, kb);
        load_scales(b);
    }
    __device__ __forceinline__ uint32_t dw(int i) const {
        return i < 12 ? __builtin_amdgcn_alignbit(v[i][1], v[i][0], sh) : __builtin_amdgcn_alignbit(s[i - 11], s[i - 12], sh);
    }
    // step st = 2 * half + 16 columns of 32: four groups
    __device__ __forceinline__ void load_step(int st, const char *b, int kb) {
        const int h = st >> 1, hf = st & 1;
        load(b, 4 * h + hf, kb);
        load(b, 4 * h + 2 + hf, kb);
        load(b, 8 + 2 * h + hf, kb);
    }
    __device__ __forceinline__ void form(int st, half4_t (&w)[4]) const {
        const int h = st >> 1, hf = st & 1;
        const uint32_t la = dw(4 * h + hf), lb = dw(4 * h + 2 + hf), qh = dw(8 + 2 * h + hf);
        const uint32_t q[4] = {(la & 0x0F0F0F0Fu) | ((qh << 4) & 0x30303030u), (lb & 0x0F0F0F0Fu) | ((qh << 2) & 0x30303030u),
                               ((la >> 4) & 0x0F0F0F0Fu) | (qh & 0x30303030u), ((lb >> 4) & 0x0F0F0F0Fu) | ((qh >> 2) & 0x30303030u)};
#pragma unroll
        for (int k = 0; k < 4; k++) w[k] = bytes_to_halves(q[k], static_cast<_Float16>(1056.f));
    }
    __device__ __forceinline__ uint32_t scale() const { return s[4] >> sh; }
};
template <>
struct Raw<SHV_GGML_Q8_0> {
    uint32_t v[8][3];
    uint16_t d[8];
    static __device__ __forceinline__ int offset(int wave) { return wave * 272; }
    __device__ __forceinline__ void load(const char *b, int g, int kb) {
        const char *blk = b + 34 * g;
        d[g] = *reinterpret_cast<const uint16_t *>(blk);
        const uint32_t *q = reinterpret_cast<const uint32_t *>(blk + (g & 1) * 2 + 8 * kb);  // an odd block's levels start on a dword, an even one's two bytes past it
        v[g][0] = q[0];
        v[g][1] = q[1];
        v[g][2] = (g & 1) ? 0u : q[2];
    }
    __device__ __forceinline__ void load(const char *b, int, int kb, int) {
#pragma unroll
        for (int g = 0; g < 8; g++) load(b, g, kb);
    }
    __device__ __forceinline__ void levels(int g, uint32_t &q0, uint32_t &q1) const {
        q0 = (g & 1) ? v[g][0] : __builtin_amdgcn_alignbit(v[g][1], v[g][0], 16);
        q1 = (g & 1) ? v[g][1] : __builtin_amdgcn_alignbit(v[g][2], v[g][1], 16);
    }
};

// grid: blocks that walk the tiles of 16 weight rows, kW waves.
// The products' sixteen activation rows hold the three parts of each of SETS * 4 = 4 rows, one product doing for all of them (and
// the lane that has a row's three sums adds them up); SETS = 0: sixteen rows, their parts one after another into the same sums.
template <int TYPE, int SETS>
__global__ __launch_bounds__(64 * kW) void gemv_q68_kernel(shv_gemv_args a, int t0, int nt) {
    constexpr int M = SETS > 0 ? SETS : 3;    // products a group
    constexpr int A = SETS > 0 ? SETS : 1;    // sums of them
    constexpr int OUT = SETS > 0 ? SETS : 4;  // outputs of a lane
    using P = Shape<TYPE>;
    constexpr int D = P::D;
    extern __shared__ __align__(16) char smem[];
    float *part = reinterpret_cast<float *>(smem + D * P::SLOT);  // [2][wave][lane][4]
    float *factor = part + 2 * P::PART / 4;
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, kb = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n_tiles = (a.n + 15) / 16;
    // ---- the tiles' way into LDS ----
    constexpr int FULL = P::ASKS / kW, MORE = P::ASKS % kW;  // asks of every wave, waves with one more
    const int asks = FULL + (wave < MORE ? 1 : 0);
    uint32_t prow[P::PER], poff[P::PER];
#pragma unroll
    for (int i = 0; i < P::PER; i++) {
        const int p = std::min((i * kW + wave) * 64 + lane, 16 * P::PIECES - 1);
        prow[i] = p / P::PIECES;
        poff[i] = std::min(p % P::PIECES, P::ROW / 16 - 1) * 16;
    }
    auto ask = [&](int tile, int slot) {
        const char *src = static_cast<const char *>(a.w) + static_cast<size_t>(tile) * 16 * P::ROW;
        const uint32_t last = a.n - 1 - tile * 16;  // rows past the matrix read its last
#pragma unroll
        for (int i = 0; i < P::PER; i++)
            if (i < asks)
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src + (std::min(prow[i], last) * P::ROW + poff[i])),
                                                 (__attribute__((address_space(3))) void *)(smem + slot * P::SLOT + (i * kW + wave) * 1024), 16, 0, 0);
    };
    const int first = blockIdx.x, step = gridDim.x;
#pragma unroll
    for (int i = 0; i < D; i++)
        if (first + i * step < n_tiles) ask(first + i * step, i);
    // ---- the activations: lane (token n, kb) holds its columns of the wave's range, as the products will ask for them ----
    constexpr int G = TYPE == SHV_GGML_Q6_K ? 16 : 8;   // products a super-block
    constexpr int C = 64 / G;                           // columns of a lane in one of them: 4, 8
    _Float16 xf[G][M][C];
    constexpr int LOADS = SETS > 0 ? SETS : 1;
    float v[LOADS][G][C];
#pragma unroll
    for (int set = 0; set < LOADS; set++) {
        const int tok = std::min(SETS > 0 ? set * 4 + (n >> 2) : n, nt - 1);
        const float *x = a.x + static_cast<size_t>(t0 + tok) * (a.x_stride > 0 ? a.x_stride : a.k) + wave * 256;
        const float *gm = a.gamma ? a.gamma + wave * 256 : nullptr;
        float ss = 0.f, mx = 0.f;
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int c = 0; c < C; c += 4) {
                const int at = g * (256 / G) + kb * C + c;
                const float4 q = *reinterpret_cast<const float4 *>(x + at);
                ss = fmaf(q.x, q.x, fmaf(q.y, q.y, fmaf(q.z, q.z, fmaf(q.w, q.w, ss))));
                float4 u = {1.f, 1.f, 1.f, 1.f};
                if (gm) u = *reinterpret_cast<const float4 *>(gm + at);
                v[set][g][c] = q.x * u.x; v[set][g][c + 1] = q.y * u.y; v[set][g][c + 2] = q.z * u.z; v[set][g][c + 3] = q.w * u.w;
#pragma unroll
                for (int j = 0; j < 4; j++) mx = fmaxf(mx, fabsf(v[set][g][c + j]));
            }
        ss += __shfl_xor(ss, 16, 64);
        ss += __shfl_xor(ss, 32, 64);
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        if (kb == 0) {
            part[(set * kW + wave) * 32 + n] = ss;
            part[(set * kW + wave) * 32 + 16 + n] = mx;
        }
    }
    __syncthreads();
#pragma unroll
    for (int set = 0; set < LOADS; set++) {
        const int tok = SETS > 0 ? set * 4 + (n >> 2) : n;
        float ss = 0.f, mx = 0.f;
#pragma unroll
        for (int w = 0; w < kW; w++) {
            ss += part[(set * kW + w) * 32 + n];
            mx = fmaxf(mx, part[(set * kW + w) * 32 + 16 + n]);
        }
        int e = 0;
        // (a row with an infinity: its finite values go below it, as small as they can be told from zero or smaller)
        if (mx > 0.f) e = mx < INFINITY ? std::max(-120, std::min(120, 14 - ilogbf(mx))) : -114;
        if (wave == 0 && kb == 0 && tok < nt) factor[tok] = ldexpf(a.gamma ? 1.f / sqrtf(ss / static_cast<float>(a.k) + a.eps) : 1.f, -e);
#pragma unroll
        for (int g = 0; g < G; g++)
#pragma unroll
            for (int c = 0; c < C; c++) {
                const float u = ldexpf(v[set][g][c], e);
                const _Float16 h = static_cast<_Float16>(u);
                const float u1 = mx < INFINITY ? u - static_cast<float>(h) : 0.f;
                const _Float16 m = static_cast<_Float16>(u1), l = static_cast<_Float16>(u1 - static_cast<float>(m));
                if constexpr (SETS > 0) {
                    xf[g][set][c] = (n & 3) == 0 ? h : (n & 3) == 1 ? m : (n & 3) == 2 ? l : static_cast<_Float16>(0.f);
                } else {
                    xf[g][0][c] = h;
                    xf[g][1][c] = m;
                    xf[g][2][c] = l;
                }
            }
    }
    __syncthreads();  // part is free again
    // ---- the outputs of a tile: thread o adds up row o % 16 of token o / 16 over the waves ----
    const int o_row = tid & 15, o_tok = tid >> 4, o_kb = SETS > 0 ? o_tok : o_tok >> 2, o_i = SETS > 0 ? o_tok >> 2 : o_tok;
    const bool mine = o_tok < nt;
    const float scale = mine ? factor[o_tok] : 0.f;
    const size_t y_at = static_cast<size_t>(t0 + (mine ? o_tok : 0)) * (a.y_stride > 0 ? a.y_stride : a.n);
    const float *from = part + ((o_kb & 3) * 16 + o_row) * OUT + (o_i & 3) % OUT;
    auto put = [&](int tile, int buf) {
        const int row = tile * 16 + o_row;
        if (!mine || row >= a.n) return;
        float v = from[buf * (P::PART / 4)];
#pragma unroll
        for (int w = 1; w < kW; w++) v += from[buf * (P::PART / 4) + w * (64 * OUT)];
        v *= scale;
        a.y[y_at + row] = a.residual ? v + a.residual[y_at + row] : v;
    };
    Raw<TYPE> raw;
    int slot = 0, buf = 0, prev = -1;  // the tile whose sums are in LDS
    // multiplies the tile in `raw` and reads the next one's bytes, at `b`, behind the last use of each
    auto sum_of = [](const float4_t (&c)[A], int i) {
        if constexpr (SETS > 0) return (c[i][0] + c[i][1]) + c[i][2];
        else return c[0][i];
    };
    half4_t w[4];
    auto multiply = [&](const char *b) {
        float4_t y = {0.f, 0.f, 0.f, 0.f};
        if constexpr (TYPE == SHV_GGML_Q6_K) {
            // four steps of four groups; a step's products run while the next one's weights are formed (`w`: the first of this tile
            // when it begins, of the next one when it ends)
            float ys[OUT];
#pragma unroll
            for (int i = 0; i < OUT; i++) ys[i] = 0.f;
            float4_t acc[2][4][A];
            auto add = [&](int st) {
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const int g = 8 * (st >> 1) + 2 * k + (st & 1);
                    const float f = static_cast<float>(static_cast<int8_t>(raw.dw(12 + (g >> 2)) >> (8 * (g & 3))));
#pragma unroll
                    for (int i = 0; i < OUT; i++) ys[i] = fmaf(f, sum_of(acc[st & 1][k], i), ys[i]);
                }
            };
#pragma unroll
            for (int st = 0; st < 4; st++) {
                half4_t wn[4];
                if (st == 0) raw.load_step(0, b, kb);
                raw.form((st + 1) & 3, wn);
                if (st < 3) raw.load_step(st + 1, b, kb);
#pragma unroll
                for (int k = 0; k < 4; k++)
#pragma unroll
                    for (int s = 0; s < A; s++) acc[st & 1][k][s] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int m = 0; m < M; m++)
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const _Float16(&x)[C] = xf[8 * (st >> 1) + 2 * k + (st & 1)][m];
                        float4_t &c = acc[st & 1][k][SETS > 0 ? m : 0];
                        c = __builtin_amdgcn_mfma_f32_16x16x16f16(half4_t{x[0], x[1], x[2], x[3]}, w[k], c, 0, 0, 0);
                    }
                if (st > 0) add(st - 1);
#pragma unroll
                for (int i = 0; i < 4 * M; i++) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // a product,
                    __builtin_amdgcn_sched_group_barrier(0x2, 12 / M, 0);  // some of the vector instructions
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int k = 0; k < 4; k++) w[k] = wn[k];
            }
            add(3);
            const float d = f16_bits_to_f32(raw.scale());
            raw.load_scales(b);
#pragma unroll
            for (int i = 0; i < OUT; i++) y[i] = d * ys[i];
        } else {
#pragma unroll
            for (int g = 0; g < 8; g++) {
                uint32_t q0, q1;
                raw.levels(g, q0, q1);
                const float d = f16_bits_to_f32(raw.d[g]);
                raw.load(b, g, kb);
                __builtin_amdgcn_sched_barrier(0);
                const half4_t w0 = bytes_to_halves(q0 ^ 0x80808080u, static_cast<_Float16>(1152.f)), w1 = bytes_to_halves(q1 ^ 0x80808080u, static_cast<_Float16>(1152.f));
                const half8_t w = {w0[0], w0[1], w0[2], w0[3], w1[0], w1[1], w1[2], w1[3]};
                float4_t acc[A];
#pragma unroll
                for (int s = 0; s < A; s++) acc[s] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int m = 0; m < M; m++) {
                    const _Float16(&f)[C] = xf[g][m];
                    float4_t &c = acc[SETS > 0 ? m : 0];
                    c = __builtin_amdgcn_mfma_f32_16x16x32_f16(half8_t{f[0], f[1], f[2], f[3], f[4 % C], f[5 % C], f[6 % C], f[7 % C]}, w, c, 0, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < OUT; i++) y[i] = fmaf(d, sum_of(acc, i), y[i]);
            }
        }
#pragma unroll
        for (int i = 0; i < OUT; i++) part[buf * (P::PART / 4) + (wave * 64 + lane) * OUT + i] = y[i];  // row n, activation row kb of set i (4 kb + i)
        buf ^= 1;
    };
    // Behind it everyone's pieces of the tile have come which is followed by `behind` others on their way (a wave's own: when no
    // more than theirs are still out), everyone has read the tile before, and its sums are in LDS.
    auto arrive = [&](bool all, auto behind) {
        constexpr int N1 = decltype(behind)::value * (FULL + 1), N0 = decltype(behind)::value * FULL;
        if (all) __builtin_amdgcn_s_waitcnt(0x0F70);
        else if (wave < MORE) __builtin_amdgcn_s_waitcnt(0x0F70 | (N1 & 15) | ((N1 >> 4) << 14));
        else __builtin_amdgcn_s_waitcnt(0x0F70 | (N0 & 15) | ((N0 >> 4) << 14));
        __builtin_amdgcn_s_waitcnt(0xC07F);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    const char *mine_at = smem + n * P::PITCH + Raw<TYPE>::offset(wave);
    arrive(first + (D - 1) * step >= n_tiles, std::integral_constant<int, D - 1>());
    raw.load(mine_at, wave, kb, 0);
    if constexpr (TYPE == SHV_GGML_Q6_K) raw.form(0, w);
    for (int tile = first; tile < n_tiles; tile += step) {
        arrive(tile + (D - 1) * step >= n_tiles, std::integral_constant<int, D - 2>());  // the next tile
        if (tile + D * step < n_tiles) ask(tile + D * step, slot);                       // where this one was
        slot = slot + 1 == D ? 0 : slot + 1;
        if (prev >= 0) put(prev, buf ^ 1);
        multiply(mine_at + slot * P::SLOT);  // behind the last tile: whatever is there, not multiplied
        prev = tile;
    }
    __syncthreads();
    if (prev >= 0) put(prev, buf ^ 1);
}

template <int TYPE, int SETS>
int launch_sets(shv_ctx *ctx, const shv_gemv_args &a, int t0, int nt) {
    using P = Shape<TYPE>;
    static std::atomic<bool> raised{false};
    if (!raised.load(std::memory_order_acquire)) {
        SHV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&gemv_q68_kernel<TYPE, SETS>), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(P::LDS)));
        raised.store(true, std::memory_order_release);
    }
    SHV_LAUNCH(ctx, (gemv_q68_kernel<TYPE, SETS>), dim3(std::min((a.n + 15) / 16, ctx->prop.multiProcessorCount)), dim3(64 * kW), P::LDS, a, t0, nt);
    return SHV_OK;
}

template <int TYPE>
int launch(shv_ctx *ctx, const shv_gemv_args &a) {
    const int rows = a.n_tok > 0 ? a.n_tok : 1;
    for (int t0 = 0; t0 < rows; t0 += kTokens) {
        const int nt = std::min(kTokens, rows - t0);
        // Q6_K keeps the vector units and the matrix cores busy (and the two do not run side by side here): up to four rows, a
        // third of the products.  Q8_0 waits for its bytes either way.
        const int rc = TYPE == SHV_GGML_Q6_K && nt <= 4 ? launch_sets<TYPE, TYPE == SHV_GGML_Q6_K>(ctx, a, t0, nt) : launch_sets<TYPE, 0>(ctx, a, t0, nt);
        if (rc != SHV_OK) return rc;
    }
    return SHV_OK;
}

}  // namespace

// The one row length that is built: a wave's 256 columns of it are 96 registers of activations, which leave room for the rest.
// (4096 columns would take sixteen waves, or twice the registers; fewer columns fewer waves: neither has been built or measured,
// such matrices go lane by lane, gemv_any.hip.)  And rows of x that 16-byte loads can read.
bool shv_gemv_q68_covers(const shv_gemv_args &a) {
    if ((a.type != SHV_GGML_Q6_K && a.type != SHV_GGML_Q8_0) || a.k != 2048) return false;
    return shv_aligned16(a.x) && (!a.gamma || shv_aligned16(a.gamma)) && (a.n_tok <= 1 || a.x_stride % 4 == 0);
}

int shv_launch_gemv_q68(shv_ctx *ctx, const shv_gemv_args &a) {
    return a.type == SHV_GGML_Q6_K ? launch<SHV_GGML_Q6_K>(ctx, a) : launch<SHV_GGML_Q8_0>(ctx, a);
}
