// The experts of long passes (lists of more than fifteen tokens on average): every expert against the tokens that listed it, up to 32, 64 or
// 96 of them at a time (walk_tiles), on the products of long_tiles.hpp.  A block takes 128 gate rows and the up rows of the same numbers, or 512 down rows.  Up
// to 64 tokens a wave has two tiles of 32 weight rows, so that a fragment read from LDS serves both; 65 to 96 one tile against three of
// tokens, whose accumulators fill the registers, and a weight is formed once for all of them: with 64 at most an expert of 80 tokens would
// form its weights twice (4096 rows over 512 experts: 1016 us a layer, 908 so).  Three blocks a compute unit instead of two, with fewer
// registers: 960.
// Bounded by the matrix cores and vector issue at 2.0 to 2.2 GHz (4096 rows: up 41 % and 34 % of the time, down 34 % and 26 %), below 20 tokens an expert by forming weights
// for tiles half empty.  us, gate/up + down of one layer of 512 experts, top 10, lists and staging included, before (16 x 16 tiles, up to 48
// tokens a walk) / now:   800 rows 462 / 387   1024 505 / 403   1531 558 / 468   2048 625 / 559   4096 1102 / 908
// Error of a layer's outputs against float64 0.71e-6 (before 0.78e-6).
#include "long_tiles.hpp"
#include "shv_internal.hpp"

namespace {

using namespace shv;
using namespace shv_moe;
using namespace shv_long;

// A wave a row.
template <int K>
__global__ __launch_bounds__(256) void moe_long_stage_kernel(const float *x, int rows, char *staged) {
    const int lane = threadIdx.x & 63, t = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= rows) return;
    float v[K / 256][4];
#pragma unroll
    for (int i = 0; i < K / 256; i++) {
        const float4 q = *reinterpret_cast<const float4 *>(x + static_cast<size_t>(t) * K + 256 * i + 4 * lane);
        v[i][0] = q.x, v[i][1] = q.y, v[i][2] = q.z, v[i][3] = q.w;
    }
    stage_row<K>(v, t, rows, staged);
}

// TILES: the tiles of 32 tokens that a walk over an expert's weights takes at most.

// Which expert and which of its rows a block takes.  The shared expert's blocks come first, `walk` tokens each; the routed experts follow in
// the order of the group workspace (longest list first), every one with all of its list.  The `parts` blocks of one expert and list are
// eight apart, on one die.
struct LongUnit {
    int expert;  // -1: the shared expert
    int part, first, count;
};
__device__ __forceinline__ LongUnit long_unit(int b, int parts, int walk, int n_expert, int n_tok, int n_used, const int32_t *group) {
    LongUnit u;
    const int shared = (n_tok + walk - 1) / walk;
    const int unit = (b / (8 * parts)) * 8 + (b & 7);
    u.part = (b >> 3) % parts;
    if (unit < shared) {
        u.expert = -1;
        u.first = unit * walk;
        u.count = n_tok - u.first < walk ? n_tok - u.first : walk;
    } else if (unit < shared + n_expert) {
        u.expert = __builtin_amdgcn_readfirstlane(group[n_expert + 1 + n_tok * n_used + unit - shared]);
        u.first = __builtin_amdgcn_readfirstlane(group[u.expert]);
        u.count = __builtin_amdgcn_readfirstlane(group[u.expert + 1]) - u.first;
    } else {
        u.expert = 0;
        u.first = u.count = 0;
    }
    return u;
}
int long_blocks(int n_tok, int n_expert, int parts, int walk) { return ((n_tok + walk - 1) / walk + n_expert + 7) / 8 * 8 * parts; }

// The pair (token * (n_used + 1) + slot) at place i of the m that begin at t0; a place past them repeats the first (nothing of it is stored).
__device__ __forceinline__ int pair_at(const LongUnit &u, int t0, int i, int m, int n_used, int n_expert, const int32_t *group) {
    const int at = u.first + t0 + (i < m ? i : 0);
    return u.expert < 0 ? at * (n_used + 1) + n_used : group[n_expert + 1 + at];
}

// ---- gate and up ----

constexpr int kUpThreads = 256, kUpCols = 128;  // a block: 128 gate rows and the up rows of the same numbers
constexpr int kActPitch = kUpCols + 4;
typedef half8_t act8_t __attribute__((aligned(4)));  // act is on a float's grid here; the down projection asks for sixteen bytes'
constexpr int up_room(int tiles) { return stream_lds(tiles) > 32 * tiles * kActPitch * 4 ? stream_lds(tiles) : 32 * tiles * kActPitch * 4; }
constexpr size_t up_lds(int tiles) { return up_room(tiles) + 64 * tiles * sizeof(int32_t); }

// One pass of up to 32 NTT tokens over the gate and up rows of 64 R columns from col0 on (of the block's expert, bank at `at`).  R 2: a wave
// has a tile of 32 gate rows and one of the up rows of the same numbers; R 1: a tile of sixteen gate rows and sixteen up rows.
template <int K, int TILES, int R, int NTT>
__device__ __forceinline__ void up_pass(const shv_moe_up_args &a, const char *gate, const char *up, const char *staged, char *act_sums, const LongUnit &u, int t0, int m, int col0, char *smem,
                                        int wave) {
    constexpr int ROWB = K / 256 * SHV_Q4K_BYTES, COLS = 64 * R;
    const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
    int32_t *pair_s = reinterpret_cast<int32_t *>(smem + up_room(TILES)), *back_s = pair_s + 32 * TILES;
    uint32_t rows[NTT];
#pragma unroll
    for (int i = 0; i < NTT; i++) {
        const int at = (wave * NTT + i) * 8 + (lane >> 3), pair = pair_at(u, t0, at, m, a.n_used, a.n_expert, a.group);
        rows[i] = static_cast<uint32_t>(pair / (a.n_used + 1)) * (K * 4) + chunk_piece(lane, at);
        if ((lane & 7) == 0) pair_s[at] = pair;  // read behind the products' barriers
    }
    // the tile whose sums this wave brings, and the exponents of its rows
    const int tok = pair_at(u, t0, (wave % NTT) * 32 + n, m, a.n_used, a.n_expert, a.group) / (a.n_used + 1);
    if (wave < NTT && h == 0) back_s[wave * 32 + n] = reinterpret_cast<const int32_t *>(staged + row_exps_offset(a.n_tok, K))[tok];
    const char *rp[R];
    if constexpr (R == 2) {
        rp[0] = gate + static_cast<size_t>(col0 + wave * 32 + n) * ROWB;
        rp[1] = up + static_cast<size_t>(col0 + wave * 32 + n) * ROWB;
    } else {
        rp[0] = (n < 16 ? gate : up) + static_cast<size_t>(col0 + wave * 16 + (n & 15)) * ROWB;
    }
    float *act_s = reinterpret_cast<float *>(smem);
    stream_products<K / 256, R, NTT>(rp, 1, 0, smem, wave, buffer_of(staged, a.n_tok * (K * 4)), rows, buffer_of(staged + row_sums_offset(a.n_tok, K), a.n_tok * (K / 256 * 32)),
                                        tok * (K / 256 * 32) + h * 16, kSumUnit, [&](int, const float16_t (&y)[R][NTT]) {
        // by way of LDS, where the chunks lay, to threads that hold eight columns of a row
        landed_barrier<0>();
#pragma unroll
        for (int tt = 0; tt < NTT; tt++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int r = 32 * tt + 8 * (i >> 2) + 4 * h + (i & 3), back = back_s[r];
                float v = ldexpf(y[0][tt][i], back);
                if constexpr (R == 2) v = v * sigmoid_exact(v) * ldexpf(y[1][tt][i], back);
                act_s[r * kActPitch + wave * 32 + n] = v;
            }
    });
    constexpr int PER = COLS / 8;  // threads a row
#pragma unroll
    for (int it = 0; it < 32 * NTT * PER / kUpThreads; it++) {
        const int at = it * kUpThreads + threadIdx.x, i = at / PER, c = (at % PER) * 8;
        const size_t pair = static_cast<size_t>(pair_s[i]);
        const int col = col0 + c;
        const float *from = act_s + i * kActPitch + (R == 2 ? c : (c >> 4) * 32 + (c & 15));
        float v[8], sum = 0.f;
        {
            // the sum is of the values as they are stored (no product and sum in one rounding where R is 1), so that a pair's result
            // is the same bit for bit whichever pass of its list it falls to: the order of a list changes from call to call
#pragma clang fp contract(off)
#pragma unroll
            for (int j = 0; j < 8; j++) {
                v[j] = from[j];
                if constexpr (R == 1) v[j] = v[j] * sigmoid_exact(v[j]) * from[16 + j];
                sum += v[j];
            }
        }
        const float o[8] = {v[0], v[2], v[1], v[3], v[4], v[6], v[5], v[7]};
        sum += __shfl_xor(sum, 1, 64);
        sum += __shfl_xor(sum, 2, 64);
        if (i >= m) continue;
        if (!a.act_packed) {
            float *dst = a.act + pair * a.ffn + col;
#pragma unroll
            for (int j = 0; j < 8; j++) dst[j] = v[j];
            continue;
        }
        half8_t hi, lo;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const _Float16 w = static_cast<_Float16>(o[j]);
            hi[j] = w;
            lo[j] = static_cast<_Float16>(o[j] - static_cast<float>(w));
        }
        char *dst = reinterpret_cast<char *>(a.act) + pair * (a.ffn * 4) + row_at(col);
        *reinterpret_cast<act8_t *>(dst) = hi;
        *reinterpret_cast<act8_t *>(dst + 32) = lo;
        if ((c & 31) == 0) {
            const _Float16 w = static_cast<_Float16>(sum);
            _Float16 *sp = reinterpret_cast<_Float16 *>(act_sums + (pair * (a.ffn / 256) + (col >> 8)) * 32) + ((col >> 5) & 7);
            sp[0] = w;
            sp[8] = static_cast<_Float16>(sum - static_cast<float>(w));
        }
    }
    __syncthreads();  // the chunks' room and the list are read to the end
}

// grid: long_blocks(n_tok, n_expert, ffn / kUpCols, 32 TILES); K = n_embd.
template <int K, int TILES>
__global__ __launch_bounds__(kUpThreads, 2) void moe_up_long_kernel(shv_moe_up_args a, const char *staged, char *act_sums) {
    extern __shared__ __align__(16) char smem[];
    constexpr size_t weight_bytes = K / 256 * SHV_Q4K_BYTES;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const LongUnit u = long_unit(blockIdx.x, a.ffn / kUpCols, 32 * TILES, a.n_expert, a.n_tok, a.n_used, a.group);
    if (u.count <= 0) return;
    const size_t at = static_cast<size_t>(u.expert < 0 ? 0 : u.expert) * a.ffn * weight_bytes;
    const char *gate = static_cast<const char *>(u.expert < 0 ? a.gate_sh : a.gate_exps) + at, *up = static_cast<const char *>(u.expert < 0 ? a.up_sh : a.up_exps) + at;
    const int col0 = u.part * kUpCols;
    for (int t0 = 0; t0 < u.count; t0 += 32 * TILES) {
        const int m = u.count - t0 < 32 * TILES ? u.count - t0 : 32 * TILES;
        if constexpr (TILES == 3) {
            if (m > 64) {
                for (int half = 0; half < 2; half++) up_pass<K, TILES, 1, 3>(a, gate, up, staged, act_sums, u, t0, m, col0 + half * 64, smem, wave);
                continue;
            }
        }
        if constexpr (TILES >= 2) {
            if (m > 32) {
                up_pass<K, TILES, 2, 2>(a, gate, up, staged, act_sums, u, t0, m, col0, smem, wave);
                continue;
            }
        }
        up_pass<K, TILES, 2, 1>(a, gate, up, staged, act_sums, u, t0, m, col0, smem, wave);
    }
}

// ---- down ----

constexpr int kDownThreads = 256;
constexpr int kDownParts = 4;  // blocks an expert's rows go to
constexpr size_t down_lds(int tiles) { return stream_lds(tiles) + 32 * tiles * sizeof(int32_t); }

// A pass of up to 32 NTT act rows against a block's weight rows, 128 R at a time.
template <int K, int TILES, int R, int NTT>
__device__ __forceinline__ void down_pass(const shv_moe_down_args &a, const char *base, const char *act_sums, const LongUnit &u, int t0, int m, int row0, int n_rows, char *smem, int wave) {
    constexpr int SBS = K / 256, ROWB = SBS * SHV_Q4K_BYTES;
    const int lane = threadIdx.x & 63, n = lane & 31, h = lane >> 5;
    int32_t *pair_s = reinterpret_cast<int32_t *>(smem + stream_lds(TILES));
    uint32_t rows[NTT];
#pragma unroll
    for (int i = 0; i < NTT; i++) {
        const int at = (wave * NTT + i) * 8 + (lane >> 3), pair = pair_at(u, t0, at, m, a.n_used, a.n_expert, a.group);
        rows[i] = static_cast<uint32_t>(pair) * (K * 4) + chunk_piece(lane, at);
        if ((lane & 7) == 0) pair_s[at] = pair;
    }
    const int pair = pair_at(u, t0, (wave % NTT) * 32 + n, m, a.n_used, a.n_expert, a.group);
    const int first = row0 + wave * (32 * R) + n;
    const char *rp[R];
#pragma unroll
    for (int r = 0; r < R; r++) rp[r] = base + static_cast<size_t>(first + 32 * r) * ROWB;
    float *out = a.pairs + first;
    stream_products<SBS, R, NTT>(rp, n_rows / (128 * R), 128 * R * ROWB, smem, wave, buffer_of(reinterpret_cast<const char *>(a.act), a.n_tok * (a.n_used + 1) * (K * 4)), rows,
                                 buffer_of(act_sums, a.n_tok * (a.n_used + 1) * (SBS * 32)), pair * (SBS * 32) + h * 16, 1.f,
                                 [&](int unit, const float16_t (&y)[R][NTT]) {
#pragma unroll
        for (int tt = 0; tt < NTT; tt++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int p = 32 * tt + 8 * (i >> 2) + 4 * h + (i & 3);
                if (p < m) {
#pragma unroll
                    for (int r = 0; r < R; r++) out[unit * (128 * R) + 32 * r + static_cast<size_t>(pair_s[p]) * a.n_embd] = y[r][tt][i];
                }
            }
    });
}

// grid: long_blocks(n_tok, n_expert, kDownParts, 32 TILES); K = ffn; act is operands (act_packed).
template <int K, int TILES>
__global__ __launch_bounds__(kDownThreads, 2) void moe_down_long_kernel(shv_moe_down_args a, const char *act_sums) {
    extern __shared__ __align__(16) char smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const LongUnit u = long_unit(blockIdx.x, kDownParts, 32 * TILES, a.n_expert, a.n_tok, a.n_used, a.group);
    if (u.count <= 0) return;
    constexpr size_t weight_bytes = static_cast<size_t>(K / 256) * SHV_Q4K_BYTES;
    const char *base = static_cast<const char *>(u.expert < 0 ? a.down_sh : a.down_exps) + static_cast<size_t>(u.expert < 0 ? 0 : u.expert) * a.n_embd * weight_bytes;
    const int per = a.n_embd / kDownParts, row0 = u.part * per;
    for (int t0 = 0; t0 < u.count; t0 += 32 * TILES) {
        const int m = u.count - t0 < 32 * TILES ? u.count - t0 : 32 * TILES;
        if constexpr (TILES == 3) {
            if (m > 64) {
                down_pass<K, TILES, 1, 3>(a, base, act_sums, u, t0, m, row0, per, smem, wave);
                continue;
            }
        }
        if constexpr (TILES >= 2) {
            if (m > 32) {
                down_pass<K, TILES, 2, 2>(a, base, act_sums, u, t0, m, row0, per, smem, wave);
                continue;
            }
        }
        down_pass<K, TILES, 2, 1>(a, base, act_sums, u, t0, m, row0, per, smem, wave);
    }
}

template <typename Kern>
int raise_lds(Kern kern, size_t lds) {
    SHV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    return SHV_OK;
}

template <int TILES>
int launch_up(shv_ctx *ctx, const shv_moe_up_args &a) {
    static const int raised = raise_lds(&moe_up_long_kernel<2048, TILES>, up_lds(TILES));
    if (raised != SHV_OK) return raised;
    SHV_LAUNCH(ctx, (moe_up_long_kernel<2048, TILES>), dim3(long_blocks(a.n_tok, a.n_expert, a.ffn / kUpCols, 32 * TILES)), dim3(kUpThreads), up_lds(TILES), a,
               static_cast<const char *>(ctx->gemm_stage), reinterpret_cast<char *>(ctx->gemm_part));
    return SHV_OK;
}

template <int TILES>
int launch_down(shv_ctx *ctx, const shv_moe_down_args &a) {
    static const int raised = raise_lds(&moe_down_long_kernel<512, TILES>, down_lds(TILES));
    if (raised != SHV_OK) return raised;
    SHV_LAUNCH(ctx, (moe_down_long_kernel<512, TILES>), dim3(long_blocks(a.n_tok, a.n_expert, kDownParts, 32 * TILES)), dim3(kDownThreads), down_lds(TILES), a,
               reinterpret_cast<const char *>(ctx->gemm_part));
    return SHV_OK;
}

// Tiles of a walk, by the tokens an expert has on average: a kernel that takes no more of them has registers to spare (up: 189, none
// spilled, of one; 256 and 13 spilled of two, 39 of three).  us a layer with one, two and three, lists drawn evenly:
//   15.6 tokens an expert 387 / 403 / 416   22.5: 412 / 425 / 434   25.4: 448 / 438 / 454   30: 510 / 468 / 491   40: 698 / 559 / 578
//   58.6: 840 / 686 / 695   64.5: 921 / 777 / 757   80: 1111 / 961 / 920
// Of lists drawn unevenly the longest, which one expert's blocks walk pass after pass, takes longer than all the others, whichever kernel it is:
// us by the logarithms' deviation over the experts, 0 / 1 / 2 / one expert that every token chose (before: 16 x 16 tiles, up to 48 tokens a walk)
//    800 rows 382 / 418 / 568 / 1009 (before 459 / 444 / 636 / 1255)   1531: 477 / 565 / 1199 / 1357 (563 / 780 / 1984 / 2349)
//   4096: 910 / 1300 / 3022 / 4343 (1095 / 1647 / 4303 / 6187)
int walk_tiles(int n_tok, int n_used, int n_expert) {
    const long long pairs = static_cast<long long>(n_tok) * n_used;
    return pairs <= 24ll * n_expert ? 1 : pairs <= 60ll * n_expert ? 2 : 3;
}

}  // namespace

size_t shv_moe_long_stage_bytes(int n_tok, int n_embd) { return row_bytes(n_tok, n_embd); }

// The rows as operands and the gate/up products of a pass whose lists are made (n_embd 2048, ffn 512).
int shv_launch_moe_up_long(shv_ctx *ctx, const shv_moe_up_args &a) {
    SHV_LAUNCH(ctx, moe_long_stage_kernel<2048>, dim3((a.n_tok + 3) / 4), dim3(256), 0, a.xn, a.n_tok, ctx->gemm_stage);
    const int tiles = walk_tiles(a.n_tok, a.n_used, a.n_expert);
    return tiles == 1 ? launch_up<1>(ctx, a) : tiles == 2 ? launch_up<2>(ctx, a) : launch_up<3>(ctx, a);
}

int shv_launch_moe_down_long(shv_ctx *ctx, const shv_moe_down_args &a) {
    static_assert(2048 % (kDownParts * 256) == 0, "whole tiles");
    const int tiles = walk_tiles(a.n_tok, a.n_used, a.n_expert);
    return tiles == 1 ? launch_down<1>(ctx, a) : tiles == 2 ? launch_down<2>(ctx, a) : launch_down<3>(ctx, a);
}
