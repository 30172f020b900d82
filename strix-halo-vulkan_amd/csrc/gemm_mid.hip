// Q4_K projections of 9 to some hundreds of activation rows: y[t] = W pro(x[t]) (+ residual[t]).
//
// A block takes 16 R weight rows and all their columns, a wave 256 or 512 of the columns: it reads its weights once, forms
// n * sc of them in registers and keeps them there while the pass's tiles of 16 activation rows go by.  A tile's fragments
// come straight from L2, where a launch before this one left them in operand order (a fragment is one contiguous kilobyte,
// three are asked for ahead of the one in use); the waves' partial tiles meet in LDS behind one barrier a tile.  No slab is
// staged, no column part is left for another launch to join.
//   products   v_mfma_f32_16x16x32_f16, activations x weights: a lane holds one weight row (its scales, its d); the
//              activations as two binary16 parts, the weights as the whole numbers n * sc, exact in binary16, one
//              accumulator a super-block
//   min term   per super-block one v_mfma_f32_16x16x32_bf16 of the sub-blocks' sums with the rows' mins: a float32 sum is exactly
//              three bfloat16 parts, and it leaves binary16's range long before one of its 32 activations does.  (Two
//              v_mfma_f32_16x16x4_f32 of the sums as they are: 12352 x 2048 of 150 rows 30.2 us, of 512 rows 78.9.)
// Up to 64 rows the weights' way through memory and the two launches bound it; from there the fragments' way from L2: 128 KB
// a tile and block of 64 weight rows go at 31 bytes a clock and compute unit (1.7 us a tile), whatever their number in
// flight, where the products alone would take half of that.  More rows a block would need more registers than there are:
// 64 rows of 2048 columns, formed, are 256 of a compute unit's 512 KB, and forming them again for each tile costs what it saves.
// us, with the staging launch, two dozen matrices in turn (n x k, rows), and what the launches of 16, of 64 rows and their joins
// took that this kernel has replaced:
//   12352 x 2048   9: 20.3, now 9.6   16: 24.6, 9.5   150: 69.1, 27.3   255: 49.0, 40   512: 90, 72.4
//    2048 x 4096   9: 16.0, now 8.5   16: 16.5, 8.8   150: 51.5, 18.6   255: 59.7, 23.5   512: 65, 36.0
// Error against float64 of 4096 x 2048 over normal activations: 0.4e-6; of the kernels of 16 and of 64 rows 2.1e-6.
#include <algorithm>
#include <atomic>

#include "gemm_rows.hpp"
#include "moe_staged.hpp"

namespace {

using namespace shv;
using namespace shv_gemm;
using namespace shv_moe;

// The staged activations of a pass: fragments [tile of 16 rows][super-block][v][part] of 1 KB, v = nibble half * 4 + block of
// 8 columns: lane (row n, group kb) holds columns 64 kb + 32 half + 8 block .. + 7 of the super-block, in the order a
// payload dword's nibbles come; then the sub-blocks' sums [tile][super-block] of 1 KB: lane (n, kb) those of sub-blocks
// 2 kb and 2 kb + 1, first parts, second, third, two zeros; then where each row's outputs go (a ring's row takes divisions and two loads to find).
constexpr int kMidFrag = 1024, kMidSb = 16 * kMidFrag, kMidSums = 64 * 16;
__host__ __device__ constexpr size_t mid_sums_offset(int tiles, int k) { return static_cast<size_t>(tiles) * (k / 256) * kMidSb; }
__host__ __device__ constexpr size_t mid_rows_offset(int tiles, int k) { return mid_sums_offset(tiles, k) + static_cast<size_t>(tiles) * (k / 256) * kMidSums; }
__host__ __device__ constexpr size_t mid_bytes(int tiles, int k) { return mid_rows_offset(tiles, k) + static_cast<size_t>(tiles) * 16 * sizeof(size_t); }

// grid: (column parts, 4 quartets of rows of a tile, tiles), 256 threads: a wave takes one row's 64 quads of a super-block
// at a time; rows past the pass's are written as zeros.  SBS: the super-blocks of a row, 0: a.k / 256 of them, asked for.
// A launch of a few dozen small blocks is as long as its chain of trips to memory, so everything that waits for nothing is asked for
// first (the whole row for its norm, the position for the ring's row, gamma) and nothing sits behind a branch: a row past the
// pass's reads the last one's.  With a norm that took a trip a super-block, and row, position, gate
// and gamma one behind the other, a pass of 16 layers (two of these launches in each) was longer: one token of 12 sequences
// 1719 us, now 1686, prompts of 9, 40 and 150 rows 1462 (1434), 3163 (3142) and 5305 (5278).
template <int PRO, int SBS>
__global__ __launch_bounds__(256) void gemm_mid_stage_kernel(shv_gemv_q4k_args a, char *staged, int tiles, float *x_out) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int sbs = SBS > 0 ? SBS : a.k / 256, K = sbs * 256, c = 4 * lane;  // c: within the super-block
    const int n = blockIdx.y * 4 + wave, t = blockIdx.z * 16 + n;
    const bool on = t < a.n_tok;
    const int from = on ? t : a.n_tok - 1;
    // which row of its sequence, and where that sequence stands in the ring
    const int sl = a.seq_len > 0 ? a.seq_len : a.n_tok, seq = from / sl, in_seq = from % sl;
    int32_t pos = 0, slot = seq;
    if (a.ring_slots > 0) {
        if (a.pos) pos = load_in_turn(a.pos + seq);
        if (a.slot) slot = load_in_turn(a.slot + seq);
    }
    const float *x = a.x + static_cast<size_t>(from) * a.x_stride;
    const int first = blockIdx.x;
    float4 v = *reinterpret_cast<const float4 *>(x + first * 256 + c), g = make_float4(1.f, 1.f, 1.f, 1.f), z = g;
    if constexpr (PRO == SHV_PRO_RMSNORM) g = *reinterpret_cast<const float4 *>(a.gamma + first * 256 + c);
    if constexpr (PRO == SHV_PRO_GATED_NORM) g = *reinterpret_cast<const float4 *>(a.gamma + (c & (a.head_dim - 1)));
    float scale = 1.f;
    if constexpr (PRO == SHV_PRO_RMSNORM) {
        float ss = 0.f;
        const auto square = [&](const float4 &r) { ss = fmaf(r.x, r.x, fmaf(r.y, r.y, fmaf(r.z, r.z, fmaf(r.w, r.w, ss)))); };
        if constexpr (SBS > 0) {
            float4 row[SBS];
#pragma unroll
            for (int i = 0; i < SBS; i++) row[i] = *reinterpret_cast<const float4 *>(x + i * 256 + c);
#pragma unroll
            for (int i = 0; i < SBS; i++) square(row[i]);
        } else {
            for (int i = 0; i < sbs; i++) square(*reinterpret_cast<const float4 *>(x + i * 256 + c));
        }
        scale = 1.f / sqrtf(wave_sum_all(ss) / static_cast<float>(K) + a.eps);
    }
    size_t ring_row = 0;
    if (a.ring_slots > 0)
        ring_row = static_cast<size_t>(__builtin_amdgcn_readfirstlane(slot)) * a.ring_slots + static_cast<size_t>((__builtin_amdgcn_readfirstlane(pos) + in_seq) % a.ring_slots);
    constexpr bool GATED = PRO == SHV_PRO_GATED_NORM || PRO == SHV_PRO_MUL_SIGMOID;
    const float *gate = nullptr;
    if constexpr (GATED) gate = a.z_ring ? a.z + ring_row * a.ring_stride : a.z + static_cast<size_t>(from) * a.z_stride;
    for (int sb = first; sb < sbs; sb += gridDim.x) {
        const int col = sb * 256 + c;
        if constexpr (GATED) {
            const int zi = PRO == SHV_PRO_MUL_SIGMOID && a.head_dim > 0 ? (col & ~(a.head_dim - 1)) * 2 + a.head_dim + (col & (a.head_dim - 1)) : col;
            z = *reinterpret_cast<const float4 *>(gate + zi);
        }
        if (sb != first) {
            v = *reinterpret_cast<const float4 *>(x + col);
            if constexpr (PRO == SHV_PRO_RMSNORM) g = *reinterpret_cast<const float4 *>(a.gamma + col);
        }
        float o[4] = {v.x, v.y, v.z, v.w};
        const float gg[4] = {g.x, g.y, g.z, g.w}, zz[4] = {z.x, z.y, z.z, z.w};
        if constexpr (PRO == SHV_PRO_RMSNORM) {
#pragma unroll
            for (int j = 0; j < 4; j++) o[j] *= scale * gg[j];
        } else if constexpr (PRO == SHV_PRO_GATED_NORM) {
            float ss = fmaf(o[0], o[0], fmaf(o[1], o[1], fmaf(o[2], o[2], o[3] * o[3])));
            const int span = a.head_dim / 4;  // lanes a head spans: a power of two up to 64
            if (span >= 2) ss += dpp_f32<kDppXor1>(ss);
            if (span >= 4) ss += dpp_f32<kDppXor2>(ss);
            if (span >= 8) ss += dpp_f32<kDppHalfMirror>(ss);
            if (span >= 16) ss += dpp_f32<kDppMirror>(ss);
            if (span >= 32) ss += __shfl_xor(ss, 16, 64);
            if (span >= 64) ss += __shfl_xor(ss, 32, 64);
            const float head = 1.f / sqrtf(ss / static_cast<float>(a.head_dim) + a.eps);
#pragma unroll
            for (int j = 0; j < 4; j++) o[j] = o[j] * head * gg[j] * sigmoid_fast(zz[j]);
        } else if constexpr (PRO == SHV_PRO_MUL_SIGMOID) {
#pragma unroll
            for (int j = 0; j < 4; j++) o[j] *= sigmoid_fast(zz[j]);
        }
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] = on ? o[j] : 0.f;
        // the transformed row itself, for a caller that also needs it as plain float32 (the router's xn)
        if (x_out && on) *reinterpret_cast<float4 *>(x_out + static_cast<size_t>(t) * K + col) = make_float4(o[0], o[1], o[2], o[3]);
        const float sum = sum8_all((o[0] + o[1]) + (o[2] + o[3]));
        const int sub = c >> 5, kb = sub >> 1, u = (sub & 1) * 4 + ((c & 31) >> 3);
        const size_t at = static_cast<size_t>(blockIdx.z) * sbs + sb;
        const float next = dpp_f32<kDppMirror>(sum);  // the sub-block's after it, which the next eight lanes hold
        if ((c & 63) == 0) *reinterpret_cast<u32x4_t *>(staged + mid_sums_offset(tiles, K) + at * kMidSums + (kb * 16 + n) * 16) = bf16_parts_pair(sum, next);
        const float in_order[4] = {o[0], o[2], o[1], o[3]};
        half4_t h, l;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const _Float16 hi = static_cast<_Float16>(in_order[j]);
            h[j] = hi;
            l[j] = static_cast<_Float16>(in_order[j] - static_cast<float>(hi));
        }
        char *e = staged + at * kMidSb + u * (2 * kMidFrag) + (kb * 16 + n) * 16 + ((c & 7) >> 2) * 8;
        *reinterpret_cast<half4_t *>(e) = h;
        *reinterpret_cast<half4_t *>(e + kMidFrag) = l;
    }
    // where the row's outputs go
    if (blockIdx.x == 0 && lane == 0)
        reinterpret_cast<size_t *>(staged + mid_rows_offset(tiles, K))[t] = !on ? 0 : a.ring_slots > 0 && !a.z_ring ? ring_row * a.ring_stride : static_cast<size_t>(t) * a.y_stride;
}

typedef const __attribute__((address_space(1))) void *mid_global_t;
typedef __attribute__((address_space(3))) void *mid_lds_t;
typedef const __attribute__((address_space(3))) char *mid_bytes_t;
typedef const __attribute__((address_space(3))) u32x4_t *mid_quad_t;

// A barrier behind which the waves' LDS writes are seen; fragments and stores in flight stay in flight.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// grid: (groups of 16 R weight rows, chunks of the pass's tiles), W waves: wave w takes columns 256 S w .. of every tile.
template <int R, int S, int W>
__global__ __launch_bounds__(64 * W) void gemm_mid_kernel(shv_gemv_q4k_args a, const char *staged, int tiles, int per_chunk) {
    extern __shared__ __align__(16) char smem[];
    float *cpart = reinterpret_cast<float *>(smem);  // [2][W][R][64][4]
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, kb = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int SBS = S * W, ROWB = SBS * SHV_Q4K_BYTES;
    const int row0 = blockIdx.x * (16 * R), tile0 = blockIdx.y * per_chunk;
    const int tile_end = tile0 + per_chunk < tiles ? tile0 + per_chunk : tiles;
    const NibbleMasks nc = nibble_masks();
    // The wave's weights first, its columns of every row one piece of 144 S bytes, by way of a corner of LDS of its own: asked for by the
    // lanes that form them they are sixteen bytes of 64 lines a load, 64 cycles of the cache's address unit each, and 12 loads for 9 (a
    // pass of 16 layers, so and now: 9 rows 1352 and 1337 us, 40 rows 2924 and 2882, 150 rows 4918 and 4879, 12 sequences 1620 and 1606).
    constexpr int PIECES = 9 * S, ASKED = 16 * R * PIECES;
    char *corner = smem + 2 * W * R * 1024 + wave * (ASKED * 16);
    const char *wbase = static_cast<const char *>(a.w) + static_cast<size_t>(row0) * ROWB + wave * (S * SHV_Q4K_BYTES);
#pragma unroll
    for (int i = 0; i < (ASKED + 63) / 64; i++) {
        const int at = i * 64 + lane, rr = min(at / PIECES, a.n - 1 - row0);
        if ((i + 1) * 64 <= ASKED || at < ASKED)
            __builtin_amdgcn_global_load_lds((mid_global_t)(wbase + static_cast<uint32_t>(rr * ROWB + at % PIECES * 16)), (mid_lds_t)(corner + i * 1024), 16, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    const char *frag = staged + (static_cast<size_t>(tile0) * SBS + wave * S) * kMidSb + lane * 16;
    const char *sums = staged + mid_sums_offset(tiles, a.k) + (static_cast<size_t>(tile0) * SBS + wave * S) * kMidSums + lane * 16;
    constexpr int D = 4;  // fetches held; eight are no faster
    auto ask = [&](const char *fp, int i, half8_t (&f)[2]) {
#pragma unroll
        for (int p = 0; p < 2; p++) f[p] = *reinterpret_cast<const half8_t *>(fp + (i * 2 + p) * kMidFrag);
    };
    half8_t f[D][2];
    bf16x8_t sx[S];
#pragma unroll
    for (int i = 0; i < D - 1; i++) ask(frag, i, f[i]);
#pragma unroll
    for (int s = 0; s < S; s++) sx[s] = *reinterpret_cast<const bf16x8_t *>(sums + s * kMidSums);
    __builtin_amdgcn_sched_barrier(0);
    static_assert(2 * (D - 1) + S < 16, "vmcnt");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (2 * (D - 1) + S));  // all but the fragments and sums: the weights have landed
    __builtin_amdgcn_sched_barrier(0);
    const mid_bytes_t held = (mid_bytes_t)(corner) + n * (PIECES * 16);
    // n * sc of the wave's columns, held for every tile of the chunk
    half8_t wt[S][R][8];
    uint32_t am[S][R];
    float d[S][R], dmin[S][R];
#pragma unroll
    for (int s = 0; s < S; s++)
#pragma unroll
        for (int r = 0; r < R; r++) {
            const mid_bytes_t at = held + r * (16 * PIECES * 16) + s * SHV_Q4K_BYTES;
            const u32x4_t h = *(mid_quad_t)(at), q0 = *(mid_quad_t)(at + 16 + kb * 32), q1 = *(mid_quad_t)(at + 32 + kb * 32);
            uint32_t sc, mn;
            q4k_group_scale_min(make_uint4(h.x, h.y, h.z, h.w), kb, sc, mn);
#pragma unroll
            for (int v = 0; v < 8; v++) {
                const u32x4_t &x = (v & 2) ? q1 : q0;
                const uint32_t d0 = (v & 1) ? x.z : x.x, d1 = (v & 1) ? x.w : x.y;
                wt[s][r][v] = v < 4 ? weights8<false>(d0, d1, sc & 0xFFu, nc) : weights8<true>(d0, d1, sc >> 8, nc);
            }
            am[s][r] = bf16_pair(mn & 0xFFu, mn >> 8);
            d[s][r] = f16_bits_to_f32(h.x);
            dmin[s][r] = f16_bits_to_f32(h.x >> 16);
        }
    constexpr int PER = R * 256 >= 64 * W ? R * 256 / (64 * W) : 1;  // outputs a lane adds up over the waves
    static_assert(PER == 1 || PER == 2 || PER == 4, "a lane's share of a tile");
    const int o = tid * PER < R * 256 ? tid * PER : 0, row = row0 + 16 * (o >> 8) + ((o >> 2) & 15), t_in = 4 * (o >> 6 & 3) + (o & 3);
    const bool mine = tid * PER < R * 256 && row < a.n;
    const size_t *rows = reinterpret_cast<const size_t *>(staged + mid_rows_offset(tiles, a.k));
    size_t to_at[PER];
    float res[PER];
    auto find = [&](int tile) {
        const int t = tile * 16 + t_in;
#pragma unroll
        for (int j = 0; j < PER; j++) {
            to_at[j] = rows[t + j];
            res[j] = a.residual && mine ? a.residual[static_cast<size_t>(t + j < a.n_tok ? t + j : a.n_tok - 1) * a.y_stride + row] : 0.f;
        }
    };
    int buf = 0;
    for (int tile = tile0; tile < tile_end; tile++) {
        const bool more = tile + 1 < tile_end;
        const char *fnext = more ? frag + SBS * kMidSb : frag, *snext = more ? sums + SBS * kMidSums : sums;
        find(tile);  // asked for here, needed at the tile's end
        float4_t y[R];
        bf16x8_t sn[S];
#pragma unroll
        for (int s = 0; s < S; s++) {
            float4_t acc[R];
#pragma unroll
            for (int r = 0; r < R; r++) acc[r] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int at = s * 8 + i, to = at + D - 1;
                if (to < S * 8) ask(frag, to, f[to % D]);
                else ask(fnext, to - S * 8, f[to % D]);
                if (to == S * 8) {
#pragma unroll
                    for (int s2 = 0; s2 < S; s2++) sn[s2] = *reinterpret_cast<const bf16x8_t *>(snext + s2 * kMidSums);
                }
                __builtin_amdgcn_sched_barrier(0);  // the fragments stay ahead of their use
#pragma unroll
                for (int p = 0; p < 2; p++)
#pragma unroll
                    for (int r = 0; r < R; r++) acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[at % D][p], wt[s][r][i], acc[r], 0, 0, 0);
            }
            // the super-block ends: its sums take the row's d, its mins the row's dmin
#pragma unroll
            for (int r = 0; r < R; r++) {
                const u32x4_t m3 = {am[s][r], am[s][r], am[s][r], 0u};  // the same two mins against each part
                const float4_t cm = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sx[s], __builtin_bit_cast(bf16x8_t, m3), float4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float m = -dmin[s][r] * cm[j];
                    y[r][j] = s == 0 ? fmaf(d[s][r], acc[r][j], m) : fmaf(d[s][r], acc[r][j], y[r][j] + m);
                }
            }
        }
        frag = fnext; sums = snext;
#pragma unroll
        for (int s = 0; s < S; s++) sx[s] = sn[s];
        // ---- the waves' columns meet: every lane adds up its share of the tile in wave order ----
        float *cp = cpart + buf * (W * R * 256);
#pragma unroll
        for (int r = 0; r < R; r++) *reinterpret_cast<float4_t *>(cp + ((wave * R + r) * 64 + lane) * 4) = y[r];
        lds_barrier();
        if (mine) {
#pragma unroll
            for (int j = 0; j < PER; j++) {
                float v = cp[o + j];
#pragma unroll
                for (int w = 1; w < W; w++) v += cp[w * (R * 256) + o + j];
                if (tile * 16 + t_in + j < a.n_tok) a.y[to_at[j] + row] = v + res[j];  // C[activation row 4 kb + j][weight row n]
            }
        }
        buf ^= 1;
    }
}

// ------------------------------------------- few rows against a matrix of many rounds ---------
// The vocabulary projection of five to sixteen rows.  A block of eight waves, two a compute unit, walks groups of 16 weight rows: a
// group's 18 KB go by way of LDS, the two after it on their way while it is multiplied, and a wave keeps its 256 columns of the one
// tile of activations in registers.  Sums and their order are gemm_mid_kernel's.
// Bound by HBM as far as two blocks out of step hide each other's waits (one of 32 rows a group: 52 us).  151936 x 2048, us of 5 / 8 / 9 / 16 rows
// with the staging launch: gemm_q4k.hip's walk to eight rows and gemm_mid_kernel from nine 74.8 / 73.6 / 64.2 / 66.9, here 46.0 / 45.0 / 45.2 / 47.2, error
// against float64 0.95 and the same.  A group loaded 64 bytes of sixteen rows at a time, rows' pieces side by side, took 2 us more.
// Two to four rows gain 7 us alone (52 to 45) and nothing in a pass, gemv_mrows.hip needing no staging launch: they stay there.
constexpr int kFewRows = 16, kFewSlots = 3, kFewSlot = kFewRows * 8 * SHV_Q4K_BYTES, kFewLoads = kFewSlot / 1024;
constexpr size_t kFewLds = static_cast<size_t>(kFewSlots) * kFewSlot + 8 * 1024;

__global__ __launch_bounds__(512, 4) void gemm_few_kernel(shv_gemv_q4k_args a, const char *staged) {
    constexpr int W = 8, ROWB = W * SHV_Q4K_BYTES, PIECES = ROWB / 16, NL = (kFewLoads + W - 1) / W;
    extern __shared__ __align__(16) char smem[];  // the groups' weights, then the waves' sums
    float *cpart = reinterpret_cast<float *>(smem + kFewSlots * kFewSlot);
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, kb = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const NibbleMasks nc = nibble_masks();
    const int groups = (a.n + kFewRows - 1) / kFewRows, step = gridDim.x;
    // a group is one piece of memory, a kilobyte a load, but that a row's pieces of 16 bytes come turned by nine places a row: sixteen
    // rows' pieces of one number are in different banks
    int from_row[NL];
    uint32_t from[NL];
#pragma unroll
    for (int i = 0; i < NL; i++) {
        const int at = (wave + W * i) * 64 + lane, row = at / PIECES;
        from_row[i] = row;
        from[i] = row * ROWB + (at % PIECES + 2 * PIECES - 9 * (row % kFewRows)) % PIECES * 16;
    }
    const auto ask = [&](int group, char *slot) {
        const char *w = static_cast<const char *>(a.w) + static_cast<size_t>(group) * kFewSlot;
        const int last = a.n - 1 - group * kFewRows;  // rows past it are it again: what they give is not stored
#pragma unroll
        for (int i = 0; i < NL; i++)
            if (wave + W * i < kFewLoads)
                __builtin_amdgcn_global_load_lds((mid_global_t)(w + (from[i] - max(from_row[i] - last, 0) * ROWB)), (mid_lds_t)(slot + (wave + W * i) * 1024), 16, 0, 0);
    };
    const auto piece = [&](int p) { return (n * PIECES + (p + 9 * n) % PIECES) * 16; };
    const int head_at = piece(9 * wave), q0_at = piece(9 * wave + 1 + 2 * kb), q1_at = piece(9 * wave + 2 + 2 * kb);
    int group = blockIdx.x;
    // the pass's rows, then the first groups: loads come back in order
    half8_t f[8][2];
    const char *frag = staged + wave * kMidSb + lane * 16;
#pragma unroll
    for (int v = 0; v < 8; v++)
#pragma unroll
        for (int p = 0; p < 2; p++) f[v][p] = *reinterpret_cast<const half8_t *>(frag + (v * 2 + p) * kMidFrag);
    const bf16x8_t sx = *reinterpret_cast<const bf16x8_t *>(staged + mid_sums_offset(1, a.k) + wave * kMidSums + lane * 16);
    // this thread's output: row of a group, and of the pass
    const int o_row = (tid >> 2) & 15, o_tok = 4 * (tid >> 6 & 3) + (tid & 3);
    const bool mine = tid < 256 && o_tok < a.n_tok;
    const size_t to = reinterpret_cast<const size_t *>(staged + mid_rows_offset(1, a.k))[o_tok];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < kFewSlots; k++)
        if (group + k * step < groups) ask(group + k * step, smem + k * kFewSlot);
#pragma unroll 1
    for (int b = 0; group < groups; group += step, b = b + 1 == kFewSlots ? 0 : b + 1) {
        char *slot = smem + b * kFewSlot;
        __builtin_amdgcn_sched_barrier(0);
        // this group has landed: all but what this wave has asked for of the ones after it
        constexpr int behind = kFewSlots - 1, whole = kFewLoads / W;
        static_assert(behind * (whole + 1) < 16, "vmcnt");
        if (group + behind * step >= groups) __builtin_amdgcn_s_waitcnt(0x0F70);
        else if (wave < kFewLoads % W) __builtin_amdgcn_s_waitcnt(0x0F70 | behind * (whole + 1));
        else __builtin_amdgcn_s_waitcnt(0x0F70 | behind * whole);
        lds_barrier();
        const mid_bytes_t rows = (mid_bytes_t)(slot);
        const u32x4_t h = *(mid_quad_t)(rows + head_at), q0 = *(mid_quad_t)(rows + q0_at), q1 = *(mid_quad_t)(rows + q1_at);
        uint32_t sc, mn;
        q4k_group_scale_min(make_uint4(h.x, h.y, h.z, h.w), kb, sc, mn);
        float4_t acc = {0.f, 0.f, 0.f, 0.f}, y;
#pragma unroll
        for (int v = 0; v < 8; v++) {
            const u32x4_t &x = (v & 2) ? q1 : q0;
            const uint32_t d0 = (v & 1) ? x.z : x.x, d1 = (v & 1) ? x.w : x.y;
            const half8_t w8 = v < 4 ? weights8<false>(d0, d1, sc & 0xFFu, nc) : weights8<true>(d0, d1, sc >> 8, nc);
#pragma unroll
            for (int p = 0; p < 2; p++) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[v][p], w8, acc, 0, 0, 0);
        }
        const uint32_t am = bf16_pair(mn & 0xFFu, mn >> 8);
        const u32x4_t m3 = {am, am, am, 0u};  // the same two mins against each part
        const float4_t cm = __builtin_amdgcn_mfma_f32_16x16x32_bf16(sx, __builtin_bit_cast(bf16x8_t, m3), float4_t{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        const float d = f16_bits_to_f32(h.x), dmin = f16_bits_to_f32(h.x >> 16);
#pragma unroll
        for (int j = 0; j < 4; j++) y[j] = fmaf(d, acc[j], -dmin * cm[j]);
        *reinterpret_cast<float4_t *>(cpart + (wave * 64 + lane) * 4) = y;
        lds_barrier();
        const int row = group * kFewRows + o_row;
        if (mine && row < a.n) {
            float v = cpart[tid];
#pragma unroll
            for (int w = 1; w < W; w++) v += cpart[w * 256 + tid];
            a.y[to + row] = v + (a.residual ? a.residual[static_cast<size_t>(o_tok) * a.y_stride + row] : 0.f);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (group + kFewSlots * step < groups) ask(group + kFewSlots * step, slot);
    }
}

// ------------------------------------------------------------ the router of a long pass -------
// logits[t][e] = xn[t] . W[e] for float32 rows W (the router's experts and, as one more row, the shared expert's gate)
// against the staged rows of a pass, in the same way: a block keeps 16 R router rows in registers.  A float32 weight enters
// as two binary16 values (hi, and the remainder scaled by 2^11 so that it stays a normal number); x_hi*w_hi + x_lo*w_hi run
// in one accumulator, x_hi*w_lo in a second one that carries the 2^11: about 22 bits of either operand, float32 sums.
// A wave takes 256 columns, w, w + 8, ...: with more than 2048 columns its weights are read again for every tile.
// Bound by the fragments' way from L2, as above, and below some 500 rows by the launches.  Slabs of 64 rows staged through LDS
// took 46 us whatever the pass's height, 27 blocks of them at 150 rows: with its staging and the selection after it the router
// went from 58 to 24 us a layer at 150 rows of 513 x 2048, from 60 to 31 at 512, from 76 to 62 at 2048.
// A fragment of the next tile asked for when this tile's is multiplied: 98.5 to 90.2 us at 4096 rows, 50.4 to 46.7 at 1531; a
// die's blocks on neighbouring tiles: to 80.7 and 43.3 (150 rows 25.1 to 24.6).
// A router row's 64 columns asked for by the lane that multiplies them are sixteen bytes of 64 lines a load, all eight waves' more
// than L1 holds; by four lanes 64 bytes at a time and exchanged through LDS (513 x 2048, with its staging):
// 128 rows 18.6 to 13.7 us, 150 19.1 to 14.5, 512 23.3 to 18.9, 1531 32.8 to 29.0, 4096 60.4 to 56.7.
template <int R>
__global__ __launch_bounds__(512) void router_rows_kernel(const float *W, const float *extra_row, int n_rows, int K, int n_tok, const char *staged, float *logits,
                                                          int logits_stride, int tiles, int per_chunk) {
    constexpr int NW = 8;
    __shared__ __align__(16) float cpart[2][NW][R * 256];
    __shared__ float4_t turn[NW][256];
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, kb = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // Workgroup i goes to die i % 8, each with an L2 of its own: a die takes neighbouring (chunk, rows), so that it reads two or
    // three chunks of the staged rows and not all of them.
    const int count = gridDim.x * gridDim.y, id = blockIdx.x + gridDim.x * blockIdx.y, die = id & 7;
    const int item = die * (count >> 3) + min(die, count & 7) + (id >> 3);
    const int sbs = K / 256, row0 = item % gridDim.x * (16 * R), tile0 = item / gridDim.x * per_chunk;
    const int tile_end = tile0 + per_chunk < tiles ? tile0 + per_chunk : tiles;
    half8_t wh[R][8], wl[R][8];
    auto form = [&](int sb) {  // this lane's 64 columns of every row, read 64 bytes of a row by four lanes and turned in the wave's corner of LDS
        const int lr = lane >> 2, ls = lane & 3;
        // a row's sixteen quads, places exchanged by row: neither the four rows of a store nor the sixteen of a load meet in a bank
        float4_t *mine = turn[wave];
        const int to_x = ((lr & 3) << 2) | (lr >> 2), from_x = ((n & 3) << 2) | (n >> 2);
#pragma unroll
        for (int r = 0; r < R; r++) {
            // rows past the end read the last row (their results are dropped); row n_rows - 1 may live apart
            const int rr = row0 + 16 * r + lr < n_rows ? row0 + 16 * r + lr : n_rows - 1;
            const float *wp = ((extra_row && rr == n_rows - 1) ? extra_row : W + static_cast<size_t>(rr) * K) + sb * 256 + ls * 4;
            float4_t w[16];  // 16 columns of each 64, of all four
#pragma unroll
            for (int i = 0; i < 16; i++) w[i] = *reinterpret_cast<const float4_t *>(wp + (i & 3) * 64 + (i >> 2) * 16);
#pragma unroll
            for (int v = 0; v < 8; v++) {
                if (v % 2 == 0) {
#pragma unroll
                    for (int g = 0; g < 4; g++) mine[lr * 16 + ((g * 4 + ls) ^ to_x)] = w[2 * v + g];
                }
                const float4_t p = mine[n * 16 + ((kb * 4 + v % 2 * 2) ^ from_x)], q = mine[n * 16 + ((kb * 4 + v % 2 * 2 + 1) ^ from_x)];
                // slot order of the eight columns, as the rows were staged: [0, 2, 1, 3, 4, 6, 5, 7]
                const float o[8] = {p.x, p.z, p.y, p.w, q.x, q.z, q.y, q.w};
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const _Float16 hi = static_cast<_Float16>(o[j]);
                    wh[r][v][j] = hi;
                    wl[r][v][j] = static_cast<_Float16>((o[j] - static_cast<float>(hi)) * 2048.f);
                }
            }
        }
    };
    // a fragment of the next tile is asked for as soon as this tile's is multiplied (and the first tile's before the weights are formed)
    half8_t f[8][2];
    auto ask = [&](int tile, int sb, int v) {
        const char *frag = staged + (static_cast<size_t>(tile) * sbs + sb) * kMidSb + lane * 16;
#pragma unroll
        for (int p = 0; p < 2; p++) f[v][p] = *reinterpret_cast<const half8_t *>(frag + (v * 2 + p) * kMidFrag);
    };
    if (wave < sbs) {
#pragma unroll
        for (int v = 0; v < 8; v++) ask(tile0, wave, v);
        form(wave);
    }
    const int o = tid % (R * 256), out_row = row0 + 16 * (o >> 8) + ((o >> 2) & 15), t_in = 4 * (o >> 6 & 3) + (o & 3);
    const bool mine = tid < R * 256 && out_row < n_rows;
    int buf = 0;
    for (int tile = tile0; tile < tile_end; tile++) {
        float4_t ym[R], yl[R];
#pragma unroll
        for (int r = 0; r < R; r++) ym[r] = yl[r] = float4_t{0.f, 0.f, 0.f, 0.f};
        for (int sb = wave; sb < sbs; sb += NW) {
            if (sbs > NW) form(sb);
            const int sb_next = sb + NW < sbs ? sb + NW : wave, tile_next = sb + NW < sbs ? tile : tile + 1 < tile_end ? tile + 1 : tile;
#pragma unroll
            for (int v = 0; v < 8; v++) {
#pragma unroll
                for (int r = 0; r < R; r++) {
                    ym[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[v][0], wh[r][v], ym[r], 0, 0, 0);
                    ym[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[v][1], wh[r][v], ym[r], 0, 0, 0);
                    yl[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(f[v][0], wl[r][v], yl[r], 0, 0, 0);
                }
                ask(tile_next, sb_next, v);
                __builtin_amdgcn_sched_barrier(0);  // (here, and not all of them behind the last product)
            }
        }
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int j = 0; j < 4; j++) cpart[buf][wave][(r * 64 + lane) * 4 + j] = fmaf(yl[r][j], 1.f / 2048.f, ym[r][j]);
        lds_barrier();
        const int t = tile * 16 + t_in;
        if (mine && t < n_tok) {
            float v = cpart[buf][0][o];
#pragma unroll
            for (int w = 1; w < NW; w++) v += cpart[buf][w][o];
            logits[static_cast<size_t>(t) * logits_stride + out_row] = v;
        }
        buf ^= 1;
    }
}

// The same logits for lower passes of 2048 columns, where launches and trips to memory are the time and not the products: a block
// takes 16 R experts and 16 tokens, each of its eight waves an eighth of the columns, on the float32 matrix instruction (nothing
// is split into halves), and no staging launch comes before.  The norm's factor is the last thing applied:
// logit = factor * sum((h * gamma) . w); xn = h * (factor * gamma) for whoever needs the row.  Rows come and are exchanged as above.
// No chain is longer than 16 products: against float64 the logits' error is 0.9 of the row kernel's below 128 rows (rms 4.4e-7 and
// 4.9e-7 of logits of 3.7) and 0.63 of the staged form's.  Of the time, 3 us a block are its 256 KB by way of L1; with sixteen bytes
// of 16 rows a load it took 7.  513 x 2048, before (row kernel to 127 rows, staged from there) and now: 65 rows 15.0
// and 7.8 us, 100 19.9 and 8.0, 121 22.4 and 8.1, 150 14.5 and 10.4, 256 16.7 and 10.6, 300 17.9 and 16.0, 384 19.2 and 16.7.
template <int R, int PER_CU>
__global__ __launch_bounds__(512, 2 * PER_CU) void router_norm_kernel(shv_moe_router_args a, int tiles) {
    constexpr int K = 2048, NW = 8;
    __shared__ __align__(16) float g[K];
    __shared__ float squares[NW][16], gate[NW][16], part[NW][R * 256];
    __shared__ float4_t turn[NW][256];
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 15, kb = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // a die takes neighbouring items, the tiles of 16 experts one behind the other: it reads an eighth of the router and all tokens
    const int count = gridDim.x, die = blockIdx.x & 7, item = die * (count >> 3) + min(die, count & 7) + (blockIdx.x >> 3);
    const int group = item / tiles, row0 = group * 16 * R, t0 = item % tiles * 16, groups = count / tiles;
    const int c0 = wave * 256, lr = lane >> 2, ls = lane & 3;
    // rows past the end read the last one: what they give is dropped
    const float *hp = a.h + static_cast<size_t>(min(t0 + lr, a.n_tok - 1)) * a.h_stride + c0 + 4 * ls, *wp[R];
#pragma unroll
    for (int r = 0; r < R; r++) wp[r] = a.router + static_cast<size_t>(min(row0 + 16 * r + lr, a.n_expert - 1)) * K + c0 + 4 * ls;
    // sixteen columns of each 64 at a time, the next asked for when these are in LDS (two steps ahead: 0.3 us more)
    float4_t h[4], w[R][4], sum[R];
    const auto ask = [&](int q) {
#pragma unroll
        for (int i = 0; i < 4; i++) h[i] = *reinterpret_cast<const float4_t *>(hp + (q * 4 + i) * 16);
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int i = 0; i < 4; i++) w[r][i] = *reinterpret_cast<const float4_t *>(wp[r] + (q * 4 + i) * 16);
    };
    const float4_t gm = *reinterpret_cast<const float4_t *>(a.gamma + c0 + 4 * lane);
    ask(0);
    *reinterpret_cast<float4_t *>(g + c0 + 4 * lane) = gm;  // read by this wave, and behind the barrier by all
    float4_t *mine = turn[wave];
    const int to_x = ((lr & 3) << 2) | (lr >> 2), from_x = ((n & 3) << 2) | (n >> 2);
    float ss = 0.f;
#pragma unroll
    for (int r = 0; r < R; r++) sum[r] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 4; q++) {
        __builtin_amdgcn_sched_barrier(0);
        float4_t x[4], wq[R][4];
#pragma unroll
        for (int i = 0; i < 4; i++) mine[lr * 16 + ((i * 4 + ls) ^ to_x)] = h[i];
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = mine[n * 16 + ((kb * 4 + i) ^ from_x)];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float4_t gi = *reinterpret_cast<const float4_t *>(g + c0 + (q * 4 + kb) * 16 + 4 * i);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                ss = fmaf(x[i][j], x[i][j], ss);
                x[i][j] *= gi[j];
            }
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
#pragma unroll
            for (int i = 0; i < 4; i++) mine[lr * 16 + ((i * 4 + ls) ^ to_x)] = w[r][i];
#pragma unroll
            for (int i = 0; i < 4; i++) wq[r][i] = mine[n * 16 + ((kb * 4 + i) ^ from_x)];
        }
        if (PER_CU > 1) __builtin_amdgcn_sched_barrier(0);  // (not before these are read: two blocks of a compute unit share its registers)
        if (q < 3) ask(q + 1);
#pragma unroll
        for (int r = 0; r < R; r++) {
            float4_t acc[4];
#pragma unroll
            for (int j = 0; j < 4; j++) acc[j] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i][j], wq[r][i][j], acc[j], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < 4; j++) sum[r][j] += (acc[0][j] + acc[1][j]) + (acc[2][j] + acc[3][j]);
        }
    }
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    if (kb == 0) squares[wave][n] = ss;
    // the shared expert's gate, one row more: a token of the tile to each of its blocks
    for (int t = group; a.shared_gate && t < 16; t += groups) {
        const float4_t x = *reinterpret_cast<const float4_t *>(a.h + static_cast<size_t>(min(t0 + t, a.n_tok - 1)) * a.h_stride + c0 + 4 * lane);
        const float4_t v = *reinterpret_cast<const float4_t *>(a.shared_gate + c0 + 4 * lane);
        const float gs = wave_sum_all((x[0] * gm[0] * v[0] + x[1] * gm[1] * v[1]) + (x[2] * gm[2] * v[2] + x[3] * gm[3] * v[3]));
        if (lane == 0) gate[wave][t] = gs;
    }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int j = 0; j < 4; j++) part[wave][(r * 64 + lane) * 4 + j] = sum[r][j];
    __syncthreads();
    const auto over_waves = [](const float *v, int stride) {
        return ((v[0] + v[stride]) + (v[2 * stride] + v[3 * stride])) + ((v[4 * stride] + v[5 * stride]) + (v[6 * stride] + v[7 * stride]));
    };
    const auto factor = [&](int t) { return 1.f / sqrtf(over_waves(&squares[0][t], 16) / static_cast<float>(K) + a.eps); };
    if (tid < R * 256) {
        // value j of a product's lane l: token 4 (l / 16) + j, router row l % 16
        const int r = tid >> 8, t = tid >> 4 & 15, row = row0 + 16 * r + (tid & 15), o = (r * 64 + (t >> 2) * 16 + (tid & 15)) * 4 + (t & 3);
        if (t0 + t < a.n_tok && row < a.n_expert) a.logits[static_cast<size_t>(t0 + t) * (a.n_expert + 1) + row] = over_waves(&part[0][o], R * 256) * factor(t);
    }
    if (a.shared_gate && tid < 16 && tid % groups == group && t0 + tid < a.n_tok)
        a.logits[static_cast<size_t>(t0 + tid) * (a.n_expert + 1) + a.n_expert] = over_waves(&gate[0][tid], 16) * factor(tid);
    // the normed rows themselves, 128 columns at a time by the tile's blocks in turn
    const int t = tid >> 5;
    if (t0 + t < a.n_tok) {
        const float f = factor(t);
        for (int c = group * 128 + (tid & 31) * 4; c < K; c += groups * 128) {
            const float4_t v = *reinterpret_cast<const float4_t *>(a.h + static_cast<size_t>(t0 + t) * a.h_stride + c), gc = *reinterpret_cast<const float4_t *>(g + c);
            float4_t x;
#pragma unroll
            for (int j = 0; j < 4; j++) x[j] = v[j] * (f * gc[j]);
            *reinterpret_cast<float4_t *>(a.xn + static_cast<size_t>(t0 + t) * K + c) = x;
        }
    }
}

// How many of a pass's tiles a block walks, `blocks` of them side by side over the weight rows: as few as blocks on every compute
// unit, one each, leave it (more blocks would form the weights again).
int tiles_a_block(const shv_ctx *ctx, int tiles, int blocks) {
    const int chunks = std::min(std::max(ctx->prop.multiProcessorCount / blocks, 1), tiles);
    return (tiles + chunks - 1) / chunks;
}

template <int R, int S, int W>
int launch(shv_ctx *ctx, const shv_gemv_q4k_args &a, int tiles) {
    constexpr size_t lds = static_cast<size_t>(W) * R * (2048 + 16 * S * SHV_Q4K_BYTES);  // the waves' sums of two tiles, then their weights
    if (lds > 48 * 1024) {
        static std::atomic<bool> raised{false};
        if (!raised.load(std::memory_order_acquire)) {
            SHV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_mid_kernel<R, S, W>), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
            raised.store(true, std::memory_order_release);
        }
    }
    const int blocks = (a.n + 16 * R - 1) / (16 * R);
    const int per = tiles_a_block(ctx, tiles, blocks);
    SHV_LAUNCH(ctx, (gemm_mid_kernel<R, S, W>), dim3(blocks, (tiles + per - 1) / per), dim3(64 * W), lds, a, static_cast<const char *>(ctx->gemm_stage), tiles, per);
    return SHV_OK;
}

int launch_stage(shv_ctx *ctx, const shv_gemv_q4k_args &a, int tiles, float *x_out) {
    const int sbs = a.k / 256;
    // Only the RMSNorm prologue needs the whole row before a column of it: its blocks take column parts until they fill the
    // chip, every one of them summing the whole row
    int parts = sbs;
    if (a.prologue == SHV_PRO_RMSNORM)
        for (parts = 1; parts < sbs && parts * 4 * tiles < 512;) parts *= 2;
    const dim3 grid(parts, 4, tiles), block(256);
    switch (a.prologue) {
        case SHV_PRO_NONE: SHV_LAUNCH(ctx, (gemm_mid_stage_kernel<SHV_PRO_NONE, 0>), grid, block, 0, a, ctx->gemm_stage, tiles, x_out); break;
        case SHV_PRO_RMSNORM:
            if (a.k == 2048) SHV_LAUNCH(ctx, (gemm_mid_stage_kernel<SHV_PRO_RMSNORM, 8>), grid, block, 0, a, ctx->gemm_stage, tiles, x_out);
            else SHV_LAUNCH(ctx, (gemm_mid_stage_kernel<SHV_PRO_RMSNORM, 0>), grid, block, 0, a, ctx->gemm_stage, tiles, x_out);
            break;
        case SHV_PRO_GATED_NORM: SHV_LAUNCH(ctx, (gemm_mid_stage_kernel<SHV_PRO_GATED_NORM, 0>), grid, block, 0, a, ctx->gemm_stage, tiles, x_out); break;
        default: SHV_LAUNCH(ctx, (gemm_mid_stage_kernel<SHV_PRO_MUL_SIGMOID, 0>), grid, block, 0, a, ctx->gemm_stage, tiles, x_out); break;
    }
    return SHV_OK;
}

}  // namespace

// A pass of five to sixteen rows against a matrix of eight groups of rows a block and more (the caller has seen to shv_gemm_q4k_covers).
bool shv_gemm_few_covers(const shv_ctx *ctx, const shv_gemv_q4k_args &a) {
    return ctx->gemm_stage && a.k == 2048 && a.n_tok >= 5 && a.n_tok <= 16 && !a.fold && !a.amax_best && !a.y_flat && a.n >= 8 * kFewRows * 2 * ctx->prop.multiProcessorCount &&
           (a.prologue != SHV_PRO_GATED_NORM || 256 % a.head_dim == 0);
}

int shv_launch_gemm_few(shv_ctx *ctx, const shv_gemv_q4k_args &a) {
    static std::atomic<bool> raised{false};
    if (!raised.load(std::memory_order_acquire)) {
        SHV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_few_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kFewLds)));
        raised.store(true, std::memory_order_release);
    }
    const int rc = launch_stage(ctx, a, 1, nullptr);
    if (rc != SHV_OK) return rc;
    SHV_LAUNCH(ctx, gemm_few_kernel, dim3(2 * ctx->prop.multiProcessorCount), dim3(512), kFewLds, a, static_cast<const char *>(ctx->gemm_stage));
    return SHV_OK;
}

// From nine rows, where the kernels that form every weight once for up to eight of them end, to 512, but for the passes that
// shv_one_group names.  Past 512 gemm_long.hip's blocks read less from L2.
bool shv_gemm_mid_covers(const shv_ctx *ctx, const shv_gemv_q4k_args &a) {
    if (!ctx->gemm_stage || (a.k != 2048 && a.k != 4096) || a.n_tok < 9 || a.n_tok > 512) return false;
    if (shv_one_group(a.n_tok)) return false;
    if (a.prologue == SHV_PRO_GATED_NORM && 256 % a.head_dim != 0) return false;
    return mid_bytes((a.n_tok + 15) / 16, a.k) <= static_cast<size_t>(shv_ctx::kGemmStageBytes);
}

int shv_launch_gemm_mid(shv_ctx *ctx, const shv_gemv_q4k_args &a) {
    if (shv_gemm_few_covers(ctx, a)) return shv_launch_gemm_few(ctx, a);
    const int tiles = (a.n_tok + 15) / 16;
    const int rc = launch_stage(ctx, a, tiles, nullptr);
    if (rc != SHV_OK) return rc;
    // 64 weight rows a block where the columns are 2048; of 4096, 32 fill the registers as well, and a single tile of
    // activations is quicker over twice the blocks (10.7 against 12.1 us of 16 rows)
    if (a.k == 2048) return launch<4, 1, 8>(ctx, a, tiles);
    return tiles == 1 ? launch<1, 2, 8>(ctx, a, tiles) : launch<2, 2, 8>(ctx, a, tiles);
}

// The router of a pass of many rows: xn = rmsnorm(h) * gamma written as float32 (and staged, by the form that multiplies staged
// rows), then every token's n_expert (+ 1, the shared expert's gate) logits on the matrix cores.
// Which form, of 2048 columns: the float32 blocks while one a compute unit is enough, of 16 experts or of 32 (150 rows of 512 experts,
// 256 compute units: 11.5 and 10.4 us), and by turns while three are (384 rows 16.7 us, staged 19.2); at 512 rows they lose, 20.3 to 18.9.
// Below, the row kernel goes through its tokens a few at a time (17 rows 7.8 us to 7.6, 32 10.4 to 7.7, 48 12.5 to 7.8) and is quicker
// of 16; shv_one_group's passes stay with it.
namespace {

bool router_aligned(const shv_moe_router_args &a) {
    return a.gamma && a.xn && a.h_stride % 4 == 0 && shv_aligned16(a.h) && shv_aligned16(a.gamma) && shv_aligned16(a.xn) && shv_aligned16(a.router) &&
           (!a.shared_gate || shv_aligned16(a.shared_gate));
}

enum class RouterNorm { none, sixteen, thirty_two, sixteen_by_turns };
RouterNorm router_norm_form(const shv_ctx *ctx, const shv_moe_router_args &a) {
    const long long cus = ctx->prop.multiProcessorCount, tiles = (a.n_tok + 15) / 16, ones = (a.n_expert + 15) / 16 * tiles, twos = (a.n_expert + 31) / 32 * tiles;
    if (a.n_embd != 2048 || a.n_tok < 17 || shv_one_group(a.n_tok) || ones > 3 * cus) return RouterNorm::none;
    return ones <= cus ? RouterNorm::sixteen : twos <= cus ? RouterNorm::thirty_two : RouterNorm::sixteen_by_turns;
}

}  // namespace

bool shv_router_rows_covers(const shv_ctx *ctx, const shv_moe_router_args &a) {
    if (!router_aligned(a)) return false;
    if (router_norm_form(ctx, a) != RouterNorm::none) return true;
    if (!ctx->gemm_stage || a.n_tok < 128 || a.n_embd % 256 != 0 || a.n_embd < 256) return false;
    return mid_bytes((a.n_tok + 15) / 16, a.n_embd) <= static_cast<size_t>(shv_ctx::kGemmStageBytes);
}

int shv_launch_router_rows(shv_ctx *ctx, const shv_moe_router_args &a) {
    const int tiles = (a.n_tok + 15) / 16;
    const dim3 ones((a.n_expert + 15) / 16 * tiles), twos((a.n_expert + 31) / 32 * tiles), block(512);
    switch (router_norm_form(ctx, a)) {
        case RouterNorm::sixteen: SHV_LAUNCH(ctx, (router_norm_kernel<1, 1>), ones, block, 0, a, tiles); return SHV_OK;
        case RouterNorm::thirty_two: SHV_LAUNCH(ctx, (router_norm_kernel<2, 1>), twos, block, 0, a, tiles); return SHV_OK;
        case RouterNorm::sixteen_by_turns: SHV_LAUNCH(ctx, (router_norm_kernel<1, 2>), ones, block, 0, a, tiles); return SHV_OK;
        case RouterNorm::none: break;
    }
    shv_gemv_q4k_args g{};
    g.x = a.h;
    g.gamma = a.gamma;
    g.k = a.n_embd;
    g.n_tok = a.n_tok;
    g.prologue = SHV_PRO_RMSNORM;
    g.eps = a.eps;
    g.x_stride = a.h_stride;
    const int n_rows = a.n_expert + (a.shared_gate ? 1 : 0);
    const int rc = launch_stage(ctx, g, tiles, a.xn);
    if (rc != SHV_OK) return rc;
    constexpr int R = 2;
    const int blocks = (n_rows + 16 * R - 1) / (16 * R), per = tiles_a_block(ctx, tiles, blocks);
    SHV_LAUNCH(ctx, (router_rows_kernel<R>), dim3(blocks, (tiles + per - 1) / per), dim3(512), 0, a.router, a.shared_gate, n_rows, a.n_embd, a.n_tok,
               static_cast<const char *>(ctx->gemm_stage), a.logits, a.n_expert + 1, tiles, per);
    return SHV_OK;
}
