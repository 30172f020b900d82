// The experts of a pass of middling length, grouped by expert: tens to hundreds of rows, whose lists hold a few tokens an
// expert.  Such a pass reads every expert it touches once and multiplies it with little, so what bounds it is HBM: all
// 512 experts of a layer are 604 MB of gate and up rows and 302 MB of down rows.  The kernels of moe_grouped.hip bring an
// expert's tokens through LDS for blocks of eight waves, one block a compute unit, and over short lists are a chain of
// slab barriers (217 us for the gate/up rows of a 150-row pass, 2.8 TB/s).  Here no wave waits for another:
//   a wave      = kR = 4 row tiles of 16 weight rows against up to 16 listed tokens; its loads put 9 KB chunks of weights
//                 into its own LDS a chunk ahead of the products, the tokens' operands come to registers; no barrier
//   products    = v_mfma_f32_16x16x32_f16, tokens x weights: a lane holds one weight row (its scales, its d) and four
//                 token rows; the weights are the whole numbers n * sc, exact in binary16, one accumulator a super-block
//   operands    = a token's values scaled by a power of two, as two binary16 parts (binary16_parts); what a token's products
//                 come to is scaled back where they leave.  A token's own row has one exponent, known when it is staged; a
//                 SwiGLU row is written by sixteen waves that know their sub-block's alone, and the waves that read it bring
//                 its sub-blocks to the row's largest, 2^-k being exact.  Error of a layer's outputs against float64, whatever
//                 the activations' size: 0.5e-6 to 0.7e-6 (slot by slot 4.2e-6; without the exponents 240e-6 at xn of 0.02)
//   up to eight tokens: the high and the low parts of a token are two rows of ONE operand (a product for both parts,
//                 the halves of a result in neighbouring registers of a lane); nine to sixteen: an operand for each part
//                 (the parts of a sum are added at its end in the one, along it in the other: the lists come in order of
//                 their tokens, so that a pair meets the same one from call to call)
//   min term    = per super-block one v_mfma_f32_16x16x16_bf16 a part of the sub-blocks' sums of x (float32 values, each
//                 exactly three bfloat16 ones) with the rows' mins (whole numbers), times the row's dmin
// Gate/up of a 150-row pass 217 -> 131 us (4.4 TB/s), down 115 -> 64.  The chunks' loads alone take 100 us of the 131, the
// arithmetic alone 87; two waves a SIMD hide most of one under the other.  The same waves as a persistent walk over a work
// list, the next unit's loads behind the last one's products, measured the same (the waits are not at a unit's ends).
#include <type_traits>

#include "moe_staged.hpp"
#include "shv_internal.hpp"

namespace {

using namespace shv;
using namespace shv_moe;

constexpr int kR = 4;          // weight row tiles a wave multiplies together
constexpr int kListThreads = 256;
constexpr int kDownUnits = 4;  // 64-row units of the down projection a wave takes with the same tokens

// A chunk is 9 KB of weights that nine loads of a wave bring into its own LDS.  A load takes 64 bytes of each of sixteen
// rows, neighbouring loads the neighbouring bytes, so lines come through L1 once: lanes that fetch their own header and
// payload of a super-block, 12 loads where these are 9, reach 3.5 TB/s with no arithmetic at all, chunks 5.2 to 5.9.
//   S 4: four super-blocks of one row tile (576 bytes a row, 5.9 TB/s), where the tokens' operands of four super-blocks
//        fit the registers (eight tokens)
//   S 2: two super-blocks of two row tiles (288 bytes a row, 5.2 TB/s; whole rows of a down projection, 6.0)
// Piece p of 16 bytes of row n of a tile (9 S a row: header, 8 of payload, S times) lies at p * 256 + n * 16 of the tile's
// part: sixteen rows' pieces are neighbours, which is how they are read.  With S 2 a tile's part is the 4 KB at
// t * 4096, pieces 16 and 17 at 8192 + t * 512.
constexpr int kChunk = 9 * 1024;
constexpr int kRing = 2 * kChunk;  // a wave's LDS: a chunk being multiplied, the next on its way

typedef const __attribute__((address_space(1))) void *global_ptr_t;
typedef __attribute__((address_space(3))) void *lds_ptr_t;
typedef const __attribute__((address_space(3))) char *lds_bytes_t;
typedef const __attribute__((address_space(3))) u32x4_t *lds_quad_t;

// w: the first row of the chunk's (first) tile, at the first of its super-blocks (the same in every lane).  on false: as many
// loads, all of the chunk's first lines.  A wave's last chunk is waited for by their count; with the whole first chunk asked for
// again behind it a ninth of what the kernels read was read for nothing: a layer of 66 rows 171 to 168 us, of 150 rows 226 to
// 223, of 700 rows 404 to 399 (prompts of 65, 150 and 700 rows of 16 layers 3725 to 3679 us, 5000 to 4938, 10793 to 10723).
// A branch around the loads costs the gate/up kernel 156 spills.
template <int ROWB, int S>
__device__ __forceinline__ void ask_chunk(const char *w, char *lds, int lane, bool on = true) {
    const int n = lane & 15, kb = lane >> 4;
    const uint32_t at = on ? n * ROWB + kb * 16 : 0;
    if constexpr (S == 4) {
#pragma unroll
        for (int i = 0; i < 9; i++) __builtin_amdgcn_global_load_lds((global_ptr_t)(w + i * 64 + at), (lds_ptr_t)(lds + i * 1024), 16, 0, 0);
    } else {
        const uint32_t tail = on ? ((kb >> 1) * 16 + n) * ROWB + 256 + (kb & 1) * 16 : 0;
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                __builtin_amdgcn_global_load_lds((global_ptr_t)(w + t * 16 * ROWB + i * 64 + at), (lds_ptr_t)(lds + t * 4096 + i * 1024), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((global_ptr_t)(w + tail), (lds_ptr_t)(lds + 8192), 16, 0, 0);
    }
}

// header and the 32 payload bytes of the lane's group (kb) of super-block s of the chunk's tile t
template <int S>
struct TileSb {
    u32x4_t h, q0, q1;
    // head: ring slot + n * 16; body: head + kb * 512; tail: body, with S 2 moved for the group that lies behind both tiles
    __device__ __forceinline__ void read(lds_bytes_t head, lds_bytes_t body, lds_bytes_t tail, int t, int s) {
        h = *(lds_quad_t)(head + t * 4096 + s * (9 * 256));
        lds_bytes_t q = S == 2 && s == 1 ? tail + t * 512 : body + t * 4096 + s * (9 * 256);
        if (S == 2 && s == 1) {
            q0 = *(lds_quad_t)(q);
            q1 = *(lds_quad_t)(q + 256);
        } else {
            q0 = *(lds_quad_t)(q + 256);
            q1 = *(lds_quad_t)(q + 512);
        }
    }
};

struct AsStaged {};

// A wave's share of one expert: row tiles of K columns against the tokens whose operands the lane reads at tok (and sums
// at sum).  A unit is four tiles, w0 and w1 the first rows of its two pairs (the same in every lane); `units` of them
// follow one another unit_bytes apart.  done(unit, y) takes a unit's sums: y[r][j] of lane (n, kb) is weight row n of
// tile r against operand row 4 kb + j.
// settle(b, sx) brings operands that are not all of one exponent to one, when they have come (AsStaged: they are).
// PARTS 1: operand row 2 t + p is part p of token t (up to eight); PARTS 2: operand row t, parts one after the other.
// A lane (n, kb) of a tile takes group kb of row n's super-blocks, so one decode of the header serves a super-block.  The
// tokens' operands of S super-blocks stay in registers over the chunks that meet them.
template <int K, int PARTS, int S, typename Settle, typename Done>
__device__ __forceinline__ void stream_tiles(const char *w0, const char *w1, int units, int unit_bytes, char *ring, const char *staged, uint32_t tok, const char *sums, uint32_t sum,
                                             Settle &&settle, Done &&done) {
    constexpr int SBS = K / SHV_Q4K_BLOCK, ROWB = SBS * SHV_Q4K_BYTES, STEPS = SBS / S;
    constexpr int TC = 4 / S, CHUNKS = kR / TC;  // tiles a chunk, chunks a step
    static_assert((S == 2 || S == 4) && CHUNKS % 2 == 0, "chunk shape");
    const int lane = threadIdx.x & 63, n = lane & 15, kb = lane >> 4;
    const NibbleMasks nc = nibble_masks();
    half8_t b[S][8][PARTS];
    short4_t sx[S][PARTS];
    auto ask_tok = [&](int sb, int s) {
#pragma unroll
        for (int v = 0; v < 8; v++)
#pragma unroll
            for (int p = 0; p < PARTS; p++)
                b[s][v][p] = *reinterpret_cast<const half8_t *>(staged + sb * (8 * kStSubBytes) + (tok + v * 128 + p * 64));
#pragma unroll
        for (int p = 0; p < PARTS; p++) sx[s][p] = *reinterpret_cast<const short4_t *>(sums + sb * kListSumBytes + (sum + p * 32));
    };
    // where chunk c of a step begins: tiles TC c .. of the unit
    auto chunk_at = [&](int st, int c) {
        const char *w = c * TC >= 2 ? w1 : w0;
        return w + ((c * TC) & 1) * (16 * ROWB) + st * (S * SHV_Q4K_BYTES);
    };
    if constexpr (!std::is_same_v<Settle, AsStaged>) {
        // the operands first, settled while the first chunk is on its way (with the second chunk asked for here as well the
        // loop has a case more, and 51 registers of the sixteen-token kernel go to memory where 27 do)
        static_assert(STEPS == 1, "operands that stay");
#pragma unroll
        for (int s = 0; s < S; s++) ask_tok(s, s);
        __builtin_amdgcn_sched_barrier(0);
        ask_chunk<ROWB, S>(chunk_at(0, 0), ring, lane);
        __builtin_amdgcn_s_waitcnt(0x0F79);  // vmcnt(9)
        __builtin_amdgcn_sched_barrier(0);
        settle(b, sx);
    } else {
        ask_chunk<ROWB, S>(chunk_at(0, 0), ring, lane);
#pragma unroll
        for (int s = 0; s < S; s++) ask_tok(s, s);
    }
    float4_t y[kR];
#pragma unroll 1
    for (int u = 0; u < units; u++) {
#pragma unroll
        for (int r = 0; r < kR; r++) y[r] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int st = 0; st < STEPS; st++) {
#pragma unroll
            for (int c = 0; c < CHUNKS; c++) {
                // the chunk after this one; behind the last of the last unit loads that nobody reads
                const bool more = c + 1 < CHUNKS || st + 1 < STEPS || u + 1 < units;
                const char *next;
                if (c + 1 < CHUNKS) next = chunk_at(st, c + 1);
                else if (st + 1 < STEPS) next = chunk_at(st + 1, 0);
                else {
                    if (u + 1 < units) w0 += unit_bytes, w1 += unit_bytes;
                    next = chunk_at(0, 0);
                }
                const int sn = st + 1 < STEPS ? S * (st + 1) : 0;  // and the super-blocks whose operands it meets
                __builtin_amdgcn_sched_barrier(0);  // everything read from the slot the next chunk goes to has been used
                ask_chunk<ROWB, S>(next, ring + ((c + 1) & 1) * kChunk, lane, more);
                __builtin_amdgcn_s_waitcnt(0x0F79);  // vmcnt(9), all but those nine: this chunk has landed, and the tokens' operands
                __builtin_amdgcn_sched_barrier(0);
                const lds_bytes_t head = (lds_bytes_t)(ring + (c & 1) * kChunk) + n * 16, body = head + kb * 512;
                const lds_bytes_t tail = S == 4 ? body : kb == 3 ? head + 8192 : body + 10 * 256;
                TileSb<S> cur, nxt;
                cur.read(head, body, tail, 0, 0);
#pragma unroll
                for (int s = 0; s < S; s++) {
#pragma unroll
                    for (int t = 0; t < TC; t++) {
                        const int i = s * TC + t + 1;
                        // (with S 2 the second super-block's payload of the first three groups lies in the tiles' parts)
                        if (i < 4) nxt.read(head, body, S == 2 && i % TC == 1 ? (kb == 3 ? tail : tail + 4096 - 512) : tail, i % TC, i / TC);
                        const int r = TC * c + t;
                        const uint4 hdr = make_uint4(cur.h.x, cur.h.y, cur.h.z, cur.h.w);
                        uint32_t sc, mn;
                        q4k_group_scale_min(hdr, kb, sc, mn);
                        float4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int v = 0; v < 8; v++) {
                            const u32x4_t &d = (v & 2) ? cur.q1 : cur.q0;
                            const uint32_t d0 = (v & 1) ? d.z : d.x, d1 = (v & 1) ? d.w : d.y;
                            const half8_t w8 = v < 4 ? weights8<false>(d0, d1, sc & 0xFFu, nc) : weights8<true>(d0, d1, sc >> 8, nc);
#pragma unroll
                            for (int p = 0; p < PARTS; p++) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[s][v][p], w8, acc, 0, 0, 0);
                        }
                        // the super-block ends: its sums take the row's d, its mins the row's dmin
                        const u32x2_t am = static_cast<u32x2_t>(bf16_pair(mn & 0xFFu, mn >> 8));
                        float4_t cm = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int p = 0; p < PARTS; p++) cm = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(sx[s][p], __builtin_bit_cast(short4_t, am), cm, 0, 0, 0);
                        const float d = f16_bits_to_f32(hdr.x), dmin = f16_bits_to_f32(hdr.x >> 16);
#pragma unroll
                        for (int j = 0; j < 4; j++) y[r][j] = fmaf(-dmin, cm[j], fmaf(d, acc[j], y[r][j]));
                        cur = nxt;
                    }
                    if (c + 1 == CHUNKS && STEPS > 1) ask_tok(sn + s, s);  // this super-block's operands are done with
                }
            }
        }
        done(u, y);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load may write LDS after the wave has moved on
}

// Which expert and which of its rows a block takes.  The shared expert's blocks come first, TOK tokens each; the routed
// experts follow in the order of the group workspace (longest list first), every one with all of its list.
struct ListUnit {
    int expert;   // -1: the shared expert
    int part;     // of the expert's rows, `parts` blocks
    int first, count;  // positions in the expert's list (routed) or token numbers (shared)
};
template <int TOK>
__device__ __forceinline__ ListUnit list_unit(int b, int parts, int n_expert, int n_tok, int n_used, const int32_t *group) {
    ListUnit u;
    const int shared = parts * ((n_tok + TOK - 1) / TOK);
    if (b >= shared) {
        b -= shared;
        // the same in every lane, and known to be: what is reached from here has scalar addresses
        u.expert = __builtin_amdgcn_readfirstlane(group[n_expert + 1 + n_tok * n_used + b / parts]);
        u.part = b % parts;
        u.first = __builtin_amdgcn_readfirstlane(group[u.expert]);
        u.count = __builtin_amdgcn_readfirstlane(group[u.expert + 1]) - u.first;
    } else {
        u.expert = -1;
        u.part = b % parts;
        u.first = (b / parts) * TOK;
        u.count = n_tok - u.first < TOK ? n_tok - u.first : TOK;
    }
    return u;
}

// The pair (token * (n_used + 1) + slot) at place i of the pass that begins at t0, of m; a place past the list repeats
// the first (its products are not stored).
__device__ __forceinline__ int pair_at(const ListUnit &u, int t0, int i, int m, int n_used, int n_expert, const int32_t *group) {
    const int at = u.first + t0 + (i < m ? i : 0);
    return u.expert < 0 ? at * (n_used + 1) + n_used : group[n_expert + 1 + at];
}

// One pass of a gate/up wave over m <= 8 (PARTS 1) or m <= 16 (PARTS 2) tokens: rows row0 .. + 31 of gate and up.  act
// goes out as the operands the down projection reads (the 32 rows are one sub-block of them), or as floats.
template <int K, int PARTS>
__device__ __forceinline__ void up_list_pass(const shv_moe_up_args &a, const char *gate, const char *up, char *ring, const char *staged, const ListUnit &u, int t0, int m, int row0,
                                             char *act_sums) {
    const int lane = threadIdx.x & 63, n = lane & 15, kb = lane >> 4;
    const int pair = pair_at(u, t0, PARTS == 1 ? n >> 1 : n, m, a.n_used, a.n_expert, a.group);
    const int t = pair / (a.n_used + 1);
    const int part = PARTS == 1 ? n & 1 : 0;
    const uint32_t tok = t * ((K / 32) * kStSubBytes) + kb * 16 + part * 64;
    const uint32_t sum = t * (K / 256 * kListSumBytes) + part * 32 + kb * 8;
    const int exponent = reinterpret_cast<const int32_t *>(staged + list_exps_offset(a.n_tok, K))[t];
    const int row = row0 + n, sub = row0 >> 5;
    uint8_t *act_exps = reinterpret_cast<uint8_t *>(act_sums + list_act_exps_offset(static_cast<long long>(a.n_tok) * (a.n_used + 1), a.ffn));
    // column n (and n + 16) of the sub-block: its slot of [0, 2, 1, 3, 4, 6, 5, 7]
    const int p8 = n & 7, slot = (p8 & 4) | ((p8 & 1) << 1) | ((p8 & 2) >> 1);
    stream_tiles<K, PARTS, PARTS == 1 ? 4 : 2>(gate, up, 1, 0, ring, staged, tok, staged + staged_sums_offset(a.n_tok, K), sum,
                                                  AsStaged(), [&](int, const float4_t (&y)[kR]) {
        constexpr int NT = PARTS == 1 ? 2 : 4;  // tokens whose sums this lane holds
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const int i = NT * kb + j;
            const int back = __shfl(exponent, PARTS == 1 ? 2 * i : i, 64) - kListOne;
            float v[2];
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const float gv = ldexpf(PARTS == 1 ? y[r][2 * (j & 1)] + y[r][2 * (j & 1) + 1] : y[r][j], back);
                const float uv = ldexpf(PARTS == 1 ? y[2 + r][2 * (j & 1)] + y[2 + r][2 * (j & 1) + 1] : y[2 + r][j], back);
                v[r] = gv * sigmoid_exact(gv) * uv;
            }
            const size_t to = static_cast<size_t>(__shfl(pair, PARTS == 1 ? 2 * i : i, 64));
            if (!a.act_packed) {
                if (i < m) {
#pragma unroll
                    for (int r = 0; r < 2; r++) a.act[to * a.ffn + row + 16 * r] = v[r];
                }
                continue;
            }
            const float sum32 = group_sum<16>(v[0] + v[1]);
            const int e = biased_exponent(max16_all(fmaxf(fabsf(v[0]), fabsf(v[1]))));
            if (i < m) {
                char *at = reinterpret_cast<char *>(a.act) + to * (a.ffn / 32) * kStSubBytes + list_block(sub, n >> 3) + slot * 2;
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    _Float16 hi, lo;
                    binary16_parts(ldexpf(v[r], kListOne - e), hi, lo);
                    *reinterpret_cast<_Float16 *>(at + r * 256) = hi;
                    *reinterpret_cast<_Float16 *>(at + r * 256 + 64) = lo;
                }
                if (n == 0) act_exps[to * (a.ffn / 32) + sub] = static_cast<uint8_t>(e);
                if (n == 0) list_sum_put(act_sums + (to * (a.ffn / 256) + (sub >> 3)) * kListSumBytes, sub, sum32);
            }
        }
    });
}

// grid: parts * (ceil(n_tok / TOK) + n_expert) blocks of four waves, parts = ffn / 128: a wave takes 32 gate rows and the
// up rows of the same numbers.  K = n_embd.
template <int K, int TOK>
__global__ __launch_bounds__(kListThreads, 2) void moe_up_list_kernel(shv_moe_up_args a, const char *staged, char *act_sums) {
    extern __shared__ __align__(16) char smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const ListUnit u = list_unit<TOK>(blockIdx.x, a.ffn / 128, a.n_expert, a.n_tok, a.n_used, a.group);
    constexpr size_t row_bytes = static_cast<size_t>(K / SHV_Q4K_BLOCK) * SHV_Q4K_BYTES;
    const int row0 = u.part * 128 + wave * 32;
    const size_t at = (static_cast<size_t>(u.expert < 0 ? 0 : u.expert) * a.ffn + row0) * row_bytes;
    const char *gate = static_cast<const char *>(u.expert < 0 ? a.gate_sh : a.gate_exps) + at;
    const char *up = static_cast<const char *>(u.expert < 0 ? a.up_sh : a.up_exps) + at;
    char *ring = smem + wave * kRing;
    for (int t0 = 0; t0 < u.count; t0 += TOK) {
        const int m = u.count - t0 < TOK ? u.count - t0 : TOK;
        if (TOK == 8 || m <= 8) up_list_pass<K, 1>(a, gate, up, ring, staged, u, t0, m, row0, act_sums);
        else up_list_pass<K, 2>(a, gate, up, ring, staged, u, t0, m, row0, act_sums);
    }
}

template <int K, int PARTS>
__device__ __forceinline__ void down_list_pass(const shv_moe_down_args &a, const char *base, char *ring, const char *act_sums, const ListUnit &u, int t0, int m, int row0) {
    constexpr int ROWB = K / SHV_Q4K_BLOCK * SHV_Q4K_BYTES;
    const int lane = threadIdx.x & 63, n = lane & 15, kb = lane >> 4;
    const int pair = pair_at(u, t0, PARTS == 1 ? n >> 1 : n, m, a.n_used, a.n_expert, a.group);
    const int part = PARTS == 1 ? n & 1 : 0;
    const uint32_t tok = pair * ((K / 32) * kStSubBytes) + kb * 16 + part * 64;
    const uint32_t sum = pair * (K / 256 * kListSumBytes) + part * 32 + kb * 8;
    static_assert(K == 512, "sixteen sub-blocks, an exponent of a byte each");
    const u32x4_t exps = *reinterpret_cast<const u32x4_t *>(act_sums + list_act_exps_offset(static_cast<long long>(a.n_tok) * (a.n_used + 1), K) + static_cast<size_t>(pair) * 16);
    int exponent = 0;  // the row's: its largest sub-block's
    auto settle = [&](half8_t(&b)[2][8][PARTS], short4_t(&sx)[2][PARTS]) {
#pragma unroll
        for (int i = 0; i < 16; i++) exponent = max(exponent, static_cast<int>(exps[i >> 2] >> (8 * (i & 3)) & 255));
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const uint32_t two = ((kb & 2) ? exps[2 * s + 1] : exps[2 * s]) >> (16 * (kb & 1));  // of this lane's sub-blocks 8 s + 2 kb and the next
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int down = static_cast<int>(two >> (8 * h) & 255) - exponent;
                const _Float16 f = static_cast<_Float16>(ldexpf(1.f, max(down, -24)));
#pragma unroll
                for (int v = 4 * h; v < 4 * h + 4; v++)
#pragma unroll
                    for (int p = 0; p < PARTS; p++) b[s][v][p] *= static_cast<half8_t>(f);
                if (__any(down < -24)) {  // binary16 knows no smaller power
                    const _Float16 f2 = static_cast<_Float16>(ldexpf(1.f, min(down + 24, 0)));
#pragma unroll
                    for (int v = 4 * h; v < 4 * h + 4; v++)
#pragma unroll
                        for (int p = 0; p < PARTS; p++) b[s][v][p] *= static_cast<half8_t>(f2);
                }
            }
#pragma unroll
            for (int p = 0; p < PARTS; p++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    sx[s][p][i] = static_cast<short>(__float_as_uint(ldexpf(__uint_as_float(static_cast<uint32_t>(static_cast<uint16_t>(sx[s][p][i])) << 16), kListOne - exponent)) >> 16);
        }
    };
    stream_tiles<K, PARTS, 2>(base, base + 32 * ROWB, kDownUnits, 16 * kR * ROWB, ring, reinterpret_cast<const char *>(a.act), tok, act_sums, sum, settle,
                              [&](int unit, const float4_t (&y)[kR]) {
        constexpr int NT = PARTS == 1 ? 2 : 4;
#pragma unroll
        for (int j = 0; j < NT; j++) {
            const int i = NT * kb + j;
            const size_t to = static_cast<size_t>(__shfl(pair, PARTS == 1 ? 2 * i : i, 64));
            const int back = __shfl(exponent, PARTS == 1 ? 2 * i : i, 64) - kListOne;
            float *dst = a.pairs + to * a.n_embd + row0 + unit * 16 * kR + n;
            if (i < m) {
#pragma unroll
                for (int r = 0; r < kR; r++) dst[16 * r] = ldexpf(PARTS == 1 ? y[r][2 * (j & 1)] + y[r][2 * (j & 1) + 1] : y[r][j], back);
            }
        }
    });
}

// grid: parts * (ceil(n_tok / TOK) + n_expert) blocks of four waves, parts = n_embd / (256 kDownUnits): a wave takes
// kDownUnits times 64 output rows.  K = ffn; act is operands (act_packed).
template <int K, int TOK>
__global__ __launch_bounds__(kListThreads, 2) void moe_down_list_kernel(shv_moe_down_args a, const char *act_sums) {
    extern __shared__ __align__(16) char smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const ListUnit u = list_unit<TOK>(blockIdx.x, a.n_embd / (4 * 16 * kR * kDownUnits), a.n_expert, a.n_tok, a.n_used, a.group);
    constexpr size_t row_bytes = static_cast<size_t>(K / SHV_Q4K_BLOCK) * SHV_Q4K_BYTES;
    const int row0 = (u.part * 4 + wave) * (16 * kR * kDownUnits);
    const char *base = static_cast<const char *>(u.expert < 0 ? a.down_sh : a.down_exps) +
                       (static_cast<size_t>(u.expert < 0 ? 0 : u.expert) * a.n_embd + row0) * row_bytes;
    char *ring = smem + wave * kRing;
    for (int t0 = 0; t0 < u.count; t0 += TOK) {
        const int m = u.count - t0 < TOK ? u.count - t0 : TOK;
        if (TOK == 8 || m <= 8) down_list_pass<K, 1>(a, base, ring, act_sums, u, t0, m, row0);
        else down_list_pass<K, 2>(a, base, ring, act_sums, u, t0, m, row0);
    }
}

}  // namespace

// Where the lists are short enough for these kernels, and how many tokens a wave takes at a time (0: not these kernels).
// Gate/up + down of one layer over 512 experts, top 10, us with the lists made: per-(token, slot) or grouped kernels / eight
// tokens a time / sixteen
//   37 rows (0.7 pairs an expert)  120 / 118 / 132      300 rows (5.9)  380 / 280 / 284
//   64 (1.25)                      185 / 158 / 168      400 (7.8)       400 / 321 / 312
//   150 (2.9)                      352 / 215 / 229      600 (11.7)      453 / 413 / 379
//   200 (3.9)                      366 / 240 / 247      800 (15.6)      480 / 510 / 460      1000 (19.5)  494 / 608 / 542
// (Taken with operands as they were and no exponents; with them 66 rows 182, 150 rows 224, 300 rows 270, 400 rows 315, 750 rows
// 431, a part in a hundred to a part in thirty more: the line at 15 pairs an expert is as good as level.)
// Below the first line most experts a pass touches are touched once, and reading them row by row costs no list.  Passes of 40
// to 64 rows would be a seventh faster here and no less exact (5e-7 against 4e-6 of a layer's outputs, against float64): they
// keep the other kernels so that a short prompt's results stay the ones they were, since where a token's tenth expert and
// its eleventh are level its choice is carried through every token decoded after it.
int shv_moe_list_tokens(int n_tok, int n_used, int n_expert) {
    const long long pairs = static_cast<long long>(n_tok) * n_used;
    if (n_tok <= 64 || 4 * pairs < 3ll * n_expert || pairs > 15ll * n_expert) return 0;
    return pairs <= 6ll * n_expert ? 8 : 16;
}

// The gate/up products of a pass whose lists are made and whose rows are staged (moe_grouped.hip launches both).
template <typename Kern>
static int raise_lds(Kern kern) {
    SHV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, 4 * kRing));
    return SHV_OK;
}
template <int TOK>
static int launch_up(shv_ctx *ctx, const shv_moe_up_args &a) {
    static const int raised = raise_lds(&moe_up_list_kernel<2048, TOK>);
    if (raised != SHV_OK) return raised;
    const int parts = a.ffn / 128, tiles = (a.n_tok + TOK - 1) / TOK;
    SHV_LAUNCH(ctx, (moe_up_list_kernel<2048, TOK>), dim3(parts * (tiles + a.n_expert)), dim3(kListThreads), 4 * kRing, a, static_cast<const char *>(ctx->gemm_stage),
               reinterpret_cast<char *>(ctx->gemm_part));
    return SHV_OK;
}
template <int TOK>
static int launch_down(shv_ctx *ctx, const shv_moe_down_args &a) {
    static const int raised = raise_lds(&moe_down_list_kernel<512, TOK>);
    if (raised != SHV_OK) return raised;
    const int parts = a.n_embd / (4 * 16 * kR * kDownUnits), tiles = (a.n_tok + TOK - 1) / TOK;
    SHV_LAUNCH(ctx, (moe_down_list_kernel<512, TOK>), dim3(parts * (tiles + a.n_expert)), dim3(kListThreads), 4 * kRing, a, reinterpret_cast<const char *>(ctx->gemm_part));
    return SHV_OK;
}

int shv_launch_moe_up_lists(shv_ctx *ctx, const shv_moe_up_args &a) {
    return shv_moe_list_tokens(a.n_tok, a.n_used, a.n_expert) == 8 ? launch_up<8>(ctx, a) : launch_up<16>(ctx, a);
}

int shv_launch_moe_down_lists(shv_ctx *ctx, const shv_moe_down_args &a) {
    return shv_moe_list_tokens(a.n_tok, a.n_used, a.n_expert) == 8 ? launch_down<8>(ctx, a) : launch_down<16>(ctx, a);
}
