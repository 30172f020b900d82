// The experts of a pass of many rows, grouped by expert on the matrix cores (the prompt side of
// MoETrace.Experts, llm/moe.go:289-409; the reference batches a chunk's tokens per expert in
// llm_moe_gemv.comp's multi-row arm).  The per-(token, expert) GEMV reads and unpacks an expert's
// weights once per token that chose it, this path once per 96 such tokens: it pays when tokens
// outnumber experts (2048 rows choosing 10 of 512: 40 tokens an expert).  Passes whose experts have
// up to fifteen tokens each go on from the same lists in moe_lists.hip.
//
//   moe_group_kernel          per-expert lists of (token, slot) pairs from topk (one block; long passes:
//                             moe_group_count_kernel + moe_group_place_kernel, sixteen blocks)
//   moe_long.hip              the rows made into operands, gate/up + SwiGLU, and the down projection
//                             over act rows that are operands (act_packed)
//   moe_down_grouped_kernel   the down projection over act rows that are floats, 48 at a time, made into
//                             operands by the block, 512 columns (a whole row) at a time
//   moe_combine_kernel        out[t] = residual[t] + sum over slots of weights[t][s]*pairs[t][s],
//                             slots in order
// The shared expert is an expert every token lists.
#include "moe_staged.hpp"
#include "shv_internal.hpp"

namespace {

using namespace shv;
using namespace shv_moe;


constexpr int kWaves = 8;       // 256 registers a lane: the streams, the accumulators of four row tiles and the operands fit without spilling
constexpr int kThreads = kWaves * 64;
constexpr int kTT = 3;            // matrix-core tiles of 16 tokens a block multiplies per pass over the weights
constexpr int kTok = 16 * kTT;    // tokens of such a pass
constexpr int kTiles = 4;         // weight row tiles of 16 a wave owns
constexpr int kSlab = 512;        // columns of the tokens' rows staged at a time
constexpr int kSlabSubs = kSlab / 32;
constexpr int kFrag = 64 * 16;    // one operand: a lane's eight halves
constexpr int kMaxExperts = 1024;

// The caller's `group` workspace: [0, n_expert] start of each expert's list (one more: the total),
// then n_tok * n_used pair ids (token * (n_used + 1) + slot), then the experts in the order their
// blocks are launched: longest list first, so that the blocks which walk their weights two or
// three times start early and the launch does not end on them.  A list's order is whatever the
// arrivals made it, but for the list kernels (moe_group_place_kernel): in the others no value depends
// on it, every pair's products being formed and added alike in whatever column they are.
__global__ __launch_bounds__(1024) void moe_group_kernel(const int32_t *topk, int n_tok, int n_used, int n_expert, int32_t *group) {
    __shared__ int32_t s_cnt[kMaxExperts + 1];
    __shared__ __align__(16) int32_t s_len[kMaxExperts];
    const int tid = threadIdx.x, n_pairs = n_tok * n_used;
    for (int e = tid; e <= n_expert; e += blockDim.x) s_cnt[e] = 0;
    for (int e = tid; e < kMaxExperts; e += blockDim.x) s_len[e] = -1;  // past n_expert: shorter than any list
    // A thread's selections are asked for once, all together, and stay in registers for both passes (the count and
    // the placement): up to NQ quads of four a thread, i.e. 4096 * NQ pairs; a longer pass reads the rest again.
    constexpr int NQ = 8;
    // whole quads of an aligned table; the tail and what does not fit the registers go one by one
    const int n_quads = (reinterpret_cast<uintptr_t>(topk) & 15) == 0 ? n_pairs / 4 : 0;
    int4 q[NQ];
#pragma unroll
    for (int b = 0; b < NQ; b++) {
        const int i = tid + b * 1024;
        q[b] = i < n_quads ? reinterpret_cast<const int4 *>(topk)[i] : make_int4(-1, -1, -1, -1);
    }
    const int rest0 = (n_quads < NQ * 1024 ? n_quads : NQ * 1024) * 4;
    __syncthreads();
    auto count = [&](int e) {
        if (e >= 0 && e < n_expert) atomicAdd(&s_cnt[e], 1);
    };
#pragma unroll
    for (int b = 0; b < NQ; b++) {
        count(q[b].x);
        count(q[b].y);
        count(q[b].z);
        count(q[b].w);
    }
    for (int i = rest0 + tid; i < n_pairs; i += 1024) count(topk[i]);
    __syncthreads();
    {
        // starts = running sum of the counts: thread e takes expert e (the block has a thread for each)
        __shared__ int32_t s_wsum[16];
        const int lane = tid & 63, wave = tid >> 6;
        const int c = tid < n_expert ? s_cnt[tid] : 0;
        int incl = c;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int up = __shfl_up(incl, o, 64);
            if (lane >= o) incl += up;
        }
        if (lane == 63) s_wsum[wave] = incl;
        __syncthreads();
        int base = 0;
        for (int w = 0; w < wave; w++) base += s_wsum[w];
        if (tid < n_expert) {
            s_cnt[tid] = base + incl - c;
            s_len[tid] = c;
        }
        if (tid == n_expert - 1) s_cnt[n_expert] = base + incl;
    }
    __syncthreads();
    for (int e = tid; e <= n_expert; e += blockDim.x) group[e] = s_cnt[e];
    // rank by list length, longer first, equal lengths by index: an expert's place in the launch.  32 threads an
    // expert, each against every 32nd length, 32 experts a round: with a thread an expert half the block idles
    // through E comparisons each.
    int32_t *order = group + n_expert + 1 + n_pairs;
    {
        const int part = tid & 31;
        for (int e = tid >> 5; e < n_expert; e += 32) {
            const int ce = s_len[e];
            int rank = 0;
            for (int o = part; o < n_expert; o += 32) {
                const int co = s_len[o];
                rank += (co > ce || (co == ce && o < e)) ? 1 : 0;
            }
            rank += __shfl_xor(rank, 16, 64);
            rank += __shfl_xor(rank, 8, 64);
            rank += __shfl_xor(rank, 4, 64);
            rank += __shfl_xor(rank, 2, 64);
            rank += __shfl_xor(rank, 1, 64);
            if (part == 0) order[rank] = e;
        }
    }
    __syncthreads();  // the starts are copied out before the placement moves them
    int32_t *list = group + n_expert + 1;
    auto place = [&](int e, int i) {
        if (e >= 0 && e < n_expert) list[atomicAdd(&s_cnt[e], 1)] = (i / n_used) * (n_used + 1) + i % n_used;
    };
#pragma unroll
    for (int b = 0; b < NQ; b++) {
        const int i = 4 * (tid + b * 1024);
        place(q[b].x, i);
        place(q[b].y, i + 1);
        place(q[b].z, i + 2);
        place(q[b].w, i + 3);
    }
    for (int i = rest0 + tid; i < n_pairs; i += 1024) place(topk[i], i);
}

// The same lists by several blocks in two launches, for passes long enough that one block's count and placement
// (one compute unit's scattered stores) are most of the grouping: block b takes pairs [b * chunk, (b + 1) * chunk).
// First launch: every block's count of its pairs per expert, to counts[b][e].  Second: every block adds up the
// counts (an expert's total, and what the blocks before it hold of it), forms the starts, and places its own pairs
// behind those of the blocks before it; block 0 also writes the starts and the experts' launch order.
// In order: a list's pairs lie by token (chunks of at most a pair a thread).  The list kernels add a token's two parts earlier
// or later as a pass over its list has more than eight tokens or not, so a place that changes from call to call would change
// its last bit.  The waves then place their pairs one after the other, a lane behind the lanes before it with the same expert
// (150 rows of ten experts: 224.2 us a layer with the pairs as they arrive, 224.9 so; 750 rows 430.5 and 430.9).
constexpr int kGroupBlocks = 16;
__global__ __launch_bounds__(1024) void moe_group_count_kernel(const int32_t *topk, int n_pairs, int chunk, int n_expert, int32_t *counts) {
    __shared__ int32_t s_cnt[kMaxExperts];
    const int tid = threadIdx.x;
    for (int e = tid; e < n_expert; e += 1024) s_cnt[e] = 0;
    __syncthreads();
    const int lo = blockIdx.x * chunk, hi = lo + chunk < n_pairs ? lo + chunk : n_pairs;
    for (int i = lo + tid; i < hi; i += 1024) {
        const int e = topk[i];
        if (e >= 0 && e < n_expert) atomicAdd(&s_cnt[e], 1);
    }
    __syncthreads();
    for (int e = tid; e < n_expert; e += 1024) counts[blockIdx.x * n_expert + e] = s_cnt[e];
}

// Rows x [rows][k] staged for the list kernels: whole rows, k / 256 of a block's sixteen waves each.
__device__ __forceinline__ void stage_rows(const float *x, int rows, int k, char *staged, int block) {
    __shared__ float s_max[16];
    const int tid = threadIdx.x, quad = block * 1024 + tid, t = quad / (k / 4), c = (quad % (k / 4)) * 4, per = k / 256;
    const float4 v = t < rows ? *reinterpret_cast<const float4 *>(x + static_cast<size_t>(t) * k + c) : float4{0.f, 0.f, 0.f, 0.f};
    float largest = wave_max_all(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    if ((tid & 63) == 0) s_max[tid >> 6] = largest;
    __syncthreads();
    for (int w = 0, w0 = (tid >> 6) / per * per; w < per; w++) largest = fmaxf(largest, s_max[w0 + w]);
    const int e = biased_exponent(largest);
    if (t < rows) {
        stage_list_quad(v, e, t, c, k, rows, staged);
        if (c == 0) reinterpret_cast<int32_t *>(staged + list_exps_offset(rows, k))[t] = e;
    }
}

// The wave's inclusive sums, lane by lane, and the sums of its halves in their last lanes: DPP steps.  By way of LDS each of
// eleven exchanges was a trip of its own, and the experts' order took two comparisons a length: a layer's lists and products
// of 66 rows 168.2 to 167.0 us, of 150 rows 224.3 to 222.7; passes of 65 and 150 rows of 16 layers 3634 to 3609 and 4848 to 4839.
__device__ __forceinline__ int wave_prefix_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr:1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, kDppBcast15, 0xA, 0xF, false);
    return v + __builtin_amdgcn_update_dpp(0, v, kDppBcast31, 0xC, 0xF, false);
}
__device__ __forceinline__ int half_wave_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, kDppXor1, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, kDppXor2, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, kDppHalfMirror, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, kDppMirror, 0xF, 0xF, false);
    return v + __builtin_amdgcn_update_dpp(0, v, kDppBcast15, 0xA, 0xF, false);
}

// counts NULL: no launch before; every block counts all pairs itself, those before its own chunk apart.  Blocks past the sixteen,
// when the launch has them, stage the list kernels' rows x meanwhile.
__global__ __launch_bounds__(1024) void moe_group_place_kernel(const int32_t *topk, int n_pairs, int chunk, int n_used, int n_expert, const int32_t *counts,
                                                               int32_t *group, int in_order, const float *x, int rows, int k, char *staged) {
    if (blockIdx.x >= kGroupBlocks) return stage_rows(x, rows, k, staged, blockIdx.x - kGroupBlocks);
    __shared__ int32_t s_cnt[kMaxExperts + 1];
    __shared__ __align__(16) int32_t s_len[kMaxExperts];
    __shared__ int32_t s_wsum[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nb = kGroupBlocks, b = blockIdx.x;
    // thread e: expert e's total, and the pairs of it the blocks before this one hold
    int c = 0, before = 0;
    if (!counts) {
        s_cnt[tid] = s_len[tid] = 0;
        __syncthreads();
        constexpr int NB = 8;
        for (int i0 = tid; i0 < n_pairs; i0 += NB * 1024) {
            int e[NB];
#pragma unroll
            for (int u = 0; u < NB; u++) e[u] = i0 + u * 1024 < n_pairs ? topk[i0 + u * 1024] : -1;
#pragma unroll
            for (int u = 0; u < NB; u++)
                if (e[u] >= 0 && e[u] < n_expert) {
                    atomicAdd(&s_len[e[u]], 1);
                    if (i0 + u * 1024 < b * chunk) atomicAdd(&s_cnt[e[u]], 1);
                }
        }
        __syncthreads();
        c = s_len[tid], before = s_cnt[tid];
    } else if (tid < n_expert) {
        // all of them asked for together: one after the other they are sixteen trips to memory
        int v[kGroupBlocks];
#pragma unroll
        for (int o = 0; o < kGroupBlocks; o++) v[o] = o < nb ? counts[o * n_expert + tid] : 0;
#pragma unroll
        for (int o = 0; o < kGroupBlocks; o++) {
            c += v[o];
            before += o < b ? v[o] : 0;
        }
    }
    const int incl = wave_prefix_sum(c);
    if (lane == 63) s_wsum[wave] = incl;
    // what orders the experts in one word (a list's length, then the lower index): shapes_covered keeps pairs below 2^19
    s_len[tid] = tid < n_expert ? (c << 10) | (kMaxExperts - 1 - tid) : -1;  // past n_expert: shorter than any list
    __syncthreads();
    int base = 0;
    for (int w = 0; w < wave; w++) base += s_wsum[w];
    const int start = base + incl - c;
    if (tid < n_expert) s_cnt[tid] = start + before;
    if (b == 0) {
        if (tid < n_expert) group[tid] = start;
        if (tid == n_expert - 1) group[n_expert] = start + c;
    }
    // An expert's place in the launch: longer lists first, equal lengths by index.  Each block ranks its share of
    // the experts, 32 threads an expert (each against every 32nd quad of lengths), instead of one block all of them with a
    // thread an expert: E^2 comparisons are most of what one block would spend on a pass's lists.
    {
        const int per = (n_expert + nb - 1) / nb, e0 = b * per;
        const int part = tid & 31;
        for (int eb = tid >> 5; eb < per; eb += 32) {
            const int e = e0 + eb;
            const bool live = e < n_expert;
            const int mine = live ? s_len[e] : 0;
            int rank = 0;
            for (int o = 4 * part; o < n_expert; o += 128) {
                const int4 k = *reinterpret_cast<const int4 *>(s_len + o);
                rank += (k.x > mine) + (k.y > mine) + (k.z > mine) + (k.w > mine);
            }
            rank = half_wave_sum(rank);
            if (live && part == 31) group[n_expert + 1 + n_pairs + rank] = e;
        }
    }
    __syncthreads();
    int32_t *list = group + n_expert + 1;
    const int lo = b * chunk, hi = lo + chunk < n_pairs ? lo + chunk : n_pairs;
    if (in_order) {
        const int i = lo + tid, e = i < hi ? topk[i] : -1;
        const bool on = e >= 0 && e < n_expert;
        uint64_t same = __ballot(on);  // the lanes with this lane's expert
        for (int bit = 1; bit < kMaxExperts; bit <<= 1) {
            const uint64_t set = __ballot(e & bit);
            same &= e & bit ? set : ~set;
        }
        const int ahead = __popcll(same & ((1ull << lane) - 1));
        for (int w = 0; w * 64 < hi - lo; w++) {
            if (wave == w && on) {
                const int at = s_cnt[e];
                if (ahead == 0) s_cnt[e] = at + __popcll(same);
                list[at + ahead] = (i / n_used) * (n_used + 1) + i % n_used;
            }
            __syncthreads();
        }
        return;
    }
    for (int i = lo + tid; i < hi; i += 1024) {
        const int e = topk[i];
        if (e >= 0 && e < n_expert) list[atomicAdd(&s_cnt[e], 1)] = (i / n_used) * (n_used + 1) + i % n_used;
    }
}

// Columns [col0, col0 + kSlab) of up to kTok listed rows (each a row of floats at rows_s[i]) into
// operand order: the fragment of (sub-block, part hi / lo, token tile) is 64 lanes x 16 bytes,
// lane = token in the tile + 16 * (k block of 8 columns), the eight columns in slot order
// [0, 2, 1, 3, 4, 6, 5, 7]; sxs[sub][token] is the sub-block's sum of x.
__device__ __forceinline__ void gather_slab(const float *const *rows_s, int m, int col0, char *frags, float *sxs) {
    constexpr int QPR = kSlab / 4;             // quads a row's slab
    constexpr int RPI = kThreads / QPR;        // rows an iteration of the block covers
    const int tid = threadIdx.x;
    const int c = 4 * (tid % QPR);
    const int sub = c >> 5, kb = (c & 31) >> 3, qh = (c & 7) >> 2;
    // six rows' quads are asked for before the first is used: two memory latencies a slab, not one a row
    constexpr int NI = kTok / RPI, NB = 6;
    static_assert(kTok % RPI == 0 && NI % NB == 0, "whole batches");
#pragma unroll 1
    for (int b0 = 0; b0 < NI; b0 += NB) {
        if (b0 * RPI >= m) break;
        float4 vv[NB];
#pragma unroll
        for (int it = 0; it < NB; it++) {
            const int i = (b0 + it) * RPI + tid / QPR;
            vv[it] = *reinterpret_cast<const float4 *>(rows_s[i < m ? i : 0] + col0 + c);
        }
#pragma unroll
        for (int it = 0; it < NB; it++) {
            const int i = (b0 + it) * RPI + tid / QPR;
            const bool on = i < m;
            float4 v = vv[it];
            if (!on) v = float4{0.f, 0.f, 0.f, 0.f};
            float sum = (v.x + v.y) + (v.z + v.w);
            sum += __shfl_xor(sum, 1, 64);
            sum += __shfl_xor(sum, 2, 64);
            sum += __shfl_xor(sum, 4, 64);
            if (on) {
                if ((c & 31) == 0) sxs[sub * kTok + i] = sum;
                const float o[4] = {v.x, v.z, v.y, v.w};
                half4_t h, l;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const _Float16 hi = static_cast<_Float16>(o[j]);
                    h[j] = hi;
                    l[j] = static_cast<_Float16>(o[j] - static_cast<float>(hi));
                }
                char *e = frags + static_cast<size_t>((sub * 2) * kTT + (i >> 4)) * kFrag + (kb * 16 + (i & 15)) * 16 + qh * 8;
                *reinterpret_cast<half4_t *>(e) = h;
                *reinterpret_cast<half4_t *>(e + kTT * kFrag) = l;
            }
        }
    }
}

// A wave's place in its R weight rows' streams: the header of the super-block it is in, the next
// super-block's header and the payload of the next 64-weight group, both on their way.
template <int R>
struct RowStream {
    uint4 hdr[R], hdr_next[R];
    uint2 q_next[R];
    // group G = 4 * super-block + g, clamped to the last one so that the loads are unconditional
    __device__ __forceinline__ void ask_group(const char *const (&rp)[R], int G, int G_last, int kb) {
        const int Gc = G < G_last ? G : G_last;
#pragma unroll
        for (int r = 0; r < R; r++)
            q_next[r] = *reinterpret_cast<const uint2 *>(rp[r] + static_cast<size_t>(Gc >> 2) * SHV_Q4K_BYTES + 16 + (Gc & 3) * 32 + kb * 8);
    }
    __device__ __forceinline__ void ask_header(const char *const (&rp)[R], int sb, int sb_last) {
        const int sc = sb < sb_last ? sb : sb_last;
#pragma unroll
        for (int r = 0; r < R; r++) hdr_next[r] = *reinterpret_cast<const uint4 *>(rp[r] + static_cast<size_t>(sc) * SHV_Q4K_BYTES);
    }
};

// The 64-weight groups [G0, G0 + NG) of R row tiles (lane rows at rp[r]) against the staged slab,
// whose first sub-block is the first of group G0:
// y[r][tt][j] += sum over those columns of W[row of tile r][.] * x[token 16 tt + 4 kb + j][.].
// A sub-block's eight weights per lane are formed once, as the whole numbers n * sc, and multiplied
// with every token tile; the matrix accumulators run over a super-block and take its d at its end,
// the min term is subtracted per sub-block: y = sum_sb d * (sum x * n * sc) - sum_sub dmin * m * sum(x).
template <int NG, int R>
__device__ __forceinline__ void slab_times_tiles(const char *const (&rp)[R], RowStream<R> &st, int G0, int G_last, const char *frags,
                                                 const float *sxs, int lane, int n_tt, float4_t (&acc)[R][kTT], float4_t (&y)[R][kTT]) {
    const int kb = lane >> 4;
    const NibbleConsts nc = nibble_consts();
#pragma unroll 1
    for (int gi = 0; gi < NG; gi++) {
        const int G = G0 + gi, g = G & 3;
        uint2 q[R];
#pragma unroll
        for (int r = 0; r < R; r++) q[r] = st.q_next[r];
        st.ask_group(rp, G + 1, G_last, kb);
        uint32_t sc[R], mn[R];
        float dmin[R];
#pragma unroll
        for (int r = 0; r < R; r++) {
            q4k_group_scale_min(st.hdr[r], g, sc[r], mn[r]);
            dmin[r] = f16_bits_to_f32(st.hdr[r].x >> 16);
        }
#pragma unroll
        for (int hi = 0; hi < 2; hi++) {
            const int sub = gi * 2 + hi;
            half8_t b[R];
            float dm[R];
#pragma unroll
            for (int r = 0; r < R; r++) {
                const uint32_t q0 = q[r].x, q1 = q[r].y;
                typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
                u32x4 v;
                if (hi == 0) {
                    v.x = ((q0 << 4) & nc.mask) | nc.one; v.y = ((q0 >> 4) & nc.mask) | nc.one;
                    v.z = ((q1 << 4) & nc.mask) | nc.one; v.w = ((q1 >> 4) & nc.mask) | nc.one;
                } else {
                    v.x = (q0 & nc.mask) | nc.one; v.y = ((q0 >> 8) & nc.mask) | nc.one;
                    v.z = (q1 & nc.mask) | nc.one; v.w = ((q1 >> 8) & nc.mask) | nc.one;
                }
                // the halves 64 + n become n * sc: whole numbers up to 15 * 63, exact in binary16 (as is
                // 64 * sc, should the two steps be fused), so one accumulator runs over the super-block
                const _Float16 s16 = static_cast<_Float16>(static_cast<float>(hi ? sc[r] >> 8 : sc[r] & 0xFFu));
                b[r] = (__builtin_bit_cast(half8_t, v) - static_cast<half8_t>(static_cast<_Float16>(64.f))) * static_cast<half8_t>(s16);
                dm[r] = dmin[r] * static_cast<float>(hi ? mn[r] >> 8 : mn[r] & 0xFFu);
            }
#pragma unroll
            for (int tt = 0; tt < kTT; tt++) {
                if (tt >= n_tt) break;
                const char *f = frags + static_cast<size_t>((sub * 2) * kTT + tt) * kFrag + lane * 16;
                const half8_t xh = *reinterpret_cast<const half8_t *>(f);
                const half8_t xl = *reinterpret_cast<const half8_t *>(f + kTT * kFrag);
                const float4 sx = *reinterpret_cast<const float4 *>(sxs + sub * kTok + 16 * tt + 4 * kb);
                const float sxv[4] = {sx.x, sx.y, sx.z, sx.w};
#pragma unroll
                for (int r = 0; r < R; r++) {
                    acc[r][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xh, b[r], acc[r][tt], 0, 0, 0);
                    acc[r][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xl, b[r], acc[r][tt], 0, 0, 0);
#pragma unroll
                    for (int j = 0; j < 4; j++) y[r][tt][j] = fmaf(-dm[r], sxv[j], y[r][tt][j]);
                }
            }
        }
        if (g == 3) {
            // the super-block ends: its sums take its d, the next one's header moves in
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float dd = f16_bits_to_f32(st.hdr[r].x);
#pragma unroll
                for (int tt = 0; tt < kTT; tt++) {
#pragma unroll
                    for (int j = 0; j < 4; j++) y[r][tt][j] = fmaf(dd, acc[r][tt][j], y[r][tt][j]);
                    acc[r][tt] = float4_t{0.f, 0.f, 0.f, 0.f};
                }
            }
            // asked for only now: a header a super-block ahead costs sixteen registers these kernels do not have
            st.ask_header(rp, (G >> 2) + 1, G_last >> 2);
#pragma unroll
            for (int r = 0; r < R; r++) st.hdr[r] = st.hdr_next[r];
        }
    }
}

// All K columns of up to kTok listed rows against a wave's kTiles row tiles: the rows go through
// LDS a slab at a time, the weights of the next super-block are on their way while a slab is staged.
template <int K>
__device__ __forceinline__ void rows_times_tiles(const char *const (&rp)[kTiles], const float *const *rows_s, int m, char *frags, float *sxs,
                                                 int lane, float4_t (&y)[kTiles][kTT]) {
    constexpr int GROUPS = K / 64, NG = kSlab / 64;
    static_assert(K % kSlab == 0, "whole slabs");
    const int n_tt = (m + 15) >> 4;
#pragma unroll
    for (int r = 0; r < kTiles; r++)
#pragma unroll
        for (int tt = 0; tt < kTT; tt++) y[r][tt] = float4_t{0.f, 0.f, 0.f, 0.f};
    float4_t acc[kTiles][kTT];
#pragma unroll
    for (int r = 0; r < kTiles; r++)
#pragma unroll
        for (int tt = 0; tt < kTT; tt++) acc[r][tt] = float4_t{0.f, 0.f, 0.f, 0.f};
    RowStream<kTiles> st;
    st.ask_header(rp, 0, GROUPS / 4 - 1);
#pragma unroll
    for (int r = 0; r < kTiles; r++) st.hdr[r] = st.hdr_next[r];
    st.ask_group(rp, 0, GROUPS - 1, lane >> 4);
#pragma unroll 1
    for (int sl = 0; sl < K / kSlab; sl++) {
        __syncthreads();   // the list is written / the slab before this one has been multiplied
        gather_slab(rows_s, m, sl * kSlab, frags, sxs);
        __syncthreads();
        slab_times_tiles<NG, kTiles>(rp, st, sl * NG, GROUPS - 1, frags, sxs, lane, n_tt, acc, y);
    }
}

// Which expert, which part of its rows and which of its tokens a block takes.  The first
// parts * ceil(n_tok / 16) blocks are the shared expert, one per (part, tile of 16 tokens); the
// rest are the routed experts (every token tile of the expert's list in turn).
struct Unit {
    int expert;   // -1: the shared expert
    int part;
    int first, count;  // positions in the expert's list (routed) or token numbers (shared)
};
__device__ __forceinline__ Unit unit_of(int b, int parts, int n_expert, int n_tok, int n_used, const int32_t *group) {
    Unit u;
    const int shared = parts * ((n_tok + kTok - 1) / kTok);  // the shared expert's blocks come first: all of them have work
    if (b >= shared) {
        b -= shared;
        u.expert = group[n_expert + 1 + n_tok * n_used + b / parts];
        u.part = b % parts;
        u.first = group[u.expert];
        u.count = group[u.expert + 1] - u.first;
    } else {
        u.expert = -1;
        u.part = b % parts;
        u.first = (b / parts) * kTok;
        u.count = n_tok - u.first < kTok ? n_tok - u.first : kTok;
    }
    return u;
}

struct Staging {
    char *frags;
    float *sxs;
    const float **rows_s;
    int32_t *pair_s;
    __device__ __forceinline__ explicit Staging(char *smem) {
        frags = smem;
        sxs = reinterpret_cast<float *>(smem + static_cast<size_t>(kSlabSubs) * 2 * kTT * kFrag);
        rows_s = reinterpret_cast<const float **>(sxs + kSlabSubs * kTok);
        pair_s = reinterpret_cast<int32_t *>(rows_s + kTok);
    }
};
constexpr size_t kGroupedLds = static_cast<size_t>(kSlabSubs) * 2 * kTT * kFrag + static_cast<size_t>(kSlabSubs) * kTok * 4 + kTok * sizeof(float *) + kTok * 4;

// grid: n_expert * parts + parts * ceil(n_tok / 48) blocks, parts = n_embd / 512: a part is 512
// output rows = 32 tiles, wave w takes tiles 4w .. 4w + 3.  K = ffn.
template <int K>
__global__ __launch_bounds__(kThreads) void moe_down_grouped_kernel(shv_moe_down_args a) {
    extern __shared__ __align__(16) char smem[];
    const Staging st(smem);
    const int32_t *group = a.group;
    float *pairout = a.pairs;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, kb = lane >> 4;
    const int parts = a.n_embd / 512;
    const Unit u = unit_of(blockIdx.x, parts, a.n_expert, a.n_tok, a.n_used, group);
    if (u.count <= 0) return;
    const size_t row_bytes = static_cast<size_t>(K / SHV_Q4K_BLOCK) * SHV_Q4K_BYTES;
    const int row0 = u.part * 512 + wave * 64 + n;
    const char *base = static_cast<const char *>(u.expert < 0 ? a.down_sh : a.down_exps) +
                       (static_cast<size_t>(u.expert < 0 ? 0 : u.expert) * a.n_embd + row0) * row_bytes;
    const char *rp[kTiles] = {base, base + 16 * row_bytes, base + 32 * row_bytes, base + 48 * row_bytes};
    for (int t0 = 0; t0 < u.count; t0 += kTok) {
        const int m = u.count - t0 < kTok ? u.count - t0 : kTok;
        if (tid < m) {
            const int pair = u.expert < 0 ? (u.first + t0 + tid) * (a.n_used + 1) + a.n_used : group[a.n_expert + 1 + u.first + t0 + tid];
            st.pair_s[tid] = pair;
            st.rows_s[tid] = a.act + static_cast<size_t>(pair) * K;
        }
        float4_t y[kTiles][kTT];
        rows_times_tiles<K>(rp, st.rows_s, m, st.frags, st.sxs, lane, y);
#pragma unroll
        for (int tt = 0; tt < kTT; tt++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int i = 16 * tt + 4 * kb + j;
                if (i < m) {
                    float *dst = pairout + static_cast<size_t>(st.pair_s[i]) * a.n_embd + row0;
#pragma unroll
                    for (int r = 0; r < kTiles; r++) dst[16 * r] = y[r][tt][j];
                }
            }
        __syncthreads();
    }
}

// grid: (ceil(n_embd / 1024), n_tok), 256 threads, four outputs a thread.
__global__ __launch_bounds__(256) void moe_combine_kernel(shv_moe_down_args a) {
    const float *pairout = a.pairs;
    const int t = blockIdx.y, c = (blockIdx.x * 256 + threadIdx.x) * 4;
    if (c >= a.n_embd) return;
    const float *w = a.weights + static_cast<size_t>(t) * (a.n_used + 1);
    float4 v = {0.f, 0.f, 0.f, 0.f};
    if (a.residual) v = *reinterpret_cast<const float4 *>(a.residual + static_cast<size_t>(t) * a.res_stride + c);
    for (int s = 0; s <= a.n_used; s++) {
        const float ws = w[s];
        const float4 p = *reinterpret_cast<const float4 *>(pairout + (static_cast<size_t>(t) * (a.n_used + 1) + s) * a.n_embd + c);
        v.x = fmaf(ws, p.x, v.x); v.y = fmaf(ws, p.y, v.y); v.z = fmaf(ws, p.z, v.z); v.w = fmaf(ws, p.w, v.w);
    }
    *reinterpret_cast<float4 *>(a.out + static_cast<size_t>(t) * a.out_stride + c) = v;
}

// The per-expert lists of a pass: one block for short passes of few experts, kGroupBlocks in two launches from 2048
// pairs or 128 experts on (ranking the experts by length is E^2 comparisons, a block's share of them a sixteenth)
// (their counts meet in the library's scratch, which nothing else on the stream is using between the two).
// x: rows of k floats to stage for the list kernels, whose lists are in order and few enough pairs for every block to count them
// all: one launch (a pass of 16 layers, with the count in a launch of its own and so: 65 rows 3749 and 3720 us, 150 rows 4989
// and 4965, 300 rows 6600 and 6580, 700 rows 10844 and 10837; the long passes' lists gain nothing, 1531 rows 14298 and 14297).
int launch_group(shv_ctx *ctx, const int32_t *topk, int n_tok, int n_used, int n_expert, int32_t *group, const float *x = nullptr, int k = 0) {
    const int n_pairs = n_tok * n_used;
    if (!x && ((n_pairs < 2048 && n_expert < 128) || !ctx->gemm_part || ctx->moe_group_one_block)) {
        SHV_LAUNCH(ctx, moe_group_kernel, dim3(1), dim3(1024), 0, topk, n_tok, n_used, n_expert, group);
        return SHV_OK;
    }
    static_assert(static_cast<size_t>(kGroupBlocks) * kMaxExperts * 4 <= static_cast<size_t>(shv_ctx::kGemmPartBytes), "the blocks' counts fit the scratch");
    int32_t *counts = reinterpret_cast<int32_t *>(ctx->gemm_part);
    const int chunk = (n_pairs + kGroupBlocks - 1) / kGroupBlocks;
    const int stage_blocks = x ? static_cast<int>((static_cast<long long>(n_tok) * (k / 4) + 1023) / 1024) : 0;
    if (!x) SHV_LAUNCH(ctx, moe_group_count_kernel, dim3(kGroupBlocks), dim3(1024), 0, topk, n_pairs, chunk, n_expert, counts);
    SHV_LAUNCH(ctx, moe_group_place_kernel, dim3(kGroupBlocks + stage_blocks), dim3(1024), 0, topk, n_pairs, chunk, n_used, n_expert, x ? nullptr : counts, group,
               x && chunk <= 1024 ? 1 : 0, x, n_tok, k, ctx->gemm_stage);
    return SHV_OK;
}

template <typename Kern>
int raise_lds(Kern kern, size_t lds) {
    SHV_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
    return SHV_OK;
}

bool shapes_covered(const shv_ctx *ctx, int n_tok, int n_embd, int ffn, int n_used, int n_expert) {
    return n_tok >= ctx->moe_group_min && (n_tok >= 128 || ctx->moe_group_forced || shv_moe_list_tokens(n_tok, n_used, n_expert) > 0) && n_embd == 2048 && ffn == 512 && n_expert >= 1 && n_expert <= kMaxExperts && n_used >= 1 &&
           static_cast<long long>(n_tok) * (n_used + 1) < (1ll << 30) / 2048;
}

}  // namespace

// Whether a pass takes the grouped path: a workspace from the caller, rows enough for experts to
// repeat, the shapes the kernels are built for, and a selection that is already made (topk from
// the router).  The launchers in moe.hip have checked that every bank is Q4_K.
bool shv_moe_up_grouped_covers(const shv_ctx *ctx, const shv_moe_up_args &a) {
    const bool lists = shv_moe_list_tokens(a.n_tok, a.n_used, a.n_expert) > 0;
    return a.group && !a.logits && shv_aligned16(a.xn) && shapes_covered(ctx, a.n_tok, a.n_embd, a.ffn, a.n_used, a.n_expert) && ctx->gemm_stage &&
           (lists ? list_bytes(a.n_tok, a.n_embd) : shv_moe_long_stage_bytes(a.n_tok, a.n_embd)) <= static_cast<size_t>(shv_ctx::kGemmStageBytes);
}

bool shv_moe_down_grouped_covers(const shv_ctx *ctx, const shv_moe_down_args &a) {
    // (act as floats, rows that used to go slot by slot: they still do, in float32)
    if (!a.act_packed && a.n_tok < 128 && !ctx->moe_group_forced) return false;
    return a.group && a.pairs && shv_aligned16(a.act) && shv_aligned16(a.pairs) && shapes_covered(ctx, a.n_tok, a.n_embd, a.ffn, a.n_used, a.n_expert);
}

// Lists, the rows as operands, then the grouped gate/up products.
int shv_launch_moe_up_grouped(shv_ctx *ctx, const shv_moe_up_args &a) {
    // refused before anything is enqueued: an error return leaves no half pass on the stream
    const bool short_lists = shv_moe_list_tokens(a.n_tok, a.n_used, a.n_expert) > 0;
    const long long n_pairs = static_cast<long long>(a.n_tok) * (a.n_used + 1);
    SHV_REQUIRE(!a.act_packed || (ctx->gemm_part && (short_lists ? list_act_bytes(n_pairs, a.ffn) : packed_sums_bytes(n_pairs, a.ffn)) <= static_cast<size_t>(shv_ctx::kGemmPartBytes)),
                "moe_up: %d rows are too many for act_packed", a.n_tok);
    if (short_lists) {
        // short lists: streamed, wave by wave
        if (const int rc = launch_group(ctx, a.topk, a.n_tok, a.n_used, a.n_expert, a.group, a.xn, a.n_embd); rc != SHV_OK) return rc;
        ctx->moe_stamp = {a.topk, a.group, a.act, a.n_tok, a.n_used, true, a.act_packed != 0};
        return shv_launch_moe_up_lists(ctx, a);
    }
    if (const int rc = launch_group(ctx, a.topk, a.n_tok, a.n_used, a.n_expert, a.group); rc != SHV_OK) return rc;
    if (const int rc = shv_launch_moe_up_long(ctx, a); rc != SHV_OK) return rc;
    ctx->moe_stamp = {a.topk, a.group, a.act, a.n_tok, a.n_used, true, a.act_packed != 0};
    return SHV_OK;
}

// The down projection makes its own lists from the same selection (the gate/up products may have
// gone another road: banks of other types), writes every pair's products to the caller's `pairs`
// and folds them per token in slot order.
int shv_launch_moe_down_grouped(shv_ctx *ctx, const shv_moe_down_args &a) {
    SHV_REQUIRE(a.n_embd % 4 == 0 && a.out_stride % 4 == 0 && shv_aligned16(a.out) &&
                    (!a.residual || (a.res_stride % 4 == 0 && shv_aligned16(a.residual))),
                "moe_down: the grouped path moves 16 bytes at a time");
    // the lists are this pass's only if the grouped gate/up launch of this very pass made them
    const shv_ctx::MoeStamp &st = ctx->moe_stamp;
    const bool lists = a.group_ready && st.grouped && st.topk == a.topk && st.group == a.group && st.n_tok == a.n_tok && st.n_used == a.n_used;
    SHV_REQUIRE(!a.act_packed || (lists && st.packed && st.act == a.act && ctx->gemm_part),
                "moe_down: act_packed, but the shv_moe_up before this call did not leave act as operands for this pass");
    if (!lists) {
        if (const int rc = launch_group(ctx, a.topk, a.n_tok, a.n_used, a.n_expert, const_cast<int32_t *>(a.group)); rc != SHV_OK) return rc;
    }
    const int parts = a.n_embd / 512, tiles = (a.n_tok + kTok - 1) / kTok;
    if (a.act_packed && shv_moe_list_tokens(a.n_tok, a.n_used, a.n_expert) > 0) {
        if (const int rc = shv_launch_moe_down_lists(ctx, a); rc != SHV_OK) return rc;
    } else if (a.act_packed) {
        if (const int rc = shv_launch_moe_down_long(ctx, a); rc != SHV_OK) return rc;
    } else {
        constexpr size_t lds = kGroupedLds;
        static const int raised = raise_lds(&moe_down_grouped_kernel<512>, lds);
        if (raised != SHV_OK) return raised;
        SHV_LAUNCH(ctx, moe_down_grouped_kernel<512>, dim3(a.n_expert * parts + parts * tiles), dim3(kThreads), lds, a);
    }
    SHV_LAUNCH(ctx, moe_combine_kernel, dim3((a.n_embd + 1023) / 1024, a.n_tok), dim3(256), 0, a);
    return SHV_OK;
}
