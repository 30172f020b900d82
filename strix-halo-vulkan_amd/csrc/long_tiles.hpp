// Q4_K weight rows against tiles of 32 activation rows on the matrix cores: what the projections and the experts of long passes share.
//
// A wave owns R tiles of 32 weight rows and NTT tiles of activations: v_mfma_f32_32x32x16_f16, activations x weights, so that a lane holds
// one weight row of a tile (its scales, its d) and sixteen activation rows.  The weights are the whole numbers n * sc, exact in binary16,
// one accumulator a super-block; the activations two binary16 parts; the min term one product a super-block, the eight sub-blocks' sums in
// two parts against the whole numbers m.  (One accumulator an output, carried from super-block to super-block by a multiplication with the
// quotient of their d, would leave registers for half as many tiles again; its error against float64 is 1.3 to 2 times this one's.)
//
// A step is 16 columns of a chunk of 64: step 2 nib + j takes, in the lanes of half h, columns 32 nib + 16 h + 8 j .. + 7, the low (nib 0)
// or high nibbles of payload bytes 16 h + 8 j .. + 7, which lane (row n, half h) of the weights has loaded.
#pragma once
#include "moe_staged.hpp"
#include "shv_internal.hpp"

namespace shv_long {

using namespace shv;
using namespace shv_moe;

typedef float float16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void *lds_ptr_t;

// A row of k columns as operands, its own 4 k bytes together: [chunk of 64][step][part][half] x 16 bytes, the eight columns in the order
// a payload dword's nibbles come.  After all rows their sums over sub-blocks, [row][super-block][part] x 16 bytes; then the rows' exponents,
// where they have been scaled (binary16_parts).
__host__ __device__ constexpr size_t row_sums_offset(long long rows, int k) { return static_cast<size_t>(rows) * k * 4; }
__host__ __device__ constexpr size_t row_exps_offset(long long rows, int k) { return row_sums_offset(rows, k) + static_cast<size_t>(rows) * (k / 256) * 32; }
__host__ __device__ constexpr size_t row_bytes(long long rows, int k) { return row_exps_offset(rows, k) + static_cast<size_t>(rows) * sizeof(int32_t); }
// columns c .. c + 7 of a row, their first part (the second 32 bytes on)
__host__ __device__ constexpr int row_at(int c) { return (c >> 6) * 256 + (((c >> 5) & 1) * 2 + ((c >> 3) & 1)) * 64 + ((c >> 4) & 1) * 16; }

// A row's columns 4 lane + 256 i as operands, scaled, with its sums and exponent; a wave a row, every lane here.
template <int K>
__device__ __forceinline__ void stage_row(const float (&x)[K / 256][4], int t, int rows, char *staged) {
    constexpr int NQ = K / 256;
    const int lane = threadIdx.x & 63;
    float largest = 0.f;
#pragma unroll
    for (int i = 0; i < NQ; i++) largest = fmaxf(largest, fmaxf(fmaxf(fabsf(x[i][0]), fabsf(x[i][1])), fmaxf(fabsf(x[i][2]), fabsf(x[i][3]))));
    const int e = biased_exponent(wave_max_all(largest));
    if (lane == 0) reinterpret_cast<int32_t *>(staged + row_exps_offset(rows, K))[t] = e - kListOne;
    char *to = staged + static_cast<size_t>(t) * (K * 4) + row_at(4 * lane) + (lane & 1) * 8;
    char *sums = staged + row_sums_offset(rows, K) + static_cast<size_t>(t) * (NQ * 32) + (lane >> 3) * 2;
#pragma unroll
    for (int i = 0; i < NQ; i++) {
        const float o[4] = {ldexpf(x[i][0], kListOne - e), ldexpf(x[i][2], kListOne - e), ldexpf(x[i][1], kListOne - e), ldexpf(x[i][3], kListOne - e)};
        half4_t hi, lo;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            _Float16 p, q;
            binary16_parts(o[j], p, q);
            hi[j] = p;
            lo[j] = q;
        }
        *reinterpret_cast<half4_t *>(to + i * 1024) = hi;
        *reinterpret_cast<half4_t *>(to + i * 1024 + 32) = lo;
        // over 64: 32 values of up to 2^15 stay within binary16
        const float sum = sum8_all((o[0] + o[2]) + (o[1] + o[3])) * (1.f / 64.f);
        if ((lane & 7) == 0) {
            _Float16 p, q;
            binary16_parts(sum, p, q);
            *reinterpret_cast<_Float16 *>(sums + i * 32) = p;
            *reinterpret_cast<_Float16 *>(sums + i * 32 + 16) = q;
        }
    }
}
constexpr float kSumUnit = 64.f;  // of stage_row's sums

// A chunk of 64 columns of 32 NTT rows in LDS is [half of the columns][8 rows] x 1 KB, what one load of a wave brings: 128 bytes, a line,
// of each of eight rows, its lane 8 r + i the sixteen bytes i ^ (row / 2 mod 8) of row r, so that the sixteen rows whose like bytes are
// read together lie in all the banks.
constexpr int kFrag = 1024;
__host__ __device__ constexpr int chunk_lds(int ntt) { return ntt * 8 * kFrag; }
__device__ __forceinline__ uint32_t chunk_piece(int lane, int row) { return ((lane & 7) ^ ((row >> 1) & 7)) * 16; }
// LDS of a stream: the chunk being multiplied and the next, and the sums of a super-block, [tile] lane (row, part) x 16 bytes.
__host__ __device__ constexpr int stream_lds(int ntt) { return 2 * chunk_lds(ntt) + ntt * kFrag; }

// Sixteen bytes a lane to LDS, at `to` + 16 lane: base + at + fixed, the first and the last the same in every lane.
typedef __amdgpu_buffer_rsrc_t buffer_t;
__device__ __forceinline__ buffer_t buffer_of(const char *base, uint32_t bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(base), 0, bytes, 0x00027000); }
// (An offset in the instruction itself would move the place in LDS as well.)
__device__ __forceinline__ void load_lds16(buffer_t base, uint32_t at, uint32_t fixed, char *to) { __builtin_amdgcn_raw_ptr_buffer_load_lds(base, (lds_ptr_t)to, 16, at, fixed, 0, 0); }

// Where lane (row n of a tile, half h) finds its sixteen bytes of part p of an even (odd) step in a chunk: at[odd][p].
struct ChunkReader {
    uint32_t at[2][2];
    __device__ __forceinline__ ChunkReader(int lane) {
        const int n = lane & 31, h = lane >> 5;
#pragma unroll
        for (int o = 0; o < 2; o++)
#pragma unroll
            for (int p = 0; p < 2; p++) at[o][p] = n * 128 + (((o * 4 + p * 2 + h) ^ ((n >> 1) & 7)) * 16);
    }
};

// acc[r][tt] += the products of a chunk's 64 columns.
template <int R, int NTT>
__device__ __forceinline__ void chunk_products(const char *from, const ChunkReader &at, const uint4 (&q)[R], const uint4 (&hdr)[R], int chunk, const NibbleMasks &nc, float16_t (&acc)[R][NTT]) {
    uint32_t sc[R], mn;
#pragma unroll
    for (int r = 0; r < R; r++) q4k_group_scale_min(hdr[r], chunk, sc[r], mn);
#pragma unroll
    for (int st = 0; st < 4; st++) {
        half8_t f[NTT][2];
#pragma unroll
        for (int tt = 0; tt < NTT; tt++)
#pragma unroll
            for (int p = 0; p < 2; p++) f[tt][p] = *reinterpret_cast<const half8_t *>(from + (st >> 1) * (NTT * 4 * kFrag) + tt * (4 * kFrag) + at.at[st & 1][p]);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const uint32_t d0 = (st & 1) ? q[r].z : q[r].x, d1 = (st & 1) ? q[r].w : q[r].y;
            const half8_t w = st < 2 ? weights8<false>(d0, d1, sc[r] & 0xFFu, nc) : weights8<true>(d0, d1, sc[r] >> 8, nc);
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int tt = 0; tt < NTT; tt++) acc[r][tt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f[tt][p], w, acc[r][tt], 0, 0, 0);
        }
    }
}

// A super-block ends: y += d acc - dmin unit (m . sums), sums: the lane's sixteen bytes of the first tile's, in units of `unit`.
template <int R, int NTT>
__device__ __forceinline__ void add_scaled(const uint4 (&hdr)[R], const float16_t (&acc)[R][NTT], const char *sums, float unit, float16_t (&y)[R][NTT]) {
#pragma unroll
    for (int r = 0; r < R; r++) {
        const float d = f16_bits_to_f32(hdr[r].x);
#pragma unroll
        for (int tt = 0; tt < NTT; tt++)
#pragma unroll
            for (int i = 0; i < 16; i++) y[r][tt][i] = fmaf(d, acc[r][tt][i], y[r][tt][i]);
    }
    half8_t m[R];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            uint32_t sc, mn;
            q4k_group_scale_min(hdr[r], g, sc, mn);
            m[r][2 * g] = static_cast<_Float16>(static_cast<float>(mn & 0xFFu));
            m[r][2 * g + 1] = static_cast<_Float16>(static_cast<float>(mn >> 8));
        }
#pragma unroll
    for (int tt = 0; tt < NTT; tt++) {
        const half8_t sx = *reinterpret_cast<const half8_t *>(sums + tt * kFrag);
#pragma unroll
        for (int r = 0; r < R; r++) {
            float16_t cm;
#pragma unroll
            for (int i = 0; i < 16; i++) cm[i] = 0.f;
            cm = __builtin_amdgcn_mfma_f32_32x32x16_f16(sx, m[r], cm, 0, 0, 0);
            const float dmin = -unit * f16_bits_to_f32(hdr[r].x >> 16);
#pragma unroll
            for (int i = 0; i < 16; i++) y[r][tt][i] = fmaf(dmin, cm[i], y[r][tt][i]);
        }
    }
}

template <int R, int NTT>
__device__ __forceinline__ void clear(float16_t (&v)[R][NTT]) {
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int tt = 0; tt < NTT; tt++)
#pragma unroll
            for (int i = 0; i < 16; i++) v[r][tt][i] = 0.f;
}

// A barrier behind which what the waves asked for before their last N loads has landed in LDS.  (__syncthreads() waits for no load that
// writes LDS by itself.)
template <int N>
__device__ __forceinline__ void landed_barrier() {
    static_assert(N < 64, "vmcnt");
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070 | (N & 15) | (N >> 4) << 14);  // vmcnt(N) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Weight rows of SBS super-blocks at first (this lane's of each of the wave's tiles), and those unit_bytes on, `units` times, against staged
// activations that stream through LDS chunk by chunk; done(u, y) takes a unit's sums: y[r][tt][i] of lane (n, h) is weight row n of tile r
// against activation row 8 (i / 4) + 4 h + i % 4 of tile tt.  (A chunk that nobody reads may be on its way to LDS still.)
// rows[i] (chunk_piece in it) is where this lane's line of its wave's i-th eight rows begins in `staged`, sum where its sixteen bytes of the
// sums of tile `wave` (waves 0 .. NTT - 1) begin in `sums`, in units of sum_unit.  A chunk's weights are asked for four chunks ahead, as soon
// as their registers are free; where a row is short (SBS 1, 2; 4 of one tile), a super-block's all together, so that a line is fetched once
// (2048 x 512 expert rows 5 % faster, 12352 x 1024 of 4096 rows, one tile, 247 to 235 us; rows of eight super-blocks, whose waves wait for
// more at a time then, 5 % slower).
// Every wave of a block of four calls it; smem: stream_lds(NTT).
//
// What bounds it: the card's power, then vector issue.  12352 x 2048 of 4096 rows: the clock falls to 1.8 GHz, the matrix cores are busy 55 %
// of it, vector instructions (five beside each matrix instruction) issue 41 %; without forming weights the same time, without LDS reads 10 % less, with the
// matrix instructions alone 27 % less.  More chunks on their way (two to four buffers), fragments read a step ahead, a wave's priority and
// the order of its instructions changed nothing beyond 2 %.
template <int SBS, int R, int NTT, typename Done>
__device__ __forceinline__ void stream_products(const char *const (&first)[R], int units, int unit_bytes, char *smem, int wave, buffer_t staged, const uint32_t (&rows)[NTT],
                                                buffer_t sums, uint32_t sum, float sum_unit, Done &&done) {
    static_assert(NTT <= 4, "a tile's sums a wave");
    constexpr bool whole = SBS <= 2 || (R == 1 && SBS <= 4);
    const int lane = threadIdx.x & 63, h = lane >> 5;
    const ChunkReader at(lane);
    char *sums_s = smem + 2 * chunk_lds(NTT);
    const char *rp[R];  // of the super-block the chunks are in
    uint4 q[4][R], hdr[R], hdr_next[R];
    auto ask = [&](int k, int b) {
#pragma unroll
        for (int i = 0; i < NTT; i++) {
            load_lds16(staged, rows[i], k * 256, smem + b * chunk_lds(NTT) + (wave * NTT + i) * kFrag);
            load_lds16(staged, rows[i], k * 256 + 128, smem + b * chunk_lds(NTT) + (NTT * 4 + wave * NTT + i) * kFrag);
        }
    };
    auto ask_sums = [&](int sb) {
        if (wave < NTT) load_lds16(sums, sum, sb * 32, sums_s + wave * kFrag);
    };
    auto ask_weights = [&](int step, int c, uint4 (&to)[R]) {
#pragma unroll
        for (int r = 0; r < R; r++) to[r] = *reinterpret_cast<const uint4 *>(rp[r] + step + 16 + c * 32 + h * 16);
    };
    auto ask_header = [&](int step) {
#pragma unroll
        for (int r = 0; r < R; r++) hdr_next[r] = *reinterpret_cast<const uint4 *>(rp[r] + step);
    };
#pragma unroll
    for (int r = 0; r < R; r++) {
        rp[r] = first[r];
        hdr[r] = *reinterpret_cast<const uint4 *>(rp[r]);
    }
    ask(0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 4; c++) ask_weights(0, c, q[c]);
    __builtin_amdgcn_s_waitcnt(0x0F70 | 4 * R);  // vmcnt: all but the weights
    const NibbleMasks nc = nibble_masks();
#pragma unroll 1
    for (int u = 0; u < units; u++) {
        float16_t y[R][NTT];
        clear(y);
#pragma unroll 1
        for (int sb = 0; sb < SBS; sb++) {
            // the super-block after this one: behind a unit's last the next unit's first (the last unit's: its own again)
            const int step = sb + 1 < SBS ? SHV_Q4K_BYTES : u + 1 < units ? unit_bytes - (SBS - 1) * SHV_Q4K_BYTES : 0;
            const int nsb = sb + 1 < SBS ? sb + 1 : 0;
            float16_t acc[R][NTT];
            clear(acc);
#pragma unroll
            for (int c = 0; c < 4; c++) {
                // this chunk is here, the other one's room is read to its end; what has been asked for since the chunk is weights
                if (!whole) landed_barrier<R>();
                else if (c == 0) landed_barrier<4 * R>();
                else landed_barrier<0>();
                if (c == 0) ask_sums(sb);
                ask(c < 3 ? 4 * sb + c + 1 : 4 * nsb, 1 - (c & 1));
                if (c == 0 && !whole) ask_header(step);
                __builtin_amdgcn_sched_barrier(0);
                chunk_products<R, NTT>(smem + (c & 1) * chunk_lds(NTT), at, q[c], hdr, c, nc, acc);
                if (!whole) {
                    ask_weights(step, c, q[c]);
                } else if (c == 3) {
                    ask_header(step);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int i = 0; i < 4; i++) ask_weights(step, i, q[i]);
                }
            }
            add_scaled(hdr, acc, sums_s + lane * 16, sum_unit, y);
#pragma unroll
            for (int r = 0; r < R; r++) {
                hdr[r] = hdr_next[r];
                rp[r] += step;
            }
        }
        done(u, y);
    }
    landed_barrier<0>();  // nothing is on its way to LDS any more, and nobody reads it
}

}  // namespace shv_long
