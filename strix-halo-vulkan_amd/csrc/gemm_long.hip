// Q4_K projections of long passes: y[t] = W pro(x[t]) (+ residual[t]) for some hundreds to 4096 activation rows, on the products of
// long_tiles.hpp: a launch makes the rows into operands, scaled row by row by a power of two, a second one multiplies groups of 64 of them
// with 256 or 128 weight rows a block.  The matrix cores' power bounds it (1.05 PFLOP/s of binary16 products at 4096 rows, 1.36 with
// nothing but the matrix instructions left).
// us, two dozen matrices in turn (n x k, rows), before / now; before: slabs of 128 columns, 16 x 16 tiles, one fragment read from LDS a
// matrix instruction, two reads of the activations' sums and values unscaled
//   12352 x 2048   576: 78 / 75   1024: 145 / 130   1531: 207 / 173   2048: 266 / 236   4096: 507 / 434
//    9216 x 2048        73 / 65         111 / 99          147 / 138         192 / 175         363 / 316
//    2048 x 4096        58 / 52          59 / 56           86 / 78           97 / 89          163 / 159
// Error against float64 of 4096 x 2048: 0.40e-6 (before 0.45e-6; activations of 0.02 2.1e-6, of mean 3 6.5e-6 against 4.0e-6 now).
#include "gemm_rows.hpp"
#include "long_tiles.hpp"

namespace {

using namespace shv;
using namespace shv_gemm;
using namespace shv_moe;
using namespace shv_long;

// A pass's rows as operands (long_tiles.hpp), up to whole groups, then where each row's outputs go.
__host__ __device__ constexpr size_t long_places_offset(int padded, int k) { return (row_bytes(padded, k) + 15) / 16 * 16; }
__host__ __device__ constexpr size_t long_bytes(int padded, int k) { return long_places_offset(padded, k) + static_cast<size_t>(padded) * sizeof(size_t); }

// A wave a row.
template <int K>
__global__ __launch_bounds__(256) void gemm_long_stage_kernel(shv_gemv_q4k_args a, char *staged, int padded) {
    constexpr int NQ = K / 256;
    const int lane = threadIdx.x & 63, t = blockIdx.x * 4 + (threadIdx.x >> 6);
    const bool on = t < a.n_tok;
    float x[NQ][4];
    float scale = 1.f;
    if (a.prologue == SHV_PRO_RMSNORM && on) {
        const float *xr = a.x + static_cast<size_t>(t) * a.x_stride + 4 * lane;
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < NQ; i++) {
            const float4 v = *reinterpret_cast<const float4 *>(xr + 256 * i);
            ss = fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, fmaf(v.w, v.w, ss))));
        }
        scale = 1.f / sqrtf(wave_sum_all(ss) / static_cast<float>(K) + a.eps);
    }
#pragma unroll
    for (int i = 0; i < NQ; i++) {
        x[i][0] = x[i][1] = x[i][2] = x[i][3] = 0.f;
        if (on) pro_quad(a, t, 256 * i + 4 * lane, scale, x[i]);
    }
    if (lane == 0) reinterpret_cast<size_t *>(staged + long_places_offset(padded, K))[t] = on ? out_offset(a, t) : 0;
    stage_row<K>(x, t, padded, staged);
}

// Four waves of 32 R weight rows each against a group of 64 activation rows.
constexpr int kThreads = 256, kTiles = 2, kTok = 32 * kTiles;
constexpr size_t kLds = stream_lds(kTiles) + kTok * (sizeof(size_t) + sizeof(int32_t));
template <int K, int R>
__global__ __launch_bounds__(kThreads, R == 1 ? 4 : 2) void gemm_long_kernel(shv_gemv_q4k_args a, const char *staged, int padded, int groups, int row_blocks) {
    extern __shared__ __align__(16) char smem[];
    constexpr int SBS = K / 256, ROWB = SBS * SHV_Q4K_BYTES;
    const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, h = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // blocks of one die (every eighth) take neighbouring tiles, eight groups of activations by some row blocks at a time
    int group, rb;
    {
        const int total = groups * row_blocks, per = (total + 7) >> 3;
        const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
        if (tile >= total) return;
        const int strip = 8 * row_blocks, s = tile / strip, in = tile - s * strip;
        const int width = groups - 8 * s < 8 ? groups - 8 * s : 8;
        rb = in / width;
        group = 8 * s + in - rb * width;
    }
    size_t *place_s = reinterpret_cast<size_t *>(smem + stream_lds(kTiles));
    int32_t *exps_s = reinterpret_cast<int32_t *>(place_s + kTok);
    if (tid < kTok) {
        place_s[tid] = reinterpret_cast<const size_t *>(staged + long_places_offset(padded, K))[group * kTok + tid];
        exps_s[tid] = reinterpret_cast<const int32_t *>(staged + row_exps_offset(padded, K))[group * kTok + tid];
    }
    const int row0 = rb * (128 * R) + wave * (32 * R);
    const char *rp[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int row = row0 + 32 * r + n < a.n ? row0 + 32 * r + n : a.n - 1;
        rp[r] = static_cast<const char *>(a.w) + static_cast<size_t>(row) * ROWB;
    }
    uint32_t rows[kTiles];
#pragma unroll
    for (int i = 0; i < kTiles; i++) {
        const int t = (wave * kTiles + i) * 8 + (lane >> 3);
        rows[i] = t * (K * 4) + chunk_piece(lane, t);
    }
    stream_products<SBS, R, kTiles>(rp, 1, 0, smem, wave, buffer_of(staged + static_cast<size_t>(group) * (kTok * K * 4), kTok * K * 4), rows,
                                    buffer_of(staged + row_sums_offset(padded, K) + static_cast<size_t>(group) * (kTok * SBS * 32), kTok * SBS * 32),
                                    ((wave % kTiles) * 32 + n) * (SBS * 32) + h * 16, kSumUnit, [&](int, const float16_t (&y)[R][kTiles]) {
        // C[activation row 8 (i >> 2) + 4 h + (i & 3)][weight row n]
#pragma unroll
        for (int tt = 0; tt < kTiles; tt++)
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const int m = 32 * tt + 8 * (i >> 2) + 4 * h + (i & 3), t = group * kTok + m, back = exps_s[m];
                const size_t to = place_s[m];
#pragma unroll
                for (int r = 0; r < R; r++) {
                    const int row = row0 + 32 * r + n;
                    if (t < a.n_tok && row < a.n) {
                        float v = ldexpf(y[r][tt][i], back);
                        if (a.residual) v += a.residual[static_cast<size_t>(t) * a.y_stride + row];
                        a.y[to + row] = v;
                    }
                }
            }
    });
}

template <int K, int R>
int launch(shv_ctx *ctx, const shv_gemv_q4k_args &a, int padded) {
    const int groups = padded / kTok, row_blocks = (a.n + 128 * R - 1) / (128 * R), per = (groups * row_blocks + 7) / 8;
    SHV_LAUNCH(ctx, (gemm_long_kernel<K, R>), dim3(8 * per), dim3(kThreads), kLds, a, static_cast<const char *>(ctx->gemm_stage), padded, groups, row_blocks);
    return SHV_OK;
}

int padded_rows(int n_tok) { return (n_tok + kTok - 1) / kTok * kTok; }

template <int K>
int launch_k(shv_ctx *ctx, const shv_gemv_q4k_args &a) {
    static_assert(kLds <= 48 * 1024, "no more than a launch may have without asking");
    const int padded = padded_rows(a.n_tok), cus = ctx->prop.multiProcessorCount;
    const long long groups = padded / kTok;
    SHV_LAUNCH(ctx, gemm_long_stage_kernel<K>, dim3(padded / 4), dim3(256), 0, a, ctx->gemm_stage, padded);
    // Short rows: blocks of 128.  Of 256 columns up to two of them a compute unit, and past that as longer rows: what such a block does is write
    // its sums, and three and four at a time on a unit do it faster on some cards and slower on others (2048 x 256 of 3000 rows, blocks of 128
    // 16.8 to 27.4 us, of 256 18.6 to 21.4).  us, before (slabs, 16 x 16 tiles) / chosen as longer rows are / so:
    //                     512 rows             1024                 1531                 2048                 4096
    //    2048 x 256   10.4 / 10.0 / 10.0   11.1 / 11.0 / 11.0   13.7 / 15.2 / 13.1   15.4 / 16.5 / 14.6   23.4 / 23.8 / 23.8
    //    2048 x 512   12.8 / 13.1 / 13.1   13.9 / 15.0 / 14.8   19.0 / 21.6 / 19.8   21.7 / 23.0 / 21.1   33.0 / 34.5 / 33.2
    //    2048 x 1024  18.5 / 19.1 / 19.1   21.2 / 22.5 / 22.2   29.6 / 32.1 / 30.1   32.7 / 35.8 / 34.0   51.7 / 53.9 / 52.6
    //    4096 x 512   13.6 / 14.1 / 14.1   20.1 / 22.2 / 20.1   28.8 / 27.0 / 27.0   31.1 / 32.2 / 30.9   54.7 / 55.2 / 51.1
    //   12352 x 512   26.6 / 27.9 / 26.7   48.2 / 48.4 / 41.8   63.6 / 61.0 / 57.7   82.0 / 79.7 / 71.2    174 / 148  / 134
    //   12352 x 1024  41.5 / 42.3 / 42.1   84.8 / 77.4 / 69.9    111 / 97   / 97      145 / 135  / 124     289 / 241  / 233
    // (2048 x 1024 of 1024 and 2048 rows, 4096 x 1024 of 2048 and 300 x 512 are left 4 to 7 % behind the slabs.)
    if (K == 512 || K == 1024 || (K == 256 && (a.n + 127) / 128 * groups <= 2ll * cus)) return launch<K, 1>(ctx, a, padded);
    // Blocks of 256 weight rows, two a compute unit, or of 128, four a unit, which read the activations twice as often but leave less of the
    // chip idle where there are few.  Their rounds of the chip, in rounds of full units: a unit with one block of 256 takes 0.58 of what two
    // take; 1, 2, 3 blocks of 128 take 0.37, 0.6, 0.82 of what four take, and four a tenth more than two of 256.  us, of 256 / of 128:
    //              576 rows    1024       1531       2048       4096
    //   12352x2048  75 / 80   135 / 130  172 / 184  236 / 236  434 / 453
    //    9216x2048  70 / 65   109 / 99   139 / 137  176 / 175  316 / 338
    //    2048x4096  72 / 52    74 / 56    78 / 82    89 / 92   159 / 168
    const auto rounds = [cus](long long blocks, int a_unit, const double *part) {
        const long long full = blocks / (static_cast<long long>(cus) * a_unit), rest = blocks - full * cus * a_unit;
        return static_cast<double>(full) + part[(rest + cus - 1) / cus];
    };
    static const double two[] = {0., 0.58, 1.}, four[] = {0., 0.37, 0.6, 0.82, 1.};
    const double wide = rounds((a.n + 255) / 256 * groups, 2, two), narrow = 1.1 * rounds((a.n + 127) / 128 * groups, 4, four);
    return narrow < wide ? launch<K, 1>(ctx, a, padded) : launch<K, 2>(ctx, a, padded);
}

}  // namespace

// Passes past gemm_mid.hip's: its blocks of 64 weight rows read the activations from L2 once each, these once per 128 or 256
// (9216 x 2048 of 512 rows 71 us there, 64 here; 12352 x 2048 72 and 75; 2048 x 4096 36 and 51).  Other widths than its: from the
// fourth group of 64 rows, below which gemm_q4k.hip's kernel of one group splits the columns.
bool shv_gemm_long_covers(const shv_ctx *ctx, const shv_gemv_q4k_args &a) {
    if (!ctx->gemm_stage || (a.k != 256 && a.k != 512 && a.k != 1024 && a.k != 2048 && a.k != 4096) || a.n_tok <= (a.k >= 2048 ? 512 : 192)) return false;
    if (a.prologue == SHV_PRO_GATED_NORM && 256 % a.head_dim != 0) return false;
    return long_bytes(padded_rows(a.n_tok), a.k) <= static_cast<size_t>(shv_ctx::kGemmStageBytes);
}

int shv_launch_gemm_long(shv_ctx *ctx, const shv_gemv_q4k_args &a) {
    switch (a.k) {
        case 256: return launch_k<256>(ctx, a);
        case 512: return launch_k<512>(ctx, a);
        case 1024: return launch_k<1024>(ctx, a);
        case 2048: return launch_k<2048>(ctx, a);
        default: return launch_k<4096>(ctx, a);
    }
}
