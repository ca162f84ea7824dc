// 32-bit matrix products on the matrix cores:  C[M,N] = A[M,K] * W[N,K]^T (+ bias[N]), float in, float out.
// v_mfma_f32_16x16x4_f32 multiplies and adds in 32-bit (no reduced-precision mode) at the rate of the vector units, but takes
// its operands from registers that a wave fills with 16-byte loads, so nothing but memory bounds the products of few rows.
//
//   gemm32_stream  M <= 64, K >= 512: the weight is read once, straight into the matrix instruction; a workgroup owns 8, 16 or 32
//                  weight rows, its waves share K out in chunks of 32 and add their sums up in LDS in a fixed order, which the
//                  number of weight rows decides and the number of rows does not.
//   gemm32_tile    the rest: tiles through LDS, the next steps' loads in flight while the present one is multiplied; a result is
//                  the sum of its products from the first column to the last, to the bit what gemm_fma gives.
//
// Both: K and the row stride of A multiples of 4, A and W 16-byte aligned (the host checks; what does not fit goes to
// gemm_fma); M and N are arbitrary.  Loads go through a buffer that ends with the workgroup's last row; rows and columns that
// do not exist are asked for beyond its end, which brings zeros and touches no memory (and no branch surrounds a load).
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

// Operand layout: lane l holds A[i = l % 16][k = l / 16] and B[k = l / 16][j = l % 16]; result D[i = 4 (l / 16) + r][j = l % 16].
// i = weight row, j = row of A.  One instruction adds its four products one after the other, each rounded.  In the stream a
// lane's four consecutive columns 4g .. 4g + 3 (one 16-byte load) serve four instructions: the sum over K takes the columns
// of a group of 16 in another order, the same one for both operands.
__device__ __forceinline__ void fma_16x16x16(f32x4& acc, f32x4 w, f32x4 x) {
#pragma unroll
    for (int r = 0; r < 4; ++r) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w[r], x[r], acc, 0, 0, 0);
}

#define NOWHERE 0x80000000u
// The rows first .. first + rows - 1 (those below `all`) of a matrix with `ld` columns a row, `cols` of them used.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_buffer(const float* p, int first, int rows, int all, int ld, int cols) {
    const unsigned bytes = (unsigned)(min(rows, all - first) - 1) * (unsigned)ld * 4u + (unsigned)cols * 4u;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p + (size_t)first * ld), 0, bytes, 0x00020000);
}
// four columns from k on of the row that starts `row` bytes into the buffer
__device__ __forceinline__ f32x4 load_columns(__amdgpu_buffer_rsrc_t b, unsigned row, int k, int K) {
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(b, k < K ? row + (unsigned)k * 4u : NOWHERE, 0, 0));
}
__device__ __forceinline__ unsigned row_offset(int row, int rows, int ld) { return row < rows ? (unsigned)row * ld * 4u : NOWHERE / 2; }

// ------------------------------------------------------------------------------ few rows
// Bound by reading the weight: 32000 x 2048 (262 MB) at 2 rows takes 48 microseconds (5.4 TB/s), 11264 x 2048 22 (4.1 TB/s),
// 2048 x 2048 6 (a launch and one wait for memory); the multiply-add kernel, whose workgroup brings 64 weight rows through
// LDS 4 bytes a load whatever the number of rows, takes 272, 210 and 202.  At 64 rows 118, 58 and 22: from some 20 rows on
// every workgroup's reading of all rows of X out of L2 weighs more than the weight.
// HALVES (up to 8 rows of A): a tile is 8 weight rows, and rows 8 to 15 of both operands hold the same rows' columns of another share of
// K, so that D[i][j] and D[i + 8][j + 8] are two parts of one sum (the other two blocks of D mean nothing).  A weight of few rows
// then has a workgroup on twice as many compute units, and each spends half the time in its matrix instructions.  8 waves with two
// shares each sum what 16 waves sum elsewhere, in the same order: a row's result is the same bits whether 1 or 64 rows come with it.
// 2 rows against 2048 x 5632 17.3 -> 10.9 microseconds, 1024 x 4096 12.9 -> 8.0, 2048 x 2048 7.9 -> 6.3, 512 x 512 5.5 -> 3.6 (16 waves
// with two shares each, whose sums are others: 12.1, 8.6, 7.0 and 4.0; with 4 chunks a round instead of 2: 12.1, 8.4, 6.4 and 4.1).
template <int MB, int NT, int WAVES, int UNROLL, bool HALVES = false, bool GATED = false>
__global__ __launch_bounds__(WAVES* LLMS_WAVE) void gemm32_stream_kernel(float* __restrict__ C, const float* __restrict__ X,
                                                                         const float* __restrict__ W,
                                                                         const float* __restrict__ bias, int M, int N, int K,
                                                                         int ldx, int ldc, int wide) {
    static_assert(!HALVES || (MB == 1 && NT == 1), "halves: one tile of up to 8 rows");
    static_assert(!GATED || (MB == 1 && NT == 1 && !HALVES), "gated: one tile of 8 units");
    constexpr int ROWS = HALVES ? 8 : 16, SHARES = HALVES ? 2 * WAVES : WAVES;  // rows of a tile, sums that K is shared out to
    __shared__ f32x4 red[WAVES][NT * MB][LLMS_WAVE];
    const int wave = threadIdx.x / LLMS_WAVE, lane = threadIdx.x % LLMS_WAVE;
    const int r16 = lane % ROWS, g = lane / 16, later = HALVES ? (lane / 8 % 2) * WAVES * 32 : 0;
    const int n0 = blockIdx.x * (GATED ? 8 : ROWS * NT);
    // (gated: from the first gate row to the last up row, W = [gate; up] of N units each)
    const __amdgpu_buffer_rsrc_t w_buf = rows_buffer(W, n0, GATED ? N + 8 : ROWS * NT, GATED ? 2 * N : N, K, K), x_buf = rows_buffer(X, 0, ROWS * MB, M, ldx, K);
    unsigned wrow[NT], xrow[MB];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        if constexpr (GATED) wrow[t] = n0 + r16 % 8 < N ? row_offset(r16 % 8 + (r16 < 8 ? 0 : N), 2 * N, K) : NOWHERE / 2;
        else wrow[t] = row_offset(t * 16 + r16, N - n0, K);
    }
#pragma unroll
    for (int b = 0; b < MB; ++b) xrow[b] = row_offset(b * 16 + r16, M, ldx);
    f32x4 acc[NT][MB];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int b = 0; b < MB; ++b) acc[t][b] = (f32x4){0.f, 0.f, 0.f, 0.f};

    const int chunks = (K + 31) / 32;
    for (int c0 = wave; c0 < chunks; c0 += SHARES * UNROLL) {
        f32x4 wv[UNROLL][NT][2];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int s = 0; s < 2; ++s) wv[u][t][s] = load_columns(w_buf, wrow[t], (c0 + u * SHARES) * 32 + later + s * 16 + g * 4, K);
        f32x4 xv[UNROLL][MB][2];
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
#pragma unroll
            for (int b = 0; b < MB; ++b)
#pragma unroll
                for (int s = 0; s < 2; ++s) xv[u][b][s] = load_columns(x_buf, xrow[b], (c0 + u * SHARES) * 32 + later + s * 16 + g * 4, K);
        // (all of them are asked for before the first is used: with the rows of X asked for one by one behind the weights,
        // 2048 x 5632 at 2 rows took 21 microseconds instead of 19)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < UNROLL; ++u)
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int b = 0; b < MB; ++b)
#pragma unroll
                    for (int t = 0; t < NT; ++t) fma_16x16x16(acc[t][b], wv[u][t][s], xv[u][b][s]);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int b = 0; b < MB; ++b) red[wave][t * MB + b][lane] = acc[t][b];
    __syncthreads();
    for (int idx = threadIdx.x; idx < NT * MB * LLMS_WAVE; idx += WAVES * LLMS_WAVE) {
        const int part = idx / LLMS_WAVE, l = idx % LLMS_WAVE;
        const int n = n0 + (part / MB) * 16 + 4 * (l / 16), m = (part % MB) * 16 + l % 16;
        if (m >= M || n >= N || ((HALVES || GATED) && l >= 32)) continue;
        // (added up in 64 bits and rounded once: the few sums of a thread wait for LDS, not for arithmetic)
        double wide_sum[4] = {};
#pragma unroll
        for (int w = 0; w < WAVES; ++w)
#pragma unroll
            for (int r = 0; r < 4; ++r) wide_sum[r] += (double)red[w][part][l][r];
        if constexpr (HALVES) {  // (rows 8 .. 15 by rows 8 .. 15 of X)
#pragma unroll
            for (int w = 0; w < WAVES; ++w)
#pragma unroll
                for (int r = 0; r < 4; ++r) wide_sum[r] += (double)red[w][part][l + 40][r];
        }
        f32x4 s = {(float)wide_sum[0], (float)wide_sum[1], (float)wide_sum[2], (float)wide_sum[3]};
        if constexpr (GATED) {  // (rows 8 .. 15: the same units' up)
            double up[4] = {};
#pragma unroll
            for (int w = 0; w < WAVES; ++w)
#pragma unroll
                for (int r = 0; r < 4; ++r) up[r] += (double)red[w][part][l + 32][r];
#pragma unroll
            for (int r = 0; r < 4; ++r) s[r] = s[r] / (1.f + expf(-s[r])) * (float)up[r];
        }
        float* c = C + (size_t)m * ldc + n;
        if (wide && n + 4 <= N) {
            if (bias)
#pragma unroll
                for (int r = 0; r < 4; ++r) s[r] += bias[n + r];
            *reinterpret_cast<f32x4*>(c) = s;
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n + r < N) c[r] = s[r] + (bias ? bias[n + r] : 0.f);
        }
    }
}

// ------------------------------------------------------------------------------ tiles
// Bound by the matrix cores (157 TFLOP/s in 32-bit) once there are several large tiles for every compute unit: an instruction of 32
// cycles needs 8 bytes of LDS per lane, so one buffer and a plain order of stages are enough (4096 x 4096 at 2,048 rows 502
// microseconds, 137 TFLOP/s).  With few rows a compute unit has one or two workgroups, which wait for each stage in turn: the small
// tiles have two buffers (TWO), and a step's products run beside the writing of the next one's tile and the loads of the two behind it,
// which made a step of 32 x 64 x 64 1.0 -> 0.72 microseconds (0.43 in its matrix instructions).  Two buffers for 64 x 64 gain
// nothing (105 and 104 microseconds for 11264 x 2048 at 130 rows): fewer workgroups fit.
template <int BM, int BN, int BK, int WM, bool TWO>
__global__ __launch_bounds__(256) void gemm32_tile_kernel(float* __restrict__ C, const float* __restrict__ A,
                                                          const float* __restrict__ W, const float* __restrict__ bias, int M,
                                                          int N, int K, int lda, int ldc, int tiles_m, int wide) {
    constexpr int WN = 4 / WM, TM = BM / WM / 16, TN = BN / WN / 16, LD = BK + 4;
    constexpr int PER_ROW = BK / 4, CA = BM * PER_ROW / 256, CB = BN * PER_ROW / 256, STEP = 256 / PER_ROW;
    __shared__ __attribute__((aligned(16))) float As[TWO ? 2 : 1][BM * LD];
    __shared__ __attribute__((aligned(16))) float Bs[TWO ? 2 : 1][BN * LD];
    // workgroups are dealt round-robin to the 8 XCDs: each XCD gets a contiguous run of tiles, rows fastest, so that the tiles
    // which share a weight slab share an L2
    const int nblk = gridDim.x, pid = blockIdx.x;
    const int full = nblk / 8, rem = nblk % 8, xcd = pid % 8;
    const int t = xcd * full + min(xcd, rem) + pid / 8;
    const int m0 = (t % tiles_m) * BM, n0 = (t / tiles_m) * BN;
    const int tid = threadIdx.x, wave = tid / LLMS_WAVE, lane = tid % LLMS_WAVE;
    const int wm = (wave % WM) * (BM / WM), wn = (wave / WM) * (BN / WN);
    const int r16 = lane % 16, g = lane / 16;
    const int row = tid / PER_ROW, col = (tid % PER_ROW) * 4, place = (col & ~15) + (col & 15) / 4;

    const __amdgpu_buffer_rsrc_t a_buf = rows_buffer(A, m0, BM, M, lda, K), w_buf = rows_buffer(W, n0, BN, N, K, K);
    unsigned ap[CA], wp[CB];
#pragma unroll
    for (int c = 0; c < CA; ++c) ap[c] = row_offset(row + c * STEP, M - m0, lda);
#pragma unroll
    for (int c = 0; c < CB; ++c) wp[c] = row_offset(row + c * STEP, N - n0, K);
    f32x4 ra[TWO ? 2 : 1][CA], rb[TWO ? 2 : 1][CB], acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    // piece p of a step's loads (rows of A, then of W; beyond K: from nowhere)
    auto fetch = [&](auto set, int p, int k0) {
        constexpr int q = decltype(set)::n;
        if (p < CA) ra[q][p] = load_columns(a_buf, ap[p], k0 + col, K);
        else rb[q][p - CA] = load_columns(w_buf, wp[p - CA], k0 + col, K);
    };
    auto put = [&](auto set, int p) {
        constexpr int q = decltype(set)::n;
        // column 4 q + r of a group of 16 lies at 4 r + q: what a lane reads in one piece, its instructions take in the order
        // of the columns, so that a result is the sum of its products from the first column to the last
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (p < CA) As[q][(row + p * STEP) * LD + place + 4 * r] = ra[q][p][r];
            else Bs[q][(row + (p - CA) * STEP) * LD + place + 4 * r] = rb[q][p - CA][r];
        }
    };
    f32x4 xf[2][TM], wf[2][TN];
    auto read = [&](auto set, int s) {
        constexpr int q = decltype(set)::n;
#pragma unroll
        for (int i = 0; i < TM; ++i) xf[s % 2][i] = *reinterpret_cast<const f32x4*>(&As[q][(wm + i * 16 + r16) * LD + s * 16 + g * 4]);
#pragma unroll
        for (int j = 0; j < TN; ++j) wf[s % 2][j] = *reinterpret_cast<const f32x4*>(&Bs[q][(wn + j * 16 + r16) * LD + s * 16 + g * 4]);
    };
    auto multiply = [&](int s) {
        // (four columns of K for every tile before the next four: a tile's instructions do not follow on one another)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[s % 2][j][r], xf[s % 2][i][r], acc[i][j], 0, 0, 0);
    };
    // LDS only is waited for: the loads of the steps behind stay in flight
    auto meet = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // A step: its tile lies in one buffer; the next step's goes into the other (whose readers met behind the step before), the one
    // behind that is asked for, and the step's products run beside both, a group of 16 columns at a time.  (With all of the next
    // tile written before the first read, the reads queued behind 96 writes of the workgroup.)
    constexpr int GROUPS = BK / 16, PIECES = CA + CB;
    auto one = [&](auto now, auto next, int k0) {
        read(now, 0);
#pragma unroll
        for (int s = 0; s < GROUPS; ++s) {
            if (s + 1 < GROUPS) read(now, s + 1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(s);
#pragma unroll
            for (int p = PIECES * s / GROUPS; p < PIECES * (s + 1) / GROUPS; ++p) {
                put(next, p);
                fetch(next, p, k0 + 3 * BK);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        meet();
    };
    if constexpr (TWO) {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) fetch(Number<0>(), p, 0);
#pragma unroll
        for (int p = 0; p < PIECES; ++p) fetch(Number<1>(), p, BK);
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
            put(Number<0>(), p);
            fetch(Number<0>(), p, 2 * BK);
        }
        meet();
        for (int k0 = 0; k0 < K; k0 += 2 * BK) {  // (a step beyond K adds zeros; a branch around it made the compiler wait for every load)
            one(Number<0>(), Number<1>(), k0);
            one(Number<1>(), Number<0>(), k0 + BK);
        }
    } else {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) fetch(Number<0>(), p, 0);
        for (int k0 = 0; k0 < K; k0 += BK) {
            __syncthreads();  // (every wave is done with the tile before)
#pragma unroll
            for (int p = 0; p < PIECES; ++p) put(Number<0>(), p);
            __syncthreads();
            if (k0 + BK < K)
#pragma unroll
                for (int p = 0; p < PIECES; ++p) fetch(Number<0>(), p, k0 + BK);
#pragma unroll
            for (int s = 0; s < GROUPS; ++s) {
                read(Number<0>(), s);
                multiply(s);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int m = m0 + wm + i * 16 + r16;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int n = n0 + wn + j * 16 + g * 4;
            f32x4 s = acc[i][j];
            float* c = C + (size_t)m * ldc + n;
            if (wide && n + 4 <= N) {
                if (bias)
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[r] += bias[n + r];
                *reinterpret_cast<f32x4*>(c) = s;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n + r < N) c[r] = s[r] + (bias ? bias[n + r] : 0.f);
            }
        }
    }
}

template <int BM, int BN, int BK, int WM, bool TWO>
static int launch_tile(float* C, const float* A, const float* W, const float* bias, int M, int N, int K, int lda, int ldc, int wide,
                       hipStream_t stream) {
    const int tiles_m = (M + BM - 1) / BM;
    const long long blocks = (long long)tiles_m * ((N + BN - 1) / BN);
    LLMS_REQUIRE(blocks < (1ll << 31), "gemm32: too many tiles");
    gemm32_tile_kernel<BM, BN, BK, WM, TWO><<<(unsigned)blocks, 256, 0, stream>>>(C, A, W, bias, M, N, K, lda, ldc, tiles_m, wide);
    LLMS_LAUNCH_CHECK();
}

// A tile and what it costs, microseconds: `fixed`, `round` more for each round of tiles over the compute units, `step` for each step of
// bk columns, and `round_step` more for each step of each round.  Fitted to two thirds of 2,929 products (4 to 2,048 rows, 256 to 11,264
// weight rows, 4 to 11,008 columns): the tile that costs least by them takes 0.3 % longer than the best in the mean and 13 % at most,
// on the third that was left out 0.3 % and 10 %.
struct Tile32 {
    int bm, bn, bk;
    bool two;
    float fixed, round, step, round_step;
};
static const Tile32 TILES32[] = {{32, 32, 64, true, 2.17f, 0.35f, 0.093f, 0.290f},
                                 {32, 64, 64, true, 2.22f, 0.51f, 0.164f, 0.551f},
                                 {32, 64, 64, false, 2.0f, 0.415f, 0.33f, 0.526f},
                                 {64, 64, 64, false, 2.06f, 1.07f, 0.41f, 0.957f},
                                 {128, 128, 32, false, 0.f, 3.66f, 0.71f, 1.83f}};

extern "C" {

// The tile (a place in TILES32) that takes least.  Larger ones read each operand less often, smaller ones fill the last round; two
// buffers hide the answers of memory behind the steps, of which a short K has none: with one step they fetch two more and multiply
// one in vain (512 rows against 11264 x 64: 32 x 64 with two buffers 22 microseconds, with one 13; 100 against 2560 x 64: 32 x 32
// 4.1, 32 x 64 with one buffer 3.3; 1,900 against 2048 x 128: 16.6 and 14.8).  At K of 2,048 and more: 65 rows against 2048 x 2048 16
// (in tiles of 32 x 64 with one buffer 31), 2048 x 5632 37 (78); 130 rows 25 (31), 59 (78), 11264 x 2048 72 (105 in 64 x 64).
int llms_gemm32_tile(int M, int N, int K, int cus) {
    int best = 0;
    float least = 0.f;
    for (int t = 0; t < (int)(sizeof(TILES32) / sizeof(TILES32[0])); ++t) {
        const Tile32& tile = TILES32[t];
        const long long tiles = (long long)((M + tile.bm - 1) / tile.bm) * ((N + tile.bn - 1) / tile.bn);
        int steps = (K + tile.bk - 1) / tile.bk;
        if (tile.two) steps += steps % 2;
        const float rounds = (float)((tiles + cus - 1) / cus);
        const float cost = tile.fixed + tile.round * rounds + (tile.step + tile.round_step * rounds) * (float)steps;
        if (t == 0 || cost < least) best = t, least = cost;
    }
    return best;
}

int llms_gemm32(void* c, const void* a, const void* w, const void* b, int M, int N, int K, int lda, int ldc, int cus,
                hipStream_t stream) {
    LLMS_REQUIRE(M > 0 && N > 0 && K > 0, "gemm32: sizes must be positive");
    LLMS_REQUIRE(K % 4 == 0 && lda % 4 == 0, "gemm32: K and the row stride of A must be multiples of 4");
    LLMS_REQUIRE((uintptr_t)a % 16 == 0 && (uintptr_t)w % 16 == 0, "gemm32: A and W must be 16-byte aligned");
    LLMS_REQUIRE(lda >= K && ldc >= N, "gemm32: leading dimensions too small");
    LLMS_REQUIRE(cus > 0, "gemm32: no compute units");
    // (offsets within a tile of 128 rows stay below the one that stands for nothing)
    LLMS_REQUIRE((long long)lda * 4 * 128 < (1ll << 30) && (long long)K * 4 * 128 < (1ll << 30), "gemm32: rows are too long");
    float* C = (float*)c;
    const float *A = (const float*)a, *W = (const float*)w, *bias = (const float*)b;
    const int wide = ldc % 4 == 0 && (uintptr_t)c % 16 == 0;
    // Rows of fewer than 512 columns give the stream's waves a chunk each at most.  They go to the tiles (2 rows of 508 columns
    // against 512 weight rows 5.4 microseconds, of 512 columns in the stream 3.5; 40 rows 5.6 and 8.1; the multiply-add kernel 48 to
    // 53), whose sums in the order of the columns are to the bit what small models gave before.
    if (M <= 64 && K >= 512) {
        const unsigned tiles = (N + 15) / 16, pairs = (N + 31) / 32;
        if (M <= 16) {
            // 16 waves a tile while the tiles alone do not fill the chip, 8 beyond (with two chunks a round: more in flight than memory
            // answers at once costs time; 2 rows against 32000 x 2048 48.5 microseconds with four, 46.5 with two, 49.3 with one)
            // tiles of 8 weight rows where there are no more of them than compute units and up to 8 rows of A
            if (M <= 8 && (N + 7) / 8 <= cus) gemm32_stream_kernel<1, 1, 8, 2, true><<<(N + 7) / 8, 512, 0, stream>>>(C, A, W, bias, M, N, K, lda, ldc, wide);
            else if (tiles <= 2u * cus) gemm32_stream_kernel<1, 1, 16, 4><<<tiles, 1024, 0, stream>>>(C, A, W, bias, M, N, K, lda, ldc, wide);
            else gemm32_stream_kernel<1, 1, 8, 2><<<tiles, 512, 0, stream>>>(C, A, W, bias, M, N, K, lda, ldc, wide);
        } else if (M <= 32) {
            if (tiles <= 2u * cus) gemm32_stream_kernel<2, 1, 16, 4><<<tiles, 1024, 0, stream>>>(C, A, W, bias, M, N, K, lda, ldc, wide);
            else gemm32_stream_kernel<2, 2, 8, 2><<<pairs, 512, 0, stream>>>(C, A, W, bias, M, N, K, lda, ldc, wide);
        } else {
            if (tiles <= 2u * cus) gemm32_stream_kernel<4, 1, 16, 2><<<tiles, 1024, 0, stream>>>(C, A, W, bias, M, N, K, lda, ldc, wide);
            else gemm32_stream_kernel<4, 2, 8, 2><<<pairs, 512, 0, stream>>>(C, A, W, bias, M, N, K, lda, ldc, wide);
        }
        LLMS_LAUNCH_CHECK();
    }
    switch (llms_gemm32_tile(M, N, K, cus)) {
        case 0: return launch_tile<32, 32, 64, 2, true>(C, A, W, bias, M, N, K, lda, ldc, wide, stream);
        case 1: return launch_tile<32, 64, 64, 1, true>(C, A, W, bias, M, N, K, lda, ldc, wide, stream);
        case 2: return launch_tile<32, 64, 64, 1, false>(C, A, W, bias, M, N, K, lda, ldc, wide, stream);
        case 3: return launch_tile<64, 64, 64, 2, false>(C, A, W, bias, M, N, K, lda, ldc, wide, stream);
    }
    return launch_tile<128, 128, 32, 2, false>(C, A, W, bias, M, N, K, lda, ldc, wide, stream);
}

// c[M, inter] = silu(a wg^T) * (a wu^T), w = [wg; wu] of `inter` rows each: up to 16 rows, the activation in the product's epilogue (4.7
// microseconds a launch of its own), with the sums and the arithmetic of llms_gemm32 and the activation behind it, to the bit (5632 x 2048 at 2
// rows 21.7 microseconds with four chunks a round in flight, 20.2 with two).
int llms_gemm32_gated(void* c, const void* a, const void* w, int M, int inter, int K, int lda, int ldc, int cus, hipStream_t stream) {
    LLMS_REQUIRE(M > 0 && M <= 16 && inter > 0 && K >= 512 && cus > 0, "gemm32_gated: 1 to 16 rows of 512 columns and more");
    LLMS_REQUIRE(K % 4 == 0 && lda % 4 == 0 && (uintptr_t)a % 16 == 0 && (uintptr_t)w % 16 == 0, "gemm32_gated: rows of multiples of 4, 16-byte aligned");
    LLMS_REQUIRE(lda >= K && ldc >= inter, "gemm32_gated: leading dimensions too small");
    LLMS_REQUIRE((long long)(inter + 8) * K * 4 < (1ll << 30) && (long long)lda * 4 * 128 < (1ll << 30), "gemm32_gated: too large");
    float* C = (float*)c;
    const float *A = (const float*)a, *W = (const float*)w;
    const int wide = ldc % 4 == 0 && (uintptr_t)c % 16 == 0;
    const unsigned tiles = (inter + 7) / 8;
    if ((2 * inter + 15) / 16 <= 2 * cus) gemm32_stream_kernel<1, 1, 16, 4, false, true><<<tiles, 1024, 0, stream>>>(C, A, W, nullptr, M, inter, K, lda, ldc, wide);
    else gemm32_stream_kernel<1, 1, 8, 2, false, true><<<tiles, 512, 0, stream>>>(C, A, W, nullptr, M, inter, K, lda, ldc, wide);
    LLMS_LAUNCH_CHECK();
}

}  // extern "C"
