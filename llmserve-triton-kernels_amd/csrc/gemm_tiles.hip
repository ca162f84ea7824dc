// bfloat16 matrix products of many rows (prompts, portions of prompts, large decode batches):  X[M,K] * W[N,K]^T on the
// matrix cores with 32-bit sums, and what used to be a kernel behind the product in its epilogue:
//
//   plain    C[M,N] (+ bias), bfloat16 or float
//   parts    K shared out to several workgroups a tile, one array of 32-bit sums per part, for a norm to add up
//   gated    W = [gate; up]: C[M,N/2] = silu(gate) * up (or the clamped unit, or gelu(gate) * up)
//   rotary   W = [q; k; v]: C = rotated q; rotated k and v go to the tokens' cache slots
//
// Arrangement.  A workgroup owns a tile of BM rows of X by BN rows of W and walks K in steps of 64.  A step's rows come into LDS by
// loads that go there directly (8 rows of 128 bytes an instruction), some steps ahead; a piece of 16 bytes lies at its place XOR
// the row, so that the 16 rows of a matrix operand are read without bank conflicts.  Fragments are held twice: while the first half
// of a step is multiplied its second half is read, and while that is multiplied the next step's first half is, so LDS and matrix
// cores work side by side and a step needs one barrier.  Instructions per wave tile of (BM / WM) x (BN / WN): the larger, the fewer
// bytes of LDS per product, so the large tiles run at 1.4 PFLOP/s in the loop and the small ones fill the chip when there are few rows.
//
// Who loads, and in which order.  A compute unit has some 40 KB of answers outstanding, however many buffers there are (more than 10
// instructions of 1 KB a wave in flight change nothing), and they come back in the order they were asked for: a row of X from L2 behind
// a row of W from memory waits as long as that.  So what counts is how often the queue stands still for memory, and the order decides
// it: U = 2 to 4 steps of W asked for in one piece, then X step by step, stand still once where a step of X and a step of W in turn
// stand still every time (loads alone, 128 x 128 tiles of 2048 x 5632 at 2,048 rows 52.8 -> 45.3 microseconds; 192 x 128 of 11264 x
// 2048 at 333 22.8 -> 19.7; weights in the memory-side cache: no difference).  That needs waves that do nothing but load (NP of them,
// one per SIMD): where the waves that multiply ask for four steps' worth at once, their matrix instructions wait behind their own loads
// (192 x 128 at 333 rows 26.6 -> 27.8, and 25.5 with waves for it).  The rings of X (SX steps) and of W (SW) are as long as LDS allows.
// Taller tiles of fewer weight rows (192 x 96, 256 x 96) ask memory for less.  Tiles of one wave per SIMD that load for themselves (NP
// = 0) stay where a compute unit holds two workgroups, where the weight mostly lies in the memory-side cache, and for 256 x 256, whose
// accumulators leave no registers for more waves.  There the buffers are variables of their own and the loop is unrolled over them: only
// so does the compiler know that a read of one buffer need not wait for the loads into another.
//
// Measured (microseconds, weights from memory; in brackets one wave per SIMD that loads for itself):
//   11264 x 2048 gated     333 rows 23.4 (26.5), 512: 27.6 (29.8), 544: 31.7 (32.6), 768: 35.9 (39.7)
//   2048 x 5632 in parts   512 rows 21.2 (24.4), 640: 26.4 (29.0); one part, 2,048 rows: 51.5 (57.1)
//   2560 x 2048            333 rows 10.3 (11.0), 640: 13.5 (15.6), 2,048: 26.1 (27.4);   2048 x 2048, 2,048 rows 21.5 (22.9)
//   12288 x 4096           256 rows 36.9 (46.8), 333: 42.1 (47.8), 2,048: 170.8 (181.7); 22016 x 4096 gated, 1,024 rows 162 (175)
// What bounds them: the loads, up to some 600 rows (without matrix instructions the same launches take 0.85 to 0.95 of the time);
// beyond, matrix cores at the clock they hold (1.5 to 1.7 PFLOP/s without loads) and how evenly the tiles fill 256 compute units.
//
// Compute units without a tile bring a weight that a later kernel multiplies with nearer (`near`).
//
// K must be a multiple of 64 (the host checks), N of 16, rows of X and W 16-byte aligned; M is arbitrary: rows beyond M
// are read as zeros or as row 0 and never stored.
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

#define GT_PLAIN 0
#define GT_FLOAT 1  // plain or parts, 32-bit result
#define GT_GATED 2
#define GT_ROTARY 3

// A weight that a kernel further on reads, for workgroups to bring nearer: into the 256 MB memory-side cache.
struct Near {
    const void* from;
    unsigned bytes;  // (the host checks: below 2 GB)
    int workers;     // workgroups that do so, behind those of the kernel's own work; 0: none
};

// Worker `at` of them, NW waves: a number of every 128-byte line goes to LDS, where nobody looks at it; `lds`: 256 bytes per wave.  Reads
// stay inside the weight (its buffer descriptor), nothing is written to memory.
template <int NW>
__device__ __forceinline__ void bring_near(const Near& n, int at, void* lds) {
#if defined(__HIP_DEVICE_COMPILE__)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LLMS_WAVE), lane = threadIdx.x % LLMS_WAVE;
    const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(n.from), 0, n.bytes, 0x00020000);
    const unsigned piece = LLMS_WAVE * 128u, stride = (unsigned)(n.workers * NW) * piece;  // (up to 2^30: no offset wraps)
    for (unsigned o = (unsigned)(at * NW + wave) * piece; o < n.bytes; o += stride)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (__attribute__((address_space(3))) void*)((char*)lds + wave * 256), 4, o + lane * 128u, 0, 0, 0);
    __builtin_amdgcn_s_waitcnt(0);  // (no load may find the workgroup gone)
#endif
}

struct TilesArgs {
    const bf16* X;
    const bf16* W;
    const bf16* bias;
    void* C;
    int M, N, K, ldx, ldc;
    int tiles_m, tiles;          // tiles along M, tiles in all (of one part)
    int band, band_tiles;        // tiles along M that are walked together, tiles of such a band
    int workgroups;              // of the tiles in all parts
    int steps;                   // of 64 columns, of one part
    long long part_stride;       // elements from one part's sums to the next's
    int inter, unit;             // GATED; unit 0 SiLU, 1 clamped, 3 gelu
    float limit;
    int n_heads, n_kv_heads, head_dim, block_size, bs_shift;  // ROTARY (bs_shift: log2 of the page size, or -1)
    const float* angles;         // [M][head_dim / 2] (sine, cosine), or null: nothing turns
    const int* slots;            // or null: nothing is stored
    bf16 *k_pool, *v_pool;
    int wide;                    // PLAIN, GATED: rows of C start on 16 bytes, not only on 8
    Near near;                   // for the workgroups behind those of the tiles
};

// Row of W behind row `r` (a multiple of 8) of the product's columns in the order the epilogue wants them: blocks of 16
// columns that belong together (gate and up, both halves of a head) alternate.
template <int EPI>
__device__ __forceinline__ int gt_weight_row(const TilesArgs& a, int r) {
    const int block = r / 16, within = r % 16;
    if (EPI == GT_GATED) return (block & 1) * a.inter + (block / 2) * 16 + within;
    if (EPI == GT_ROTARY) {
        const int halves = a.head_dim / 32, turned = 2 * (a.n_heads + a.n_kv_heads) * halves;  // blocks of q and k
        if (block < turned) {
            const int pair = block / 2, head = pair / halves;
            return head * a.head_dim + (pair - head * halves) * 16 + (block & 1) * (a.head_dim / 2) + within;
        }
    }
    return r;
}

__device__ __forceinline__ void gt_store4(bf16* p, float a, float b, float c, float d) {
    *reinterpret_cast<u32x2*>(p) = (u32x2){pack_bf16x2(a, b), pack_bf16x2(c, d)};
}

// 16 bytes of a result's row; `wide`: rows start on 16 bytes, not on 8
__device__ __forceinline__ void gt_store16(void* p, u32x4 v, int wide) {
    if (wide) {
        *reinterpret_cast<u32x4*>(p) = v;
    } else {
        reinterpret_cast<u32x2*>(p)[0] = (u32x2){v[0], v[1]};
        reinterpret_cast<u32x2*>(p)[1] = (u32x2){v[2], v[3]};
    }
}

// Four units at once.  (UNIT is a constant: with a branch on it around every unit the compiler works one after the other, each a
// chain of some 35 instructions.)
template <int UNIT>
__device__ __forceinline__ u32x2 gt_units(const TilesArgs& a, const f32x4& gate, const f32x4& up) {
    float y[4];
    if constexpr (UNIT == 0) {  // (the projections' results and SiLU are bfloat16 before they are multiplied)
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
            const uint32_t g = pack_bf16x2(gate[r], gate[r + 1]), u = pack_bf16x2(up[r], up[r + 1]);
            const uint32_t s = pack_bf16x2(silu_of_bf16(__uint_as_float(g << 16)), silu_of_bf16(__uint_as_float(g & 0xffff0000u)));
            y[r] = __uint_as_float(s << 16) * __uint_as_float(u << 16);
            y[r + 1] = __uint_as_float(s & 0xffff0000u) * __uint_as_float(u & 0xffff0000u);
        }
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (UNIT == 1) {
                const float g = fminf(gate[r], a.limit), v = fminf(fmaxf(up[r], -a.limit), a.limit);
                y[r] = g / (1.f + expf(-1.702f * g)) * (v + 1.f);
            } else {
                y[r] = gelu_tanh(gate[r]) * up[r];
            }
        }
    }
    return (u32x2){pack_bf16x2(y[0], y[1]), pack_bf16x2(y[2], y[3])};
}

// Workgroups beyond those of the tiles bring a weight that a later kernel multiplies with nearer (`near`).  A tile's loads are
// answered in order, those of weights from memory hold up those of rows from L2 behind them, and no depth of fetching ahead made
// up for it; with its weight in the memory-side cache 2048 x 5632 at 512 rows in 2
// parts takes 17.1 microseconds where it takes 22.9 from memory, 2048 x 2048 8.9 and 11.8.  A layer's four products of the 1.1B shape at
// 512 rows: 93.7 microseconds, 85.8 where q, k, v bring o_proj's weight (16 compute units without a tile) and gate and up
// down_proj's (20).  What bounds a worker is what a compute unit has of misses in flight: 57 GB/s.
//
// NP: waves that only load; without, every wave loads.  SX, SW: steps that LDS holds of X and of W; U: steps of W asked for at once.
template <int BM, int BN, int WM, int WN, int NP, int SX, int SW, int U, int EPI>
__global__ __launch_bounds__((WM * WN + NP) * LLMS_WAVE) void gemm_tiles_kernel(const TilesArgs a) {
    constexpr int NW = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16;
    constexpr int NL = NP ? NP : NW;                   // waves that load
    constexpr int LM = BM / 8 / NL, LN = BN / 8 / NL;  // loads of 8 rows, per wave
    static_assert(LM * NL * 8 == BM && LN * NL * 8 == BN && TM * WM * 16 == BM && TN * WN * 16 == BN, "tile does not divide");
    static_assert(TN % 2 == 0, "columns that belong together lie in one wave");
    static_assert(NP ? SW % U == 0 && SW > U && SX > 2 : SX == SW && U == 1 && (SX == 2 || SX == 4), "buffers");
    // lds0 with NP: SX steps of rows of X, then SW steps of rows of W.  Without: each buffer holds a step of both.
    constexpr int XT = BM * 128, WT = BN * 128, LDS = NP ? SX * XT + SW * WT : XT + WT;
    __shared__ __attribute__((aligned(1024))) uint8_t lds0[LDS];
    __shared__ __attribute__((aligned(1024))) uint8_t lds1[NP ? 16 : LDS];
    __shared__ __attribute__((aligned(1024))) uint8_t lds2[NP || SX < 4 ? 16 : LDS];
    __shared__ __attribute__((aligned(1024))) uint8_t lds3[NP || SX < 4 ? 16 : LDS];

    const int part = EPI == GT_FLOAT ? blockIdx.x / a.tiles : 0, pid = blockIdx.x - part * a.tiles;
    const int first = part * a.steps, steps = min(a.steps, a.K / 64 - first);
    // workgroups are dealt round-robin to the 8 XCDs: each XCD gets a contiguous run of tiles, in bands of `band` tiles along M, rows
    // fastest, so that the tiles which share rows of X or weight rows share an L2
    const int full = a.tiles / 8, rem = a.tiles % 8, xcd = pid % 8;
    const int t = xcd * full + min(xcd, rem) + pid / 8;
    int above = 0, in_band = t, high = a.tiles_m;
    if (a.band < a.tiles_m) {  // (a division that most launches do without)
        const int b = t / a.band_tiles;
        above = b * a.band;
        in_band = t - b * a.band_tiles;
        high = min(a.band, a.tiles_m - above);
    }
    const int m0 = (above + in_band % high) * BM, n0 = in_band / high * BN;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / LLMS_WAVE), lane = tid % LLMS_WAVE;
    const int loader = NP ? wave - NW : wave;  // (NP: the last waves load, the others multiply)
    const int wm = (wave % WM) * (BM / WM), wn = (wave / WM) * (BN / WN);
    const int r16 = lane % 16, g = lane / 16;

    int slots[TM];  // (asked for here, used in the epilogue)
    if constexpr (EPI == GT_ROTARY) {
#pragma unroll
        for (int j = 0; j < TM; ++j) slots[j] = a.slots ? a.slots[min(m0 + wm + j * 16 + r16, a.M - 1)] : -1;
    }

    // A load brings 8 rows: lane l row l / 8, the piece (l % 8) ^ (l / 8) of its 128 bytes, to place l.  Each load has a
    // buffer of its own that starts with its first row and ends with the matrix (groups of rows beyond it: with row 0).
    // Steps beyond the last are asked for beyond the buffers' ends: zeros, and no memory is touched.
    const int lr = lane / 8, lc = ((lane % 8) ^ lr) * 16;
    const unsigned x_off = (unsigned)(lr * a.ldx * 2 + lc), w_off = (unsigned)(lr * a.K * 2 + lc);
    __amdgpu_buffer_rsrc_t xb[LM], wb[LN];
#pragma unroll
    for (int i = 0; i < LM; ++i) {
        int r = m0 + (loader * LM + i) * 8;
        r = r < a.M ? r : 0;
        xb[i] = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(a.X + (size_t)r * a.ldx), 0,
                                                  (unsigned)((min(8, a.M - r) - 1) * a.ldx + a.K) * 2u, 0x00020000);
    }
#pragma unroll
    for (int i = 0; i < LN; ++i) {
        const int c = n0 + (loader * LN + i) * 8;
        wb[i] = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(a.W + (size_t)(c < a.N ? gt_weight_row<EPI>(a, c) : 0) * a.K), 0,
                                                  (unsigned)(8 * a.K) * 2u, 0x00020000);
    }
    auto fetch_x = [&](uint8_t* x, int step) {
#if defined(__HIP_DEVICE_COMPILE__)
        const bool live = step < steps;
        const int so = live ? (first + step) * 128 : 0;
        const unsigned off = live ? x_off : 0x80000000u;
#pragma unroll
        for (int i = 0; i < LM; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xb[i], (__attribute__((address_space(3))) void*)(x + (loader * LM + i) * 1024), 16, off, so, 0, 0);
#endif
    };
    auto fetch_w = [&](uint8_t* w, int step) {
#if defined(__HIP_DEVICE_COMPILE__)
        const bool live = step < steps;
        const int so = live ? (first + step) * 128 : 0;
        const unsigned off = live ? w_off : 0x80000000u;
#pragma unroll
        for (int i = 0; i < LN; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wb[i], (__attribute__((address_space(3))) void*)(w + (loader * LN + i) * 1024), 16, off, so, 0, 0);
#endif
    };

    // v_mfma_f32_16x16x32_bf16 as everywhere in this folder: i = weight row (4 g + register), j = row of X (lane % 16)
    f32x4 acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    bf16x8 wf[2][TN], xf[2][TM];
    auto read = [&](const uint8_t* x, const uint8_t* w, int half) {
        const int q = ((half * 4 + g) ^ (r16 & 7)) * 16;
#pragma unroll
        for (int i = 0; i < TN; ++i) wf[half][i] = *reinterpret_cast<const bf16x8*>(w + (wn + i * 16 + r16) * 128 + q);
#pragma unroll
        for (int j = 0; j < TM; ++j) xf[half][j] = *reinterpret_cast<const bf16x8*>(x + (wm + j * 16 + r16) * 128 + q);
    };
    auto multiply = [&](int half) {
#pragma unroll
        for (int j = 0; j < TM; ++j)
#pragma unroll
            for (int i = 0; i < TN; ++i) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[half][i], xf[half][j], acc[i][j], 0, 0, 0);
    };
    // the order in which the scheduler puts a stage: some matrix instructions, one LDS read, one load, and again
    auto interleave = [&](auto loads) {
        constexpr int READS = TM + TN, EACH = TM * TN / READS > 0 ? TM * TN / READS : 1;
#pragma unroll
        for (int i = 0; i < READS; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x8, EACH, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            if (i < decltype(loads)::n) __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x8, TM * TN, 0);
    };
    // waits until at most `left` loads of this wave are in flight (and its LDS reads are done), then for all waves
    auto arrive = [&](auto left) {
        constexpr int n = decltype(left)::n;
        static_assert(n < 64, "the counter of loads in flight");
        __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | 0x0070);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // (Here and not at the start: behind a branch there the arguments would be asked for a second time, 0.4 microseconds a launch; what
    // a worker has worked out so far is in bounds and not used.  Products that come in parts have no workers, and were 0.4 slower with
    // this code in their kernel.)
    if constexpr (EPI == GT_GATED || EPI == GT_ROTARY) {
        if (__builtin_expect((int)blockIdx.x >= a.workgroups, 0)) {
            bring_near<NW + NP>(a.near, blockIdx.x - a.workgroups, lds0);
            return;
        }
    }
    if constexpr (NP == 0) {
        // One step: `now` holds it, its first half is in registers; `next` holds the step behind it.  At the barrier every wave
        // has read all of `now`, which then takes the step SX further on.
        int step = 0;
        auto fetch = [&](uint8_t* lds, int at) {
            fetch_x(lds, at);
            fetch_w(lds + XT, at);
        };
        auto one = [&](uint8_t* now, uint8_t* next) {
            read(now, now + XT, 1);
            multiply(0);
            interleave(Number<0>());
            __builtin_amdgcn_sched_barrier(0);
            arrive(Number<(SX - 2) * (LM + LN)>());
            __builtin_amdgcn_sched_barrier(0);
            fetch(now, step + SX);
            read(next, next + XT, 0);
            multiply(1);
            interleave(Number<LM + LN>());
            __builtin_amdgcn_sched_barrier(0);
            ++step;
        };
        fetch(lds0, 0);
        fetch(lds1, 1);
        if constexpr (SX == 4) {
            fetch(lds2, 2);
            fetch(lds3, 3);
        }
        arrive(Number<(SX - 1) * (LM + LN)>());
        read(lds0, lds0 + XT, 0);
        for (int rounds = (steps + SX - 1) / SX; rounds > 0; --rounds) {
            one(lds0, lds1);
            if constexpr (SX == 2) {
                one(lds1, lds0);
            } else {
                one(lds1, lds2);
                one(lds2, lds3);
                one(lds3, lds0);
            }
        }
        arrive(Number<0>());  // (no load may find the workgroup gone)
    } else if (wave >= NW) {
        // What is asked for at the barrier behind step t, where the places of that step are free: if it is the last of U, U steps of W,
        // then a step of X.  Step s + 1 is there when at most `left` loads are in flight: those asked for behind it until then.
        int xs = 0, ws = 0;  // the places that are asked for next
        auto next_x = [&](int step) {
            fetch_x(lds0 + xs * XT, step);
            xs = xs + 1 < SX ? xs + 1 : 0;
        };
        auto next_w = [&](int from) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                fetch_w(lds0 + SX * XT + ws * WT, from + u);
                ws = ws + 1 < SW ? ws + 1 : 0;
            }
        };
        constexpr int BEFORE = SX > SW - U + 1 ? SX : SW - U + 1;
#pragma unroll
        for (int t = -BEFORE; t < -1; ++t) {
            if ((t + 64 * U) % U == U - 1 && t + SW - U + 1 >= 0) next_w(t + SW - U + 1);
            if (t + SX >= 0) next_x(t + SX);
        }
        // (from -1 on: there the first step is waited for)
        auto go = [&](int t, auto phase) {  // phase: t modulo U
            constexpr int P = decltype(phase)::n, J = (P + 1) % U;
            constexpr int BACK_X = SX - 1, BACK_W = SW - U + J;  // step t + 1 was asked for that many barriers ago: X, W
            constexpr auto asked = [](int back) {      // loads asked for at the `back - 1` barriers before this one
                int n = 0;
                for (int b = 1; b < back; ++b) n += LM + ((P - b + 64 * U) % U == U - 1 ? U * LN : 0);
                return n;
            };
            constexpr int X_LEFT = asked(BACK_X), W_LEFT = asked(BACK_W) + (U - 1 - J) * LN + LM;
            constexpr int LEFT = X_LEFT < W_LEFT ? X_LEFT : W_LEFT;
            arrive(Number<(LEFT < 63 ? LEFT : 63)>());
            if (P == U - 1) next_w(t + SW - U + 1);
            next_x(t + SX);
        };
        int t = -1;
        go(t++, Number<U - 1>());
        while (t < steps - 1) {
            go(t++, Number<0>());
            if constexpr (U > 1) {
                if (t >= steps - 1) break;
                go(t++, Number<1>());
            }
            if constexpr (U > 2) {
                if (t >= steps - 1) break;
                go(t++, Number<2>());
            }
            if constexpr (U > 3) {
                if (t >= steps - 1) break;
                go(t++, Number<3>());
            }
        }
        arrive(Number<0>());  // (no load may find the workgroup gone, nor what the epilogue keeps in LDS)
        return;
    } else {
        int xs = 0, ws = 0;
        arrive(Number<63>());
        read(lds0, lds0 + SX * XT, 0);
        for (int step = 0; step < steps - 1; ++step) {
            const uint8_t* x = lds0 + xs * XT;
            const uint8_t* w = lds0 + SX * XT + ws * WT;
            read(x, w, 1);
            multiply(0);
            interleave(Number<0>());
            __builtin_amdgcn_sched_barrier(0);
            arrive(Number<63>());
            __builtin_amdgcn_sched_barrier(0);
            xs = xs + 1 < SX ? xs + 1 : 0;
            ws = ws + 1 < SW ? ws + 1 : 0;
            read(lds0 + xs * XT, lds0 + SX * XT + ws * WT, 0);
            multiply(1);
            interleave(Number<0>());
            __builtin_amdgcn_sched_barrier(0);
        }
        read(lds0 + xs * XT, lds0 + SX * XT + ws * WT, 1);
        multiply(0);
        multiply(1);
        arrive(Number<63>());
    }

    // ---- epilogue: a lane holds 4 consecutive columns of row m in each acc[i][j]; blocks i and i + 1 (i even) belong together
    if constexpr (EPI == GT_ROTARY) {
        const int D = a.head_dim, half = D / 2, bs = a.block_size, nkv = a.n_kv_heads, turned = (a.n_heads + nkv) * D;
        // The angles of a pair of blocks are asked for before the pair in front of them is stored: behind the stores, each row's
        // would be waited for on its own (the compiler cannot know that they do not overlap), which took 10 microseconds of
        // the 36 that q, k and v of 2,048 rows of the 1.1B shape took.
        constexpr int AHEAD = NW + NP == 4 || TM * TN <= 24 ? 2 : 1;  // (8 waves with large tiles leave no registers for a second pair's)
        f32x4 table[AHEAD][TM][2];
        auto ask = [&](int i) {
            const int c = n0 + wn + i * 16;  // (the same for all lanes: the branches on it are uniform)
            if (!a.angles || c >= turned) return;
            const int row = gt_weight_row<EPI>(a, c) + g * 4, d = row % D;
#pragma unroll
            for (int j = 0; j < TM; ++j) {
                const int m = min(m0 + wm + j * 16 + r16, a.M - 1);
                const f32x4* from = reinterpret_cast<const f32x4*>(a.angles + ((size_t)m * half + d) * 2);
                table[(i / 2) % AHEAD][j][0] = from[0];
                table[(i / 2) % AHEAD][j][1] = from[1];
            }
        };
        if (AHEAD == 2) ask(0);
#pragma unroll
        for (int i = 0; i < TN; i += 2) {
            if (AHEAD == 1) ask(i);
            else if (i + 2 < TN) ask(i + 2);
            const int c = n0 + wn + i * 16;
            if (c >= a.N) continue;
            const int row_lo = gt_weight_row<EPI>(a, c) + g * 4, row_hi = gt_weight_row<EPI>(a, c + 16) + g * 4;
            const int head = row_lo / D, d = row_lo - head * D;
            float b_lo[4] = {}, b_hi[4] = {};
            if (a.bias) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    b_lo[r] = bf16_bits_to_f32(a.bias[row_lo + r].bits);
                    b_hi[r] = bf16_bits_to_f32(a.bias[row_hi + r].bits);
                }
            }
#pragma unroll
            for (int j = 0; j < TM; ++j) {
                const int m = m0 + wm + j * 16 + r16;
                if (m >= a.M) continue;
                const int slot = slots[j];
                const int page = a.bs_shift >= 0 ? slot >> a.bs_shift : slot / bs, off = slot - page * bs;  // (used where slot >= 0)
                float lo[4], hi[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {  // (the projection's result is bfloat16 before it is rotated)
                    lo[r] = round_to<bf16>(acc[i][j][r] + b_lo[r]);
                    hi[r] = round_to<bf16>(acc[i + 1][j][r] + b_hi[r]);
                }
                if (c < turned) {
                    if (a.angles) {
                        const f32x4 s0 = table[(i / 2) % AHEAD][j][0], s1 = table[(i / 2) % AHEAD][j][1];
                        const float sn[4] = {s0[0], s0[2], s1[0], s1[2]}, cs[4] = {s0[1], s0[3], s1[1], s1[3]};
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float2 v = rotate_pair(lo[r], hi[r], cs[r], sn[r]);
                            lo[r] = v.x;
                            hi[r] = v.y;
                        }
                    }
                    bf16* to = nullptr;
                    if (head < a.n_heads) to = reinterpret_cast<bf16*>(a.C) + (size_t)m * a.ldc + head * D + d;
                    else if (slot >= 0) to = a.k_pool + (((size_t)page * nkv + (head - a.n_heads)) * bs + off) * D + d;
                    if (to) {
                        gt_store4(to, lo[0], lo[1], lo[2], lo[3]);
                        gt_store4(to + half, hi[0], hi[1], hi[2], hi[3]);
                    }
                } else if (slot >= 0) {
                    // a page holds [kv head][dimension][token]: 16 lanes are 16 tokens, mostly side by side in a page
                    bf16* v = a.v_pool + (size_t)page * nkv * D * bs + off;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        v[(size_t)(row_lo - turned + r) * bs].bits = f32_to_bf16_bits(lo[r]);
                        v[(size_t)(row_hi - turned + r) * bs].bits = f32_to_bf16_bits(hi[r]);
                    }
                }
            }
        }
        return;
    }
    if constexpr (EPI == GT_FLOAT) {
#pragma unroll
        for (int j = 0; j < TM; ++j) {
            const int m = m0 + wm + j * 16 + r16;
            if (m >= a.M) continue;
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                const int n = n0 + wn + i * 16 + g * 4;
                if (n >= a.N) continue;
                f32x4 s = acc[i][j];
                if (a.bias) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) s[r] += bf16_bits_to_f32(a.bias[n + r].bits);
                }
                *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.C) + part * a.part_stride + (size_t)m * a.ldc + n) = s;
            }
        }
        return;
    }
    // bfloat16 rows go through LDS, a chunk of JC blocks of rows at a time, and leave in 16-byte pieces along whole rows of the
    // tile: as the lanes hold them (8 bytes of 16 rows an instruction) a matrix of 2,048 x 5,632 takes 11.2 microseconds to
    // store, in pieces along rows 5.6.  (32-bit rows have 64 bytes together as the lanes hold them: through LDS 17.3 microseconds for
    // 512 rows of 2048 x 2048, directly 17.0.)  With four units worked out side by side gate and up of the 1.1B shape went from 32.2
    // to 26.4 microseconds at 333 rows, from 34.9 to 29.3 at 512, and from 92.9 to 82.5 at 2,048.
    constexpr int ROW = EPI == GT_GATED ? BN : BN * 2, PITCH = ROW + 16;  // bytes
    constexpr int FIT = LDS / (WM * 16 * PITCH), JC = FIT < TM ? FIT : TM, CHUNKS = (TM + JC - 1) / JC;
    static_assert(JC > 0, "a block of rows fits");
    constexpr int RC = WM * JC * 16, PP = ROW / 16, THREADS = NW * LLMS_WAVE;
    const int left = EPI == GT_GATED ? a.inter - n0 / 2 : a.N - n0;  // columns from the tile's first on
    bf16* const first_row = reinterpret_cast<bf16*>(a.C) + (size_t)m0 * a.ldc + (EPI == GT_GATED ? n0 / 2 : n0);
#pragma unroll
    for (int chunk = 0; chunk < CHUNKS; ++chunk) {
        const int j0 = chunk * JC;
        static_assert(NP == 0 || CHUNKS == 1, "the tile fits");
        uint8_t* const stage = chunk % 2 ? lds1 : lds0;
        uint8_t* const mine = stage + ((wave % WM) * (JC * 16) + r16) * PITCH;
        if constexpr (EPI == GT_GATED) {
            auto units = [&](auto unit) {
#pragma unroll
                for (int j = j0; j < j0 + JC && j < TM; ++j)
#pragma unroll
                    for (int i = 0; i < TN; i += 2)
                        *reinterpret_cast<u32x2*>(mine + (j - j0) * 16 * PITCH + (wn / 2 + i * 8 + g * 4) * 2) =
                            gt_units<decltype(unit)::n>(a, acc[i][j], acc[i + 1][j]);
            };
            if (a.unit == 0) units(Number<0>());
            else if (a.unit == 1) units(Number<1>());
            else units(Number<3>());
        } else {
#pragma unroll
            for (int i = 0; i < TN; ++i) {
                const int n = n0 + wn + i * 16 + g * 4;
                f32x4 b = (f32x4){0.f, 0.f, 0.f, 0.f};
                if (a.bias && n < a.N) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) b[r] = bf16_bits_to_f32(a.bias[n + r].bits);
                }
#pragma unroll
                for (int j = j0; j < j0 + JC && j < TM; ++j) {
                    const f32x4 s = acc[i][j] + b;
                    *reinterpret_cast<u32x2*>(mine + (j - j0) * 16 * PITCH + (wn + i * 16 + g * 4) * 2) =
                        (u32x2){pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])};
                }
            }
        }
        // (LDS alone is waited for: stores to memory stay in flight)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0xc07f);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int k = 0; k < (RC * PP + THREADS - 1) / THREADS; ++k) {
            const int p = tid + k * THREADS, r = p / PP, q = p % PP, within = r % (JC * 16);
            const int row = r / (JC * 16) * (BM / WM) + j0 * 16 + within;  // (of the tile; the last chunk may have fewer blocks)
            if (p >= RC * PP || j0 * 16 + within >= TM * 16 || m0 + row >= a.M || q * 8 >= left) continue;
            gt_store16(first_row + (size_t)row * a.ldc + q * 8, *reinterpret_cast<const u32x4*>(stage + r * PITCH + q * 16), a.wide);
        }
    }
}

// How many tiles along M an XCD walks together.  Of the rows that its `run` of tiles asks L2 for, those of X that lie in the band and those of W
// behind the columns that the run then reaches, the fewest: what the tiles do not share comes from the memory-side cache, and a row from
// there holds up those behind it.  (All of M together, as it is where few rows leave few tiles along M, and in bands, microseconds, weights from
// memory, at 2,048 rows: 2560 x 2048 23.4 and 22.0, 2048 x 2048 18.7 and 18.0, 2048 x 5632 52.1 and 49.2, 4096 x 4096 57.4 and 56.2, 4096 x
// 11008 147.5 and 144.6; 11264 x 2048 gated 87.9 and 87.3, 22016 x 4096 gated 303.3 and 301.4.  A
// few rows less are not worth it, since a weight row that two XCDs ask for comes from memory and one of X does not: 2048 x 5632 in two parts at
// 513 rows, 800 for 832.)
static int gt_band(int tiles_m, int bm, int bn, int run) {
    int best = tiles_m;
    long long least = -1;
    for (int bands = 1; bands <= tiles_m && bands <= 64; ++bands) {
        const int high = (tiles_m + bands - 1) / bands;
        const long long rows = (long long)high * bm + (long long)((run + high - 1) / high) * bn;
        if (least < 0 || rows < least - least / 8) {
            least = rows;
            best = high;
        }
    }
    return best;
}

template <int BM, int BN, int WM, int WN, int NP, int SX, int SW, int U>
static int launch(int epilogue, TilesArgs a, int parts, hipStream_t stream) {
    LLMS_REQUIRE(a.K % 64 == 0, "gemm_tiles: K must be a multiple of 64");
    const int tiles_n = (a.N + BN - 1) / BN;
    a.tiles_m = (a.M + BM - 1) / BM;
    LLMS_REQUIRE((long long)a.tiles_m * tiles_n * parts < (1ll << 31), "gemm_tiles: too many tiles");
    a.tiles = a.tiles_m * tiles_n;
    const int held = 2 * (SX * BM + SW * BN) * 128 <= 163840 ? 2 : 1, each = (a.tiles + 7) / 8;  // tiles a compute unit has at once; of an XCD
    a.band = gt_band(a.tiles_m, BM, BN, each < 32 * held ? each : 32 * held);
    a.band_tiles = a.band * tiles_n;
    a.steps = (a.K / 64 + parts - 1) / parts;
    LLMS_REQUIRE((long long)(parts - 1) * a.steps < a.K / 64, "gemm_tiles: a part of K is empty");
    a.workgroups = a.tiles * parts;
    LLMS_REQUIRE((long long)a.workgroups + a.near.workers < (1ll << 31), "gemm_tiles: too many workgroups");
    const dim3 grid((unsigned)(a.workgroups + a.near.workers)), block((WM * WN + NP) * LLMS_WAVE);
    if (epilogue == GT_PLAIN) gemm_tiles_kernel<BM, BN, WM, WN, NP, SX, SW, U, GT_PLAIN><<<grid, block, 0, stream>>>(a);
    else if (epilogue == GT_FLOAT) gemm_tiles_kernel<BM, BN, WM, WN, NP, SX, SW, U, GT_FLOAT><<<grid, block, 0, stream>>>(a);
    else if (epilogue == GT_GATED) gemm_tiles_kernel<BM, BN, WM, WN, NP, SX, SW, U, GT_GATED><<<grid, block, 0, stream>>>(a);
    else gemm_tiles_kernel<BM, BN, WM, WN, NP, SX, SW, U, GT_ROTARY><<<grid, block, 0, stream>>>(a);
    LLMS_LAUNCH_CHECK();
}

extern "C" {

// epilogue: 0 plain bfloat16, 1 plain float (parts > 1: `parts` arrays of sums, part_stride elements apart), 2 gated, 3 rotary.
// tile: a place in the table of ops/library.py (GEMM_TILES).
// near_workers (gated, rotary): that many workgroups more bring `near_bytes` of `near` nearer.
int llms_gemm_tiles(int tile, int epilogue, void* C, const void* X, const void* W, const void* bias, int M, int N, int K, int ldx,
                    int ldc, int parts, long long part_stride, int unit, float limit, int n_heads, int n_kv_heads, int head_dim,
                    int block_size, const float* angles, const int* slots, void* k_pool, void* v_pool, const void* near,
                    unsigned near_bytes, int near_workers, hipStream_t stream) {
    LLMS_REQUIRE(M > 0 && N > 0 && K > 0 && parts > 0, "gemm_tiles: sizes must be positive");
    LLMS_REQUIRE(N % 16 == 0 && ldx % 8 == 0 && ldx >= K, "gemm_tiles: N in multiples of 16, rows of X of multiples of 8");
    LLMS_REQUIRE((uintptr_t)X % 16 == 0 && (uintptr_t)W % 16 == 0, "gemm_tiles: X and W must be 16-byte aligned");
    LLMS_REQUIRE(ldx < (1 << 26) && K < (1 << 26), "gemm_tiles: rows are too long");
    LLMS_REQUIRE(epilogue >= GT_PLAIN && epilogue <= GT_ROTARY, "gemm_tiles: epilogue");
    LLMS_REQUIRE(parts == 1 || (epilogue == GT_FLOAT && bias == nullptr), "gemm_tiles: only plain 32-bit sums come in parts");
    LLMS_REQUIRE(C != nullptr && ldc % 4 == 0 && (uintptr_t)C % (epilogue == GT_FLOAT ? 16 : 8) == 0 && part_stride % 4 == 0,
                 "gemm_tiles: rows of the result must start on 4 elements");
    const int cols = epilogue == GT_GATED ? N / 2 : epilogue == GT_ROTARY ? n_heads * head_dim : N;
    LLMS_REQUIRE(ldc >= cols, "gemm_tiles: leading dimension of the result too small");
    TilesArgs a{};
    a.X = (const bf16*)X;
    a.W = (const bf16*)W;
    a.bias = (const bf16*)bias;
    a.C = C;
    a.M = M;
    a.N = N;
    a.K = K;
    a.ldx = ldx;
    a.ldc = ldc;
    a.part_stride = part_stride;
    a.near = Near{near, near_bytes, near_workers};
    LLMS_REQUIRE(near_workers >= 0 && near_workers <= 4096 && (near_workers == 0 || (near && (uintptr_t)near % 4 == 0 && near_bytes < (1u << 31))),
                 "gemm_tiles: up to 4,096 workgroups bring up to 2 GB nearer, aligned to 4 bytes");
    LLMS_REQUIRE(near_workers == 0 || epilogue == GT_GATED || epilogue == GT_ROTARY, "gemm_tiles: workers go with the gated and rotary epilogues");
    a.wide = ldc % 8 == 0 && (uintptr_t)C % 16 == 0;
    if (epilogue == GT_GATED) {
        LLMS_REQUIRE(N % 32 == 0 && bias == nullptr, "gemm_tiles: the gated epilogue takes blocks of 16 units and no bias");
        LLMS_REQUIRE(unit == 0 || unit == 1 || unit == 3, "gemm_tiles: unit 0, 1 or 3");
        a.inter = N / 2;
        a.unit = unit;
        a.limit = limit;
    }
    if (epilogue == GT_ROTARY) {
        LLMS_REQUIRE(n_heads > 0 && n_kv_heads > 0 && head_dim > 0 && head_dim % 32 == 0 && N == (n_heads + 2 * n_kv_heads) * head_dim,
                     "gemm_tiles: the rotary epilogue takes q, k and v of heads in multiples of 32");
        LLMS_REQUIRE(slots == nullptr || (k_pool && v_pool && block_size > 0 && (uintptr_t)k_pool % 8 == 0), "gemm_tiles: slots without pools");
        LLMS_REQUIRE((uintptr_t)angles % 16 == 0, "gemm_tiles: the table of angles must be 16-byte aligned");
        a.n_heads = n_heads;
        a.n_kv_heads = n_kv_heads;
        a.head_dim = head_dim;
        a.block_size = block_size;
        a.bs_shift = -1;
        for (int s = 0; s < 31; ++s)
            if ((1 << s) == block_size) a.bs_shift = s;
        a.angles = angles;
        a.slots = slots;
        a.k_pool = (bf16*)k_pool;
        a.v_pool = (bf16*)v_pool;
    }
    switch (tile) {
        case 0: return launch<64, 64, 2, 2, 0, 4, 4, 1>(epilogue, a, parts, stream);
        case 1: return launch<96, 64, 2, 2, 0, 4, 4, 1>(epilogue, a, parts, stream);
        case 2: return launch<128, 64, 2, 2, 0, 4, 4, 1>(epilogue, a, parts, stream);
        case 3: return launch<96, 128, 2, 2, 4, 4, 4, 2>(epilogue, a, parts, stream);
        case 4: return launch<128, 128, 2, 2, 4, 4, 4, 2>(epilogue, a, parts, stream);
        case 5: return launch<160, 192, 2, 2, 4, 3, 3, 1>(epilogue, a, parts, stream);
        case 6: return launch<192, 128, 2, 2, 4, 4, 4, 2>(epilogue, a, parts, stream);
        case 7: return launch<192, 128, 2, 2, 0, 2, 2, 1>(epilogue, a, parts, stream);
        case 8: return launch<256, 128, 2, 2, 4, 3, 4, 2>(epilogue, a, parts, stream);
        case 9: return launch<192, 96, 4, 1, 4, 4, 4, 2>(epilogue, a, parts, stream);
        case 10: return launch<192, 192, 2, 2, 4, 3, 3, 1>(epilogue, a, parts, stream);
        case 11: return launch<256, 256, 2, 4, 0, 2, 2, 1>(epilogue, a, parts, stream);
        case 12: return launch<64, 64, 2, 2, 4, 8, 8, 4>(epilogue, a, parts, stream);
        case 13: return launch<96, 64, 2, 2, 4, 6, 8, 4>(epilogue, a, parts, stream);
        case 14: return launch<128, 64, 2, 2, 4, 4, 8, 4>(epilogue, a, parts, stream);
        case 15: return launch<192, 64, 2, 2, 4, 4, 8, 4>(epilogue, a, parts, stream);
        case 16: return launch<256, 96, 4, 1, 4, 3, 4, 2>(epilogue, a, parts, stream);
    }
    LLMS_REQUIRE(false, "gemm_tiles: no such tile");
}

}  // extern "C"
