// The composed attention on the matrix cores, bfloat16, where a column meets the values before heads are mixed.
//
// With mixed heads a result is sum_g talk[h, g] sum_j w_g(j) v_h(j).  Mixing the weights w_g first needs them normalised, so
// two walks over the keys, and every head's weights of a token through LDS.  Here each score column g is multiplied with the
// values of *all* key/value heads in one walk, u_g[k] = sum_j w_g(j) v_k(j), and the results are mixed once at the end:
// o_h = sum_g talk[h, g] u_g[kv(h)]: a plain online softmax whose values are kv_heads * dv wide.  Up to 256 columns of values (64
// registers of results a lane) it is the faster way.  Two score maps are the same walk with a map's columns as columns of their
// own, over the values of their key/value head.
//
// Mixing may subtract heads that are nearly alike, and then a rounding of each head's weights is not small beside what is left.  So
// with mixed heads a weight is two bfloat16 numbers, itself rounded and the remainder rounded (2^-18 of it is lost), and the values
// are multiplied with both: at 4 key/value heads of 64, 32 of 36 matrix instructions are value products, where the kernel that
// mixes weights has 4 of 12 in its two walks.  Relative error of the result in the norm against 64 bits, 32 heads of 64 on 4, 100 and
// 1,000 keys: 1.6 to 2.0e-3 for the identity with noise, random matrices, heads minus their mean and minus the next head with
// queries of 0.01 to 1, and pairs of heads subtracted whose queries are 0.01 to 0.3 apart; where the mixed weights are rounded 2.2
// to 2.5e-3; with one rounded number a weight 2.0e-3 to 1.2e-1, the pairs up to 0.7.  A third number changes the fourth digit.
//
// A unit is 16 columns that share a key row: `tpw` neighbouring tokens times the `grp` query heads of a key/value head.  Per
// step of 32 keys (two tiles of 16) a wave forms S^T = K Q^T with v_mfma_f32_16x16x32_bf16, two products whose rows are the keys
// 8 (i / 4) + 4 u + i % 4; a lane then holds keys 8 q4 .. + 7 of the 32 for its column, which is the B operand of O^T = V^T P^T, and the
// values' A operand is one load of 16 bytes.  (With a tile a product, a lane's keys were 4 of each tile and its values two loads of 8: a load
// instruction takes its turn whatever it brings.  Microseconds, 32 heads of 64 on 4: 2 tokens behind 1,278 64 -> 55, 333 tokens 27.2 ->
// 24.9, 2,048 tokens 174 -> 157, 4 single tokens behind 1,000 13.2 -> 12.3; two maps, 2,048 tokens 105 -> 91; 210 tokens behind 890
// 31.9 -> 33.0, and 29.8 since the scores do not wait for the values.)  Pages hold a multiple of 16 keys, so a tile's page and place are scalars, and a lane chooses between two.
//
//   attend_wide_kernel<.., PARTS = true>   requests that bring one token: the keys go to `shares` workgroups, whose maxima, sums
//       and results (32-bit) a second kernel joins: combine_mixed_kernel or combine_maps_kernel.
//   PARTS = false   portions of prompts.  With mixed heads a workgroup holds all heads of its tokens, and mixes in LDS (32-bit
//       matrix instructions), one key/value head's values at a time; else it holds a key/value head's one or two maps.
//
// Why it is a kernel of its own, and a short one: attention_composed_mfma.hip is 31 to 41 KB of straight code that a decoding wave
// goes through once or twice (twice the waves a request and keys asked for a group ahead left its time as it was: it waits for
// its instructions), and its places are looked up lane by lane; this one is 5 to 9 KB.  What bounds it now: for single tokens the
// chain of two launches and of lengths -> table -> keys -> results; for portions the answers to a step's values.
// Measured against that kernel, microseconds (mixed: 32 heads of 64 on 4 key/value heads; maps: 16 heads of two maps of 64 on 2,
// values of 128):
//     4 requests, one token behind   300 keys    mixed 22.1 -> 10.8    maps 18.4 ->  8.5
//     4 requests, one token behind 1,000 keys    mixed 24.9 -> 12.0    maps 31.7 ->  9.4
//   256 requests, one token behind 1,000 keys    mixed  130 ->   66    maps 50.4 -> 50.4 (5 TB/s of keys and values)
//     a prompt of   333 tokens                   mixed  152 ->   23    maps 35.7 -> 12.3
//     a prompt of 2,048 tokens                   mixed  819 ->  152    maps  284 ->   86
// (Mixed with two numbers a weight costs 0 to 8 % more than with one.)  Two maps, whose weights are one number in both kernels, are 2.2 to
// 2.5e-3 from 64 bits in both.
//
// Masks as in attention_composed_mfma.hip: a column at position i sees j <= i with j >= its chunk's start and (i - j < window or
// j < keep_first).
#include "common.h"

#define LOG2E 1.4426950408889634f
#define NOTHING_YET (-1.0e30f)
#define AW_SHARES 16  // most workgroups that share a request's keys
#define AW_NO_KEY 0x40000000
#define AW_AT_ONCE 256  // workgroups: one a compute unit
#define AW_PIECES 2  // of a weight, where heads are mixed behind the value products

typedef __attribute__((ext_vector_type(8))) short s16x8;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8v;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4;

struct WideArgs {
    bf16* out;
    const bf16* q;
    const bf16* k_pool;
    const bf16* v_pool;
    const int* block_tables;
    const int* table_rows;
    const int* cu_seqlens;
    const int* context_lens;
    const float* slopes;
    const float* talk;
    float* ws_o;      // [share][request][heads * maps][DT * 16]
    float* ws_stats;  // [share][request][heads * maps][2]: maximum (units of log 2) and sum
    int out_stride, q_stride, max_blocks;
    int seq_begin, n_seqs;
    int heads, grp, maps, score_heads, heads_per_wg;
    int dv, block_size, k_page, v_page;  // k_page, v_page: elements of a page
    int window, keep_first, chunk;
    int tok, tpw, shares;
    int ordered;  // workgroups go by their keys (`block_of`)
    int talk_at;  // where the mixing matrix lies in LDS (portions of prompts; in floats)
    unsigned bs_magic;  // ceil(2^32 / block_size)
    unsigned tok_magic;  // ceil(2^32 / tok) (0: tok is 1)
    float scale, lambda, eps, out_scale;
    int head_norm, sink;
};

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Four weights of two tiles each as operands of the value products, rounded to bfloat16; the first is the weights rounded, each
// further one what is then left of them.
template <int PIECES>
__device__ __forceinline__ void weight_pieces(float p[2][4], bf16x8v pf[PIECES]) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
        u32x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            float &a = p[e / 2][2 * (e % 2)], &b = p[e / 2][2 * (e % 2) + 1];
            w[e] = pack_bf16x2(a, b);
            a -= __uint_as_float(w[e] << 16), b -= __uint_as_float(w[e] & 0xffff0000u);
        }
        pf[i] = __builtin_bit_cast(bf16x8v, w);
    }
}

__device__ __forceinline__ uint32_t low_half_mask(int keep) { return keep <= 0 ? 0u : keep == 1 ? 0xffffu : 0xffffffffu; }

// Workgroup i's request and block of tokens; the workgroups that find none lie behind all that do.  With a grid of every request's longest
// possible portion, workgroups without tokens lay between those with some, and as workgroups go around the parts of the chip in
// turn, parts of it met only empty ones (32 heads of 64 on 4, microseconds: 811, 890, 150 and 197 tokens 156 -> 91, twice 1,024 beside
// two of 1 token 190 -> 104, without those 104; 16 heads of two maps on 2: 57 -> 48 and 73 -> 56; 77 and 44 are the first and third now).
// One request after the other, each from its last block to its first, where the chip takes all workgroups at once or the requests are more than a
// wave's lanes, whose portions are short.  Otherwise (`ordered`) the block with the i-th most keys, so that no long one begins late, and among equals
// in the order of the requests, so that portions of one length meet the parts of the chip as their requests do and a part reads few requests'
// keys.  A block's height is its place from its request's beginning, in blocks: request s has the heights from .. upto - 1; the height is looked for in
// quarters, a turn of three sums over the lanes.  (The order for up to 8 requests alone, whose sums went over them one by one, and for more one request
// after the other, microseconds: 16 of 64 tokens behind 100, 32 heads of 128 on 8, 20.3 -> 16.1; 32 of 64 behind 300 61 -> 41; 16 of 128, 32 mixed
// heads of 64 on 8 of 32, 48 -> 41, on 4 of 64 42 -> 37.)
// `add` over the numbers of a lane and of those before it.
template <typename F>
__device__ __forceinline__ int up_to_lane(int v, F add) {
    v = add(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true));  // from 1, 2, 4 and 8 lanes before, in rows of 16
    v = add(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true));
    v = add(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true));
    v = add(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true));
    v = add(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));  // the last lane of the row before, and of the half before
    return add(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));
}
__device__ __forceinline__ bool block_of(const WideArgs& a, int i, int lane, int& bi, int& blk, int& row0, int& count, int& end) {
    auto blocks = [&](int tokens) { return a.tok_magic ? (int)__umulhi((unsigned)tokens, a.tok_magic) : tokens; };
    int from, upto, row, tokens, keys;
    auto heights = [&](int base) {  // of request base + lane
        from = upto = row = tokens = keys = 0;
        const int s = a.seq_begin + base + lane;
        if (base + lane >= a.n_seqs) return;
        row = a.cu_seqlens[s], tokens = a.cu_seqlens[s + 1] - row, keys = a.context_lens[s];
        if (keys <= 0 || tokens <= 0) return;
        from = blocks(keys > tokens ? keys - tokens : 0);
        upto = from + blocks(tokens + a.tok - 1);
    };
    auto found = [&](int at, int request, int block) {
        bi = request, blk = block;
        row0 = __builtin_amdgcn_readlane(row, at), count = __builtin_amdgcn_readlane(tokens, at), end = __builtin_amdgcn_readlane(keys, at);
        return true;
    };
    if (a.n_seqs == 1) {  // (nothing to look for: 0.1 microseconds less)
        row0 = a.cu_seqlens[a.seq_begin], count = a.cu_seqlens[a.seq_begin + 1] - row0, end = a.context_lens[a.seq_begin];
        bi = 0, blk = blocks(count + a.tok - 1) - 1 - i;
        return count > 0 && end > 0 && blk >= 0;
    }
    auto sum = [](int x, int y) { return x + y; };
    if (a.ordered) {
        heights(0);
        auto most = [](int x, int y) { return x > y ? x : y; };
        auto over_lanes = [&](int v, auto add) { return __builtin_amdgcn_readlane(up_to_lane(v, add), LLMS_WAVE - 1); };
        auto of_height = [&](int h) { return over_lanes(most(upto - most(from, h), 0), sum); };  // blocks of height h and more
        const int all_blocks = over_lanes(upto - from, sum), highest = over_lanes(upto, most);
        const int depth = over_lanes(upto > from ? highest - from : 0, most);  // (from the highest block down to the lowest)
        if (all_blocks <= i) return false;
        int lo = highest - depth, hi = highest, above = 0;  // a height that more than i blocks reach, and one that `above` blocks do, at most i
        while (hi - lo > 1) {
            const int quarter = (hi - lo + 3) / 4, m1 = lo + quarter, m2 = min(m1 + quarter, hi), m3 = min(m2 + quarter, hi);
            const int n1 = of_height(m1), n2 = of_height(m2), n3 = of_height(m3);
            if (n1 <= i) hi = m1, above = n1;
            else if (n2 <= i) lo = m1, hi = m2, above = n2;
            else if (n3 <= i) lo = m2, hi = m3, above = n3;
            else lo = m3;
        }
        const bool there = from <= lo && lo < upto;
        const unsigned long long all = __ballot(there);
        const int at = __ffsll(__ballot(there && __popcll(all & ((1ull << lane) - 1)) == i - above)) - 1;
        return found(at, at, lo - __builtin_amdgcn_readlane(from, at));
    }
    for (int base = 0; base < a.n_seqs; base += LLMS_WAVE) {
        heights(base);
        const int last = up_to_lane(upto - from, sum);  // behind request base + lane's blocks
        const unsigned long long behind = __ballot(last > i);
        if (behind) {
            const int at = __ffsll(behind) - 1;
            return found(at, base + at, __builtin_amdgcn_readlane(last, at) - 1 - i);
        }
        i -= __builtin_amdgcn_readlane(last, LLMS_WAVE - 1);
    }
    return false;
}

template <int TK, int DT, int U, bool PARTS, bool SHARED, bool MIXED>
__global__ __launch_bounds__(PARTS ? 256 : 512) void attend_wide_kernel(const WideArgs a) {
    extern __shared__ float lds[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / LLMS_WAVE), lane = threadIdx.x % LLMS_WAVE;
    const int nwaves = blockDim.x / LLMS_WAVE;
    const int col = lane % 16, q4 = lane / 16;
    int bi = blockIdx.x, blk = 0, row0, count, end;
    if constexpr (PARTS) {
        row0 = a.cu_seqlens[a.seq_begin + bi], count = a.cu_seqlens[a.seq_begin + bi + 1] - row0, end = a.context_lens[a.seq_begin + bi];
        if (count <= 0 || end <= 0) return;  // (the same for every thread of the workgroup, as below)
    } else if (!block_of(a, blockIdx.x, lane, bi, blk, row0, count, end)) return;
    const int b = a.seq_begin + bi, t0 = blk * a.tok;
    const int ntok = count - t0 < a.tok ? count - t0 : a.tok;
    const int pos_lo = end - count + t0, pos_hi = pos_lo + ntok - 1;
    // (the constant address space: a page's number stays a scalar load also behind a barrier, where the compiler would take it for
    // memory that may have changed, load it as a vector and wait for every load in flight before it)
    const auto table = (const __attribute__((address_space(4))) int*)(uintptr_t)(
        a.block_tables + (size_t)(a.table_rows ? a.table_rows[b] : b) * a.max_blocks);
    const int head = blockIdx.z * a.heads_per_wg + wave;
    if (PARTS && head >= a.score_heads) return;
    const int kvh = head / a.maps, map = head - kvh * a.maps;
    const int share = blockIdx.y, bs = a.block_size;
    constexpr int PIECES = MIXED ? AW_PIECES : 1;
    constexpr int DK = 32 * TK, HALVES = (DT > 8 && !PARTS && !SHARED) ? 2 : 1;  // (16 tiles of values and their results fill a wave's registers)

    // tiles of 16 keys: the kept first keys that the window has passed, then what the first token reaches to the last's own
    const int lo_chunk = a.chunk > 0 ? pos_lo / a.chunk * a.chunk : 0;
    const int lo_win = (a.window > 0 && pos_lo - a.window + 1 > 0) ? pos_lo - a.window + 1 : 0;
    const int main_begin = (lo_chunk > lo_win ? lo_chunk : lo_win) / 16, main_end = pos_hi / 16 + 1;
    const int sink_begin = lo_chunk / 16;
    int sink_end = (a.keep_first + 15) / 16;
    if (sink_end > main_begin) sink_end = main_begin;
    if (a.window <= 0 || sink_end < sink_begin) sink_end = sink_begin;
    const int n_sink = sink_end - sink_begin, n_tiles = n_sink + main_end - main_begin, n_steps = (n_tiles + 1) / 2;
    auto tile_start = [&](int i) { return 16 * (i < n_sink ? sink_begin + i : main_begin + (i - n_sink)); };

    bool valid[U];
    int pos[U], pmin[U], pmax[U], chunk_lo[U];
    bf16x8v qf[U][TK];
    const int h = kvh * a.grp + col % a.grp;
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int first = u * a.tpw, tl = first + col / a.grp;
        valid[u] = col < a.tpw * a.grp && tl < ntok;
        pos[u] = pos_lo + tl;
        pmin[u] = pos_lo + first;
        pmax[u] = pmin[u] + a.tpw - 1 < pos_hi ? pmin[u] + a.tpw - 1 : pos_hi;
        chunk_lo[u] = a.chunk > 0 ? pos[u] / a.chunk * a.chunk : 0;
        const bf16* qrow = a.q + (size_t)(row0 + t0 + tl) * a.q_stride + (size_t)(h * a.maps + map) * DK + 8 * q4;
#pragma unroll
        for (int t = 0; t < TK; ++t)
            qf[u][t] = valid[u] ? *reinterpret_cast<const bf16x8v*>(qrow + 32 * t) : __builtin_bit_cast(bf16x8v, s16x8{0, 0, 0, 0, 0, 0, 0, 0});
    }
    const bool sloped = a.slopes != nullptr;
    const float slope = sloped ? a.slopes[h] * LOG2E : 0.f;
    const float scale2 = a.scale * LOG2E;

    // a lane's keys of a step: as a row of the score products the key 8 (col / 4) + 4 u + col % 4 of product u, as a column of them the
    // keys 8 q4 .. 8 q4 + 7, of 32: both of one tile
    const bool k_second = col >= 8, second = q4 >= 2;
    const int first_key = 8 * (q4 % 2);
    const bf16* k_head = a.k_pool + (size_t)head * bs * DK + (8 * (col / 4 % 2) + col % 4) * DK + 8 * q4;
    const bf16* v_head = a.v_pool + (size_t)(MIXED ? 0 : kvh) * a.dv * bs + col * bs + first_key;
    struct Place {
        int page, in_page;
    };
    // a step's second tile may not exist: it reads the last one again, and its keys lie behind every position
    auto place_of = [&](int i) {
        const int j = tile_start(i < n_tiles ? i : n_tiles - 1), block = (int)__umulhi((unsigned)j, a.bs_magic);
        const int page = table[block];
        return Place{page < 0 ? 0 : page, j - block * bs};
    };
    auto ask_keys = [&](const Place at[2], bf16x8v kf[2][TK]) {
        const size_t rows[2] = {(size_t)at[0].page * a.k_page + at[0].in_page * DK, (size_t)at[1].page * a.k_page + at[1].in_page * DK};
        const bf16* row = k_head + (k_second ? rows[1] : rows[0]);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int t = 0; t < TK; ++t) kf[u][t] = *reinterpret_cast<const bf16x8v*>(row + 4 * u * DK + 32 * t);
    };

    f32x4 o[U][DT];
    float run_m[U], run_l[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        run_m[u] = NOTHING_YET, run_l[u] = 0.f;
#pragma unroll
        for (int d = 0; d < DT; ++d) o[u][d] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // SHARED: a step's values go through LDS (1,500 tokens of 32 heads on 8 of 32: 100 microseconds with or without), [tile][dimension][16 keys] as in a page, in two turns: the waves of the workgroup
    // (one per key/value head) all read all of them.  A chunk is 32 dimensions of a tile, 16 bytes a lane;
    // the two halves of dimensions 8 to 15 of every 16 change places, so that 32 lanes read 64 banks.
    constexpr int CHUNKS = SHARED ? DT / 4 : 1;
    uint16_t* v_lds = reinterpret_cast<uint16_t*>(lds);
    u32x4 staged[CHUNKS];
    int staged_keep[CHUNKS];  // keys of a lane's 8 that lie before the request's end
    auto ask_chunks = [&](const Place at[2], int step) {
#pragma unroll
        for (int i = 0; i < CHUNKS; ++i) {
            const int own = wave + i * nwaves, c = own < DT ? own : DT - 1, tt = c / (DT / 2), dim = 32 * (c - tt * (DT / 2)) + lane / 2;
            const Place& p = tt ? at[1] : at[0];
            staged[i] = *reinterpret_cast<const u32x4*>(a.v_pool + (size_t)p.page * a.v_page + (size_t)dim * bs + p.in_page + 8 * (lane % 2));
            staged_keep[i] = (2 * step + tt < n_tiles ? end - tile_start(2 * step + tt) : 0) - 8 * (lane % 2);
        }
    };
    auto store_chunks = [&](int turn) {
#pragma unroll
        for (int i = 0; i < CHUNKS; ++i) {
            const int c = wave + i * nwaves;
            if (c >= DT) continue;
            u32x4 v = staged[i];
            if (__any(staged_keep[i] < 8)) {  // values behind the request's end may be anything, also NaN
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] &= low_half_mask(staged_keep[i] - 2 * e);
            }
            *reinterpret_cast<u32x4*>(v_lds + turn * (DT * 512) + c * 512 + lane / 2 * 16 + 8 * ((lane ^ (lane >> 4)) & 1)) = v;
        }
    };

    // A step asks for the next step's keys (and values, where they are shared) before anything else; the places of the step after
    // that are looked up at the same time, so that no step waits for a page's number.
    bf16x8v kf[2][TK], next_kf[2][TK];
    Place at[2], next_at[2];
    if (share < n_steps) {
        at[0] = place_of(2 * share), at[1] = place_of(2 * share + 1);
        next_at[0] = place_of(2 * (share + a.shares)), next_at[1] = place_of(2 * (share + a.shares) + 1);
        if constexpr (SHARED) ask_chunks(at, share);
        ask_keys(at, kf);
        if constexpr (SHARED) store_chunks(0);
    }
    if constexpr (MIXED && !PARTS) {  // the mixing matrix, [h][g] with a row of H + 1, behind what else is in LDS: it comes beside the first step's keys
        for (int h0 = wave; h0 < a.heads; h0 += 8 * nwaves)
            for (int g = lane; g < a.heads; g += LLMS_WAVE) {
                float t[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int hr = h0 + e * nwaves;
                    t[e] = a.talk[(size_t)(hr < a.heads ? hr : h0) * a.heads + g];
                }
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    if (h0 + e * nwaves < a.heads) lds[a.talk_at + (h0 + e * nwaves) * (a.heads + 1) + g] = t[e];
            }
    }
    int turn = 0;
    // ALWAYS: the next keys are asked for also where there is no further step (the last tile's again).  With a branch around them the compiler
    // counts on none of them, and the score products wait for the step's values as well.  (Mixed heads and single tokens, but those of 128
    // columns of keys of 64, have enough waves beside one another that the needless keys weigh more: 64 single tokens of 8 heads on 8 of 32
    // behind 1,000 keys 36.5 -> 37.6 microseconds, 16 of two maps of 64 on 2, values of 128, 23.3 -> 22.3.)
    constexpr bool ALWAYS = !MIXED && (!PARTS || (DT == 8 && TK == 2));
    auto walk = [&](int step, bf16x8v (&kf)[2][TK], bf16x8v (&next_kf)[2][TK]) {
        const int next = step + a.shares;
        if constexpr (SHARED) {
            __syncthreads();  // this step's values are in LDS, and the turn before has been read
            if (next < n_steps) ask_chunks(next_at, next);
        }
        u32x4 vf[HALVES][DT / HALVES];
        auto ask_values = [&](int half) {
            const size_t tiles[2] = {(size_t)at[0].page * a.v_page + at[0].in_page, (size_t)at[1].page * a.v_page + at[1].in_page};
            const bf16* vt = v_head + (second ? tiles[1] : tiles[0]) + (size_t)half * (DT / HALVES) * 16 * bs;
#pragma unroll
            for (int d = 0; d < DT / HALVES; ++d) vf[half][d] = *reinterpret_cast<const u32x4*>(vt + (size_t)16 * d * bs);
        };
        if constexpr (!SHARED) ask_values(0);
        if (ALWAYS || next < n_steps) ask_keys(next_at, next_kf);
        if constexpr (SHARED) {  // (all of them, asked for before the scores: their way through LDS passes beside the softmax)
            const uint16_t* from = v_lds + turn * (DT * 512) + (q4 / 2) * (DT * 256) + col * 16 + 8 * ((q4 % 2) ^ (col / 8));
#pragma unroll
            for (int d = 0; d < DT; ++d) vf[0][d] = *reinterpret_cast<const u32x4*>(from + 256 * d);
            __builtin_amdgcn_sched_barrier(0);
        }
        const Place after_at[2] = {place_of(2 * (next + a.shares)), place_of(2 * (next + a.shares) + 1)};
        int j0[2];
        j0[0] = tile_start(2 * step), j0[1] = 2 * step + 1 < n_tiles ? tile_start(2 * step + 1) : AW_NO_KEY;
        const int lane_key = (second ? j0[1] : j0[0]) + first_key;
        bf16x8v pf[U][PIECES];
        float corr[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float sc[2][4], mx = -INFINITY;
            // every column of the unit sees all 32 keys (the same answer in every lane)
            bool whole = true;
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
                whole = whole && j0[tt] + 15 <= pmin[u] && (a.chunk <= 0 || j0[tt] >= pmax[u] / a.chunk * a.chunk) &&
                        (a.window <= 0 || pmax[u] - j0[tt] < a.window);
#pragma unroll
            for (int tt = 0; tt < 2; ++tt) {
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int t = 0; t < TK; ++t) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[tt][t], qf[u][t], acc, 0, 0, 0);
                const int key0 = lane_key + 4 * tt;
#pragma unroll
                for (int r = 0; r < 4; ++r) sc[tt][r] = acc[r] * scale2;
                if (sloped) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) sc[tt][r] -= slope * ((float)(pos[u] - key0) - (float)r);
                }
                if (!whole) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int key = key0 + r;
                        const bool seen = key <= pos[u] && key >= chunk_lo[u] && (a.window <= 0 || pos[u] - key < a.window || key < a.keep_first);
                        sc[tt][r] = seen ? sc[tt][r] : -INFINITY;
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) mx = fmaxf(mx, sc[tt][r]);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16, LLMS_WAVE));
            mx = fmaxf(mx, __shfl_xor(mx, 32, LLMS_WAVE));
            const float m_new = fmaxf(fmaxf(run_m[u], mx), NOTHING_YET);
            corr[u] = fast_exp2(run_m[u] - m_new);
            float p[2][4], sum = 0.f;
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int r = 0; r < 4; ++r) p[tt][r] = fast_exp2(sc[tt][r] - m_new), sum += p[tt][r];
            run_l[u] = run_l[u] * corr[u] + sum;
            run_m[u] = m_new;
            weight_pieces<PIECES>(p, pf[u]);
        }
        if (HALVES == 2) ask_values(1);
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (__any(corr[u] != 1.f)) {
#pragma unroll
                for (int d = 0; d < DT; ++d) o[u][d] *= corr[u];
            }
        const bool tail = j0[0] + 15 >= end || j0[1] + 15 >= end;  // values behind the request's end may be anything, also NaN
#pragma unroll
        for (int half = 0; half < HALVES; ++half) {
            if (!SHARED && tail) {
#pragma unroll
                for (int d = 0; d < DT / HALVES; ++d)
#pragma unroll
                    for (int e = 0; e < 4; ++e) vf[half][d][e] &= low_half_mask(end - lane_key - 2 * e);
            }
#pragma unroll
            for (int d = 0; d < DT / HALVES; ++d) {
                const bf16x8v v = __builtin_bit_cast(bf16x8v, vf[half][d]);
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    f32x4& to = o[u][half * (DT / HALVES) + d];
#pragma unroll
                    for (int i = 0; i < PIECES; ++i) to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, pf[u][i], to, 0, 0, 0);
                }
            }
        }
        if constexpr (SHARED) {
            turn ^= 1;
            if (next < n_steps) store_chunks(turn);
        }
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) at[tt] = next_at[tt], next_at[tt] = after_at[tt];
    };
    if constexpr (!SHARED) {
        // Two steps a turn, whose keys change places: to copy them is to wait for them at the end of each step.  Both together, microseconds, at
        // 2 tokens behind 1,278 others: two maps of 64 on 2, values of 128, 35.1 -> 33.1, on 4, values of 64, 32.5 -> 30.2 (16 heads);
        // 8 mixed heads of 128 on 1 43.2 -> 41.8; 32 of 64 on 4 55.0 -> 53.4; one map of 64 on 4, 7 tokens behind 890, 24.2 -> 22.5.
        // (Shared values wait at a barrier a step either way, and have no registers left.)
        for (int step = share; step < n_steps; step += 2 * a.shares) {
            walk(step, kf, next_kf);
            if (step + a.shares < n_steps) walk(step + a.shares, next_kf, kf);
        }
    } else {
        for (int step = share; step < n_steps; step += a.shares) {
            walk(step, kf, next_kf);
#pragma unroll
            for (int tt = 0; tt < 2; ++tt)
#pragma unroll
                for (int t = 0; t < TK; ++t) kf[tt][t] = next_kf[tt][t];
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
        run_l[u] += __shfl_xor(run_l[u], 16, LLMS_WAVE);
        run_l[u] += __shfl_xor(run_l[u], 32, LLMS_WAVE);
    }

    if constexpr (PARTS) {
        if (!valid[0]) return;
        const size_t at_col = ((size_t)share * a.n_seqs + bi) * (a.heads * a.maps) + h * a.maps + map;
        if (q4 == 0) a.ws_stats[2 * at_col] = run_m[0], a.ws_stats[2 * at_col + 1] = run_l[0];
        float* part = a.ws_o + at_col * (DT * 16) + 4 * q4;
#pragma unroll
        for (int d = 0; d < DT; ++d) *reinterpret_cast<f32x4*>(part + 16 * d) = o[0][d];
    } else if constexpr (!MIXED) {
        // the second map's waves leave their results in LDS, lane by lane, for those of the first with the same columns
        float mul[U];
#pragma unroll
        for (int u = 0; u < U; ++u) mul[u] = 1.f / (a.sink ? run_l[u] + fast_exp2(-run_m[u]) : run_l[u]);
        f32x4* other = reinterpret_cast<f32x4*>(lds) + lane;
        if (a.maps == 2) {
            if (map == 1) {
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int d = 0; d < DT; ++d) other[(u * DT + d) * LLMS_WAVE] = o[u][d] * (mul[u] * a.lambda);
            }
            __syncthreads();
            if (map == 1) return;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float ss = 0.f;
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                o[u][d] *= mul[u];
                if (a.maps == 2) o[u][d] -= other[(u * DT + d) * LLMS_WAVE];
#pragma unroll
                for (int r = 0; r < 4; ++r) ss = fmaf(o[u][d][r], o[u][d][r], ss);
            }
            ss += __shfl_xor(ss, 16, LLMS_WAVE);
            ss += __shfl_xor(ss, 32, LLMS_WAVE);
            const float norm = a.head_norm ? a.out_scale / sqrtf(ss / (float)(DT * 16) + a.eps) : 1.f;
            if (!valid[u]) continue;
            bf16* orow = a.out + (size_t)(row0 + t0 + u * a.tpw + col / a.grp) * a.out_stride + (size_t)h * (DT * 16) + 4 * q4;
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const f32x4 v = o[u][d] * norm;
                *reinterpret_cast<u32x2*>(orow + 16 * d) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            }
        }
    } else {
        // one key/value head's values at a time: [token][head g][dv + 16] in LDS (the pad puts 4 heads on different banks),
        // then a job is a token's 16 dimensions of that key/value head's query heads, 4 heads g an instruction
        const int H = a.heads, dv = a.dv, dvt = dv / 16, pad = dv + 16, G = H / a.grp;
        const float* talk_s = lds + a.talk_at;
        float inv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) inv[u] = 1.f / run_l[u];
        for (int k = 0; k < G; ++k) {
            if (SHARED || k) __syncthreads();
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (valid[u]) {
                    float* at_col = lds + ((size_t)(u * a.tpw + col / a.grp) * H + h) * pad + 4 * q4;
#pragma unroll
                    for (int d = 0; d < DT; ++d)  // (constant indexes of the results: the others are skipped)
                        if ((unsigned)(d - k * dvt) < (unsigned)dvt) *reinterpret_cast<f32x4*>(at_col + 16 * (d - k * dvt)) = o[u][d] * inv[u];
                }
            __syncthreads();
            for (int job = wave; job < ntok * dvt; job += nwaves) {
                const int tl = job / dvt, d0 = 16 * (job - tl * dvt);
                const bool mine = col < a.grp;
                const int ho = k * a.grp + (mine ? col : 0);
                const float* from = lds + (size_t)tl * H * pad + d0 + col;
                f32x4 mixed = {0.f, 0.f, 0.f, 0.f};
                // 4 * quads heads are asked for before the first product: 32, and 8 at a time of what is left (with 32 for every count, 8
                // heads asked for 24 that are not there: 8 on 8 of 32, 2 tokens 15.7 microseconds, 11.8 now, 100 tokens 34.3 and 25.1; 8 of 128
                // on 1, 333 tokens 20.8 and 17.9; 32 on 4 of 64, 333 tokens 24.4 and 23.6)
                auto mix = [&](int g0, auto quads) {
                    constexpr int Q = decltype(quads)::n;
                    float ug[Q], tg[Q];
#pragma unroll
                    for (int e = 0; e < Q; ++e) {
                        const int g = g0 + 4 * e + q4, gr = g < H ? g : H - 1;
                        ug[e] = from[gr * pad], tg[e] = talk_s[ho * (H + 1) + gr];
                        if (g >= H) ug[e] = 0.f, tg[e] = 0.f;
                    }
#pragma unroll
                    for (int e = 0; e < Q; ++e) mixed = __builtin_amdgcn_mfma_f32_16x16x4f32(ug[e], tg[e], mixed, 0, 0, 0);
                };
                int g0 = 0;
                for (; g0 + 32 <= H; g0 += 32) mix(g0, Number<8>());
                for (; g0 < H; g0 += 8) mix(g0, Number<2>());
                if (mine) {
                    *reinterpret_cast<u32x2*>(a.out + (size_t)(row0 + t0 + tl) * a.out_stride + (size_t)ho * dv + d0 + 4 * q4) =
                        u32x2{pack_bf16x2(mixed[0], mixed[1]), pack_bf16x2(mixed[2], mixed[3])};
                }
            }
        }
    }
}

// A column's factors for its shares' results: exp2(m_s - max m) / sum, 0 for a share that saw no key (its results are not used).
template <bool SINK>
__device__ __forceinline__ void share_factors(const float* stats, size_t stride, int shares, float f[AW_SHARES]) {
    float m[AW_SHARES], l[AW_SHARES], top = NOTHING_YET, total = 0.f;
#pragma unroll
    for (int s = 0; s < AW_SHARES; ++s) {
        const float2 ml = *reinterpret_cast<const float2*>(stats + (s < shares ? s : shares - 1) * stride);
        m[s] = ml.x, l[s] = s < shares ? ml.y : 0.f;
    }
#pragma unroll
    for (int s = 0; s < AW_SHARES; ++s) top = fmaxf(top, l[s] > 0.f ? m[s] : NOTHING_YET);
#pragma unroll
    for (int s = 0; s < AW_SHARES; ++s) {
        f[s] = l[s] > 0.f ? fast_exp2(m[s] - top) : 0.f;
        total += f[s] * l[s];
    }
    if (SINK) total += fast_exp2(-top);
    const float inv = 1.f / total;
#pragma unroll
    for (int s = 0; s < AW_SHARES; ++s) f[s] *= inv;
}

// Mixed heads: a workgroup takes one request, the query heads of one key/value head and 16 of its dimensions.
__global__ __launch_bounds__(256) void combine_mixed_kernel(const WideArgs a, int width) {
    extern __shared__ float lds[];  // [g][16 + 4] results, then this key/value head's rows of the mixing matrix [grp][H]
    const int b = a.seq_begin + blockIdx.x, H = a.heads, grp = a.grp, k = blockIdx.y, d0 = k * a.dv + 16 * blockIdx.z;
    const int row = a.cu_seqlens[b];
    if (a.cu_seqlens[b + 1] <= row || a.context_lens[b] <= 0) return;
    float* talk_s = lds + H * 20;
    for (int i = threadIdx.x; i < grp * H; i += blockDim.x) talk_s[i] = a.talk[(size_t)k * grp * H + i];
    for (int i = threadIdx.x; i < 4 * H; i += blockDim.x) {
        const int g = i / 4, c = 4 * (i % 4);
        const size_t col = (size_t)blockIdx.x * H + g, stride = (size_t)a.n_seqs * H;
        f32x4 part[AW_SHARES];
#pragma unroll
        for (int s = 0; s < AW_SHARES; ++s)  // (a share that does not exist reads the last one and counts for nothing)
            part[s] = *reinterpret_cast<const f32x4*>(a.ws_o + (col + (s < a.shares ? s : a.shares - 1) * stride) * width + d0 + c);
        float f[AW_SHARES];
        share_factors<false>(a.ws_stats + 2 * col, 2 * stride, a.shares, f);
        f32x4 u = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < AW_SHARES; ++s) u += f[s] * part[s];
        *reinterpret_cast<f32x4*>(lds + g * 20 + c) = u;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < grp * 16; i += blockDim.x) {
        const int hh = i / 16, d = i % 16;
        float sum = 0.f;
        for (int g = 0; g < H; ++g) sum = fmaf(talk_s[hh * H + g], lds[g * 20 + d], sum);
        a.out[(size_t)row * a.out_stride + (size_t)(k * grp + hh) * a.dv + 16 * blockIdx.z + d] = from_f32<bf16>(sum);
    }
}

// One or two maps: a wave takes a request's head; a half of it is a map, a lane 4 dimensions (dv <= 128).
template <bool SINK>
__global__ __launch_bounds__(64) void combine_maps_kernel(const WideArgs a) {
    const int b = a.seq_begin + blockIdx.x, h = blockIdx.y, lane = threadIdx.x, map = lane / 32, c = 4 * (lane % 32);
    const int row = a.cu_seqlens[b];
    if (a.cu_seqlens[b + 1] <= row || a.context_lens[b] <= 0) return;
    const bool mine = map < a.maps && c < a.dv;
    const int n = a.heads * a.maps;
    const size_t col = (size_t)blockIdx.x * n + h * a.maps + (map < a.maps ? map : 0), stride = (size_t)a.n_seqs * n;
    f32x4 part[AW_SHARES];
#pragma unroll
    for (int s = 0; s < AW_SHARES; ++s)
        part[s] = *reinterpret_cast<const f32x4*>(a.ws_o + (col + (s < a.shares ? s : a.shares - 1) * stride) * a.dv + (mine ? c : 0));
    float f[AW_SHARES];
    share_factors<SINK>(a.ws_stats + 2 * col, 2 * stride, a.shares, f);
    f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < AW_SHARES; ++s) o += f[s] * part[s];
    if (!mine) o = f32x4{0.f, 0.f, 0.f, 0.f};
    float ss = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float other = __shfl_xor(o[r], 32, LLMS_WAVE);
        if (a.maps == 2) o[r] -= a.lambda * other;  // (the upper half's numbers are not used)
        ss = fmaf(o[r], o[r], ss);
    }
#pragma unroll
    for (int mask = 1; mask < 32; mask *= 2) ss += __shfl_xor(ss, mask, LLMS_WAVE);
    const float norm = a.head_norm ? a.out_scale / sqrtf(ss / (float)a.dv + a.eps) : 1.f;
    if (map == 0 && mine) {
        *reinterpret_cast<u32x2*>(a.out + (size_t)row * a.out_stride + (size_t)h * a.dv + c) =
            u32x2{pack_bf16x2(o[0] * norm, o[1] * norm), pack_bf16x2(o[2] * norm, o[3] * norm)};
    }
}

template <int TK, int DT, int U, bool PARTS, bool MIXED, bool SHARED = false>
static int launch_one(const WideArgs& a, dim3 grid, int threads, size_t lds, hipStream_t stream) {
    auto kernel = attend_wide_kernel<TK, DT, U, PARTS, SHARED, MIXED>;
    if (lds > 48 * 1024) LLMS_HIP_CHECK(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    kernel<<<grid, threads, lds, stream>>>(a);
    LLMS_LAUNCH_CHECK();
}

template <int U, bool PARTS, bool MIXED>
static int launch(const WideArgs& a, int dk, int width, dim3 grid, int threads, size_t lds, hipStream_t stream) {
    if constexpr (U == 1 && MIXED) {
        if (width == 256)
            return dk == 64 ? launch_one<2, 16, U, PARTS, MIXED>(a, grid, threads, lds, stream)
                            : launch_one<4, 16, U, PARTS, MIXED>(a, grid, threads, lds, stream);
    }
    LLMS_REQUIRE(width <= 128, "attend_composed_wide: 256 columns of values go with mixed heads and one unit");
    if (dk == 64)
        return width == 64 ? launch_one<2, 4, U, PARTS, MIXED>(a, grid, threads, lds, stream)
                           : launch_one<2, 8, U, PARTS, MIXED>(a, grid, threads, lds, stream);
    return width == 64 ? launch_one<4, 4, U, PARTS, MIXED>(a, grid, threads, lds, stream)
                       : launch_one<4, 8, U, PARTS, MIXED>(a, grid, threads, lds, stream);
}

template <int U, bool PARTS>
static int launch(const WideArgs& a, int dk, int width, dim3 grid, int threads, size_t lds, hipStream_t stream) {
    return a.talk ? launch<U, PARTS, true>(a, dk, width, grid, threads, lds, stream)
                  : launch<U, PARTS, false>(a, dk, width, grid, threads, lds, stream);
}

extern "C" {

// `rows`: rows of q.  `units` > 0: portions of prompts, workgroups of `units` (1, or 2 up to 128 columns of values) units of tokens.  units = 0:
// requests that bring one token, their keys shared out to `shares` workgroups, with the workspaces ws_o and ws_stats.
int llms_attend_composed_wide(void* out, int out_stride, const void* q, int q_stride, const void* k_pool, const void* v_pool,
                              const int* block_tables, const int* table_rows, int max_blocks, const int* cu_seqlens,
                              const int* context_lens, int seq_begin, int n_seqs, int max_new, int rows, int heads, int kv_heads, int maps,
                              int dk, int dv, int block_size, int window, int keep_first, int chunk, float scale,
                              const float* slopes, const float* talk, float lambda, int head_norm, float eps, float out_scale,
                              int sink, int units, int shared, int shares, float* ws_o, float* ws_stats, hipStream_t stream) {
    const int width = talk ? kv_heads * dv : dv;
    LLMS_REQUIRE(n_seqs > 0 && max_new > 0 && rows >= 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && heads / kv_heads <= 16,
                 "attend_composed_wide: up to 16 query heads per key/value head");
    LLMS_REQUIRE((maps == 1 || maps == 2) && !(talk && (maps != 1 || sink || head_norm)), "attend_composed_wide: one or two maps; mixed heads with one, no sink and no norm");
    LLMS_REQUIRE((dk == 64 || dk == 128) && dv > 0 && dv % 16 == 0 && (width == 64 || width == 128 || width == 256) && (talk || dv <= 128),
                 "attend_composed_wide: keys of 64 or 128, values of 64, 128 or 256 a column");
    LLMS_REQUIRE(block_size > 0 && block_size % 16 == 0 && max_blocks > 0, "attend_composed_wide: pages of a multiple of 16 keys");
    LLMS_REQUIRE(q_stride % 8 == 0 && out_stride % 4 == 0, "attend_composed_wide: query rows must be 16-byte aligned, result rows 8-byte");
    LLMS_REQUIRE(window >= 0 && keep_first >= 0 && chunk >= 0, "attend_composed_wide: window, keep_first and chunk are >= 0");
    LLMS_REQUIRE((size_t)kv_heads * maps * block_size * dk < (1u << 31) && (size_t)kv_heads * dv * block_size < (1u << 31),
                 "attend_composed_wide: a page is too large");
    WideArgs a;
    a.out = (bf16*)out, a.q = (const bf16*)q, a.k_pool = (const bf16*)k_pool, a.v_pool = (const bf16*)v_pool;
    a.block_tables = block_tables, a.table_rows = table_rows, a.cu_seqlens = cu_seqlens, a.context_lens = context_lens;
    a.slopes = slopes, a.talk = talk, a.ws_o = ws_o, a.ws_stats = ws_stats;
    a.out_stride = out_stride, a.q_stride = q_stride, a.max_blocks = max_blocks, a.seq_begin = seq_begin, a.n_seqs = n_seqs;
    a.heads = heads, a.grp = heads / kv_heads, a.maps = maps, a.score_heads = kv_heads * maps;
    a.dv = dv, a.block_size = block_size, a.k_page = kv_heads * maps * block_size * dk, a.v_page = kv_heads * dv * block_size;
    a.window = window, a.keep_first = keep_first, a.chunk = chunk;
    a.scale = scale, a.lambda = lambda, a.eps = eps, a.out_scale = out_scale, a.head_norm = head_norm, a.sink = sink;
    a.tpw = 16 / a.grp;
    a.bs_magic = (unsigned)((0x100000000ull + block_size - 1) / block_size);
    if (units > 0) {
        a.heads_per_wg = talk ? kv_heads : maps, a.shares = 1;
        LLMS_REQUIRE((units == 1 || (units == 2 && width <= 128)) && a.heads_per_wg <= 8, "attend_composed_wide: up to 8 waves, of two units up to 128 columns of values");
        a.tok = units * a.tpw, a.tok_magic = a.tok > 1 ? (unsigned)((0x100000000ull + a.tok - 1) / a.tok) : 0;
        const size_t results = (size_t)a.tok * heads * (dv + 16), turns = shared ? (size_t)width * 32 : 0;  // (floats; they take turns in LDS)
        a.talk_at = (int)(results > turns ? results : turns);
        const size_t lds = talk        ? ((size_t)a.talk_at + (size_t)heads * (heads + 1)) * sizeof(float)
                           : maps == 2 ? (size_t)units * 16 * dv * sizeof(float)
                                       : 0;
        LLMS_REQUIRE(lds <= 160 * 1024, "attend_composed_wide: too many heads for the LDS");
        const long most = (long)n_seqs * ((max_new + a.tok - 1) / a.tok), held = rows / a.tok + n_seqs;  // (blocks of portions as long as the longest, and that `rows` rows make)
        const dim3 grid((unsigned)(held < most ? held : most), 1, talk ? 1 : kv_heads);
        a.ordered = n_seqs > 1 && n_seqs <= LLMS_WAVE && (long)grid.x * grid.z > AW_AT_ONCE;
        if (shared) {
            LLMS_REQUIRE(talk && units == 1 && kv_heads >= 4 && dk == 64 && width == 256, "attend_composed_wide: shared values with 4 to 8 mixed key/value heads, keys of 64 and 256 columns of values");
            return launch_one<2, 16, 1, false, true, true>(a, grid, kv_heads * LLMS_WAVE, lds, stream);
        }
        return units == 2 ? launch<2, false>(a, dk, width, grid, a.heads_per_wg * LLMS_WAVE, lds, stream)
                          : launch<1, false>(a, dk, width, grid, a.heads_per_wg * LLMS_WAVE, lds, stream);
    }
    LLMS_REQUIRE(max_new == 1 && shares >= 1 && shares <= AW_SHARES && ws_o && ws_stats, "attend_composed_wide: one token a request, up to 16 shares, and their workspaces");
    a.heads_per_wg = a.score_heads < 4 ? a.score_heads : 4;
    a.tok = 1, a.shares = shares, a.ordered = 0;
    const int zs = (a.score_heads + a.heads_per_wg - 1) / a.heads_per_wg;
    LLMS_REQUIRE(zs <= 65535 && heads <= 65535, "attend_composed_wide: too many heads");
    const size_t mix_lds = ((size_t)heads * 20 + (size_t)a.grp * heads) * sizeof(float);
    LLMS_REQUIRE(!talk || mix_lds <= 48 * 1024, "attend_composed_wide: too many heads for the LDS");
    const int rc = launch<1, true>(a, dk, width, dim3(n_seqs, shares, zs), a.heads_per_wg * LLMS_WAVE, 0, stream);
    if (rc != LLMS_OK) return rc;
    if (talk) combine_mixed_kernel<<<dim3(n_seqs, kv_heads, dv / 16), 256, mix_lds, stream>>>(a, width);
    else if (sink) combine_maps_kernel<true><<<dim3(n_seqs, heads), 64, 0, stream>>>(a);
    else combine_maps_kernel<false><<<dim3(n_seqs, heads), 64, 0, stream>>>(a);
    LLMS_LAUNCH_CHECK();
}

}  // extern "C"
