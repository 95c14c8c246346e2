// Mapped MoE calls on the tile kernel (tile_gemm.hpp, nint_tile.hpp): activations in row order, the work list, the kernel and its
// launch, shared by the grouped matmul and by its form with the fused act(gate) * up output.
//
// A shared expert is one more expert of the same launches, whose pairs are the tokens in order: as calls of its own its two products cost
// two layouts of the activations, an elementwise launch and ends of launches that nothing else filled (2048 tokens, 8 of 128 experts of
// 2048 x 2048 and 2048 x 1024: 78 us of 454, the block now 409; 256 tokens 160, now 130; 32 experts of 2880 x 2880 at 128 tokens 114, 99).
//
// The (token, route) pairs of an expert are cut into chunks of nearly equal size of at most kMoeTiles row tiles (16 pairs each); a
// block takes one chunk against a tile of the expert's neurons.  One launch runs chunks of every size and cohorts of every
// profile, largest chunks first: the body is chosen per block, so that no launch stands empty and the small chunks fill the end.
//
// 2048 tokens, 8 of 128 experts of 2048 x 2048 gate/up and 2048 x 1024 down in 2 to 5 bits and a shared expert: gate/up 206 us and down
// 132 us; three launches over an older body without this loop took 286 and 208 without the shared expert (chunks of 128 pairs and a
// remainder that unpacked its expert once more), one 198 and 132.  The matrix cores are busy 47 and 35 % of the time, waves wait 20 and
// 26 % of theirs: a block walks a short K (64 to 80 slices) and then has its results to write, and two blocks on a compute unit fill each
// other's start and end in part only.  Three row-blocks per wave instead of two cut that share (202 and 140 us).  61 tokens, 8 of 64
// experts of 4096 x 4096 and 4096 x 2048 and a shared one, a tile or two each: 134 and 80 us, 4.3 and 3.6 TB/s of weights, matrix cores
// 13 and 11 %.  Chunks of five and seven tiles run the bodies of six and eight: 64 experts of those 2048 x 2048 with 72 to 112 pairs each
// are 2 to 27 % faster in every profile than on the bodies of five to eight tiles before.
#pragma once
#include "common.hpp"
#include "nint_body.hpp"
#include "tune.hpp"

namespace mfq {

constexpr int kMaxPools = 8;
struct MoePools {
    NintK k[kMaxPools];
    const uint8_t *w[kMaxPools];
    int spw[kMaxPools];
    int n;
};

constexpr int kMoeTileM = 16;  // (token, route) pairs of one expert per tile of the route map
constexpr int kMoeTiles = 9;   // row tiles of the largest chunk: two blocks of 9 x 8 KB of activations share a compute unit

// Row-blocks of a wave (of units of that many dwords), slices of an LDS stage, stages of the ring and weight units in flight of a body of mt row tiles.  Up to two tiles the
// weight stream sets the pace: four row-blocks share an activation fragment and a whole step of weights is in flight.  Up to four
// the minimum term runs inside the loop (its sums fit the registers).
constexpr int moe_nb(int mt, int dwords) { return dwords > 5 ? 2 : mt <= 2 ? 4 : 3; }
constexpr int moe_sl(int mt) { return mt <= 3 ? 4 : 2; }
constexpr int kMoeRing = 4;
constexpr int moe_sets(int mt, int d) { return d <= 2 || (mt <= 3 && d * moe_nb(mt, d) <= 20) ? 4 : 2; }
constexpr int moe_fused(int mt) { return mt <= 4 ? mt : 0; }
// Nine row tiles of three row-blocks of NINT5-28 are the body that needs the most registers: its act(gate) * up form reloaded eleven
// addresses per step from scratch, each reload behind a wait for every request in flight (64 experts of 2048 x 2048, 136 pairs each:
// 137 us, now 112).  Bodies that do not spill are up to 2 % slower with the shorter addresses.
constexpr bool moe_short(int mt, int d) { return mt >= 9 && d == 5; }
// Few pairs an expert: chunks of at most kMoeFewTiles tiles on a kernel of their own, whose bodies fit half the registers, so that four
// blocks of two row-blocks a wave share a compute unit where two of four did; nothing but the weight stream counts there.
constexpr int kMoeFewTiles = 2, kMoeFewNb = 2;
constexpr int moe_few_sets(int mt, int d) { return mt * d <= 6 ? 4 : 2; }
constexpr int kMoeTableBytes = 2048;  // rows of a chunk: source, destination, scale
constexpr size_t kMoeTileLds = kMoeTableBytes + 1024 * static_cast<size_t>(kMoeTiles * kMoeRing * moe_sl(kMoeTiles));
constexpr size_t kMoeFewLds = kMoeTableBytes + 1024 * static_cast<size_t>(kMoeFewTiles * kMoeRing * moe_sl(kMoeFewTiles));
static_assert(12 * 16 * kMoeTiles <= kMoeTableBytes && 2 * kMoeTileLds <= kMaxDynamicLds, "two blocks per compute unit");

// Activations of a mapped call in row order (GatherCopy), one copy per groupsize among the cohorts:
//     xr[row][slice][kb][8] = x16[row][(4 u + kb) gs + 8 mm ...], slice = u * NM + mm, zeros behind a group's last value and K
//     xg[row][step][kb][8]  = group sums of groups 16 s + 4 j + kb (j = 0..3) as fp16, then what that rounding left out
constexpr int kMoeGroupSizes = 5;  // 16, 24, 28, 32, 48
struct MoeActs {
    int n, gs[kMoeGroupSizes], nsteps[kMoeGroupSizes];
    uint16_t *xr[kMoeGroupSizes], *xg[kMoeGroupSizes];
    int8_t of_pool[kMaxPools];  // which of them a cohort reads
    // Cohorts by bytes per weight, most first: the order in which their chunks of a size run, so that short blocks fill the end.
    // Chunks of one or two tiles run the other way round in the kernel of all sizes (61 tokens, 8 of 64 experts: gate/up 127 us, 138
    // heaviest first); in the one for few pairs, four blocks to a compute unit, heaviest first is the faster (the block 250 us, then 246).
    int8_t turn[kMaxPools];
    float *xscale;
};

// What moe_rows does besides: the list of chunks (lists[0] = their number, lists[4 + 4 i] = {first pair, end of pairs, cohort, expert
// in the cohort} of chunk i; largest first, and those of a cohort, which run the same code, together) and zeros in the output rows of pairs without an expert of these cohorts.
struct MoeRowsArgs {
    MoeActs acts;
    const uint16_t *x;
    int64_t ldx;
    int rows, K, routed, R, n_pairs, E, cap, tiles;  // tiles: of the largest chunk
    int T, shared;  // shared: cohort of a tensor that every token goes through (pair n_pairs + t), or -1
    const int32_t *ids, *expert_pool, *expert_local, *expert_bounds;
    int32_t *lists;
    void *out;
    int64_t ldo;
    int width, out_bytes;  // elements of an output row and their size
};
int moe_rows(const MoeRowsArgs &a, int x_dtype, hipStream_t st);

struct MoeTileArgs {
    NintK k[kMaxPools];
    const uint8_t *w[kMaxPools];
    const uint16_t *xr[kMaxPools], *xg[kMaxPools];
    const float *xscale;
    const int32_t *ids_dst, *lists;
    int out_per_expert, routed, R, ncol, n_pairs;  // pairs from n_pairs on: the tokens, of the tensor that all of them go through
    int row0, n_rows;  // the pass's rows of the activations (a buffer window spans less than 4 GiB)
    void *out;
    int64_t ldo;
    int gelu, f16;
};

// Starts moe_tile_kernel (moe_tile.hpp) for plain results / for act(gate) * up.
int moe_tile_plain(const MoeTileArgs &t, unsigned grid, hipStream_t st);
int moe_tile_glu(const MoeTileArgs &t, unsigned grid, hipStream_t st);
int moe_tile_few_plain(const MoeTileArgs &t, unsigned grid, hipStream_t st);
int moe_tile_few_glu(const MoeTileArgs &t, unsigned grid, hipStream_t st);

inline size_t moe_align256(size_t v) { return (v + 255) & ~static_cast<size_t>(255); }
// Chunks of a call of at most `most` tiles: one per expert with pairs, and one more per `most` row tiles.
inline int moe_chunks(int E, int n_pairs, int most = kMoeTiles) {
    const int hit = E < n_pairs ? E : n_pairs;
    return hit + (n_pairs / kMoeTileM + hit) / most + 1;
}
constexpr int kMoeChunkCap = 18432;  // of the list
constexpr size_t kMoeListBytes = 16 * (1 + kMoeChunkCap);
inline bool moe_prefill_unit(const mfq_nint_desc &d) { return d.kind == 1 || (d.bits == 5 && d.gs == 28); }
inline bool moe_prefill_pools(const mfq_moe_pool *pools, int n_pools) {  // every cohort has a prefill unit
    for (int i = 0; i < n_pools; ++i)
        if (!moe_prefill_unit(pools[i].desc) || 4 * pools[i].desc.rowblock_bytes >= (1ll << 31)) return false;
    return true;
}

// The kernel for few pairs: up to 20 per expert on average, and rows (those of a shared tensor too) for at most kMoeFewBlocks full blocks
// a compute unit: with more, what a chunk of two tiles costs to unpack counts, and not the stream alone.  Whole feed-forward blocks,
// kernel of all sizes / this one, us.
//   Routes spread evenly, no shared expert in the launch: 64 experts of 4096 x 4096 and 4096 x 2048, 8 a token, at 61 / 128 / 160 / 224 /
//   256 tokens (8 / 16 / 20 / 28 / 32 pairs an expert) 261 / 312 / 340 / 382 / 392 and 262 / 309 / 329 / 394 / 450; 128 of 2048 x 2048 and
//   2048 x 1024 at 32 / 192 / 256 / 448 / 512 tokens 158 / 202 / 225 / 251 / 260 and 144 / 188 / 209 / 248 / 276; 32 of 2880 x 2880 and
//   2880 x 1440, 4 a token, at 61 / 128 / 192 / 256 tokens 117 / 141 / 154 / 167 and 95 / 116 / 140 / 173.
//   A shared expert in the launch and few routes a token, so that it has a third or half of the rows: those 128, one route, 320 / 1280 /
//   2048 tokens (1.3 / 5 / 8 blocks a compute unit) 164 / 206 / 225 and 140 / 189 / 221 (with calls of its own for the shared expert,
//   either kernel, 179 / 226 / 247 at best), two, 320 / 1000 / 1280 tokens 175 / 197 / 220 and 154 / 190 / 207; 64 of 4096, one route,
//   320 / 640 / 1280 tokens (2.5 / 5 / 10) 302 / 324 / 388 and 267 / 307 / 380.  128 of 4096, one, 512 / 768 / 1024 / 2560 tokens (4 / 6 /
//   8 / 20) 438 / 483 / 495 / 661 and 438 / 480 / 513 / 720; 256 of 2048 x 2048, one, 1536 / 2048 / 5120 tokens (6 / 8 / 20) 313 / 322 / 432
//   and 309 / 331 / 477.
//   Pairs on a part of the experts, no shared one: 256 of 2048 x 2048, 8 a token, at 4 / 6 / 8 / 10 blocks a compute unit on 8 of them 102 /
//   120 / 126 / 142 and 92 / 110 / 131 / 163, on 128 182 / 200 / 210 / 229 and 165 / 181 / 221 / 274, on all 265 / 282 / 301 / 312 and 254 /
//   269 / 286 / 302; 128 of 4096 on 8 144 / 153 / 190 / 254 and 130 / 160 / 204 / 252, on 64 267 / 312 / 308 / 331 and 253 / 284 / 366 /
//   462, on all 418 / 442 / 467 / 475 and 418 / 438 / 464 / 490.  What an even spread could gain above seven is 6 %, what an uneven one
//   could lose 40 %.
constexpr int kMoeFewBlocks = 7;
inline bool moe_few(int E, int out_per_expert, int n_pairs, int shared_rows) {
    const int64_t rows = n_pairs + static_cast<int64_t>(shared_rows);
    // (a block has 4 waves of kMoeFewNb row-blocks, half of them gate rows where there is a GLU)
    const int64_t blocks = ceil_div(rows, 16 * kMoeFewTiles) * ceil_div(out_per_expert, 64 * kMoeFewNb);
    return n_pairs <= 20 * static_cast<int64_t>(E) && blocks <= static_cast<int64_t>(kMoeFewBlocks) * device_cu_count() &&
           moe_chunks(E + (shared_rows > 0), static_cast<int>(rows), kMoeFewTiles) <= kMoeChunkCap;
}

inline void moe_fill_k(NintK &k, const mfq_nint_desc &d) { k = to_k(&d); }

// Row bytes of a cohort's activations in row order
inline size_t moe_row_bytes(const mfq_nint_desc &d) { return static_cast<size_t>(d.nsteps) * 4 * ((d.gs + 7) / 8) * 64; }

// Workspace of x_rows activation rows, carved at base (null: its size only); 0 when a cohort has no prefill body.
inline size_t moe_prefill_carve(const mfq_moe_pool *pools, int n_pools, int x_rows, uint8_t *base, MoeActs *acts, int32_t **lists) {
    if (!pools || n_pools < 1 || n_pools > kMaxPools || x_rows < 1 || !moe_prefill_pools(pools, n_pools)) return 0;
    const size_t rows = static_cast<size_t>(x_rows);
    size_t at = moe_align256(kMoeListBytes), scale_at = at;
    at += moe_align256(rows * 4);
    MoeActs a{};
    for (int i = 0; i < n_pools; ++i) {
        const mfq_nint_desc &d = pools[i].desc;
        int g = 0;
        while (g < a.n && a.gs[g] != d.gs) ++g;
        a.of_pool[i] = static_cast<int8_t>(g);
        if (g < a.n) continue;
        a.gs[a.n] = d.gs;
        a.nsteps[a.n] = d.nsteps;
        a.xr[a.n] = reinterpret_cast<uint16_t *>(base + at);
        at += moe_align256(rows * moe_row_bytes(d));
        a.xg[a.n++] = reinterpret_cast<uint16_t *>(base + at);
        at += moe_align256(rows * d.nsteps * 64);
    }
    for (int i = 0; i < n_pools; ++i) {
        int t = 0;
        for (int j = 0; j < n_pools; ++j)
            t += pools[j].desc.rowblock_bytes > pools[i].desc.rowblock_bytes || (pools[j].desc.rowblock_bytes == pools[i].desc.rowblock_bytes && j < i);
        a.turn[i] = static_cast<int8_t>(t);
    }
    if (base) {
        a.xscale = reinterpret_cast<float *>(base + scale_at);
        *acts = a;
        *lists = reinterpret_cast<int32_t *>(base);
    }
    return at;
}

// A mapped call can take the tile kernel: every cohort has a body, the chunk list and the activations are within their limits, the
// workspace is large enough.
inline bool moe_prefill_eligible(const mfq_moe_pool *pools, int n_pools, int E, int K, int routed_input, int n_pairs, int T,
                                 const void *workspace, size_t workspace_bytes, bool shared = false) {
    const int all = n_pairs + (shared ? T : 0), x_rows = routed_input ? all : T;
    if (!workspace || !moe_prefill_pools(pools, n_pools) || moe_chunks(E + shared, all) > kMoeChunkCap) return false;
    int64_t k = K;
    for (int i = 0; i < n_pools; ++i) {
        const int64_t whole = static_cast<int64_t>(pools[i].desc.nsteps) * 16 * pools[i].desc.gs;
        if (whole > k) k = whole;
    }
    return static_cast<int64_t>(x_rows) * ceil_div(k, 32) * 64 < (1ll << 32) &&
           workspace_bytes >= moe_prefill_carve(pools, n_pools, x_rows, nullptr, nullptr, nullptr);
}

// P holds the cohorts, with `shared` the last of them a tensor that every token goes through, in rows n_pairs + t of out (and, routed,
// of x); out: float [pairs, ldo], or with glu uint16_t [pairs, ldo].
int moe_prefill_launch(bool glu, const MoePools &P, const mfq_moe_pool *pools, int n_pools, const int32_t *expert_pool,
                       const int32_t *expert_local, int E, int out_per_expert, int K, const void *x, int x_dtype, int64_t ldx,
                       int routed_input, const int32_t *ids, int n_pairs, int T, int R, const int32_t *ids_dst,
                       const int32_t *expert_bounds, void *out, int64_t ldo, int gelu, int f16, void *workspace, bool shared, hipStream_t st);

}  // namespace mfq
