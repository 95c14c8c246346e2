// Activations of mapped MoE calls in row order and their list of chunks (moe_prefill.hpp).
#include "moe_prefill.hpp"
#include "xfrag.hpp"

namespace mfq {

// A row's share of the threads (t of nt) lays it out for one groupsize.  A thread makes whole 16-byte pieces in the order in which
// they lie, so stores are contiguous; what it reads is a permutation inside four groups, from LDS or for long rows from cache (the row
// was just searched for its maximum).
template <int GS, int XF16, int AT_ONCE>
__device__ __forceinline__ void lay_out_row(const uint16_t *x, int K, int nsteps, float inv, uint16_t *__restrict__ xr,
                                            uint16_t *__restrict__ xg, int t, int nt) {
    constexpr int NM = (GS + 7) / 8;
    const int pieces = nsteps * 16 * NM;
    for (int d0 = t; d0 < pieces; d0 += AT_ONCE * nt) {
        u32x4_t v[AT_ONCE];
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i) {
            const int d = d0 + i * nt, sl = d >> 2, u = sl / NM, mm = sl - u * NM, k0 = (4 * u + (d & 3)) * GS + 8 * mm;
            v[i] = u32x4_t{0u, 0u, 0u, 0u};
            if (d < pieces) {
                if constexpr (GS % 8 == 0) {
                    if (k0 < K) v[i] = *reinterpret_cast<const u32x4_t *>(x + k0);
                } else {
                    if (k0 < K) {
                        const u32x2_t h = *reinterpret_cast<const u32x2_t *>(x + k0);
                        v[i].x = h.x; v[i].y = h.y;
                    }
                    if (8 * mm + 8 <= GS && k0 + 4 < K) {
                        const u32x2_t h = *reinterpret_cast<const u32x2_t *>(x + k0 + 4);
                        v[i].z = h.x; v[i].w = h.y;
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i)
            if (d0 + i * nt < pieces) *reinterpret_cast<u32x4_t *>(xr + 8 * (d0 + i * nt)) = scaled_f16<XF16>(v[i], inv);
    }
    for (int g = t; g < nsteps * 16; g += nt) {
        // pieces of eight values (of four where the groups are no multiple of eight), added in k order
        constexpr int EL = GS % 8 == 0 ? 8 : 4, N = GS / EL;
        u32x4_t v[N];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            v[i] = u32x4_t{0u, 0u, 0u, 0u};
            const int k0 = g * GS + EL * i;
            if (k0 < K) {
                if constexpr (EL == 8) {
                    v[i] = *reinterpret_cast<const u32x4_t *>(x + k0);
                } else {
                    const u32x2_t h = *reinterpret_cast<const u32x2_t *>(x + k0);
                    v[i].x = h.x; v[i].y = h.y;
                }
            }
        }
        float X = 0.f;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const u32x4_t h = scaled_f16<XF16>(v[i], inv);
#pragma unroll
            for (int q = 0; q < EL / 2; ++q) X = dot2<1>(h[q], 0x3c003c00u, X);
        }
        const uint16_t hi = f32_to_f16_rne(X);
        uint16_t *o = xg + ((g >> 4) * 4 + (g & 3)) * 8 + ((g >> 2) & 3);
        o[0] = hi;
        o[4] = f32_to_f16_rne(X - f16_to_f32(hi));
    }
}

// The chunks of all experts, counted and then placed by size and cohort.  An expert of t tiles has n = ceil(t / a.tiles) chunks,
// the first t - n * (t / n) of them one tile larger than the rest.  (The order inside a bucket is that of the atomics: it decides
// when a chunk runs and nothing else.)
__device__ __forceinline__ void list_chunks(const MoeRowsArgs &a) {
    constexpr int NBUCKET = kMoeTiles * kMaxPools;
    static_assert(NBUCKET <= 128, "two buckets per lane");
    __shared__ int bucket[NBUCKET];
    const int tid = threadIdx.x, nt = blockDim.x;
    auto split = [&](int e, int &lo, int &end, int &pool, int &small, int &large_n) -> int {  // number of chunks
        pool = e < a.E ? a.expert_pool[e] : a.shared;
        if (pool < 0) return 0;
        lo = e < a.E ? a.expert_bounds[e] : a.n_pairs;
        end = e < a.E ? a.expert_bounds[e + 1] : a.n_pairs + a.T;
        const int tiles = (end - lo + 15) >> 4, n = (tiles + a.tiles - 1) / a.tiles;
        small = n > 0 ? tiles / n : 0;
        large_n = tiles - n * small;
        return n;
    };
    auto at = [&](int cls, int pool) -> int & {
        const int turn = a.acts.turn[pool];
        return bucket[(kMoeTiles - cls) * kMaxPools + (cls <= 2 && a.tiles > kMoeFewTiles ? kMaxPools - 1 - turn : turn)];
    };
    const int experts = a.E + (a.shared >= 0 ? 1 : 0);
    int lo, end, pool, small, large_n;
    for (int i = tid; i < NBUCKET; i += nt) bucket[i] = 0;
    __syncthreads();
    for (int e = tid; e < experts; e += nt) {
        const int n = split(e, lo, end, pool, small, large_n);
        if (n > 0) atomicAdd(&at(small, pool), n - large_n);
        if (n > 0 && large_n > 0) atomicAdd(&at(small + 1, pool), large_n);
    }
    __syncthreads();
    if (tid < 64) {  // exclusive sums
        const int v0 = 2 * tid < NBUCKET ? bucket[2 * tid] : 0, v1 = 2 * tid + 1 < NBUCKET ? bucket[2 * tid + 1] : 0;
        int inc = v0 + v1;
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(inc, o, 64);
            if (tid >= o) inc += v;
        }
        if (2 * tid < NBUCKET) bucket[2 * tid] = inc - v0 - v1;
        if (2 * tid + 1 < NBUCKET) bucket[2 * tid + 1] = inc - v1;
        if (tid == 63) a.lists[0] = min(inc, a.cap);
    }
    __syncthreads();
    for (int e = tid; e < experts; e += nt) {
        const int n = split(e, lo, end, pool, small, large_n);
        if (n <= 0) continue;
        const int local = e < a.E ? a.expert_local[e] : 0;
        int pos_large = large_n > 0 ? atomicAdd(&at(small + 1, pool), large_n) : 0, pos_small = atomicAdd(&at(small, pool), n - large_n);
        for (int c = 0; c < n; ++c) {
            const int first = lo + 16 * (c * small + min(c, large_n)), last = min(end, first + 16 * (small + (c < large_n ? 1 : 0)));
            const int pos = c < large_n ? pos_large++ : pos_small++;
            if (pos < a.cap) *reinterpret_cast<int4 *>(a.lists + 4 + 4 * pos) = make_int4(first, last, pool, local);
        }
    }
}

constexpr int kMoeKeepWave = 64 * 4 * 8;  // values a wave holds of a row

// Block 0 lists the chunks; the others take WPR waves per activation row: its scale (2^(e - 9), e the exponent of its largest finite
// magnitude), its fp16 values in the order of every groupsize that reads it -- all of them where the routes of a token share the
// row (gridDim.y blocks share them), that of the expert's cohort where a row belongs to one pair -- and zeros in the output rows
// without an expert.
// A row is requested before its expert is looked up; up to kMoeKeepWave values a wave (WHOLE) pass through LDS to their places, where
// they were read from memory once more.  That is bound by the chain of a row's round trips, and by HBM for many rows: 18432 hidden rows
// of 1024 values took 30 us (traced), now 23; the block of 2048 tokens, 8 of 128 experts 408 and now 400; 61 tokens, 8 of 64 experts 241, now 238.
template <int XF16, int WPR, bool WHOLE>
__global__ __launch_bounds__(256) void moe_rows_kernel(MoeRowsArgs a) {
    if (blockIdx.x == 0) {
        if (blockIdx.y == 0) list_chunks(a);
        return;
    }
    constexpr int NT = 64 * WPR, KEEP = kMoeKeepWave / 512;
    __shared__ uint32_t red[4];
    __shared__ u32x4_t kept[WHOLE ? 256 * KEEP : 1];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), m = (blockIdx.x - 1) * (4 / WPR) + (WPR == 1 ? wave : 0);
    const int t = WPR == 1 ? threadIdx.x & 63 : threadIdx.x;
    if (m >= a.rows) return;
    const uint16_t *x = a.x + static_cast<int64_t>(m) * a.ldx;
    const u32x4_t *xv = reinterpret_cast<const u32x4_t *>(x);
    const int nch = a.K >> 3;
    u32x4_t head[KEEP];
#pragma unroll
    for (int i = 0; i < KEEP; ++i) head[i] = xv[min(t + i * NT, nch - 1)];
    auto pool_of = [&](int pair) {
        const int e = a.ids[pair];
        return e >= 0 && e < a.E ? a.expert_pool[e] : -1;
    };
    const int p0 = a.routed ? m : m * a.R, np = a.routed ? (m < a.n_pairs ? 1 : 0) : a.R;
    int pool = a.shared;
    for (int q = 0; q < np; ++q) {
        pool = pool_of(p0 + q);
        if (pool >= 0 || blockIdx.y > 0) continue;
        if (a.out_bytes == 4) {
            float *o = static_cast<float *>(a.out) + (p0 + q) * a.ldo;
            for (int c = t; c < a.width; c += NT) o[c] = 0.f;
        } else {
            uint16_t *o = static_cast<uint16_t *>(a.out) + (p0 + q) * a.ldo;
            for (int c = t; c < a.width; c += NT) o[c] = 0;
        }
    }
    constexpr uint32_t kInf = XF16 ? 0x7c00u : 0x7f80u;
    auto row_max = [&](uint32_t top) {
        for (int o = 32; o > 0; o >>= 1) top = max(top, static_cast<uint32_t>(__shfl_xor(static_cast<int>(top), o, 64)));
        if constexpr (WPR > 1) {
            __syncthreads();
            if ((threadIdx.x & 63) == 0) red[wave] = top;
            __syncthreads();
            top = max(max(red[0], red[1]), max(red[2], red[3]));
        }
        return top;
    };
    u16x2_t big = u16x2_t{0, 0};
    u32x4_t *const row = kept + (WHOLE && WPR == 1 ? wave * 64 * KEEP : 0);
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        if constexpr (WHOLE) row[t + i * NT] = head[i];
        big = pair_top(big, head[i]);
    }
    if constexpr (WHOLE && WPR == 1) wave_sync();  // (else row_max meets)
    for (int c = t + KEEP * NT; !WHOLE && c < nch; c += 4 * NT) {
        u32x4_t v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = xv[min(c + i * NT, nch - 1)];
#pragma unroll
        for (int i = 0; i < 4; ++i) big = pair_top(big, v[i]);
    }
    uint32_t top = row_max(max(big.x, big.y));
    if (top >= kInf) {  // infinities and NaNs (rare) are left out
        top = 0;
        for (int c = t; c < nch; c += NT) top = finite_top<XF16>(top, xv[c]);
        top = row_max(top);
    }
    const int e = row_exp<XF16>(top);
    const float inv = ldexpf(1.f, 9 - e);
    if (t == 0 && blockIdx.y == 0) a.acts.xscale[m] = ldexpf(1.f, e - 9);
    const int first = a.routed ? (pool >= 0 ? a.acts.of_pool[pool] : a.acts.n) : static_cast<int>(blockIdx.y);
    const int last = a.routed ? min(first + 1, a.acts.n) : a.acts.n;
    const uint16_t *from = WHOLE ? reinterpret_cast<const uint16_t *>(row) : x;
    for (int g = first; g < last; g += gridDim.y) {
        const int nsteps = a.acts.nsteps[g];
        uint16_t *xg = a.acts.xg[g] + static_cast<int64_t>(m) * nsteps * 32;
        switch (a.acts.gs[g]) {
#define MFQ_ROW_GS(G)                                                                                                                              \
    case G:                                                                                                                                        \
        lay_out_row<G, XF16, WHOLE ? 2 : 4>(from, a.K, nsteps, inv, a.acts.xr[g] + static_cast<int64_t>(m) * nsteps * (128 * ((G + 7) / 8)), xg, t, NT); \
        break;
            MFQ_ROW_GS(16) MFQ_ROW_GS(24) MFQ_ROW_GS(28) MFQ_ROW_GS(32) MFQ_ROW_GS(48)
#undef MFQ_ROW_GS
        }
    }
}

int moe_rows(const MoeRowsArgs &a, int x_dtype, hipStream_t st) {
    // a wave per row from the number of rows on that fills the chip that way
    const bool per_wave = a.rows >= 8 * device_cu_count();
    const dim3 grid(static_cast<unsigned>(1 + (per_wave ? ceil_div(a.rows, 4) : a.rows)),
                    static_cast<unsigned>(!per_wave && !a.routed && a.rows < 2 * device_cu_count() ? a.acts.n : 1));
    const bool whole = a.K <= (per_wave ? kMoeKeepWave : 4 * kMoeKeepWave), f16 = x_dtype == MFQ_X_F16;
    auto start = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, a); };
    if (per_wave) {
        if (f16) whole ? start(moe_rows_kernel<1, 1, true>) : start(moe_rows_kernel<1, 1, false>);
        else whole ? start(moe_rows_kernel<0, 1, true>) : start(moe_rows_kernel<0, 1, false>);
    } else {
        if (f16) whole ? start(moe_rows_kernel<1, 4, true>) : start(moe_rows_kernel<1, 4, false>);
        else whole ? start(moe_rows_kernel<0, 4, true>) : start(moe_rows_kernel<0, 4, false>);
    }
    return check_launch("moe_rows");
}

int moe_prefill_launch(bool glu, const MoePools &P, const mfq_moe_pool *pools, int n_pools, const int32_t *expert_pool,
                              const int32_t *expert_local, int E, int out_per_expert, int K, const void *x, int x_dtype,
                              int64_t ldx, int routed_input, const int32_t *ids, int n_pairs, int T, int R, const int32_t *ids_dst,
                              const int32_t *expert_bounds, void *out, int64_t ldo, int gelu, int f16, void *workspace, bool shared,
                              hipStream_t st) {
    const int all = n_pairs + (shared ? T : 0), x_rows = routed_input ? all : T;
    const int rbs = glu ? out_per_expert / 32 : out_per_expert / 16;
    MoeRowsArgs a{};
    moe_prefill_carve(pools, n_pools, x_rows, static_cast<uint8_t *>(workspace), &a.acts, &a.lists);
    a.x = static_cast<const uint16_t *>(x); a.ldx = ldx; a.rows = x_rows; a.K = K; a.routed = routed_input; a.R = R;
    const bool few = moe_few(E, out_per_expert, n_pairs, all - n_pairs);
    a.T = T; a.shared = shared ? n_pools - 1 : -1;
    a.n_pairs = n_pairs; a.E = E; a.cap = kMoeChunkCap; a.tiles = few ? kMoeFewTiles : kMoeTiles;
    a.ids = ids; a.expert_pool = expert_pool; a.expert_local = expert_local; a.expert_bounds = expert_bounds;
    a.out = out; a.ldo = ldo; a.width = rbs * 16; a.out_bytes = glu ? 2 : 4;
    if (int rc = moe_rows(a, x_dtype, st)) return rc;
    MoeTileArgs t{};
    size_t row_bytes = 1;
    int dwords = 0;
    for (int i = 0; i < n_pools; ++i) {
        t.k[i] = P.k[i];
        t.w[i] = P.w[i];
        if (pools[i].desc.dwords > dwords) dwords = pools[i].desc.dwords;
        if (moe_row_bytes(pools[i].desc) > row_bytes) row_bytes = moe_row_bytes(pools[i].desc);
    }
    t.ids_dst = ids_dst; t.lists = a.lists; t.xscale = a.acts.xscale;
    t.out_per_expert = out_per_expert; t.routed = routed_input; t.R = R; t.n_pairs = n_pairs; t.out = out; t.ldo = ldo; t.gelu = gelu; t.f16 = f16;
    t.ncol = static_cast<int>(ceil_div(rbs, (glu ? 2 : 4) * (few ? kMoeFewNb : moe_nb(kMoeTiles, dwords))));
    const unsigned grid = static_cast<unsigned>(ceil_div(moe_chunks(E + shared, all, a.tiles), 8) * 8 * t.ncol);
    const int per_pass = static_cast<int>(0xffffffffull / row_bytes);
    for (t.row0 = 0; t.row0 < x_rows; t.row0 += per_pass) {
        t.n_rows = x_rows - t.row0 < per_pass ? x_rows - t.row0 : per_pass;
        for (int i = 0; i < n_pools; ++i) {
            const int g = a.acts.of_pool[i];
            t.xr[i] = a.acts.xr[g] + t.row0 * moe_row_bytes(pools[i].desc) / 2;
            t.xg[i] = a.acts.xg[g] + static_cast<size_t>(t.row0) * pools[i].desc.nsteps * 32;
        }
        if (int rc = few ? (glu ? moe_tile_few_glu(t, grid, st) : moe_tile_few_plain(t, grid, st)) : glu ? moe_tile_glu(t, grid, st) : moe_tile_plain(t, grid, st)) return rc;
    }
    return MFQ_OK;
}

}  // namespace mfq
