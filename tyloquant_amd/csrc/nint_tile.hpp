// Packed NINT weights as a policy of the tile kernel (tile_gemm.hpp): a wave's row-blocks are read straight from HBM in
// the R16 layout and decoded in registers, one slice ahead of the matrix cores.
//
// Measured on NINT4-32 with random codes and normal activations, kernel alone, the quickest of twelve in a row on one card: 12288 x 4096
// at 512 / 2048 rows 56 / 171 us (0.92 / 1.2 PFLOP/s), gate/up 24576 x 4096 with the GLU at 2048 rows 338 us, 4096 x 12288 at 128 / 512 /
// 2048 rows 21 / 51 / 170 us.  At 2048 rows the clock falls as they repeat (medians 178, 398 and 204), and cards differ by up to 9 %.  The
// tile of eight waves side by side with two row-blocks each took 60 / 205, 430 and 40 / 80 / 190 on a card of its time.
// With the GLU at 2048 rows the matrix cores are busy 67 % of the time at 1.9 GHz (2.4 nominal: random data), with 2.8 vector-ALU and a
// quarter of an LDS instruction per matrix-core instruction; 4096 x 12288 61 % and 2.5, NINT5-28 and NINT3-24 tensors at 1024 rows 36 and
// 49 %, 3.3 and 3.1: there it is the walk of one tile through K.
#pragma once
#include "tile_gemm.hpp"

namespace mfq {

// D dwords of a lane's unit; UNI: constants in the scalar offset
template <int D, bool UNI>
__device__ __forceinline__ void tile_load_unit(__amdgpu_buffer_rsrc_t win, uint32_t voff, int soff, uint32_t (&q)[D]) {
#pragma unroll
    for (int i = 0; i + 4 <= D; i += 4) {
        const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(win, UNI ? voff : voff + 4 * i, UNI ? soff + 4 * i : soff, 0);
        q[i] = v.x; q[i + 1] = v.y; q[i + 2] = v.z; q[i + 3] = v.w;
    }
    constexpr int I = D / 4 * 4;
    if constexpr (UNI) soff += 4 * I;
    else voff += 4 * I;
    if constexpr (D % 4 == 3) {
        const auto v = __builtin_amdgcn_raw_buffer_load_b96(win, voff, soff, 0);
        q[I] = v[0]; q[I + 1] = v[1]; q[I + 2] = v[2];
    } else if constexpr (D % 4 == 2) {
        const u32x2_t v = __builtin_amdgcn_raw_buffer_load_b64(win, voff, soff, 0);
        q[I] = v.x; q[I + 1] = v.y;
    } else if constexpr (D % 4 == 1) {
        q[I] = __builtin_amdgcn_raw_buffer_load_b32(win, voff, soff, 0);
    }
}
template <int D>
constexpr int tile_unit_loads() { return (D + 3) / 4; }

// SLV, SETS: slices of a stage and units in registers where the defaults are not wanted.  MF > 0: the minimum term of MF row tiles
// runs inside the loop, into sums of its own (s2): one more instruction per step, row tile and row-block on the scales that the
// codes need anyway, and the group sums straight from memory a step ahead.  It saves the pass over the scales ahead of the loop,
// which tiles with few rows notice, where the weights and not the matrix cores set the pace.
// UNI: for bodies that are short of registers.  What is the same for the wave in the address of a request goes into its scalar offset,
// where otherwise the lane's offset plus each row-block's, constants included, take a vector register apiece over the whole loop; and
// the addresses of what follows the loop are computed after it.
template <class U, int NB, int SLV = 0, int SETS = 0, int MF = 0, bool UNI = false>
struct NintTileB {
    static constexpr bool SHORT = UNI;
    static constexpr int NBLK = NB, D = U::D, NM = U::NPAIR / 4, BITS = U::CBITS;
    static constexpr int NCLS = BITS == 0 ? 1 : (BITS == 3 ? 3 : 2);
    // Eight-bit codes times a sub-scale need up to 16 bits where fp16 has 11, so they are decoded around 128: the one rounding
    // then falls on a number of the finished weight's size (error against 64 bits 2.1e-4; 2.6e-4 with uniform codes and 5.2e-4
    // with quantized normal weights where code * sub_scale itself was rounded).  The body adds back what the centre took off.
    static constexpr int CENTER = U::CODE_BITS == 8 ? 128 : 0, BIAS = 16 + CENTER / 64;  // BIAS: (1024 + CENTER) / 64
    static constexpr int STEP = 4 * NM, SL = SLV ? SLV : NM % 2 == 0 ? 2 : 3, NBUF = 2, MINF = MF;
    // sub-steps (units) in registers: the one being decoded and those in flight
    static constexpr int NSET = SETS ? SETS : D <= 2 ? 4 : 2;
    __amdgpu_buffer_rsrc_t win;
    uint32_t qoff[NB], toff, soff_lane, lane_q;  // byte offsets inside the window: row-block, the lane's tail, scales, unit
    int sb, s_last;
    uint32_t q[NSET][NB][D], tails[NB], tailsn[NB], sx[NB], sy[NB];
    half2_t S[NB], C[NB], Sc[NCLS], Cc[NCLS];
    u32x4_t bf[2][NB];
    __amdgpu_buffer_rsrc_t gwin;
    uint32_t goff[MF ? MF : 1];
    u32x4_t xg[MF ? MF : 1], bm[MF ? NB : 1];
    float4_t s2[MF ? MF : 1][NB];

    // vector-memory requests of issue<i>
    static constexpr int loads(int i) {
        const int j = i / NM, mm = i % NM;
        int n = 0;
        if (mm == NM - 1) n += NB * tile_unit_loads<D>();
        if (mm == 0 && j == 1) n += NB * (U::TAIL ? 2 : 1);
        if (mm == 0 && j == 3) n += NB;
        if (i == 1) n += MF;
        return n;
    }
    static constexpr int loads_before(int i, int n) {  // of the n slices before slice i
        int t = 0;
        for (int d = 1; d <= n; ++d) t += loads(((i - d) % STEP + STEP) % STEP);
        return t;
    }
    __device__ static __forceinline__ float4_t mfma(u32x4_t b, u32x4_t a, float4_t c) { return mfma16(b, a, c); }

    // Row-blocks rb0 + b of the tensor; those at or past rb_end repeat the last one (nobody stores their sums), so that
    // every request lies inside the tensor.
    __device__ __forceinline__ void init(const NintK &k, const uint8_t *wt, int rb0, int rb_end, int lane) {
        const uint32_t rbb = static_cast<uint32_t>(k.rowblock_bytes);
        const int rw = min(rb0, rb_end - 1), n = min(NB, rb_end - rw);
        sb = static_cast<int>(k.step_bytes);
        s_last = k.nsteps - 1;
        win = wave_window(wt + static_cast<int64_t>(rw) * k.rowblock_bytes, n * rbb);
#pragma unroll
        for (int b = 0; b < NB; ++b) qoff[b] = min(b, n - 1) * rbb;
        toff = 1024u * D + lane * 4u;
        soff_lane = 1024u * D + (U::TAIL ? 256u : 0u) + lane * 8u;
        lane_q = lane * (D * 4u);
    }
    // Minimum term inside the loop: group sums in row order, 64 bytes per row and step; off[a]: the lane's bytes of row tile a.
    __device__ __forceinline__ void init_min(__amdgpu_buffer_rsrc_t group_sums, const uint32_t (&off)[MF ? MF : 1], int s) {
        gwin = group_sums;
#pragma unroll
        for (int a = 0; a < MF; ++a) {
            goff[a] = off[a];
#pragma unroll
            for (int b = 0; b < NB; ++b) s2[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};
        }
        load_sums(s);
    }
    __device__ __forceinline__ void load_sums(int s) {
        const int so = __builtin_amdgcn_readfirstlane(min(s, s_last) * 64);
#pragma unroll
        for (int a = 0; a < MF; ++a) xg[a] = __builtin_amdgcn_raw_buffer_load_b128(gwin, goff[a], so, 0);
    }
    __device__ __forceinline__ void load_units(int u, uint32_t (&dst)[NB][D]) {  // unit u = 4 * step + j
        const int so = __builtin_amdgcn_readfirstlane(min(u >> 2, s_last) * sb + (u & 3) * 256 * D);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if constexpr (UNI) tile_load_unit<D, true>(win, lane_q, __builtin_amdgcn_readfirstlane(so + qoff[b]), dst[b]);
            else tile_load_unit<D, false>(win, qoff[b] + lane_q, so, dst[b]);
        }
    }
    template <int HALF>
    __device__ __forceinline__ void load_scales(int s, uint32_t (&dst)[NB]) {
        const int so = __builtin_amdgcn_readfirstlane(min(s, s_last) * sb);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if constexpr (UNI) dst[b] = __builtin_amdgcn_raw_buffer_load_b32(win, soff_lane, __builtin_amdgcn_readfirstlane(so + qoff[b] + 4 * HALF), 0);
            else dst[b] = __builtin_amdgcn_raw_buffer_load_b32(win, qoff[b] + soff_lane + 4 * HALF, so, 0);
        }
    }
    __device__ __forceinline__ void load_tails(int s, uint32_t (&dst)[NB]) {
        const int so = __builtin_amdgcn_readfirstlane(min(s, s_last) * sb);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            dst[b] = 0;
            if constexpr (U::TAIL && UNI) dst[b] = __builtin_amdgcn_raw_buffer_load_b32(win, toff, __builtin_amdgcn_readfirstlane(so + qoff[b]), 0);
            else if constexpr (U::TAIL) dst[b] = __builtin_amdgcn_raw_buffer_load_b32(win, qoff[b] + toff, so, 0);
        }
    }
    __device__ __forceinline__ void prologue(int s) {
#pragma unroll
        for (int u = 0; u < NSET; ++u) load_units(4 * s + u, q[u]);
        load_scales<0>(s, sx);
        load_scales<1>(s, sy);
        load_tails(s, tails);
    }
    // sub_min bytes of a step as an fp16 fragment: groups j = 0 .. 3, twice (the halves of the group sums)
    __device__ static __forceinline__ u32x4_t min_fragment(uint32_t x, uint32_t y) {
        const uint32_t b01 = __builtin_bit_cast(uint32_t, pk_h2(ubyte_f32(x, 1), ubyte_f32(x, 3)));
        const uint32_t b23 = __builtin_bit_cast(uint32_t, pk_h2(ubyte_f32(y, 1), ubyte_f32(y, 3)));
        return u32x4_t{b01, b23, b01, b23};
    }
    // scale and bias of sub-step j: S = sub_scale / 64, C = -1024 S, both exact, from the byte dropped into the mantissa of
    // 1024.0; those of a pair whose field sits at mantissa offset o are 2^-o times that and made per fragment.  Centred codes:
    // C = -1152 S, rounded to fp16 (exact up to sub_scale = 227).
    __device__ __forceinline__ void scales(int b, int j) {
        uint32_t scw = (j < 2) ? sx[b] : sy[b];
        asm volatile("" : "+v"(scw));
        const uint32_t sel = 0x03000100u | ((4u + 2u * (j & 1)) << 16) | (4u + 2u * (j & 1));
        const half2_t X = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(scw, kMagicH2, sel));
        const _Float16 f = static_cast<_Float16>(1.f / 64.f), g16 = static_cast<_Float16>(16.f), g = static_cast<_Float16>(1.f * BIAS),
                       h = static_cast<_Float16>(1024.f * BIAS);
        S[b] = __builtin_elementwise_fma(X, half2_t{f, f}, half2_t{-g16, -g16});
        C[b] = __builtin_elementwise_fma(X, half2_t{-g, -g}, half2_t{h, h});
    }
    // pairs [p0, p1) (4 per row-block) of the fragments of slice (j, mm) of unit set `set`
    template <int P0, int P1, int J, int MM, int SET>
    __device__ __forceinline__ void decode(u32x4_t (&dst)[NB]) {
        static_for<P1 - P0>([&](auto P) {
            constexpr int p = P0 + P.value, b = p / 4, t = p % 4;
            // The codes of a row-block become visible to the compiler here and not earlier: the unpack has no side effects,
            // and hoisted to where the unit arrives it would keep a whole unit of pairs in registers.
            if constexpr (t == 0) {
                if constexpr (BITS == 4) asm volatile("" : "+v"(q[SET][b][MM]));
                else
#pragma unroll
                    for (int d = 0; d < D; ++d) asm volatile("" : "+v"(q[SET][b][d]));
            }
            if constexpr (MM == 0 && t == 0) scales(b, J);
            if constexpr (t == 0) {
#pragma unroll
                for (int c = 0; c < NCLS; ++c) {
                    const _Float16 f = static_cast<_Float16>(1.f / static_cast<float>(1 << (BITS * c)));
                    Sc[c] = c ? S[b] * half2_t{f, f} : S[b];
                    Cc[c] = c ? C[b] * half2_t{f, f} : C[b];
                }
            }
            uint32_t v[U::NPAIR];
            U::unpack(q[SET][b], (tails[b] >> (8 * J)) & 0xffu, v);
            dst[b][t] = __builtin_bit_cast(uint32_t, h2_fma(v[4 * MM + t], Sc[U::cls(4 * MM + t)], Cc[U::cls(4 * MM + t)]));
        });
    }
    __device__ __forceinline__ void first(int) { decode<0, 4 * NB, 0, 0, 0>(bf[0]); }
    template <int I>
    __device__ __forceinline__ void issue(int s) {
        constexpr int j = I / NM, mm = I % NM;
        if constexpr (mm == NM - 1) load_units(4 * s + j + NSET, q[j % NSET]);
        if constexpr (mm == 0 && j == 1) {
            load_scales<0>(s + 1, sx);
            if constexpr (U::TAIL) load_tails(s + 1, tailsn);
        }
        if constexpr (mm == 0 && j == 3) load_scales<1>(s + 1, sy);
        if constexpr (MF > 0 && I == 1) load_sums(s + 1);
    }
    template <int I, int PART, int PARTS>
    __device__ __forceinline__ void produce(int) {
        constexpr int n = (I + 1) % STEP, j = n / NM, mm = n % NM;
        if constexpr (U::TAIL && n == 0 && PART == 0) {
#pragma unroll
            for (int b = 0; b < NB; ++b) tails[b] = tailsn[b];
        }
        if constexpr (MF > 0 && I == 0) {  // both halves of the step's scales are here, the next ones not yet requested
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if constexpr (PART == 0) bm[b] = min_fragment(sx[b], sy[b]);
                s2[PART][b] = mfma16(bm[b], xg[PART], s2[PART][b]);
            }
        }
        decode<PART * 4 * NB / PARTS, (PART + 1) * 4 * NB / PARTS, j, mm, j % NSET>(bf[(I + 1) & 1]);
    }
    template <int MT>
    __device__ static __forceinline__ void schedule() {
        __builtin_amdgcn_sched_barrier(0);
    }
};

// What a launch works on.  With GLU the tensor is a [2 W, K] gate/up pair: rb_half = W / 16 row-blocks of gate rows, then as
// many of up rows, and y is uint16_t [M, ldy].
struct NintTileArgs {
    NintK k;
    const uint8_t *w;
    const uint16_t *xf, *xg;  // fragment-ordered activations and group sums (x_frag)
    const float *xscale;
    void *y;
    int64_t ldy, zstride;     // zstride: floats between the partial results of two splits over K
    int M, spz;               // steps per split
    int rb_half, gelu, f16;
};

// The activation rows of a tile: consecutive ones in fragment order, or any rows in row order (tile_gemm.hpp).
struct FragRows {
    const uint16_t *xf, *xg;
    const float *xscale;
    int mb0, mb_total, M;
    static constexpr bool PAIRED = true;
    template <int MBS, int SL, int NW> using Copy = TileCopy<MBS, SL, NW>;
    __device__ __forceinline__ uint32_t lane_off(int lane) const { return static_cast<uint32_t>(lane) * 16u; }
    __device__ __forceinline__ int request() const { return 0; }
    __device__ __forceinline__ float tables(int) const { return 0.f; }
    __device__ __forceinline__ void scales(float) const {}
    template <class C>
    __device__ __forceinline__ void init(C &c, const uint16_t *x, int slices, int lane, int wave) const {
        c.init(x, slices, mb0, mb_total, lane, wave);
    }
    __device__ __forceinline__ float scale(int a, int r) const { return xscale[min(mb0 + a, mb_total - 1) * 16 + r]; }
    __device__ __forceinline__ int dst(int a, int r) const {  // row of y, or -1
        const int m = (mb0 + a) * 16 + r;
        return m < M ? m : -1;
    }
};
struct GatherRows {
    const uint16_t *xf, *xg;
    const float *xscale;
    const int32_t *pairs;    // the tile's rows of y, n of them (null: first, first + 1, ...)
    int n, per_src;          // rows of y that share a row of xf
    int row0, n_rows;        // first row and rows of xf / xg / xscale; a row of y whose source lies outside is not this call's
    int *srcv, *dstv;        // LDS tables of the tile's rows: row of xf / xg / xscale (always valid), row of y or -1,
    float *scalev;           // xscale of the row
    int entries;             // of the tables
    int first;
    // The tables, in pieces between which other requests go: the rows, their indices, their scales.
    __device__ __forceinline__ int request() const {
        const int i = min(static_cast<int>(threadIdx.x), n - 1);
        return pairs ? pairs[i] : first + i;
    }
    __device__ __forceinline__ float tables(int pair) const {
        const int src = pair / per_src - row0;
        const bool mine = src >= 0 && src < n_rows;
        if (static_cast<int>(threadIdx.x) < entries) {
            srcv[threadIdx.x] = mine ? src : 0;
            dstv[threadIdx.x] = mine && static_cast<int>(threadIdx.x) < n ? pair : -1;
        }
        // a bare barrier: the fence of __syncthreads would wait for the weights
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        return xscale[mine ? src : 0];
    }
    __device__ __forceinline__ void scales(float s) const {
        if (static_cast<int>(threadIdx.x) < entries) scalev[threadIdx.x] = s;
    }
    static constexpr bool PAIRED = false;
    template <int MBS, int SL, int NW> using Copy = GatherCopy<MBS, SL, NW>;
    __device__ __forceinline__ uint32_t lane_off(int lane) const { return row_order_lane(lane); }
    template <class C>
    __device__ __forceinline__ void init(C &c, const uint16_t *x, int slices, int lane, int wave) const {
        c.init(x, slices, srcv, n_rows, lane, wave);
    }
    __device__ __forceinline__ float scale(int a, int r) const { return scalev[16 * a + r]; }
    __device__ __forceinline__ int dst(int a, int r) const { return dstv[16 * a + r]; }
};

// Where the neurons of a tile lie and where its results go: output row-blocks [0, rbs) are the row-blocks rb_first + ... of the
// tensor, with GLU the gate ones followed by as many up ones; cols = columns of y that are stored.
struct TileOut {
    int rb_first, rbs, cols;
    void *y;
    int64_t ldy;
    int gelu, f16;
};

// One tile: the 16 * MT activation rows of `rows` against NW * NB row-blocks of the tensor, from output row-block tn * NWN * NB on.
//     y = xscale[m] * 64 ns[n] * (S1 - nm[n] / (64 ns[n]) * S2),  S1 = sum of sub_scale * code / 64 * x,
//     S2 = sum_g sub_min_g * X_g
// S2 runs first, through the same accumulators, which are then multiplied by -nm / (64 ns) per neuron.  A neuron with
// ns = 0 has no S1; 2^-80 in its place makes what S1 adds vanish next to a minimum term (and the factor 64 ns is 0 where
// nm is 0 too).  Codes decoded around a centre: S1 also gets sum_g (-C_g - 16 sub_scale_g) X_g, one more instruction per step
// and fragment here; it goes straight into the accumulators, so S2 takes registers of its own for a chunk of steps.
// GLU: the lower half of the waves takes gate row-blocks, the upper half the matching up row-blocks; they exchange results in the
// ring's LDS.
// B::MINF > 0: S2 runs inside the K loop, in row order only, and the two terms meet as y = xscale * (64 ns * S1 - nm * S2).
template <class B, int NW, int MT, int R, bool GLU, class Rows>
__device__ __forceinline__ void nint_tile_body(const NintK &k, const uint8_t *wt, const Rows &rows, const TileOut &out, int tn, int s_begin,
                                               int s_end, uint8_t *lds) {
    constexpr int NB = B::NBLK;
    constexpr bool FUSED = B::MINF > 0;
    static_assert(!FUSED || (B::MINF == MT && B::CENTER == 0), "the minimum term of every row tile");
    constexpr int NWN = GLU ? NW / 2 : NW;  // waves side by side on the neurons of the output
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int lane = tid & 63, r = lane & 15, kb = lane >> 4;
    const int rb_out = (tn * NWN + wave % NWN) * NB;  // first row-block of the wave in the output
    const int rbs = out.rbs;
    const int nrb = min(NB, rbs - rb_out);
    const bool up = GLU && wave >= NWN;
    const int rb0 = out.rb_first + rb_out + (up ? rbs : 0), rb_end = out.rb_first + (up ? 2 * rbs : rbs);
    B w;
    w.init(k, wt, rb0, rb_end, lane);
    const int row = rows.request();
    w.prologue(s_begin);
    const float row_scale = rows.tables(row);
    float4_t acc[MT][NB];
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};

    const float *anchors = reinterpret_cast<const float *>(wt + k.anchors_off);
    auto row_of = [&](int b) { return min(rb0 + b, rb_end - 1) * 16 + 4 * kb; };
    float4_t min_factor[NB], ns[NB], nm[NB];
    auto load_anchors = [&]() {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            ns[b] = *reinterpret_cast<const float4_t *>(anchors + row_of(b));
            nm[b] = *reinterpret_cast<const float4_t *>(anchors + 16 * k.n_rowblocks + row_of(b));
        }
    };
    auto load_min_factor = [&]() {
        load_anchors();
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) min_factor[b][v] = -nm[b][v] / (64.f * (ns[b][v] == 0.f ? 0x1p-80f : ns[b][v]));
    };
    if constexpr (B::CENTER != 0) load_min_factor();

    const uint32_t lane_off = rows.lane_off(lane);
    typename Rows::template Copy<MT, B::SL, NW> cp;
    rows.init(cp, rows.xf, k.nsteps * B::STEP, lane, wave);
    if constexpr (FUSED) {
        uint32_t off[MT];
#pragma unroll
        for (int a = 0; a < MT; ++a) off[a] = static_cast<uint32_t>(rows.srcv[16 * a + r]) * static_cast<uint32_t>(k.nsteps) * 64u + kb * 16u;
        w.init_min(wave_window(reinterpret_cast<const uint8_t *>(rows.xg), static_cast<uint32_t>(rows.n_rows) * static_cast<uint32_t>(k.nsteps) * 64u), off,
                   s_begin);
    } else {
        // Minimum term: group sums of SC steps (a stage) at a time through the two stages of the ring that the first products need
        // last, the next stage on its way while one is multiplied.  The products' own first stages are requested before all of that,
        // the last of them in place of a next stage, so that only one wait for memory stands at the head of a tile (it was one per
        // four steps and one more: NINT4-32 12288 x 4096 on blocks of eight waves at 1024 and 2048 rows 113.4 and 190.4 us, then 109.6 and
        // 185.9).
        constexpr int SC = B::SL, SLOT = MT * SC * 1024;
        typename Rows::template Copy<MT, SC, NW> cg;
        rows.init(cg, rows.xg, k.nsteps, lane, wave);
        const int n = (s_end - s_begin + SC - 1) / SC;
        u32x2_t sc[SC][NB], next[SC][NB];
        auto slot = [&](int i) { return lds + (R - 1 - ((n - 1 - i) & 1)) * SLOT; };  // stage n - 1 in the ring's last
        auto load_sub = [&](int i, u32x2_t (&dst)[SC][NB]) {
#pragma unroll
            for (int t = 0; t < SC; ++t) {
                const int so = __builtin_amdgcn_readfirstlane(min(s_begin + i * SC + t, w.s_last) * w.sb);
#pragma unroll
                for (int b = 0; b < NB; ++b) dst[t][b] = __builtin_amdgcn_raw_buffer_load_b64(w.win, w.qoff[b] + w.soff_lane, so, 0);
            }
        };
        load_sub(0, sc);
        cg.issue(slot(0), s_begin);
        if (n > 1) {
            load_sub(1, next);
            cg.issue(slot(1), s_begin + SC);
        } else {
            cp.issue(lds + (R - 2) * SLOT, s_begin * B::STEP + (R - 2) * B::SL);
        }
#pragma unroll
        for (int i = 0; i < R - 2; ++i) cp.issue(lds + i * SLOT, s_begin * B::STEP + i * B::SL);
        for (int i = 0; i < n; ++i) {
            const int c0 = s_begin + i * SC;
            const uint8_t *sums = slot(i);
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
            __syncthreads();
            if (i > 0) {
#pragma unroll
                for (int t = 0; t < SC; ++t)
#pragma unroll
                    for (int b = 0; b < NB; ++b) sc[t][b] = next[t][b];
                if (i + 1 < n) {
                    load_sub(i + 1, next);
                    cg.issue(slot(i + 1), c0 + SC);
                } else {
                    cp.issue(lds + (R - 2) * SLOT, s_begin * B::STEP + (R - 2) * B::SL);
                }
            }
            if constexpr (B::CENTER != 0) {
                // Fragments of one value per group, groups j = 0 .. 3 twice: a byte dropped into the mantissa of 1024 and packed
                // fp16 arithmetic (16 s is exact, and so is what it leaves of the rounded BIAS s).
                const _Float16 k1 = static_cast<_Float16>(1024.f), k16 = static_cast<_Float16>(16.f), kb16 = static_cast<_Float16>(1.f * B::BIAS),
                               k1k = static_cast<_Float16>(16384.f), kbk = static_cast<_Float16>(1024.f * B::BIAS);
                auto sub_min = [&](uint32_t v) {
                    const half2_t X = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(v, kMagicH2, 0x03070105u));
                    return __builtin_bit_cast(uint32_t, X - half2_t{k1, k1});
                };
                auto off_centre = [&](uint32_t v) {
                    const half2_t X = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(v, kMagicH2, 0x03060104u));
                    const half2_t c = __builtin_elementwise_fma(X, half2_t{kb16, kb16}, half2_t{-kbk, -kbk});
                    return __builtin_bit_cast(uint32_t, c - __builtin_elementwise_fma(X, half2_t{k16, k16}, half2_t{-k1k, -k1k}));
                };
                float4_t s2[MT][NB];
#pragma unroll
                for (int a = 0; a < MT; ++a)
#pragma unroll
                    for (int b = 0; b < NB; ++b) s2[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int t = 0; t < SC; ++t) {
                    if (c0 + t < s_end) {
                        u32x4_t bm[NB], bc[NB];
#pragma unroll
                        for (int b = 0; b < NB; ++b) {
                            const uint32_t m01 = sub_min(sc[t][b].x), m23 = sub_min(sc[t][b].y);
                            const uint32_t c01 = off_centre(sc[t][b].x), c23 = off_centre(sc[t][b].y);
                            bm[b] = u32x4_t{m01, m23, m01, m23};
                            bc[b] = u32x4_t{c01, c23, c01, c23};
                        }
#pragma unroll
                        for (int a = 0; a < MT; ++a) {
                            const u32x4_t ax = *reinterpret_cast<const u32x4_t *>(sums + (a * SC + t) * 1024 + lane_off);
#pragma unroll
                            for (int b = 0; b < NB; ++b) {
                                s2[a][b] = mfma16(bm[b], ax, s2[a][b]);
                                acc[a][b] = mfma16(bc[b], ax, acc[a][b]);
                            }
                        }
                    }
                }
#pragma unroll
                for (int a = 0; a < MT; ++a)
#pragma unroll
                    for (int b = 0; b < NB; ++b)
#pragma unroll
                        for (int v = 0; v < 4; ++v) acc[a][b][v] = fmaf(min_factor[b][v], s2[a][b][v], acc[a][b][v]);
            } else {
#pragma unroll
                for (int t = 0; t < SC; ++t) {
                    if (c0 + t < s_end) {
                        u32x4_t bm[NB];
#pragma unroll
                        for (int b = 0; b < NB; ++b) bm[b] = B::min_fragment(sc[t][b].x, sc[t][b].y);
#pragma unroll
                        for (int a = 0; a < MT; ++a) {
                            const u32x4_t ax = *reinterpret_cast<const u32x4_t *>(sums + (a * SC + t) * 1024 + lane_off);
#pragma unroll
                            for (int b = 0; b < NB; ++b) acc[a][b] = mfma16(bm[b], ax, acc[a][b]);
                        }
                    }
                }
            }
        }
    }
    if constexpr (B::CENTER == 0 && !FUSED) {
        load_min_factor();
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int a = 0; a < MT; ++a)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[a][b][v] *= min_factor[b][v];
    }

    rows.scales(row_scale);
    tile_loop<B, MT, R, !FUSED, Rows::PAIRED>(w, cp, lds, s_begin, s_end, lane_off, acc);
    if constexpr (B::SHORT) {
        int late = threadIdx.x;
        asm volatile("" : "+v"(late));
        lane = late & 63;
        r = lane & 15;
        kb = lane >> 4;
    }

    float xs[MT];
#pragma unroll
    for (int a = 0; a < MT; ++a) xs[a] = rows.scale(a, r);
    load_anchors();
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if constexpr (FUSED) {
#pragma unroll
            for (int a = 0; a < MT; ++a)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[a][b][v] = xs[a] * (64.f * ns[b][v] * acc[a][b][v] - nm[b][v] * w.s2[a][b][v]);
        } else {
            float4_t f;
#pragma unroll
            for (int v = 0; v < 4; ++v) f[v] = 64.f * (ns[b][v] != 0.f ? ns[b][v] : nm[b][v] != 0.f ? 0x1p-80f : 0.f);
#pragma unroll
            for (int a = 0; a < MT; ++a)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[a][b][v] = xs[a] * (f[v] * acc[a][b][v]);
        }
    }
    const bool wide = (out.ldy & 3) == 0 && (reinterpret_cast<uintptr_t>(out.y) & 15) == 0;
    const bool wide16 = (out.ldy & 7) == 0 && (reinterpret_cast<uintptr_t>(out.y) & 15) == 0;
    if constexpr (GLU) {
        // Both halves of the waves compute: gate waves the row tiles below A0 and up waves the others, after handing each other
        // their sums of the rest.
        constexpr int A0 = (MT + 1) / 2;
        uint8_t *ex = lds + (wave % NWN) * (MT * NB * 1024) + lane * 16;
#pragma unroll
        for (int a = 0; a < MT; ++a)
#pragma unroll
            for (int b = 0; b < NB; ++b)
                if (up == (a < A0)) *reinterpret_cast<float4_t *>(ex + (a * NB + b) * 1024) = acc[a][b];
        __syncthreads();
        auto store = [&](auto F16, auto A, auto UP) {
            constexpr int a = A.value;
            u32x2_t o[NB];
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const float4_t o4 = *reinterpret_cast<const float4_t *>(ex + (a * NB + b) * 1024);
                uint32_t h[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float hv = UP.value ? glu_value(o4[v], acc[a][b][v], out.gelu != 0) : glu_value(acc[a][b][v], o4[v], out.gelu != 0);
                    h[v] = F16.value ? f32_to_f16_rne(hv) : f32_to_bf16_rne(hv);
                }
                o[b] = u32x2_t{h[0] | (h[1] << 16), h[2] | (h[3] << 16)};
            }
            // by way of what the wave has just read there: its own exchange of this row tile
            wave_sync();
            store_rows16(lds + ((wave % NWN) * MT + a) * (NB * 1024), o, lane, rb_out * 16, rb_out * 16 + nrb * 16, static_cast<uint16_t *>(out.y), out.ldy, wide16,
                         [&](int row) { return rows.dst(a, row); });
        };
        auto store_half = [&](auto F16) {
            if (up) static_for<MT - A0>([&](auto I) { store(F16, std::integral_constant<int, A0 + I.value>{}, std::true_type{}); });
            else static_for<A0>([&](auto I) { store(F16, I, std::false_type{}); });
        };
        if (out.f16) store_half(std::true_type{});
        else store_half(std::false_type{});
    } else {
        float *y = static_cast<float *>(out.y);
#pragma unroll
        for (int a = 0; a < MT; ++a)
            store_rows(lds + wave * kRowsOut, acc[a], lane, rb_out * 16, min(out.cols, (rb_out + nrb) * 16), y, out.ldy, wide,
                       [&](int row) { return rows.dst(a, row); });
    }
}

template <class U, int NW, int MT, int NB, int R, bool GLU>
__global__ __launch_bounds__(64 * NW, 2) void nint_tile_kernel(NintTileArgs p, int tiles_n, int tiles_m) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t tile_lds[];
    int tn, tm;
    if (!tile_of_block(tiles_n, tiles_m, tn, tm)) return;
    const int z = blockIdx.y, s_begin = z * p.spz, s_end = min(p.k.nsteps, s_begin + p.spz);
    const FragRows rows{p.xf, p.xg, p.xscale, tm * MT, (p.M + 15) >> 4, p.M};
    const TileOut out{0, GLU ? p.rb_half : p.k.n_rowblocks, p.k.out, GLU ? p.y : static_cast<float *>(p.y) + z * p.zstride, p.ldy, p.gelu, p.f16};
    nint_tile_body<NintTileB<U, NB, 0, NB == 4 ? 2 : 0, 0, NB == 4>, NW, MT, R, GLU>(p.k, p.w, rows, out, tn, s_begin, s_end, tile_lds);
}

// row-blocks of a wave that the registers hold (four of three bits spill at the head of a tile: 383 us for 172)
constexpr int nint_tile_widest(int bits, int dwords) { return dwords > 5 ? 2 : dwords > 4 || bits == 3 ? 3 : 4; }
template <class U, int SHAPE, bool GLU>
static int nint_tile_start(const NintTileArgs &a, int splits, hipStream_t st) {
    constexpr int MT = kTileShape[SHAPE].mt, NB = kTileShape[SHAPE].nb, NW = kTileShape[SHAPE].nw;
    if constexpr (NB > nint_tile_widest(U::CODE_BITS, U::D)) {
        return fail(MFQ_ERR_UNSUPPORTED, "nint_tile: no registers for %d units of %d dwords", NB, U::D);
    } else {
        constexpr int SL = NintTileB<U, NB>::SL, R = SL == 3 && NW == 4 ? 3 : 4;
        // the ring; with GLU the up results
        constexpr size_t blocks = MT * R * SL, up = GLU ? MT * NB * (NW / 2) : 0;
        constexpr size_t lds = 1024 * (blocks > up ? blocks : up);
        const int rbs = GLU ? a.rb_half : a.k.n_rowblocks;
        const int tn = static_cast<int>(ceil_div(rbs, (GLU ? NW / 2 : NW) * NB)), tm = static_cast<int>(ceil_div(a.M, 16 * MT));
        auto kern = nint_tile_kernel<U, NW, MT, NB, R, GLU>;
        if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), lds, "nint_tile")) return rc;
        hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(ceil_div(static_cast<int64_t>(tn) * tm, 8) * 8), static_cast<unsigned>(splits)),
                           dim3(64 * NW), lds, st, a, tn, tm);
        return check_launch("nint_tile");
    }
}

template <class U>
static int nint_tile_launch(const NintTileArgs &a, int shape, bool glu, int splits, hipStream_t st) {
    switch (shape) {
#define MFQ_TILE_SHAPE_CASE(S) case S: return glu ? nint_tile_start<U, S, true>(a, splits, st) : nint_tile_start<U, S, false>(a, splits, st);
        MFQ_TILE_SHAPE_CASE(0) MFQ_TILE_SHAPE_CASE(1) MFQ_TILE_SHAPE_CASE(2) MFQ_TILE_SHAPE_CASE(3) MFQ_TILE_SHAPE_CASE(4) MFQ_TILE_SHAPE_CASE(5)
#undef MFQ_TILE_SHAPE_CASE
    }
    return fail(MFQ_ERR_UNSUPPORTED, "nint_tile: shape %d", shape);
}

}  // namespace mfq
