// Row-major weights as policies of the tile kernel (tile_gemm.hpp): the payload's own bytes (OCP MX, Q8_0 codes), or fp16
// fragments that another kernel has left in a workspace.  Nothing is repacked in memory: which k sits in which of an instruction's 32
// slots is free as long as the activations (x_frag) agree.
//
// Measured, whole calls with bf16 activations (the fp16 copy and 128 x 128 GEMM they replace): MXFP4 12288 x 4096 at 64 / 601 / 2048 rows
// 23 / 62 / 184 us (43 / 223 / 446), NINT8-0 there at 64 / 2048 rows 31 / 222 us (103 / 446), 4096 x 12288 fp16 at 333 rows 66 us (226).
#pragma once
#include "tile_gemm.hpp"

namespace mfq {

struct RowTileArgs {
    const uint8_t *w, *scales;   // values and scales of the whole tensor (fp16: its fragments)
    int64_t row_bytes;           // of a neuron's values
    int row0, N, K, M;           // neurons [row0, row0 + N) against M activation rows
    const uint16_t *xf;          // fragment-ordered activations (x_frag, groups of RowUnit::GS values)
    const float *xscale, *wscale;  // per activation row; per neuron of the call (null: 1)
    float *y;
    int64_t ldy, zstride;        // zstride: floats between the partial results of two splits over K
    int slices, nsteps, spz;     // slices of a row-block of xf; steps of K, and of a split
};

// A unit is 64 bytes of a neuron: a lane multiplies GS values of it, NM = GS / 8 fragments.
template <int KIND> struct RowUnit { static constexpr int GS = KIND == kRowMx4 || KIND == kRowMx4F16 ? 32 : KIND == kRowF16 ? 8 : 16; };

// fp16 fragments (a KB per 16 neurons and 32 k, frag16_at): loaded three slices ahead into the registers the matrix cores read
// them from.  Row-blocks past the end repeat the last one.
template <int NB>
struct RowTileF16 {
    static constexpr int NBLK = NB, STEP = 8, SL = 2, NBUF = 4, LDS_WAVE = 0;
    static constexpr bool PAIRED = false;
    __amdgpu_buffer_rsrc_t win;
    uint32_t off[NB];
    int slices;
    u32x4_t bf[NBUF][NB];
    static constexpr int loads(int) { return NB; }
    static constexpr int loads_before(int, int n) { return n * NB; }
    __device__ static __forceinline__ float4_t mfma(u32x4_t b, u32x4_t a, float4_t c) { return mfma16(b, a, c); }
    __device__ __forceinline__ void init(const RowTileArgs &p, int rb0, int lane) {
        slices = static_cast<int>(p.row_bytes >> 6);
        const int rbs = (p.N + 15) >> 4, first = min(rb0, rbs - 1), n = min(NB, rbs - first);
        win = wave_window(p.w + static_cast<int64_t>(first) * slices * 1024, static_cast<uint32_t>(n * slices) * 1024u);
#pragma unroll
        for (int b = 0; b < NB; ++b) off[b] = static_cast<uint32_t>(min(b, n - 1) * slices) * 1024u + lane * 16u;
    }
    __device__ __forceinline__ void load(int t, u32x4_t (&dst)[NB]) {
#pragma unroll
        for (int b = 0; b < NB; ++b)
            dst[b] = __builtin_amdgcn_raw_buffer_load_b128(win, t < slices ? off[b] : kNoStep, __builtin_amdgcn_readfirstlane(t * 1024), 0);
    }
    __device__ __forceinline__ void prologue(int s) {
#pragma unroll
        for (int i = 0; i < NBUF - 1; ++i) load(s * STEP + i, bf[i]);
    }
    __device__ __forceinline__ void first(int) {}
    template <int I>
    __device__ __forceinline__ void issue(int s) { load(s * STEP + I + NBUF - 1, bf[(I + NBUF - 1) % NBUF]); }
    template <int I, int PART, int PARTS>
    __device__ __forceinline__ void produce(int) {}
    template <int MT>
    __device__ static __forceinline__ void schedule() { __builtin_amdgcn_sched_barrier(0); }
};

// Packed rows: units decoded one slice ahead of the matrix cores.
//
// A request whose neighbouring lanes lie in different rows occupies a compute unit's address path four times as long as one where four
// lanes share 64 bytes, and with one such request per lane's 16 bytes that path set the pace.  So a request takes 64 contiguous bytes
// of each of 16 neurons (four lanes a neuron, "row order" as in GatherCopy), waits RS units ahead in registers, and passes through a
// KB of LDS of the wave's own on its way to the lane (r, kb) that multiplies it; the scales of a step go the same way, two per lane.
// LDS operations of a wave happen in order, so the pieces need no waits between them, only the compiler kept from moving them.
// Whole calls, before (every lane asked for 16 bytes of its own row) and after: NINT8-0 4096 x 12288 fp16 at 333 rows 81.4 and 69.1
// us, MXFP4 12288 x 4096 bf16 at 601 rows 65.4 and 61.4.
//   Q8      fp16 scale per 32 values.  Code byte -> mantissa of 8 (9 + code / 128 exactly), minus 9, times the scale taken
//           relative to the row's power of two (wscale), which puts the row's largest into [2^14, 2^15): one rounding per
//           weight, and no scale loses bits before it is 2^-29 of the largest (with whole codes it would at 2^-23).
//   MX      the hardware's conversion multiplies by the power of two in the exponent field of its scale operand: an E8M0 byte
//           shifted into place.  bf16 activations: exact, unscaled (bf16 has the exponents of E8M0).  fp16 activations: the
//           scale relative to the row's largest (wscale), exact unless the element is 2^-24 and more below it.
template <int KIND, int NB>
struct RowTilePacked {
    typedef RowUnit<KIND> U;
    static constexpr bool MX4 = KIND == kRowMx4 || KIND == kRowMx4F16, MX8 = KIND == kRowMx8 || KIND == kRowMx8F16;
    static constexpr bool BF16 = KIND == kRowMx4 || KIND == kRowMx8, PAIRED = KIND == kRowQ8;
    // units per step, in registers as the lane multiplies them, and in flight
    static constexpr int NM = U::GS / 8, UPS = 8 / NM, NSET = 2, RS = MX8 && NB == 3 ? 2 : UPS;  // (no registers for more)
    static constexpr int NBLK = NB, STEP = 8, SL = 2, NBUF = 2;
    static constexpr int SCALE_BYTES = MX8 ? 0 : KIND == kRowQ8 ? 256 : 128;  // of the eight groups of a step, 16 rows
    static constexpr int SCALE_AT = NM * (UPS - NSET);  // slice from which the units to come are those of the next step
    static constexpr int LDS_WAVE = NB * (1024 + SCALE_BYTES);
    __amdgpu_buffer_rsrc_t win, swin;
    uint32_t off[NB], soff[NB], rel[NB];  // rel: bits of the row's 2^(7 - p) (Q8) or its largest E8M0 byte (MX against fp16)
    uint8_t *area;
    uint32_t to, at, sto, sat;   // where the lane leaves a request's 16 bytes and finds those of its unit; the same for scales
    int ulim, slim;              // a lane's 16 bytes of unit u lie inside the row if 4 u < ulim, its scales of step (MX8: unit) u by slim
    u32x4_t raw[RS][NB];
    uint32_t rsc[2][NB];
    uint32_t q[NSET][NB][4], sc[NSET][NB];
    float scale[NB];
    half2_t scale2[NB];
    u32x4_t bf[NBUF][NB];

    static constexpr int loads(int i) {
        return (i % NM == NM - 1 ? NB * (MX8 ? 2 : 1) : 0) + (!MX8 && i == SCALE_AT ? 2 * NB : 0);
    }
    static constexpr int loads_before(int i, int n) {
        int t = 0;
        for (int d = 1; d <= n; ++d) t += loads(((i - d) % STEP + STEP) % STEP);
        return t;
    }
    __device__ static __forceinline__ float4_t mfma(u32x4_t b, u32x4_t a, float4_t c) {
        if constexpr (BF16)
            return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b), __builtin_bit_cast(bf16x8_t, a), c, 0, 0, 0);
        else
            return mfma16(b, a, c);
    }
    // Row-blocks rb0 + b of the call; rows past the end repeat the last one (nobody stores their sums).  A lane whose columns do not
    // exist asks outside the window and gets zeros.
    __device__ __forceinline__ void init(const RowTileArgs &p, int rb0, int lane, uint8_t *lds) {
        const int kb = lane >> 4, quarter = row_order_quarter(lane >> 2, lane & 3);
        area = lds;
        to = lane * 16;
        at = row_order_lane(lane);
        sto = NB * 1024 + lane * (KIND == kRowQ8 ? 4 : 2);
        sat = NB * 1024 + (KIND == kRowQ8 ? (lane & 15) * 16 + (kb >> 1) * 2 : (lane & 15) * 8 + kb);
        ulim = p.K / U::GS - quarter;
        slim = MX8 ? p.K / U::GS - kb : p.K / 32 - 2 * (lane & 3);
        const int first = min(rb0 * 16, p.N - 1), n = min(NB * 16, p.N - first), r0 = p.row0 + first;
        win = wave_window(p.w + static_cast<int64_t>(r0) * p.row_bytes, static_cast<uint32_t>(n * p.row_bytes));
        // a neuron's scales: K / 32 of SB bytes, or those of its 128-row band
        constexpr int SB = KIND == kRowQ8 ? 2 : 1;
        const int64_t per_row = MX8 ? p.K / 128 : static_cast<int64_t>(p.K / 32) * SB;
        const int base = MX8 ? r0 / 128 : r0, count = MX8 ? (r0 + n - 1) / 128 - base + 1 : n;
        swin = wave_window(p.scales + base * per_row, static_cast<uint32_t>(count * per_row));
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int row = min(16 * b + (lane & 15), n - 1), mine = min(16 * b + (lane >> 2), n - 1);
            off[b] = static_cast<uint32_t>(mine) * static_cast<uint32_t>(p.row_bytes) + quarter * 16;
            if constexpr (MX8) soff[b] = static_cast<uint32_t>((r0 + row) / 128 - base) * static_cast<uint32_t>(per_row);
            else soff[b] = static_cast<uint32_t>(mine) * static_cast<uint32_t>(per_row) + (lane & 3) * 2 * SB;
            rel[b] = 0;
            if constexpr (!BF16) {
                const uint32_t bits = __float_as_uint(p.wscale[first + row]);
                rel[b] = KIND == kRowQ8 ? (261u << 23) - bits : bits >> 23;  // Q8: 2^7 / wscale
            }
        }
    }
    __device__ __forceinline__ void load_unit(int u, u32x4_t (&dst)[NB]) {
        const bool in = 4 * u < ulim;
        const int so = __builtin_amdgcn_readfirstlane(u * 64);
#pragma unroll
        for (int b = 0; b < NB; ++b) dst[b] = __builtin_amdgcn_raw_buffer_load_b128(win, in ? off[b] : kNoStep, so, 0);
    }
    // Groups 2 (lane % 4) and the next one of step u's eight, in two requests because an odd number of groups puts every other row
    // off any wider boundary.
    __device__ __forceinline__ void load_scales(int u) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool in = 8 * u + h < slim;
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                if constexpr (KIND == kRowQ8)
                    rsc[h][b] = __builtin_amdgcn_raw_buffer_load_b16(swin, in ? soff[b] + 2 * h : kNoStep, __builtin_amdgcn_readfirstlane(u * 16), 0);
                else
                    rsc[h][b] = __builtin_amdgcn_raw_buffer_load_b8(swin, in ? soff[b] + h : kNoStep, __builtin_amdgcn_readfirstlane(u * 8), 0);
            }
        }
    }
    // MX8: the scale of unit u's band, one byte for most or all of the lanes
    __device__ __forceinline__ void load_band(int u, uint32_t (&dst)[NB]) {
        const bool in = 4 * u < slim;
        const int so = __builtin_amdgcn_readfirstlane(u >> 1);
#pragma unroll
        for (int b = 0; b < NB; ++b) dst[b] = __builtin_amdgcn_raw_buffer_load_b8(swin, in ? soff[b] : kNoStep, so, 0);
    }
    // the scales of the next step become those in LDS; SCALE_AT is behind the last read of the current ones
    __device__ __forceinline__ void turn_scales(int next) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            uint8_t *dst = area + sto + b * SCALE_BYTES;
            if constexpr (KIND == kRowQ8) *reinterpret_cast<uint32_t *>(dst) = rsc[0][b] | (rsc[1][b] << 16);
            else *reinterpret_cast<uint16_t *>(dst) = static_cast<uint16_t>(rsc[0][b] | (rsc[1][b] << 8));
        }
        wave_sync();
        load_scales(next);
    }
    // unit u, number J of its step: from the order of the request (set IN) into that of the matrix cores; the unit RS on is requested
    template <int J, int IN>
    __device__ __forceinline__ void turn(int u) {
        constexpr int OUT = J % NSET;
        if constexpr (MX8) load_band(u, sc[OUT]);
#pragma unroll
        for (int b = 0; b < NB; ++b) *reinterpret_cast<u32x4_t *>(area + to + b * 1024) = raw[IN][b];
        wave_sync();
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const u32x4_t v = *reinterpret_cast<const u32x4_t *>(area + at + b * 1024);
            q[OUT][b][0] = v.x; q[OUT][b][1] = v.y; q[OUT][b][2] = v.z; q[OUT][b][3] = v.w;
            if constexpr (KIND == kRowQ8) sc[OUT][b] = *reinterpret_cast<const uint16_t *>(area + sat + b * SCALE_BYTES + 4 * J);
            else if constexpr (MX4) sc[OUT][b] = area[sat + b * SCALE_BYTES + 4 * J];
        }
        wave_sync();
        load_unit(u + RS, raw[IN]);
    }
    __device__ __forceinline__ void prologue(int s) {
        if constexpr (!MX8) load_scales(s);
#pragma unroll
        for (int u = 0; u < RS; ++u) load_unit(UPS * s + u, raw[u]);
    }
    __device__ __forceinline__ void unit_scale(int b, uint32_t raw) {
        if constexpr (KIND == kRowQ8) {
            const float v = f16_to_f32(static_cast<uint16_t>(raw)) * __uint_as_float(rel[b]);
            const _Float16 h = static_cast<_Float16>(v);
            scale2[b] = half2_t{h, h};
        } else if constexpr (BF16) {
            scale[b] = __uint_as_float(raw << 23);
        } else {
            // 2^(raw - largest): exact down to 2^-126, zero below; a NaN scale stays one
            const int e = static_cast<int>(raw) - static_cast<int>(rel[b]) + 127;
            scale[b] = __uint_as_float(raw == 255u ? 0x7f800000u : e > 0 ? static_cast<uint32_t>(e) << 23 : 0u);
        }
    }
    // dwords [P0, P1) (four per row-block) of the fragments of slice (j, MM) of unit set SET
    template <int P0, int P1, int MM, int SET>
    __device__ __forceinline__ void decode(u32x4_t (&dst)[NB]) {
        static_for<P1 - P0>([&](auto P) {
            constexpr int p = P0 + P.value, b = p / 4, t = p % 4;
            // visible to the compiler here and not earlier: hoisted to the unit's arrival the conversions would keep a whole
            // unit of pairs in registers
            if constexpr (MX4) {
                if constexpr (t == 0) asm volatile("" : "+v"(q[SET][b][MM]));
            } else {
                if constexpr (t % 2 == 0) asm volatile("" : "+v"(q[SET][b][2 * MM + t / 2]));
            }
            if constexpr (MM == 0 && t == 0) {
                asm volatile("" : "+v"(sc[SET][b]));
                unit_scale(b, sc[SET][b]);
            }
            uint32_t v;
            if constexpr (MX4) {
                if constexpr (BF16) v = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(q[SET][b][MM], scale[b], t));
                else v = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(q[SET][b][MM], scale[b], t));
            } else if constexpr (MX8) {
                const uint32_t d = q[SET][b][2 * MM + t / 2];
                if constexpr (BF16) v = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(d, scale[b], t % 2 == 1));
                else v = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(d, scale[b], t % 2 == 1));
            } else {
                const uint32_t d = q[SET][b][2 * MM + t / 2] ^ 0x80808080u;
                const half2_t c = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(d, 0x48004800u, t % 2 ? 0x03070106u : 0x03050104u));
                const _Float16 off = static_cast<_Float16>(-9.f);
                v = __builtin_bit_cast(uint32_t, (c + half2_t{off, off}) * scale2[b]);
            }
            dst[b][t] = v;
        });
    }
    __device__ __forceinline__ void first(int s) {
        if constexpr (!MX8) turn_scales(s + 1);
        static_for<NSET>([&](auto J) { turn<J.value, J.value>(UPS * s + J.value); });
        decode<0, 4 * NB, 0, 0>(bf[0]);
    }
    template <int I>
    __device__ __forceinline__ void issue(int s) {
        constexpr int j = I / NM, n = j + NSET;
        if constexpr (!MX8 && I == SCALE_AT) turn_scales(s + 2);
        if constexpr (I % NM == NM - 1) turn<n % UPS, n % RS>(UPS * s + n);
    }
    template <int I, int PART, int PARTS>
    __device__ __forceinline__ void produce(int) {
        constexpr int n = (I + 1) % STEP;
        decode<PART * 4 * NB / PARTS, (PART + 1) * 4 * NB / PARTS, n % NM, n / NM % NSET>(bf[(I + 1) & 1]);
    }
    template <int MT>
    __device__ static __forceinline__ void schedule() { __builtin_amdgcn_sched_barrier(0); }
};

template <int KIND, int NB> struct RowPolicy { typedef RowTilePacked<KIND, NB> type; };
template <int NB> struct RowPolicy<kRowF16, NB> { typedef RowTileF16<NB> type; };

// y[m, n] = xscale[m] * wscale[n] * sum; blocks are dealt to the XCDs as in nint_tile_kernel.
template <int KIND, int NW, int MT, int NB, int R>
__global__ __launch_bounds__(64 * NW, 2) void row_tile_kernel(RowTileArgs p, int tiles_n, int tiles_m) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t tile_lds[];
    typedef typename RowPolicy<KIND, NB>::type B;
    int tn, tm;
    if (!tile_of_block(tiles_n, tiles_m, tn, tm)) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, kb = lane >> 4;
    const int mb0 = tm * MT, mb_total = (p.M + 15) >> 4, rb0 = (tn * NW + wave) * NB;
    const int z = blockIdx.y, s_begin = z * p.spz, s_end = min(p.nsteps, s_begin + p.spz);
    B w;
    if constexpr (KIND == kRowF16) w.init(p, rb0, lane);
    else w.init(p, rb0, lane, tile_lds + 1024 * MT * R * B::SL + wave * B::LDS_WAVE);
    w.prologue(s_begin);
    float4_t acc[MT][NB];
#pragma unroll
    for (int a = 0; a < MT; ++a)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = float4_t{0.f, 0.f, 0.f, 0.f};
    TileCopy<MT, B::SL, NW> cp;
    cp.init(p.xf, p.slices, mb0, mb_total, lane, wave);
    tile_loop<B, MT, R, false, B::PAIRED>(w, cp, tile_lds, s_begin, s_end, static_cast<uint32_t>(lane) * 16u, acc);

    float xs[MT];
#pragma unroll
    for (int a = 0; a < MT; ++a) xs[a] = p.xscale[min(mb0 + a, mb_total - 1) * 16 + r];
    float4_t ws[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        ws[b] = float4_t{1.f, 1.f, 1.f, 1.f};
        if (p.wscale)
#pragma unroll
            for (int v = 0; v < 4; ++v) ws[b][v] = p.wscale[min((rb0 + b) * 16 + 4 * kb + v, p.N - 1)];
    }
    float *y = p.y + static_cast<int64_t>(z) * p.zstride;
    const bool wide = (p.ldy & 3) == 0 && (reinterpret_cast<uintptr_t>(p.y) & 15) == 0;
#pragma unroll
    for (int a = 0; a < MT; ++a) {
        float4_t o[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int v = 0; v < 4; ++v) o[b][v] = acc[a][b][v] * ws[b][v] * xs[a];
        store_rows(tile_lds + wave * kRowsOut, o, lane, rb0 * 16, min(p.N, (rb0 + NB) * 16), y, p.ldy, wide, [&](int row) {
            const int m = (mb0 + a) * 16 + row;
            return m < p.M ? m : -1;
        });
    }
}

constexpr int row_tile_widest(int kind) { return kind == kRowQ8 ? 2 : kind == kRowF16 ? 4 : 3; }
template <int KIND, int SHAPE>
static int row_tile_start(const RowTileArgs &a, int splits, hipStream_t st) {
    constexpr int MT = kTileShape[SHAPE].mt, NB = kTileShape[SHAPE].nb, NW = kTileShape[SHAPE].nw;
    if constexpr (NB > row_tile_widest(KIND)) {
        return fail(MFQ_ERR_UNSUPPORTED, "row_tile: no registers for %d row-blocks of kind %d", NB, KIND);
    } else {
        typedef typename RowPolicy<KIND, NB>::type B;
        constexpr int R = 4;
        constexpr size_t lds = static_cast<size_t>(1024) * MT * R * B::SL + NW * B::LDS_WAVE;
        const int tn = static_cast<int>(ceil_div(a.N, 16 * NW * NB)), tm = static_cast<int>(ceil_div(a.M, 16 * MT));
        auto kern = row_tile_kernel<KIND, NW, MT, NB, R>;
        if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), lds, "row_tile")) return rc;
        hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(ceil_div(static_cast<int64_t>(tn) * tm, 8) * 8), static_cast<unsigned>(splits)),
                           dim3(64 * NW), lds, st, a, tn, tm);
        return check_launch("row_tile");
    }
}

template <int KIND>
static int row_tile_launch(const RowTileArgs &a, int shape, int splits, hipStream_t st) {
    switch (shape) {
        case 0: return row_tile_start<KIND, 0>(a, splits, st);
        case 1: return row_tile_start<KIND, 1>(a, splits, st);
        case 2: return row_tile_start<KIND, 2>(a, splits, st);
        case 3: return row_tile_start<KIND, 3>(a, splits, st);
        case 4: return row_tile_start<KIND, 4>(a, splits, st);
        case 5: return row_tile_start<KIND, 5>(a, splits, st);
    }
    return fail(MFQ_ERR_UNSUPPORTED, "row_tile: shape %d", shape);
}

}  // namespace mfq
