// Block-tiled matrix-core matmul of prefill batches: y[m, n] = sum_k x[m, k] * w[n, k], fp32 accumulation.
//
// Both operands are kept in "fragment order": the 16 rows x 32 k-values one v_mfma_f32_16x16x32 consumes are 1 KB that
// a wave reads as 16 bytes per lane, lane (r, kb) = row r, eight k-values of quarter kb (a "slice" of the 16 rows).  The
// activations come that way from x_frag_kernel; a weight policy leaves the weight fragments of a wave's row-blocks in
// registers, by decoding packed units or by loading 16-bit fragments.
//
// Block = four or eight waves side by side on the neurons; a wave owns MT * 16 tokens x NB * 16 neurons.  The activation slices
// of the block's tokens go from global memory straight into a ring of stages in LDS, with no padding and no swizzle:
// every copy and every read is one contiguous KB (no bank conflicts counted).  NINT units and fp16 fragments go from memory straight
// into registers; row-major weights and their scales pass through LDS_WAVE bytes of the wave's own behind the ring (row_tile.hpp).  Per
// slice a wave reads MT fragments from LDS for MT * NB matrix-core instructions, one for two to four of them (kTileShape).  Results
// leave through the ring's LDS (store_rows).
// The loop is software-pipelined inside the wave: the activation fragments of the next few instructions are read, and
// the weight fragments of the next slice made, between the matrix-core instructions of the current one.
#pragma once
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "gemv_common.hpp"
#include "nint_mfma.hpp"
#include "tune.hpp"

namespace mfq {

typedef __attribute__((address_space(3))) void *lds_void_t;
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

template <class F, int... I>
__device__ __forceinline__ void static_for_seq(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_seq(static_cast<F &&>(f), std::make_integer_sequence<int, N>{});
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N < 64, "vmcnt holds six bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Copies of one wave for a stage (SL slices) of the block's MBS 16-row blocks of activations.
template <int MBS, int SL, int NW>
struct TileCopy {
    static constexpr int REQ = MBS * SL, PER = (REQ + NW - 1) / NW;  // 1 KB requests of a stage / of a wave
    __amdgpu_buffer_rsrc_t win;
    uint32_t voff;
    int wave, mb_last, T;
    __device__ __forceinline__ void init(const uint16_t *xf, int slices, int mb0, int mb_total, int lane, int wave_) {
        T = slices;
        wave = wave_;
        const int rows = min(MBS, mb_total - mb0);
        mb_last = rows - 1;
        win = wave_window(reinterpret_cast<const uint8_t *>(xf) + static_cast<int64_t>(mb0) * slices * 1024,
                          static_cast<uint32_t>(rows) * static_cast<uint32_t>(slices) * 1024u);
        voff = static_cast<uint32_t>(lane) * 16u;
    }
    // lds: start of the stage's buffer, layout [mb][slice][1 KB].  Row-blocks and slices past the end repeat the last.
    __device__ __forceinline__ void issue(uint8_t *lds, int t0) const {
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            int q = wave + NW * p;
            if (REQ % NW != 0) q = min(q, REQ - 1);  // every wave issues the same number of requests
            const int mb = q / SL, sl = q - mb * SL;
            const int so = (min(mb, mb_last) * T + min(t0 + sl, T - 1)) * 1024;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(win, (lds_void_t)(lds + q * 1024), 16, voff,
                                                     __builtin_amdgcn_readfirstlane(so), 0, 0);
        }
    }
};

// The same for rows that are not neighbours (the pairs of an expert).  The activations are then kept row by row, 64 bytes per row
// and slice ("row order"): a request is one slice of 16 rows, four lanes per row, and leaves 1 KB in LDS of which lane (r, kb)
// reads the 16 bytes at row_order_lane.  The hardware serves a 16-byte read in four passes of 16 lanes, lanes 0-3, 12-15, 20-27 and
// 4-11, 16-19, 28-31 and the same 32 further (as far as conflict counts tell): quarter kb of a row lies at kb ^ (-(r / 4) & 3),
// with which each pass meets every bank once, as in fragment order.  Turned by r / 4 instead, reads met their banks twice (3.8
// conflict cycles each, a tenth of the kernel's time; the counters show none now).
__device__ __forceinline__ int row_order_quarter(int r, int kb) { return (kb ^ -(r >> 2)) & 3; }
__device__ __forceinline__ uint32_t row_order_lane(int lane) {
    const int r = lane & 15;
    return static_cast<uint32_t>(r * 64 + row_order_quarter(r, lane >> 4) * 16);
}
template <int MBS, int SL, int NW>
struct GatherCopy {
    static constexpr int REQ = MBS * SL, PER = (REQ + NW - 1) / NW;
    __amdgpu_buffer_rsrc_t win;
    uint32_t voff[PER];
    int wave, T;
    // src: LDS table of the source row of each of the 16 * MBS rows, all below n_rows
    __device__ __forceinline__ void init(const uint16_t *x, int slices, const int *src, int n_rows, int lane, int wave_) {
        T = slices;
        wave = wave_;
        win = wave_window(reinterpret_cast<const uint8_t *>(x), static_cast<uint32_t>(n_rows) * static_cast<uint32_t>(slices) * 64u);
        const int r = lane >> 2;
#pragma unroll
        for (int p = 0; p < PER; ++p)
            voff[p] = static_cast<uint32_t>(src[min(wave + NW * p, REQ - 1) / SL * 16 + r]) * static_cast<uint32_t>(slices) * 64u +
                      static_cast<uint32_t>(row_order_quarter(r, lane & 3) * 16);
    }
    __device__ __forceinline__ void issue(uint8_t *lds, int t0) const {
#pragma unroll
        for (int p = 0; p < PER; ++p) {
            const int q = min(wave + NW * p, REQ - 1);  // every wave issues the same number of requests
            __builtin_amdgcn_raw_ptr_buffer_load_lds(win, (lds_void_t)(lds + q * 1024), 16, voff[p],
                                                     __builtin_amdgcn_readfirstlane(min(t0 + q % SL, T - 1) * 64), 0, 0);
        }
    }
};

// The K loop over the steps [step_begin, step_end) of the tensor (a step = B::STEP slices, unrolled).
//   B::SL           slices of an LDS stage (one barrier per stage); R = stages of the ring
//   B::NBUF         weight-fragment buffers: slice i multiplies bf[i % NBUF] while produce<i>() fills
//                   bf[(i + NBUF - 1) % NBUF] with the fragments of slice i + NBUF - 1
//   B::loads(i)     vector-memory requests of issue<i>()
// lane_off: where in the 1 KB of a slice the lane's fragment lies.  The caller has made the weights' first requests (w.prologue) and,
// where PRIMED, those of the first R - 1 stages.
// PAIRED: fragments go through in pairs, the later one first.  One wait then serves both where each would have its own, and every
// instruction of the loop takes an issue slot from the matrix instructions.  Two fragments stay in flight meanwhile, so not with fewer
// than four in registers; with four row-blocks the registers do not hold the pair.  Before and after, us: FFN of NINT4-32 4096 / 12288
// at 100 rows 73.1, 71.3, at 2048 602.1, 598.5; NINT5-28 12288 x 4096 at 200 rows 57.1, 54.6; NINT8-0 12288 x 4096 at 333 and 2048
// rows 75.0 and 257.1, 73.0 and 252.2.  Nothing with the other weights of row_tile.hpp (0.5 % slower at 100 to 333 rows of 4096 x 4096),
// and 1 to 2 % slower with the routed experts' gathered rows.
template <class B, int MT, int R, bool PRIMED = false, bool PAIRED = false, class Copy>
__device__ __forceinline__ void tile_loop(B &w, const Copy &cp, uint8_t *lds, int step_begin, int step_end, uint32_t lane_off,
                                          float4_t (&acc)[MT][B::NBLK]) {
    constexpr int SL = B::SL, NB = B::NBLK, STEP = B::STEP, NBUF = B::NBUF;
    constexpr int STAGE = MT * SL * 1024;  // bytes
    constexpr int AR = MT % 4 == 0 ? 4 : MT % 3 == 0 ? 3 : MT;  // activation fragments in registers
    constexpr int PERW = Copy::PER;
    static_assert(MT % AR == 0 && STEP % SL == 0 && STEP % NBUF == 0 && R >= 3, "ring positions are compile-time constants");
    u32x4_t af[AR];
    uint32_t rd = 0, wr = (R - 1) * STAGE;  // ring positions (bytes) of the current stage and of the one the next copy goes to
    // Addresses of the current and the next stage: one register each and immediate offsets.  The position is opaque:
    // where the unrolled body is a whole number of turns of the ring the compiler would otherwise keep an address
    // register for every fragment beyond the reach of an offset.
    uint32_t cur = lane_off, nxt = lane_off + STAGE;
    auto aread = [&](uint32_t stage, int sl, int a) {
        return *reinterpret_cast<const u32x4_t *>(lds + stage + (a * SL + sl) * 1024);
    };
    if constexpr (!PRIMED) {
#pragma unroll
        for (int i = 0; i < R - 1; ++i) cp.issue(lds + i * STAGE, step_begin * STEP + i * SL);
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0), through a wait the compiler sees: it then counts only the loop's requests
    __syncthreads();
    w.first(step_begin);
#pragma unroll
    for (int a = 0; a < AR; ++a) af[a] = aread(cur, 0, a);
    for (int s = step_begin; s < step_end; ++s) {
        static_for<STEP>([&](auto I) {
            constexpr int i = I.value;
            constexpr bool last = i % SL == SL - 1;  // of its stage: the reads ahead enter the next stage
            if constexpr (last) {
                // The next stage was requested R - 2 stages ago; what is younger than it: the copies of the R - 3 stages
                // after it and the weight requests made since.  After the barrier every wave has consumed the stage
                // before the current one, whose buffer takes the next copy.
                __builtin_amdgcn_sched_barrier(0);
                wait_vmcnt<(R - 3) * PERW + B::loads_before(i, (R - 2) * SL)>();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                cp.issue(lds + wr, s * STEP + i + 1 + (R - 2) * SL);
                // The count above holds only if all copies come before issue<i>'s requests: where the compiler put two of
                // those in between, ten requests were admitted with eight younger than the last copy.
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                wr = wr + STAGE == R * STAGE ? 0u : wr + STAGE;
            }
            w.template issue<i>(s);
            auto next_of = [&](int a) {
                if (a + AR < MT) return aread(cur, i % SL, a + AR);
                if (last) return aread(nxt, 0, a + AR - MT);
                return aread(cur, i % SL + 1, a + AR - MT);
            };
            if constexpr (PAIRED && AR == 4 && NB < 4) {
                static_for<MT / 2>([&](auto A) {
                    constexpr int a = 2 * A.value;
#pragma unroll
                    for (int b = 0; b < NB; ++b) acc[a + 1][b] = B::mfma(w.bf[i % NBUF][b], af[(a + 1) % AR], acc[a + 1][b]);
#pragma unroll
                    for (int b = 0; b < NB; ++b) acc[a][b] = B::mfma(w.bf[i % NBUF][b], af[a % AR], acc[a][b]);
                    w.template produce<i, a, MT>(s);
                    af[a % AR] = next_of(a);
                    af[(a + 1) % AR] = next_of(a + 1);
                    w.template produce<i, a + 1, MT>(s);
                    B::template schedule<MT>();
                });
            } else {
                static_for<MT>([&](auto A) {
                    constexpr int a = A.value;
#pragma unroll
                    for (int b = 0; b < NB; ++b) acc[a][b] = B::mfma(w.bf[i % NBUF][b], af[a % AR], acc[a][b]);
                    af[a % AR] = next_of(a);
                    w.template produce<i, a, MT>(s);
                    B::template schedule<MT>();
                });
            }
            if constexpr (last) {
                cur = nxt;
                rd = rd + STAGE == R * STAGE ? 0u : rd + STAGE;
                const uint32_t ahead = rd + STAGE == R * STAGE ? 0u : rd + STAGE;
                nxt = lane_off + ahead;
                asm volatile("" : "+v"(nxt));
            }
        });
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // late copies must not land in reused LDS
    __syncthreads();
}

// Results of 16 rows by 16 * NB columns, four consecutive columns of row lane % 16 in each of a lane's vectors: they leave through
// the wave's own kRowsOut bytes of LDS so that neighbouring lanes of a store lie side by side in a row.  Stored as they come, every
// lane of a store is in another row, which occupies a compute unit's address path four times as long.  dst(r): the row of y that
// row r of the tile goes to, or -1; columns [n0, n_end) are stored, n_end - n0 <= 16 * NB.  wide: rows of y at 16 bytes.
// NINT4-32 12288 x 4096 at 512 / 1024 / 2048 rows on blocks of eight waves 55.9 / 109.6 / 185.9 us, then 53.6 / 106.2 / 179.2.
constexpr int kRowsOut = 16 * (4 * 64 + 16);
template <int NB, class Dst>
__device__ __forceinline__ void store_rows(uint8_t *area, const float4_t (&v)[NB], int lane, int n0, int n_end, float *y, int64_t ldy, bool wide, Dst dst) {
    constexpr int PITCH = NB * 64 + 16;  // an odd number of 16-byte pieces: the lanes of a write meet every bank once
    static_assert(NB <= 4, "kRowsOut");
    uint8_t *to = area + (lane & 15) * PITCH + (lane >> 4) * 16;
#pragma unroll
    for (int b = 0; b < NB; ++b) *reinterpret_cast<float4_t *>(to + b * 64) = v[b];
    wave_sync();
    float4_t o[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int i = lane + 64 * j;
        o[j] = *reinterpret_cast<const float4_t *>(area + i / (4 * NB) * PITCH + i % (4 * NB) * 16);
    }
    wave_sync();
#pragma unroll
    for (int j = 0; j < NB; ++j) {
        const int i = lane + 64 * j, n = n0 + i % (4 * NB) * 4, m = dst(i / (4 * NB));
        if (m < 0 || n >= n_end) continue;
        float *p = y + static_cast<int64_t>(m) * ldy + n;
        if (wide && n + 4 <= n_end) {
            *reinterpret_cast<float4_t *>(p) = o[j];
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                if (n + t < n_end) p[t] = o[j][t];
        }
    }
}
// The same for results of two bytes, two packed per word.
template <int NB, class Dst>
__device__ __forceinline__ void store_rows16(uint8_t *area, const u32x2_t (&v)[NB], int lane, int n0, int n_end, uint16_t *y, int64_t ldy, bool wide, Dst dst) {
    constexpr int PITCH = NB * 32 + 16;
    uint8_t *to = area + (lane & 15) * PITCH + (lane >> 4) * 8;
#pragma unroll
    for (int b = 0; b < NB; ++b) *reinterpret_cast<u32x2_t *>(to + b * 32) = v[b];
    wave_sync();
    constexpr int PIECES = 32 * NB, PER = (PIECES + 63) / 64;  // of 16 bytes
    u32x4_t o[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = min(lane + 64 * j, PIECES - 1);
        o[j] = *reinterpret_cast<const u32x4_t *>(area + i / (2 * NB) * PITCH + i % (2 * NB) * 16);
    }
    wave_sync();
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const int i = lane + 64 * j;
        if (i >= PIECES) continue;
        const int n = n0 + i % (2 * NB) * 8, m = dst(i / (2 * NB));
        if (m < 0 || n >= n_end) continue;
        uint16_t *p = y + static_cast<int64_t>(m) * ldy + n;
        if (wide && n + 8 <= n_end) {
            *reinterpret_cast<u32x4_t *>(p) = o[j];
        } else {
#pragma unroll
            for (int t = 0; t < 8; ++t)
                if (n + t < n_end) p[t] = static_cast<uint16_t>(o[j][t >> 1] >> (16 * (t & 1)));
        }
    }
}

// Blocks go to the XCDs in turn: XCD x takes a contiguous range of the tiles, which are ordered in bands of GM row tiles, rows
// fastest inside a band: the 32 or 64 tiles an XCD has in flight are about as tall as wide, so both their activations and
// their weights are read into its L2 a few times only (all row tiles in one band: 3 to 5 % slower at 2048 rows).
__device__ __forceinline__ bool tile_of_block(int tiles_n, int tiles_m, int &tn, int &tm) {
    constexpr int GM = 8;
    const int total = tiles_n * tiles_m, per = (total + 7) / 8, b = blockIdx.x;
    const int t = (b & 7) * per + (b >> 3);
    if (t >= total || (b >> 3) >= per) return false;
    const int band = t / (GM * tiles_n), rows = min(GM, tiles_m - band * GM), in = t - band * GM * tiles_n;
    tn = in / rows;
    tm = band * GM + in % rows;
    return true;
}

// Tile shapes a launch can take: 16 * MT tokens x 16 * NB * NW neurons (half of that with GLU) per block of NW waves.  Two
// blocks of four waves share a compute unit, and one fills the other's start and end; a block of eight fetches the same
// activations once for twice the neurons (4096 x 12288 at 2048 rows: 172 us against 178; 8 x 3 x 8 was never more than 2 %
// ahead of 8 x 3 x 4).  Four row-blocks a wave read a fragment of activations for four instructions, and take every register of the
// profiles that have enough: gate/up 24576 x 4096 NINT4-32 at 2048 rows 342 us with three and 322 with four, 12288 x 4096 177 and 170.
struct NintTileShape { int mt, nb, nw; };
constexpr int kTileShapes = 6;
constexpr NintTileShape kTileShape[kTileShapes] = {{8, 2, 8}, {8, 3, 4}, {8, 2, 4}, {4, 3, 4}, {4, 2, 4}, {8, 4, 4}};

// The tile and split over K of a launch with the smallest modelled time (nint_tile.hip): rbs row-blocks of output neurons, nsteps
// steps of per_step slices; widest: row-blocks of a wave that the registers hold; halves: gate and up waves side by side; weight: what a
// fragment of weights takes to make (NINT of two and four bits; NINT of other widths; MX rows and fp16 copies; NINT8-0 rows).
enum TileWeight { kTileLight, kTileDecoded, kTileRows, kTileHeavy };
struct TilePlan {
    int shape, splits, spz;
    double us;
};
// pieces of a split over K whose partial results fit behind the first `used` bytes of a workspace (at most 8, at least 1)
inline int splits_that_fit(size_t ws_bytes, size_t used, int M, int out) {
    const size_t n = ws_bytes > used ? (ws_bytes - used) / (static_cast<size_t>(M) * out * 4) : 0;
    return n < 1 ? 1 : n > 8 ? 8 : static_cast<int>(n);
}
TilePlan tile_plan(int rbs, int nsteps, int per_step, int rows, int out, int max_splits, int widest, TileWeight weight, bool halves);

}  // namespace mfq
