// Activations of the tile kernels (tile_gemm.hpp) in fragment order.
#include "tune.hpp"
#include "xfrag.hpp"

namespace mfq {

// steps of a round: about a thousand values of a row
constexpr int x_frag_steps(int gs) { return 1024 / (16 * gs) > 0 ? 1024 / (16 * gs) : 1; }

// chunk c of a row: eight values, zeros past K and past the last of nch chunks
template <bool VEC>
__device__ __forceinline__ u32x4_t x_chunk(const uint16_t *__restrict__ xr, int c, int nch, int K) {
    u32x4_t v = u32x4_t{0u, 0u, 0u, 0u};
    if (c < nch) {
        if constexpr (VEC) {
            v = reinterpret_cast<const u32x4_t *>(xr)[c];
        } else {
#pragma unroll
            for (int t = 0; t < 8; ++t)
                if (8 * c + t < K) v[t >> 1] |= static_cast<uint32_t>(xr[8 * c + t]) << (16 * (t & 1));
        }
    }
    return v;
}

// xscale of every row by itself, a block per row (rows past M: 0).
template <int XF16, bool VEC>
__global__ __launch_bounds__(256) void x_row_scale_kernel(const uint16_t *__restrict__ x, int64_t ldx, int M, int K, float *__restrict__ xscale) {
    __shared__ uint32_t red[4];
    const int m = blockIdx.x, tid = threadIdx.x, nch = (K + 7) >> 3;
    if (m >= M) {
        if (tid == 0) xscale[m] = 0.f;
        return;
    }
    const uint16_t *xr = x + static_cast<int64_t>(m) * ldx;
    uint32_t top = 0;
    for (int c = tid; c < nch; c += 2048) {
        u32x4_t v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = x_chunk<VEC>(xr, c + 256 * i, nch, K);
#pragma unroll
        for (int i = 0; i < 8; ++i) top = finite_top<XF16>(top, v[i]);
    }
    for (int o = 32; o > 0; o >>= 1) top = max(top, static_cast<uint32_t>(__shfl_xor(static_cast<int>(top), o, 64)));
    if ((tid & 63) == 0) red[tid >> 6] = top;
    __syncthreads();
    if (tid == 0) xscale[m] = ldexpf(1.f, row_exp<XF16>(max(max(red[0], red[1]), max(red[2], red[3]))) - 9);
}

// One block = the 16 rows of row-block blockIdx.x, a row per wave.  The whole row is requested at once into registers (the
// first KEEP * 512 values; what is longer is read a second time), its largest finite magnitude gives the power of two that
// brings the row maximum into [256, 512) in fp16, and rounds of about a thousand values per row pass through LDS, from where
// every wave writes whole 1 KB fragments:
//     xf[mb][slice][lane (r, kb)][8] = x[16 mb + r][(4 u + kb) GS + 8 mm ...], slice = u * NM + mm, NM = ceil(GS / 8)
// with zeros behind a group's last value, behind K and in rows past M.  With xg != null also the group sums in two fp16
// halves, xg[mb][step][lane][8] = Xhi of groups 16 s + 4 j + kb (j = 0..3), then Xlo; X summed in k order.
// SCALE = 0 keeps bf16 activations as they are (xscale = 1), for weights that are exact in bf16.
// gridDim.y > 1 (few rows): the blocks of a row-block all read the rows and share the rounds.
// KEEP = 0: x_row_scale_kernel has left xscale, and a block reads the pieces of its rounds only.
// Behind the row-blocks' columns of the grid, blocks for the neurons of rs (groups of 16 only; x_frag_scales says when).
// The launch moves 4 bytes per activation: 2048 rows of 4096 / 12288 values take 9 / 30 us (3.7 / 3.3 TB/s), a few hundred of
// 4096 6 to 7 us.
template <int GS, int XF16, bool VEC, bool SCALE, int KEEP>
__global__ __launch_bounds__(1024) void x_frag_kernel(const uint16_t *__restrict__ x, int64_t ldx, int M, int K, int nsteps, uint16_t *__restrict__ xf, float *__restrict__ xscale,
                                                      uint16_t *__restrict__ xg, RowScales rs) {
    extern __shared__ __attribute__((aligned(16))) uint16_t rows[];  // [2][16][spr * 16 * GS + 8]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int mb = blockIdx.x, m = mb * 16 + wave;
    if constexpr (GS == 16 && SCALE) {
        const int extra = static_cast<int>(blockIdx.x) - ((M + 15) >> 4);
        if (extra >= 0) {
            const int block = extra * gridDim.y + blockIdx.y;
            if (block < rs.blocks)
                for (int row = block * 16 + wave; row < rs.out; row += rs.blocks * 16) row_scale(rs, row, lane);
            return;
        }
    }
    constexpr int NM = (GS + 7) / 8, spr = x_frag_steps(GS), SEG = spr * 16 * GS, LD = SEG + 8;
    const bool live = m < M;
    const uint16_t *xr = x + static_cast<int64_t>(live ? m : 0) * ldx;
    const int nch = live ? (K + 7) >> 3 : 0;  // chunks of eight values
    auto fetch = [&](int c) { return x_chunk<VEC>(xr, c, nch, K); };
    u32x4_t keep[KEEP ? KEEP : 1];
#pragma unroll
    for (int i = 0; i < KEEP; ++i) keep[i] = fetch(lane + 64 * i);
    float inv = 1.f;
    if constexpr (KEEP == 0) {
        if (live) inv = __uint_as_float((254u << 23) - __float_as_uint(xscale[m]));  // a normal power of two
    } else if constexpr (SCALE) {
        // Infinities and NaNs come out on top; a row that holds one (rare) is searched again without them.
        constexpr uint32_t kInf = XF16 ? 0x7c00u : 0x7f80u;
        u16x2_t big = u16x2_t{0, 0};
        for (int c = lane + 64 * KEEP; c < nch; c += 256) {
            u32x4_t v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = fetch(c + 64 * i);
#pragma unroll
            for (int i = 0; i < 4; ++i) big = pair_top(big, v[i]);
        }
#pragma unroll
        for (int i = 0; i < KEEP; ++i) big = pair_top(big, keep[i]);
        uint32_t top = max(big.x, big.y);
        for (int o = 32; o > 0; o >>= 1) top = max(top, static_cast<uint32_t>(__shfl_xor(static_cast<int>(top), o, 64)));
        if (top >= kInf) {
            top = 0;
            for (int c = lane; c < nch; c += 64) top = finite_top<XF16>(top, fetch(c));
            for (int o = 32; o > 0; o >>= 1) top = max(top, static_cast<uint32_t>(__shfl_xor(static_cast<int>(top), o, 64)));
        }
        const int e = row_exp<XF16>(top);
        inv = ldexpf(1.f, 9 - e);
        if (blockIdx.y == 0 && lane == 0) xscale[m] = live ? ldexpf(1.f, e - 9) : 0.f;
    } else {
        if (blockIdx.y == 0 && lane == 0) xscale[m] = live ? 1.f : 0.f;
    }
    auto conv = [&](u32x4_t v) -> u32x4_t {
        if constexpr (!SCALE) return v;
        return scaled_f16<XF16>(v, inv);
    };
    const int r = lane & 15, kb = lane >> 4;
    const int T = nsteps * 4 * NM, rounds = (nsteps + spr - 1) / spr;
    uint16_t *buf = rows;
    for (int q = blockIdx.y; q < rounds; q += gridDim.y) {
        const int c0 = q * (SEG / 8);
        uint16_t *mine = buf + wave * LD;
        if constexpr (KEEP == 0) {
            constexpr int NC = (SEG / 8 + 63) / 64;
            u32x4_t v[NC];
#pragma unroll
            for (int i = 0; i < NC; ++i) v[i] = fetch(c0 + lane + 64 * i);
#pragma unroll
            for (int i = 0; i < NC; ++i)
                if (lane + 64 * i < SEG / 8) *reinterpret_cast<u32x4_t *>(mine + 8 * (lane + 64 * i)) = conv(v[i]);
        } else {
#pragma unroll
            for (int i = 0; i < KEEP; ++i) {
                const int c = lane + 64 * i - c0;
                if (c >= 0 && c < SEG / 8) *reinterpret_cast<u32x4_t *>(mine + 8 * c) = conv(keep[i]);
            }
            for (int c = max(lane + 64 * KEEP, c0 + ((lane - c0) & 63)); c < c0 + SEG / 8; c += 64)
                *reinterpret_cast<u32x4_t *>(mine + 8 * (c - c0)) = conv(fetch(c));
        }
        __syncthreads();
        const int ns = min(spr, nsteps - q * spr);
        for (int t = wave; t < ns * 4 * NM; t += 16) {
            const int u = t / NM, mm = t - u * NM;
            const uint16_t *src = buf + r * LD + (4 * u + kb) * GS + 8 * mm;
            u32x4_t h;
            if constexpr (GS % 8 == 0) {
                h = *reinterpret_cast<const u32x4_t *>(src);
            } else {  // groups of a multiple of four values: eight-byte pieces, the last slice half empty
                const u32x2_t a = *reinterpret_cast<const u32x2_t *>(src);
                h = u32x4_t{a.x, a.y, 0u, 0u};
                if (8 * mm + 8 <= GS) {
                    const u32x2_t b = *reinterpret_cast<const u32x2_t *>(src + 4);
                    h.z = b.x; h.w = b.y;
                }
            }
            *reinterpret_cast<u32x4_t *>(xf + ((static_cast<int64_t>(mb) * T + q * spr * 4 * NM + t) * 64 + lane) * 8) = h;
        }
        if (xg) {
            // a wave takes one of the four groups j of a step at a time: lane (r, kb) leaves two of its eight halves
            for (int t = 15 - wave; t < ns * 4; t += 16) {
                const int s = t >> 2, j = t & 3;
                const u32x2_t *p = reinterpret_cast<const u32x2_t *>(buf + r * LD + (16 * s + 4 * j + kb) * GS);
                float X = 0.f;
#pragma unroll
                for (int i = 0; i < GS / 4; ++i) {
                    const u32x2_t v = p[i];
                    X = dot2<1>(v.x, 0x3c003c00u, X);
                    X = dot2<1>(v.y, 0x3c003c00u, X);
                }
                const uint16_t hi = f32_to_f16_rne(X);
                uint16_t *o = xg + ((static_cast<int64_t>(mb) * nsteps + q * spr + s) * 64 + lane) * 8 + j;
                o[0] = hi;
                o[4] = f32_to_f16_rne(X - f16_to_f32(hi));
            }
        }
        buf = buf == rows ? rows + 16 * LD : rows;  // the next round's values go to the other half: one barrier per round
    }
}

template <int GS>
static int x_frag_start(const void *x, int x_dtype, int64_t ldx, int M, int K, int nsteps, uint16_t *xf, float *xscale, uint16_t *xg,
                        bool keep_bf16, const RowScales &rs, hipStream_t st) {
    const int mbs = static_cast<int>(ceil_div(M, 16));
    const bool vec = K % 8 == 0 && ldx % 8 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0;
    constexpr int spr = x_frag_steps(GS);
    const int rounds = static_cast<int>(ceil_div(nsteps, spr));
    int share = device_cu_count() / mbs;  // few rows: several blocks share the rounds of a row-block
    share = share < 1 ? 1 : share;
    dim3 grid(static_cast<unsigned>(mbs), static_cast<unsigned>(share < rounds ? share : rounds));
    // Several blocks per row-block would each read its rows whole to find their scale: two launches take 4.6 + 4.8 us at 300 rows
    // of 12288 values (one: 14.1), 5.1 + 6.1 at 300 of 17408 (20.4), 3.5 + 4.0 at 200 of 6144 (9.3), and 5.4 + 7.4 at 1024 of
    // 8192 (12.8), 3.3 + 3.8 at 200 of 4096 (6.3).
    const bool long_rows = K > 6144 && share >= 6;
    const size_t lds = 2 * 16 * (static_cast<size_t>(spr) * 16 * GS + 8) * 2;
    const uint16_t *xp = static_cast<const uint16_t *>(x);
#define MFQ_XFRAG_K(F, V, S, KEEP)                                                                                     \
    do {                                                                                                               \
        auto kern = x_frag_kernel<GS, F, V, S, KEEP>;                                                                  \
        if (GS == 16 && S) grid.x += static_cast<unsigned>(ceil_div(rs.blocks, grid.y));                               \
        if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(kern), lds, "x_frag")) return rc;                \
        hipLaunchKernelGGL(kern, grid, dim3(1024), lds, st, xp, ldx, M, K, nsteps, xf, xscale, xg, rs);                \
        return check_launch("x_frag");                                                                                 \
    } while (0)
    // 8 chunks of a lane are a row of 4096 values, 16 one of 8192 (the 128 registers of such a block hold no more).
#define MFQ_XFRAG(F, S)                                                                                                \
    do {                                                                                                               \
        if (S && long_rows) {                                                                            \
            if (vec) hipLaunchKernelGGL((x_row_scale_kernel<F, true>), dim3(static_cast<unsigned>(16 * mbs)), dim3(256), 0, st, xp, ldx, M, K, xscale); \
            else hipLaunchKernelGGL((x_row_scale_kernel<F, false>), dim3(static_cast<unsigned>(16 * mbs)), dim3(256), 0, st, xp, ldx, M, K, xscale);    \
            if (int rc = check_launch("x_row_scale")) return rc;                                                       \
            grid.y = static_cast<unsigned>(rounds);                                                                    \
            if (!vec) MFQ_XFRAG_K(F, false, S, 0);                                                                     \
            MFQ_XFRAG_K(F, true, S, 0);                                                                                \
        }                                                                                                              \
        if (!vec) MFQ_XFRAG_K(F, false, S, 8);                                                                         \
        if (K <= 4096) MFQ_XFRAG_K(F, true, S, 8);                                                                     \
        MFQ_XFRAG_K(F, true, S, 16);                                                                                   \
    } while (0)
    if (x_dtype == MFQ_X_F16) MFQ_XFRAG(1, true);
    if constexpr (GS == 16 || GS == 32) {
        if (keep_bf16) MFQ_XFRAG(0, false);
    }
    MFQ_XFRAG(0, true);
#undef MFQ_XFRAG
#undef MFQ_XFRAG_K
}

// xf: ceil(M / 16) * nsteps * 4 * ceil(GS / 8) KB, xscale: 16 * ceil(M / 16) floats, xg (or null): ceil(M / 16) * nsteps KB.
// GS = 8 is the plain order of 32 k-values per slice; keep_bf16 (groups of 16 and 32) copies bf16 rows unscaled.
int x_frag(const void *x, int x_dtype, int64_t ldx, int M, int K, int GS, int nsteps, uint16_t *xf, float *xscale, uint16_t *xg,
           bool keep_bf16, hipStream_t st) {
    MFQ_REQUIRE(static_cast<int64_t>(nsteps) * 16 * GS >= K, MFQ_ERR_INVALID, "x_frag: %d steps of 16 groups of %d for K = %d", nsteps, GS, K);
    switch (GS) {
#define MFQ_XFRAG_GS(G) case G: return x_frag_start<G>(x, x_dtype, ldx, M, K, nsteps, xf, xscale, xg, keep_bf16, RowScales{}, st);
        MFQ_XFRAG_GS(8) MFQ_XFRAG_GS(16) MFQ_XFRAG_GS(24) MFQ_XFRAG_GS(28) MFQ_XFRAG_GS(32) MFQ_XFRAG_GS(48)
#undef MFQ_XFRAG_GS
    }
    return fail(MFQ_ERR_UNSUPPORTED, "x_frag: groups of %d", GS);
}
__global__ __launch_bounds__(256) void row_scale_kernel(RowScales rs) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (row < rs.out) row_scale(rs, row, threadIdx.x & 63);
}
// The same in groups of 16, and the powers of two of a tensor's neurons: in that launch, one block a compute unit, up to 128 activation
// rows or four neurons a wave.  Whole calls of NINT8-0, a launch of their own and in that launch, us: 4096 x 4096 at 64 / 333 / 2048
// rows 24.1 / 39.9 / 86.5 and 21.6 / 37.9 / 85.0, 12288 x 4096 33.4 / 72.4 / 226 and 31.4 / 70.4 / 222, 4096 x 12288 at 333 67.3 and
// 65.1.  Beyond, the blocks of the neurons hold the activations' up: 37984 x 4096 at 64 rows 66.5 and 66.1, at 333 and 1024 161 and 383,
// 163 and 388 (with four neurons requested at a time the same, and 4096 x 4096 0.7 us slower).
int x_frag_scales(const void *x, int x_dtype, int64_t ldx, int M, int K, int nsteps, uint16_t *xf, float *xscale, const uint16_t *scales, int ng,
                  int out, float *rowscale, hipStream_t st) {
    MFQ_REQUIRE(static_cast<int64_t>(nsteps) * 256 >= K, MFQ_ERR_INVALID, "x_frag: %d steps of 256 for K = %d", nsteps, K);
    const int blocks = static_cast<int>(ceil_div(out, 16)), cus = device_cu_count();
    RowScales rs{scales, ng, out, blocks < cus ? blocks : cus, rowscale};
    if (M > 128 && out > 64 * cus) {
        rs.blocks = 0;
        hipLaunchKernelGGL(row_scale_kernel, dim3(static_cast<unsigned>(ceil_div(out, 4))), dim3(256), 0, st, rs);
        if (int rc = check_launch("row_scale")) return rc;
    }
    return x_frag_start<16>(x, x_dtype, ldx, M, K, nsteps, xf, xscale, nullptr, false, rs, st);
}

}  // namespace mfq
