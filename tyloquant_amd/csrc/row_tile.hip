// Launches of the tile kernel on row-major weights (row_tile.hpp), their workspaces, and the dense product of formats that are
// dequantized to fp16 fragments first.
#include "row_tile.hpp"

namespace mfq {

int x_frag(const void *x, int x_dtype, int64_t ldx, int M, int K, int GS, int nsteps, uint16_t *xf, float *xscale, uint16_t *xg,
           bool keep_bf16, hipStream_t st);
int prefill_sum_splits(const float *part, int64_t ystride, int splits, int M, int N, float *y, int64_t ldy, hipStream_t st);
int row_tile_q8(const RowTileArgs &a, int shape, int splits, hipStream_t st);
int row_tile_mx4(const RowTileArgs &a, bool f16, int shape, int splits, hipStream_t st);
int row_tile_mx8(const RowTileArgs &a, bool f16, int shape, int splits, hipStream_t st);

static int row_gs(int kind) { return kind == kRowF16 ? 8 : kind == kRowMx8 || kind == kRowMx8F16 ? 16 : 32; }
// A step is 256 columns; x_frag writes whole runs of 16 groups, and zeros for as many steps as the kernel walks.
static int row_steps(int K) { return static_cast<int>(ceil_div(K, 256)); }
static int row_xf_steps(int kind, int K) { return static_cast<int>(ceil_div(row_steps(K) * 256, 16 * row_gs(kind))); }
static TilePlan row_plan(int kind, int N, int K, int M, int room = 8) {  // room: splits the workspace holds
    const int nsteps = row_steps(K), most = N % 4 ? 1 : nsteps / 2 < 8 ? nsteps / 2 : 8, splits = most < room ? most : room;
    return tile_plan(static_cast<int>(ceil_div(N, 16)), nsteps, 8, M, N, splits, kind != kRowQ8, false);
}
static size_t align256(size_t v) { return (v + 255) & ~static_cast<size_t>(255); }
struct RowCarve { size_t xf, xscale, wscale, part; };
static RowCarve row_carve(int kind, int N, int K, int M) {
    const size_t mbs = static_cast<size_t>(ceil_div(M, 16));
    RowCarve c;
    c.xf = 0;
    c.xscale = c.xf + mbs * row_xf_steps(kind, K) * (2 * row_gs(kind) / 4) * 1024;
    c.wscale = c.xscale + align256(mbs * 64);
    c.part = c.wscale + align256(static_cast<size_t>(N) * 4);
    return c;
}
// What a call makes use of (the activations, a scale per neuron, the partial results of its split over K), and what it cannot
// do without, which grows with the rows.
size_t row_tile_workspace(int kind, int N, int K, int M) {
    const int splits = row_plan(kind, N, K, M).splits;
    return row_carve(kind, N, K, M).part + (splits > 1 ? align256(static_cast<size_t>(splits) * M * N * 4) : 0);
}
size_t row_tile_workspace_least(int kind, int N, int K, int M) { return row_carve(kind, N, K, M).part; }
float *row_tile_wscale(int kind, int N, int K, int M, void *ws) {
    return reinterpret_cast<float *>(static_cast<uint8_t *>(ws) + row_carve(kind, N, K, M).wscale);
}
// modelled time of a call, the launch that orders the activations included (5 us up to a few hundred rows)
double row_tile_us(int kind, int N, int K, int M) { return row_plan(kind, N, K, M).us + 5.0; }
bool row_tile_fits(int64_t row_bytes, const void *w) { return 64 * row_bytes < (1ll << 31) && (reinterpret_cast<uintptr_t>(w) & 3) == 0; }

// y of M activation rows against neurons [row0, row0 + N).  scaled: row_tile_wscale's array holds a factor per neuron.
// ws_bytes: at least row_tile_workspace_least; with less than row_tile_workspace K is split into fewer pieces.
int row_tile(int kind, const void *w, const void *scales, int64_t row_bytes, int row0, int N, int K, bool scaled, const void *x, int x_dtype,
             int64_t ldx, int M, float *y, int64_t ldy, void *ws, size_t ws_bytes, hipStream_t st) {
    const RowCarve c = row_carve(kind, N, K, M);
    const TilePlan pl = row_plan(kind, N, K, M, splits_that_fit(ws_bytes, c.part, M, N));
    uint8_t *base = static_cast<uint8_t *>(ws);
    uint16_t *xf = reinterpret_cast<uint16_t *>(base + c.xf);
    float *xscale = reinterpret_cast<float *>(base + c.xscale), *wscale = reinterpret_cast<float *>(base + c.wscale);
    float *part = reinterpret_cast<float *>(base + c.part);
    const int gs = row_gs(kind), xs = row_xf_steps(kind, K);
    if (int rc = x_frag(x, x_dtype, ldx, M, K, gs, xs, xf, xscale, nullptr, kind == kRowMx4 || kind == kRowMx8, st)) return rc;
    const bool split = pl.splits > 1;
    const RowTileArgs a{static_cast<const uint8_t *>(w), static_cast<const uint8_t *>(scales), row_bytes, row0, N, K, M, xf, xscale,
                        scaled ? wscale : nullptr, split ? part : y, split ? N : ldy, static_cast<int64_t>(M) * N, xs * (gs / 2),
                        row_steps(K), pl.spz};
    int rc;
    switch (kind) {
        case kRowF16: rc = row_tile_launch<kRowF16>(a, pl.shape, pl.splits, st); break;
        case kRowQ8: rc = row_tile_q8(a, pl.shape, pl.splits, st); break;
        case kRowMx4: case kRowMx4F16: rc = row_tile_mx4(a, kind == kRowMx4F16, pl.shape, pl.splits, st); break;
        default: rc = row_tile_mx8(a, kind == kRowMx8F16, pl.shape, pl.splits, st); break;
    }
    if (rc) return rc;
    return split ? prefill_sum_splits(part, a.zstride, pl.splits, M, N, y, ldy, st) : MFQ_OK;
}

// ---- formats that are dequantized to fp16 fragments first --------------------------------------------------------------------
// Workspace: w16, [N rounded up to 16, Kp] in fragment order (frag16_at), Kp = K rounded up to 32 (the padding is zero), then
// that of the tile kernel.
//
// Codebook formats with a prefill kernel of their own (NVQ D4, NEPQ1) look every weight up again in each tile of 64 or 128
// tokens, which leaves that kernel at 0.5 .. 0.7 PFLOP/s; the copy costs one pass over the tensor (17 to 30 us for 12288 x 4096)
// and then runs at the tile kernel's rate.  It wins from about 1.5 million outputs on, once a 64 x 96 tile falls to every
// compute unit, but not below 256 rows (128 rows of 12288 x 4096 / 17408 x 5120: 55 / 102 us against 52 / 87).  Whole calls, fragments
// from the codebooks against the copy, bf16 activations:
//     NVQ3J-512  12288 x 4096 at 256 / 512 / 1024 / 2048 rows   74 /  92 / 175 / 284   63 /  81 / 116 / 204 us
//                17408 x 5120                                  112 / 211 / 318 / 569  108 / 155 / 225 / 386
//                4096 x 12288 at 256 / 384 / 1024 / 2048        66 / 105 / 188 / 266   76 /  86 / 135 / 209
//                1536 x 2048 at 512 / 768 / 1024 / 2048         30 /  32 /  37 /  50   30 /  33 /  33 /  38
//     NEPQ1-S    12288 x 4096 at 256 / 512 / 1024 / 2048        68 /  88 / 166 / 261   61 /  79 / 113 / 192
//                4096 x 4096 at 256 / 384 / 1024 / 2048         38 /  49 /  70 /  97   36 /  40 /  56 /  78
// A copy of more than half a gigabyte (a vocabulary-sized head) is not taken: it would be the call's largest allocation by far.
bool prefill_by_copy(int N, int K, int M) {
    return M >= 256 && static_cast<int64_t>(M) * N >= 1500000 && static_cast<int64_t>(N) * K <= (1ll << 28);
}
static size_t copy_bytes(int N, int K) { return static_cast<size_t>(ceil_div(N, 16)) * static_cast<size_t>(ceil_div(K, 32)) * 1024; }
size_t dequant_gemm_workspace(int N, int K, int M) { return copy_bytes(N, K) + row_tile_workspace(kRowF16, N, K, M); }
size_t dequant_gemm_workspace_least(int N, int K, int M) { return copy_bytes(N, K) + row_tile_workspace_least(kRowF16, N, K, M); }
void dequant_gemm_carve(void *ws, int N, int K, int M, uint16_t *&w16, float *&wscale, int &Kp) {
    Kp = static_cast<int>(ceil_div(K, 32)) * 32;
    w16 = static_cast<uint16_t *>(ws);
    wscale = row_tile_wscale(kRowF16, N, K, M, static_cast<uint8_t *>(ws) + copy_bytes(N, K));
}
int dequant_gemm(void *ws, size_t ws_bytes, int N, int K, const void *x, int x_dtype, int64_t ldx, int M, float *y, int64_t ldy, hipStream_t st) {
    const size_t copy = copy_bytes(N, K);
    const int64_t row_bytes = 2 * ceil_div(K, 32) * 32;
    MFQ_REQUIRE(row_tile_fits(row_bytes, ws), MFQ_ERR_UNSUPPORTED, "dequant_gemm: rows of %d columns, workspace at %p", K, ws);
    return row_tile(kRowF16, ws, nullptr, row_bytes, 0, N, K, true, x, x_dtype, ldx, M, y, ldy, static_cast<uint8_t *>(ws) + copy,
                    ws_bytes - copy, st);
}

}  // namespace mfq
