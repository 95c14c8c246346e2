// Launches of the tile kernel on row-major weights (row_tile.hpp), their workspaces, and the dense product of formats that are
// dequantized to fp16 fragments first.
#include "row_tile.hpp"

namespace mfq {

int x_frag(const void *x, int x_dtype, int64_t ldx, int M, int K, int GS, int nsteps, uint16_t *xf, float *xscale, uint16_t *xg,
           bool keep_bf16, hipStream_t st);
int x_frag_scales(const void *x, int x_dtype, int64_t ldx, int M, int K, int nsteps, uint16_t *xf, float *xscale, const uint16_t *scales, int ng,
                  int out, float *rowscale, hipStream_t st);
int prefill_sum_splits(const float *part, int64_t ystride, int splits, int M, int N, float *y, int64_t ldy, hipStream_t st);
int row_tile_q8(const RowTileArgs &a, int shape, int splits, hipStream_t st);
int row_tile_mx4(const RowTileArgs &a, bool f16, int shape, int splits, hipStream_t st);
int row_tile_mx8(const RowTileArgs &a, bool f16, int shape, int splits, hipStream_t st);

static int row_gs(int kind) { return kind == kRowF16 ? 8 : kind == kRowMx4 || kind == kRowMx4F16 ? 32 : 16; }
// A step is 256 columns; x_frag writes whole runs of 16 groups, and zeros for as many steps as the kernel walks.
static int row_steps(int K) { return static_cast<int>(ceil_div(K, 256)); }
static int row_xf_steps(int kind, int K) { return static_cast<int>(ceil_div(row_steps(K) * 256, 16 * row_gs(kind))); }
static TilePlan row_plan(int kind, int N, int K, int M, int room = 8) {  // room: splits the workspace holds
    const int nsteps = row_steps(K), most = N % 4 ? 1 : nsteps / 2 < 8 ? nsteps / 2 : 8, splits = most < room ? most : room;
    return tile_plan(static_cast<int>(ceil_div(N, 16)), nsteps, 8, M, N, splits, row_tile_widest(kind),
                     kind == kRowQ8 ? kTileHeavy : kTileRows, false);
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
// modelled time of a call, the activations included: 5 us up to a few hundred rows, and two launches for long rows
double row_tile_us(int kind, int N, int K, int M) { return row_plan(kind, N, K, M).us + (K > 6144 ? 9.0 : 5.0); }
bool row_tile_fits(int64_t row_bytes, const void *w) { return 64 * row_bytes < (1ll << 31) && (reinterpret_cast<uintptr_t>(w) & 3) == 0; }

// y of M activation rows against neurons [row0, row0 + N).  scaled: a factor per neuron, which the caller has left in
// row_tile_wscale's array, or for kRowQ8 (whole tensors, row0 = 0) the launch that lays the activations out leaves there.
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
    if (int rc = kind == kRowQ8 ? x_frag_scales(x, x_dtype, ldx, M, K, xs, xf, xscale, static_cast<const uint16_t *>(scales), K / 32, N, wscale, st)
                                : x_frag(x, x_dtype, ldx, M, K, gs, xs, xf, xscale, nullptr, kind == kRowMx4 || kind == kRowMx8, st))
        return rc;
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
// and then runs at the tile kernel's rate.  It wins from about 1.5 million outputs on, but not below 256 rows (128 rows of
// 12288 x 4096: 55 us against 52).  A copy of more than 2^26 weights, half the last-level cache, goes through memory twice, about
// 1 us per million weights: it is taken where that and the tile kernel are cheaper than the codebook kernel's rounds of 128 x
// 256 tiles (round_us per 1024 columns each), and not where that kernel splits K.  Whole calls on two weights in turn, bf16,
// fragments from the codebooks / the copy, us ("-" behind it: not taken):
//     rows                        256      300      400      640      777     1024     2048
//     NVQ3J-512   4096 x 4096                     50/45    70/55    73/62    74/64   104/88
//                12288 x 4096    76/65    77/78   90/82    99/91  171/116  173/122  284/218
//                17408 x 5120  117/133- 116/137- 208/161  213/167  233/219- 317/227  569/391
//                32000 x 4096  116/184- 179/199- 189/227- 278/292- 361/336  376/398- 739/600
//                5120 x 17408    -      144/161- 255/180  260/201  329/259  334/286  664/444
//     NEPQ1-S     4096 x 4096                     47/41    64/49    66/57    67/59    97/81
//                12288 x 4096    70/63    70/70   85/81    91/89  162/112  164/118  262/210
//                24576 x 4096   95/131- 162/154- 161/170- 174/214- 254/274- 259/275- 505/449
// A copy of more than half a gigabyte (a vocabulary-sized head) is not taken: it would be the call's largest allocation by far.
bool prefill_by_copy(int N, int K, int M, double round_us) {
    const int64_t weights = static_cast<int64_t>(N) * K;
    if (M < 256 || static_cast<int64_t>(M) * N < 1500000 || weights > 1ll << 28) return false;
    if (weights >= 1ll << 26 && ceil_div(N, 256) * ceil_div(M, 64) <= 128) return false;
    if (weights <= 1ll << 26) return true;
    const int64_t rounds = ceil_div(ceil_div(N, 256) * ceil_div(M, 128), device_cu_count());
    return 0.95e-6 * static_cast<double>(weights) + row_tile_us(kRowF16, N, K, M) < 0.92 * round_us * (K / 1024.0) * static_cast<double>(rounds);
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

extern "C" int mfq_hip_row_tile_plan(int kind, int N, int K, int M, int *splits) {
    if (kind < mfq::kRowF16 || kind > mfq::kRowMx8F16 || N < 1 || K < 1 || M < 1) return -1;
    const mfq::TilePlan pl = mfq::row_plan(kind, N, K, M);
    if (splits) *splits = pl.splits;
    return pl.shape;
}
