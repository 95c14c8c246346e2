// Which tile shape and split over K a NINT prefill batch takes, its workspace and its launch (nint_tile.hpp).
#include "nint_tile.hpp"
#include "tune.hpp"

namespace mfq {

int x_frag(const void *x, int x_dtype, int64_t ldx, int M, int K, int GS, int nsteps, uint16_t *xf, float *xscale, uint16_t *xg,
           bool keep_bf16, hipStream_t st);
int prefill_sum_splits(const float *part, int64_t ystride, int splits, int M, int N, float *y, int64_t ldy, hipStream_t st);

#define MFQ_TILE_UNITS(X) X(4, 32) X(4, 24) X(4, 16) X(4, 48) X(3, 24) X(2, 16) X(2, 32) X(5, 28) X(6, 24) X(8, 48)
#define MFQ_TILE_DECL(B, G) int nint_tile_##B##_##G(const NintTileArgs &a, int shape, bool glu, int splits, hipStream_t st);
MFQ_TILE_UNITS(MFQ_TILE_DECL)
#undef MFQ_TILE_DECL

// Every profile with a unit: the paired layouts and NINT5-28 / NINT6-24 / NINT8-48.
bool nint_tile_capable(const mfq_nint_desc *d) {
    return (d->kind == 1 || (d->bits == 5 && d->gs == 28) || (d->bits == 6 && d->gs == 24) || (d->bits == 8 && d->gs == 48)) &&
           d->neuron_len >= 8 && 4 * d->rowblock_bytes < (1ll << 31);
}

// The tile and split over K with the smallest modelled time.  With nc = blocks per compute unit, rounded up, a launch takes
//     6.5 us + slices of K per split * (nc / 2 * u2 + nc % 2 * u1)  (+ 1.6 us + 0.33 us per MB of partial results)
// where u2 is the time of a slice in two blocks on one compute unit (side by side, or for the block of eight waves one after
// the other) and u1 that of one alone.  Those of the first five shapes were fitted over 12 batches (48 .. 2048 rows) x 7 tensors (1536 ..
// 24576 neurons, K 2048 .. 17408) of NINT4-32 with random codes (random data costs clock).  The sixth against
// the second, whole calls: 24576 x 4096 at 512 / 1024 / 2048 rows 110 / 179 / 334 us and 102 / 182 / 349, 12288 x 4096 at 601 rows 73 and 86,
// 4096 x 4096 at 2048 rows 76 and 89; by these constants, which leave out the launch that lays the activations out, 91 / 140 / 260 and
// 75 / 143 / 279, 55 and 75, 55 and 75.
// Weights that take longer to make than NINT's of two and four bits cost another tenth in 4 x 2 x 4, where a fragment serves fewest
// instructions, and NINT8-0's 1.4 times as much everywhere (without, 23 % at worst: 4096 x 4096 at 601 rows 65 us for 53).  For NINT the
// tenth does not hold from 65 to 192 rows, where the blocks of a launch are few and wait for memory more than for issue slots, and it
// only keeps calls off the best shape (with fewer rows it leaves them to the streaming kernel: NINT5-28 FFN 4096 / 12288 at 10 rows 59.7 us,
// without 61.6).  With it / without, us, at 100 rows NINT5-28 4096 x 4096 25.9 / 24.9; at 160 rows NINT5-28 FFN 5120 / 5120 90.6 / 79.0,
// NINT3-24 2560 x 8192 33.1 / 30.3, NINT6-24 there 35.4 / 31.9, NINT5-28 4096 x 12288 50.2 / 47.5, NINT8-48 there 46.3 / 43.6; against it,
// at 100 rows, NINT5-28 4096 x 12288 38.0 / 39.2, NINT8-48 12288 x 4096 36.1 / 36.7.  MX rows and fp16 copies have it at all sizes (at 100
// rows MXFP4 4096 x 12288 31.6 / 33.2; NVQ2J there at 200 rows 86.0 / 90.2, though 2560 x 8192 at 256 rows 45.5 / 43.5).
// The choice against the best of all shapes over 5 tensors (2560 .. 24576 neurons, K 4096 .. 12288) x 17 batches, on average and at
// worst, 48 to 192 / 200 to 333 / 400 to 2048 rows, %: NINT4-32 0.9, 10 / 0, 0 / 0.3, 4; NINT3-24 0.4, 4 / 1.2, 9 / 0.7, 8; NINT5-28 1.0, 6 /
// 2.1, 14 / 1.9, 19; NINT8-0 0.9, 6 / 1.9, 11 / 0.8, 7; MXFP4 1.0, 11 / 0.6, 5 / 0.5, 8; NVQ2J (fp16 copy) 1.6, 7 / 1.4, 8 / 0.5, 9.
// Pieces of K are not looked at from three tiles a compute unit on: by this model they would gain at most 1.4 %, in 51 of 8460 cases (1024
// .. 24576 neurons, K 2048 .. 17408, 128 .. 4096 rows), and the search is host time of every call.
TilePlan tile_plan(int rbs, int nsteps, int per_step, int rows, int out, int max_splits, int widest, TileWeight weight, bool halves) {
    const int M = static_cast<int>(ceil_div(rows, 64) * 64);  // one plan per 64 rows: the workspace then grows with the rows inside them
    static const int env_shape = tune_env("MFQ_TILE_SHAPE", 0), env_splits = tune_env("MFQ_PREFILL_SPLITS", 0);
    static const double u1[kTileShapes] = {0.351, 0.301, 0.219, 0.195, 0.138, 0.380}, u2[kTileShapes] = {0.774, 0.533, 0.378, 0.318, 0.213, 0.660};
    const bool slow_narrow = weight == kTileDecoded ? M <= 64 || M > 192 : weight != kTileLight;
    const int cu = device_cu_count();
    TilePlan best{2, 1, nsteps, 1e30};
    for (int shape = 0; shape < kTileShapes; ++shape) {
        const int mt = kTileShape[shape].mt, nb = kTileShape[shape].nb, nw = kTileShape[shape].nw;
        if (nb > widest) continue;
        if (env_shape > 0 && shape != env_shape - 1) continue;
        const int64_t tiles = ceil_div(rbs, (halves ? nw / 2 : nw) * nb) * ceil_div(M, 16 * mt);
        for (int sp = 1; sp == 1 || (sp <= max_splits && tiles < 3 * cu); ++sp) {
            if (env_splits > 0 && env_splits <= max_splits && sp != env_splits) continue;
            const int spz = static_cast<int>(ceil_div(nsteps, sp));
            if (ceil_div(nsteps, spz) != sp) continue;  // no empty split
            const int64_t nc = ceil_div(tiles * sp, cu);
            const double f = (weight == kTileHeavy ? 1.4 : 1.0) * (mt == 4 && nb == 2 && slow_narrow ? 1.1 : 1.0);
            const double t = 6.5 + spz * per_step * f * (static_cast<double>(nc / 2) * u2[shape] + static_cast<double>(nc % 2) * u1[shape]) +
                             (sp > 1 ? 1.6 + 0.33e-6 * sp * M * 4.0 * out : 0.0);
            if (t < best.us) best = TilePlan{shape, sp, spz, t};
        }
    }
    return best;
}
static TilePlan nint_tile_plan(const mfq_nint_desc *d, int rows, bool glu, int room = 8) {  // room: splits the workspace holds
    int max_splits = glu || d->out % 4 ? 1 : d->nsteps / 2 < 8 ? d->nsteps / 2 : 8;
    if (max_splits > room) max_splits = room;
    return tile_plan(glu ? d->n_rowblocks / 2 : d->n_rowblocks, d->nsteps, 4 * ((d->gs + 7) / 8), rows, d->out, max_splits, nint_tile_widest(d->bits, d->dwords), d->bits <= 4 && d->bits != 3 ? kTileLight : kTileDecoded, glu);
}

int nint_tile_shape(const mfq_nint_desc *d, int M, bool glu, int *splits) {
    const TilePlan pl = nint_tile_plan(d, M, glu);
    if (splits) *splits = pl.splits;
    return pl.shape;
}

static size_t tile_align(size_t v) { return (v + 255) & ~static_cast<size_t>(255); }
struct TileCarve { size_t xf, xscale, xg, part; };
static TileCarve nint_tile_carve(const mfq_nint_desc *d, int M) {
    const size_t mbs = static_cast<size_t>(ceil_div(M, 16));
    TileCarve c;
    c.xf = 0;
    c.xscale = c.xf + mbs * d->nsteps * 4 * static_cast<size_t>((d->gs + 7) / 8) * 1024;
    c.xg = c.xscale + tile_align(mbs * 64);
    c.part = c.xg + mbs * d->nsteps * 1024;
    return c;
}
// What a call makes use of: the activations, and the partial results of its split over K (a call with the GLU has none).
size_t nint_tile_workspace(const mfq_nint_desc *d, int M) {
    const int splits = nint_tile_plan(d, M, false).splits;
    return nint_tile_carve(d, M).part + (splits > 1 ? static_cast<size_t>(splits) * M * d->out * 4 : 0);
}
// What a call cannot do without.  It grows with the rows, which the other does not: a split belongs to small batches.
size_t nint_tile_workspace_least(const mfq_nint_desc *d, int M) { return nint_tile_carve(d, M).part; }

// Modelled time of a plain call, the activations included: 5 us up to a few hundred rows, and two launches for long rows.
double nint_tile_us(const mfq_nint_desc *d, int M) { return nint_tile_plan(d, M, false).us + (d->neuron_len > 6144 ? 9.0 : 5.0); }

// Fused act(gate) * up: whole row-blocks of both halves, and either no slower than the plain call, which may split K (2 us: part
// of what its elementwise kernel costs), or a batch of 512 rows and more whose 64 x 256 tiles fill half the chip: those callers
// always had the fused form (NINT4-32 4096 x 8192 at 600 rows 78 us, two launches 76; NINT3-24 5120 x 8192 at 512 rows 87, 79).
bool nint_tile_glu_pays(const mfq_nint_desc *d, int M) {
    if (!nint_tile_capable(d) || d->out % 32 != 0) return false;
    if (M >= 512 && ceil_div(d->n_rowblocks, 16) * ceil_div(M, 64) > 128) return true;
    return nint_tile_plan(d, M, true).us <= nint_tile_plan(d, M, false).us + 2.0;
}

// y (float [M, ldy], or with glu uint16_t [M, ldy]) of M activation rows; ws_bytes of at least nint_tile_workspace_least(d, M):
// with less than nint_tile_workspace(d, M) it splits K into fewer pieces
int nint_tile(const mfq_nint_desc *d, const void *weight, const void *x, int x_dtype, int64_t ldx, int M, void *y, int64_t ldy,
              bool glu, int gelu, int f16, void *ws, size_t ws_bytes, hipStream_t st) {
    const TileCarve c = nint_tile_carve(d, M);
    const TilePlan pl = nint_tile_plan(d, M, glu, splits_that_fit(ws_bytes, c.part, M, d->out));
    uint8_t *base = static_cast<uint8_t *>(ws);
    uint16_t *xf = reinterpret_cast<uint16_t *>(base + c.xf), *xg = reinterpret_cast<uint16_t *>(base + c.xg);
    float *xscale = reinterpret_cast<float *>(base + c.xscale), *part = reinterpret_cast<float *>(base + c.part);
    if (int rc = x_frag(x, x_dtype, ldx, M, d->neuron_len, d->gs, d->nsteps, xf, xscale, xg, false, st)) return rc;
    const bool split = pl.splits > 1;
    const NintTileArgs a{to_k(d), static_cast<const uint8_t *>(weight), xf, xg, xscale, split ? part : y, split ? d->out : ldy,
                         static_cast<int64_t>(M) * d->out, M, pl.spz, d->n_rowblocks / 2, gelu, f16};
    int rc = MFQ_ERR_UNSUPPORTED;
#define MFQ_TILE_CASE(B, G) if (d->bits == B && d->gs == G) rc = nint_tile_##B##_##G(a, pl.shape, glu, pl.splits, st);
    MFQ_TILE_UNITS(MFQ_TILE_CASE)
#undef MFQ_TILE_CASE
    if (rc) return rc == MFQ_ERR_UNSUPPORTED ? fail(rc, "nint_tile: no kernel for NINT%d-%d", d->bits, d->gs) : rc;
    return split ? prefill_sum_splits(part, a.zstride, pl.splits, M, d->out, static_cast<float *>(y), ldy, st) : MFQ_OK;
}

}  // namespace mfq
