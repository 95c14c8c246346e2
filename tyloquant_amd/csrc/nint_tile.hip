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
// the other) and u1 that of one alone.  Fitted over 5 shapes x 12 batches (48 .. 2048 rows) x 7 tensors (1536 .. 24576
// neurons, K 2048 .. 17408) of NINT4-32 with random codes (random data costs clock); the choice is within 1 % of the best on
// average and 10 % at worst there, for NINT3-24 and NINT2-16 too, whose slices cost 5 to 15 % more in all shapes alike.
// Weights that take longer to make than NINT's of two and four bits cost another tenth in 4 x 2 x 4, where a fragment serves fewest
// instructions, and NINT8-0's 1.4 times as much everywhere: over 5 tensors x 7 batches (200 .. 2048 rows) the choice is 0.3 to 1.3 %
// behind the best by format; without, 2.9 % for NINT8-0 and 23 % at worst (4096 x 4096 at 601 rows 65 us for 53).
TilePlan tile_plan(int rbs, int nsteps, int per_step, int rows, int out, int max_splits, int widest, TileWeight weight, bool halves) {
    const int M = static_cast<int>(ceil_div(rows, 64) * 64);  // one plan per 64 rows: the workspace then grows with the rows inside them
    static const int env_shape = tune_env("MFQ_TILE_SHAPE", 0), env_splits = tune_env("MFQ_PREFILL_SPLITS", 0);
    static const double u1[kTileShapes] = {0.351, 0.301, 0.219, 0.195, 0.138, 0.380}, u2[kTileShapes] = {0.774, 0.533, 0.378, 0.318, 0.213, 0.660};
    const int cu = device_cu_count();
    TilePlan best{2, 1, nsteps, 1e30};
    for (int shape = 0; shape < kTileShapes; ++shape) {
        const int mt = kTileShape[shape].mt, nb = kTileShape[shape].nb, nw = kTileShape[shape].nw;
        if (nb > widest) continue;
        if (env_shape > 0 && shape != env_shape - 1) continue;
        const int64_t tiles = ceil_div(rbs, (halves ? nw / 2 : nw) * nb) * ceil_div(M, 16 * mt);
        for (int sp = 1; sp == 1 || (sp <= max_splits && tiles < 3 * cu); ++sp) {  // (a full chip needs no pieces)
            if (env_splits > 0 && env_splits <= max_splits && sp != env_splits) continue;
            const int spz = static_cast<int>(ceil_div(nsteps, sp));
            if (ceil_div(nsteps, spz) != sp) continue;  // no empty split
            const int64_t nc = ceil_div(tiles * sp, cu);
            const double f = (weight == kTileHeavy ? 1.4 : 1.0) * (mt == 4 && nb == 2 && weight != kTileLight ? 1.1 : 1.0);
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
