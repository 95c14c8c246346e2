// Kernel of mapped MoE calls (moe_prefill.hpp); compiled side by side for its two outputs.
#pragma once
#include "moe_prefill.hpp"
#include "nint_tile.hpp"

namespace mfq {

template <class U, int MT, bool GLU>
__device__ __forceinline__ void moe_tile_run(const NintK &k, const uint8_t *w, const GatherRows &rows, const TileOut &out, int tn, uint8_t *lds) {
    typedef NintTileB<U, moe_nb(MT, U::D), moe_sl(MT), moe_sets(MT, U::D), moe_fused(MT), moe_short(MT, U::D)> B;
    nint_tile_body<B, 4, MT, kMoeRing, GLU>(k, w, rows, out, tn, 0, k.nsteps, lds);
}

template <class U, int MT, bool GLU>
__device__ __forceinline__ void moe_tile_run_few(const NintK &k, const uint8_t *w, const GatherRows &rows, const TileOut &out, int tn, uint8_t *lds) {
    typedef NintTileB<U, kMoeFewNb, moe_sl(MT), moe_few_sets(MT, U::D), moe_fused(MT)> B;
    nint_tile_body<B, 4, MT, kMoeRing, GLU>(k, w, rows, out, tn, 0, k.nsteps, lds);
}

// Block b: XCD b % 8 (blocks go to the XCDs in turn) takes chunk (b / 8 / ncol) * 8 + b % 8, neuron tile (b / 8) % ncol -- the
// blocks that share a chunk's activation rows run next to each other on one XCD and find them in its L2.  Chunks of a tile or two have
// few rows to share and few chunks to spread: there the tiles of a chunk go to all XCDs (66 chunks, 9 on two of the XCDs and 8 on the
// others: 61 tokens, 8 of 64 experts and a shared one 252 us by chunk, 250 spread).
template <bool GLU, class Run>
__device__ __forceinline__ void moe_tile_block(const MoeTileArgs &p, uint8_t *lds, bool few, Run run) {
    const int b = blockIdx.x, j = b >> 3, item = few ? b / p.ncol : (j / p.ncol) * 8 + (b & 7), tn = few ? b % p.ncol : j % p.ncol;
    if (item >= p.lists[0]) return;
    const int lo = p.lists[4 + 4 * item], hi = p.lists[5 + 4 * item], pool = p.lists[6 + 4 * item], local = p.lists[7 + 4 * item];
    const int tiles = (hi - lo + 15) >> 4, rbe = p.out_per_expert >> 4, rbs = GLU ? rbe >> 1 : rbe;
    const NintK &k = p.k[pool];
    if (tn * (GLU ? 2 : 4) * (few ? kMoeFewNb : moe_nb(tiles, k.dwords)) >= rbs) return;  // small chunks take more neurons per block
    int *srcv = reinterpret_cast<int *>(lds);
    const bool own = lo >= p.n_pairs;  // a chunk of the shared tensor: tokens in order
    const GatherRows rows{p.xr[pool], p.xg[pool], p.xscale + p.row0, own ? nullptr : p.ids_dst + lo, hi - lo, p.routed || own ? 1 : p.R,
                          p.row0 + (own && !p.routed ? p.n_pairs : 0), p.n_rows, srcv, srcv + 16 * kMoeTiles,
                          reinterpret_cast<float *>(srcv + 32 * kMoeTiles), 16 * kMoeTiles, lo};
    const TileOut out{local * rbe, rbs, rbs * 16, p.out, p.ldo, p.gelu, p.f16};
    run(k, p.w[pool], rows, out, tn, tiles);
}
#define MFQ_MOE_UNITS(MANY, FEW)                                                                                       \
    if (k.kind == 1) {                                                                                                 \
        MANY(PairedUnit, 4, 24)                                                                                        \
        else MANY(PairedUnit, 3, 24)                                                                                   \
        else MANY(PairedUnit, 2, 16)                                                                                   \
        else MANY(PairedUnit, 4, 32)                                                                                   \
        else FEW(PairedUnit, 4, 16)                                                                                    \
        else FEW(PairedUnit, 4, 48)                                                                                    \
        else FEW(PairedUnit, 2, 32)                                                                                    \
    } else {                                                                                                           \
        MANY(GenericUnit, 5, 28)                                                                                       \
    }
template <bool GLU>
__global__ __launch_bounds__(256, 2) void moe_tile_kernel(MoeTileArgs p) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t moe_lds[];
    moe_tile_block<GLU>(p, moe_lds, false, [&](const NintK &k, const uint8_t *w, const GatherRows &rows, const TileOut &out, int tn, int tiles) __attribute__((always_inline)) {
    // Bodies by row tiles; sizes without one of their own run the next larger (of the profiles that mixed files of experts are not
    // written in, for the sake of the build, more of them).
#define MFQ_MOE_MT(MT, UNIT, B, G) moe_tile_run<UNIT<B, G>, MT, GLU>(k, w, rows, out, tn, moe_lds + kMoeTableBytes); break;
#define MFQ_MOE_UNIT(UNIT, B, G)                                                                                       \
    if (k.bits == B && k.gs == G) {                                                                                    \
        switch (tiles) {                                                                                               \
            case 1: MFQ_MOE_MT(1, UNIT, B, G)                                                                          \
            case 2: MFQ_MOE_MT(2, UNIT, B, G)                                                                          \
            case 3: MFQ_MOE_MT(3, UNIT, B, G)                                                                          \
            case 4: MFQ_MOE_MT(4, UNIT, B, G)                                                                          \
            case 5: case 6: MFQ_MOE_MT(6, UNIT, B, G)                                                                  \
            case 7: case 8: MFQ_MOE_MT(8, UNIT, B, G)                                                                  \
            case 9: MFQ_MOE_MT(9, UNIT, B, G)                                                                          \
        }                                                                                                              \
    }
#define MFQ_MOE_UNIT_FEW(UNIT, B, G)                                                                                   \
    if (k.bits == B && k.gs == G) {                                                                                    \
        switch (tiles) {                                                                                               \
            case 1: case 2: MFQ_MOE_MT(2, UNIT, B, G)                                                                  \
            case 3: case 4: MFQ_MOE_MT(4, UNIT, B, G)                                                                  \
            case 5: case 6: MFQ_MOE_MT(6, UNIT, B, G)                                                                  \
            case 7: case 8: case 9: MFQ_MOE_MT(9, UNIT, B, G)                                                          \
        }                                                                                                              \
    }
        MFQ_MOE_UNITS(MFQ_MOE_UNIT, MFQ_MOE_UNIT_FEW)
    });
#undef MFQ_MOE_UNIT
#undef MFQ_MOE_UNIT_FEW
#undef MFQ_MOE_MT
}

// Chunks of one or two row tiles (kMoeFewTiles).
template <bool GLU>
__global__ __launch_bounds__(256, 4) void moe_tile_few_kernel(MoeTileArgs p) {
    extern __shared__ __attribute__((aligned(1024))) uint8_t moe_lds[];
    moe_tile_block<GLU>(p, moe_lds, true, [&](const NintK &k, const uint8_t *w, const GatherRows &rows, const TileOut &out, int tn, int tiles) __attribute__((always_inline)) {
#define MFQ_MOE_UNIT(UNIT, B, G)                                                                                       \
    if (k.bits == B && k.gs == G) {                                                                                    \
        if (tiles <= 1) moe_tile_run_few<UNIT<B, G>, 1, GLU>(k, w, rows, out, tn, moe_lds + kMoeTableBytes);           \
        else moe_tile_run_few<UNIT<B, G>, 2, GLU>(k, w, rows, out, tn, moe_lds + kMoeTableBytes);                      \
    }
        MFQ_MOE_UNITS(MFQ_MOE_UNIT, MFQ_MOE_UNIT)
#undef MFQ_MOE_UNIT
    });
}

template <bool GLU>
static int moe_tile_start(const MoeTileArgs &t, unsigned grid, hipStream_t st) {
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void *>(&moe_tile_kernel<GLU>), kMoeTileLds, "moe_tile")) return rc;
    hipLaunchKernelGGL(moe_tile_kernel<GLU>, dim3(grid), dim3(256), kMoeTileLds, st, t);
    return check_launch("moe_tile");
}
template <bool GLU>
static int moe_tile_few_start(const MoeTileArgs &t, unsigned grid, hipStream_t st) {
    hipLaunchKernelGGL(moe_tile_few_kernel<GLU>, dim3(grid), dim3(256), kMoeFewLds, st, t);
    return check_launch("moe_tile_few");
}

}  // namespace mfq
