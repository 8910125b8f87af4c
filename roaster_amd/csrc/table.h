/*
 * table.h -- internal layout of the HBM expert table (table.hip).
 */
#ifndef ROASTER_TABLE_H
#define ROASTER_TABLE_H

#include <vector>
#include "decode.h"

/* Device addresses of one layer's matrices in the MFMA tile layout (tile.h). */
struct TileLayer {
    const uint8_t *gate, *up, *down;      /* [E] consecutive matrices */
    const uint8_t *sgate, *sup, *sdown;
    /* the router as the prefill router's MFMA operand: [E / 32, rounded up][H /
     * 32][4][64 lanes][4]: load q of K chunk c gives lane n + 32 h columns 32 c
     * + 8 q + 4 h .. + 3 of expert 32 b + n (zero past E); NULL past 256 experts,
     * which prefill refuses.  A load of a wave is a
     * contiguous kilobyte; the row-major router's 32 rows, H floats apart,
     * measured 9.6 us in place of 8.5 at 45 tokens and 35.6 in place of 30.7
     * at 2048 (E 256, H 2048). */
    const float *router;
};

/* Types, sizes and offsets of one layer's matrices (types may differ by layer). */
struct LayerGeo {
    int q6[3], sh_q6[3];                  /* 0 = Q4_K, 1 = Q6_K */
    size_t eb[3], sb[3];                  /* GGML bytes: one routed expert's matrix / the shared one's */
    size_t off_exps[3], off_sh[3];        /* offsets inside the layer's GGML region */
    size_t teb[3], tsb[3];                /* the same in the tile layout */
    size_t toff_exps[3], toff_sh[3];
    size_t base, tbase;                   /* the layer's offsets in qmem / tmem */
};

struct RoasterTable {
    RoasterTableDesc d;
    std::vector<LayerGeo> geo;
    size_t qbytes, tbytes, fbytes;
    uint8_t *qmem = nullptr; /* quantised matrices (GGML layout), all layers */
    uint8_t *tmem = nullptr; /* the same matrices in the MFMA tile layout (prefill GEMM operands) */
    float *fmem = nullptr;   /* routers and gate vectors, then the routers' operand copies */
    std::vector<DecLayer> layers_h;
    DecLayer *layers_d = nullptr;
    std::vector<TileLayer> tlayers_h;
    float *dbound = nullptr; /* [n_layers][E + 1]: bound on the L1 norm of any row of each down matrix */
};

#endif
