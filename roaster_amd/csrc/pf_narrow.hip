/*
 * pf_narrow.hip -- grouped expert GEMMs of the prefill path on 32-row tiles
 * with exact integer weights.
 *
 * A wave owns 32 weight rows (gate/up: 16 gate rows and the 16 up rows of the
 * same columns) and reads each lane's half super-block straight from the MFMA
 * tile layout (tile.h) into registers.  The MFMA operand is the block's integer
 * part, which fp16 holds exactly -- Q4_K: sc q (at most 945); Q6_K: sc (q - 32)
 * (up to 4096, exact up to 2048 and rounded to 11 bits above, with the
 * remainder as a second operand in split mode) -- and the super-block's d is
 * applied in f32 to the 32 x 32 sums of its sixteen k-slices.  Q4_K's minimum
 * term, sum over sub-blocks of m_s (sum of x over s), is one more MFMA per
 * super-block: its operands are the eight 6-bit m_s and the eight sub-block
 * sums of the row (fp16 hi + lo, scaled by 2^-6), prepared with the rows.
 * (kernels.c:1844-1874: d sc q - dmin m and d sc (q - 32).)
 *
 * Activations are fp16, scaled per row by a power of two.  PF_F16 tiles have up
 * to 32 rows.  PF_SPLIT tiles have up to 16: operand row r holds the fp16 hi
 * part of tile row r and operand row 16 + r its lo part (22 bits together), so
 * one MFMA per slice forms both products and a lane adds its accumulators i
 * and i + 8.  Against the bf16 hi + lo operands of gemm.h, which serve
 * PF_SPLIT where this file does not, the weights lose nothing and the
 * activations 6 bits less, down to about 2^-22 of their row's largest; below that
 * an element's error stays at 2^-39 of the largest, where bf16 hi + lo has 2^-17 of
 * the element.  Against 64 bits, N(0, 1) activations, 256 tokens of a layer: 7.2e-6
 * -> 3.0e-7.
 */
#include <type_traits>

#include "internal.h"
#include "gemm.h"
#include "prefill.h"
#include "pf_tile.h"

#define NW_ROWS 32                /* operand rows */
#define NW_SUM GK                 /* a staged row: 256 activations, 16 sub-block sums, padding */
#define NW_LD (GK + 16 + 8)       /* fp16 row pitch: 35 16-byte granules, so the 32 rows of an operand
                                     read start in different bank groups */
#define NW_BUF (NW_ROWS * NW_LD)  /* fp16 elements of one staged super-block */

/* Tile rows and accumulators per lane. */
template <bool SPLIT> struct NwTile { static constexpr int ROWS = SPLIT ? 16 : 32, ACC = ROWS / 2; };
template <int N> struct NwAcc { float v[N]; };

/* Loads at a uniform base plus a 32-bit lane offset (one address register). */
__device__ __forceinline__ uint4 gld_u4o(const void *base, uint32_t off)
{
    const gu32x4 v = *(const GAS gu32x4 *)((const GAS uint8_t *)base + off);
    return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ void nw_load(RawQ6 &r, const uint8_t *base, uint32_t off)
{
    uint4 s[7];
#pragma unroll
    for (int i = 0; i < 7; i++) s[i] = gld_u4o(base + 1024 * i, off);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        r.L[4 * i] = s[i].x; r.L[4 * i + 1] = s[i].y; r.L[4 * i + 2] = s[i].z; r.L[4 * i + 3] = s[i].w;
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        r.Hh[4 * i] = s[4 + i].x; r.Hh[4 * i + 1] = s[4 + i].y; r.Hh[4 * i + 2] = s[4 + i].z; r.Hh[4 * i + 3] = s[4 + i].w;
    }
    r.S[0] = s[6].x;
    r.S[1] = s[6].y;
    r.d = s[6].z;                     /* d in the low 16 bits, the rest is 0 */
}

__device__ __forceinline__ void nw_load(RawQ4 &r, const uint8_t *base, uint32_t off)
{
    uint4 s[5];
#pragma unroll
    for (int i = 0; i < 5; i++) s[i] = gld_u4o(base + 1024 * i, off);
    r.hd[0] = s[0].x; r.hd[1] = s[0].y; r.hd[2] = s[0].z; r.hd[3] = s[0].w;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        r.Q[4 * i] = s[1 + i].x; r.Q[4 * i + 1] = s[1 + i].y; r.Q[4 * i + 2] = s[1 + i].z; r.Q[4 * i + 3] = s[1 + i].w;
    }
}

/* ---- one super-block: acc += d (integer weights . x) [- dmin (m . sums)] ---- */
__device__ __forceinline__ f16x2 splat2(int v) { const _Float16 f = (_Float16)v; return (f16x2){ f, f }; }

template <bool SPLIT>
struct NwQ4 {
    f16x2 sc[4], bias[4];
    __device__ __forceinline__ NwQ4(const RawQ4 &r, int h)
    {
        const uint32_t s03 = r.hd[1], s811 = r.hd[3];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const uint32_t lo = byte_of(s03, i) & 63, hi = (byte_of(s811, i) & 15) | ((byte_of(s03, i) >> 6) << 4);
            const int v = (int)(h ? hi : lo);
            sc[i] = splat2(v);
            bias[i] = splat2(-1024 * v);             /* exact: 63 * 1024 < 65504 */
        }
    }
    /* the operand of k-slice j + 8 u; exact, so there is no remainder */
    __device__ __forceinline__ void slice8(const RawQ4 &r, int j, int u, f16x8 &b, f16x8 &) const
    {
        b = slice(r.Q[8 * u + j], 2 * u);
    }
    __device__ __forceinline__ f16x8 slice(uint32_t q, int s) const
    {
        const uint32_t lo = q & 0x0F0F0F0Fu, hi = (q >> 4) & 0x0F0F0F0Fu;
        const f16x2 a = __builtin_elementwise_fma(magic_lo(lo), sc[s], bias[s]);
        const f16x2 b = __builtin_elementwise_fma(magic_hi(lo), sc[s], bias[s]);
        const f16x2 c = __builtin_elementwise_fma(magic_lo(hi), sc[s + 1], bias[s + 1]);
        const f16x2 d = __builtin_elementwise_fma(magic_hi(hi), sc[s + 1], bias[s + 1]);
        return (f16x8){ a[0], a[1], b[0], b[1], c[0], c[1], d[0], d[1] };
    }
};

template <bool SPLIT>
struct NwQ6 {
    f16x2 sc[8];
    __device__ __forceinline__ NwQ6(const RawQ6 &r, int)
    {
#pragma unroll
        for (int s = 0; s < 8; s++) sc[s] = splat2((int)(int8_t)((r.S[s >> 2] >> (8 * (s & 3))) & 0xFFu));
    }
    __device__ __forceinline__ void quad(uint32_t q, int s, f16x2 &h0, f16x2 &h1, f16x2 &l0, f16x2 &l1) const
    {
        const f16x2 off = { (_Float16)-1056.0f, (_Float16)-1056.0f };
        const f16x2 u = magic_lo(q) + off, v = magic_hi(q) + off;        /* q - 32, exact */
        h0 = u * sc[s];
        h1 = v * sc[s];
        if (SPLIT) {
            l0 = __builtin_elementwise_fma(u, sc[s], -h0);               /* what the product rounded off: 0 or +-1 */
            l1 = __builtin_elementwise_fma(v, sc[s], -h1);
        }
    }
    __device__ __forceinline__ void slice8(const RawQ6 &r, int j, int u, f16x8 &b, f16x8 &e) const
    {
        const uint32_t A = r.L[j], B = r.L[8 + j], C = r.Hh[j];
        const uint32_t qa = u ? ((A >> 4) & 0x0F0F0F0Fu) | (C & 0x30303030u) : (A & 0x0F0F0F0Fu) | ((C << 4) & 0x30303030u);
        const uint32_t qb = u ? ((B >> 4) & 0x0F0F0F0Fu) | ((C >> 2) & 0x30303030u)
                              : (B & 0x0F0F0F0Fu) | ((C << 2) & 0x30303030u);
        const int s = (j >> 2) + 4 * u;
        f16x2 h[4], l[4];
        quad(qa, s, h[0], h[1], l[0], l[1]);
        quad(qb, s + 2, h[2], h[3], l[2], l[3]);
        b = (f16x8){ h[0][0], h[0][1], h[1][0], h[1][1], h[2][0], h[2][1], h[3][0], h[3][1] };
        if (SPLIT) e = (f16x8){ l[0][0], l[0][1], l[1][0], l[1][1], l[2][0], l[2][1], l[3][0], l[3][1] };
    }
};

template <bool Q6, bool SPLIT> struct NwOf;
template <bool SPLIT> struct NwOf<true, SPLIT> { typedef NwQ6<SPLIT> T; };
template <bool SPLIT> struct NwOf<false, SPLIT> { typedef NwQ4<SPLIT> T; };

__device__ __forceinline__ float nw_d(const RawQ6 &r) { return f16_bits_to_f32(r.d); }
__device__ __forceinline__ float nw_d(const RawQ4 &r) { return f16_bits_to_f32(r.hd[0] & 0xFFFFu); }

template <int N>
__device__ __forceinline__ void nw_min(NwAcc<N> &, const RawQ6 &, const _Float16 *) {}
template <int N>
__device__ __forceinline__ void nw_min(NwAcc<N> &acc, const RawQ4 &r, const _Float16 *xs)
{
    const uint32_t s47 = r.hd[2], s811 = r.hd[3];
    f16x8 m;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        m[i] = (_Float16)(int)(byte_of(s47, i) & 63);
        m[4 + i] = (_Float16)(int)((byte_of(s811, i) >> 4) | ((byte_of(s47, i) >> 6) << 4));
    }
    const f16x8 x = *(const f16x8 *)xs;
    const f32x16 z = __builtin_amdgcn_mfma_f32_32x32x16_f16(x, m, (f32x16){}, 0, 0, 0);
    const float dm = f16_bits_to_f32(r.hd[0] >> 16) * -64.0f;            /* the sums carry 2^-6 */
#pragma unroll
    for (int i = 0; i < N; i++) {
        acc.v[i] = fmaf(dm, z[i], acc.v[i]);                             /* (operand rows 16.. of a split tile: unused) */
        asm volatile("" : "+v"(acc.v[i]));                               /* done here: z is not kept over the slices */
    }
}

template <bool Q6, bool SPLIT, int N>
__device__ __forceinline__ void nw_block(NwAcc<N> &acc, const _Float16 *Xs, const typename RawOf<Q6>::T &r, int l)
{
    const int h = l >> 5, n = l & 31;
    const _Float16 *xa = Xs + n * NW_LD + 8 * h;
    nw_min(acc, r, xa + NW_SUM);
    __builtin_amdgcn_sched_barrier(0);
    const typename NwOf<Q6, SPLIT>::T c(r, h);
    f32x16 z = {};
#pragma unroll
    for (int j = 0; j < 16; j++) {
        /* slices 0, 8, 1, 9, ...: Q6_K slices j and j + 8 share their dwords */
        const int k = (j >> 1) + 8 * (j & 1);
        f16x8 b, e;
        c.slice8(r, j >> 1, j & 1, b, e);
        const f16x8 x = *(const f16x8 *)(xa + 16 * k);
        z = __builtin_amdgcn_mfma_f32_32x32x16_f16(x, b, z, 0, 0, 0);
        if (SPLIT && Q6) z = __builtin_amdgcn_mfma_f32_32x32x16_f16(x, e, z, 0, 0, 0);
        if (j & 1) __builtin_amdgcn_sched_barrier(0);
    }
    const float d = nw_d(r);
#pragma unroll
    for (int i = 0; i < N; i++) acc.v[i] = fmaf(d, SPLIT ? z[i] + z[(i + 8) & 15] : z[i], acc.v[i]);
}

/* ---- gate/up -----------------------------------------------------------------
 * Bound by the weights' bytes: short prompts touch nearly every expert with a
 * few rows each.  Four waves (64 columns) per workgroup and three workgroups
 * per CU (168 registers, 36 KB of LDS) keep 60-84 KB of weights in flight per
 * CU, each super-block's loads issued a whole step ahead, and one workgroup's
 * barriers, prologue and epilogue run under the others' loads; 45 tokens make
 * 1,568 workgroups of even size where one workgroup per CU over 128-column
 * units left a fourth round for a quarter of the CUs.  Q4_K, 256 experts,
 * hidden 2048, inter 512, kernel trace: 45 tokens 100 -> 54 us (257 MB of
 * weights: 4.8 TB/s, the rate of a large copy), 512 skewed tokens 133 -> 86.
 * Split mode (16-row tiles), 256 tokens: gate/up 671 -> 75 us against the
 * 64 x 64 tiles of gemm.h; 32-row tiles with separate hi and lo products took
 * 100 us (twice the MFMAs and staging registers, two waves per SIMD). */
struct NwMeta {
    int tok[NW_ROWS];
    float fwd[NW_ROWS];
};

#define NWG_W 4                   /* waves per gate/up workgroup */

template <bool Q6, bool SPLIT>
__device__ __forceinline__ void nw_gu_body(const PfGemmArgs &A, const PfGroup &G, NwMeta &meta, int m0, int mlen, int j0,
                                           _Float16 *Xb)
{
    constexpr int NT = 64 * NWG_W, RPP = NT / 32, NP = NW_ROWS / RPP;      /* operand rows per staging round, rounds */
    constexpr int ROWS = NwTile<SPLIT>::ROWS, NA = NwTile<SPLIT>::ACC, TB = TL_BYTES(Q6);
    const int t = threadIdx.x, l = t & 63, h = l >> 5, w = t >> 6, n = l & 31;
    const int nkb = A.H / GK;
    const bool up = n >= 16;
    const int jrow = j0 + 16 * w + (n & 15);
    /* both matrices from the lower one's address (a table's tile layout keeps
     * a layer's gate and up regions within 4 GiB) */
    const uint8_t *wb = G.tg < G.tu ? G.tg : G.tu;
    const uint32_t wo = (uint32_t)((up ? G.tu : G.tg) - wb) + (uint32_t)(jrow / TL_ROWS) * nkb * TB +
                        16u * ((jrow & (TL_ROWS - 1)) + 32 * h);
    /* the rows' tokens first (a wave's loads return in order), then the first
     * super-block's weights, which stay in flight over the barrier */
    int tok = 0;
    if (t < NW_ROWS) {
        const int r = m0 + min(t, mlen - 1);
        tok = G.tok ? G.tok[r] : G.tok0 + r;
    }
    typename RawOf<Q6>::T r[2];
    nw_load(r[0], wb, wo);
    if (t < NW_ROWS) meta.tok[t] = tok;
    lds_barrier();
    /* staging: piece i of a thread is 16 bytes of operand row t / 32 + i RPP,
     * tile row (that) % ROWS; rounds past the tile's last row are skipped, rows
     * past it repeat it */
    const int xrow = t >> 5;
    uint32_t xo[NP];
#pragma unroll
    for (int i = 0; i < NP; i++)
        xo[i] = 2u * ((uint32_t)meta.tok[(xrow + i * RPP) % ROWS] * (uint32_t)A.H + 8u * (t & 31));
    const uint32_t so = 32u * (uint32_t)meta.tok[(t >> 1) % ROWS] * (uint32_t)nkb + 16u * (t & 1);
    const uint8_t *x16 = (const uint8_t *)A.X16, *x16l = (const uint8_t *)A.X16l, *xs16 = (const uint8_t *)A.xs16;
    uint4 xr[NP], sr;
    auto x_load = [&](int kb) {
#pragma unroll
        for (int i = 0; i < NP; i++)
            if (i * RPP % ROWS < mlen) xr[i] = gld_u4o((i * RPP < ROWS ? x16 : x16l) + 2 * GK * kb, xo[i]);
        if (!Q6) sr = gld_u4o(xs16 + 32 * kb, so);
    };
    auto x_store = [&](int buf) {
        _Float16 *dst = Xb + buf * NW_BUF;
#pragma unroll
        for (int i = 0; i < NP; i++)
            if (i * RPP % ROWS < mlen) *(uint4 *)(dst + (xrow + i * RPP) * NW_LD + 8 * (t & 31)) = xr[i];
        if (!Q6 && t < 2 * ROWS) *(uint4 *)(dst + (t >> 1) * NW_LD + NW_SUM + 8 * (t & 1)) = sr;
    };
    x_load(0);
    if (t < NW_ROWS) meta.fwd[t] = A.xfwd[tok];                          /* read in the epilogue */
    x_store(0);
    lds_barrier();
    NwAcc<NA> acc = {};
    /* super-block kb with kb + 1's loads issued ahead of it: activations (from
     * L2) before weights, so that the staging store waits for the former only */
    auto step = [&](auto bc, int kb) {
        constexpr int buf = decltype(bc)::value;
        x_load(kb + 1);
        nw_load(r[buf ^ 1], wb + (size_t)(kb + 1) * TB, wo);
        __builtin_amdgcn_sched_barrier(0);
        nw_block<Q6, SPLIT>(acc, Xb + buf * NW_BUF, r[buf], l);
        __builtin_amdgcn_sched_barrier(0);
        x_store(buf ^ 1);
        lds_barrier();
    };
    using B0 = std::integral_constant<int, 0>;
    using B1 = std::integral_constant<int, 1>;
    int kb = 0;
    for (; kb + 2 < nkb; kb += 2) {
        step(B0(), kb);
        step(B1(), kb + 1);
    }
    if (kb + 1 < nkb) {
        step(B0(), kb);
        nw_block<Q6, SPLIT>(acc, Xb + NW_BUF, r[1], l);
    } else {
        nw_block<Q6, SPLIT>(acc, Xb, r[0], l);
    }
    /* epilogue: lane n < 16 holds gate and lane n + 16 up of column j0 + 16 w +
     * (n & 15).  One lane swap per row pair (i, i + 1) gives lanes n < 16 both
     * values of row i and lanes n >= 16 both of row i + 1.  The 16-lane maximum
     * of |act| is the row's part maximum; fp16 mode stores act scaled by its
     * power of two, split mode stores it in f32. */
    const int npart = A.I / 16, part = (j0 >> 4) + w;
#pragma unroll
    for (int i = 0; i < NA; i += 2) {
        if (8 * (i >> 2) >= mlen) continue;                              /* wave-uniform */
        const float v0 = acc.v[i], v1 = acc.v[i + 1];
        const float mine = up ? v1 : v0, other = up ? v0 : v1;
        const auto sw = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, other),
                                                         __builtin_bit_cast(uint32_t, other), false, false);
        const float got = __builtin_bit_cast(float, (uint32_t)(up ? sw[0] : sw[1]));
        const int m = 8 * (i >> 2) + 4 * h + (i & 3) + (up ? 1 : 0);
        const float f = meta.fwd[m];
        const float g = (up ? got : mine) * f, u = (up ? mine : got) * f;
        const float e = SPLIT ? pf_silu_mul(g, u) : pf_silu_mul_fast(g, u);
        uint32_t mb = __builtin_bit_cast(uint32_t, e) & 0x7FFFFFFFu;
        mb = max(mb, (uint32_t)dpp_i<DPP_XOR1>((int)mb));
        mb = max(mb, (uint32_t)dpp_i<DPP_XOR2>((int)mb));
        mb = max(mb, (uint32_t)dpp_i<DPP_HALF_MIRROR>((int)mb));
        mb = max(mb, (uint32_t)dpp_i<DPP_MIRROR>((int)mb));
        const float mx = __builtin_bit_cast(float, mb);
        if (m < mlen) {
            const size_t slot = (size_t)(G.slot0 + m0 + m);
            if (SPLIT) {
                A.act[slot * A.I + jrow] = e;
            } else {
                float pinv, pfwd;
                row_scale(mx, pinv, pfwd);
                const _Float16 v = (_Float16)(e * pinv);
                A.act16[slot * A.I + jrow] = __builtin_bit_cast(uint16_t, v);
            }
            if ((n & 15) == 0) A.pmax[slot * npart + part] = mx;
        }
    }
}

template <bool SPLIT>
__global__ void __launch_bounds__(64 * NWG_W, 3) pfn_gu_kernel(PfGemmArgs A)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t nw_lds[];
    __shared__ NwMeta meta;
    const int nblk = A.I / (16 * NWG_W), R = *A.gu_ntiles * nblk;
    if ((int)blockIdx.x >= R) return;
    const int v = pf_virtual_block(blockIdx.x, R);
    const PfTile tile = A.gu_tiles[v / nblk];
    const PfGroup &G = A.groups[tile.grp];
    const int mlen = min(NwTile<SPLIT>::ROWS, G.n - tile.m0), j0 = (v % nblk) * 16 * NWG_W;
    if (G.gq6) nw_gu_body<true, SPLIT>(A, G, meta, tile.m0, mlen, j0, (_Float16 *)nw_lds);
    else nw_gu_body<false, SPLIT>(A, G, meta, tile.m0, mlen, j0, (_Float16 *)nw_lds);
}

/* ---- down (inter <= 512) -----------------------------------------------------
 * A workgroup (4 waves) stages its tile's activations once, every super-block
 * of the SiLU*up rows with their sub-block sums, and walks dn_nt blocks of 128
 * output rows, the next block's weights loaded as each super-block's registers
 * come free.  Split mode: the f32 rows, scaled by the row's power of two (from
 * its part maxima) and split into fp16 hi + lo; f32 products.  fp16 mode: the
 * fp16 rows, each 16-column part moved from its own power of two onto the
 * row's; the products leave in fp16, scaled by 2^-e, e the exponent of the
 * bound max|act| * dbnd, as the wide down GEMMs store them (pf_gemm.hip).
 * 256 tokens split, Q6_K: 386 -> 60 us against the 64 x 64 tiles of gemm.h;
 * 8-wave workgroups 65 us. */
#define NWD_T 256
#define NWD_N (NWD_T / 2)         /* output rows per block: 32 a wave */

struct NwDnMeta {
    float inv[NW_ROWS], fwd[NW_ROWS];
    int8_t psh[NW_ROWS][32];      /* fp16 mode: part scale exponent - row scale exponent (<= 0) */
};

template <bool Q6, bool SPLIT, int NKB>
__device__ __forceinline__ void nw_dn_body(const PfGemmArgs &A, const PfGroup &G, NwDnMeta &meta, int m0, int mlen, int n0,
                                           int nt_count, _Float16 *Xb)
{
    constexpr int ROWS = NwTile<SPLIT>::ROWS, TB = TL_BYTES(Q6), NP = ROWS * NKB * 32 / NWD_T, NR = ROWS * 16 / NWD_T;
    const int t = threadIdx.x, l = t & 63, h = l >> 5, w = t >> 6, n = l & 31;
    const size_t slot0 = (size_t)(G.slot0 + m0);
    /* part maxima: 16 lanes per row, NKB of its 16 NKB parts each */
    float pm[NR][NKB];
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const float *pp = A.pmax + (slot0 + min((t >> 4) + i * (NWD_T / 16), mlen - 1)) * (16 * NKB) + (t & 15) * NKB;
#pragma unroll
        for (int k = 0; k < NKB; k++) pm[i][k] = pp[k];
    }
    /* activations: piece i of a thread is 8 columns of row idx / (32 NKB) */
    float4 xa[NP][2];
    uint4 xh[NP];
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const int idx = t + i * NWD_T, row = min(idx / (32 * NKB), mlen - 1), c = idx % (32 * NKB);
        const size_t at = (slot0 + row) * (GK * NKB) + 8 * c;
        if (SPLIT) {
            xa[i][0] = gld_f4(A.act + at);
            xa[i][1] = gld_f4(A.act + at + 4);
        } else {
            xh[i] = gld_u4(A.act16 + at);
        }
    }
    typename RawOf<Q6>::T r[NKB];
    const uint8_t *wt = G.td + (size_t)((n0 + 32 * w) / TL_ROWS) * NKB * TB;
    constexpr size_t TN = (size_t)(NWD_N / TL_ROWS) * NKB * TB;          /* one block of output rows on */
#pragma unroll
    for (int k = 0; k < NKB; k++) nw_load(r[k], wt + (size_t)k * TB, 16 * l);
#pragma unroll
    for (int i = 0; i < NR; i++) {
        const int row = (t >> 4) + i * (NWD_T / 16);
        float mx = pm[i][0];
#pragma unroll
        for (int k = 1; k < NKB; k++) mx = fmaxf(mx, pm[i][k]);
        mx = fmaxf(mx, dpp_f<DPP_XOR1>(mx));
        mx = fmaxf(mx, dpp_f<DPP_XOR2>(mx));
        mx = fmaxf(mx, dpp_f<DPP_HALF_MIRROR>(mx));
        mx = fmaxf(mx, dpp_f<DPP_MIRROR>(mx));
        float inv, fwd;
        if (SPLIT) {
            row_scale_wide(mx, inv, fwd);
        } else {
            row_scale(mx, inv, fwd);
            const int er = pf_scale_exp(mx), sp = pf_scale_exp(mx * G.dbnd);
            fwd = __builtin_bit_cast(float, (uint32_t)(127 + max(-126, min(126, er - sp))) << 23);
            if ((t & 15) == 0 && row < mlen && n0 == 0) A.oexp[slot0 + row] = (int8_t)sp;
#pragma unroll
            for (int k = 0; k < NKB; k++)
                meta.psh[row][(t & 15) * NKB + k] = (int8_t)max(pf_scale_exp(pm[i][k]) - er, -64);
        }
        if ((t & 15) == 0) {
            meta.inv[row] = inv;
            meta.fwd[row] = fwd;
        }
    }
    lds_barrier();
#pragma unroll
    for (int i = 0; i < NP; i++) {
        const int idx = t + i * NWD_T, row = idx / (32 * NKB), c = idx % (32 * NKB), kb = c >> 5, c8 = 8 * (c & 31);
        if (i * NWD_T / (32 * NKB) >= mlen) break;                       /* workgroup-uniform */
        _Float16 *dh = Xb + kb * NW_BUF + row * NW_LD;
        const int s0 = perm_slot4(c8), s1 = perm_slot4(c8 + 4);
        f32x8 e;
        if (SPLIT) {
            const float s = meta.inv[row];
            e = (f32x8){ xa[i][0].x, xa[i][0].y, xa[i][0].z, xa[i][0].w, xa[i][1].x, xa[i][1].y, xa[i][1].z, xa[i][1].w } * s;
        } else {
            const int sh = (int)meta.psh[row][c >> 1];
            const f16x8 hv = __builtin_bit_cast(f16x8, xh[i]);
#pragma unroll
            for (int k = 0; k < 8; k++) e[k] = __builtin_ldexpf((float)hv[k], sh);
        }
        const f16x8 hi = __builtin_convertvector(e, f16x8);
        const uint4 hu = __builtin_bit_cast(uint4, hi);
        *(uint2 *)(dh + s0) = make_uint2(hu.x, hu.y);
        *(uint2 *)(dh + s1) = make_uint2(hu.z, hu.w);
        if (SPLIT) {
            const f32x8 back = __builtin_convertvector(hi, f32x8);
            const uint4 lu = __builtin_bit_cast(uint4, __builtin_convertvector(e - back, f16x8));
            *(uint2 *)(dh + ROWS * NW_LD + s0) = make_uint2(lu.x, lu.y);
            *(uint2 *)(dh + ROWS * NW_LD + s1) = make_uint2(lu.z, lu.w);
        } else {
            e = __builtin_convertvector(hi, f32x8);                      /* the sums of what the products see */
        }
        if (!Q6) {
            /* a sub-block is four neighbouring lanes' pieces */
            float sum = ((e[0] + e[1]) + (e[2] + e[3])) + ((e[4] + e[5]) + (e[6] + e[7]));
            sum = group_sum<4>(sum) * 0.015625f;
            const _Float16 sh = (_Float16)sum, sl = (_Float16)(sum - (float)sh);
            if ((t & 3) == 0) {
                dh[NW_SUM + (c8 >> 5)] = sh;
                dh[NW_SUM + 8 + (c8 >> 5)] = sl;
            }
        }
    }
    lds_barrier();
    for (int nt = 0; nt < nt_count; nt++) {
        /* the last block reloads its own weights: a fixed number of loads per
         * block, so that each wait counts only the loads it needs */
        wt += nt + 1 < nt_count ? TN : 0;
        NwAcc<NwTile<SPLIT>::ACC> acc = {};
#pragma unroll
        for (int k = 0; k < NKB; k++) {
            __builtin_amdgcn_sched_barrier(0);
            nw_block<Q6, SPLIT>(acc, Xb + k * NW_BUF, r[k], l);
            __builtin_amdgcn_sched_barrier(0);
            nw_load(r[k], wt + (size_t)k * TB, 16 * l);
        }
        /* addresses and scales are formed here, not kept over the blocks */
        int hh = h;
        asm volatile("" : "+v"(hh));
        const size_t o0 = slot0 * A.H + n0 + nt * NWD_N;
        if (SPLIT) {
            float *ob = A.out + o0;
            const uint32_t oo = (uint32_t)(4 * hh * A.H + 32 * w + n);
#pragma unroll
            for (int q = 0; q < ROWS / 8; q++) {
                if (8 * q >= mlen) break;                                /* wave-uniform */
                const float4 f = *(const float4 *)(meta.fwd + 8 * q + 4 * hh);
                const float v[4] = { acc.v[4 * q] * f.x, acc.v[4 * q + 1] * f.y, acc.v[4 * q + 2] * f.z, acc.v[4 * q + 3] * f.w };
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (8 * q + 4 * hh + i < mlen) ob[oo + (uint32_t)((8 * q + i) * A.H)] = v[i];
            }
        } else {
            /* lanes n and n ^ 1 swap one value of each row pair: the even lane
             * stores the first row's two columns, the odd lane the second's */
            const bool odd = (n & 1) != 0;
            uint16_t *ob = A.out16 + o0;
            const uint32_t oo = (uint32_t)((4 * hh + (odd ? 1 : 0)) * A.H + 32 * w + (n & ~1));
#pragma unroll
            for (int q = 0; q < ROWS / 8; q++) {
                if (8 * q >= mlen) break;                                /* wave-uniform */
                const float4 f = *(const float4 *)(meta.fwd + 8 * q + 4 * hh);
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                    const float v0 = acc.v[4 * q + i] * (i ? f.z : f.x), v1 = acc.v[4 * q + i + 1] * (i ? f.w : f.y);
                    const float got = dpp_f<DPP_XOR1>(odd ? v0 : v1);
                    const f16x2 pk = { (_Float16)(odd ? got : v0), (_Float16)(odd ? v1 : got) };
                    if (8 * q + 4 * hh + i + (odd ? 1 : 0) < mlen)
                        *(uint32_t *)(ob + oo + (uint32_t)((8 * q + i) * A.H)) = __builtin_bit_cast(uint32_t, pk);
                }
            }
        }
    }
}

template <bool SPLIT>
__global__ void __launch_bounds__(NWD_T, 3) pfn_down_kernel(PfGemmArgs A)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t nw_lds[];
    __shared__ __attribute__((aligned(16))) NwDnMeta meta;
    const int nt = A.dn_nt, nblk = A.H / NWD_N / nt, R = *A.gu_ntiles * nblk;
    if ((int)blockIdx.x >= R) return;
    const int v = pf_virtual_block(blockIdx.x, R);
    const PfTile tile = A.gu_tiles[v / nblk];
    const PfGroup &G = A.groups[tile.grp];
    const int mlen = min(NwTile<SPLIT>::ROWS, G.n - tile.m0), n0 = (v % nblk) * nt * NWD_N;
    _Float16 *Xb = (_Float16 *)nw_lds;
    if (A.I > GK) {
        if (G.dq6) nw_dn_body<true, SPLIT, 2>(A, G, meta, tile.m0, mlen, n0, nt, Xb);
        else nw_dn_body<false, SPLIT, 2>(A, G, meta, tile.m0, mlen, n0, nt, Xb);
    } else {
        if (G.dq6) nw_dn_body<true, SPLIT, 1>(A, G, meta, tile.m0, mlen, n0, nt, Xb);
        else nw_dn_body<false, SPLIT, 1>(A, G, meta, tile.m0, mlen, n0, nt, Xb);
    }
}

/* ---- host ----------------------------------------------------------------- */
int pf_narrow_rows(bool split) { return split ? NwTile<true>::ROWS : NwTile<false>::ROWS; }

/* The down GEMM beside it: the wide one is level with this on Q6_K from 45
 * tokens on (45 tokens 129.5 us a layer, here 131.9; 512 skewed 180, here 184;
 * 4 tokens 55.4, here 52.8), and slower on Q4_K, whose dequantisation there
 * costs twice the instructions (200 tokens 157 us, here 149; 512 skewed 175,
 * here 170). */
bool pf_narrow_f16_down(int T, int E, int q6) { return !q6 || 8 * (long long)T <= E; }

int pf_narrow_gu_launch(const PfGemmArgs &A, int max_tiles, bool split)
{
    const dim3 g((unsigned)(max_tiles * (A.I / (16 * NWG_W)))), b(64 * NWG_W);
    const size_t lds = 2 * (size_t)NW_BUF * 2;
    if (split) hipLaunchKernelGGL(pfn_gu_kernel<true>, g, b, lds, rt().stream, A);
    else hipLaunchKernelGGL(pfn_gu_kernel<false>, g, b, lds, rt().stream, A);
    return rt_check(hipGetLastError(), "prefill gate/up launch") ? ROASTER_EDEVICE : 0;
}

/* Where the line lies: fp16 mode's wide tiles (pf_gemm.hip) dequantise a weight
 * once per 96 rows, these once per 32, but run at three waves per SIMD and
 * balance in units of 64 columns.  Measured per layer (256 experts, hidden
 * 2048, inter 512, Q6_K down; wide -> narrow, us): Q4_K gate/up 512 tokens 205
 * -> 173, 768 224 -> 190, 1152 (the line) 257 -> 241, 1792 288 -> 297; Q6_K gate/up
 * 512 210 -> 196, 896 (the line) 236 -> 225, 1152 262 -> 268, 1792 283 -> 319.  At
 * the line of other shapes, Q4_K / Q6_K: hidden 1024 167 -> 151 / 149 -> 137, inter
 * 256 187 -> 167 / 163 -> 148, inter 768 412 -> 402 / 382 -> 381, inter 1024 505 ->
 * 502 / 470 -> 470, 64 experts 107 -> 81 / 99 -> 77, 8 experts 77 -> 45 / 69 -> 46.
 * Where a few experts take every token the narrow tiles run out first: 8 of 256,
 * 768 tokens 136 -> 122 / 135 -> 126, but 1152 166 -> 173, Q6_K 896 136 -> 141. */
bool pf_narrow_f16(int T, int E, int q6) { return 8 * (long long)T <= (long long)E * (q6 ? 28 : 36); }

int pf_narrow_down_launch(const PfGemmArgs &A, int max_tiles, bool split)
{
    PfGemmArgs D = A;
    const int nb = A.H / NWD_N;                      /* even: H is a multiple of 256 */
    D.dn_nt = 2;                                     /* 1 / 2 / 4 / 8 blocks: 256 tokens 2 and 4 within 1%, 8 +3% */
    const dim3 g((unsigned)(max_tiles * (nb / D.dn_nt))), b(NWD_T);
    const size_t lds = (size_t)(A.I / GK) * NW_BUF * 2;
    if (split) hipLaunchKernelGGL(pfn_down_kernel<true>, g, b, lds, rt().stream, D);
    else hipLaunchKernelGGL(pfn_down_kernel<false>, g, b, lds, rt().stream, D);
    return rt_check(hipGetLastError(), "prefill down launch") ? ROASTER_EDEVICE : 0;
}
