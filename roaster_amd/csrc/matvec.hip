/*
 * matvec.hip -- multi-job quantised matvec / small-T matmul and the small
 * vector kernels behind kernels.h.
 *
 * Reference: kernel_matvec_quant_batch (kernels.c:1582-1646: all jobs of a call
 * in one submit), kernel_matmul_quant_batch (kernels.c:1916-2069,
 * Y[t*rows + r] = dot(W[r], X[t])), and the CPU vector kernels
 * (kernels.c:102-148, 584-719).
 *
 * One wave serves a task = (job, group of rows).  Lane layout per row:
 * lpr = lanes_per_row(blocks) lanes (qdot.h), 8 per 256-weight super-block
 * (qdot.h); each lane's quant chunk is loaded once and applied to all T tokens.
 */
#include "internal.h"
#include "qdot.h"
#include "matvec.h"
#include "pf_tile.h"

#include <type_traits>

#define MV_THREADS 256

template <bool Q6>
__device__ __forceinline__ void matvec_task(const MvJob &J, int task, int lane)
{
    const int nb = J.cols / RQK;
    const int lpr = lanes_per_row(nb), rpw = 64 / lpr;
    const int rw = lane / lpr, lr = lane % lpr, c = lr & 7, lb = lr >> 3;
    const int row = (task - J.task0) * rpw + rw;
    const bool live = row < J.rows;
    const size_t bs = Q6 ? RQ6K_BYTES : RQ4K_BYTES;
    const uint8_t *wrow = J.W + (size_t)(live ? row : 0) * nb * bs;
    for (int t = 0; t < J.T; t++) {
        const float *x = J.X + (size_t)t * J.cols;
        float part = 0.0f;
        for (int b = lb; live && b < nb; b += 8) {
            QChunk ch = q_load<Q6>(wrow + (size_t)b * bs, c);
            const int ca = b * RQK + q_run_a<Q6>(c), cb = ca + q_run_b_off<Q6>();
            part += q_chunk_dot<Q6>(ch, c, x + ca, x + cb, sum16(x + ca), sum16(x + cb));
        }
        part = group_sum_w(part, lpr);
        if (live && lr == 0) J.Y[(size_t)t * J.rows + row] = part;
    }
}

__global__ void __launch_bounds__(MV_THREADS) matvec_jobs_kernel(const MvJob *jobs, int njobs, int ntasks)
{
    const int lane = threadIdx.x & 63;
    const int gw = blockIdx.x * (MV_THREADS / 64) + (threadIdx.x >> 6), nw = gridDim.x * (MV_THREADS / 64);
    for (int task = gw; task < ntasks; task += nw) {
        int j = 0;
        while (j + 1 < njobs && jobs[j + 1].task0 <= task) j++;
        const MvJob J = jobs[j];
        if (J.q6) matvec_task<true>(J, task, lane);
        else matvec_task<false>(J, task, lane);
    }
}

/* ---- dense projections on device buffers ---------------------------------
 * y[t][r] = W[r] . x[t] for a [rows x cols] Q4_K / Q6_K matrix and T <= 8
 * tokens: the dense projections around the MoE block and the LM head
 * (model.c:795-800, 1284-1290, 1344-1347, 1368-1370; the same products
 * tensor_matvec_f32_or_quant, model.c:113-121, sends to kernel_matvec_q*_k).
 * cols <= 4096: one lane group covers a whole row (8 lanes per super-block,
 * lanes_per_row(blocks) lanes per row, 64 / lpr rows per wave pass), past 2048
 * columns with two super-blocks a lane.
 * Each lane's activation runs are fixed for every row it serves: with one
 * token they sit in registers for the whole kernel, with more in LDS.  Every
 * wave keeps the next row pass's loads in flight while it computes one. */
static int g_dense_mfma_t = 2;             /* tokens from which dense_mm8_kernel serves a call */

/* 16 (8) bytes at a 2-byte aligned address as the aligned dwords around them;
 * shift 0 or 16 brings them back.  A vector load that is not 4-byte aligned
 * is split by the memory pipe: the LM head (Q6_K [248320 x 2048], one token)
 * took 109 us with 2-byte aligned loads and takes 104 with these. */
struct U5 { uint4 v; uint32_t w; };

__device__ __forceinline__ U5 gld_5(const uint8_t *p)    /* p 4-byte aligned */
{
    typedef gu32x4 __attribute__((aligned(4))) gu32x4_a4;
    const gu32x4 v = *(const GAS gu32x4_a4 *)p;
    U5 r;
    r.v = make_uint4(v.x, v.y, v.z, v.w);
    r.w = gld_u32(p + 16);
    return r;
}

__device__ __forceinline__ uint4 u5_fix(const U5 &a, uint32_t sh)
{
    return make_uint4(__builtin_amdgcn_alignbit(a.v.y, a.v.x, sh), __builtin_amdgcn_alignbit(a.v.z, a.v.y, sh),
                      __builtin_amdgcn_alignbit(a.v.w, a.v.z, sh), __builtin_amdgcn_alignbit(a.w, a.v.w, sh));
}

/* A lane's chunk as loaded (q_load's bytes) and the QChunk it stands for.  DW:
 * as the aligned dwords around it, for Q6_K blocks at even addresses (a block
 * is 210 bytes, so all of a matrix's are even or none). */
template <bool Q6, bool DW> struct QRaw {
    QChunk ch;
    __device__ __forceinline__ void load(const uint8_t *blk, int c) { ch = q_load<Q6>(blk, c); }
    __device__ __forceinline__ QChunk chunk() const { return ch; }
};
template <> struct QRaw<true, true> {
    U5 q, h;
    uint32_t s[3], dd, sh;
    __device__ __forceinline__ void load(const uint8_t *blk, int c)
    {
        const uint8_t *al = (const uint8_t *)((uintptr_t)blk & ~(uintptr_t)3);
        const int n = c >> 2, p = c & 3;
        sh = ((uint32_t)(uintptr_t)blk & 2u) * 8u;
        q = gld_5(al + 16 * c);
        h = gld_5(al + 128 + 32 * n + 16 * (p & 1));
        typedef gu32x2 __attribute__((aligned(4))) gu32x2_a4;
        const gu32x2 v = *(const GAS gu32x2_a4 *)(al + 192 + 8 * n);
        s[0] = v.x;
        s[1] = v.y;
        s[2] = gld_u32(al + 192 + 8 * n + (sh ? 8 : 4));    /* not past the block's end */
        dd = gld_u16(blk + 208);
    }
    __device__ __forceinline__ QChunk chunk() const
    {
        QChunk ch;
        ch.q = u5_fix(q, sh);
        ch.h = u5_fix(h, sh);
        ch.s = make_uint2(__builtin_amdgcn_alignbit(s[1], s[0], sh), __builtin_amdgcn_alignbit(s[2], s[1], sh));
        ch.dd = dd;
        return ch;
    }
};

template <bool Q6, bool ONE, int KB, bool DW = Q6>
__global__ void __launch_bounds__(MV_THREADS) dense_mv_kernel(const uint8_t *W, const float *X, float *Y, int rows,
                                                              int cols, int T)
{
    extern __shared__ __align__(16) float xs[];            /* [T][cols] + run sums [T][cols / 16] (T > 1) */
    const int lane = threadIdx.x & 63;
    const int nb = cols / RQK, lpr = lanes_per_row(nb), rpw = 64 / lpr;
    const int rw = lane / lpr, lr = lane % lpr, c = lr & 7, lb = lr >> 3;
    const size_t bs = Q6 ? RQ6K_BYTES : RQ4K_BYTES, row_bytes = (size_t)nb * bs;
    /* KB super-blocks per lane: lb, lb + 8 (rows of more than 8 blocks) */
    bool blk_live[KB];
    int ca[KB], cb[KB];
#pragma unroll
    for (int k = 0; k < KB; k++) {
        blk_live[k] = lb + 8 * k < nb;
        ca[k] = (lb + 8 * k) * RQK + q_run_a<Q6>(c);
        cb[k] = ca[k] + q_run_b_off<Q6>();
    }
    float4 xa[KB][4], xb[KB][4];
    float sxa[KB], sxb[KB];
    float *xsum = xs + (size_t)T * cols;
    if (ONE) {
#pragma unroll
        for (int k = 0; k < KB; k++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                xa[k][i] = blk_live[k] ? gld_f4(X + ca[k] + 4 * i) : make_float4(0.f, 0.f, 0.f, 0.f);
                xb[k][i] = blk_live[k] ? gld_f4(X + cb[k] + 4 * i) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
            sxa[k] = ((xa[k][0].x + xa[k][0].y) + (xa[k][0].z + xa[k][0].w)) + ((xa[k][1].x + xa[k][1].y) + (xa[k][1].z + xa[k][1].w)) +
                     (((xa[k][2].x + xa[k][2].y) + (xa[k][2].z + xa[k][2].w)) + ((xa[k][3].x + xa[k][3].y) + (xa[k][3].z + xa[k][3].w)));
            sxb[k] = ((xb[k][0].x + xb[k][0].y) + (xb[k][0].z + xb[k][0].w)) + ((xb[k][1].x + xb[k][1].y) + (xb[k][1].z + xb[k][1].w)) +
                     (((xb[k][2].x + xb[k][2].y) + (xb[k][2].z + xb[k][2].w)) + ((xb[k][3].x + xb[k][3].y) + (xb[k][3].z + xb[k][3].w)));
        }
    } else {
        for (int i = threadIdx.x; i < T * cols / 4; i += MV_THREADS) ((float4 *)xs)[i] = gld_f4(X + 4 * i);
        __syncthreads();
        for (int i = threadIdx.x; i < T * cols / 16; i += MV_THREADS) xsum[i] = sum16(xs + 16 * i);
        __syncthreads();
    }
    const int gw = blockIdx.x * (MV_THREADS / 64) + (threadIdx.x >> 6), nw = gridDim.x * (MV_THREADS / 64);
    const int npass = (rows + rpw - 1) / rpw;
    /* the next pass's chunks are in flight while the current one's are dotted;
     * rows and blocks past the end read the last one, unused, so that the loads
     * carry no branches and each wait counts its own loads only */
    QRaw<Q6, DW> cur[KB], nxt[KB];
    auto load = [&](QRaw<Q6, DW> (&ch)[KB], int pass) {
        const int row = min(min(pass, npass - 1) * rpw + rw, rows - 1);
#pragma unroll
        for (int k = 0; k < KB; k++)
            ch[k].load(W + (size_t)row * row_bytes + (size_t)min(lb + 8 * k, nb - 1) * bs, c);
    };
    auto compute = [&](const QRaw<Q6, DW> (&ch)[KB], int pass) {
        const int row = pass * rpw + rw;
        const bool live = row < rows;
        QChunk qc[KB];
#pragma unroll
        for (int k = 0; k < KB; k++) qc[k] = ch[k].chunk();
        for (int t = 0; t < (ONE ? 1 : T); t++) {
            float part = 0.0f;
#pragma unroll
            for (int k = 0; k < KB; k++) {
                if (live && blk_live[k]) {
                    if (ONE) {
                        part += q_chunk_dot_r<Q6>(qc[k], c, xa[k], xb[k], sxa[k], sxb[k]);
                    } else {
                        const float *x = xs + (size_t)t * cols, *sx = xsum + (size_t)t * (cols / 16);
                        part += q_chunk_dot<Q6>(qc[k], c, x + ca[k], x + cb[k], sx[ca[k] >> 4], sx[cb[k] >> 4]);
                    }
                }
            }
            part = group_sum_w(part, lpr);
            if (live && lr == 0) Y[(size_t)t * rows + row] = part;
        }
    };
    if (gw >= npass) return;
    load(cur, gw);
    if (gw + nw >= npass) {                              /* this wave's only pass */
        compute(cur, gw);
        return;
    }
    for (int p = gw; p < npass; p += 2 * nw) {
        load(nxt, p + nw);
        __builtin_amdgcn_sched_barrier(0);
        compute(cur, p);
        if (p + nw >= npass) break;
        load(cur, p + 2 * nw);
        __builtin_amdgcn_sched_barrier(0);
        compute(nxt, p + nw);
    }
}

/* ---- tokens on MFMA -----------------------------------------------------------
 * y[t][r] = W[r] . x[t] with 16 weight rows per wave on
 * v_mfma_f32_16x16x32_f16 and the block's integer part as the operand, which
 * fp16 holds exactly:
 *   B = 16 rows x 32 columns: Q4_K sc q (at most 945), Q6_K sc (q - 32) with
 *       what its rounding to 11 bits drops (above 2048 in magnitude) as a
 *       second operand; lane l holds row l % 16 and 8 columns of its run;
 *   A = the tokens' activations, scaled per (token, super-block) by a power of
 *       two (max |x| in [2^14, 2^15)) and split into fp16 parts: up to 4 tokens
 *       three parts (every bit of an f32), rows 4 t + part, 5..8 tokens two
 *       (22 bits), rows 2 t + part, so that the accumulators of lane l are the
 *       parts of token l / 16 (of tokens 2 (l / 16), + 1) and add up in the
 *       lane;
 *   d, the scale's inverse and (Q4_K) dmin times the sub-block minima's
 *       product with the sub-block sums (one more MFMA: minima 2 g, 2 g + 1 in
 *       lane group g) are applied in f32 once per super-block; the sums are f32
 *       in three fp16 parts, the third, with 5..8 tokens, beside the second in
 *       its row (the minima stand there again)
 * (the reference's fold, kernels.c:1844-1874: d sc sum(q x) - dmin m sum(x),
 * d sc sum((q - 32) x)).  Every workgroup prepares A in LDS itself while its
 * first weights are on the way; each wave streams 16-row groups, the next
 * super-block's quants in flight while one computes. */
#define MM8_T 512
#define MM8_W (MM8_T / 64)
#define MM8_RED (2 * MM8_W * 64 * 8)      /* static LDS of dense_mm8_kernel */

/* LDS of one call: A fragments [cols / 256][8][64 lanes] (16 bytes), sub-block
 * sums [cols / 256][64 lanes] (MM8_SUM fp16), scales [cols / 256][8 tokens] (2^-e). */
#define MM8_SUM(Q6, PARTS) (!(Q6) && (PARTS) == 2 ? 4 : 2)
__host__ __device__ static inline size_t mm8_frag_bytes(size_t cols) { return cols * 32; }
template <bool Q6, int PARTS>
__host__ __device__ static inline size_t mm8_sum_bytes(size_t cols) { return cols / 2 * MM8_SUM(Q6, PARTS); }
template <bool Q6, int PARTS>
__host__ __device__ static inline size_t mm8_lds_bytes(size_t cols)
{
    return mm8_frag_bytes(cols) + mm8_sum_bytes<Q6, PARTS>(cols) + cols / RQK * 8 * 4;
}

/* Super-block kb of the activations into LDS (one wave): lane (t = l / 8, c =
 * l % 8) takes columns 32 c .. + 31 of token t. */
template <bool Q6, int PARTS>
__device__ __forceinline__ void mm8_prep(const float *X, int cols, int T, int kb, uint8_t *lds, int lane)
{
    const int t = lane >> 3, c = lane & 7;
    /* lane group g's columns in slice f follow its 16-byte runs of quants
     * (mm8_load): Q6_K 64 (f / 2) + 16 g + 8 (f % 2) .. + 7, Q4_K 128 (f / 4) +
     * 64 (g / 2) + 32 ((f / 2) % 2) + 16 (g % 2) + 8 (f % 2) .. + 7 */
    f16x8 *frag = (f16x8 *)lds + (size_t)kb * 512 +
                  (Q6 ? 128 * (c >> 1) + 32 * (c & 1) : 256 * (c >> 2) + 128 * (c & 1) + 32 * ((c >> 1) & 1));
    _Float16 *sums = (_Float16 *)(lds + mm8_frag_bytes(cols)) + kb * 64 * MM8_SUM(Q6, PARTS);
    float *ge = (float *)(lds + mm8_frag_bytes(cols) + mm8_sum_bytes<Q6, PARTS>(cols)) + kb * 8;
    if (t >= T) return;
    const float *xp = X + (size_t)t * cols + RQK * kb + 32 * c;
    float4 v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = gld_f4(xp + 4 * i);
    float mx = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++)
        mx = fmaxf(mx, fmaxf(fmaxf(fabsf(v[i].x), fabsf(v[i].y)), fmaxf(fabsf(v[i].z), fabsf(v[i].w))));
    mx = fmaxf(mx, dpp_f<DPP_XOR1>(mx));
    mx = fmaxf(mx, dpp_f<DPP_XOR2>(mx));
    mx = fmaxf(mx, dpp_f<DPP_HALF_MIRROR>(mx));
    int e = 0;
    if (mx > 0.0f && mx <= 3.0e38f) {
        int E;
        (void)frexpf(mx, &E);
        e = min(max(15 - E, -100), 100);
    }
    const float up = ldexpf(1.0f, e);
    if (c == 0) ge[t] = ldexpf(1.0f, -e);
    const int row = PARTS == 3 ? 4 * t : 2 * t;
    float sum = 0.0f;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        f32x8 w = { v[2 * g].x, v[2 * g].y, v[2 * g].z, v[2 * g].w, v[2 * g + 1].x, v[2 * g + 1].y, v[2 * g + 1].z, v[2 * g + 1].w };
        w = w * up;
        sum += ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
#pragma unroll
        for (int p = 0; p < PARTS; p++) {
            const f16x8 h = __builtin_convertvector(w, f16x8);
            frag[64 * (g & 1) + 16 * (g >> 1) + row + p] = h;
            w = w - __builtin_convertvector(h, f32x8);
        }
    }
    /* sub-block c's sum, in lane group c / 2's slot c % 2; two rows a token: the
     * third part in the second row's slot 2 + c % 2, lanes c and c ^ 1 swapping
     * what the other's row holds, so that each stores one row's four slots */
    sum *= 0.015625f;
    _Float16 sp[3];
#pragma unroll
    for (int p = 0; p < 3; p++) {
        sp[p] = (_Float16)sum;
        sum -= (float)sp[p];
    }
    if constexpr (MM8_SUM(Q6, PARTS) == 4) {
        const bool odd = (c & 1) != 0;
        const f16x2 mine = odd ? (f16x2){ sp[0], (_Float16)0.0f } : (f16x2){ sp[1], sp[2] };
        const f16x2 got = __builtin_bit_cast(f16x2, dpp_i<DPP_XOR1>(__builtin_bit_cast(int, mine)));
        *(f16x4 *)(sums + (16 * (c >> 1) + row + (odd ? 1 : 0)) * 4) =
            odd ? (f16x4){ got[0], sp[1], got[1], sp[2] } : (f16x4){ sp[0], got[0], (_Float16)0.0f, (_Float16)0.0f };
    } else {
#pragma unroll
        for (int p = 0; p < PARTS; p++) sums[(16 * (c >> 1) + row + p) * 2 + (c & 1)] = sp[p];
    }
}

/* Lane group g's share of a super-block: 16-byte runs, so that the four lanes
 * of a row read 64 contiguous bytes a load.  Q4_K: qs bytes 64 k + 16 g
 * (sub-blocks 4 k + 2 (g / 2), + 1); Q6_K, by half n: ql bytes 64 n + 16 g
 * (scales 8 n + g, + 4) and the qh bytes under them. */
struct Mm8Q4 { uint4 hd, p[2]; };
struct Mm8Q6 { U5 l[2], h[2], sc; uint32_t d, sh; };

__device__ __forceinline__ void mm8_load(Mm8Q4 &r, const uint8_t *blk, int g)
{
    r.hd = gld_u4(blk);
#pragma unroll
    for (int k = 0; k < 2; k++) r.p[k] = gld_u4(blk + 16 + 64 * k + 16 * g);
}

__device__ __forceinline__ void mm8_load(Mm8Q6 &r, const uint8_t *blk, int g)
{
    const uint8_t *al = (const uint8_t *)((uintptr_t)blk & ~(uintptr_t)3);
    r.sh = ((uint32_t)(uintptr_t)blk & 2u) * 8u;
#pragma unroll
    for (int n = 0; n < 2; n++) {
        r.l[n] = gld_5(al + 64 * n + 16 * g);
        r.h[n] = gld_5(al + 128 + 32 * n + 16 * (g & 1));
    }
    typedef gu32x4 __attribute__((aligned(4))) gu32x4_a4;
    const gu32x4 v = *(const GAS gu32x4_a4 *)(al + 192);
    r.sc.v = make_uint4(v.x, v.y, v.z, v.w);
    r.sc.w = gld_u32(al + (r.sh ? 208 : 204));
    r.d = gld_u16(blk + 208);
}

__device__ __forceinline__ uint32_t u4_word(const uint4 &v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

/* Scale / minimum j (a byte offset of 0..2 with j + 1 in the same half) and
 * the next of a lane group whose sub-blocks lie in the header's lower (lo) or
 * upper half; sh = 8 j. */
__device__ __forceinline__ uint32_t q4_pair6(uint32_t own, uint32_t s811, int nib, int sh, bool lo)
{
    const uint32_t a = own >> sh, b = s811 >> (sh + nib);
    const uint32_t x = a & 0x3F3Fu, y = (b & 0x0F0Fu) | ((a >> 2) & 0x3030u);
    return lo ? x : y;                                   /* bytes 0 and 1 */
}

/* z: the integer products of one super-block; zm: the minima's (Q4_K). */
template <int PARTS>
__device__ __forceinline__ void mm8_block(const Mm8Q4 &r, const uint8_t *frag, const uint8_t *sums, int lane, f32x4 (&z)[2],
                                          f32x4 &zm)
{
    const uint32_t s03 = r.hd.y, s47 = r.hd.z, s811 = r.hd.w;
    const int g = lane >> 4;
    {
        /* minima 2 g, 2 g + 1 of lane group g against the sums of those sub-blocks */
        const uint32_t m = q4_pair6(s47, s811, 4, 16 * (g & 1), g < 2);
        const _Float16 o = (_Float16)0.0f;
        const _Float16 m0 = (_Float16)(int)(m & 0xFF), m1 = (_Float16)(int)(m >> 8);
        f16x8 mb = { m0, m1, o, o, o, o, o, o }, xa = { o, o, o, o, o, o, o, o };
        if constexpr (PARTS == 2) {
            const f16x4 xs = *(const f16x4 *)(sums + 8 * lane);
            mb[2] = m0, mb[3] = m1;
            xa[0] = xs[0], xa[1] = xs[1], xa[2] = xs[2], xa[3] = xs[3];
        } else {
            const f16x2 xs = *(const f16x2 *)(sums + 4 * lane);
            xa[0] = xs[0], xa[1] = xs[1];
        }
        zm = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa, mb, (f32x4){}, 0, 0, 0);
    }
    z[0] = z[1] = (f32x4){};
#pragma unroll
    for (int k = 0; k < 2; k++) {
        /* sub-blocks 4 k + 2 (g / 2) (low nibbles) and + 1 (high) */
        const uint32_t scs = q4_pair6(s03, s811, 0, 16 * (g >> 1), k == 0);
#pragma unroll
        for (int hi = 0; hi < 2; hi++) {
            const _Float16 sf = (_Float16)(int)(hi ? scs >> 8 : scs & 0xFF);
            const f16x2 scv = { sf, sf };
            const f16x2 bias = scv * (f16x2){ (_Float16)-1024.0f, (_Float16)-1024.0f };   /* exact: 63 * 1024 < 65504 */
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const uint32_t p = u4_word(r.p[k], 2 * i), q = u4_word(r.p[k], 2 * i + 1);
                const uint32_t x = (hi ? p >> 4 : p) & 0x0F0F0F0Fu, y = (hi ? q >> 4 : q) & 0x0F0F0F0Fu;
                const f16x2 w0 = __builtin_elementwise_fma(magic_lo(x), scv, bias), w1 = __builtin_elementwise_fma(magic_hi(x), scv, bias);
                const f16x2 w2 = __builtin_elementwise_fma(magic_lo(y), scv, bias), w3 = __builtin_elementwise_fma(magic_hi(y), scv, bias);
                const f16x8 b = { w0[0], w0[1], w1[0], w1[1], w2[0], w2[1], w3[0], w3[1] };
                const f16x8 a = *(const f16x8 *)(frag + (4 * k + 2 * hi + i) * 1024 + lane * 16);
                z[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, z[i], 0, 0, 0);
            }
        }
    }
}

template <int PARTS>
__device__ __forceinline__ void mm8_block(const Mm8Q6 &r, const uint8_t *frag, const uint8_t *, int lane, f32x4 (&z)[2], f32x4 &)
{
    const int g = lane >> 4, qs = 2 * (g >> 1);             /* qh bits of the low nibbles' columns */
    const f16x2 off = { (_Float16)-1056.0f, (_Float16)-1056.0f };
    z[0] = z[1] = (f32x4){};
    const uint4 scv = u5_fix(r.sc, r.sh);
#pragma unroll
    for (int n = 0; n < 2; n++) {
        const uint4 rl = u5_fix(r.l[n], r.sh), rh = u5_fix(r.h[n], r.sh);
        uint32_t hs[4];
#pragma unroll
        for (int i = 0; i < 4; i++) hs[i] = u4_word(rh, i) >> qs;
#pragma unroll
        for (int hi = 0; hi < 2; hi++) {
            const uint32_t sw = u4_word(scv, 2 * n + hi);
            const _Float16 sf = (_Float16)(short)__builtin_amdgcn_sbfe((int)sw, 8 * g, 8);
            const f16x2 sc = { sf, sf };
#pragma unroll
            for (int i = 0; i < 2; i++) {
                f16x2 w[4], e[4];
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const uint32_t lw = u4_word(rl, 2 * i + k), hw = hs[2 * i + k];
                    const uint32_t q = hi ? ((lw >> 4) & 0x0F0F0F0Fu) | (hw & 0x30303030u) : (lw & 0x0F0F0F0Fu) | ((hw << 4) & 0x30303030u);
                    const f16x2 u = magic_lo(q) + off, v = magic_hi(q) + off;    /* q - 32 */
                    w[2 * k] = u * sc;
                    w[2 * k + 1] = v * sc;
                    e[2 * k] = __builtin_elementwise_fma(u, sc, -w[2 * k]);
                    e[2 * k + 1] = __builtin_elementwise_fma(v, sc, -w[2 * k + 1]);
                }
                const f16x8 b = { w[0][0], w[0][1], w[1][0], w[1][1], w[2][0], w[2][1], w[3][0], w[3][1] };
                const f16x8 be = { e[0][0], e[0][1], e[1][0], e[1][1], e[2][0], e[2][1], e[3][0], e[3][1] };
                const f16x8 a = *(const f16x8 *)(frag + (4 * n + 2 * hi + i) * 1024 + lane * 16);
                z[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, z[0], 0, 0, 0);
                z[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, be, z[1], 0, 0, 0);
            }
        }
    }
}

/* One super-block of a 16-row group: its products added (live) to y, the sums
 * of this lane's tokens (PARTS == 3: token l / 16; 2: tokens 2 (l / 16), + 1). */
template <bool Q6, int PARTS, class Raw>
__device__ __forceinline__ void mm8_add(const Raw &raw, const uint8_t *lds, int cols, int kb, bool live, int lane,
                                        float (&y)[2])
{
    f32x4 z[2], zm;
    mm8_block<PARTS>(raw, lds + (size_t)kb * 8192, lds + mm8_frag_bytes(cols) + kb * 128 * MM8_SUM(Q6, PARTS), lane, z, zm);
    const float *ge = (const float *)(lds + mm8_frag_bytes(cols) + mm8_sum_bytes<Q6, PARTS>(cols)) + kb * 8;
    const int g = lane >> 4;
    float d, dm;
    if constexpr (Q6) {
        d = f16_bits_to_f32(raw.d);
        dm = 0.0f;
    } else {
        d = f16_bits_to_f32(raw.hd.x & 0xFFFFu);
        dm = f16_bits_to_f32(raw.hd.x >> 16) * -64.0f;   /* the sums carry 2^-6 */
    }
    const f32x4 s = z[0] + z[1];
    if (PARTS == 3) {
        float v = d * ((s[0] + s[1]) + s[2]);
        if (!Q6) v = fmaf(dm, (zm[0] + zm[1]) + zm[2], v);
        y[0] = live ? fmaf(v, ge[g], y[0]) : y[0];
    } else {
        float v0 = d * (s[0] + s[1]), v1 = d * (s[2] + s[3]);
        if (!Q6) {
            v0 = fmaf(dm, zm[0] + zm[1], v0);
            v1 = fmaf(dm, zm[2] + zm[3], v1);
        }
        const float2 g2 = *(const float2 *)(ge + 2 * g);
        y[0] = live ? fmaf(v0, g2.x, y[0]) : y[0];
        y[1] = live ? fmaf(v1, g2.y, y[1]) : y[1];
    }
}

template <int PARTS>
__device__ __forceinline__ void mm8_store(float *Y, int rows, int T, int r, int lane, const float (&y)[2])
{
    if (r >= rows) return;
    const int t0 = PARTS == 3 ? lane >> 4 : 2 * (lane >> 4);
    if (t0 < T) Y[(size_t)t0 * rows + r] = y[0];
    if (PARTS == 2 && t0 + 1 < T) Y[(size_t)(t0 + 1) * rows + r] = y[1];
}

template <bool Q6, int PARTS>
__global__ void __launch_bounds__(MM8_T, 4) dense_mm8_kernel(const uint8_t *W, const float *X, float *Y, int rows, int cols,
                                                             int T, int split)
{
    extern __shared__ __align__(16) uint8_t mm8_lds[];
    constexpr size_t BS = Q6 ? RQ6K_BYTES : RQ4K_BYTES;
    typedef typename std::conditional<Q6, Mm8Q6, Mm8Q4>::type Raw;
    const int nb = cols / RQK;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g4 = lane >> 4;
    const int ngroups = (rows + 15) >> 4;
    /* a workgroup is 8 / split teams of split waves; a team takes a 16-row
     * group, its member m the super-blocks m, m + split, ..., and member 0 adds
     * the members' sums in their order */
    const int member = wv & (split - 1), tpw = MM8_W / split;
    const int team = blockIdx.x * tpw + wv / split, nteam = gridDim.x * tpw;
    const int iters = (ngroups + nteam - 1) / nteam, per = (nb + split - 1) / split, total = iters * per;
    __shared__ float2 red[2][MM8_W][64];
    static_assert(sizeof(red) == MM8_RED, "the launch counts it");
    /* item i: super-block member + (i % per) split of group team + (i / per)
     * nteam; past either end the last one again, so that every wave runs the
     * same items and barriers */
    auto blk = [&](int item) {
        const int g = min(team + (item / per) * nteam, ngroups - 1), kb = min(member + (item % per) * split, nb - 1);
        const int r = min(16 * g + (lane & 15), rows - 1);
        return W + ((size_t)r * nb + kb) * BS;
    };
    Raw ra, rb;
    mm8_load(ra, blk(0), g4);
    for (int kb = wv; kb < nb; kb += MM8_W) mm8_prep<Q6, PARTS>(X, cols, T, kb, mm8_lds, lane);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   /* LDS only: the weights stay in flight */
    float y[2] = { 0.0f, 0.0f };
    auto compute = [&](const Raw &raw, int item) {
        const int it = item / per, j = item - it * per, kb = member + j * split;
        mm8_add<Q6, PARTS>(raw, mm8_lds, cols, min(kb, nb - 1), kb < nb, lane, y);   /* no branch: the loads stay ahead */
        if (j != per - 1) return;
        const int g = team + it * nteam;
        if (split > 1) {
            red[it & 1][wv][lane] = make_float2(y[0], y[1]);
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if (member == 0)
                for (int w = 1; w < split; w++) {
                    const float2 b = red[it & 1][wv + w][lane];
                    y[0] += b.x;
                    y[1] += b.y;
                }
        }
        if (member == 0 && g < ngroups) mm8_store<PARTS>(Y, rows, T, 16 * g + (lane & 15), lane, y);
        y[0] = y[1] = 0.0f;
    };
    /* the loads are unconditional, so that the wait before a computation counts
     * only its own loads, not the next item's behind them */
    for (int it = 0;; it += 2) {
        mm8_load(rb, blk(min(it + 1, total - 1)), g4);
        compute(ra, it);
        if (it + 1 >= total) break;
        mm8_load(ra, blk(min(it + 2, total - 1)), g4);
        compute(rb, it + 1);
        if (it + 2 >= total) break;
    }
}

/* The same with the weights staged in LDS, for many rows: 16 waves, each on
 * 16-row groups of its own.  Loaded where they are used, a Q6_K super-block's
 * 16 x 210 bytes take a wave eleven loads of 64-byte pieces at 2-byte alignment,
 * and a 128-byte line is fetched by several of them, after the CU's other waves
 * have driven it out of its cache.  Here a wave takes them in order, 13 chunks of
 * 16 bytes a row (Q4_K 9), with four loads and one for the last four bytes, two
 * super-blocks in flight, and picks its quants up from its own slice of LDS.
 * Groups go round the CUs before the waves of one.  LM head (Q6_K [248320 x
 * 2048]), five tokens: 124.5 -> 100.4 us (4.15 TB/s); [60000 x 2048] 37.4 -> 27.9. */
#define MM8S_T 1024
#define MM8S_W (MM8S_T / 64)

/* A lane's share of a staged super-block: its chunks; Q6_K: bytes 206..209 of
 * the lane's own row and the shift of its bytes. */
template <bool Q6>
struct Mm8S {
    static constexpr int CH = Q6 ? 13 : 9, N = 16 * CH, NL = (N + 63) / 64;   /* chunks a row (odd: 8 rows' 16-byte reads
                                                                                  fall in different banks), a group, loads */
    uint4 c[NL];
    uint32_t t, sh;
};

template <bool Q6, int PARTS>
__global__ void __launch_bounds__(MM8S_T, 1) dense_mm8s_kernel(const uint8_t *W, const float *X, float *Y, int rows, int cols,
                                                               int T)
{
    extern __shared__ __align__(16) uint8_t mm8_lds[];
    typedef Mm8S<Q6> Raw;
    constexpr unsigned BS = Q6 ? RQ6K_BYTES : RQ4K_BYTES;
    const int nb = cols / RQK;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, g4 = lane >> 4;
    const int ngroups = (rows + 15) >> 4, nw = gridDim.x * MM8S_W;
    uint8_t *slice = mm8_lds + mm8_lds_bytes<Q6, PARTS>(cols) + wv * 16 * Raw::N;
    /* load i of this lane: chunk ck of the group's row cr (past the last chunk
     * that one again, to the same place) */
    int cr[Raw::NL], ck[Raw::NL];
#pragma unroll
    for (int i = 0; i < Raw::NL; i++) {
        const int idx = min(64 * i + lane, Raw::N - 1);
        cr[i] = idx / Raw::CH;
        ck[i] = 16 * (idx - Raw::CH * cr[i]);
    }
    const int g0 = wv * gridDim.x + blockIdx.x;
    int lg = g0, lkb = 0;                               /* the next super-block to load */
    auto rowp = [&](int r) { return W + (size_t)min(16 * min(lg, ngroups - 1) + r, rows - 1) * nb * BS; };
    const uint8_t *wr[Raw::NL], *own;
    auto rowset = [&]() {
#pragma unroll
        for (int i = 0; i < Raw::NL; i++) wr[i] = rowp(cr[i]);
        own = rowp(lane & 15);
    };
    rowset();
    auto load = [&](Raw &r) {                           /* past the last group that one again, unused */
        typedef gu32x4 __attribute__((aligned(4))) gu32x4_a4;
        const unsigned at = (unsigned)lkb * BS;
#pragma unroll
        for (int i = 0; i < Raw::NL; i++) {
            const uint8_t *al = wr[i] + at;
            if (Q6) al = (const uint8_t *)((uintptr_t)al & ~(uintptr_t)3);
            const gu32x4 v = *(const GAS gu32x4_a4 *)(al + ck[i]);
            r.c[i] = make_uint4(v.x, v.y, v.z, v.w);
        }
        if constexpr (Q6) {
            typedef uint32_t __attribute__((aligned(2))) u32_a2;
            const uint8_t *b = own + at;
            r.t = *(const GAS u32_a2 *)(b + 206);
            r.sh = ((uint32_t)(uintptr_t)b & 2u) * 8u;
        }
        if (++lkb == nb) {
            lkb = 0;
            lg += nw;
            rowset();
        }
    };
    Raw ra, rb;
    load(ra);
    load(rb);
    for (int kb = wv; kb < nb; kb += MM8S_W) mm8_prep<Q6, PARTS>(X, cols, T, kb, mm8_lds, lane);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   /* LDS only: the weights stay in flight */
    if (g0 >= ngroups) return;
    float y[2] = { 0.0f, 0.0f };
    int g = g0, kb = 0;                                 /* the super-block to compute */
    /* the slice's stores and loads of one step and the next stay in order, for
     * all lanes (LDS serves a wave's accesses in order: no instructions) */
    auto wave_fence = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    auto step = [&](Raw &r) {                           /* whether it was the last */
        wave_fence();
#pragma unroll
        for (int i = 0; i < Raw::NL; i++) *(uint4 *)(slice + 16 * min(64 * i + lane, Raw::N - 1)) = r.c[i];
        wave_fence();
        const uint32_t tail = r.t, sh = r.sh;
        load(r);
        const uint8_t *row = slice + (lane & 15) * (16 * Raw::CH);
        if constexpr (Q6) {
            auto u5 = [&](int at) { return U5{ *(const uint4 *)(row + at), *(const uint32_t *)(row + at + 16) }; };
            Mm8Q6 q;
#pragma unroll
            for (int n = 0; n < 2; n++) {
                q.l[n] = u5(64 * n + 16 * g4);
                q.h[n] = u5(128 + 32 * n + 16 * (g4 & 1));
            }
            q.sc = U5{ *(const uint4 *)(row + 192), tail };
            q.d = tail >> 16;
            q.sh = sh;
            mm8_add<true, PARTS>(q, mm8_lds, cols, kb, true, lane, y);
        } else {
            Mm8Q4 q;
            q.hd = *(const uint4 *)row;
#pragma unroll
            for (int k = 0; k < 2; k++) q.p[k] = *(const uint4 *)(row + 16 + 64 * k + 16 * g4);
            mm8_add<false, PARTS>(q, mm8_lds, cols, kb, true, lane, y);
        }
        if (++kb != nb) return false;
        mm8_store<PARTS>(Y, rows, T, 16 * g + (lane & 15), lane, y);
        y[0] = y[1] = 0.0f;
        kb = 0;
        g += nw;
        return g >= ngroups;
    };
    for (;;) {
        if (step(ra)) break;
        if (step(rb)) break;
    }
}

static bool mat_odd(const uint8_t *W, int q6) { return q6 && ((uintptr_t)W & 1); }

bool dense_mm8_takes(const uint8_t *W, int q6, size_t cols, size_t T)
{
    return T >= (size_t)g_dense_mfma_t && cols <= 4096 && !mat_odd(W, q6);
}

int dense_mm8_launch(const uint8_t *W, int q6, const float *X, float *Y, size_t rows, size_t cols, int T)
{
    const size_t lds = q6 ? mm8_lds_bytes<true, 3>(cols) : T <= 4 ? mm8_lds_bytes<false, 3>(cols) : mm8_lds_bytes<false, 2>(cols);
    const size_t ng = (rows + 15) / 16;
    const size_t slds = lds + MM8S_W * 256 * (q6 ? Mm8S<true>::CH : Mm8S<false>::CH);
    const dim3 gs((unsigned)rt().n_cu), bs(MM8S_T);
#define MM8S(Q6_, P_) hipLaunchKernelGGL((dense_mm8s_kernel<Q6_, P_>), gs, bs, slds, rt().stream, W, X, Y, (int)rows, (int)cols, T)
    /* staged from 4 groups per CU on (256 CUs: 16384 rows), where a wave with a
     * group to itself is no longer short of others (Q6_K / Q4_K, five tokens:
     * [16384 x 768] 7.3 / 5.7 us staged, 7.9 / 5.7 not; [8192 x 2048] 11.8 / 8.4
     * and 11.0 / 8.4), while the slices fit beside the activations (Q6_K: 3328
     * columns) */
    if (ng >= 4 * (size_t)rt().n_cu && slds <= 160 * 1024) {
        if (T <= 4) {
            if (q6) MM8S(true, 3);
            else MM8S(false, 3);
        } else {
            if (q6) MM8S(true, 2);
            else MM8S(false, 2);
        }
#undef MM8S
        return rt_check(hipGetLastError(), "dense MFMA launch") ? ROASTER_EDEVICE : 0;
    }
    /* workgroups resident at once, by LDS (up to 2048 columns two per CU) */
    const size_t cap = (size_t)(2 * (lds + MM8_RED) <= 160 * 1024 ? 2 : 1) * rt().n_cu;
    const int nb = (int)(cols / RQK);
    /* waves per group: the split whose waves run the fewest super-blocks one
     * after the other (a few groups need several waves each to fill the CUs) */
    int split = 1;
    size_t best = 0;
    for (int sp = 1; sp <= MM8_W && sp <= nb; sp *= 2) {
        const size_t teams = cap * (MM8_W / sp), cost = (ng + teams - 1) / teams * ((nb + sp - 1) / sp);
        if (!best || cost < best) best = cost, split = sp;
    }
    size_t blocks = (ng + MM8_W / split - 1) / (MM8_W / split);
    if (blocks > cap) blocks = cap;
    const dim3 gd((unsigned)blocks), bd(MM8_T);
#define MM8(Q6_, P_) hipLaunchKernelGGL((dense_mm8_kernel<Q6_, P_>), gd, bd, lds, rt().stream, W, X, Y, (int)rows, (int)cols, T, split)
    if (T <= 4) {
        if (q6) MM8(true, 3);
        else MM8(false, 3);
    } else {
        if (q6) MM8(true, 2);
        else MM8(false, 2);
    }
#undef MM8
    return rt_check(hipGetLastError(), "dense MFMA launch") ? ROASTER_EDEVICE : 0;
}

/* eh = (g / (1 + exp(-g))) * u over n elements (kernels.c:2191, model.c:1124). */
__global__ void silu_mul_kernel(float *g, const float *u, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        const float a = g[i];
        g[i] = (a / (1.0f + expf(-a))) * u[i];
    }
}

/* f32 matvec rows (kernel_matvec_f32 / kernel_dot_f32): one wave per row. */
__global__ void __launch_bounds__(MV_THREADS) matvec_f32_kernel(const float *W, const float *x, float *y, size_t rows,
                                                                size_t cols)
{
    const int lane = threadIdx.x & 63;
    const size_t gw = (size_t)blockIdx.x * (MV_THREADS / 64) + (threadIdx.x >> 6);
    const size_t nw = (size_t)gridDim.x * (MV_THREADS / 64);
    for (size_t r = gw; r < rows; r += nw) {
        const float *row = W + r * cols;
        float acc = 0.0f;
        for (size_t i = lane; i < cols; i += 64) acc = fmaf(row[i], x[i], acc);
        acc = group_sum<64>(acc);
        if (lane == 0) y[r] = acc;
    }
}

/* ---- host launchers ------------------------------------------------------- */
int mv_launch(const MvJob *jobs_dev, int njobs, int ntasks)
{
    if (ntasks <= 0) return 0;
    const int wpb = MV_THREADS / 64;
    int blocks = (ntasks + wpb - 1) / wpb;
    if (blocks > 8 * rt().n_cu) blocks = 8 * rt().n_cu;
    hipLaunchKernelGGL(matvec_jobs_kernel, dim3(blocks), dim3(MV_THREADS), 0, rt().stream, jobs_dev, njobs, ntasks);
    return rt_check(hipGetLastError(), "matvec launch") ? ROASTER_EDEVICE : 0;
}

int mv_tasks_for(int rows, size_t cols)
{
    const int nb = (int)(cols / RQK);
    const int lpr = lanes_per_row(nb);
    const int rpw = 64 / lpr;
    return (rows + rpw - 1) / rpw;
}

extern "C" int roaster_matvec_q(const void *W, int q6, const float *X, float *Y, size_t rows, size_t cols, int T)
{
    std::lock_guard<std::recursive_mutex> g(rt_lock());
    if (rt_init_locked()) return ROASTER_EDEVICE;
    if (!W || !X || !Y || !rows || !cols || cols % RQK || cols > 4096 || T < 1 || T > 8 || rows > (size_t)INT32_MAX)
        return rt_fail(ROASTER_EINVAL, "roaster_matvec_q: need cols a multiple of 256 and <= 4096, 1 <= T <= 8");
    if (dense_mm8_takes((const uint8_t *)W, q6, cols, T))   /* several tokens: quants on MFMA */
        return dense_mm8_launch((const uint8_t *)W, q6, X, Y, rows, cols, T);
    const int nb = (int)(cols / RQK), rpw = 64 / lanes_per_row(nb);
    const size_t npass = (rows + rpw - 1) / rpw;
    /* a grid that is resident at once (registers: 5 workgroups per CU for Q6_K,
     * 6 for Q4_K, 3 past 8 super-blocks), its waves with equal numbers of
     * passes: the LM head with one token 104 us on 8 workgroups per CU, 99.5 on
     * 5, 96 with the next pass's loads under the current one's dots; 8192 rows
     * of 2048 7.8 -> 6.2 us */
    const size_t per_cu = nb > 8 ? 3 : q6 ? 5 : 6, waves = 4 * per_cu * rt().n_cu;
    const size_t iters = (npass + waves - 1) / waves, blocks = (npass + 4 * iters - 1) / (4 * iters);
    const size_t lds = T > 1 ? (size_t)T * cols * 4 + (size_t)T * (cols / 16) * 4 : 0;
    const dim3 gd((unsigned)blocks), bd(MV_THREADS);
    const uint8_t *w = (const uint8_t *)W;
    const int r = (int)rows, cc = (int)cols;
#define DMV(...) hipLaunchKernelGGL((dense_mv_kernel<__VA_ARGS__>), gd, bd, lds, rt().stream, w, X, Y, r, cc, T)
    if (mat_odd(w, q6)) {                              /* Q6_K blocks at odd addresses: loaded as they lie */
        if (nb <= 8 && T == 1) DMV(true, true, 1, false);
        else if (nb <= 8) DMV(true, false, 1, false);
        else if (T == 1) DMV(true, true, 2, false);
        else DMV(true, false, 2, false);
    } else if (nb <= 8) {
        if (q6 && T == 1) DMV(true, true, 1);
        else if (q6) DMV(true, false, 1);
        else if (T == 1) DMV(false, true, 1);
        else DMV(false, false, 1);
    } else {
        if (q6 && T == 1) DMV(true, true, 2);
        else if (q6) DMV(true, false, 2);
        else if (T == 1) DMV(false, true, 2);
        else DMV(false, false, 2);
    }
#undef DMV
    return rt_check(hipGetLastError(), "dense matvec launch") ? ROASTER_EDEVICE : 0;
}

/* roaster_dense_mfma_min_tokens: calls with at least this many tokens run
 * on dense_mm8_kernel; 0 = query. */
extern "C" int roaster_dense_mfma_min_tokens(int t)
{
    std::lock_guard<std::recursive_mutex> g(rt_lock());
    if (t > 0) g_dense_mfma_t = t;
    return g_dense_mfma_t;
}

int silu_mul_launch(float *g, const float *u, size_t n)
{
    int blocks = (int)((n + 255) / 256);
    if (blocks > 4096) blocks = 4096;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(silu_mul_kernel, dim3(blocks), dim3(256), 0, rt().stream, g, u, n);
    return rt_check(hipGetLastError(), "silu launch") ? ROASTER_EDEVICE : 0;
}

int matvec_f32_launch(const float *W, const float *x, float *y, size_t rows, size_t cols)
{
    size_t blocks = (rows + 3) / 4;
    if (blocks > 4096) blocks = 4096;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(matvec_f32_kernel, dim3((unsigned)blocks), dim3(MV_THREADS), 0, rt().stream, W, x, y, rows,
                       cols);
    return rt_check(hipGetLastError(), "matvec_f32 launch") ? ROASTER_EDEVICE : 0;
}
