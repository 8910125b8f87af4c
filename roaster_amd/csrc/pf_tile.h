/*
 * pf_tile.h -- device helpers shared by the MFMA GEMMs, first those that read weights in
 * the MFMA tile layout (tile.h): raw lane records and their loads, the fp16
 * bit-pattern conversions of quants, the permuted K order of a super-block,
 * power-of-two scale exponents and the block numbering of a launch.
 */
#ifndef ROASTER_PF_TILE_H
#define ROASTER_PF_TILE_H

#include "gemm.h"
#include "tile.h"

static __device__ __forceinline__ float pf_silu_mul(float g, float u) { return (g / (1.0f + expf(-g))) * u; }
/* The exponent s of row_scale(amax): fwd = 2^s, clamped to [-100, 100]. */
static __device__ __forceinline__ int pf_scale_exp(float amax)
{
    const int s = (int)((__builtin_bit_cast(uint32_t, amax) >> 23) & 255u) - 127 - 14;
    return s < -100 ? -100 : (s > 100 ? 100 : s);
}
/* SiLU(g) * u with the hardware exp and reciprocal (v_exp_f32, v_rcp_f32: a
 * few ulp in f32; the result is rounded to fp16 for the next GEMM anyway). */
static __device__ __forceinline__ float pf_silu_mul_fast(float g, float u)
{
    return g * __builtin_amdgcn_rcpf(1.0f + __expf(-g)) * u;
}

/* A workgroup barrier that orders LDS accesses only: every wave's LDS reads
 * and writes complete, global loads may stay in flight (__syncthreads()
 * waits for those too). */
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

/* Virtual block id: blocks b < R = ntiles * nblk run; on a grid dispatched
 * round-robin over the 8 XCDs, XCD b % 8 takes the contiguous range of
 * virtual ids [(b % 8) * R / 8, ...), so the n-blocks of one tile and the
 * consecutive tiles of one expert share an L2. */
__device__ __forceinline__ int pf_virtual_block(int b, int R)
{
    return (R & 7) ? b : (b & 7) * (R >> 3) + (b >> 3);
}

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

/* One lane's raw share of a super-block: half h (weights 128h .. 128h+127). */
struct RawQ6 { uint32_t L[16], Hh[8], S[2], d; };
struct RawQ4 { uint32_t hd[4], Q[16]; };
template <bool Q6> struct RawOf;
template <> struct RawOf<true> { typedef RawQ6 T; };
template <> struct RawOf<false> { typedef RawQ4 T; };

/* fp16 pairs (1024 + b0, 1024 + b1) and (1024 + b2, 1024 + b3) of the bytes of q. */
__device__ __forceinline__ f16x2 magic_lo(uint32_t q) { return __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(q, 0x64646464u, 0x00050004u)); }
__device__ __forceinline__ f16x2 magic_hi(uint32_t q) { return __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(q, 0x64646464u, 0x00070006u)); }

/* Natural position p (multiple of 4) of a super-block -> its permuted slot. */
__device__ __forceinline__ int perm_slot4(int p)
{
    const int h = p >> 7, q = p & 127, hi = q >> 6, r = q & 63;
    const int l0 = r < 32 ? r : r - 32, i0 = r < 32 ? 0 : 4;
    return (8 * hi + (l0 >> 2)) * 16 + 8 * h + i0;
}

__device__ __forceinline__ void tile_load(RawQ6 &r, const uint8_t *tile, int lane)
{
    const uint8_t *p = tile + 16 * lane;
    uint4 s[6];
#pragma unroll
    for (int i = 0; i < 6; i++) s[i] = gld_u4(p + 1024 * i);
    const uint3 s6 = gld_u3(p + 1024 * 6);          /* the record's last dword is padding */
#pragma unroll
    for (int i = 0; i < 4; i++) {
        r.L[4 * i] = s[i].x; r.L[4 * i + 1] = s[i].y; r.L[4 * i + 2] = s[i].z; r.L[4 * i + 3] = s[i].w;
    }
#pragma unroll
    for (int i = 0; i < 2; i++) {
        r.Hh[4 * i] = s[4 + i].x; r.Hh[4 * i + 1] = s[4 + i].y; r.Hh[4 * i + 2] = s[4 + i].z; r.Hh[4 * i + 3] = s[4 + i].w;
    }
    r.S[0] = s6.x;
    r.S[1] = s6.y;
    r.d = s6.z & 0xFFFFu;
}

__device__ __forceinline__ void tile_load(RawQ4 &r, const uint8_t *tile, int lane)
{
    const uint8_t *p = tile + 16 * lane;
    uint4 s[5];
#pragma unroll
    for (int i = 0; i < 5; i++) s[i] = gld_u4(p + 1024 * i);
    r.hd[0] = s[0].x; r.hd[1] = s[0].y; r.hd[2] = s[0].z; r.hd[3] = s[0].w;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        r.Q[4 * i] = s[1 + i].x; r.Q[4 * i + 1] = s[1 + i].y; r.Q[4 * i + 2] = s[1 + i].z; r.Q[4 * i + 3] = s[1 + i].w;
    }
}

#endif
