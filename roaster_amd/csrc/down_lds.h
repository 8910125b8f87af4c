/*
 * down_lds.h -- the dynamic LDS of dec_down_kernel: n slots' SiLU*up rows of I
 * floats, then their sums over runs of 16.  The launch sizes the allocation and
 * the kernels index it by this structure alone (n is 9 in the decode path and
 * the call's expert count, 1 to 9, in kernel_ffn_fused).
 */
#ifndef ROASTER_DOWN_LDS_H
#define ROASTER_DOWN_LDS_H

#include <stddef.h>

#ifdef __HIPCC__
#define DOWN_LDS_FN __host__ __device__ inline
#else
#define DOWN_LDS_FN inline
#endif

struct DownLds {
    int n, I;
    DOWN_LDS_FN int units() const { return n * I / 4; }              /* 16-byte units of the rows */
    DOWN_LDS_FN int unit(int k) const { return k < units() ? k : units() - 1; }
    DOWN_LDS_FN int sums_at() const { return n * I; }                /* floats before the sums */
    DOWN_LDS_FN int sums() const { return n * (I / 16); }
    DOWN_LDS_FN size_t bytes() const { return (size_t)(sums_at() + sums()) * 4; }
};

#endif
