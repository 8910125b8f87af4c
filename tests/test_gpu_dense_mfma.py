"""roaster_matvec_q of several tokens on MFMA (dense_mm8_kernel) where its splits
and operands can go wrong, against the oracle: one row, a row past a 16-row
group, groups that need every wave of a workgroup and groups that fill the
grid with one wave each; one, three and nine super-blocks (a wave's members and
items ragged); 4 tokens in three fp16 parts and 5 in two, and the ends; Q6_K
scales over the whole int8 range (sc (q - 32) past 2048 needs the second weight
operand).  One token runs the pipelined matvec on the same shapes.

Bar 5e-6 of max|y|: 22-bit activations (2^-22 per product, random in sign) and
f32 sums of up to 3584 terms on both sides, about 1e-6 each."""
import ctypes as C

import numpy as np
import pytest

import roaster_amd as R
from gpu_util import Dev, alloc_w
from oracle import oracle as O
from test_gpu_dense import run, weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q6", [0, 1])
@pytest.mark.parametrize("rows,cols", [(1, 256), (17, 2304), (300, 768), (33000, 256), (70001, 768)])
def test_splits(q6, rows, cols):
    W = weights(q6, rows, cols, 70 + cols)
    if q6:
        b = W.reshape(-1, R.Q6K_BYTES)
        b[:, 192:208] = np.random.default_rng(3).integers(0, 256, (len(b), 16), dtype=np.uint8)
    X = np.stack([R.synth_normal(71, R.synth_stream(t, cols, 5), cols) for t in range(8)])
    X[1, : cols // 2] *= 2.0 ** 12                # super-blocks of very different size
    ref = [O.matvec(q6, W, x, rows, cols) for x in X]
    for T in (1, 2, 4, 5, 8):
        Y = run(q6, W, X[:T], rows, cols)
        for t in range(T):
            err = np.max(np.abs(Y[t] - ref[t])) / np.max(np.abs(ref[t]))
            assert err <= 5e-6, (T, t, err)


@pytest.mark.parametrize("q6", [0, 1])
@pytest.mark.parametrize("rows,cols", [(16368, 256), (16369, 512), (16400, 3328), (16400, 3584)])
def test_staged(q6, rows, cols):
    """The weights staged in LDS (from 1024 16-row groups on 256 CUs): the last
    size before and the first after, the widest that fits with Q6_K and one
    past it."""
    W = weights(q6, rows, cols, 90 + cols)
    X = np.stack([R.synth_normal(91, R.synth_stream(t, cols, 5), cols) for t in range(6)])
    ref = {t: O.matvec(q6, W, X[t], rows, cols) for t in (0, 1, 5)}
    for T in (2, 6):
        Y = run(q6, W, X[:T], rows, cols)
        for t in (t for t in ref if t < T):
            err = np.max(np.abs(Y[t] - ref[t])) / np.max(np.abs(ref[t]))
            assert err <= 5e-6, (T, t, err)


@pytest.mark.parametrize("off", [1, 2, 3])
@pytest.mark.parametrize("q6", [0, 1])
@pytest.mark.parametrize("rows,cols", [(37, 512), (37, 2304), (16400, 256)])
def test_unaligned_matrix(q6, rows, cols, off):
    """A matrix that begins at any byte gives what it gives at an aligned address
    (the Q6_K kernels that read aligned dwords take even ones only)."""
    W = weights(q6, rows, cols, 95 + cols)
    X = np.stack([R.synth_normal(96, R.synth_stream(t, cols, 5), cols) for t in range(8)])
    moved = Dev(np.concatenate([np.zeros(off, np.uint8), W]))
    for T in (1, 2, 5, 8):
        Y = run(q6, W, X[:T], rows, cols)
        dx, dy = Dev(X[:T]), Dev(nbytes=T * rows * 4, shape=(T, rows))
        R.check(R.lib().roaster_matvec_q(moved.p + off, q6, dx.p, dy.p, rows, cols, T), "matvec_q")
        R.check(R.lib().roaster_sync(), "sync")
        err = np.max(np.abs(dy.get() - Y)) / np.max(np.abs(Y))
        assert err <= 5e-6, (T, err)


@pytest.mark.parametrize("q6", [0, 1])
def test_unaligned_matrix_batch(q6):
    """The same through kernel_matmul_quant_batch, from weight memory at an odd address."""
    rows, cols, T = 100, 512, 5
    W = weights(q6, rows, cols, 97)
    X = np.stack([R.synth_normal(98, R.synth_stream(t, cols, 5), cols) for t in range(T)])
    p = alloc_w(np.concatenate([np.zeros(1, np.uint8), W]))
    Y = np.empty((T, rows), np.float32)
    job = R.KernelMatmulJob(q6, p + 1, X.ctypes.data, Y.ctypes.data, rows, cols, T)
    assert R.lib().kernel_matmul_quant_batch(C.byref(job), 1) == 0
    for t in range(T):
        ref = O.matvec(q6, W, X[t], rows, cols)
        assert np.max(np.abs(Y[t] - ref)) <= 5e-6 * np.max(np.abs(ref))


@pytest.mark.parametrize("T", [4, 5, 8])
def test_minima_keep_f32_sums(T):
    """Q4_K's minimum term takes the sub-block sums with all 24 bits of an f32: scales
    of zero and one minimum of one per super-block leave y = -dmin x for an x with a
    single 24-bit entry in each super-block's sub-block, here exactly."""
    rows, cols = 64, 512
    W = np.zeros((rows, cols // 256, R.Q4K_BYTES), np.uint8)
    W[:, 0, 2:4] = np.frombuffer(np.float16(1.0).tobytes(), np.uint8)     # dmin of the first super-block
    sub = np.arange(rows) % 8
    for r, s in enumerate(sub):
        W[r, 0, 8 + s] = 1 if s < 4 else 1 << 4                           # minimum 1 in sub-block s
    rng = np.random.default_rng(6)
    X = np.zeros((T, cols), np.float32)
    big = rng.integers(2 ** 23, 2 ** 24, (T, 8)) | 1
    for t in range(T):
        X[t, 32 * np.arange(8) + t] = big[t]
    Y = run(0, W.reshape(-1), X, rows, cols)
    np.testing.assert_array_equal(Y, -big[:, sub].astype(np.float32))
