"""GPU check of the two ways prefill buckets and plans: by the last workgroup of
the token kernel (up to 512 tokens) and by two more kernels (above).

One set of 513 tokens goes through the second way; its first T tokens go
through the first, T about the word size of the bit map, a batch of picks (256
tokens) and the line.  A token's row of Y depends on neither its tile nor its
neighbours (with Q6_K down matrices and E < 8 T every call has the same GEMMs), so the
rows are equal bit for bit wherever every list, rank, offset and tile is right.
Routes are uniform or on twelve experts (lists of up to T tokens).  Three calls
a case: the workgroup counter has to be back at zero.

logits_out may be logits_in: each token's logits, biased, replace its own and
nothing else changes, also where T leaves waves of the last workgroup idle (T not
a multiple of 4; both ways)."""
import ctypes as C

import numpy as np
import pytest

import roaster_amd as R
from gpu_util import Dev, SynthTable, prefill

pytestmark = pytest.mark.gpu

E, H, T_ALL = 256, 256, 513


@pytest.fixture(scope="module")
def table():
    t = SynthTable(21, n_experts=E, hidden=H, inter=256, q6=(0, 0, 1), sh_q6=(0, 0, 1))
    yield t
    t.destroy()


@pytest.fixture(scope="module", params=["uniform", "twelve"])
def whole(table, request):
    rng = np.random.default_rng(2)
    X = rng.standard_normal((T_ALL, H)).astype(np.float32)
    lg = rng.standard_normal((T_ALL, E)).astype(np.float32)
    if request.param == "twelve":
        lg[:, rng.permutation(E)[:12]] += 100.0
    return X, lg, prefill(table, X, logits_in=lg)


@pytest.mark.parametrize("T", [33, 63, 64, 65, 255, 256, 257, 511, 512])
def test_one_launch_buckets(table, whole, T):
    X, lg, (Y, _, ids, w, _) = whole
    for _ in range(3):
        Yt, _, idt, wt, counts = prefill(table, X[:T], logits_in=lg[:T])
        assert np.array_equal(idt, ids[:T]) and np.array_equal(wt, w[:T])
        assert np.array_equal(counts, np.bincount(idt.ravel(), minlength=E))
        assert np.array_equal(Yt, Y[:T])


@pytest.mark.parametrize("T", [1, 2, 3, 5, 45, 510, 513])
def test_logits_in_place(table, T):
    rng = np.random.default_rng(T)
    X = rng.standard_normal((T, H)).astype(np.float32)
    lg = rng.standard_normal((T, E)).astype(np.float32)
    b = (4 * rng.standard_normal(E)).astype(np.float32)
    Y, out, ids, w, counts = prefill(table, X, logits_in=lg, bias=b)
    assert np.array_equal(out, lg + b)
    dx, dl, db, dy = Dev(X), Dev(lg), Dev(b), Dev(nbytes=T * H * 4, shape=(T, H))
    di, dw = Dev(nbytes=T * 32, dtype=np.int32, shape=(T, 8)), Dev(nbytes=T * 32, shape=(T, 8))
    o = R.RoasterPrefillOpts(R.PREC_F16, dl.p, db.p, dl.p, di.p, dw.p, None)
    R.check(R.lib().roaster_moe_prefill(table.t, 0, dx.p, T, dy.p, C.byref(o)), "prefill")
    R.check(R.lib().roaster_sync(), "sync")
    assert np.array_equal(dl.get(), out)
    assert np.array_equal(di.get(), ids) and np.array_equal(dw.get(), w)
    assert np.array_equal(dy.get(), Y)
