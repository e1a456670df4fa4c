"""GPU parity of the attention kernel for few query rows (keys split over waves
and workgroups, V read untransposed) against the oracle."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def note(msg):
    print(f"[case] {msg}", file=sys.stderr, flush=True)


def run(rk, q, k, v, h, kv, d, scale, softcap=0.0, mode=0, window=-1, q0=0, k0=0):
    n_q, n_kv = q.shape[0], k.shape[0]
    b = [rk.DeviceBuffer.from_array(t.view(np.uint16)) for t in (q, k, v)]
    o = rk.DeviceBuffer(n_q * h * d * 2)
    assert rk.lib().rk_attention_dev(b[0].ptr, b[1].ptr, b[2].ptr, n_q, n_kv, h, kv, d, scale, softcap, mode, window,
                                     q0, k0, o.ptr, None) == 0, rk.lib().rk_last_error()
    rk.synchronize()
    return o.download((n_q, h * d), np.uint16).view(np.float16).astype(np.float32)


def data(seed, n_q, n_kv, h, kv, d):
    r = np.random.default_rng(seed)
    return [r.standard_normal(s).astype(np.float16) for s in ((n_q, h * d), (n_kv, kv * d), (n_kv, kv * d))]


# fp16 results of f32 sums against the oracle's: one rounding (2^-11) and P in
# two fp16 halves (2^-22); the bound of the other attention tests
def check(orc, got, ref):
    assert np.isfinite(got).all()
    assert orc.cosine(got, ref) >= 0.9999 and orc.max_rel(got, ref) <= 1e-2


# Every head dim; one row and a full row tile; key counts of less than a chunk,
# a chunk's edge, one chunk per wave and several per wave over several splits.
@pytest.mark.parametrize("d", [32, 48, 64, 72, 80, 96, 112, 128, 256])
@pytest.mark.parametrize("n_q,n_kv,h,kv", [(1, 1, 1, 1), (1, 33, 8, 2), (4, 131, 8, 2), (17, 1000, 2, 1),
                                           (1, 4097, 4, 4), (64, 70, 1, 1), (150, 4100, 14, 1)])
def test_rows_head_dims_and_edges(rk, orc, d, n_q, n_kv, h, kv):
    note(f"rows attention d={d} n_q={n_q} n_kv={n_kv} {h}/{kv}")
    q, k, v = data(d + n_kv, n_q, n_kv, h, kv, d)
    q0 = max(0, n_kv - n_q)
    for mode in (0, 1):
        got = run(rk, q, k, v, h, kv, d, d ** -0.5, mode=mode, q0=q0)
        check(orc, got, orc.attention_ref(q, k, v, h, kv, d, d ** -0.5, 0.0, mode, -1, q0, 0))
        # the merge order is the split order: the same bits each time
        assert (got == run(rk, q, k, v, h, kv, d, d ** -0.5, mode=mode, q0=q0)).all()


@pytest.mark.parametrize("mode,window,softcap,q0,k0", [
    (2, 40, 0.0, 500, 0), (3, 100, 0.0, 600, 0), (3, 64, 20.0, 700, 300),
    (1, -1, 0.0, 0, 100),    # rows before the first key: no visible key, the mean of V
    (2, 8, 0.0, 5000, 0),    # a window past the last key
    (1, -1, 30.0, 2000, 0),
])
def test_rows_masks(rk, orc, mode, window, softcap, q0, k0):
    note(f"rows attention mode={mode} window={window} softcap={softcap} q0={q0} k0={k0}")
    h, kv, d, n_q, n_kv = 6, 2, 64, 9, 777
    q, k, v = data(mode + q0 + k0, n_q, n_kv, h, kv, d)
    got = run(rk, q, k, v, h, kv, d, 0.125, softcap, mode, window, q0, k0)
    check(orc, got, orc.attention_ref(q, k, v, h, kv, d, 0.125, softcap, mode, window, q0, k0))


def test_rows_large_scores(rk, orc):
    """Scores in the hundreds, rising along the keys: the running maximum moves in every chunk."""
    note("rows attention, rising scores")
    h, kv, d, n_kv = 4, 1, 128, 2000
    q, k, v = data(7, 1, n_kv, h, kv, d)
    k = (k * np.linspace(0.1, 6, n_kv)[:, None]).astype(np.float16)
    check(orc, run(rk, q, k, v, h, kv, d, 1.0), orc.attention_ref(q, k, v, h, kv, d, 1.0))


def test_rows_unaligned_v_keeps_its_kernel(rk, orc):
    """V at an address that is not a multiple of 16 bytes goes to the kernel that takes it."""
    note("rows attention, V 4 bytes off")
    h, kv, d, n_q, n_kv = 4, 2, 64, 3, 200
    q, k, v = data(5, n_q, n_kv, h, kv, d)
    b = [rk.DeviceBuffer.from_array(t.view(np.uint16)) for t in (q, k)]
    dv = rk.DeviceBuffer.from_array(np.concatenate([np.zeros(2, np.uint16), v.view(np.uint16).reshape(-1)]))
    o = rk.DeviceBuffer(n_q * h * d * 2)
    assert rk.lib().rk_attention_dev(b[0].ptr, b[1].ptr, dv.ptr + 4, n_q, n_kv, h, kv, d, 0.125, 0.0, 0, -1, 0, 0,
                                     o.ptr, None) == 0, rk.lib().rk_last_error()
    rk.synchronize()
    check(orc, o.download((n_q, h * d), np.uint16).view(np.float16).astype(np.float32),
          orc.attention_ref(q, k, v, h, kv, d, 0.125))
