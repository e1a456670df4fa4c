"""The expert kernel for tiles of few rows against the one for any rows, bit for
bit, at the edges of its row classes and with K that ends inside a stage; and
the bucket lists a call builds."""
import ctypes
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def note(msg):
    print(f"[case] {msg}", file=sys.stderr, flush=True)


# 1, 8, 9, 16, 17, 32 rows of the fullest expert (33: the other kernel both
# times); hidden and inter of one block, a stage, and blocks past a stage.
@pytest.mark.parametrize("rows", [1, 8, 9, 16, 17, 32, 33])
@pytest.mark.parametrize("hidden,inter", [(32, 32), (128, 96), (416, 160), (1024, 512)])
def test_few_row_tiles_equal_the_ring_kernel(rk, rows, hidden, inter, monkeypatch):
    note(f"MoE few rows={rows} hidden={hidden} inter={inter}")
    lib, r = rk.lib(), np.random.default_rng(rows + hidden)
    E, K = 5, 3
    w = [(r.standard_normal(s) * 0.05).astype(np.float32) for s in ((E, inter, hidden), (E, inter, hidden),
                                                                    (E, hidden, inter))]
    wid = rk.pack_moe_f32(*w)
    # every token goes to expert 3 and to two others in any order
    ids = np.stack([r.permutation([3, *r.choice([0, 1, 2, 4], 2, replace=False)]) for _ in range(rows)])
    ids = np.ascontiguousarray(ids, np.uint32)
    wts = np.ascontiguousarray(r.uniform(0.1, 1, (rows, K)), np.float32)
    x = r.standard_normal((rows, hidden)).astype(np.float32)
    dx, dy, da = rk.DeviceBuffer.from_array(x), rk.DeviceBuffer(x.nbytes), rk.DeviceBuffer(rows * K * inter * 4)
    got = []
    for knob in (None, "128"):
        if knob:
            monkeypatch.setenv("RK_MOE_ROWS", knob)
        assert lib.rk_moe_experts_dev(int(wid), dx.ptr, rows, K, ids.ctypes.data, wts.ctypes.data, dy.ptr, None) == 0
        rk.synchronize()
        y = dy.download((rows, hidden), np.float32)
        plan = ctypes.c_void_p()
        assert lib.rk_moe_plan_create(int(wid), rows, K, ids.ctypes.data, wts.ctypes.data, ctypes.byref(plan)) == 0
        assert lib.rk_moe_gate_up_dev(int(wid), plan, dx.ptr, da.ptr, None) == 0
        rk.synchronize()
        got.append((y, da.download((rows * K, inter), np.float32)))
        assert lib.rk_moe_plan_destroy(plan) == 0
    assert np.isfinite(got[0][0]).all()
    assert (got[0][0] == got[1][0]).all() and (got[0][1] == got[1][1]).all()


@pytest.mark.parametrize("s", [1, 300, 700])
def test_lists_of_a_call_and_of_a_plan(rk, s):
    """One copy and two copies of the lists, calls of changing size, repeated and missing
    experts, against the planned form; a bad id is refused before anything runs."""
    note(f"MoE lists s={s}")
    lib, r = rk.lib(), np.random.default_rng(s)
    E, K, H, I = 16, 4, 128, 64
    w = [(r.standard_normal(t) * 0.05).astype(np.float32) for t in ((E, I, H), (E, I, H), (E, H, I))]
    wid = rk.pack_moe_f32(*w)
    ids = np.ascontiguousarray(r.integers(0, E // 2, (s, K)) * 2, np.uint32)
    wts = np.ascontiguousarray(r.uniform(0.1, 1, (s, K)), np.float32)
    x = r.standard_normal((s, H)).astype(np.float32)
    dx, dy, dz = rk.DeviceBuffer.from_array(x), rk.DeviceBuffer(x.nbytes), rk.DeviceBuffer(x.nbytes)
    plan = ctypes.c_void_p()
    assert lib.rk_moe_plan_create(int(wid), s, K, ids.ctypes.data, wts.ctypes.data, ctypes.byref(plan)) == 0
    assert lib.rk_moe_experts_planned_dev(int(wid), plan, dx.ptr, dz.ptr, None) == 0
    assert lib.rk_moe_experts_dev(int(wid), dx.ptr, s, K, ids.ctypes.data, wts.ctypes.data, dy.ptr, None) == 0
    rk.synchronize()
    want = dz.download((s, H), np.float32)
    assert (dy.download((s, H), np.float32) == want).all()
    assert lib.rk_moe_plan_destroy(plan) == 0
    ids[-1, -1] = E
    assert lib.rk_moe_experts_dev(int(wid), dx.ptr, s, K, ids.ctypes.data, wts.ctypes.data, dy.ptr, None) == rk.RK_E_SHAPE
    assert (dy.download((s, H), np.float32) == want).all()
