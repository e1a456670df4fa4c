"""GPU parity of the group-wise int8 path (weight groups of 64 and 128, and the
activation quantizer's group sizes) against the oracle, through the C ABI."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def note(msg):
    print(f"[case] {msg}", file=sys.stderr, flush=True)


def quantize_dev(rk, x, group):
    m, k = x.shape
    dx, dq, ds = rk.DeviceBuffer.from_array(x), rk.DeviceBuffer(m * k), rk.DeviceBuffer(m * (k // group) * 4)
    assert rk.lib().rk_quantize_rows_dev(dx.ptr, m, k, group, dq.ptr, ds.ptr, None) == 0, rk.lib().rk_last_error()
    rk.synchronize()
    return dq, ds


@pytest.mark.parametrize("group", [32, 64, 96, 128, 256, 512])
@pytest.mark.parametrize("m", [1, 3, 70])
def test_quantize_groups_is_bit_exact(rk, orc, m, group):
    k = 3 * group
    note(f"quantize_rows m={m} k={k} group={group}")
    r = np.random.default_rng(m * group)
    x = (r.standard_normal((m, k)) * r.uniform(0, 8, (m, k))).astype(np.float32)
    x[0, :group] = 0.0  # a zero group: the scale floor
    x[-1, -1] = np.nan  # ignored by the group maximum, as fmaxf ignores it
    dq, ds = quantize_dev(rk, x, group)
    x[-1, -1] = 0.0
    q, s = orc.quantize_rows(x, group)
    got = dq.download((m, k), np.int8)
    if group != 96:  # (one workgroup per row: its maximum is NaN there)
        assert (ds.download((m, k // group), np.float32).view(np.uint32) == s.view(np.uint32)).all()
        got[-1, -1] = q[-1, -1] = 0
        assert (got == q).all()
    else:
        assert (got[:, :-group] == q[:, :-group]).all()


# The pipelined kernel: its 64x64 tiles at their edges, one group, an odd number of groups (64: a
# stage that holds one group), columns and rows that end inside a tile (those of few tiles only reach it
# with RK_SKINNY=0; as they are they run on the few-tile kernels), and its 128x64 tiles with two stages and
# with ten, more than its ring of three holds, of which the last is half filled (group 64).
SHAPES = [(1, 128, 1), (63, 192, 65), (65, 384, 200), (129, 1152, 1000), (2050, 256, 1090), (2050, 1216, 1090)]


@pytest.mark.parametrize("group", [64, 128])
@pytest.mark.parametrize("m,k,n,skinny", [(*s, v) for s in SHAPES for v in ("1", "0") if v == "1" or s[0] < 2000])
def test_group_gemm(rk, orc, monkeypatch, m, k, n, skinny, group):
    monkeypatch.setenv("RK_SKINNY", skinny)
    if k % group:
        k += group - k % group
    note(f"group gemm m={m} k={k} n={n} group={group} RK_SKINNY={skinny}")
    r = np.random.default_rng(m + k + n + group)
    x = r.standard_normal((m, k)).astype(np.float32)
    w = (r.standard_normal((n, k)) * 0.02).astype(np.float32)
    wid = rk.pack_i8(w, group)
    wq, ws = orc.quantize_rows(w, group)
    for a_group in (group, k):
        aq, a_s = orc.quantize_rows(x, a_group)
        da, ds = rk.DeviceBuffer.from_array(aq), rk.DeviceBuffer.from_array(a_s)
        ref = orc.emu_matmul_gw(aq, a_s, a_group, wq, ws, group)
        for f16out in (False, True):
            dc = rk.DeviceBuffer(m * n * (2 if f16out else 4))
            fn = rk.lib().rk_matmul_w8a8_f16out_dev if f16out else rk.lib().rk_matmul_w8a8_dev
            assert fn(int(wid), da.ptr, ds.ptr, a_group, m, k, dc.ptr, None) == 0, rk.lib().rk_last_error()
            rk.synchronize()
            if f16out:  # one rounding of 2^-11 on top
                got = dc.download((m, n), np.uint16).view(np.float16).astype(np.float32)
                assert (np.abs(got - ref) <= 2.0 ** -11 * np.abs(ref) + 1e-5 * np.abs(ref).max()).all()
            else:  # f32 sums of k / group terms, each rounded at 2^-24
                got = dc.download((m, n), np.float32)
                assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()
