"""The order of the sums: of the scaled int8 products (groups ascending, whatever kernel a
call's size takes: rows do not depend on the batch they come in), and of fused against plain
products, through the C ABI."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def note(msg):
    print(f"[case] {msg}", file=sys.stderr, flush=True)


def q8(rk, orc, w):
    n, k = w.shape
    return rk.pack_q8_0(orc.q8_0_blocks(*orc.q8_0_quantize(w)), n, k)


def product(rk, fn, wid, da, ds, a_group, m, k, n, f16):
    dc = rk.DeviceBuffer(m * n * (2 if f16 else 4))
    assert fn(int(wid), da.ptr, ds.ptr, a_group, m, k, dc.ptr, None) == 0, rk.lib().rk_last_error()
    rk.synchronize()
    return dc.download((m, n), np.uint16 if f16 else np.uint32)


# K of one to three stages, ending inside a stage, and of many stages; N odd, from a few
# tiles (one round of workgroups at every M) to more than a round at most M; group 32
# with fp16 scales (Q8_0) and with f32 scales, 64, 128.
@pytest.mark.parametrize("k,n", [(128, 33), (416, 200), (1024, 3072), (3072, 1000), (4288, 70), (128, 4100),
                                 (288, 1300), (416, 3001)])
@pytest.mark.parametrize("group", ["q8_0", 32, 64, 128])
def test_int8_rows_do_not_depend_on_the_batch(rk, orc, monkeypatch, k, n, group):
    g = 32 if group == "q8_0" else group
    k = -(-k // g) * g
    r = np.random.default_rng(k + n + g)
    x = r.standard_normal((260, k)).astype(np.float32)
    w = (r.standard_normal((n, k)) * 0.02).astype(np.float32)
    wid = q8(rk, orc, w) if group == "q8_0" else rk.pack_i8(w, g)
    for a_group in (g, k):
        note(f"int8 rows k={k} n={n} group={group} a_group={a_group}")
        aq, a_s = orc.quantize_rows(x, a_group)
        da, ds = rk.DeviceBuffer.from_array(aq), rk.DeviceBuffer.from_array(a_s)
        for f16 in (False, True):
            fn = rk.lib().rk_matmul_w8a8_f16out_dev if f16 else rk.lib().rk_matmul_w8a8_dev
            monkeypatch.setenv("RK_SKINNY", "0")
            want = product(rk, fn, wid, da, ds, a_group, len(x), k, n, f16)
            monkeypatch.delenv("RK_SKINNY")
            for m in (1, 12, 17, 33, 128, 256):
                assert (product(rk, fn, wid, da, ds, a_group, m, k, n, f16) == want[:m]).all(), (m, f16)


def test_int8_groups_are_summed_in_ascending_order(rk, orc):
    """acc = fma(P_g, w_s[n, g], acc) over ascending g, then a_s[m]·acc, in numpy: a product of a 20-bit
    and a 24-bit number is exact in 64 bits, and so the sum is rounded twice once in 2^29."""
    m, k, n = 12, 3072, 96
    note(f"int8 ascending order m={m} k={k} n={n}")
    r = np.random.default_rng(5)
    x, w = r.standard_normal((m, k)).astype(np.float32), (r.standard_normal((n, k)) * 0.02).astype(np.float32)
    wq, wd = orc.q8_0_quantize(w)
    d = wd.view(np.float16).astype(np.float64)
    aq, a_s = orc.quantize_rows(x, k)
    p = np.einsum("mbj,nbj->bmn", aq.reshape(m, -1, 32).astype(np.int64), wq.reshape(n, -1, 32).astype(np.int64))
    acc = np.zeros((m, n), np.float32)
    for b in range(k // 32):
        acc = (p[b].astype(np.float64) * d[None, :, b] + acc).astype(np.float32)
    want = a_s.reshape(m, 1).astype(np.float32) * acc
    got = product(rk, rk.lib().rk_matmul_w8a8_dev, q8(rk, orc, w), rk.DeviceBuffer.from_array(aq),
                  rk.DeviceBuffer.from_array(a_s), k, m, k, n, False)
    assert (got == want.view(np.uint32)).all()


# Rows on both sides of the limits of the plain and of the fused form.
@pytest.mark.parametrize("m,k,n", [(30, 416, 100), (161, 1024, 3072), (200, 416, 1000), (256, 1024, 3072),
                                   (400, 128, 3000)])
def test_int8_gate_up_equals_products_then_glue(rk, orc, monkeypatch, m, k, n):
    note(f"int8 gate|up m={m} k={k} n={n}")
    lib, r = rk.lib(), np.random.default_rng(m + n)
    x = r.standard_normal((m, k)).astype(np.float32)
    w = [(r.standard_normal((n, k)) * 0.05).astype(np.float32) for _ in range(2)]
    aq, a_s = orc.quantize_rows(x, k)
    da, ds = rk.DeviceBuffer.from_array(aq), rk.DeviceBuffer.from_array(a_s)
    g, u = [product(rk, lib.rk_matmul_w8a8_dev, q8(rk, orc, t), da, ds, k, m, k, n, False).view(np.float32) for t in w]
    wid = rk.pack_q8_0_glu(*[orc.q8_0_blocks(*orc.q8_0_quantize(t)) for t in w], n, k)
    dy = rk.DeviceBuffer(m * n * 4)
    for kind, glue in ((rk.GLU_SILU, rk.silu_mul), (rk.GLU_GELU, rk.gelu_mul)):
        assert lib.rk_matmul_w8a8_glu_dev(int(wid), da.ptr, ds.ptr, m, k, kind, dy.ptr, 0, None) == 0
        rk.synchronize()
        assert (dy.download((m, n), np.float32) == glue(g, u)).all()
        half = []  # fp16 results: those of the tiled kernels
        for knob in ("1", "0"):
            monkeypatch.setenv("RK_SKINNY", knob)
            assert lib.rk_matmul_w8a8_glu_dev(int(wid), da.ptr, ds.ptr, m, k, kind, dy.ptr, 1, None) == 0
            rk.synchronize()
            half.append(dy.download((m, n), np.uint16))
        monkeypatch.delenv("RK_SKINNY")
        assert (half[0] == half[1]).all()


# K below 768 in each tile the few-tile kernel has; from there one row tile, tiles as wide
# as a plain product's and twice as wide, K over eight waves, over four (the fused form with
# four accumulator sets: 16, 13, 19, 25 and 14 stages, full and ragged tiles) and unsplit.
@pytest.mark.parametrize("m,k,n", [(24, 128, 1500), (40, 96, 1500), (20, 192, 4200), (12, 136, 4300), (8, 1024, 3072),
                                   (33, 1024, 3072), (64, 1024, 3072), (128, 1024, 3072), (256, 776, 1000),
                                   (20, 1160, 4300), (100, 1160, 1900), (70, 776, 3001), (450, 1600, 1000),
                                   (500, 1160, 1000), (257, 888, 1000), (300, 1024, 3072)])
def test_fp16_gate_up_equals_products_then_glue(rk, orc, m, k, n):
    note(f"fp16 gate|up m={m} k={k} n={n}")
    lib, r = rk.lib(), np.random.default_rng(m + k + n)
    x = r.standard_normal((m, k)).astype(np.float16)
    w = [(r.standard_normal((n, k)) * 0.05).astype(np.float32) for _ in range(2)]
    dx, dy = rk.DeviceBuffer.from_array(x.view(np.uint16)), rk.DeviceBuffer(m * n * 4)
    prods = []
    for t in w:
        assert lib.rk_matmul_f16_dev(int(rk.pack(t)), dx.ptr, m, k, dy.ptr, None) == 0, lib.rk_last_error()
        rk.synchronize()
        prods.append(dy.download((m, n), np.uint16).view(np.float16))
        ref = x.astype(np.float64) @ t.astype(np.float16).astype(np.float64).T
        # f32 sums of K products (1e-5 of the largest, as in the few-tile tests), then one fp16 rounding
        assert (np.abs(prods[-1] - ref) <= 1e-5 * np.abs(ref).max() + 2.0 ** -11 * np.abs(ref)).all()
    wid = rk.pack_f16_glu(*w)
    for kind, glue in ((rk.GLU_SILU, rk.silu_mul), (rk.GLU_GELU, rk.gelu_mul)):
        want = glue(*[p.astype(np.float32) for p in prods])
        for f16 in (0, 1):
            assert lib.rk_matmul_f16_glu_dev(int(wid), dx.ptr, m, k, kind, dy.ptr, f16, None) == 0
            rk.synchronize()
            if f16:  # (the glue op on fp16 operands computes in f32 and rounds once)
                assert (dy.download((m, n), np.uint16) == glue(*prods).view(np.uint16)).all()
            else:
                assert (dy.download((m, n), np.float32) == want).all()


# Calls whose rows move in chunks: a short last chunk (688 + 12 rows, 1376 + 24), and chunks that by
# themselves would split K over eight waves where the whole call splits it over four.
@pytest.mark.parametrize("m,k,n", [(700, 1024, 3072), (1400, 1024, 3072), (9000, 768, 32)])
def test_fp16_rows_of_a_host_call_follow_one_order(rk, m, k, n):
    note(f"fp16 host call m={m} k={k} n={n}")
    lib, r = rk.lib(), np.random.default_rng(m + n)
    x = r.standard_normal((m, k)).astype(np.float16)
    wid = rk.pack((r.standard_normal((n, k)) * 0.05).astype(np.float32))
    dx, dy = rk.DeviceBuffer.from_array(x.view(np.uint16)), rk.DeviceBuffer(m * n * 2)
    assert lib.rk_matmul_f16_dev(int(wid), dx.ptr, m, k, dy.ptr, None) == 0, lib.rk_last_error()
    rk.synchronize()
    want = dy.download((m, n), np.uint16).view(np.float16)
    assert (rk.matmul(x.astype(np.float32), wid) == want.astype(np.float32)).all()
    c = np.empty((m, n), np.float16)
    assert lib.rk_matmul_f16(int(wid), x.ctypes.data, m, k, c.ctypes.data) == 0, lib.rk_last_error()
    assert (c == want).all()
