"""GPU parity of the GEMM kernels for few output tiles (int8 and fp16, plain and
gate|up) against the oracle: rows, columns and K at the edges of tiles and stages."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# M, K, N: one row, the 16-row tile edges, K of one block / less than one stage
# per wave / ends inside a stage / more than two stages per wave; and more tiles
# than one round of workgroups, ragged both ways (the last, 16-row tiles walked by
# one wave each).
SHAPES = [(1, 32, 1), (16, 160, 40), (33, 1152, 33), (32, 416, 200), (5, 3072, 96), (95, 4128, 65), (100, 416, 3001)]


def note(msg):
    print(f"[case] {msg}", file=sys.stderr, flush=True)


def dev(rk, a):
    return rk.DeviceBuffer.from_array(a)


def close(got, ref, f16):
    # sums of K products in another order: K·2^-24 of the largest sum at the
    # very most (1e-5 covers K = 4128 with rounding at random); fp16 outputs
    # round once more
    tol = 1e-5 * np.abs(ref).max() + (2.0 ** -10 * np.abs(ref) if f16 else 0)
    assert (np.abs(got - ref) <= tol).all(), np.abs(got - ref).max()


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("group", [32, 64, 128])
def test_skinny_i8(rk, orc, m, k, n, group):
    k = -(-k // group) * group
    note(f"skinny int8 m={m} k={k} n={n} group={group}")
    r = np.random.default_rng(m + k + n + group)
    x = r.standard_normal((m, k)).astype(np.float32)
    w = (r.standard_normal((n, k)) * 0.02).astype(np.float32)
    if group == 32:
        wq, wd = orc.q8_0_quantize(w)
        ws, wid = wd.view(np.float16).astype(np.float32), rk.pack_q8_0(orc.q8_0_blocks(wq, wd), n, k)
    else:
        (wq, ws), wid = orc.quantize_rows(w, group), rk.pack_i8(w, group)
    for a_group in (group, k):
        aq, a_s = orc.quantize_rows(x, a_group)
        da, ds = dev(rk, aq), dev(rk, a_s)
        ref = orc.emu_matmul_gw(aq, a_s, a_group, wq, ws, group)
        for f16 in (False, True):
            dc = rk.DeviceBuffer(m * n * (2 if f16 else 4))
            fn = rk.lib().rk_matmul_w8a8_f16out_dev if f16 else rk.lib().rk_matmul_w8a8_dev
            assert fn(int(wid), da.ptr, ds.ptr, a_group, m, k, dc.ptr, None) == 0, rk.lib().rk_last_error()
            rk.synchronize()
            got = dc.download((m, n), np.uint16).view(np.float16).astype(np.float32) if f16 else \
                dc.download((m, n), np.float32)
            close(got, ref, f16)


@pytest.mark.parametrize("m,k,n", [(1, 8, 1), (16, 72, 16), (17, 1152, 33), (32, 1016, 200), (5, 3072, 96), (48, 704, 1400),
                                   (40, 96, 1500), (20, 192, 4200), (12, 136, 4300), (128, 200, 1000)])
def test_skinny_f16(rk, orc, m, k, n):
    note(f"skinny fp16 m={m} k={k} n={n}")
    r = np.random.default_rng(m + k + n)
    a = r.standard_normal((m, k)).astype(np.float16)
    b = (r.standard_normal((n, k)) * 0.05).astype(np.float16)
    da, dc = dev(rk, a.view(np.uint16)), rk.DeviceBuffer(m * n * 2)
    assert rk.lib().rk_matmul_f16_dev(int(rk.pack(b)), da.ptr, m, k, dc.ptr, None) == 0, rk.lib().rk_last_error()
    rk.synchronize()
    close(dc.download((m, n), np.uint16).view(np.float16).astype(np.float32),
          (a.astype(np.float64) @ b.astype(np.float64).T).astype(np.float32), True)


# K split over the waves of 32x32 tiles (8 waves) and 64x32 tiles (4 waves, the last
# three): one row, tile edges, K of less than two stages per wave and one that ends
# inside a stage, odd N, and the largest grids of either tile. (33 rows of K = 768
# run on the 16-row tiles.)
@pytest.mark.parametrize("m,k,n", [(9, 1536, 1), (33, 768, 1050), (64, 1544, 3000), (255, 776, 1000), (300, 1160, 800),
                                   (65, 4304, 2001), (70, 776, 3001), (450, 1160, 1000), (512, 3072, 1024)])
def test_kwaves_f16(rk, orc, m, k, n):
    note(f"fp16 K over waves m={m} k={k} n={n}")
    r = np.random.default_rng(m + k + n)
    a = r.standard_normal((m, k)).astype(np.float16)
    b = (r.standard_normal((n, k)) * 0.05).astype(np.float16)
    da, dc = dev(rk, a.view(np.uint16)), rk.DeviceBuffer(m * n * 2)
    wid = rk.pack(b)
    ref = (a.astype(np.float64) @ b.astype(np.float64).T).astype(np.float32)
    for _ in range(2):  # the sums have one order
        assert rk.lib().rk_matmul_f16_dev(int(wid), da.ptr, m, k, dc.ptr, None) == 0, rk.lib().rk_last_error()
        rk.synchronize()
        got = dc.download((m, n), np.uint16).view(np.float16).astype(np.float32)
        close(got, ref, True)


@pytest.mark.parametrize("glu", ["silu", "gelu"])
@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("m,k,n", [(9, 1536, 5), (40, 776, 1900), (64, 1160, 1900), (130, 3072, 300), (100, 1160, 1900),
                                   (20, 1160, 4300), (70, 776, 3001), (450, 1600, 1000)])
def test_kwaves_f16_glu(rk, orc, m, k, n, glu, f16):
    """gate|up against the glue of float64 products rounded to fp16: a product next to a rounding
    midpoint may round the other way (one fp16 step of the gate or up value)."""
    note(f"fp16 gate|up K over waves m={m} k={k} n={n} {glu} f16={f16}")
    r = np.random.default_rng(m + k + n)
    x = r.standard_normal((m, k)).astype(np.float16)
    w = [(r.standard_normal((n, k)) * 0.05).astype(np.float16) for _ in range(2)]
    dx, dy = dev(rk, x.view(np.uint16)), rk.DeviceBuffer(m * n * 4)
    kind, glue = (rk.GLU_SILU, orc.silu_mul) if glu == "silu" else (rk.GLU_GELU, orc.gelu_mul)
    wid = rk.pack_f16_glu(*[t.astype(np.float32) for t in w])
    assert rk.lib().rk_matmul_f16_glu_dev(int(wid), dx.ptr, m, k, kind, dy.ptr, int(f16), None) == 0
    rk.synchronize()
    got = dy.download((m, n), np.uint16).view(np.float16).astype(np.float32) if f16 else dy.download((m, n), np.float32)
    g, u = [(x.astype(np.float64) @ t.astype(np.float64).T).astype(np.float16).astype(np.float32) for t in w]
    ref = glue(g, u)
    # |d silu| and |d gelu| <= 1.13; a step is 2^-10 of the value; an fp16 result rounds once more
    step = 2.0 ** -10 * 1.13 * (np.abs(g) * np.abs(u) + np.abs(g * u)) + 1e-5
    assert (np.abs(got - ref) <= step + (2.0 ** -10 * np.abs(ref) if f16 else 0)).all()


@pytest.mark.parametrize("glu", ["silu", "gelu"])
@pytest.mark.parametrize("m,k,n", [(1, 64, 3), (8, 1152, 40), (32, 416, 64), (29, 3072, 17),
                                   (24, 128, 1500), (128, 256, 72), (9, 96, 4000)])
def test_skinny_glu_equals_products_then_glue(rk, orc, m, k, n, glu):
    """The fused forms give what the two plain products and the glue op give, bit for bit (larger
    shapes: test_gpu_sum_order.py)."""
    note(f"skinny gate|up m={m} k={k} n={n} {glu}")
    lib, r = rk.lib(), np.random.default_rng(m + k + n)
    kind, glue = (rk.GLU_SILU, rk.silu_mul) if glu == "silu" else (rk.GLU_GELU, rk.gelu_mul)
    x = r.standard_normal((m, k)).astype(np.float32)
    w = [(r.standard_normal((n, k)) * 0.05).astype(np.float32) for _ in range(2)]
    dx, dy = dev(rk, x.astype(np.float16).view(np.uint16)), rk.DeviceBuffer(m * n * 4)
    prods = []
    for t in w:
        assert lib.rk_matmul_f16_dev(int(rk.pack(t)), dx.ptr, m, k, dy.ptr, None) == 0, lib.rk_last_error()
        rk.synchronize()
        prods.append(dy.download((m, n), np.uint16).view(np.float16).astype(np.float32))
    assert lib.rk_matmul_f16_glu_dev(int(rk.pack_f16_glu(*w)), dx.ptr, m, k, kind, dy.ptr, 0, None) == 0
    rk.synchronize()
    assert (dy.download((m, n), np.float32) == glue(*prods)).all()

    blocks = [orc.q8_0_blocks(*orc.q8_0_quantize(t)) for t in w]
    aq, a_s = orc.quantize_rows(x, k)
    da, ds = dev(rk, aq), dev(rk, a_s)
    prods = []
    for b in blocks:
        assert lib.rk_matmul_w8a8_dev(int(rk.pack_q8_0(b, n, k)), da.ptr, ds.ptr, k, m, k, dy.ptr, None) == 0
        rk.synchronize()
        prods.append(dy.download((m, n), np.float32))
    wid = rk.pack_q8_0_glu(*blocks, n, k)
    assert lib.rk_matmul_w8a8_glu_dev(int(wid), da.ptr, ds.ptr, m, k, kind, dy.ptr, 0, None) == 0
    rk.synchronize()
    assert (dy.download((m, n), np.float32) == glue(*prods)).all()
