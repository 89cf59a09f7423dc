"""Float weights at several columns: the f32 matrix-unit kernels (matmul_f32.hip) and the vector
kernel's column groups, at the edges of their tiles, against the oracle. The kernels' chains are
short (relative error 1.1e-7 against 64-bit products, NMSE 1.2e-14); the oracle adds K products in
order, each addition rounding by up to u = 2^-24 of a partial sum that grows as sqrt(k): NMSE about
sum_k k u^2 / 3 / K = K u^2 / 6 (2.4e-12 at K = 4096). Bound for both: (K + 16) u^2."""
import numpy as np
import pytest

import oracle as O
import scrapgpulibrary_amd as sg
from tests.test_gpu_float_weights import IDS, float_weights, run
from tests.gpu_util import check_matvec, nmse

pytestmark = pytest.mark.gpu


def bound(K):
    return (K + 16) * 2.0 ** -48

CASES = [
    # 3..8 columns: 4- and 8-column tiles, whole and partial steps of 128, a row tail, one column pad
    (sg.F16, 512, 3100, 3, 0, "float mfma tile=16x4"),
    (sg.BF16, 520, 3075, 4, 0, "float mfma tile=16x4"),
    (sg.F16, 2184, 1030, 5, 4, "float mfma tile=16x4"),  # rows on a quarter of the CUs; unaligned x
    (sg.BF16, 256, 4101, 8, 0, "float mfma tile=16x8"),
    (sg.F16, 8, 4100, 7, 0, "float mfma tile=16x8"),  # the smallest K
    (sg.BF16, 1160, 4099, 6, 4, "float mfma tile=16x8"),
    # more: 16 x 16, 32 x 32 and 64 x 32 tiles with row, column and K tails
    (sg.F32, 2048, 130, 300, 0, "float mfma tile=16x16"),
    (sg.F32, 8, 1000, 33, 0, "float mfma tile=16x16"),
    (sg.F16, 520, 2500, 9, 4, "float mfma tile=16x16"),
    (sg.F32, 1032, 513, 500, 4, "float mfma tile=32x32"),
    (sg.BF16, 72, 2001, 130, 0, "float mfma tile=32x32"),
    (sg.F32, 264, 1000, 700, 0, "float mfma tile=64x32"),
    # few 8 x 8 tiles: the vector kernel's column groups in one launch
    (sg.F32, 4096, 40, 100, 0, "float rows=8 column-groups=13"),
    (sg.F16, 136, 70, 9, 4, "float rows=8 column-groups=2"),
]


@pytest.mark.parametrize("dtype,K,M,N,xoff,form", CASES, ids=lambda v: str(v).replace(" ", "_"))
def test_float_columns(hip, dtype, K, M, N, xoff, form):
    dev, st = hip
    wbytes, wf = float_weights(dtype, M, K, 8000 + K + M)
    x = O.normal(N * K, 8001 + N).reshape(N, K)
    y = run(dev, st, dtype, wbytes, K, M, x, x_offset=xoff, row_stride=K * sg.TYPE_SIZE[dtype] + (48 if xoff else 0), check_form=False)
    if dev.info().compute_units == 256:
        assert sg.last_launch()[0].startswith(form), sg.last_launch()
    ref = O.mul_mat(dtype, wbytes, K, M, x, threads=8)
    e = check_matvec(y, ref, x, wf)
    assert e <= bound(K), f"{IDS[dtype]} NMSE {e:.3e}"


@pytest.mark.parametrize("dtype,K,Ms,N,S", [(sg.F16, 640, (2050, 40, 1100), 4, 1), (sg.F32, 328, (90, 700, 17), 70, 1), (sg.BF16, 136, (1040,), 6, 4)],
                         ids=["multi_cols", "multi_tiles", "slices"])
def test_float_columns_multi_and_slices(hip, dtype, K, Ms, N, S):
    """Row tiles across the weights of a MUL_MAT_MULTI; slices with broadcast (2 slices of x per
    slice of weights) and padded columns of x and y."""
    dev, st = hip
    bc = 2 if S > 1 else 1
    px, py = K + 4, max(Ms) + 3
    x = np.zeros((S * bc, N, px), np.float32)
    x[:, :, :K] = O.normal(S * bc * N * K, 8100).reshape(S * bc, N, K)
    xb = dev.alloc(x.nbytes)
    xt = sg.tdesc(sg.F32, (K, N, S * bc), xb, nb=[4, 4 * px, 4 * px * N, 4 * px * N * S * bc])
    st.write(xb, 0, x)
    bufs, wts, yts, ws = [xb], [], [], []
    for j, M in enumerate(Ms):
        w = [float_weights(dtype, M, K, 8101 + 9 * j + s) for s in range(S)]
        raw = np.concatenate([np.ascontiguousarray(b).view(np.uint8).reshape(-1) for b, _ in w])
        wb, yb = dev.alloc(raw.nbytes), dev.alloc(4 * py * N * S * bc)
        st.write(wb, 0, raw)
        bufs += [wb, yb]
        ws.append(w)
        wts.append(sg.tdesc(dtype, (K, M, S), wb))
        yts.append(sg.tdesc(sg.F32, (M, N, S * bc), yb, nb=[4, 4 * py, 4 * py * N, 4 * py * N * S * bc]))
    op, keep = sg.multi_op(wts, xt, yts) if len(Ms) > 1 else sg.mul_mat_op(wts[0], xt, yts[0], allow_broadcast=1)
    st.execute(op)
    st.sync()
    assert sg.last_launch()[0].startswith("float mfma") or dev.info().compute_units != 256, sg.last_launch()
    for M, yt, w, b in zip(Ms, yts, ws, bufs[2::2]):
        y = st.read(b, 0, 4 * py * N * S * bc).view(np.float32).reshape(S * bc, N, py)[:, :, :M]
        for s in range(S * bc):
            ref = O.mul_mat(dtype, w[s // bc][0], K, M, np.ascontiguousarray(x[s, :, :K]), threads=8)
            assert nmse(y[s], ref) <= bound(K), (M, s)
    for b in bufs:
        b.free()


@pytest.mark.parametrize("dtype,K,M,N", [(sg.F16, 136, 4100, 8), (sg.F32, 40, 600, 40)], ids=["cols", "tiles"])
def test_float_columns_non_finite(hip, dtype, K, M, N):
    """Inf and NaN in x and weights reach exactly the outputs they reach in the reference: the padding
    of a K tail (8 of 128 or 32 elements) and of rows and columns must not spread them."""
    dev, st = hip
    wbytes, _ = float_weights(dtype, M, K, 8200)
    x = O.normal(N * K, 8201).reshape(N, K)
    x[1, K - 1], x[2, 0] = np.inf, np.nan
    w = np.ascontiguousarray(wbytes).reshape(M, K).copy()
    w[M - 1, K - 2] = 0x7C00 if dtype == sg.F16 else np.inf
    y = run(dev, st, dtype, w, K, M, x, check_form=False)
    ref = O.mul_mat(dtype, w, K, M, x, threads=8)
    assert np.array_equal(np.isnan(y), np.isnan(ref)) and np.array_equal(np.isinf(y), np.isinf(ref))
    ok = np.isfinite(ref)
    assert np.array_equal(y[~ok & ~np.isnan(ref)], ref[~ok & ~np.isnan(ref)]) and nmse(y[ok], ref[ok]) <= bound(K)


@pytest.mark.parametrize("dtype,K,M,N", [(sg.BF16, 520, 4096, 5), (sg.F16, 4096, 3072, 8), (sg.F16, 1000, 1000, 64), (sg.BF16, 2056, 1500, 40),
                                         (sg.F32, 512, 512, 1100), (sg.F32, 1024, 300, 128), (sg.F16, 64, 1000, 30),
                                         (sg.F32, 16, 1270, 471), (sg.F32, 40, 1500, 94), (sg.F32, 120, 1150, 449)], ids=lambda v: str(v))
def test_float_columns_error(hip, dtype, K, M, N):
    """The error against 64-bit products is no larger than the vector kernel's (1 and 2 columns per call),
    on activations with outlier channels."""
    dev, st = hip
    wbytes, wf = float_weights(dtype, M, K, 8300 + K)
    x = O.normal(N * K, 8301 + N).reshape(N, K)
    x[:, 5::64] *= 8
    exact = x.astype(np.float64) @ wf.astype(np.float64).T
    y = run(dev, st, dtype, wbytes, K, M, x, check_form=False)
    assert sg.last_launch()[0].startswith("float mfma") or dev.info().compute_units != 256, sg.last_launch()
    cols = np.arange(N) if N <= 64 else np.linspace(0, N - 1, 64).astype(int)  # (a sample: some 30000 values differ by 1% in their mean error)
    v = np.concatenate([run(dev, st, dtype, wbytes, K, M, x[cols[i:i + 2]]) for i in range(0, len(cols), 2)])
    e, ev = nmse(y, exact) ** 0.5, nmse(v, exact[cols]) ** 0.5
    assert e <= ev, f"{IDS[dtype]} {M}x{K} N={N}: {e:.3e}, the vector kernel {ev:.3e}"
