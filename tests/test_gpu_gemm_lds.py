"""F16 / BF16 weights on the GEMM with both operands in LDS (gemm_lds.hip), at the edges of its tiles
and of its stage pipeline (4 or 2 stages of 64 in LDS; K splits that start and end anywhere), against
the oracle. Bounds as for the other forms of this product: the operands are f16 (x rounded once, 2^-11
relative at worst, NMSE <= 2^-22 / 3 = 8e-8) or bf16 (both 2^-8: x alone is rounded here, 2^-16 / 3 =
5e-6): 1e-6 and 2e-5."""
import numpy as np
import pytest

import oracle as O
import scrapgpulibrary_amd as sg
from tests.gpu_util import nmse
from tests.test_gpu_float_weights import IDS, PREFILL_NMSE, float_weights, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,K,M,N,form", [
    (sg.F16, 2176, 1000, 65, "gemm lds w=8 kg=2 bn=128 rows=128 split=4"),  # 34 stages in splits of 8 and 9, one token past a half tile
    (sg.BF16, 1280, 513, 257, "gemm lds w=8 kg=2 bn=128 rows=128"),         # one row past a tile, one token past two
    (sg.F16, 1408, 12289, 380, "gemm lds w=8 kg=2 bn=128 rows="),           # 22 stages (a tail of 2)
    (sg.BF16, 1664, 12288, 512, "gemm lds w=8 kg=2 bn=128 rows=192 split=1"),  # 26 stages, every CU one tile
    (sg.F16, 1920, 2000, 130, "gemm lds w=8 kg=2 bn=128 rows=128"),         # 30 stages
    (sg.F16, 4224, 12290, 380, "gemm wide w=12 kg=1 bn=128 rg=1 split=2 lds"),  # 384-row tiles, 33 stages a split
    (sg.BF16, 128, 24576, 500, "gemm wide w=12 kg=1 bn=128 rg=1 split=1 lds"),  # two stages in all
    (sg.F16, 512, 9001, 1000, "gemm lds w=8 kg=2 bn=128 rows="),            # short K: 568 tiles of 128 x 128, a last round of 56
    (sg.BF16, 896, 28672, 300, "gemm lds w=8 kg=2 bn=128 rows="),           # 672 of them
    (sg.F16, 640, 9001, 1500, "gemm w=4 kg=1 bn=128"),                      # 852: a last round two thirds full
    (sg.F16, 384, 9001, 1000, "gemm w=4 kg=1 bn=128"),                      # K below 512
], ids=lambda v: str(v).replace(" ", "_"))
def test_gemm_lds(hip, dtype, K, M, N, form):
    dev, st = hip
    wbytes, wf = float_weights(dtype, M, K, 9000 + K + M)
    x = O.normal(N * K, 9001 + N).reshape(N, K)
    x[:, ::37] *= 100.0
    y = run(dev, st, dtype, wbytes, K, M, x, row_stride=2 * K + (48 if N % 2 else 0), x_offset=4 if M % 2 else 0, check_form=False)
    if dev.info().compute_units == 256:
        assert sg.last_launch()[0].startswith(form), sg.last_launch()
    rows = np.unique(np.concatenate([np.arange(0, M, max(1, M // 500)), np.arange(max(0, M - 200), M)]))  # (the oracle on a sample of rows)
    ref = O.mul_mat(dtype, np.ascontiguousarray(wbytes[rows]), K, len(rows), x, threads=8)
    e = nmse(y[:, rows], ref)
    assert e <= PREFILL_NMSE[dtype], f"{IDS[dtype]} {M}x{K} N={N}: NMSE {e:.3e} {sg.last_launch()}"


@pytest.mark.parametrize("dtype,K,Ms,N,S", [(sg.BF16, 1152, (700, 130, 257), 150, 1), (sg.F16, 1280, (390,), 70, 4)], ids=["multi", "slices"])
def test_gemm_lds_multi_and_slices(hip, dtype, K, Ms, N, S):
    """Row tiles per weight of a MUL_MAT_MULTI; slices with broadcast and padded columns of x and y."""
    dev, st = hip
    bc = 2 if S > 1 else 1
    px, py = K + 4, max(Ms) + 3
    x = np.zeros((S * bc, N, px), np.float32)
    x[:, :, :K] = O.normal(S * bc * N * K, 9100).reshape(S * bc, N, K)
    xb = dev.alloc(x.nbytes)
    xt = sg.tdesc(sg.F32, (K, N, S * bc), xb, nb=[4, 4 * px, 4 * px * N, 4 * px * N * S * bc])
    st.write(xb, 0, x)
    bufs, wts, yts, ws = [xb], [], [], []
    for j, M in enumerate(Ms):
        w = [float_weights(dtype, M, K, 9101 + 9 * j + s) for s in range(S)]
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
    assert sg.last_launch()[0].startswith("gemm lds") or dev.info().compute_units != 256, sg.last_launch()
    for M, w, b in zip(Ms, ws, bufs[2::2]):
        y = st.read(b, 0, 4 * py * N * S * bc).view(np.float32).reshape(S * bc, N, py)[:, :, :M]
        for s in range(S * bc):
            ref = O.mul_mat(dtype, w[s // bc][0], K, M, np.ascontiguousarray(x[s, :, :K]), threads=8)
            assert nmse(y[s], ref) <= PREFILL_NMSE[dtype], (M, s)
    for b in bufs:
        b.free()


@pytest.mark.parametrize("dtype,K,M,N,form", [
    (sg.F16, 1152, 1000, 130, "gemm lds w=8 kg=2 bn=128 rows=128"),                # tails in rows, tokens and stages
    (sg.BF16, 4224, 12290, 380, "gemm wide w=12 kg=1 bn=128 rg=1 split=2 lds"),    # K in splits
    (sg.F16, 1280, 12288, 511, "gemm lds w=8 kg=2 bn=128 rows=192 split=1"),
], ids=["128_rows", "384_rows_split", "192_rows"])
def test_gemm_lds_non_finite(hip, dtype, K, M, N, form):
    """Inf and NaN in x and weights reach exactly the outputs that they reach in the reference: the last row
    and token, which the tiles' padding reads again, hold some of them."""
    dev, st = hip
    wbytes, _ = float_weights(dtype, M, K, 9200)
    x = O.normal(N * K, 9201).reshape(N, K)
    x[N - 1, K - 1], x[N - 2, 0], x[3, 64] = np.inf, np.nan, -np.inf
    w = np.ascontiguousarray(wbytes).view(np.uint16).reshape(M, K).copy()
    inf, nan = (0x7C00, 0x7E00) if dtype == sg.F16 else (0x7F80, 0x7FC0)
    w[M - 1, K - 2], w[M - 2, 1], w[7, 65] = inf, nan, inf
    y = run(dev, st, dtype, w, K, M, x, check_form=False)
    if dev.info().compute_units == 256:
        assert sg.last_launch()[0].startswith(form), sg.last_launch()
    rows = np.unique(np.concatenate([np.arange(0, M, max(1, M // 300)), [7, 8], np.arange(M - 130, M)]))
    ref = O.mul_mat(dtype, np.ascontiguousarray(w[rows]), K, len(rows), x, threads=8)
    y = y[:, rows]
    assert np.array_equal(np.isnan(y), np.isnan(ref)) and np.array_equal(np.isinf(y), np.isinf(ref))
    ok = np.isfinite(ref)
    bad = ~ok & ~np.isnan(ref)
    assert bad.any() and np.array_equal(y[bad], ref[bad]) and nmse(y[ok], ref[ok]) <= PREFILL_NMSE[dtype]


@pytest.mark.parametrize("Ms,K,N,form", [
    ((4096, 1024, 1024), 1152, 2048, "gemm lds w=8 kg=2 bn=128 rows=128 split=1"),  # 34 192-row tiles against 32 over all rows: past two rounds of the CUs
    ((4000, 1100, 1044), 4224, 1000, "gemm lds w=8 kg=2 bn=128 rows="),             # 384-row tiles in two splits would take a second round
    ((8192, 8192, 8192), 128, 512, "gemm lds w=8 kg=2 bn=128 rows="),               # two stages of K; one round of 384-row tiles over all rows, two apart
    ((3840, 1152, 1152), 4224, 1000, "gemm wide w=12 kg=1 bn=128 rg=1 split=2 lds"),  # whole 384-row tiles: as one weight
], ids=["192", "384_split", "384", "whole"])
def test_gemm_lds_multi_tiles(hip, Ms, K, N, form):
    """Several weights whose tiles are more than those of their rows together: the tiles chosen for them."""
    dev, st = hip
    dtype = sg.BF16
    x = O.normal(N * K, 9300).reshape(N, K)
    xb = dev.alloc(x.nbytes)
    xt = sg.tdesc(sg.F32, (K, N), xb)
    st.write(xb, 0, x)
    bufs, wts, yts, ws = [xb], [], [], []
    for j, M in enumerate(Ms):
        w = np.ascontiguousarray(float_weights(dtype, M, K, 9301 + j)[0]).view(np.uint16).reshape(M, K)
        wb, yb = dev.alloc(w.nbytes), dev.alloc(4 * M * N)
        st.write(wb, 0, w.view(np.uint8).reshape(-1))
        bufs += [wb, yb]
        ws.append(w)
        wts.append(sg.tdesc(dtype, (K, M), wb))
        yts.append(sg.tdesc(sg.F32, (M, N), yb))
    op, keep = sg.multi_op(wts, xt, yts)
    st.execute(op)
    st.sync()
    if dev.info().compute_units == 256:
        assert sg.last_launch()[0].startswith(form), sg.last_launch()
    cols = np.unique(np.concatenate([np.arange(0, N, 37), np.arange(N - 20, N)]))
    for M, yt, w in zip(Ms, yts, ws):
        rows = np.unique(np.concatenate([np.arange(0, M, 61), np.arange(M - 70, M)]))
        ref = O.mul_mat(dtype, np.ascontiguousarray(w[rows]), K, len(rows), np.ascontiguousarray(x[cols]), threads=8)
        y = st.download(yt).reshape(N, M)[np.ix_(cols, rows)]
        assert nmse(y, ref) <= PREFILL_NMSE[dtype], M
    for b in bufs:
        b.free()
