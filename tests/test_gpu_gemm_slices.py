"""Prefill MUL_MAT over slices in both outer dimensions (6 slices of x), the weights broadcast over one
of them or over none: the slice, row and split arithmetic of every GEMM family, against the oracle at
the prefill gate (f16 operands: NMSE 5e-5; F16 weights 1e-6)."""
import numpy as np
import pytest

import oracle as O
import scrapgpulibrary_amd as sg
from tests.gpu_util import nmse
from tests.test_gpu_float_weights import float_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w2,w3", [(3, 2), (1, 2), (3, 1)], ids=["none", "over_2", "over_3"])
@pytest.mark.parametrize("dtype,K,M,N,form", [
    (sg.Q4_K, 2048, 80, 33, "gemm w=4"),       # K in splits
    (sg.Q8_0, 1056, 48, 70, "gemm w=4"),       # a K tail
    (sg.F16, 1152, 130, 100, "gemm lds"),
    (sg.F16, 520, 70, 20, "float"),
], ids=["q4_k", "q8_0", "f16_lds", "f16_f32"])
def test_slices_in_both_dimensions(hip, dtype, K, M, N, form, w2, w3):
    dev, st = hip
    W, S2, S3 = w2 * w3, 3, 2
    if dtype == sg.F16:
        raw = np.stack([float_weights(dtype, M, K, 6200 + i)[0] for i in range(W)])
    else:
        raw = O.quantize(dtype, O.normal(W * M * K, 6200, 0.0, 0.02)).reshape(W, -1)
    wbytes = np.ascontiguousarray(raw).view(np.uint8).reshape(-1)
    wb = dev.alloc(wbytes.nbytes)
    if dtype == sg.F16:
        st.write(wb, 0, wbytes)
        wt = sg.tdesc(dtype, (K, M, w2, w3), wb)
    else:
        wt = sg.tdesc(dtype, (K, M, w2, w3), wb, layout=sg.R32)
        st.upload(wt, wbytes)
    px, py = K + 4, M + 3
    x = np.zeros((S3, S2, N, px), np.float32)
    x[..., :K] = O.normal(S3 * S2 * N * K, 6210).reshape(S3, S2, N, K)
    xb, yb = dev.alloc(x.nbytes), dev.alloc(4 * S3 * S2 * N * py)
    st.write(xb, 0, x)
    st.write(yb, 0, np.full(S3 * S2 * N * py, -7.0, np.float32))
    xt = sg.tdesc(sg.F32, (K, N, S2, S3), xb, nb=[4, 4 * px, 4 * px * N, 4 * px * N * S2])
    yt = sg.tdesc(sg.F32, (M, N, S2, S3), yb, nb=[4, 4 * py, 4 * py * N, 4 * py * N * S2])
    op, keep = sg.mul_mat_op(wt, xt, yt, allow_broadcast=1)
    st.execute(op)
    st.sync()
    got = sg.last_launch()[0]
    assert got.startswith(form) or dev.info().compute_units != 256, got
    y = st.read(yb, 0, 4 * S3 * S2 * N * py).view(np.float32).reshape(S3, S2, N, py)
    for i3 in range(S3):
        for i2 in range(S2):
            wi = i3 // (S3 // w3) * w2 + i2 // (S2 // w2)
            ref = O.mul_mat(dtype, np.ascontiguousarray(raw[wi]), K, M, np.ascontiguousarray(x[i3, i2, :, :K]), threads=8)
            e = nmse(y[i3, i2, :, :M], ref)
            assert e <= (1e-6 if dtype == sg.F16 else 5e-5), f"slice {i2},{i3}: NMSE {e:.3e} [{got}]"
    assert np.all(y[..., M:] == -7.0)
    for b in (wb, xb, yb):
        b.free()
