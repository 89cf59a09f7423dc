"""Float-weight products beside others: the kernels with both operands in LDS and those on the f32 matrix
units recorded in a plan (a HIP graph) and replayed, and one x that F16, BF16 and quantized weights read in
different orders."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
import scrapgpulibrary_amd as sg
from tests.gpu_util import nmse, upload_weights
from tests.test_gpu_float_weights import IDS, PREFILL_NMSE, float_weights
from tests.test_gpu_row_strides import build

pytestmark = pytest.mark.gpu

NAMES = {**sg.NAMES, **IDS}


def test_replays_match_the_ops_run_alone(hip):
    """Every replay, with new x and with the ops run alone between the replays, gives bit for bit what the
    ops run alone give; those match the oracle."""
    dev, st = hip
    cases = [  # (dtype, K, rows, columns, the kernel's form)
        (sg.F16, 1152, 390, 130, "gemm lds"), (sg.BF16, 2176, 1000, 70, "gemm lds"),  # (the second with K in splits)
        (sg.F16, 4224, 12290, 380, "gemm wide w=12"), (sg.BF16, 520, 3075, 4, "float mfma tile=16x4"),
        (sg.F16, 256, 4101, 8, "float mfma tile=16x8"), (sg.F32, 2048, 130, 300, "float mfma tile=16x16"),
        (sg.BF16, 72, 2001, 130, "float mfma tile=32x32"), (sg.F32, 4096, 40, 100, "float rows=8 column-groups"),
    ]
    items, bufs = [], []
    for i, (dtype, K, M, N, form) in enumerate(cases):
        wbytes, _ = float_weights(dtype, M, K, 9400 + i)
        wb, xb, yb = dev.alloc(M * K * sg.TYPE_SIZE[dtype]), dev.alloc(4 * K * N), dev.alloc(4 * M * N)
        st.write(wb, 0, np.ascontiguousarray(wbytes).view(np.uint8).reshape(-1))
        bufs += [wb, xb, yb]
        xt, yt = sg.tdesc(sg.F32, (K, N), xb), sg.tdesc(sg.F32, (M, N), yb)
        items.append((xt, yt, wbytes, sg.mul_mat_op(sg.tdesc(dtype, (K, M), wb), xt, yt)))
    plan = build(dev, [it[3] for it in items])
    ones = [np.full(4 * M * N, 0x55, np.uint8) for _, _, M, N, _ in cases]
    for rep in range(4):
        for i, (_, K, M, N, _) in enumerate(cases):
            st.upload(items[i][0], O.normal(N * K, 9420 + 10 * rep + i).reshape(N, K))
            st.write(bufs[3 * i + 2], 0, ones[i])
        sg.check(sg.lib().scrapgpu_plan_execute(st.handle, plan), "plan_execute")
        st.sync()
        got = [st.download(it[1]).copy() for it in items]
        for i, (dtype, K, M, N, form) in enumerate(cases):
            st.write(bufs[3 * i + 2], 0, ones[i])
            st.execute(items[i][3][0])
            st.sync()
            assert sg.last_launch()[0].startswith(form) or dev.info().compute_units != 256, (form, sg.last_launch())
            y = st.download(items[i][1])
            assert np.array_equal(got[i].view(np.uint32), y.view(np.uint32)), f"replay {rep}: {IDS[dtype]} {M}x{K} N={N}"
            if rep == 0:
                rows = np.unique(np.linspace(0, M - 1, 200).astype(int))
                wr = np.ascontiguousarray(np.ascontiguousarray(items[i][2]).view(np.uint8).reshape(M, -1)[rows])
                ref = O.mul_mat(dtype, wr, K, len(rows), O.normal(N * K, 9420 + i).reshape(N, K), threads=8)
                assert nmse(y.reshape(N, M)[:, rows], ref) <= (PREFILL_NMSE[dtype] if N > 8 and K % 128 == 0 and dtype != sg.F32 else 1e-10)
    sg.lib().scrapgpu_plan_free(plan)
    for b in bufs:
        b.free()


@pytest.mark.parametrize("as_plan", [False, True], ids=["multi", "plan"])
@pytest.mark.parametrize("order", [(sg.F16, sg.Q8_0, sg.F16), (sg.Q4_0, sg.F16, sg.BF16), (sg.BF16, sg.Q4_K, sg.F16), (sg.Q6_K, sg.F16, sg.Q8_0)],
                         ids=lambda o: "-".join(NAMES[d] for d in o))
@pytest.mark.parametrize("N", [20, 150])
def test_one_x_in_every_order(hip, order, N, as_plan):
    """x is kept in plain element order for F16 and BF16 weights and in pairs for the quantized ones: weights of
    both kinds in a row over one x, at a prefill size."""
    dev, st = hip
    K = 1280
    x = O.normal(N * K, 9500).reshape(N, K)
    xb = dev.alloc(x.nbytes)
    xt = sg.tdesc(sg.F32, (K, N), xb)
    st.write(xb, 0, x)
    bufs, wts, yts, refs = [xb], [], [], []
    for j, (dtype, M) in enumerate(zip(order, (1030, 512, 700))):
        if dtype in (sg.F16, sg.BF16):
            raw = float_weights(dtype, M, K, 9501 + j)[0]
            wb = dev.alloc(2 * M * K)
            st.write(wb, 0, np.ascontiguousarray(raw).view(np.uint8).reshape(-1))
            wt = sg.tdesc(dtype, (K, M), wb)
        else:
            raw = O.quantize(dtype, O.normal(M * K, 9501 + j, 0.0, 0.02))
            wb, wt = upload_weights(dev, st, dtype, raw, K, M)
        yb = dev.alloc(4 * M * N)
        bufs += [wb, yb]
        wts.append(wt)
        yts.append(sg.tdesc(sg.F32, (M, N), yb))
        refs.append(O.mul_mat(dtype, raw, K, M, x, threads=8))
    if as_plan:
        plan = build(dev, [sg.mul_mat_op(w, xt, y) for w, y in zip(wts, yts)])
        for _ in range(2):
            sg.check(sg.lib().scrapgpu_plan_execute(st.handle, plan), "plan_execute")
    else:
        op, keep = sg.multi_op(wts, xt, yts)
        st.execute(op)
    st.sync()
    for dtype, yt, ref in zip(order, yts, refs):
        e = nmse(st.download(yt).reshape(ref.shape), ref)
        assert e <= PREFILL_NMSE.get(dtype, 5e-5), f"{NAMES[dtype]}: NMSE {e:.3e}"
    if as_plan:
        sg.lib().scrapgpu_plan_free(plan)
    for b in bufs:
        b.free()
