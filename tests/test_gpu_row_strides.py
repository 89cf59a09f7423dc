"""Float weights whose rows lie at different strides, sharing one x: a MUL_MAT_MULTI, the MUL_MATs of a
plan, and the MUL_MAT_IDs of a plan that share x and ids. One launch over several weights reads all of
them at one row stride, so such weights run as one launch each. Against the oracle, at the bounds of
the single products (test_gpu_float_weights.py)."""
import ctypes as C

import numpy as np
import pytest

import oracle as O
import scrapgpulibrary_amd as sg
from tests.gpu_util import nmse
from tests.test_gpu_float_weights import IDS, PREFILL_NMSE, float_weights

pytestmark = pytest.mark.gpu


def strided(dev, st, dtype, wbytes, K, M, E, pad):
    """Weights of E slices of M rows, rows `pad` bytes longer than K elements (slices as far apart as
    with 64 bytes of padding, whatever `pad` is): (buffer, descriptor)."""
    esz = sg.TYPE_SIZE[dtype]
    rs, ss = K * esz + pad, M * (K * esz + 64)
    img = np.full(E * ss, 0x5A, np.uint8)
    for e in range(E):
        rows = img[e * ss:e * ss + M * rs].reshape(M, rs)
        rows[:, :K * esz] = np.ascontiguousarray(wbytes).view(np.uint8).reshape(E, M, K * esz)[e]
    wb = dev.alloc(img.nbytes)
    st.write(wb, 0, img)
    return wb, sg.tdesc(dtype, (K, M, E), wb, nb=[esz, rs, ss, ss * E])


def build(dev, ops):
    nodes = (sg.PlanNode * len(ops))(*[sg.PlanNode(C.sizeof(sg.PlanNode), op, 0) for op, _ in ops])
    plan = C.c_void_p()
    sg.check(sg.lib().scrapgpu_plan_build(dev.handle, C.byref(sg.PlanDesc(C.sizeof(sg.PlanDesc), nodes, len(ops))), C.byref(plan)), "plan_build")
    return plan


@pytest.mark.parametrize("as_plan", [False, True], ids=["multi", "plan"])
@pytest.mark.parametrize("dtype,K,N", [
    (sg.F32, 264, 1), (sg.F16, 520, 2), (sg.BF16, 512, 5),  # decode: the vector kernel, 4 x 4 tiles
    (sg.F32, 264, 30), (sg.F16, 520, 70),                   # columns: exact f32 products
    (sg.BF16, 512, 20), (sg.F16, 1152, 150),                # prefill: 4-wave work-groups, both operands in LDS
], ids=lambda v: str(v))
def test_mul_mats_sharing_x(hip, dtype, K, N, as_plan):
    dev, st = hip
    x = O.normal(N * K, 6000 + N).reshape(N, K)
    xb = dev.alloc(x.nbytes)
    xt = sg.tdesc(sg.F32, (K, N), xb)
    st.write(xb, 0, x)
    bufs, wts, yts, refs = [xb], [], [], []
    for i, (M, pad) in enumerate([(1100, 16), (300, 0), (130, 64)]):
        wbytes, _ = float_weights(dtype, M, K, 6001 + i)
        wb, wt = strided(dev, st, dtype, wbytes, K, M, 1, pad)
        yb = dev.alloc(4 * M * N)
        bufs += [wb, yb]
        wts.append(wt)
        yts.append(sg.tdesc(sg.F32, (M, N), yb))
        refs.append(O.mul_mat(dtype, wbytes, K, M, x, threads=8))
    if as_plan:
        ops = [sg.mul_mat_op(wt, xt, yt) for wt, yt in zip(wts, yts)]
        plan = build(dev, ops)
        for _ in range(2):
            sg.check(sg.lib().scrapgpu_plan_execute(st.handle, plan), "plan_execute")
    else:
        op, keep = sg.multi_op(wts, xt, yts)
        st.execute(op)
    st.sync()
    tol = PREFILL_NMSE[dtype] if N > 8 and K % 128 == 0 else 1e-10
    for yt, ref in zip(yts, refs):
        e = nmse(st.download(yt).reshape(ref.shape), ref)
        assert e <= tol, f"{IDS[dtype]} {ref.shape[1]} rows: NMSE {e:.3e} [{sg.last_launch()[0]}]"
    if as_plan:
        sg.lib().scrapgpu_plan_free(plan)
    for b in bufs:
        b.free()


@pytest.mark.parametrize("dtype", (sg.F32, sg.F16), ids=lambda d: IDS[d])
def test_mul_mat_ids_sharing_x(hip, dtype):
    """gate and up of a mixture of experts, the expert tensors equally far apart, their rows not."""
    dev, st = hip
    K, M, E, T, nu = 256, 48, 5, 6, 2
    ids = np.random.default_rng(6100).integers(0, E, (T, nu)).astype(np.int32)
    x = O.normal(T * K, 6101).reshape(T, 1, K)
    xb, ib = dev.alloc(x.nbytes), dev.alloc(ids.nbytes)
    st.write(xb, 0, x)
    st.write(ib, 0, ids)
    xt, it = sg.tdesc(sg.F32, (K, 1, T), xb), sg.tdesc(sg.I32, (nu, T), ib)
    bufs, ops, outs = [xb, ib], [], []
    for i, pad in enumerate((0, 48)):
        wbytes = np.stack([float_weights(dtype, M, K, 6102 + 10 * i + e)[0] for e in range(E)])
        wb, wt = strided(dev, st, dtype, wbytes, K, M, E, pad)
        yb = dev.alloc(4 * M * nu * T)
        yt = sg.tdesc(sg.F32, (M, nu, T), yb)
        bufs += [wb, yb]
        ops.append(sg.mul_mat_id_op(wt, xt, it, yt, nu))
        outs.append((yt, O.mul_mat_id(dtype, wbytes.reshape(-1), K, M, E, x, ids)))
    plan = build(dev, ops)
    for _ in range(2):
        sg.check(sg.lib().scrapgpu_plan_execute(st.handle, plan), "plan_execute")
    st.sync()
    for yt, ref in outs:
        e = nmse(st.download(yt).reshape(ref.shape), ref)
        assert e <= 1e-10, f"NMSE {e:.3e}"
    sg.lib().scrapgpu_plan_free(plan)
    for b in bufs:
        b.free()
