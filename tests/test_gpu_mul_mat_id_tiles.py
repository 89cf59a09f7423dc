"""The token tiles of the grouped MUL_MAT_ID: pair counts at the edges of a tile and of its half,
experts without pairs, and the most pairs (65535) in about as many tiles as the routing has
threads. Tolerance as
for every prefill matmul (f16 activations): NMSE 5e-5."""
import numpy as np
import pytest

import oracle as O
import scrapgpulibrary_amd as sg
from tests.test_gpu_mul_mat_id import check_grouped, run_mul_mat_id

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [sg.Q4_K, sg.Q6_K, sg.Q8_0], ids=lambda d: sg.NAMES[d])
@pytest.mark.parametrize("form", ["wide", "tiled"])
def test_pair_counts_at_tile_edges(hip, dtype, form):
    """One slot per token: expert e gets counts[e] pairs; with bn = 64 a tile of at most 32 runs
    without its second fragment."""
    dev, st = hip
    counts = [0, 1, 31, 32, 33, 63, 64, 65, 96, 97, 128, 129, 0]
    K, M = 512, 384
    if form == "wide":  # 384-row tiles need half as many experts as CUs
        counts = counts + [0, 40] * 64
    E = len(counts)
    ids = np.repeat(np.arange(E), counts).astype(np.int32)
    ids = np.random.default_rng(91).permutation(ids).reshape(-1, 1)
    T = len(ids)
    w = O.quantize(dtype, O.normal(K * M * E, 92, 0.0, 0.02))
    x = O.normal(T * K, 93).reshape(T, 1, K)
    y = run_mul_mat_id(dev, st, dtype, w, K, M, E, x, ids)
    if dev.info().compute_units == 256:
        assert sg.last_launch()[0] == ("grouped wide w=12 bn=64" if form == "wide" else "grouped w=4 bn=64"), sg.last_launch()
    check_grouped(y, O.mul_mat_id(dtype, w, K, M, E, x, ids))


def test_many_tiles_and_pairs(hip):
    """65535 pairs, the most a call may have, over 3 experts (1026 or 1027 token tiles)."""
    dev, st = hip
    K, M, E, T, nu = 256, 64, 3, 21845, 3
    rng = np.random.default_rng(94)
    ids = rng.integers(0, E, (T, nu)).astype(np.int32)
    w = O.quantize(sg.Q4_0, O.normal(K * M * E, 95, 0.0, 0.02))
    x = O.normal(T * K, 96).reshape(T, 1, K)
    y = run_mul_mat_id(dev, st, sg.Q4_0, w, K, M, E, x, ids)
    deq = O.dequantize(sg.Q4_0, w, K * M * E).reshape(E, M, K).astype(np.float64)
    xd = x[:, 0].astype(np.float64)
    per = np.stack([xd @ deq[e].T for e in range(E)], 1)  # every token against every expert
    ref = np.take_along_axis(per, ids[:, :, None], 1)
    d = ((y - ref) ** 2).sum(2) / (ref ** 2).sum(2)
    assert d.max() <= 20 * 5e-5, (d.max(), int(d.argmax()))
    assert ((y - ref) ** 2).sum() <= 5e-5 * (ref ** 2).sum()


@pytest.mark.parametrize("dtype,K", [(sg.Q4_0, 32), (sg.Q8_0, 992), (sg.Q4_0, 2016), (sg.Q8_0, 2048), (sg.Q4_K, 256), (sg.Q4_K, 1792), (sg.Q6_K, 768)],
                         ids=lambda v: str(v))
def test_x_rows_by_wave_and_by_group(hip, dtype, K):
    """The conversion of x beside the routing: a wave per row below K = 2048, 4 waves from there on;
    21 tokens with a row per slot (63 rows: the last work-group of 16 is part empty), row magnitudes
    over six decades (each row has a scale of its own)."""
    dev, st = hip
    M, E, T, nu = 96, 4, 21, 3
    rng = np.random.default_rng(97)
    ids = np.stack([rng.permutation(E)[:nu] for _ in range(T)]).astype(np.int32)
    w = O.quantize(dtype, O.normal(K * M * E, 98, 0.0, 0.02))
    x = O.normal(T * nu * K, 99).reshape(T, nu, K) * (10.0 ** rng.integers(-3, 4, (T, nu, 1))).astype(np.float32)
    y = run_mul_mat_id(dev, st, dtype, w, K, M, E, x, ids)
    ref = O.mul_mat_id(dtype, w, K, M, E, x, ids)
    d = ((y.astype(np.float64) - ref) ** 2).sum(2) / (ref.astype(np.float64) ** 2).sum(2)
    assert d.max() <= 20 * 5e-5, d.max()


def test_experts_of_many_tiles(hip):
    """Routing far from balanced: experts of more than 32 token tiles (their table is written by a wave) beside
    experts of few and of none, two of them in one wave; against every token's product with its expert in
    64 bits."""
    dev, st = hip
    K, M, E, T, nu = 256, 40, 130, 14000, 2
    rng = np.random.default_rng(100)
    ids = rng.integers(0, E, (T, nu)).astype(np.int32)
    hot = rng.random((T, nu))
    for e, lo, hi in ((3, 0.0, 0.3), (60, 0.3, 0.55), (127, 0.55, 0.85)):
        ids[(hot >= lo) & (hot < hi)] = e
    ids[ids == 61] = 62  # (no pairs beside the many)
    w = O.quantize(sg.Q8_0, O.normal(K * M * E, 101, 0.0, 0.02))
    x = O.normal(T * K, 102).reshape(T, 1, K)
    y = run_mul_mat_id(dev, st, sg.Q8_0, w, K, M, E, x, ids)
    deq = O.dequantize(sg.Q8_0, w, K * M * E).reshape(E, M, K).astype(np.float64)
    ref = np.empty(y.shape)
    for e in range(E):
        t, s = np.nonzero(ids == e)
        ref[t, s] = x[t, 0].astype(np.float64) @ deq[e].T
    d = ((y - ref) ** 2).sum(2) / (ref ** 2).sum(2)
    assert d.max() <= 20 * 5e-5, (d.max(), int(d.argmax()))
    assert ((y - ref) ** 2).sum() <= 5e-5 * (ref ** 2).sum()
