"""Products over looked-up rows of which many are one and the same (the inner vertices of parse trees): the tiles that do a
vector's work, against sums in 64 bits, at the edges of tiles and of the rows that are equal."""
import ctypes as C

import numpy as np
import pytest

from cavs_amd import hip, synth

pytestmark = pytest.mark.gpu

U24 = 2.0 ** -24


@pytest.fixture
def g():
    import gpuutil

    hip.call("cavs_init", 0)
    yield gpuutil
    gpuutil.release()


def lookups(r, n, first, V, id_):
    ids = np.floor(r.bulk_uniform(max(n, 1)) * V)[:n].astype(np.float32)
    ids[first:] = id_
    return ids


def within(got, want, mags, K, what):
    """Every element within (K + 16) roundings of the sum of the products' magnitudes: K of the sum whatever its order, and
    what is left out of the products' parts (a quarter of a rounding each)."""
    tol = (K + 16) * U24 * mags + 1e-30
    bad = np.abs(got.astype(np.float64) - want) > tol
    assert not bad.any(), f"{what}: {int(bad.sum())} of {bad.size} outside, worst {np.abs(got - want)[bad].max()} of {tol[bad].max()}"


@pytest.mark.parametrize("n,first,E,N,pad", [(129, 0, 4, 64, 0), (190, 64, 300, 512, 0), (257, 100, 37, 96, 0), (2400, 1203, 300, 2048, 0),
                                             (1000, 437, 101, 640, 160), (700, 300, 1024, 128, 0), (9600, 4900, 300, 2048, 0), (5000, 5000, 64, 2048, 0)])
def test_rows_times_weights(g, n, first, E, N, pad):
    """cavs_embed_pull_sgemm_padded on 64 x 64 tiles and on 128 x 128 ones (the last two): the product, the looked-up rows, the ids."""
    r, V = synth.SplitMix64(n + E), 211
    table, B = (r.bulk_normal(V * E).reshape(V, E) * 0.1).astype(np.float32), r.bulk_uniform(E * N, -0.2, 0.2).reshape(E, N).astype(np.float32)
    used = pad * 5 // 8
    if pad:
        B.reshape(E, N // pad, pad)[:, :, used:] = 0
    for id_ in (0.0, 7.0):
        ids = lookups(r, n, first, V, id_)
        rows = np.arange(n, dtype=np.int32)[::-1].copy()
        x = np.empty(n, np.float32)
        x[rows] = ids
        Cd, e, xs = g.zeros(n, N, fill=float("nan")), g.zeros(n, E, fill=float("nan")), g.zeros(n, fill=float("nan"))
        g.call("cavs_embed_pull_sgemm_padded", g.P(Cd), N, g.P(e), E, g.P(xs), g.P(g.devf(x)), g.P(g.devi(rows)), g.P(g.devf(table)), n, E,
               g.P(g.devf(B)), N, N, 0, 0, pad, used, g.stream())
        want = table[ids.astype(int)]
        np.testing.assert_array_equal(g.host(e), want)
        np.testing.assert_array_equal(g.host(xs), ids)
        within(g.host(Cd), want.astype(np.float64) @ B.astype(np.float64), np.abs(want).astype(np.float64) @ np.abs(B).astype(np.float64), E, "x W")


@pytest.mark.parametrize("E,none", [(1, -1.0), (1, -2.0), (2, -1.0), (2, -3.0), (4, -1.0), (300, -1.0)])
def test_rows_without_an_id(g, E, none):
    """Rows with a negative id are zero rows, also where whole wavefronts of a tile (16 rows) have none and the others have one
    and the same word: beside the first, beside the last, all of them, and in a tile that the rows do not fill."""
    n, N, r = 64 * 5 + 40, 128, synth.SplitMix64(E)
    table, B = r.bulk_normal(9 * E).reshape(9, E).astype(np.float32), r.bulk_uniform(E * N, -1, 1).reshape(E, N).astype(np.float32)
    ids = np.full(n, 7.0, np.float32)
    for a, b in ((16, 64), (64, 80), (144, 160), (192, 256), (272, 288), (320 + 16, n)):
        ids[a:b] = none
    Cd, e, xs = g.zeros(n, N, fill=float("nan")), g.zeros(n, E, fill=float("nan")), g.zeros(n, fill=float("nan"))
    g.call("cavs_embed_pull_sgemm", g.P(Cd), N, g.P(e), E, g.P(xs), g.P(g.devf(ids)), g.P(g.devi(np.arange(n))), g.P(g.devf(table)), n, E,
           g.P(g.devf(B)), N, N, 0, 0, g.stream())
    want = np.where(ids[:, None] < 0, np.float32(0), table[7])
    np.testing.assert_array_equal(g.host(e), want)
    np.testing.assert_array_equal(g.host(xs), ids)
    within(g.host(Cd), want.astype(np.float64) @ B.astype(np.float64), np.abs(want).astype(np.float64) @ np.abs(B).astype(np.float64), E, "x W")


def test_an_infinite_row_times_weights(g):
    """An infinity in the row that many vertices share: infinities and NaN as the sum of products has them, padding zero."""
    n, E, N, r = 300, 20, 128, synth.SplitMix64(5)
    table, B = r.bulk_normal(11 * E).reshape(11, E).astype(np.float32), r.bulk_uniform(E * N, -1, 1).reshape(E, N).astype(np.float32)
    table[3, 4] = np.inf
    B[4, 9] = 0
    B.reshape(E, 2, 64)[:, :, 40:] = 0
    ids = lookups(r, n, 90, 3, 3.0)
    Cd, e, xs = g.zeros(n, N), g.zeros(n, E), g.zeros(n)
    g.call("cavs_embed_pull_sgemm_padded", g.P(Cd), N, g.P(e), E, g.P(xs), g.P(g.devf(ids)), g.P(g.devi(np.arange(n))), g.P(g.devf(table)), n, E,
           g.P(g.devf(B)), N, N, 0, 0, 64, 40, g.stream())
    with np.errstate(invalid="ignore"):
        want = table[ids.astype(int)].astype(np.float64) @ B.astype(np.float64)
    want.reshape(n, 2, 64)[:, :, 40:] = 0
    got = g.host(Cd)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
    ok = np.isfinite(want)
    np.testing.assert_allclose(got[ok], want[ok], rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("n,first,E,W,start", [(70, 0, 4, 64, 0), (200, 64, 300, 512, 64), (513, 250, 36, 96, 200), (2370, 1217, 300, 2048, 1217),
                                               (2370, 1217, 304, 2048, 900), (1000, 437, 100, 640, 437), (600, 600, 64, 256, 300), (900, 30, 512, 1024, 0),
                                               (333, 300, 60, 128, 333)])
def test_gradients_of_lookups(g, n, first, E, W, start):
    """cavs_sgemm_group_lookups: d e = d (x W) W^T into the table, d W = e^T d (x W), another product beside them; rows equal from
    `first` on, looked at from `start` on."""
    import torch

    r, V = synth.SplitMix64(3 * n + E), 97
    ids = lookups(r, n, first, V, 5.0)
    table = r.bulk_normal(V * E).reshape(V, E).astype(np.float32)
    e, d, Wt = table[ids.astype(int)], r.bulk_uniform(n * W, -1, 1).reshape(n, W).astype(np.float32), r.bulk_uniform(E * W, -1, 1).reshape(E, W).astype(np.float32)
    other = r.bulk_uniform(n * 32, -1, 1).reshape(n, 32).astype(np.float32)
    de, dW, dO = torch.full((n, E), float("nan"), device="cuda"), torch.full((E, W), float("nan"), device="cuda"), torch.full((32, W), float("nan"), device="cuda")
    e_, d_, W_, o_, ids_ = g.devf(e), g.devf(d), g.devf(Wt), g.devf(other), g.devf(ids)
    descs = (hip.GemmDesc * 3)()
    descs[0] = hip.GemmDesc(0, 1, n, E, W, 1.0, 0.0, g.P(d_), W, g.P(W_), W, g.P(de), E)
    descs[1] = hip.GemmDesc(1, 0, E, W, n, 1.0, 0.0, g.P(e_), E, g.P(d_), W, g.P(dW), W)
    descs[2] = hip.GemmDesc(1, 0, 32, W, n, 1.0, 0.0, g.P(o_), 32, g.P(d_), W, g.P(dO), W)
    nbytes = hip.lib().cavs_sgemm_group_workspace(3, descs)
    ws = torch.empty(max(nbytes // 4, 1), device="cuda")
    counters = torch.zeros(4096, dtype=torch.int32, device="cuda")
    f = lambda a: a.astype(np.float64)  # noqa: E731
    rows, mags = f(d) @ f(Wt).T, np.abs(f(d)) @ np.abs(f(Wt)).T
    want, mag = np.zeros((V, E)), np.zeros((V, E))
    np.add.at(want, ids.astype(int), rows)
    np.add.at(mag, ids.astype(int), mags)
    for turn in range(2):
        grad = torch.zeros(V, E, device="cuda")
        g.call("cavs_sgemm_group_lookups", 3, descs, 0, g.P(grad), g.P(ids_), 3, start, g.P(ws), nbytes, g.P(counters), 4096, None, g.stream())
        within(g.host(grad), want, mag, W + n, "table")
        within(g.host(dW), f(e).T @ f(d), np.abs(f(e)).T @ np.abs(f(d)), n, "d W")
        within(g.host(dO), f(other).T @ f(d), np.abs(f(other)).T @ np.abs(f(d)), n, "another product")
        assert not counters.any()


def test_an_infinite_gradient_of_lookups(g):
    """An infinite row of the table that many vertices share: d W has infinities and NaN where the sum of products has them."""
    import torch

    n, first, E, W, r = 400, 100, 64, 128, synth.SplitMix64(8)
    e = r.bulk_uniform(n * E, 0.1, 1).reshape(n, E).astype(np.float32)
    e[first:] = e[first]
    e[first:, 3] = np.inf
    d, Wt = r.bulk_uniform(n * W, -1, 1).reshape(n, W).astype(np.float32), np.zeros((E, W), np.float32)
    d[:, 7] = np.abs(d[:, 7])
    d[first + 9, 11] = 0
    ids = np.where(np.arange(n) < first, np.arange(n) % 40, 50).astype(np.float32)
    de, dW, grad = torch.zeros(n, E, device="cuda"), torch.zeros(E, W, device="cuda"), torch.zeros(60, E, device="cuda")
    descs = (hip.GemmDesc * 2)()
    e_, d_, W_ = g.devf(e), g.devf(d), g.devf(Wt)
    descs[0] = hip.GemmDesc(0, 1, n, E, W, 1.0, 0.0, g.P(d_), W, g.P(W_), W, g.P(de), E)
    descs[1] = hip.GemmDesc(1, 0, E, W, n, 1.0, 0.0, g.P(e_), E, g.P(d_), W, g.P(dW), W)
    nbytes = hip.lib().cavs_sgemm_group_workspace(2, descs)
    ws, counters = torch.empty(max(nbytes // 4, 1), device="cuda"), torch.zeros(4096, dtype=torch.int32, device="cuda")
    g.call("cavs_sgemm_group_lookups", 2, descs, 0, g.P(grad), g.P(g.devf(ids)), 3, first, g.P(ws), nbytes, g.P(counters), 4096, None, g.stream())
    got = g.host(dW)
    assert np.isposinf(got[3, 7]) and np.isnan(got[3, 11]) and np.isnan(got[3, np.arange(W) % 64 != 7][20:40]).all()
    assert np.isfinite(np.delete(got, 3, axis=0)).all()


def test_gradients_whose_sum_passes_the_range_of_a_float(g):
    """Gradients of 2e37 .. 3e37: the sum of a block of 64 rows is infinite, the products with weights of 1e-6 and their sums are not."""
    import torch

    n, first, E, W, r = 400, 100, 64, 128, synth.SplitMix64(11)
    e = r.bulk_uniform(n * E, 1e-4, 1e-3).reshape(n, E).astype(np.float32)
    e[first:] = e[first]
    ids = np.where(np.arange(n) < first, np.arange(n) % 40, 50).astype(np.float32)
    d = r.bulk_uniform(n * W, 2e37, 3e37).reshape(n, W).astype(np.float32)
    Wt = r.bulk_uniform(E * W, 5e-7, 1e-6).reshape(E, W).astype(np.float32)
    de, dW, grad = torch.zeros(n, E, device="cuda"), torch.zeros(E, W, device="cuda"), torch.zeros(60, E, device="cuda")
    e_, d_, W_ = g.devf(e), g.devf(d), g.devf(Wt)
    descs = (hip.GemmDesc * 2)()
    descs[0] = hip.GemmDesc(0, 1, n, E, W, 1.0, 0.0, g.P(d_), W, g.P(W_), W, g.P(de), E)
    descs[1] = hip.GemmDesc(1, 0, E, W, n, 1.0, 0.0, g.P(e_), E, g.P(d_), W, g.P(dW), W)
    nbytes = hip.lib().cavs_sgemm_group_workspace(2, descs)
    ws, counters = torch.empty(max(nbytes // 4, 1), device="cuda"), torch.zeros(4096, dtype=torch.int32, device="cuda")
    g.call("cavs_sgemm_group_lookups", 2, descs, 0, g.P(grad), g.P(g.devf(ids)), 3, first, g.P(ws), nbytes, g.P(counters), 4096, None, g.stream())
    f = lambda a: a.astype(np.float64)  # noqa: E731
    want, rows = np.zeros((60, E)), f(d) @ f(Wt).T
    np.add.at(want, ids.astype(int), rows)
    within(g.host(grad), want, want, W + n, "table")  # (everything is positive)
    dw = f(e).T @ f(d)
    within(g.host(dW), dw, dw, n, "d W")
