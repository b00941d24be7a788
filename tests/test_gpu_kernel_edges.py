"""The matcher at the sizes where its kernels' tiles, lane groups and merges change, against the FP64 oracle at the
reference's own tolerance (validate.py:7)."""
import numpy as np
import pytest
import torch

from application_classification_amd import _lib
from application_classification_amd import workloads as W
from application_classification_amd.matcher import AC_OPT_PRUNE, AC_OPT_TAPE, ACError, Matcher
from oracle import oracle as O
from tests.conftest import allclose_report
from tests.test_gpu_adjoint import check_grad, fd_grad, gpu_grad, weights

pytestmark = pytest.mark.gpu


def g64(g):
    return O.Graph64.of(g.vfeat, g.efeat, g.src, g.dst)


def random_graph(n, m, dv, de, seed):
    r = np.random.default_rng(seed)
    return W.Graph(r.normal(size=(n, dv)).astype(np.float32), r.normal(size=(m, de)).astype(np.float32),
                   r.integers(0, n, m).astype(np.int32), r.integers(0, n, m).astype(np.int32))


def check(data, patt, n_iter=3):
    with Matcher(0) as m:
        m.set_data(data)
        m.set_pattern(patt)
        mu = m.run(n_iter)
    bad, ratio = allclose_report(mu, O.run(g64(data), g64(patt), n_iter=n_iter))
    print(f"dn={data.num_nodes} de={data.num_edges} pn={patt.num_nodes} pe={patt.num_edges}: max err/tol {ratio:.4f}", flush=True)
    assert bad == 0, ratio


@pytest.mark.parametrize("n,m,pn,pe", [
    (2, 1, 1, 1), (9, 30, 1, 3), (64, 200, 2, 1),            # a few rows, one pattern vertex or edge
    (4095, 9000, 5, 3), (4097, 5000, 17, 65),                # 8- and 16-row tiles, some vertices isolated
    (20_000, 90_000, 33, 20), (70_000, 90_000, 9, 24),       # 32- and 64-row tiles; a full block of partials
    (500, 3000, 256, 256), (1200, 2500, 3, 256), (900, 4000, 255, 64),  # the widest patterns
])
def test_vertex_pass_tiles(n, m, pn, pe):
    """Multigraphs with self-loops and isolated vertices; the tile height follows the vertex count and the pattern."""
    check(random_graph(n, m, 4, 5, n), random_graph(pn, pe, 4, 5, pn + pe))


@pytest.mark.parametrize("run_edges", [4, 8, 16, 32, 64, 128])
@pytest.mark.parametrize("prune", [0, 1])
def test_run_lengths(run_edges, prune, monkeypatch):
    """Every run length the edge count can select, on a graph with hubs of both kinds, one to hundreds of pieces: the
    pieces' atomic maxima over several iterations (each resetting the rows), pruned bundles included."""
    monkeypatch.setenv("AC_RUN_EDGES", str(run_edges))
    r = np.random.default_rng(run_edges)
    n, hub_in, hub_out = 1500, 900, 400
    src = np.concatenate([r.integers(0, n, 6000), r.integers(0, n, hub_in), np.full(hub_out, 7), r.integers(0, n, 130)])
    dst = np.concatenate([r.integers(0, n, 6000), np.full(hub_in, 3), r.integers(0, n, hub_out), np.full(130, 4)])
    data = W.Graph(r.normal(size=(n, 6)).astype(np.float32), r.normal(size=(len(src), 6)).astype(np.float32),
                   src.astype(np.int32), dst.astype(np.int32))
    patt = W.planted_pattern(data, 7, 10, 1)
    with Matcher(0) as m:
        m.set_option(AC_OPT_PRUNE, prune)
        m.set_data(data)
        m.set_pattern(patt)
        for n_iter in (0, 1, 7):
            bad, ratio = allclose_report(m.run(n_iter), O.run(g64(data), g64(patt), n_iter=n_iter))
            assert bad == 0, (n_iter, ratio)


@pytest.mark.parametrize("n,pn,k,kind", [
    (70_000, 1, 1, "random"), (6554, 10, 3, "random"), (6553, 10, 3, "random"),  # one side and the other of the size rule
    (40_000, 5, 512, "random"), (40_000, 5, 513, "random"), (300, 256, 75, "random"), (300, 256, 150, "random"),
    (50_000, 7, 40, "groups"), (50_000, 3, 9, "equal"), (20_000, 12, 20_000, "random"), (30_000, 4, 5, "nan"),
])
def test_topk_and_match_selection(n, pn, k, kind):
    """The k best of each column in order, ties by lower vertex: device and host selection, chunks of one row, values
    shared by a few vertices (groups) and by more than the device keeps (equal), and NaN columns."""
    data, patt = random_graph(n, 2 * n, 3, 2, n + k), random_graph(pn, pn, 3, 2, pn)
    if kind == "groups":
        data.vfeat[:] = data.vfeat[np.arange(n) % 900]
    elif kind == "equal":
        data.vfeat[:] = data.vfeat[0]
    elif kind == "nan":
        data.vfeat[n // 2] = np.nan
    with Matcher(0) as m:
        m.set_data(data)
        m.set_pattern(patt)
        mu = m.run(0)
        idx, val = m.topk(k)
        match = m.match(-8.0)
    if kind == "nan":
        assert np.isnan(mu).any()
        return  # no order to hold: the calls return, as they did
    want = np.stack([np.lexsort((np.arange(n), -mu[:, p]))[:k] for p in range(pn)])
    np.testing.assert_array_equal(idx, want)
    np.testing.assert_array_equal(val, np.take_along_axis(mu.T, want, axis=1))
    best = mu.argmax(axis=0)
    expect = np.zeros((n, pn), np.uint8)
    expect[best, np.arange(pn)] = np.where(mu[best, np.arange(pn)] >= -8.0, 2, 1)
    np.testing.assert_array_equal(match, expect)


@pytest.mark.parametrize("n,pn,k,ties", [(65_536, 1, 5, 4000), (65_536, 1, 5, 4200), (120_000, 7, 60, 500), (120_000, 7, 60, 30_000),
                                         (9000, 256, 3, 4096), (9000, 256, 3, 4097)])
def test_topk_keeps_up_to_a_limit_of_ties(n, pn, k, ties):
    """A stretch of vertices that share a column's best value, below and above the number of entries the device keeps."""
    data, patt = random_graph(n, n, 3, 2, n + k), random_graph(pn, pn, 3, 2, pn)
    data.vfeat[n // 3:n // 3 + ties] = patt.vfeat[0] + 1e-3
    with Matcher(0) as m:
        m.set_data(data)
        m.set_pattern(patt)
        mu = m.run(0)
        idx, val = m.topk(k)
    want = np.stack([np.lexsort((np.arange(n), -mu[:, p]))[:k] for p in range(pn)])
    np.testing.assert_array_equal(idx, want)
    np.testing.assert_array_equal(val, np.take_along_axis(mu.T, want, axis=1))


@pytest.mark.parametrize("where", ["data", "pattern"])
def test_selection_with_nan_columns(where):
    """A NaN is above nothing and nothing is above it: a column of them selects its first vertices, in order, and the other
    columns are selected as ever."""
    n, pn, k = 30_000, 4, 5
    data, patt = random_graph(n, 2 * n, 3, 2, n + k), random_graph(pn, pn, 3, 2, pn)
    (data if where == "data" else patt).vfeat[1] = np.nan
    with Matcher(0) as m:
        m.set_data(data)
        m.set_pattern(patt)
        mu = m.run(0)
        idx, val = m.topk(k)
        match = m.match(-8.0)
    expect = np.zeros((n, pn), np.uint8)
    for p in range(pn):
        nan = np.isnan(mu[:, p])
        assert nan.all() == (where == "data" or p == 1) and nan.all() == nan.any()
        want = np.arange(k) if nan.all() else np.lexsort((np.arange(n), -mu[:, p]))[:k]
        np.testing.assert_array_equal(idx[p], want)
        np.testing.assert_array_equal(val[p], mu[want, p])
        expect[want[0], p] = 2 if mu[want[0], p] >= -8.0 else 1
    np.testing.assert_array_equal(match, expect)


@pytest.mark.parametrize("run_edges", [4, 16, 128])
def test_gradients_do_not_depend_on_run_lengths(run_edges, monkeypatch):
    """The recorded least-cost out-edges and argmax in-edges of hubs in one to hundreds of pieces, equal costs among
    them: the gradients equal those of one piece per vertex to the rounding of the log-sum-exp merges (the forward
    quantities differ by about 1e-7 of their size; 2e-5 allows for the sums over iterations and edges)."""
    r = np.random.default_rng(5)
    n = 700
    src = np.concatenate([r.integers(0, n, 4000), r.integers(0, n, 600), np.full(600, 7)])
    dst = np.concatenate([r.integers(0, n, 4000), np.full(600, 3), r.integers(0, n, 600)])
    ef = r.normal(size=(len(src), 6)).astype(np.float32)
    ef[-300:] = ef[-600:-300]  # equal costs among the hub's out-edges
    data = W.Graph(r.normal(size=(n, 6)).astype(np.float32), ef, src.astype(np.int32), dst.astype(np.int32))
    patt = W.planted_pattern(data, 6, 9, 2, sigma=0.3)
    grad = np.zeros((n, 6), np.float32)
    grad[patt.vmap, np.arange(6)] = -1.0 / 6

    def run(L):
        monkeypatch.setenv("AC_RUN_EDGES", str(L))
        with Matcher(0) as m:
            m.set_option(AC_OPT_TAPE, 1)
            m.set_data(data)
            m.set_pattern(patt)
            m.run()
            return m.backward(grad)

    for got, want in zip(run(run_edges), run(4096)):
        np.testing.assert_allclose(got, want, rtol=0, atol=2e-5 * np.abs(want).max())


@pytest.mark.parametrize("pe", [3, 70, 130, 250])
@pytest.mark.parametrize("pieces", [3, 4, 5, 31, 32, 33, 300])
def test_hub_pieces(pe, pieces, monkeypatch):
    """Vertices at the piece counts where a group, a wave and a block take over, beside vertices of two and three
    pieces, for patterns that leave a wave one group of lanes to many; recorded and plain walks agree bit for bit."""
    monkeypatch.setenv("AC_RUN_EDGES", "4")
    r = np.random.default_rng(pieces)
    n, hub = 120, 4 * pieces
    src = np.concatenate([r.integers(8, n, 900), r.integers(8, n, hub), np.full(hub, 5), r.integers(8, n, hub)])
    dst = np.concatenate([r.integers(8, n, 900), np.full(hub, 3), r.integers(8, n, hub), np.full(hub, 4)])
    data = W.Graph(r.normal(size=(n, 6)).astype(np.float32), r.normal(size=(len(src), 6)).astype(np.float32),
                   src.astype(np.int32), dst.astype(np.int32))
    patt = random_graph(9, pe, 6, 6, pe)
    expect = O.run(g64(data), g64(patt), n_iter=4)
    got = []
    for tape in (0, 1):
        with Matcher(0) as m:
            m.set_option(AC_OPT_TAPE, tape)
            m.set_data(data)
            m.set_pattern(patt)
            got.append(m.run(4))
        bad, ratio = allclose_report(got[-1], expect)
        assert bad == 0, (tape, ratio)
    np.testing.assert_array_equal(got[0], got[1])


@pytest.mark.parametrize("n,m,pn,pe,K,dim", [
    (300, 900, 3, 200, 1, 3), (2000, 500, 40, 1, 2, 3), (1100, 3000, 256, 5, 1, 3),  # edges, isolated vertices, columns
    (5, 9, 1, 1, 1, 3), (17_000, 30_000, 7, 9, 3, 3),                 # less than a tile; more than 16 rows a block
    (400, 900, 16, 17, 1, 17), (400, 900, 33, 48, 1, 33), (400, 900, 49, 16, 1, 65),  # blocks of columns and features
])
def test_gradient_tiles(n, m, pn, pe, K, dim):
    """The adjoint's kernels over their tiles and lane groups, against finite differences of the oracle."""
    data = random_graph(n, m, dim, dim, n)
    patt = random_graph(pn, pe, dim, dim, pn + pe)
    patt.vmap = np.random.default_rng(pe).integers(0, n, pn)
    wv, we = weights(2, dim, dim)
    _, gv, ge = gpu_grad(data, patt, wv, we, 3, K=K)
    fv, fe = fd_grad(g64(data), g64(patt), patt.vmap, wv.copy(), we.copy(), 3)
    check_grad(np.concatenate([gv, ge]), np.concatenate([fv, fe]), f"dn={n} de={m} pn={pn} pe={pe} dim={dim}")


@pytest.mark.parametrize("pe", [3, 17, 70, 130])
@pytest.mark.parametrize("extra", [0, 500])
def test_one_vertex_takes_all_edges(pe, extra):
    """Stars in both directions with more pieces than a vertex is split into at its run length (8 edges): waves whose
    pieces are all one vertex's, with and without others among them; plain and recorded walks agree bit for bit."""
    r = np.random.default_rng(pe + extra)
    n, hub = 90, 12_000
    src = np.concatenate([r.integers(2, n, hub), np.full(hub, 1), r.integers(0, n, extra)])
    dst = np.concatenate([np.full(hub, 0), r.integers(2, n, hub), r.integers(0, n, extra)])
    data = W.Graph(r.normal(size=(n, 5)).astype(np.float32), r.normal(size=(len(src), 5)).astype(np.float32),
                   src.astype(np.int32), dst.astype(np.int32))
    patt = random_graph(9, pe, 5, 5, pe)
    expect = O.run(g64(data), g64(patt), n_iter=4)
    got = []
    for tape in (0, 1):
        with Matcher(0) as m:
            m.set_option(AC_OPT_TAPE, tape)
            m.set_data(data)
            m.set_pattern(patt)
            got.append([m.run(4) for _ in range(2)])
        bad, ratio = allclose_report(got[-1][1], expect)
        assert bad == 0, (tape, ratio)
    np.testing.assert_array_equal(got[0][0], got[0][1])
    np.testing.assert_array_equal(got[0][1], got[1][1])


@pytest.mark.parametrize("n,act,pn,pe", [(17_000, 300, 4, 5), (40_000, 3000, 9, 24), (9000, 60, 33, 40)])
def test_output_tiles_of_mostly_isolated_graphs(n, act, pn, pe):
    """Few vertices with edges among many: the iterations' tiles and the output passes' differ in height.  Plain, batched
    (a pattern's own columns beside another's) and taped runs, and the gradients."""
    data, patt = random_graph(act, 4 * act, 2, 2, n), random_graph(pn, pe, 2, 2, pn)
    r = np.random.default_rng(pe)
    ids = r.permutation(n)[:act].astype(np.int32)
    data = W.Graph(r.normal(size=(n, 2)).astype(np.float32), data.efeat, ids[data.src], ids[data.dst])
    expect = O.run(g64(data), g64(patt), n_iter=3)
    with Matcher(0) as m:
        m.set_data(data)
        m.set_pattern(patt)
        plain = m.run(3)
        m.batch_set_patterns([random_graph(5, 7, 2, 2, 1), patt])
        m.batch_run([2, 3])
        batched = m.batch_mu(1)
    for mu in (plain, batched):
        bad, ratio = allclose_report(mu, expect)
        assert bad == 0, ratio
    patt.vmap = r.integers(0, n, pn)
    wv, we = weights(2, 2, 2)
    _, gv, ge = gpu_grad(data, patt, wv, we, 2, K=1)
    fv, fe = fd_grad(g64(data), g64(patt), patt.vmap, wv.copy(), we.copy(), 2)
    check_grad(np.concatenate([gv, ge]), np.concatenate([fv, fe]), f"dn={n} act={act} pn={pn} pe={pe}")


@pytest.mark.parametrize("n,pn", [(1000, 10), (70_000, 9), (600_000, 9)])  # a direct copy, one thread's slots, four threads'
def test_page_locked_results_and_gradients(n, pn):
    """Results into, and the gradient out of, page-locked memory are those of ordinary memory."""
    data, patt = random_graph(n, n, 2, 2, n), random_graph(pn, pn, 2, 2, pn)
    grad = np.zeros((n, pn), np.float32)
    grad[np.arange(pn) * 7 % n, np.arange(pn)] = -1.0 / pn
    with Matcher(0) as m:
        m.set_option(AC_OPT_TAPE, 1)
        m.set_data(data)
        m.set_pattern(patt)
        mu = m.run(1)
        locked = torch.zeros(n, pn).pin_memory()
        _lib.check(m._L.ac_get_mu(m._h, locked.data_ptr()), m._h)
        np.testing.assert_array_equal(locked.numpy(), mu)
        want = m.backward(grad)
        locked.copy_(torch.from_numpy(grad))
        got = m.backward(locked.numpy())
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)


def test_a_pattern_that_does_not_fit_leaves_no_result(monkeypatch):
    """A pattern whose upload fails for want of memory takes the last result with it: what reads results says so, and the
    next pattern runs."""
    data, small, wide = random_graph(20_000, 40_000, 64, 4, 1), random_graph(4, 5, 64, 4, 2), random_graph(250, 20, 64, 4, 3)
    with Matcher(0) as m:
        m.set_option(AC_OPT_TAPE, 1)
        m.set_data(data)
        m.set_pattern(small)
        before = m.run(2)
        monkeypatch.setenv("AC_MAX_ALLOC_BYTES", "65536")
        with pytest.raises(ACError) as e:
            m.set_pattern(wide)
        assert e.value.code == _lib.AC_ERR_OOM
        monkeypatch.delenv("AC_MAX_ALLOC_BYTES")
        for read in (m.mu, m.match, lambda: m.topk(3), lambda: m.backward(np.zeros(m.sizes()[0::2], np.float32))):
            with pytest.raises(ACError) as e:
                read()
            assert e.value.code == _lib.AC_ERR_STATE
        m.set_pattern(small)
        np.testing.assert_array_equal(m.run(2), before)


def test_work_buffers_after_a_run_that_did_not_fit(monkeypatch):
    """A run that fails for want of memory leaves buffers of both patterns' sizes behind; the pattern that fitted runs again
    with the same result."""
    data, small, wide = random_graph(3000, 9000, 4, 4, 1), random_graph(4, 5, 4, 4, 2), random_graph(60, 90, 4, 4, 3)
    with Matcher(0) as m:
        m.set_data(data)
        m.set_pattern(small)
        before = m.run(2)
        m.set_pattern(wide)
        monkeypatch.setenv("AC_MAX_ALLOC_BYTES", str(600 * 1024))
        with pytest.raises(ACError) as e:
            m.run(2)
        assert e.value.code == _lib.AC_ERR_OOM
        m.set_pattern(small)
        np.testing.assert_array_equal(m.run(2), before)
        monkeypatch.delenv("AC_MAX_ALLOC_BYTES")
        m.set_pattern(wide)
        bad, ratio = allclose_report(m.run(2), O.run(g64(data), g64(wide), n_iter=2))
        assert bad == 0, ratio


def test_no_step_back_over_a_data_graph_that_did_not_fit(monkeypatch):
    """The graph of a taped run is gone once the next one's upload has failed; the result itself stays readable."""
    data, big = random_graph(500, 1500, 4, 4, 1), random_graph(20_000, 400, 4, 4, 2)
    with Matcher(0) as m:
        m.set_option(AC_OPT_TAPE, 1)
        m.set_data(data)
        m.set_pattern(random_graph(4, 5, 4, 4, 3))
        mu = m.run(2)
        monkeypatch.setenv("AC_MAX_ALLOC_BYTES", "65536")
        with pytest.raises(ACError) as e:
            m.set_data(big)
        assert e.value.code == _lib.AC_ERR_OOM
        np.testing.assert_array_equal(m.mu(), mu)
        with pytest.raises(ACError) as e:
            m.backward(np.zeros_like(mu))
        assert e.value.code == _lib.AC_ERR_STATE
