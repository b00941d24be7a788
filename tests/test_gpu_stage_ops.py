"""The stage operators at the edges of their kernels' tiles and dispatch rules, against plain references."""
import numpy as np
import pytest
import torch

from application_classification_amd.matcher import ac
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def dev(x):
    return torch.from_numpy(np.ascontiguousarray(x)).cuda()


@pytest.mark.parametrize("n_a,n_b,dim", [(3, 63, 5), (1, 64, 1), (4, 65, 31), (5, 257, 32), (17, 1000, 33), (33, 300, 64),
                                         (16, 524_289, 20), (24, 270_001, 35), (2, 100, 0)])
@pytest.mark.parametrize("offset", [0, 1])
def test_cdist_tiles(n_a, n_b, dim, offset):
    """Short and long b, partial tiles and chunks, groups of a rows, b rows off the 16-byte grid.  The FP64 sum is
    rounded once: within half an ulp (2^-24) of the FP64 root, and 2^-40 for the two sums' different orders."""
    r = np.random.default_rng(n_b)
    a = r.normal(size=(n_a, dim)).astype(np.float32)
    b = r.normal(size=(n_b, dim)).astype(np.float32)
    b[n_b // 2] = a[0] if dim else b[n_b // 2]
    db = torch.empty(n_b * dim + 4, device="cuda")
    db[offset:offset + n_b * dim] = dev(b.reshape(-1))
    da = dev(a) if dim else db
    out = torch.full((n_a * n_b + 64,), -7.0, device="cuda")
    ac.cdist(n_a, n_b, dim, da, db.data_ptr() + 4 * offset, out)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert (got[n_a * n_b:] == -7.0).all()  # nothing past the end
    ref = O.cdist(a, b)
    np.testing.assert_allclose(got[:n_a * n_b].reshape(n_a, n_b), ref, rtol=2.0**-24 + 2.0**-40, atol=0)


@pytest.mark.parametrize("n_a,n_b,dim", [
    (4, 95, 4), (4, 96, 4), (7, 400, 0),                              # b as a whole on both sides of the cache rule
    (15, 4166, 24), (15, 4167, 24), (15, 4167, 25), (1200, 50, 25),   # small calls of few features and others
    (16, 32_704, 25), (16, 32_705, 25), (17, 16_352, 25), (3, 64, 25), (5, 193, 300), (6000, 192, 25), (6000, 193, 25),
])
def test_cdist_split_of_small_calls(n_a, n_b, dim):
    """Both sides of the rules that choose a thread per output, groups of four a rows and short tiles."""
    test_cdist_tiles(n_a, n_b, dim, 0)


def order_key(x):
    """The total order of the scatter's maximum: floats by value, -0.0 below +0.0, NaNs beyond the infinities."""
    b = np.ascontiguousarray(x).view(np.int32).astype(np.int64)
    return np.where(b < 0, -(b & 0x7FFFFFFF) - 1, b)


@pytest.mark.parametrize("n_row,n_in,n_out,offset", [(1, 1, 1, 0), (3, 7, 2, 1), (5, 1023, 40, 2), (2, 1025, 1, 3),
                                                     (3, 8193, 700, 1), (16, 70_001, 3000, 0), (2, 0, 5, 0),
                                                     (3, 5, 4099, 1), (0, 5, 5000, 0),
                                                     (5000, 9, 4, 1), (40, 255, 60, 2), (40, 256, 60, 2)])
@pytest.mark.parametrize("fill", ["low", "mid", "special"])
def test_edge_max_reduce_edges(n_row, n_in, n_out, offset, fill):
    """Chunk edges, rows off the 16-byte grid, nodes shared by many and by neighbouring values, fills below, among and
    above the values, and infinities, signed zeros and NaNs on both sides.  A maximum: bit for bit."""
    r = np.random.default_rng(n_in)
    xe = r.normal(size=(n_row, n_in)).astype(np.float32)
    vy = np.full(n_row, {"low": -np.inf, "mid": 0.5, "special": 0.0}[fill], np.float32)
    if fill == "special":
        special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, -np.nan], np.float32)
        xe[:, :] = np.where(r.random(xe.shape) < 0.02, r.choice(special, xe.shape), xe)
        vy[:] = r.choice(special, n_row)
        xe.reshape(-1)[:2] = -0.0
    nodes = (r.integers(0, n_out, n_in) // 3 * 3 if n_in % 2 else np.sort(r.integers(0, n_out, n_in))).astype(np.int32)
    x = torch.empty(n_row * n_in + 4, device="cuda")
    x[offset:offset + n_row * n_in] = dev(xe.reshape(-1))
    out = torch.full((n_row * n_out + 8,), 3.0, device="cuda")
    ac.EdgeMaxReduce2_t(n_in, n_out, n_row, dev(vy), x.data_ptr() + 4 * offset, out, dev(nodes))
    torch.cuda.synchronize()
    key = np.repeat(order_key(vy)[:, None], n_out, axis=1)
    for i in range(n_row):
        np.maximum.at(key[i], nodes, order_key(xe[i]))
    got = out.cpu().numpy()
    np.testing.assert_array_equal(order_key(got[:n_row * n_out]).reshape(n_row, n_out), key)
    assert (got[n_row * n_out:] == 3.0).all()


@pytest.mark.parametrize("n_row,n_in,n_out,offset", [(128, 1024, 300, 1), (129, 1024, 300, 1), (257, 1023, 50, 2),
                                                     (256, 1023, 50, 2), (1, 131_072, 700, 3), (1, 131_073, 700, 3)])
@pytest.mark.parametrize("fill", ["low", "mid", "special"])
def test_edge_max_reduce_small_calls(n_row, n_in, n_out, offset, fill):
    """Both sides of the number of values up to which each has a thread of its own."""
    test_edge_max_reduce_edges(n_row, n_in, n_out, offset, fill)


def at_offset(x, offset):
    """x on the device, `offset` floats off an aligned start, and room behind it."""
    buf = torch.full((x.size + 8,), 3.0, device="cuda")
    buf[offset:offset + x.size] = dev(x.reshape(-1))
    return buf, buf.data_ptr() + 4 * offset


@pytest.mark.parametrize("n_row,n_col,offset", [(3, 1, 1), (2, 255, 0), (2, 257, 3), (3, 4096, 1), (2, 4097, 0),
                                                (2, 32_768, 2), (3, 32_769, 1), (2, 70_001, 3)])
def test_row_log_softmax_edges(n_row, n_col, offset):
    """The one-launch and three-launch rows and their blocks' edges.  Each term is an FP32 exponential of a difference of
    at most D: relative error (1 + D) 2^-23, which bounds the logarithm's; the result is rounded once."""
    r = np.random.default_rng(n_col)
    x = (r.normal(size=(n_row, n_col)) * 4).astype(np.float32)
    if n_col > 1:
        x[0, n_col // 2] = -np.inf
        x[0, n_col - 1] = x[0].max()  # the maximum more than once
    buf, ptr = at_offset(x, offset)
    ac.RowSoftmax2(n_row, n_col, ptr)
    torch.cuda.synchronize()
    got = buf.cpu().numpy()
    assert (got[offset + x.size:] == 3.0).all() and (got[:offset] == 3.0).all()
    ref = O.row_log_softmax(x.astype(np.float64))
    spread = np.ptp(np.where(np.isfinite(x), x, 0.0))
    np.testing.assert_allclose(got[offset:offset + x.size].reshape(x.shape), ref, rtol=2.0**-24,
                               atol=(1 + spread) * 2.0**-23)


@pytest.mark.parametrize("n_col", [300, 5000, 20_000, 40_000])
def test_row_log_softmax_specials(n_col):
    """One +inf takes the whole mass; two, a NaN, or nothing but -inf leave no number."""
    x = np.random.default_rng(n_col).normal(size=(5, n_col)).astype(np.float32)
    x[0, 7] = np.inf
    x[1, [3, n_col - 1]] = np.inf
    x[2, [4, n_col // 2]] = np.inf
    x[3] = -np.inf
    x[4, 9] = np.nan
    buf, ptr = at_offset(x, 0)
    ac.RowSoftmax2(5, n_col, ptr)
    torch.cuda.synchronize()
    got = buf.cpu().numpy()[:x.size].reshape(x.shape)
    assert np.isnan(got[0, 7]) and (np.delete(got[0], 7) == -np.inf).all()
    assert np.isnan(got[1:]).all()


@pytest.mark.parametrize("n_row,n_col,offset", [(256, 4097, 1), (257, 4097, 1), (257, 8192, 0), (257, 8193, 3),
                                                (300, 16_384, 2), (257, 16_385, 1)])
def test_row_log_softmax_many_rows(n_row, n_col, offset):
    """More rows than CUs take the smallest block that holds one: both sides of each width."""
    test_row_log_softmax_edges(n_row, n_col, offset)
    x = np.random.default_rng(n_col).normal(size=(n_row, n_col)).astype(np.float32)
    x[0, 7] = np.inf
    x[1, [3, n_col - 1]] = np.inf
    x[2] = -np.inf
    x[3, 9] = np.nan
    x[n_row - 1, 1:] = -np.inf
    buf, ptr = at_offset(x, offset)
    ac.RowSoftmax2(n_row, n_col, ptr)
    torch.cuda.synchronize()
    got = buf.cpu().numpy()[offset:offset + x.size].reshape(x.shape)
    assert np.isnan(got[0, 7]) and (np.delete(got[0], 7) == -np.inf).all()
    assert np.isnan(got[1:4]).all()
    assert got[n_row - 1, 0] == 0.0 and (got[n_row - 1, 1:] == -np.inf).all()


@pytest.mark.parametrize("n_row,n_col,offset", [(1, 1, 0), (300, 3, 1), (3, 32_768, 1), (3, 32_769, 2), (2, 100_001, 3),
                                                (4, 8192, 1), (4, 8193, 1)])
def test_row_max_edges(n_row, n_col, offset):
    x = -np.abs(np.random.default_rng(n_col).normal(size=(n_row, n_col))).astype(np.float32) - 1.0
    x[0, :] = -np.inf
    buf, ptr = at_offset(x, offset)
    out = torch.full((n_row + 4,), 3.0, device="cuda")
    ac.RowMax2(n_row, n_col, ptr, out)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy()[:n_row], x.max(axis=1))
    assert (out.cpu().numpy()[n_row:] == 3.0).all()


@pytest.mark.parametrize("n_row,n_col,offset", [(7, 63, 1), (5, 64, 0), (5, 65, 2), (3, 1023, 3), (3, 1024, 1),
                                                (3, 1025, 1), (70_000, 5, 1)])
def test_row_max_short_rows(n_row, n_col, offset):
    """Rows of a wave's and of a block's width."""
    test_row_max_edges(n_row, n_col, offset)


@pytest.mark.parametrize("n_row", [2**23 + 1, 2**24 + 3, 2**25 + 1])
def test_more_rows_than_one_grid_takes(n_row):
    """Row operators on rows of three: beyond 2^23 rows of 256 threads, 2^25 of 64, a launch takes a slice of them.  Maxima
    bit for bit; the log-softmax against FP64 as in test_row_log_softmax_edges, with values within [-4, 4]."""
    gen = torch.Generator("cuda").manual_seed(n_row)
    x = torch.rand(n_row, 3, device="cuda", generator=gen) * 8 - 4
    top = torch.full((n_row + 4,), 3.0, device="cuda")
    ac.RowMax2(n_row, 3, x, top)
    assert torch.equal(top[:n_row], x.amax(1)) and (top[n_row:] == 3.0).all()
    got = torch.cat([x.flatten(), torch.full((4,), 3.0, device="cuda")])
    ac.RowSoftmax2(n_row, 3, got)
    assert (got[3 * n_row:] == 3.0).all()
    worst = 0.0
    for a in range(0, n_row, 1 << 22):
        ref = torch.log_softmax(x[a:a + (1 << 22)].double(), 1)
        worst = max(worst, (got[3 * a:3 * a + ref.numel()].double().view(-1, 3) - ref).abs().max().item())
    assert worst <= 9 * 2.0**-23 + 9 * 2.0**-24, worst


@pytest.mark.parametrize("n_in,n_out,P,Q,offset", [(8, 8, 3, 5, 0), (1028, 2052, 4, 70, 0), (1028, 2052, 4, 70, 1),
                                                   (1027, 1030, 5, 130, 0), (4096, 1000, 2, 64, 0), (40, 44, 2, 700, 0),
                                                   (7, 5, 3, 0, 0)])
def test_compute_mu_edges(n_in, n_out, P, Q, offset):
    """Both widths of access, columns on one side only, no pattern edge at all, loops, and more incident pattern edges
    than one list holds.  FP64 sums in one order, rounded once: bit for bit."""
    r = np.random.default_rng(Q)
    cv, f, b = (r.normal(size=s).astype(np.float32) for s in ((P, n_out), (Q, n_in), (Q, n_in)))
    src, dst = (r.integers(0, P, Q).astype(np.int32) for _ in range(2))
    if Q:
        src[0] = dst[0] = P - 1
    keep = [at_offset(x, offset) for x in (cv, f, b)]
    mu = torch.full((P * n_out + 8,), 3.0, device="cuda")
    ac.ComputeMU2_t(n_in, Q, n_out, P, keep[0][1], keep[1][1], keep[2][1], dev(src), dev(dst),
                    mu.data_ptr() + 4 * offset)
    torch.cuda.synchronize()
    ref = -cv.astype(np.float64)
    n = min(n_in, n_out)
    for q in range(Q):
        ref[dst[q], :n] += f[q, :n]
        ref[src[q], :n] += b[q, :n]
    got = mu.cpu().numpy()
    np.testing.assert_array_equal(got[offset:offset + P * n_out].reshape(P, n_out), ref.astype(np.float32))
    assert (got[offset + P * n_out:] == 3.0).all() and (got[:offset] == 3.0).all()


@pytest.mark.parametrize("n_in,n_out,P,Q,offset", [(40, 44, 1, 192, 0), (40, 44, 1, 256, 1), (40, 44, 1, 257, 0), (1028, 2052, 2, 2100, 0),
                                                   (300, 300, 4100, 70, 0), (9, 5000, 3, 4000, 2)])
def test_compute_mu_many_incident_edges(n_in, n_out, P, Q, offset):
    """Lists that are just full, and several to a pattern vertex; more pattern vertices than the grid has rows."""
    test_compute_mu_edges(n_in, n_out, P, Q, offset)


@pytest.mark.parametrize("n_rows,n_cols", [(1, 1), (64, 64), (63, 65), (3, 1000), (1000, 3), (16, 100_003), (70_001, 12)])
def test_transpose_tiles(n_rows, n_cols):
    x = np.arange(n_rows * n_cols, dtype=np.float32).reshape(n_rows, n_cols)
    out = torch.full((x.size + 8,), -1.0, device="cuda")
    ac.transpose(dev(x), out, n_rows, n_cols)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[:x.size].reshape(n_cols, n_rows), x.T)
    assert (got[x.size:] == -1.0).all()
