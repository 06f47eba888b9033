"""Graph preprocessing on the GPU vs the oracle -- all bit-exact.

edge_list_to_csr (reference src/graph_loader.cpp:211-281), CSR validation
(src/tensor.cpp:46-86), add_self_loops (src/layers.cpp:71-144) and gcn_norm
(src/layers.cpp:158-208), including the degree and 1/sqrt(deg) arrays.
"""
import numpy as np
import pytest

import oracle
from helpers import bits, random_csr

pytestmark = pytest.mark.gpu


def _dev(gpu, a):
    import tinygnn_amd as tg
    return tg.DeviceCSR.from_numpy(a.n_rows, a.n_cols, a.row_ptr, a.col_ind, a.val)


def _edges(gpu, src, dst):
    return (gpu.from_numpy(np.ascontiguousarray(src, np.int32)).cuda(),
            gpu.from_numpy(np.ascontiguousarray(dst, np.int32)).cuda())


@pytest.mark.parametrize("n,e,dmax,seed", [
    (1, 0, 1, 0), (5, 1, 1, 1), (300, 4000, 64, 2), (2000, 60000, 900, 3),
    (500, 120000, 40000, 4),     # a bucket over 32,768: sorted through memory
    (64, 200000, 100000, 5),
])
def test_edge_list_to_csr_bitexact(gpu, restate, n, e, dmax, seed):
    import tinygnn_amd as tg
    from tinygnn_amd import synth
    if e == 0:
        src = dst = np.zeros(0, np.int32)
    elif n <= 5:
        rng = np.random.default_rng(seed)
        src = rng.integers(0, n, size=e).astype(np.int32)
        dst = rng.integers(0, n, size=e).astype(np.int32)
    else:
        src, dst = synth.powerlaw_edges(n, e, alpha=2.1, dmax=dmax, seed=seed)
    want = restate.edge_list_to_csr(src, dst, n)
    s, d = _edges(gpu, src, dst)
    got = tg.edge_list_to_csr(s, d, n)
    rp, ci, v = got.to_numpy()
    np.testing.assert_array_equal(rp, want.row_ptr)
    np.testing.assert_array_equal(ci, want.col_ind)
    np.testing.assert_array_equal(bits(v), bits(want.val))


@pytest.mark.parametrize("n,e,kind", [
    (1, 1, "uniform"), (2, 5000, "uniform"), (7, 16384, "uniform"), (7, 16385, "sorted"),
    (4096, 40000, "uniform"), (4097, 1, "uniform"), (70001, 300000, "one_row"),
    (70001, 300000, "sorted"), (1 << 22, 50000, "uniform"), ((1 << 22) + 1, 50000, "uniform"),
    (3, 32768, "one_row"), (3, 32769, "one_row"),   # LDS sort, the sort through memory
    (3, 262144, "one_row"), (3, 262145, "one_row"),  # that one, the general build
    (300000, 5000000, "hubs"),
])
def test_edge_list_to_csr_partition_edges(gpu, restate, n, e, kind):
    """The partition-and-sort build at the edges of its buckets, tiles, sort
    paths and sizes, and the general build just past them."""
    import tinygnn_amd as tg
    rng = np.random.default_rng(n + e)
    src = rng.integers(0, n, size=e).astype(np.int32)
    if kind == "sorted":
        src.sort()
    elif kind == "one_row":
        src[:] = n - 1
    elif kind == "hubs":
        src[: e // 4] = rng.integers(1000, 1020, size=e // 4)
        src[e // 4: e // 2] = n - 1 - src[e // 4: e // 2] % 4
        rng.shuffle(src)
    dst = rng.integers(0, n, size=e).astype(np.int32)
    dst[:: 7] = n - 1
    want = restate.edge_list_to_csr(src, dst, n)
    rp, ci, v = tg.edge_list_to_csr(*_edges(gpu, src, dst), n).to_numpy()
    np.testing.assert_array_equal(rp, want.row_ptr)
    np.testing.assert_array_equal(ci, want.col_ind)
    np.testing.assert_array_equal(bits(v), bits(want.val))


@pytest.mark.parametrize("lens", [
    [270000], [65, 100, 1023, 1024, 270000, 64, 2, 1],     # with every length class
    [1025, 2000, 16383, 16384, 300000, 1024, 0, 63],
    [16385, 17000, 270000, 40000, 0, 131073, 70, 1500],    # several long rows: segments, stages
])
def test_edge_list_to_csr_general_rows(gpu, restate, lens):
    """The general build, which a bucket of more than 262,144 edges takes: its
    sorts of rows up to 64, 1,024 and 16,384 entries and of several longer
    ones, beside 500 rows of a few edges."""
    import tinygnn_amd as tg
    rng = np.random.default_rng(len(lens) + lens[0])
    n = 600
    deg = rng.integers(0, 70, size=n)
    deg[rng.choice(n, size=len(lens), replace=False)] = lens
    src = np.repeat(np.arange(n), deg).astype(np.int32)
    rng.shuffle(src)
    dst = rng.integers(0, n, size=src.size).astype(np.int32)
    want = restate.edge_list_to_csr(src, dst, n)
    rp, ci, v = tg.edge_list_to_csr(*_edges(gpu, src, dst), n).to_numpy()
    np.testing.assert_array_equal(rp, want.row_ptr)
    np.testing.assert_array_equal(ci, want.col_ind)
    np.testing.assert_array_equal(bits(v), bits(want.val))


@pytest.mark.parametrize("n,rows", [
    (65536, [0]), (65536, [65535]), (60000, [30000] * 100), (5000, [0, 64, 128, 4999]),
    (5000, [64, 129, 4936]), (5000, [63, 128, 193, 4935]), ((1 << 22), [7, 1 << 20, (1 << 22) - 1]),
    (3000, [1500] * 40000),   # sorted through memory
])
def test_edge_list_to_csr_empty_rows(gpu, restate, n, rows):
    """Runs of empty rows of any length, 64 and 65 among them, between the
    rows of a few edges."""
    import tinygnn_amd as tg
    src = np.array(rows, np.int32)
    dst = np.random.default_rng(n).integers(0, n, size=src.size).astype(np.int32)
    want = restate.edge_list_to_csr(src, dst, n)
    rp, ci, v = tg.edge_list_to_csr(*_edges(gpu, src, dst), n).to_numpy()
    np.testing.assert_array_equal(rp, want.row_ptr)
    np.testing.assert_array_equal(ci, want.col_ind)
    np.testing.assert_array_equal(bits(v), bits(want.val))


@pytest.mark.parametrize("e", [1023, 1024, 1025, 262143, 262144, 262145])
def test_edge_list_to_csr_shares(gpu, restate, e):
    """The partition's shares of 1,024 edges, and whole tiles past 262,144."""
    import tinygnn_amd as tg
    rng = np.random.default_rng(e)
    src = np.sort(rng.integers(0, 9000, size=e)).astype(np.int32)
    dst = rng.integers(0, 9000, size=e).astype(np.int32)
    want = restate.edge_list_to_csr(src, dst, 9000)
    rp, ci, v = tg.edge_list_to_csr(*_edges(gpu, src, dst), 9000).to_numpy()
    np.testing.assert_array_equal(rp, want.row_ptr)
    np.testing.assert_array_equal(ci, want.col_ind)


def test_edge_list_to_csr_duplicates_and_self_edges(gpu, restate):
    import tinygnn_amd as tg
    rng = np.random.default_rng(9)
    src = rng.integers(0, 40, size=5000).astype(np.int32)
    dst = rng.integers(0, 40, size=5000).astype(np.int32)  # many duplicates, self edges
    want = restate.edge_list_to_csr(src, dst, 40)
    got = tg.edge_list_to_csr(*_edges(gpu, src, dst), 40)
    np.testing.assert_array_equal(got.to_numpy()[0], want.row_ptr)
    np.testing.assert_array_equal(got.to_numpy()[1], want.col_ind)


@pytest.mark.parametrize("bad", [("src", 7, 10), ("dst", 3, -1), ("src", 0, 4)])
def test_edge_list_to_csr_errors(gpu, restate, bad):
    """Message of graph_loader.cpp:227-242 for the first bad endpoint."""
    import tinygnn_amd as tg
    which, pos, value = bad
    src = np.arange(12, dtype=np.int32) % 4
    dst = (np.arange(12, dtype=np.int32) + 1) % 4
    (src if which == "src" else dst)[pos] = value
    (dst if which == "src" else src)[pos + 2] = 99  # a later bad edge must not be reported
    with pytest.raises(oracle.OracleError) as want:
        restate.edge_list_to_csr(src, dst, 4)
    with pytest.raises(tg.InvalidArgument) as got:
        tg.edge_list_to_csr(*_edges(gpu, src, dst), 4)
    assert str(got.value) == str(want.value)


def test_edge_list_to_csr_zero_nodes(gpu):
    import tinygnn_amd as tg
    s, d = _edges(gpu, np.zeros(0, np.int32), np.zeros(0, np.int32))
    a = tg.edge_list_to_csr(s, d, 0)
    assert a.row_ptr.cpu().tolist() == [0]
    s, d = _edges(gpu, np.zeros(1, np.int32), np.zeros(1, np.int32))
    with pytest.raises(tg.InvalidArgument, match="num_nodes is 0 but edges is non-empty"):
        tg.edge_list_to_csr(s, d, 0)


def test_csr_validate(gpu, reference):
    import tinygnn_amd as tg
    rp = np.array([0, 2, 3, 3, 5], np.int32)
    ci = np.array([0, 3, 1, 2, 0], np.int32)
    ok = oracle.CSR(4, 4, rp, ci, np.ones(5, np.float32))
    tg.csr_validate(_dev(gpu, ok))
    cases = [
        oracle.CSR(4, 4, rp, np.array([0, 3, 1, 4, 9], np.int32), np.ones(5, np.float32)),
        oracle.CSR(4, 4, np.array([0, 2, 1, 3, 5], np.int32), ci, np.ones(5, np.float32)),
        oracle.CSR(4, 4, np.array([0, 2, 3, 3, 4], np.int32), ci[:5], np.ones(5, np.float32)),
    ]
    for c in cases:
        with pytest.raises(oracle.OracleError) as want:
            reference.csr_raw(c.n_rows, c.n_cols, c.row_ptr, c.col_ind, c.val)
        with pytest.raises(tg.InvalidArgument) as got:
            tg.csr_validate(_dev(gpu, c))
        assert str(got.value) == str(want.value)


def _graph_with_diagonals(restate, seed, n=400, unsorted=False):
    rng = np.random.default_rng(seed)
    a = random_csr(rng, n, n, avg_deg=7, max_deg=300, empty_frac=0.15)
    rows = np.repeat(np.arange(n), np.diff(a.row_ptr))
    diag = rng.choice(n, size=n // 4, replace=False)
    dup = rng.choice(diag, size=n // 20, replace=False)
    src = np.concatenate([rows, diag, dup]).astype(np.int32)
    dst = np.concatenate([a.col_ind, diag, dup]).astype(np.int32)
    g = restate.edge_list_to_csr(src, dst, n)
    g.val[:] = (rng.random(g.nnz) * 3 - 1).astype(np.float32)
    if unsorted:
        for i in range(n):
            seg = slice(g.row_ptr[i], g.row_ptr[i + 1])
            p = rng.permutation(g.row_ptr[i + 1] - g.row_ptr[i])
            g.col_ind[seg] = g.col_ind[seg][p]
            g.val[seg] = g.val[seg][p]
    return g


@pytest.mark.parametrize("seed,unsorted", [(0, False), (1, False), (2, True)])
def test_add_self_loops_bitexact(gpu, restate, seed, unsorted):
    import tinygnn_amd as tg
    a = _graph_with_diagonals(restate, seed, unsorted=unsorted)
    want = restate.add_self_loops(a)
    got = tg.add_self_loops(_dev(gpu, a))
    rp, ci, v = got.to_numpy()
    np.testing.assert_array_equal(rp, want.row_ptr)
    np.testing.assert_array_equal(ci, want.col_ind)
    np.testing.assert_array_equal(bits(v), bits(want.val))


@pytest.mark.parametrize("seed,unsorted,weights", [(3, False, "unit"), (4, False, "real"),
                                                   (5, True, "real")])
def test_gcn_norm_bitexact(gpu, restate, seed, unsorted, weights):
    import tinygnn_amd as tg
    a = _graph_with_diagonals(restate, seed, unsorted=unsorted)
    if weights == "unit":
        a.val[:] = 1.0
    else:
        a.val[:] = np.abs(a.val) + 0.01  # positive degrees, non-integer sums
    want, wdeg, wdis = restate.gcn_norm(a, with_degrees=True)
    got, deg, dis = tg.gcn_norm(_dev(gpu, a), with_degrees=True)
    rp, ci, v = got.to_numpy()
    np.testing.assert_array_equal(rp, want.row_ptr)
    np.testing.assert_array_equal(ci, want.col_ind)
    np.testing.assert_array_equal(bits(deg.cpu().numpy()), bits(wdeg))
    np.testing.assert_array_equal(bits(dis.cpu().numpy()), bits(wdis))
    np.testing.assert_array_equal(bits(v), bits(want.val))


@pytest.mark.parametrize("weights", ["unit", "real", "big_int", "neg_int"])
def test_self_loops_long_rows(gpu, restate, weights):
    """Rows up to 9,000 entries (the workgroup-per-row kernels) with
    diagonals present and absent.  Unit and small signed integers take the
    exact parallel degree; real values and integers whose magnitudes sum past
    2^24 take the sequential one."""
    import tinygnn_amd as tg
    rng = np.random.default_rng(17)
    n = 3000
    a = random_csr(rng, n, n, avg_deg=20, max_deg=9000)
    rows = np.repeat(np.arange(n), np.diff(a.row_ptr))
    diag = rng.choice(n, size=n // 3, replace=False)
    src = np.concatenate([rows, diag]).astype(np.int32)
    dst = np.concatenate([a.col_ind, diag]).astype(np.int32)
    g = restate.edge_list_to_csr(src, dst, n)
    if weights == "unit":
        g.val[:] = 1.0
    elif weights == "real":
        g.val[:] = (rng.random(g.nnz) * 2 + 0.01).astype(np.float32)
    elif weights == "big_int":
        g.val[:] = rng.integers(1, 20000, g.nnz).astype(np.float32)
    else:
        g.val[:] = rng.integers(-5, 6, g.nnz).astype(np.float32)
    assert np.diff(g.row_ptr).max() > 2048
    want = restate.add_self_loops(g)
    rp, ci, v = tg.add_self_loops(_dev(gpu, g)).to_numpy()
    np.testing.assert_array_equal(rp, want.row_ptr)
    np.testing.assert_array_equal(ci, want.col_ind)
    np.testing.assert_array_equal(bits(v), bits(want.val))
    want, wdeg, wdis = restate.gcn_norm(g, with_degrees=True)
    got, deg, dis = tg.gcn_norm(_dev(gpu, g), with_degrees=True)
    np.testing.assert_array_equal(bits(deg.cpu().numpy()), bits(wdeg))
    np.testing.assert_array_equal(bits(dis.cpu().numpy()), bits(wdis))
    np.testing.assert_array_equal(bits(got.val.cpu().numpy()), bits(want.val))


@pytest.mark.parametrize("diag", ["none", "first", "last", "two", "inf"])
def test_gcn_norm_sequential_degrees(gpu, restate, diag):
    """Real-valued rows around every step of the in-order degree sums (16, 64,
    1,024 entries; more than 1,024: a workgroup with an LDS stage), columns in
    random order, the diagonal absent, at either end or twice, negative zeros
    and, in one case, an infinite degree: every bit of the degree and of
    1/sqrt(degree)."""
    import tinygnn_amd as tg
    rng = np.random.default_rng(29)
    lens = [0, 1, 2, 15, 16, 17, 31, 47, 63, 64, 65, 79, 127, 128, 129, 1007, 1022, 1023, 1024,
            1025, 1026, 1055, 1056, 1088, 2047, 2048, 2049, 3071, 4096, 7001]
    n = 8000
    rp, ci, v = [0], [], []
    for i in range(n):
        m = lens[i] if i < len(lens) else 0
        c = (i + 1 + rng.integers(0, n - 1, size=m)) % n  # never the diagonal
        if m and diag == "first":
            c[0] = i
        elif m and diag == "last":
            c[-1] = i
        elif m and diag == "two":
            c[rng.integers(0, m, size=2)] = i
        x = (rng.random(m) * 3).astype(np.float32)
        x[rng.random(m) < 0.1] = -0.0
        if diag == "inf" and m > 20:
            x[m // 2] = np.inf
        ci.append(c)
        v.append(x)
        rp.append(rp[-1] + m)
    a = oracle.CSR(n, n, np.array(rp, np.int32), np.concatenate(ci).astype(np.int32),
                   np.concatenate(v))
    _, wdeg, wdis = restate.gcn_norm(a, with_degrees=True)
    _, deg, dis = tg.gcn_norm(_dev(gpu, a), with_degrees=True)
    np.testing.assert_array_equal(bits(deg.cpu().numpy()), bits(wdeg))
    np.testing.assert_array_equal(bits(dis.cpu().numpy()), bits(wdis))


@pytest.mark.parametrize("in_off,out_off", [(0, 1), (1, 0), (1, 1), (0, 2), (3, 0)])
def test_self_loops_pointer_alignment(gpu, restate, in_off, out_off):
    """col_ind / val inputs and outputs starting 4-12 bytes past a 16-byte
    boundary (C-ABI callers may pass any element-aligned pointer): the
    128-bit read and aligned-granule copy paths and the entry-wise ones give
    the same bits."""
    import tinygnn_amd as tg
    torch = gpu
    rng = np.random.default_rng(23)
    n = 700
    a = random_csr(rng, n, n, avg_deg=12, max_deg=3000, empty_frac=0.1)
    rows = np.repeat(np.arange(n), np.diff(a.row_ptr))
    diag = rng.choice(n, size=n // 3, replace=False)
    g = restate.edge_list_to_csr(np.concatenate([rows, diag]).astype(np.int32),
                                 np.concatenate([a.col_ind, diag]).astype(np.int32), n)
    g.val[:] = (rng.random(g.nnz) * 2 + 0.01).astype(np.float32)
    assert np.diff(g.row_ptr).max() > 2048  # the workgroup-per-row kernels too

    def placed(x, off):  # x's values in a device buffer, starting off elements in
        buf = torch.zeros(x.size + off + 4, dtype=torch.from_numpy(x[:1]).dtype).cuda()
        buf[off:off + x.size] = torch.from_numpy(x).cuda()
        return buf, buf.data_ptr() + off * x.itemsize

    rp = torch.from_numpy(g.row_ptr).cuda()
    ci_buf, ci_p = placed(g.col_ind, in_off)
    v_buf, v_p = placed(g.val, in_off)
    cap = g.nnz + n
    for norm in (False, True):
        want = restate.gcn_norm(g) if norm else restate.add_self_loops(g)
        rp_o = torch.empty(n + 1, dtype=torch.int32).cuda()
        co_buf, co_p = placed(np.zeros(cap, np.int32), out_off)
        vo_buf, vo_p = placed(np.zeros(cap, np.float32), out_off)
        if norm:
            st = tg.lib.tg_gcn_norm(n, g.nnz, rp.data_ptr(), ci_p, v_p, rp_o.data_ptr(), co_p,
                                    vo_p, None, None, None, 0, None)
        else:
            st = tg.lib.tg_add_self_loops(n, g.nnz, rp.data_ptr(), ci_p, v_p, rp_o.data_ptr(),
                                          co_p, vo_p, None, 0, None)
        tg.lib.check(st)
        torch.cuda.synchronize()
        nnz = want.row_ptr[-1]
        np.testing.assert_array_equal(rp_o.cpu().numpy(), want.row_ptr)
        ci_o = co_buf.cpu().numpy()[out_off:out_off + nnz]
        v_o = vo_buf.cpu().numpy()[out_off:out_off + nnz]
        np.testing.assert_array_equal(ci_o, want.col_ind)
        np.testing.assert_array_equal(bits(v_o), bits(want.val))
        # nothing written outside the outputs
        assert not co_buf.cpu().numpy()[:out_off].any()
        assert not co_buf.cpu().numpy()[out_off + nnz:].any()


def test_gcn_norm_degree_sweep(gpu, restate):
    """1/sqrt(deg) correctly rounded for every integer degree 1..4096 (star-like
    rows of unit weights): the device sqrt and divide must round exactly as
    the host's."""
    import tinygnn_amd as tg
    n = 4097
    rows = np.arange(1, n)
    k = rows % 4096
    src = np.repeat(rows, k)
    start = np.repeat(np.cumsum(k) - k, k)
    dst = (np.arange(src.size) - start + src + 1) % n
    a = restate.edge_list_to_csr(src.astype(np.int32), dst.astype(np.int32), n)
    want, wdeg, wdis = restate.gcn_norm(a, with_degrees=True)
    got, deg, dis = tg.gcn_norm(_dev(gpu, a), with_degrees=True)
    np.testing.assert_array_equal(bits(dis.cpu().numpy()), bits(wdis))
    np.testing.assert_array_equal(bits(got.val.cpu().numpy()), bits(want.val))


def test_self_loops_known_answers(gpu):
    """test_gcn.cpp:288-327 path graph through the GPU path."""
    import tinygnn_amd as tg
    s, d = _edges(gpu, [0, 1, 1, 2], [1, 0, 2, 1])
    a = tg.edge_list_to_csr(s, d, 3)
    nrm = tg.gcn_norm(a)
    s6 = 1 / np.sqrt(6)
    np.testing.assert_array_equal(nrm.row_ptr.cpu().numpy(), [0, 2, 5, 7])
    np.testing.assert_allclose(nrm.val.cpu().numpy(), [0.5, s6, s6, 1 / 3, s6, s6, 0.5],
                               atol=1e-6)


def test_square_required(gpu):
    import tinygnn_amd as tg
    a = oracle.CSR(3, 4, np.array([0, 1, 1, 2], np.int32), np.array([1, 3], np.int32),
                   np.ones(2, np.float32))
    with pytest.raises(tg.InvalidArgument, match="square"):
        tg.add_self_loops(_dev(gpu, a))


def test_temporaries_on_streams_and_threads(gpu, restate):
    """Calls that bring no workspace, from three threads on streams of their
    own, again and again: their temporaries, reused in stream order, do not mix."""
    import threading
    import tinygnn_amd as tg
    torch = gpu
    want, dev = [], []
    for seed in (31, 32, 33):
        a = random_csr(np.random.default_rng(seed), 3000 + seed, 3000 + seed, avg_deg=8,
                       max_deg=2500)
        a.val[:] = np.abs(a.val) + 0.01
        want.append(restate.gcn_norm(a))
        dev.append(_dev(gpu, a))
    torch.cuda.synchronize()
    bad = []

    def work(k):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(10):
                rp, ci, v = tg.gcn_norm(dev[k]).to_numpy()
                if not (np.array_equal(rp, want[k].row_ptr) and
                        np.array_equal(ci, want[k].col_ind) and
                        np.array_equal(bits(v), bits(want[k].val))):
                    bad.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
