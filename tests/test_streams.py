"""Calls on an explicit stream that is not torch's current one: what they
return is finished, its size included.

Without a GPU the native calls are stood in for by ones whose work happens
when the stream is waited for, so a size read too early is a wrong size every
time; with one, the same calls run behind a long queue on the stream."""
import numpy as np
import pytest

from helpers import bits, random_csr


class _Stream:
    """A stream whose queued work runs when it is waited for."""

    def __init__(self, handle):
        self.cuda_stream, self.queue, self.waits = handle, [], 0

    def synchronize(self):
        self.waits += 1
        while self.queue:
            self.queue.pop(0)()


class _Lib:
    """Native calls of one piece of work, queued, or (`now`) done by the time
    that the caller reads a result."""

    def __init__(self, stream, work, now):
        self.stream, self.work, self.now = stream, work, now

    def check(self, status):
        assert status == 0

    def __getattr__(self, name):
        def call(*args):
            assert args[-1] == self.stream.cuda_stream
            if self.now:
                self.work(args)
            else:
                self.stream.queue.append(lambda: self.work(args))
            return 0
        return call


CALLS = ["add_self_loops", "gcn_norm", "edge_list_to_csr", "sage_forward", "gat_aggregate"]


@pytest.mark.parametrize("name", CALLS)
@pytest.mark.parametrize("current", [False, True])
def test_other_stream_is_waited_for(monkeypatch, name, current):
    import torch
    import tinygnn_amd as tg
    stream = _Stream(77)
    monkeypatch.setattr(tg, "dptr", lambda t, dtype=None: t)
    monkeypatch.setattr(torch.cuda, "current_stream",
                        lambda *a: stream if current else _Stream(0))
    n, nnz = 4, 3
    a = tg.DeviceCSR(n, n, torch.tensor([0, 1, 2, 3, 3], dtype=torch.int32),
                     torch.tensor([1, 2, 3], dtype=torch.int32), torch.ones(nnz))

    def work(args):
        if name in ("add_self_loops", "gcn_norm"):
            args[5].copy_(torch.tensor([0, 2, 4, 6, 7], dtype=torch.int32))  # row_ptr_out

    real_empty = torch.empty
    monkeypatch.setattr(torch, "empty", lambda *s, **k: real_empty(*s, **k).zero_())
    # (reading a size waits for the current stream by itself)
    monkeypatch.setattr(tg, "lib", _Lib(stream, work, now=current))
    x, w = torch.ones(n, 2), torch.ones(2, 2)
    plan = type("Plan", (), {"h": None})()
    out = {"add_self_loops": lambda: tg.add_self_loops(a, stream=stream),
           "gcn_norm": lambda: tg.gcn_norm(a, stream=stream),
           "edge_list_to_csr": lambda: tg.edge_list_to_csr(a.col_ind, a.col_ind, n, stream=stream),
           "sage_forward": lambda: tg.sage_forward(plan, a, x, w, w, stream=stream),
           "gat_aggregate": lambda: tg.gat_aggregate(plan, a, x, 1, 2, x[:, :1], x[:, :1],
                                                     stream=stream)}[name]()
    assert stream.waits == (0 if current else 1)
    if name in ("add_self_loops", "gcn_norm"):
        assert out.nnz == 7 and out.val.numel() == 7


@pytest.mark.gpu
def test_results_of_another_stream(gpu, restate):
    """The same calls behind some milliseconds of work on a stream of their own,
    read on the current stream at once."""
    import tinygnn_amd as tg
    torch = gpu
    rng = np.random.default_rng(41)
    a = random_csr(rng, 3000, 3000, avg_deg=8, max_deg=2500)
    a.val[:] = np.abs(a.val) + 0.01
    d = tg.DeviceCSR.from_numpy(a.n_rows, a.n_cols, a.row_ptr, a.col_ind, a.val)
    src = np.repeat(np.arange(3000), np.diff(a.row_ptr)).astype(np.int32)
    dsrc, ddst = torch.from_numpy(src).cuda(), torch.from_numpy(a.col_ind).cuda()
    big = torch.randn(4096, 4096, device="cuda")
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    for fn, want in ((tg.add_self_loops, restate.add_self_loops(a)),
                     (tg.gcn_norm, restate.gcn_norm(a)),
                     (lambda _, stream: tg.edge_list_to_csr(dsrc, ddst, 3000, stream=stream),
                      restate.edge_list_to_csr(src, a.col_ind, 3000))):
        with torch.cuda.stream(side):
            for _ in range(10):
                torch.mm(big, big)
        rp, ci, v = fn(d, stream=side).to_numpy()
        np.testing.assert_array_equal(rp, want.row_ptr)
        np.testing.assert_array_equal(ci, want.col_ind)
        np.testing.assert_array_equal(bits(v), bits(want.val))
