"""The device memory of calls that are given no workspace (csrc/common.hpp,
TempBuffer): reuse, its bound, and streams under capture."""
import os
import subprocess

import numpy as np
import pytest

from helpers import bits, random_csr


def test_kept_blocks_on_the_host():
    """tests/cpp/test_temporaries.cpp: the library's allocations over a stand-in
    for the runtime's memory and event calls."""
    from tinygnn_amd import build
    if not os.path.exists(build.TEMPORARIES_TEST):
        pytest.skip("test_temporaries not built")
    r = subprocess.run([build.TEMPORARIES_TEST], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr


@pytest.mark.gpu
def test_trim(gpu):
    """What a call's temporaries leave behind goes back to the driver."""
    import tinygnn_amd as tg
    torch = gpu
    n = 100_000
    d = tg.DeviceCSR(n, n, torch.arange(n + 1, dtype=torch.int32, device="cuda"),
                     torch.arange(n, dtype=torch.int32, device="cuda"),
                     torch.ones(n, device="cuda"))
    plan = tg.SpmmPlan(d.row_ptr, n, n, 256)
    x, w = torch.ones(n, 256, device="cuda"), torch.ones(256, 64, device="cuda")
    out = tg.sage_forward(plan, d, x, w, w, dataflow=tg.SAGE_CONCAT)  # 100 MB of its own
    torch.cuda.synchronize()
    kept = torch.cuda.mem_get_info()[0]
    tg.trim()
    assert torch.cuda.mem_get_info()[0] - kept >= 4 * n * 256
    assert float(out[0, 0]) == 512.0


@pytest.mark.gpu
def test_capture_needs_a_workspace(gpu, restate):
    """Under capture, in a mode that would let hipMalloc through, a call that
    would allocate is refused and the capture goes on; with a workspace it is
    captured and replays."""
    import tinygnn_amd as tg
    torch = gpu
    a = random_csr(np.random.default_rng(7), 2000, 2000, avg_deg=6, max_deg=1500)
    a.val[:] = np.abs(a.val) + 0.01
    d = tg.DeviceCSR.from_numpy(2000, 2000, a.row_ptr, a.col_ind, a.val)
    plan = tg.SpmmPlan(d.row_ptr, 2000, d.nnz, 64)
    x, w = torch.randn(2000, 64, device="cuda"), torch.randn(64, 64, device="cuda")
    s = torch.randn(2000, 1, device="cuda")
    cap = d.nnz + 2000
    rp = torch.empty(2001, dtype=torch.int32, device="cuda")
    ci = torch.empty(cap, dtype=torch.int32, device="cuda")
    v = torch.empty(cap, device="cuda")
    n_ws = tg.lib.tg_self_loops_workspace_size(2000)
    ws = torch.empty(n_ws, dtype=torch.uint8, device="cuda")
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side, capture_error_mode="relaxed"):
        for call in (lambda: tg.gcn_norm(d), lambda: tg.add_self_loops(d),
                     lambda: tg.sage_forward(plan, d, x, w, w, dataflow=tg.SAGE_CONCAT),
                     # averaged heads need room for every head
                     lambda: tg.gat_aggregate(plan, d, x, 4, 16, s.expand(-1, 4).contiguous(),
                                              s.expand(-1, 4).contiguous(), concat=False),
                     lambda: tg.edge_list_to_csr(d.col_ind, d.col_ind, 2000)):
            with pytest.raises(tg.InvalidArgument, match="workspace"):
                call()
        tg.lib.check(tg.lib.tg_gcn_norm(2000, d.nnz, d.row_ptr.data_ptr(), d.col_ind.data_ptr(),
                                        d.val.data_ptr(), rp.data_ptr(), ci.data_ptr(),
                                        v.data_ptr(), None, None, ws.data_ptr(), n_ws,
                                        tg.stream_handle()))
    want = restate.gcn_norm(a)
    for _ in range(3):
        for t in (rp, ci, v):
            t.zero_()
        g.replay()
        torch.cuda.synchronize()
        nnz = int(rp[-1])
        np.testing.assert_array_equal(rp.cpu().numpy(), want.row_ptr)
        np.testing.assert_array_equal(ci[:nnz].cpu().numpy(), want.col_ind)
        np.testing.assert_array_equal(bits(v[:nnz].cpu().numpy()), bits(want.val))
