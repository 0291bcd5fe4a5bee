"""The drop-in runners (eva_amd.coop, eva_amd.linear) on the GPU: results against the oracle,
and the reference's ownership rules (runtime/ds41/moe_coop3072.py:261-402)."""
import threading

import numpy as np
import pytest
import torch

from oracle import coop, synth
from tests.gpu_helpers import DeviceExperts, rel_err_rows, to_dev

pytestmark = pytest.mark.gpu
TOL = 1e-2
H, I, E = 256, 128, 12


@pytest.fixture(scope="module")
def case(dev):
    rng = np.random.default_rng(61)
    ex = [synth.expert(rng, H, I, 3, 1 / np.sqrt(H)) for _ in range(E)]
    return ex, DeviceExperts(ex, dev)


def _routes(rng, rows, topk):
    sel = np.stack([rng.choice(E, size=topk, replace=False) for _ in range(rows)]).astype(np.int64)
    w = rng.uniform(0.05, 1.0, size=(rows, topk)).astype(np.float32)
    return sel, w


def test_coop_runner_borrowed_output(dev, case):
    from eva_amd.coop import CoopRunner
    ex, de = case
    rng = np.random.default_rng(62)
    r = CoopRunner(dev, topk=4, hidden=H, inter=I, rows=2)
    x = rng.standard_normal((2, H)).astype(np.float16)
    sel, w = _routes(rng, 2, 4)
    rows = [de.table[i] for i in range(9)]                     # nine row views of one table
    y1 = r.run(to_dev(x, dev), to_dev(sel, dev).to(torch.int32), to_dev(w, dev), rows, 3, 10.0)
    torch.cuda.synchronize()
    ref = coop.moe_routed(x, sel, w.astype(np.float16), ex, 10.0)
    assert rel_err_rows(y1.cpu().numpy(), ref) < TOL
    y2 = r.run(to_dev(x, dev), to_dev(sel, dev), to_dev(w, dev), de.table, 3, 10.0)
    assert y2 is y1                                            # borrowed, overwritten by the next call


def test_capacity_runner_run_prepare_table(dev, case):
    from eva_amd.coop import CoopRunner3072
    ex, de = case
    rng = np.random.default_rng(63)
    r = CoopRunner3072(dev, topk=6, hidden=H, inter=I, max_rows=20)
    for rows in (20, 7):
        x = rng.standard_normal((rows, H)).astype(np.float16)
        sel, w = _routes(rng, rows, 6)
        w[1, 2] = 0.0
        y = r.run(to_dev(x, dev), to_dev(sel, dev), to_dev(w, dev), de.table, 3, 10.0)
        rw16 = w.astype(np.float16)
        assert y.shape == (rows, H) and y.data_ptr() != r.out.data_ptr()   # owned copy (moe_coop3072.py:312)
        assert rel_err_rows(y.cpu().numpy(), coop.moe_routed(x, sel, rw16, ex, 10.0)) < TOL
        assert np.array_equal(r.run_table().cpu().numpy(), coop.reference_table(sel, rw16, capacity=20))
        t = r.prepare_routes(to_dev(sel, dev), to_dev(w, dev), E)
        assert np.array_equal(t.cpu().numpy(), coop.reference_table(sel, rw16, capacity=20))
        assert np.array_equal(r.run_table().cpu().numpy(), t.cpu().numpy())
    life = r.lifecycle()
    assert not life["failed"] and not life["closed"] and life["owner_thread_matches"]
    r.close()
    assert r.lifecycle()["closed"]
    with pytest.raises(RuntimeError):
        r.run(to_dev(x, dev), to_dev(sel, dev), to_dev(w, dev), de.table, 3, 10.0)


def test_capacity_runner_bounds_poison_and_owner(dev, case):
    from eva_amd.coop import CoopRunner512
    _, de = case
    rng = np.random.default_rng(64)
    r = CoopRunner512(dev, topk=2, hidden=H, inter=I)
    x = to_dev(rng.standard_normal((2, H)).astype(np.float16), dev)
    w = to_dev(np.full((2, 2), 0.5, np.float32), dev)
    good = to_dev(np.array([[0, 1], [2, 3]], np.int64), dev)
    errors = []
    th = threading.Thread(target=lambda: errors.append(pytest.raises(RuntimeError, r.run, x, good, w, de.table, 3, 1.0)))
    th.start()
    th.join()
    assert errors                                              # wrong thread refused
    with pytest.raises(ValueError):
        r.run(x, good, w, de.table, 6, 1.0)                    # unsupported rate: argument error
    y1 = r.run(x, good, w, de.table, 3, 1.0)
    assert y1.data_ptr() == r.out.data_ptr() and y1.shape == (2, H)   # borrowed rows (moe_coop512.py:248)
    bad = to_dev(np.array([[0, 1], [2, 99]], np.int64), dev)   # 99 is outside the 12-entry table
    with pytest.raises(RuntimeError, match="outside"):
        r.run(x, bad, w, de.table, 3, 1.0)
    assert r.lifecycle()["failed"]
    with pytest.raises(RuntimeError):
        r.run(x, good, w, de.table, 3, 1.0)                    # poisoned


def test_elinear_batch_invariant(dev):
    """Up to 16 rows (decode GEMV) each row alone gives the same bits as in a 16-row call; beyond
    (MFMA path) a row gives the same bits in calls of 17, 37 and 101 rows. Both within TOL of the
    oracle."""
    from eva_amd.linear import build_linear
    rng = np.random.default_rng(65)
    tr, suh, svh = synth.projection(rng, 512, 384, 4, svh_scale=1 / np.sqrt(512))
    lin = build_linear(torch.from_numpy(suh), torch.from_numpy(svh), torch.from_numpy(tr), None, device=dev)
    x = rng.standard_normal((101, 512)).astype(np.float16)
    ref = coop.exl3_linear(x, tr, suh, svh, 4)
    y16 = lin.forward(to_dev(x[:16], dev)).cpu().numpy()
    assert rel_err_rows(y16.astype(np.float32), ref[:16].astype(np.float32)) < TOL
    for i in (0, 5, 15):                                       # each row alone gives the same bits
        yi = lin.forward(to_dev(x[i:i + 1], dev)).cpu().numpy()
        assert np.array_equal(yi[0].view(np.uint16), y16[i].view(np.uint16))
    y101 = lin.forward(to_dev(x, dev)).cpu().numpy()
    assert rel_err_rows(y101.astype(np.float32), ref.astype(np.float32)) < TOL
    y37 = lin.forward(to_dev(x[20:57], dev)).cpu().numpy()
    y17 = lin.forward(to_dev(x[84:], dev)).cpu().numpy()
    assert np.array_equal(y37.view(np.uint16), y101[20:57].view(np.uint16))
    assert np.array_equal(y17.view(np.uint16), y101[84:].view(np.uint16))


@pytest.mark.parametrize("shape,K,counts", [
    ((128, 128), 4, (17, 32, 33, 64, 65)),                     # one 128-chunk: one k-range
    ((384, 256), 2.5, (17, 63, 129, 2048)),                    # fewer chunks than k-ranges
    ((1152, 1024), 3, (33, 64, 192, 704, 1000, 6145)),         # uneven k-ranges; each kernel by size
    ((1152, 1024), 5, (49, 6399)),
    ((7168, 896), 1.5, (18, 300, 1920, 3600)),
])
def test_linear_row_kernels(dev, shape, K, counts):
    """Above 16 rows a call takes one of three kernels by its size. Every row of every call has the bits
    the row has in a 17-row call, at the edges of the 16-, 64- and 256-row tiles too; the 17-row calls are
    held to the oracle."""
    n_in, n_out = shape
    rng = np.random.default_rng(n_in + n_out)
    tr, suh, svh = synth.projection(rng, n_in, n_out, K, n_in ** -0.5)
    from eva_amd import ops
    from eva_amd.linear import build_linear
    lin = build_linear(to_dev(suh, dev), to_dev(svh, dev), to_dev(tr, dev), device=dev, strict=False)
    x = rng.standard_normal((max(counts), n_in)).astype(np.float16)
    xd = to_dev(x, dev)
    y17 = lin.forward(xd[:17].contiguous()).cpu().numpy()
    ref = coop.exl3_linear(x[:17], tr, suh, svh, K)
    assert rel_err_rows(y17.astype(np.float32), ref.astype(np.float32)) < TOL
    for rows in counts:
        y = lin.forward(xd[:rows].contiguous())
        starts = sorted({0, max(0, rows - 17), max(0, rows // 2 - 8)} | {r for r in (56, 248) if r + 17 <= rows})
        for r in starts:
            want = lin.forward(xd[r:r + 17].contiguous())
            assert torch.equal(y[r:r + 17][:rows - r].view(torch.int16), want[:min(17, rows - r)].view(torch.int16)), (rows, r)
    # an output that starts off a 16-byte boundary
    rows = max(counts)
    buf = torch.zeros(rows * n_out + 1, dtype=torch.float16, device=dev)
    ops.exl3_linear(xd, lin.trellis, lin.suh, lin.svh, K, out=buf[1:].view(rows, n_out))
    assert torch.equal(buf[1:].view(rows, n_out).view(torch.int16), lin.forward(xd).view(torch.int16))


@pytest.mark.parametrize("shape,K", [((128, 128), 4), ((512, 256), 2), ((640, 1024), 3.5), ((5120, 5120), 5), ((1280, 40960), 1.5)])
def test_linear_decode_rows_bit_identical(dev, shape, K):
    """1 to 16 rows, one 128-chunk a split: one k-split quarter and many, workgroups of four and of eight
    waves. Every row has the bits of its one-row call; those are held to the oracle."""
    n_in, n_out = shape
    rng = np.random.default_rng(n_in + n_out)
    tr, suh, svh = synth.projection(rng, n_in, n_out, K, n_in ** -0.5)
    from eva_amd.linear import build_linear
    lin = build_linear(to_dev(suh, dev), to_dev(svh, dev), to_dev(tr, dev), device=dev)
    x = rng.standard_normal((16, n_in)).astype(np.float16)
    xd = to_dev(x, dev)
    one = torch.cat([lin.forward(xd[r:r + 1]) for r in range(16)])
    for rows in (2, 3, 4, 5, 7, 8, 9, 13, 16):
        assert torch.equal(lin.forward(xd[:rows]).view(torch.int16), one[:rows].view(torch.int16)), rows
    _check_columns(one[:2], x[:2], tr, suh, svh, K, [range(0, min(n_out, 5120) // 128)])


def _check_columns(y, x, tr, suh, svh, K, spans):
    """Some 128-column groups of y = linear(x) against the oracle: a group depends on its own tiles only."""
    for groups in spans:
        a, b = 128 * groups[0], 128 * (groups[-1] + 1)
        ref = coop.exl3_linear(x, np.ascontiguousarray(tr[:, a // 16:b // 16]), suh, svh[a:b], K)
        assert rel_err_rows(y[:, a:b].cpu().numpy().astype(np.float32), ref.astype(np.float32)) < TOL, a


@pytest.mark.parametrize("shape,K", [
    ((7168, 18432), 1.5),        # 56 chunks over 29 splits: one or two each
    ((18432, 7168), 3),          # 144 over 74
    ((1152, 524288), 1.5),       # nine chunks in one split: three windows of four, five of two
    ((512, 65536), 5),           # one chunk a split, one quarter
    ((128, 4194432), 1.5),       # more column groups than a grid's second dimension takes
])
def test_linear_decode_rows_wide(dev, shape, K):
    """1 to 16 rows where a split has several 128-chunks, evenly and unevenly, in one LDS window and in
    several, and at the largest column counts. Every row has the bits of its one-row call; some column
    groups of those are held to the oracle."""
    n_in, n_out = shape
    rng = np.random.default_rng(n_in + n_out)
    tr, suh, svh = synth.projection(rng, n_in, n_out, K, n_in ** -0.5)
    from eva_amd.linear import build_linear
    lin = build_linear(to_dev(suh, dev), to_dev(svh, dev), to_dev(tr, dev), device=dev)
    x = rng.standard_normal((16, n_in)).astype(np.float16)
    xd = to_dev(x, dev)
    one = torch.cat([lin.forward(xd[r:r + 1]) for r in range(16)])
    for rows in (2, 5, 9, 16):
        assert torch.equal(lin.forward(xd[:rows]).view(torch.int16), one[:rows].view(torch.int16)), rows
    n = n_out // 128
    _check_columns(one[:2], x[:2], tr, suh, svh, K, [range(g, g + 1) for g in sorted({0, 1, n // 2, n - 2, n - 1})])


@pytest.mark.parametrize("rows", [1, 13])
def test_elinear_graph_after_larger_calls(dev, rows):
    """A captured call of up to 16 rows keeps a workspace of its own: eager calls of more rows and fresh
    allocations between its replays change neither its results nor those allocations."""
    n_in, n_out, K = 1024, 2048, 4
    rng = np.random.default_rng(5 + rows)
    tr, suh, svh = synth.projection(rng, n_in, n_out, K, n_in ** -0.5)
    from eva_amd.linear import build_linear
    lin = build_linear(to_dev(suh, dev), to_dev(svh, dev), to_dev(tr, dev), device=dev, strict=False)
    x = to_dev(rng.standard_normal((1024, n_in)).astype(np.float16), dev)
    xs = x[:rows].clone()
    want = lin.forward(xs).clone()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = lin.forward(xs)
    held = []
    for more in (17, 200, 1024):
        big = lin.forward(x[:more]).clone()
        need = [lin._ws.numel()] + [1 << s for s in range(12, 25)]
        held += [torch.full((n,), 0x5A, dtype=torch.uint8, device=dev) for n in need]
        for _ in range(3):
            y.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y.view(torch.int16), want.view(torch.int16))
        assert all(bool((t == 0x5A).all()) for t in held)
        assert torch.equal(lin.forward(x[:more]).view(torch.int16), big.view(torch.int16))
