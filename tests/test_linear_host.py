"""ELinear's workspaces on the host (no GPU): the library call is recorded instead of made."""
import pytest
import torch

from eva_amd import _lib, ops
from eva_amd.linear import GEMV_MAX_ROWS, ELinear


def _recorded(monkeypatch, n_in, n_out, bits=4):
    calls = []

    def call(x, trellis, suh, svh, k, out=None, workspace=None):
        need = _lib.lib().evamx_exl3_linear_workspace_bytes(x.shape[0], n_in, n_out)
        ws = torch.empty(need, dtype=torch.uint8) if workspace is None else workspace     # as ops.exl3_linear
        assert ws.numel() >= need > 0
        calls.append((x.shape[0], ws))                   # held, so that no later one can take its address

    monkeypatch.setattr(ops, "exl3_linear", call)
    lin = ELinear(torch.zeros(n_in // 16, n_out // 16, 16 * bits, dtype=torch.int16), torch.ones(n_in, dtype=torch.float16),
                  torch.ones(n_out, dtype=torch.float16), strict=False)
    return lin, calls


@pytest.mark.parametrize("n_in,n_out", [(128, 128), (2048, 7168), (7168, 2048)])
@pytest.mark.parametrize("first", [1, 13])
def test_decode_workspace_outlives_larger_calls(monkeypatch, n_in, n_out, first):
    """A captured call of up to 16 rows keeps its workspace's address for every replay: the module goes
    on owning that buffer, and gives it to no larger call, whatever is called in between."""
    lin, calls = _recorded(monkeypatch, n_in, n_out)
    for rows in (first, 17, 200, 2, 512, GEMV_MAX_ROWS, 1024, first):
        lin.forward(torch.zeros(rows, n_in, dtype=torch.float16))
    decode = [ws for rows, ws in calls if rows <= GEMV_MAX_ROWS]
    assert len({ws.data_ptr() for ws in decode}) == 1
    lo, hi = decode[0].data_ptr(), decode[0].data_ptr() + decode[0].numel()
    assert all(ws.data_ptr() >= hi or ws.data_ptr() + ws.numel() <= lo for rows, ws in calls if rows > GEMV_MAX_ROWS)
    assert any(v is decode[0] for v in vars(lin).values())


def test_larger_calls_keep_no_workspace(monkeypatch):
    """A module holds its decode buffer alone, whatever it has been called with: a larger call's workspace
    is the allocator's again when the call returns (a capture's pool keeps it as long as the graph)."""
    lin, calls = _recorded(monkeypatch, 1024, 1024)
    for rows in (1, 4096, 200):
        lin.forward(torch.zeros(rows, 1024, dtype=torch.float16))
    held = {v.data_ptr() for v in vars(lin).values() if isinstance(v, torch.Tensor)}
    assert not any(ws.data_ptr() in held for rows, ws in calls if rows > GEMV_MAX_ROWS)


@pytest.mark.parametrize("n_in,n_out", [(7168, 18432), (4096, 14336), (7168, 12288), (18432, 12288)])
@pytest.mark.parametrize("rows", [17, 64])
def test_few_rows_of_a_wide_output_are_split(n_in, n_out, rows):
    """A call of one 64-row tile keeps the partials of eight k-ranges however many column groups it has:
    it does not go to the 256-row workgroups, which would be all but empty."""
    assert _lib.lib().evamx_exl3_linear_workspace_bytes(rows, n_in, n_out) >= 8 * rows * n_out * 4
