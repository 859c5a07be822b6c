"""Batches whose padded pass finds no room on the device (a bound on a plan's
device memory stands for a full device): the vectors run in narrower passes,
bitwise the same as those passes alone, and a graph captured before stays."""
import numpy as np
import pytest

from conftest import make_synthetic

pytestmark = pytest.mark.gpu


def _bound(h):
    """Bytes that the plan of 8 vectors fits and the one of 16 does not: the
    workspace of 16 vectors alone."""
    w16, w8 = h.plan_stats(64, 16), h.plan_stats(64, 8)
    bound = 8 * 16 * w16["nW"]
    assert 8 * 8 * w8["nW"] + 64 * (w8["tiles"] + w8["reduces"]) < 0.8 * bound
    return bound


def _batch(h, n, seed=5):
    import torch
    return torch.from_numpy(np.random.default_rng(seed).standard_normal((n, h.n))).to("cuda:0")


def _run(h, X):
    import torch
    Y = torch.full_like(X, np.nan)
    h.matvec_multi_dev(len(X), X.data_ptr(), Y.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return Y


@pytest.mark.parametrize("executor", [0, 1])
def test_no_room_keeps_the_graph(executor, tmp_path):
    import torch
    h = make_synthetic(tmp_path / "s.rep", 900, 72, leaf=30, max_rank=12, lr_frac=0.4, diag_lr_frac=0.3)
    h.set_executor(executor)
    X = _batch(h, 9)
    y = torch.full_like(X[0], np.nan)
    torch.cuda.synchronize()
    h.graph_capture("matvec", 1, X.data_ptr(), y.data_ptr())
    h.set_pass_memory(_bound(h))
    Y = _run(h, X)
    assert torch.equal(Y[:8], _run(h, X[:8].contiguous()))
    assert torch.equal(Y[8:], _run(h, X[8:].contiguous()))
    h.graph_replay(torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(y, _run(h, X[:1].contiguous())[0])


@pytest.mark.parametrize("freed", ["precision", "tiles"])
def test_padding_returns_with_room(freed, tmp_path):
    import torch
    h = make_synthetic(tmp_path / "s.rep", 900, 72, leaf=30, max_rank=12, lr_frac=0.4, diag_lr_frac=0.3)
    X = _batch(h, 9)
    padded = _run(h, X)   # 16 wide: matrix instructions, other roundings than the narrower passes
    narrow = torch.cat([_run(h, X[:8].contiguous()), _run(h, X[8:].contiguous())])
    assert not torch.equal(padded, narrow)
    h.set_tile_bytes(65536)
    h.set_tile_bytes(131072)   # the plans go
    h.set_pass_memory(_bound(h))
    assert torch.equal(_run(h, X), narrow)
    h.set_pass_memory(0)
    if freed == "tiles":
        h.set_tile_bytes(65536)
        h.set_tile_bytes(131072)
    else:
        h.set_precision(32)
        h.set_precision(64)
    assert torch.equal(_run(h, X), padded)
