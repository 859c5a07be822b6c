"""A caller's own capture of a batch whose padded pass has no plan yet, and
whose narrower passes have theirs: nothing can be allocated under capture, so
the narrower passes are recorded, and each replay equals them bitwise."""
import numpy as np
import pytest

from conftest import make_synthetic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("executor", [0, 1])
def test_capture_of_three_after_one_and_two(executor, tmp_path):
    import torch
    h = make_synthetic(tmp_path / "s.rep", 700, 21, lr_frac=0.5, diag_lr_frac=0.3)
    h.set_executor(executor)
    X = torch.from_numpy(np.random.default_rng(3).standard_normal((3, h.n))).to("cuda:0")
    ref, Y = torch.full_like(X, np.nan), torch.full_like(X, np.nan)
    st = torch.cuda.Stream()
    torch.cuda.synchronize()
    h.upload()
    h.matvec_multi_dev(2, X.data_ptr(), ref.data_ptr(), st.cuda_stream)
    h.matvec_multi_dev(1, X[2:].data_ptr(), ref[2:].data_ptr(), st.cuda_stream)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=st, capture_error_mode="thread_local"):
        h.matvec_multi_dev(3, X.data_ptr(), Y.data_ptr(), st.cuda_stream)
    for _ in range(3):
        Y.fill_(np.nan)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(Y, ref)
