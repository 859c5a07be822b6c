"""Five vectors: one padded pass of eight, or 4 + 1 where the staged executor
works on small blocks.  Either way they are bitwise what those passes give."""
import numpy as np
import pytest

from conftest import relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size,executor,bits,split", [(8, 0, 64, True), (8, 0, 32, True), (8, 1, 64, False),
                                                      (4, 0, 64, False)])
def test_passes_of_five(size, executor, bits, split):
    import h2eri
    import torch
    from h2eri import molecules as M
    h = h2eri.H2ERI(1e-10, 1e-10, 1e-6)
    h.build_from_mol(text=M.mol_text(M.water_cluster(size, M.rng_for(1000 + size))))
    h.set_precision(bits)
    h.set_executor(executor)
    X = torch.zeros((8, h.n), dtype=torch.float64, device="cuda:0")
    X[:5] = torch.from_numpy(np.random.default_rng(size).standard_normal((5, h.n))).to("cuda:0")

    def run(Z):
        Y = torch.full_like(Z, np.nan)
        h.matvec_multi_dev(len(Z), Z.data_ptr(), Y.data_ptr(), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        return Y

    torch.cuda.synchronize()
    Y = run(X[:5].contiguous())
    four_one = torch.cat([run(X[:4].contiguous()), run(X[4:5].contiguous())])
    eight = run(X)[:5]
    assert not torch.equal(four_one, eight)   # other summation orders
    assert torch.equal(Y, four_one if split else eight)
    assert relerr(Y.cpu().numpy(), eight.cpu().numpy()) < 1e-13
