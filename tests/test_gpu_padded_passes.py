"""Batches that are not a power of two run their last vectors in a wider pass
whose spare vectors are zero.  Every vector equals its single-vector product
(1e-13: the widths sum in different orders, as the other batch tests allow),
with both executors, dense and low-rank blocks and both storage precisions;
nothing is written beyond the batch's last vector, and the input ends with
it.  Coulomb builds of as many densities equal the single builds alike."""
import numpy as np
import pytest

from conftest import make_synthetic, relerr

pytestmark = pytest.mark.gpu

COUNTS = [3, 5, 7, 9, 15, 17, 19]


@pytest.fixture(scope="module")
def tree(tmp_path_factory):
    return make_synthetic(tmp_path_factory.mktemp("pad") / "s.rep", 700, 21, lr_frac=0.5, diag_lr_frac=0.3)


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("executor", [0, 1])
@pytest.mark.parametrize("nvec", COUNTS)
def test_padded_matvec(tree, nvec, executor, bits):
    import torch
    h = tree
    h.set_precision(bits)
    h.set_executor(executor)
    X = np.random.default_rng(nvec).standard_normal((nvec, h.n))
    Xd = torch.from_numpy(X).to("cuda:0")
    Yd = torch.full((nvec + 16, h.n), 7.25, dtype=torch.float64, device="cuda:0")
    torch.cuda.synchronize()
    print(f"padded passes: {nvec} vectors, executor {executor}, {bits} bits", flush=True)
    h.matvec_multi_dev(nvec, Xd.data_ptr(), Yd.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    h.device_status()
    Y = Yd.cpu().numpy()
    assert np.all(Y[nvec:] == 7.25)
    for k in range(nvec):
        assert relerr(Y[k], h.matvec(X[k])) < 1e-13


@pytest.mark.parametrize("ndens", [1, 3, 5, 9, 17])
def test_coulomb_counts(ndens):
    import h2eri
    from h2eri import molecules as M
    rng = M.rng_for(300)
    atoms = M.water_cluster(3, rng)
    h = h2eri.H2ERI(1e-10, 1e-10, 1e-6).build_from_mol(text=M.mol_text(atoms))
    Ds = np.stack([M.density(atoms, 15, rng) for _ in range(ndens)])
    Js = h.build_coulomb_multi(Ds)
    for k in range(ndens):
        assert np.array_equal(Js[k], Js[k].T)
        assert relerr(Js[k], h.build_coulomb(Ds[k])) < 1e-13
