"""The on-the-fly matvec's Hermite potential kernels at the edges of their
tasks: sides with fewer centres than a wave has lanes (each centre then takes
several lanes), with a remainder beyond whole waves, without any centre of the
higher orders, and molecules far enough apart that every Boys argument of a
pair of fragments lies above the table (T > 40, up to some thousands).  The
GPU product equals the oracle's on the same molecule with B and D stored
dense to <= 1e-13: about 1e4 additions of FP64 terms per row leave 1e-14, as
the host emulation of the same sums does.
"""
import numpy as np
import pytest

import oracle_bind
from conftest import relerr


def _atoms(name):
    from h2eri import molecules as M
    rng = M.rng_for(77)
    if name == "h":
        return [("H", np.zeros(3))]
    if name == "h2":
        return [("H", np.zeros(3)), ("H", np.array([0.0, 0.0, 0.74]))]
    if name == "water":
        return M.water_cluster(1, rng)
    if name == "ethane":
        return M.alkane(2, rng)
    far = M.water_cluster(2, rng)   # two waters 40 angstrom apart and one 400 away
    third = M.water_cluster(1, rng)
    return ([(s, r) for s, r in far[:3]] + [(s, r + np.array([40.0, 3.0, 1.0])) for s, r in far[3:]] +
            [(s, r + np.array([-5.0, 400.0, 2.0])) for s, r in third])


NAMES = ["h", "h2", "water", "ethane", "far"]


def _pair(name, tmp_path):
    import h2eri
    from h2eri import molecules as M
    txt = M.mol_text(_atoms(name))
    hd = h2eri.H2ERI(1e-10, 1e-10, 1e-6)
    hd.set_block_compression(0)
    hd.build_from_mol(text=txt)
    p = str(tmp_path / f"{name}.rep")
    hd.save(p)
    hj = h2eri.H2ERI(1e-10, 1e-10, 1e-6)
    hj.read_mol_text(txt).process_shells().partition().build_h2(1)
    return hj, oracle_bind.Oracle(p)


@pytest.mark.parametrize("name", NAMES)
def test_emulation_equals_dense_oracle(name, tmp_path):
    hj, o = _pair(name, tmp_path)
    x = np.random.default_rng(51).standard_normal(hj.n)
    assert relerr(hj.jit_emulate(x), o.matvec(x)) < 1e-13


@pytest.mark.gpu
@pytest.mark.parametrize("name", NAMES)
def test_matvec_equals_dense_oracle(name, tmp_path):
    hj, o = _pair(name, tmp_path)
    x = np.random.default_rng(52).standard_normal(hj.n)
    print(f"on-the-fly matvec {name} N={hj.n}", flush=True)
    y = hj.matvec(x)
    assert relerr(y, o.matvec(x)) < 1e-13
    assert np.array_equal(hj.matvec(x), y)
