"""The exchange build's fused block kernel at the edges of its tiles: nodes of
fewer functions than a tile of 16, a single function, ranks below and between
multiples of 16, and (C40H82) nodes of more than 352 functions, whose K block
is cut into splits.  K equals the oracle's to 1e-12, the tolerance of the
other exchange tests (sums of up to 1e5 FP64 terms per element, in another
order: 1e-13 at most)."""
import numpy as np
import pytest

import oracle_bind
from conftest import relerr

pytestmark = pytest.mark.gpu


def _atoms(name):
    from h2eri import molecules as M
    rng = M.rng_for(88)
    if name == "h":
        return [("H", np.zeros(3))], 1
    if name == "h2":
        return [("H", np.zeros(3)), ("H", np.array([0.0, 0.0, 0.74]))], 1
    if name == "water":
        return M.water_cluster(1, rng), 5
    if name == "water5":
        return M.water_cluster(5, rng), 25
    if name == "methane":
        return M.alkane(1, rng), 5
    return M.alkane(40, rng), 161


@pytest.mark.parametrize("name", ["h", "h2", "water", "methane", "water5", "c40"])
def test_exchange_blocks(name, tmp_path):
    import h2eri
    from h2eri import molecules as M
    atoms, nocc = _atoms(name)
    D = M.density(atoms, min(nocc, len(M.bf_centers(atoms))), M.rng_for(89))
    h = h2eri.H2ERI(1e-10, 1e-10, 1e-6)
    h.build_from_mol(text=M.mol_text(atoms))
    p = str(tmp_path / f"{name}.rep")
    h.save(p)
    print(f"exchange {name}: {h.nbf} functions, N={h.n}", flush=True)
    K = h.build_exchange(D)
    assert relerr(K, oracle_bind.Oracle(p).exchange(D)) < 1e-12
    assert relerr(h.build_exchange(D), K) < 1e-14   # atomics: another order of the adds
