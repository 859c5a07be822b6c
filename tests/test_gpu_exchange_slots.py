"""The column slots of the exchange build: shells of one function only (all
singles, an odd one left over), entry lists of less than four, of exactly the
32 entries kept in registers and of more, and lists cut into several slots of
one function.  K equals the oracle's to 1e-12 (sums of up to 1e5 FP64 terms
per element, in another order: 1e-13 at most)."""
import numpy as np
import pytest

import oracle_bind
from conftest import relerr

pytestmark = pytest.mark.gpu


def _chain(n):
    return [("H", np.array([0.0, 0.0, 0.8 * k + 0.05 * (k % 3)])) for k in range(n)]


@pytest.mark.parametrize("name,n", [("chain", 3), ("chain", 17), ("chain", 48), ("water", 3), ("water", 9), ("alkane", 7)])
def test_exchange_slots(name, n, tmp_path):
    import h2eri
    from h2eri import molecules as M
    rng = M.rng_for(90 + n)
    atoms = _chain(n) if name == "chain" else (M.water_cluster(n, rng) if name == "water" else M.alkane(n, rng))
    D = M.density(atoms, max(1, n // 2) if name == "chain" else 4 * n, M.rng_for(91))
    h = h2eri.H2ERI(1e-10, 1e-10, 1e-6)
    h.build_from_mol(text=M.mol_text(atoms))
    p = str(tmp_path / "m.rep")
    h.save(p)
    print(f"exchange {name} {n}: {h.nbf} functions, N={h.n}", flush=True)
    assert relerr(h.build_exchange(D), oracle_bind.Oracle(p).exchange(D)) < 1e-12
