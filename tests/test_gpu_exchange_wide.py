"""The exchange build's block kernel with 64-bit operand offsets, which only
representations of many gigabytes take by themselves, forced on small ones: the
edges of its tiles, column slots and splits as for the 32-bit form (C40H82 has
nodes of more than 352 functions).  K equals the oracle's to 1e-12, the
tolerance of the other exchange tests, and the 32-bit form's to 1e-13 (the same
sums; only the order of the atomic adds differs)."""
import numpy as np
import pytest

import oracle_bind
from conftest import relerr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n", [("h2", 1), ("chain", 17), ("chain", 48), ("water", 1), ("water", 5), ("water", 9),
                                    ("alkane", 7), ("alkane", 40)])
def test_wide_offsets(kind, n, tmp_path):
    import h2eri
    from h2eri import molecules as M
    rng = M.rng_for(800 + n)
    if kind == "h2":
        atoms = [("H", np.zeros(3)), ("H", np.array([0.0, 0.0, 0.74]))]
    elif kind == "chain":
        atoms = [("H", np.array([0.0, 0.0, 0.8 * k + 0.05 * (k % 3)])) for k in range(n)]
    else:
        atoms = M.alkane(n, rng) if kind == "alkane" else M.water_cluster(n, rng)
    D = M.density(atoms, max(1, len(atoms) // 2), M.rng_for(801))
    h = h2eri.H2ERI(1e-10, 1e-10, 1e-6)
    h.build_from_mol(text=M.mol_text(atoms))
    p = str(tmp_path / "m.rep")
    h.save(p)
    h.set_exchange_wide(True)
    assert h.exchange_plan_shape()["wide"] == 1
    print(f"exchange, 64-bit offsets, {kind} {n}: {h.nbf} functions", flush=True)
    K = h.build_exchange(D)
    assert relerr(K, oracle_bind.Oracle(p).exchange(D)) < 1e-12
    h.set_exchange_wide(False)
    assert h.exchange_plan_shape()["wide"] == 0
    assert relerr(K, h.build_exchange(D)) < 1e-13
