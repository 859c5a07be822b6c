"""K of several handles of a process: a large molecule's block tasks take more
LDS than a small one's, whose plan is uploaded after it and must not lower the
limit of the large one's launches."""
import pytest

import oracle_bind
from conftest import relerr

pytestmark = pytest.mark.gpu


def test_small_plan_after_a_large_one(tmp_path):
    import h2eri
    from h2eri import molecules as M
    out = []
    for k, atoms in enumerate([M.alkane(20, M.rng_for(720)), M.water_cluster(2, M.rng_for(702))]):
        h = h2eri.H2ERI(1e-10, 1e-10, 1e-6)
        h.build_from_mol(text=M.mol_text(atoms))
        p = str(tmp_path / f"{k}.rep")
        h.save(p)
        h.exchange_workbuf_init()
        out.append((h, p, M.density(atoms, 10, M.rng_for(98 + k))))
    assert out[0][0].exchange_plan_shape()["lds_bytes"] > 65536 > out[1][0].exchange_plan_shape()["lds_bytes"]
    for h, p, D in out + out[:1]:
        print(f"exchange of {h.nbf} functions", flush=True)
        assert relerr(h.build_exchange(D), oracle_bind.Oracle(p).exchange(D)) < 1e-12


def test_resident_bytes_of_a_plan():
    """The host's count of what a plan makes resident is what an upload
    allocates, task lists included, also after the plan was made again."""
    import h2eri
    from h2eri import molecules as M
    h = h2eri.H2ERI(1e-10, 1e-10, 1e-6)
    h.build_from_mol(text=M.mol_text(M.water_cluster(5, M.rng_for(705))))
    for bound in (2.0 ** 31, 65536, 2.0 ** 31):
        h.set_exchange_scratch(bound)
        assert h.exchange_stats()["resident_bytes"] == h.exchange_plan_check()["resident_bytes"]
