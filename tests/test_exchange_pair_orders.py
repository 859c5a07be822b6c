"""Exchange of a representation that holds shell pairs in both orders, and
twice in one order, as a file may (every row then counts): the plan keeps each
entry of every function, and K equals the oracle's, which sums over all rows,
to 1e-12 (the tolerance of the other exchange tests)."""
import numpy as np
import pytest

import oracle_bind
from conftest import relerr


def _with_repeated_pairs(path, twice):
    """C10H22 with, in every leaf, one shell pair replaced by another one of
    its leaf with as many functions: in the reverse order, or the same."""
    import h2eri
    from h2eri import molecules as M
    atoms = M.alkane(10, M.rng_for(95))
    h = h2eri.H2ERI(1e-10, 1e-10, 1e-6)
    h.build_from_mol(text=M.mol_text(atoms))
    s, t = h.s, h.tree()
    nb = np.diff(t["shell_bf_sidx"])
    npair, changed = s.num_sp, 0
    for leaf in t["height_nodes"][0, :t["height_n_node"][0]]:
        p0, p1 = t["pt_cluster"][leaf]
        seen = {}
        for i in range(p0, p1 + 1):
            a, b = s.sp_shell_idx[i], s.sp_shell_idx[i + npair]
            if a == b:
                continue
            size = nb[a] * nb[b]
            if size in seen and size > 1:
                c, d = seen[size]
                s.sp_shell_idx[i], s.sp_shell_idx[i + npair] = (c, d) if twice else (d, c)
                changed += 1
                break
            seen[size] = (a, b)
    assert changed > 4
    h.save(path)
    return h2eri.H2ERI.load(path), atoms


@pytest.mark.parametrize("twice", [False, True])
def test_plan_keeps_every_entry(twice, tmp_path):
    h, _ = _with_repeated_pairs(str(tmp_path / "r.rep"), twice)
    assert h.exchange_plan_check()["terms"] > 0


@pytest.mark.gpu
@pytest.mark.parametrize("twice", [False, True])
def test_exchange_sums_every_row(twice, tmp_path):
    from h2eri import molecules as M
    p = str(tmp_path / "r.rep")
    h, atoms = _with_repeated_pairs(p, twice)
    D = M.density(atoms, 41, M.rng_for(96))
    print(f"exchange with repeated pairs: {h.nbf} functions, twice {twice}", flush=True)
    assert relerr(h.build_exchange(D), oracle_bind.Oracle(p).exchange(D)) < 1e-12


@pytest.mark.gpu
@pytest.mark.parametrize("twice", [False, True])
def test_coulomb_sums_every_row(twice, tmp_path):
    from h2eri import molecules as M
    p = str(tmp_path / "r.rep")
    h, atoms = _with_repeated_pairs(p, twice)
    o = oracle_bind.Oracle(p)
    o.lib.orc_set_threads(1)   # its threads add rows of one element of J without a lock
    Ds = np.stack([M.density(atoms, 41, M.rng_for(97 + k)) for k in range(5)])
    Js = h.build_coulomb_multi(Ds)
    ref = [o.coulomb(D) for D in Ds]
    o.lib.orc_set_threads(0)
    for J, R in zip(Js, ref):
        assert relerr(J, R) < 1e-12
