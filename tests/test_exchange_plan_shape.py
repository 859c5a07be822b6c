"""Shape of the exchange build's block tasks, on the host: the LDS of a
workgroup follows the row nodes of block terms alone (a column node's or a
direct block's functions take none), and nodes of more than 352 functions are
cut into splits that pass the plan's own checks."""
import numpy as np
import pytest


def _built(kind, n):
    import h2eri
    from h2eri import molecules as M
    rng = M.rng_for(700 + n)
    atoms = M.alkane(n, rng) if kind == "alkane" else M.water_cluster(n, rng)
    h = h2eri.H2ERI(1e-10, 1e-10, 1e-6)
    return h.build_from_mol(text=M.mol_text(atoms))


def _row_functions(h):
    """Basis functions of the row node of every term that is not a dense
    near-field block."""
    t, s = h.tree(), h.s
    sbf, sp, nl = t["shell_bf_sidx"], t["sp_shell_idx"].reshape(2, -1), t["n_leaf_node"]

    def functions(node):
        p0, p1 = t["pt_cluster"][node]
        return sum(int(sbf[k + 1] - sbf[k]) for k in np.unique(sp[:, p0:p1 + 1]))

    leaves = t["height_nodes"][0, :nl]
    near = [(a, s.c_D_blks[i]) for i, a in enumerate(list(leaves) + [p[0] for p in t["r_inadm_pairs"]])]
    far = [(p[0], s.c_B_blks[i]) for i, p in enumerate(t["r_adm_pairs"])]
    rows = [a for a, b in near if b and b.contents.ld < 0] + [a for a, b in far if b and b.contents.nrow > 0]
    return [functions(a) for a in set(rows)]


@pytest.mark.parametrize("kind,n,splits", [("water", 1, 1), ("water", 3, 1), ("alkane", 12, 1), ("alkane", 40, 2)])
def test_block_tasks_follow_the_row_nodes(kind, n, splits):
    h = _built(kind, n)
    r = h.exchange_plan_shape()
    nf = _row_functions(h) or [1]
    assert r["functions"] == max(nf) and r["splits"] == splits and r["wide"] == 0
    per_split = max(-(-n // -(-n // 352)) for n in nf)
    assert r["lds_bytes"] == 16 * 258 * 8 + (per_split + 1) * 16 * 8 + 4 * max(nf)
