"""The work a user of this library has it do, as cases of one pass each.

Every case is one call (or one graph replay) of a public entry point on a
seeded cc-pVDZ molecule, as an SCF program makes it in each iteration: the
representation is built and uploaded once per molecule and kept, the density
is new.  Four kinds, by "call":

* "coulomb": J matrices of `ndens` densities.  "via": "host" (host arrays in
  and out, the drop-in call), "device" (device pointers on the current stream)
  or "graph" (a captured HIP graph on fixed buffers, the densities of this
  iteration copied into them first);
* "exchange": one K matrix, device pointers;
* "on_the_fly": one J matrix with the B and D blocks evaluated from the shell
  pairs in the call (nothing but U stored), device pointers;
* "group": one matvec of every molecule of a set of alkanes in one call.

"bits" is the storage precision of U and B, "executor" 0 the staged launches,
1 the persistent one.  Geometries depend on the molecule alone (as in one SCF
calculation), densities on the seed: the damped densities of
h2eri.molecules, made on the GPU.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "h2p-eri_amd"))

import h2eri  # noqa: E402
from h2eri import molecules as M  # noqa: E402

DEV = "cuda:0"
ENTRY_BYTES = 8


def _coulomb(name, kind, n, reltol=1e-6, ndens=1, bits=64, via="device", executor=0):
    return dict(name=name, call="coulomb", molecule=kind, n=n, reltol=reltol, ndens=ndens, bits=bits, via=via,
                executor=executor)


def _exchange(name, kind, n, reltol=1e-6, bits=64):
    return dict(name=name, call="exchange", molecule=kind, n=n, reltol=reltol, bits=bits)


def listed():
    return [
        # the smallest drop-in call: propane (the exchange tests' molecule),
        # host arrays in and out, where latency and launches count
        _coulomb("j_c3h8_host", "alkane", 3, via="host"),
        # the reference's own test size, C10H22, one FP64 density on the device
        _coulomb("j_c10h22", "alkane", 10),
        # the mid-size chain in an SCF loop as a graph, FP32-stored, with the
        # persistent executor (the autotuner's choice there)
        _coulomb("j_c30h62_f32_graph", "alkane", 30, bits=32, via="graph", executor=1),
        # five response densities at once in FP64: widths 4 + 1, a ragged batch
        _coulomb("j_c30h62_x5", "alkane", 30, ndens=5),
        # the globular case: many small coupling blocks
        _coulomb("j_h2o64_f32", "water", 64, bits=32),
        # the long chain of the headline benchmark, one density per replay
        _coulomb("j_c100h202_f32_graph", "alkane", 100, reltol=1e-8, bits=32, via="graph"),
        # the same chain's batching workload: sixteen densities in one pass
        _coulomb("j_c100h202_f32_x16", "alkane", 100, reltol=1e-8, ndens=16, bits=32),
        # exchange of the reference's test size, the mid-size chain and the
        # globular cluster (hybrid functionals and Hartree-Fock build K
        # beside J in every iteration; the cluster's handle keeps U and B in
        # FP32 for its J, K itself is FP64)
        _exchange("k_c10h22", "alkane", 10),
        _exchange("k_c30h62", "alkane", 30),
        _exchange("k_h2o64", "water", 64, bits=32),
        # the memory-saving form on the mid-size chain
        dict(name="jit_c30h62", call="on_the_fly", molecule="alkane", n=30, reltol=1e-6),
        # eight small alkanes C4..C32 (fragments of one batch) in one call
        dict(name="group_c4_c32_f32", call="group", first=4, step=4, count=8, reltol=1e-6, bits=32),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    call = rng.choice(["coulomb"] * 5 + ["exchange"] * 3 + ["on_the_fly"] * 2 + ["group"])
    reltol = rng.choice([1e-6, 1e-6, 1e-8])
    kind = rng.choice(["alkane", "alkane", "water"])
    if call == "coulomb":
        n = _log_int(rng, 2, 50 if kind == "alkane" else 64)
        ndens = rng.choice([1, 1, 1, 1, 2, 3, 4, 6, 7, 8, 11, 13, 16, 16])
        return dict(call=call, molecule=kind, n=n, reltol=reltol, ndens=ndens, bits=rng.choice([32, 64]),
                    via=rng.choice(["host", "device", "device", "graph"]), executor=rng.choice([0, 0, 1]))
    if call == "exchange":
        return dict(call=call, molecule=kind, n=_log_int(rng, 2, 40), reltol=reltol, bits=rng.choice([32, 64]))
    if call == "on_the_fly":
        return dict(call=call, molecule=kind, n=_log_int(rng, 2, 24 if kind == "alkane" else 20), reltol=reltol)
    return dict(call=call, first=rng.randint(2, 6), step=rng.randint(1, 4), count=rng.randint(2, 8), reltol=reltol,
                bits=rng.choice([32, 64]))


# ---------------------------------------------------------------------------
# What a program keeps over its SCF iterations
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _atoms(kind, n):
    """Seeded geometry of a molecule (the benchmark's rules)."""
    rng = M.rng_for(1000 + n)
    return M.alkane(n, rng) if kind == "alkane" else M.water_cluster(n, rng)


@functools.lru_cache(maxsize=None)
def _handle(kind, n, reltol, bits, executor, jit, graph):
    """A built representation, uploaded; `graph` > 0: with the fixed buffers
    and the captured Coulomb graph of that many densities.  A graph belongs to
    its handle, so each form a program uses has a handle of its own."""
    h = h2eri.H2ERI(1e-10, 1e-10, reltol)
    h.read_mol_text(M.mol_text(_atoms(kind, n))).process_shells().partition().build_h2(jit)
    if jit:
        return h
    if bits != 64:
        h.set_precision(bits)
    if executor:
        h.set_executor(executor)
    h.upload()
    if graph:
        h.D_buf = torch.zeros((graph, h.nbf, h.nbf), dtype=torch.float64, device=DEV)
        h.J_buf = torch.zeros_like(h.D_buf)
        torch.cuda.synchronize()
        h.graph_capture("coulomb", graph, h.D_buf.data_ptr(), h.J_buf.data_ptr())
    return h


def _case_handle(c):
    return _handle(c["molecule"], c["n"], c["reltol"], c.get("bits", 64), c.get("executor", 0),
                   1 if c["call"] == "on_the_fly" else 0, c["ndens"] if c.get("via") == "graph" else 0)


def _group_sizes(c):
    return [c["first"] + i * c["step"] for i in range(c["count"])]


@functools.lru_cache(maxsize=None)
def _group(first, step, count, reltol, bits):
    """The molecules' handles, their group on fixed buffers and the buffers."""
    hs = [_handle("alkane", first + i * step, reltol, bits, 0, 0, 0) for i in range(count)]
    ends = np.cumsum([h.n for h in hs]).tolist()
    X = torch.zeros(ends[-1], dtype=torch.float64, device=DEV)
    Y = torch.zeros_like(X)
    parts = list(zip([0] + ends[:-1], ends))
    g = h2eri.Group(hs, [X[b:e].data_ptr() for b, e in parts], [Y[b:e].data_ptr() for b, e in parts])
    return hs, g, X, Y, [Y[b:e] for b, e in parts]


@functools.lru_cache(maxsize=None)
def _pair_rows(h):
    """Of every row of x: its two basis functions and whether their shells
    differ (row order: n * nbf(M) + m of the pair (M, N), pair after pair)."""
    t = h.tree()
    sbf, sp = t["shell_bf_sidx"], t["sp_shell_idx"].reshape(2, -1)
    a, b, d = [], [], []
    for s0, s1 in sp.T.tolist():
        m, n = np.arange(sbf[s0], sbf[s0 + 1]), np.arange(sbf[s1], sbf[s1 + 1])
        a.append(np.tile(m, len(n)))
        b.append(np.repeat(n, len(m)))
        d.append(np.full(len(m) * len(n), s0 != s1))
    return np.concatenate(a), np.concatenate(b), np.concatenate(d)


# ---------------------------------------------------------------------------
# One iteration's inputs
# ---------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _damping(kind, n):
    R = torch.from_numpy(M.bf_centers(_atoms(kind, n))).to(DEV)
    return torch.exp(-0.5 * (R[:, None, :] - R[None, :, :]).norm(dim=-1))


def _densities(kind, n, count, seed):
    """`count` densities 2 Q Q^T o exp(-0.5 |R_i - R_j|), Q the orthonormal
    basis of a seeded Gaussian nbf x nocc matrix (h2eri.molecules.density)."""
    damp = _damping(kind, n)
    nocc = 4 * n + 1 if kind == "alkane" else 5 * n
    gen = torch.Generator(device=DEV).manual_seed(int(seed))
    Ds = []
    for _ in range(count):
        Q = torch.linalg.qr(torch.randn((len(damp), nocc), dtype=torch.float64, device=DEV, generator=gen))[0]
        D = 2.0 * (Q @ Q.T) * damp
        Ds.append(0.5 * (D + D.T))
    return torch.stack(Ds)


def _uncontract(h, D):
    a, b, d = (torch.from_numpy(v).to(DEV) for v in _pair_rows(h))
    return D[b, a] * torch.where(d, 2.0, 1.0)


def prepare(case, seed):
    c = dict(case)
    if c["call"] == "group":
        hs, g, X, Y, ys = _group(c["first"], c["step"], c["count"], c["reltol"], c["bits"])
        x = torch.cat([_uncontract(h, _densities("alkane", n, 1, seed + 7919 * n)[0])
                       for h, n in zip(hs, _group_sizes(c))])
        return dict(c=c, group=g, X=X, x=x, ys=ys)
    h = _case_handle(c)
    D = _densities(c["molecule"], c["n"], c.get("ndens", 1), seed)
    if c["call"] == "coulomb" and c["via"] == "host":
        return dict(c=c, h=h, D=D.cpu().numpy())
    s = dict(c=c, h=h, D=D)
    if c["call"] == "coulomb" and c["via"] == "graph":
        return s
    s["out"] = torch.empty_like(D)
    if c["call"] == "exchange":
        h.exchange_workbuf_init()
    return s


def run(s):
    c = s["c"]
    stream = torch.cuda.current_stream().cuda_stream
    if c["call"] == "group":
        s["X"].copy_(s["x"])
        s["group"].matvec(stream)
        return s["ys"]
    h, D = s["h"], s["D"]
    if c["call"] == "coulomb" and c["via"] == "host":
        return h.build_coulomb(D[0]) if c["ndens"] == 1 else h.build_coulomb_multi(D)
    if c["call"] == "coulomb" and c["via"] == "graph":
        h.D_buf.copy_(D)
        h.graph_replay(stream)
        return h.J_buf
    out = s["out"]
    if c["call"] == "exchange":
        h.build_exchange_dev(D.data_ptr(), out.data_ptr(), stream)
    elif c.get("ndens", 1) == 1:
        h.build_coulomb_dev(D.data_ptr(), out.data_ptr(), stream)
    else:
        h.build_coulomb_multi_dev(c["ndens"], D.data_ptr(), out.data_ptr(), stream)
    return out


# ---------------------------------------------------------------------------
# Work
# ---------------------------------------------------------------------------
def _product_work(h, bits, nv, vector_bytes):
    """One product with the representation: every stored block read once (U
    and B in their storage precision, D in FP64), the vectors; 2 FLOP per
    element and side (U up and down, B and off-diagonal D both ways)."""
    b = h.matvec_bytes()
    U, B, D = 0.5 * b["U"], b["B"], b["D"]
    elements = (U + B) / (bits // 8) + D / 8
    return {"bytes": U + B + D + vector_bytes, "flops": 4.0 * elements * nv}


def _exchange_flops(h, blocks):
    """K of the block terms F = L R^T with L m0 x k and R m1 x k: the ket
    contraction |B(0)| m1 k and the bra contraction m0 |B(1)| k, B(i) the basis
    functions of node i's rows, both orientations of a row."""
    t = h.tree()
    a, b, _ = _pair_rows(h)
    lo, hi = t["mat_cluster"][:, 0], t["mat_cluster"][:, 1] + 1
    nb = {}

    def rows_bfs(n):
        if n not in nb:
            nb[n] = (hi[n] - lo[n], len(np.unique(np.concatenate([a[lo[n]:hi[n]], b[lo[n]:hi[n]]]))))
        return nb[n]

    flops = 0.0
    for kind, n0, n1, rank in blocks:
        (m0, b0), (m1, b1) = rows_bfs(n0), rows_bfs(n1)
        flops += 4.0 * rank * (b0 * m1 + m0 * b1)
    return flops


def _shape(p):
    return (p.contents.nrow, p.contents.ncol, p.contents.ld) if p else (0, 0, 0)


def work(case):
    c = dict(case)
    if c["call"] == "group":
        each = []
        for n in _group_sizes(c):
            h = _handle("alkane", n, c["reltol"], c["bits"], 0, 0, 0)
            each.append(_product_work(h, c["bits"], 1, 16.0 * h.n))
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    h = _case_handle(c)
    matrices = 2.0 * ENTRY_BYTES * h.nbf ** 2
    if c["call"] == "coulomb":
        return _product_work(h, c["bits"], c["ndens"], c["ndens"] * matrices)
    s = h.s
    if c["call"] == "on_the_fly":
        # the integrals of each block once (the counts are of both sides):
        # about 30 FLOP per primitive quartet for its centres, prefactor and
        # Boys value, 4 to apply an integral to both sides
        q = h.jit_stats()
        U = sum(r * k for r, k, _ in map(_shape, (s.U[i] for i in range(s.n_node))))
        return {"bytes": ENTRY_BYTES * U + matrices, "flops": 15.0 * q["prim_quartets"] + 2.0 * q["eri_values"] + 4.0 * U}
    t = h.tree()
    lv = t["node_level"]
    blocks = []
    for i, (n0, n1) in enumerate(t["r_adm_pairs"].tolist()):
        r, k, ld = _shape(s.c_B_blks[i])
        full = [k if lv[n1] >= lv[n0] else r, r if lv[n0] >= lv[n1] else k]
        blocks.append(("B", n0, n1, -ld if ld < 0 else min(full)))
    leaves = t["height_nodes"][0][: t["height_n_node"][0]].tolist()
    pairs = [(n, n) for n in leaves] + [tuple(p) for p in t["r_inadm_pairs"].tolist()]
    for i, (n0, n1) in enumerate(pairs):
        r, k, ld = _shape(s.c_D_blks[i])
        blocks.append(("D", n0, n1, -ld if ld < 0 else min(r, k)))
    b = h.matvec_bytes()
    return {"bytes": 0.5 * b["U"] + b["B"] + b["D"] + matrices, "flops": _exchange_flops(h, blocks)}


# ---------------------------------------------------------------------------
# The same in plain numpy and torch, 64 bits
# ---------------------------------------------------------------------------
def _mul(blk, x, transpose=False):
    kind = blk[0]
    if kind == "dense":
        return (blk[1].T if transpose else blk[1]) @ x
    U, VT = blk[1], blk[2]
    return VT @ (U.T @ x) if transpose else U @ (VT.T @ x)


def _apply(h, x):
    """A x by the definition of the representation (x: N x nv)."""
    t = h.tree()
    U, B, D = h.blocks()
    lv, nchild, children = t["node_level"], t["n_child"], t["children"]
    lo, hi = t["mat_cluster"][:, 0], t["mat_cluster"][:, 1] + 1
    order = np.argsort(-lv, kind="stable").tolist()   # leaves of the deepest level first
    up, y1 = {}, {}
    for n in order:
        if U[n] is None or U[n][1].shape[1] == 0:
            continue
        if nchild[n]:
            src = [up[k] for k in children[n][: nchild[n]].tolist() if k in up]
            src = np.concatenate(src)
        else:
            src = x[lo[n]:hi[n]]
        up[n] = U[n][1].T @ src
        y1[n] = np.zeros_like(up[n])
    y = np.zeros_like(x)
    for blk, (n0, n1) in zip(B, t["r_adm_pairs"].tolist()):
        if blk is None or 0 in blk[1].shape:
            continue
        deep0, deep1 = lv[n0] >= lv[n1], lv[n1] >= lv[n0]
        in0, in1 = (up[n1] if deep1 else x[lo[n1]:hi[n1]]), (up[n0] if deep0 else x[lo[n0]:hi[n0]])
        o0, o1 = _mul(blk, in0), _mul(blk, in1, True)
        if deep0:
            y1[n0] += o0
        else:
            y[lo[n0]:hi[n0]] += o0
        if deep1:
            y1[n1] += o1
        else:
            y[lo[n1]:hi[n1]] += o1
    for n in reversed(order):
        if n not in y1:
            continue
        o = U[n][1] @ y1[n]
        if not nchild[n]:
            y[lo[n]:hi[n]] += o
            continue
        at = 0
        for k in children[n][: nchild[n]].tolist():
            if k in y1:
                y1[k] += o[at:at + len(y1[k])]
                at += len(y1[k])
    leaves = t["height_nodes"][0][: t["height_n_node"][0]].tolist()
    for blk, n in zip(D, leaves):
        if blk is not None:
            y[lo[n]:hi[n]] += _mul(blk, x[lo[n]:hi[n]])
    for blk, (n0, n1) in zip(D[len(leaves):], t["r_inadm_pairs"].tolist()):
        if blk is not None:
            y[lo[n0]:hi[n0]] += _mul(blk, x[lo[n1]:hi[n1]])
            y[lo[n1]:hi[n1]] += _mul(blk, x[lo[n0]:hi[n0]], True)
    return y


def _exact_coulomb(h, Ds):
    a, b, d = _pair_rows(h)
    x = (Ds[:, b, a] * np.where(d, 2.0, 1.0)).T
    y = _apply(h, np.ascontiguousarray(x))
    J = np.zeros_like(Ds)
    for k in range(len(Ds)):
        np.add.at(J[k], (b, a), np.where(d, 1.0, 0.5) * y[:, k])
        J[k] = J[k] + J[k].T
    return J


def _exact_exchange(h, D):
    """K_mq = sum (mn|pq) D_np block by block: F of a block from the expanded
    bases, contracted over both orientations of its rows and columns."""
    t = h.tree()
    U, B, Dblk = h.blocks()
    lv, nchild, children = t["node_level"], t["n_child"], t["children"]
    lo, hi = t["mat_cluster"][:, 0], t["mat_cluster"][:, 1] + 1

    def dev(v):
        return torch.from_numpy(np.ascontiguousarray(v)).to(DEV)

    a, b, d = map(dev, _pair_rows(h))
    # the reference's screening: shell blocks of D without any |D| > 1e-10
    sbf = t["shell_bf_sidx"]
    shell = dev(np.repeat(np.arange(len(sbf) - 1), np.diff(sbf)))
    ns = len(sbf) - 1
    kept = torch.zeros(ns * ns, dtype=torch.bool, device=DEV)
    where = (shell[:, None] * ns + shell[None, :])
    kept[where[D.abs() > 1e-10]] = True
    D = D * kept[where]
    P = {}
    for n in np.argsort(-lv, kind="stable").tolist():
        if U[n] is None or U[n][1].shape[1] == 0:
            continue
        Un = dev(U[n][1])
        if nchild[n]:
            parts, at = [], 0
            for k in children[n][: nchild[n]].tolist():
                r = P[k].shape[1] if k in P else 0
                parts.append(P[k] @ Un[at:at + r] if r else
                             torch.zeros((hi[k] - lo[k], Un.shape[1]), dtype=torch.float64, device=DEV))
                at += r
            Un = torch.cat(parts)
        P[n] = Un
    nbf = h.nbf
    sums = [torch.zeros((nbf, nbf), dtype=torch.float64, device=DEV) for _ in range(2)]

    def contract(K, F, r0, c0):
        rows, cols = slice(r0, r0 + F.shape[0]), slice(c0, c0 + F.shape[1])
        Fr = F * d[rows, None]
        for m, n, Fm in ((a[rows], b[rows], F), (b[rows], a[rows], Fr)):
            for p, q, Fc in ((a[cols], b[cols], Fm), (b[cols], a[cols], Fm * d[None, cols])):
                T = torch.zeros((F.shape[0], nbf), dtype=torch.float64, device=DEV)
                T.index_add_(1, q, Fc * D[n][:, p])
                K.index_add_(0, m, T)

    def dense(blk):
        return dev(blk[1]) if blk[0] == "dense" else dev(blk[1]) @ dev(blk[2]).T

    leaves = t["height_nodes"][0][: t["height_n_node"][0]].tolist()
    for blk, n in zip(Dblk, leaves):
        if blk is not None:
            contract(sums[1], dense(blk), lo[n], lo[n])
    for blk, (n0, n1) in zip(Dblk[len(leaves):], t["r_inadm_pairs"].tolist()):
        if blk is not None:
            contract(sums[0], dense(blk), lo[n0], lo[n1])
    for blk, (n0, n1) in zip(B, t["r_adm_pairs"].tolist()):
        if blk is None or 0 in blk[1].shape:
            continue
        C = dense(blk)
        if lv[n1] >= lv[n0]:
            C = C @ P[n1].T
        for r in range(0, hi[n0] - lo[n0], 2048):   # row chunks bound the memory of the big nodes
            if lv[n0] >= lv[n1]:
                contract(sums[0], P[n0][r:r + 2048] @ C, lo[n0] + r, lo[n1])
            else:
                contract(sums[0], C[r:r + 2048], lo[n0] + r, lo[n1])
    return sums[0] + sums[0].T + sums[1]


def exact(case, seed):
    """The same values in 64 bits from the blocks of the representation (the
    inputs of a product; J and K are defined by them).  None for the on-the-fly
    form, whose blocks are integrals evaluated in the call, and for the
    molecules whose representation alone takes too long to build."""
    c = dict(case)
    if c["call"] == "on_the_fly":
        return None
    if c["call"] == "group":
        ys = []
        for n in _group_sizes(c):
            h = _handle("alkane", n, c["reltol"], c["bits"], 0, 0, 0)
            x = _uncontract(h, _densities("alkane", n, 1, seed + 7919 * n)[0]).cpu().numpy()
            ys.append(_apply(h, x[:, None])[:, 0])
        return ys
    if c["n"] > 64 or (c["call"] == "exchange" and c["molecule"] == "water" and c["n"] > 40):
        return None
    h = _case_handle(c)
    D = _densities(c["molecule"], c["n"], c.get("ndens", 1), seed)
    if c["call"] == "exchange":
        return _exact_exchange(h, D[0])[None]
    J = _exact_coulomb(h, D.cpu().numpy())
    return J[0] if c["via"] == "host" and c["ndens"] == 1 else J
