"""What a program does with this library, as timed cases over its public entry points.

A case is a dict of plain values whose "kind" names one of:

  theta    ``tensordot`` of two neighbouring MPS tensors: the smallest contraction of a sweep
  env      ``tensordot`` X(b, a', s, w) . Abar(a', s, b') of an environment update
  lanczos  ``one_step_lanczos``: two applications of the two-site Hamiltonian and the step's scalars
  gemms    one ``tensordot`` over many unrelated blocks (sizes log-uniform in 4 .. 768)
  split    truncating ``svd`` of a two-site state, and its factors put back together
  svds     ``svd`` of many unrelated matrices at once (sizes log-uniform in 4 .. 768)
  rho      ``eigh`` of a block-diagonal density matrix
  dmrg     a whole ``dmrg`` call that takes a small-bond state to its full bond (0 Krylov vectors: the
           one-step update; 4: the k-step update that a solve service runs), then the entanglement
           spectrum in the middle

Everything is FP64.  A program holds one context, its Hamiltonian and its tensors on the device:
``prepare`` makes those, ``run`` is the call.  Results stay on the device, as they do in a program
that goes on with them, until somebody reads an entry of what ``run`` returns.
Singular vectors are unique only up to their signs, so the factors of a split are compared through
what a program builds from them: the product U d V and the overlap U U of the new site.
"""
import math

import numpy as np
import torch  # noqa: F401  (one HIP runtime for the process: torch's is loaded first)

import quantit_amd as qa
from quantit_amd import models

U1 = (0,)
UP_DOWN = [(1, (1,)), (1, (-1,))]
CUTOFF = 1e-10
ARENA = 24 << 30

_contexts = {}


def _context(krylov=0):
    """The process's context for the one-step update (0) or the k-step one."""
    if krylov not in _contexts:
        _contexts[krylov] = qa.Context(0, arena_bytes=ARENA if krylov == 0 else 4 << 30)
        _contexts[krylov].set_lanczos(krylov, 1e-12)
    return _contexts[krylov]


class Results(dict):
    """What a call returned: device tensors, read to the host (all blocks in list order, one
    array) when an entry is asked for, and plain numbers as they are."""

    def __getitem__(self, name):
        v = super().__getitem__(name)
        return _flat(v) if isinstance(v, qa.BTensor) else v


def _flat(t):
    blocks = t.to_parts()[4]
    return np.concatenate([b.ravel() for b in blocks.values()]) if blocks else np.zeros(0)


# ---- legs and tensors on the host -------------------------------------------------------------

def _bond(D, parity, spread=3.0):
    """A U(1) bond of D states: charges 2Sz of one parity, sizes by a normal profile."""
    q = [c for c in range(-12, 13) if (c - parity) % 2 == 0]
    w = np.exp(-0.5 * (np.array(q) / spread) ** 2)
    n = np.floor(D * w / w.sum()).astype(int)
    for i in np.argsort(-w, kind="stable")[: D - int(n.sum())]:
        n[i] += 1
    return [(int(k), (c,)) for k, c in zip(n, q) if k > 0]


def _inv(leg):
    return [(n, tuple(-x for x in c)) for n, c in leg]


def _leg(parts, d):
    return list(zip(parts["secs"][d], parts["cvals"][d]))


def _structure(legs):
    """Block indices whose charges sum to zero, in lexicographic order."""
    found = [((), 0)]
    for leg in legs[:-1]:
        found = [(i + (k,), q + c[0]) for i, q in found for k, (_, c) in enumerate(leg)]
    last = {}
    for k, (_, c) in enumerate(legs[-1]):
        last.setdefault(-c[0], []).append(k)
    return [i + (k,) for i, q in found for k in last.get(q, ())]


def _parts(legs, blocks):
    return dict(groups=U1, secs=[[n for n, _ in leg] for leg in legs], cvals=[[c for _, c in leg] for leg in legs],
                sel=(0,), blocks=blocks)


def _random(legs, rng, scale=1.0):
    """Every allowed block, independent normal entries."""
    idx = _structure(legs)
    shapes = [tuple(legs[d][k][0] for d, k in enumerate(i)) for i in idx]
    x = rng.standard_normal(sum(math.prod(s) for s in shapes)) * scale
    blocks, at = {}, 0
    for i, s in zip(idx, shapes):
        n = math.prod(s)
        blocks[i] = x[at:at + n].reshape(s)
        at += n
    return _parts(legs, blocks)


def _diagonal(rows, cols, fill):
    """Unrelated matrices as the blocks of one tensor, each with a charge of its own."""
    return dict(groups=U1, secs=[[int(r) for r in rows], [int(c) for c in cols]],
                cvals=[[(i,) for i in range(len(rows))], [(-i,) for i in range(len(cols))]], sel=(0,),
                blocks={(i, i): fill(int(r), int(c)) for i, (r, c) in enumerate(zip(rows, cols))})


def _sizes(rng, n, lo=4, hi=768):
    return np.floor(np.exp(rng.uniform(np.log(lo), np.log(hi + 1), n))).astype(int).clip(lo, hi)


def _graded(rng, values, m, n, top, decades):
    """U diag(s) V^T with random orthonormal factors: the graded spectra of states."""
    k = min(m, n)
    u = np.linalg.qr(rng.standard_normal((m, k)))[0]
    v = np.linalg.qr(rng.standard_normal((n, k)))[0]
    s = top * 10.0 ** (-decades * ((np.arange(k) + values.uniform(0.0, 0.9, k)) / k) ** 0.7)
    return (u * s) @ v.T


def _sectors(legs):
    """{charge: (row blocks, column blocks)} of a two-site state split in its middle, each block
    as (indices, offset, size)."""
    out = {}
    for side, (x, y) in enumerate(((legs[0], legs[1]), (legs[2], legs[3]))):
        for i, (n, a) in enumerate(x):
            for j, (m, b) in enumerate(y):
                q = (a[0] + b[0]) * (1 if side == 0 else -1)
                rows = out.setdefault(q, ([], []))[side]
                rows.append(((i, j), sum(r[2] for r in rows), n * m))
    return {q: rc for q, rc in sorted(out.items()) if rc[0] and rc[1]}


def _two_site(D, decades, rng):
    """A normalised two-site state whose Schmidt values fall over so many decades in every sector
    (about six in the states of a cylinder, whose bond cuts them; ten or more in those of a chain,
    where the cutoff does), the wide sectors (small charges) holding most of the weight.  The
    values go by the size alone, so that every seed keeps as many of them."""
    values = np.random.default_rng([13, D])
    legs = [_bond(D, 0), UP_DOWN, UP_DOWN, _inv(_bond(D, 0))]
    blocks = {}
    for q, (rows, cols) in _sectors(legs).items():
        m, n = sum(r[2] for r in rows), sum(c[2] for c in cols)
        a = _graded(rng, values, m, n, math.exp(-q * q / 12.0), decades)
        for (i, s), r0, r in rows:
            for (t, j), c0, c in cols:
                blocks[(i, s, t, j)] = np.ascontiguousarray(a[r0:r0 + r, c0:c0 + c]).reshape(
                    legs[0][i][0], 1, 1, legs[3][j][0])
    norm = math.sqrt(sum(float(np.vdot(b, b)) for b in blocks.values()))
    return _parts(legs, {k: b / norm for k, b in blocks.items()})


def _hamiltonian(case):
    """The two centre sites of the model's MPO, as block parts."""
    w = case["width"]
    n = 8 if w == 1 else 4 * w
    bonds = models.chain_bonds(n) if w == 1 else models.cylinder_bonds(w, 4)
    parts = models.bmpo_parts(models.spin_mpo(n, bonds, delta=0.8))
    return parts[n // 2 - 1], parts[n // 2]


def _spins(case, seed):
    """A random-field XXZ chain: no symmetry beyond U(1), so that no two singular values tie."""
    n = case["sites"]
    fields = np.random.default_rng(seed).uniform(-0.8, 0.8, n)
    return models.bmpo_parts(models.spin_mpo(n, models.chain_bonds(n), delta=case["delta"], fields=fields))


def _inputs(case, seed):
    """The host tensors of a case, by name."""
    rng = np.random.default_rng([seed, 7])
    kind = case["kind"]
    if kind == "theta":
        a, b, c = _bond(case["D"], 0), _bond(case["D"], 1), _bond(case["D"], 0)
        return {"a": _random([a, UP_DOWN, _inv(b)], rng), "b": _random([b, UP_DOWN, _inv(c)], rng)}
    if kind == "env":
        w = _leg(_hamiltonian({"width": 4})[0], 2)
        a, b = _bond(case["D"], 0), _bond(case["D"], 1)
        return {"a": _random([_inv(b), a, UP_DOWN, w], rng), "b": _random([_inv(a), _inv(UP_DOWN), b], rng)}
    if kind == "lanczos":
        w1, w2 = _hamiltonian(case)
        wl, wr = _inv(_leg(w1, 0)), _inv(_leg(w2, 2))
        theta = _two_site(case["D"], 6.0, rng)
        l, r = _leg(theta, 0), _leg(theta, 3)
        scale = 1.0 / math.sqrt(case["D"])
        return {"theta": theta, "w1": w1, "w2": w2, "left": _random([_inv(l), wl, l], rng, scale),
                "right": _random([_inv(r), wr, r], rng, scale)}
    shapes = np.random.default_rng([11, case.get("items", 0)])
    if kind == "gemms":
        m, n, k = (_sizes(shapes, case["items"]) for _ in range(3))
        fill = lambda r, c: rng.standard_normal((r, c))  # noqa: E731
        return {"a": _diagonal(m, k, fill), "b": _diagonal(k, n, fill)}
    if kind == "split":
        return {"theta": _two_site(case["D"], case["decades"], rng)}
    if kind == "svds":
        m, n = (_sizes(shapes, case["items"]) for _ in range(2))
        return {"a": _diagonal(m, n, lambda r, c: rng.standard_normal((r, c)))}
    if kind == "rho":
        # the neutral sector first: an eigh's vectors carry the charge of the first one
        leg = sorted(_bond(case["D"], 0), key=lambda s: abs(s[1][0]))
        blocks = {}
        for i, (n, c) in enumerate(leg):
            u = np.linalg.qr(rng.standard_normal((n, n)))[0]
            p = math.exp(-c[0] ** 2 / 6.0) * 10.0 ** (-12.0 * (np.arange(n) + rng.uniform(0.0, 0.9, n)) / n)
            a = (u * p) @ u.T
            blocks[(i, i)] = 0.5 * (a + a.T)
        trace = sum(float(np.trace(b)) for b in blocks.values())
        return {"rho": _parts([leg, _inv(leg)], {k: b / trace for k, b in blocks.items()})}
    raise ValueError(kind)


# ---- the cases ---------------------------------------------------------------------------------

def listed():
    return [
        # the ends of a chain and small bonds: a handful of blocks, all launch latency
        {"name": "theta_D16", "kind": "theta", "D": 16},
        # the environment update of the cylinder: few columns of many sizes, long summed K
        {"name": "env_D1024", "kind": "env", "D": 1024},
        # the Hamiltonian of a chain at a small odd bond: many small blocks
        {"name": "lanczos_chain_D203", "kind": "lanczos", "D": 203, "width": 1},
        # the same step of a width-4 cylinder at the bond that its solve grows to
        {"name": "lanczos_cylinder_D1024", "kind": "lanczos", "D": 1024, "width": 4},
        # the grouped batch: unrelated blocks from 4 to 768
        {"name": "gemms_1024", "kind": "gemms", "items": 1024},
        # two-site updates: of chains at a small bond and an ordinary odd one (more decades than a
        # Gram matrix holds), and of the cylinder at the bond that its solve grows to
        {"name": "split_D48", "kind": "split", "D": 48, "decades": 10.0},
        {"name": "split_D301", "kind": "split", "D": 301, "decades": 10.0},
        {"name": "split_D1024", "kind": "split", "D": 1024, "decades": 6.0},
        # unrelated singular value decompositions, tall and wide
        {"name": "svds_96", "kind": "svds", "items": 96},
        # density matrices of a bond
        {"name": "rho_D256", "kind": "rho", "D": 256},
        # whole solves: the reference's one-step update, and the served form
        {"name": "dmrg_L32_D64", "kind": "dmrg", "sites": 32, "D": 64, "sweeps": 3, "krylov": 0, "delta": 0.9},
        {"name": "dmrg_served_L20_D48", "kind": "dmrg", "sites": 20, "D": 48, "sweeps": 3, "krylov": 4, "delta": 1.3},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["theta", "env", "lanczos", "gemms", "split", "split", "svds", "rho", "dmrg"])
    if kind == "theta":
        return {"kind": kind, "D": log(6, 512)}
    if kind == "env":
        return {"kind": kind, "D": log(40, 1000)}
    if kind == "lanczos":
        return {"kind": kind, "D": log(30, 1000), "width": rng.choice([1, 4])}
    if kind == "gemms":
        return {"kind": kind, "items": log(24, 1000)}
    if kind == "split":
        return {"kind": kind, "D": log(16, 1000), "decades": round(rng.uniform(4.0, 11.0), 2)}
    if kind == "svds":
        return {"kind": kind, "items": rng.randint(8, 90)}
    if kind == "rho":
        return {"kind": kind, "D": log(16, 256)}
    return {"kind": kind, "sites": 2 * rng.randint(6, 15), "D": rng.randint(16, 60), "sweeps": rng.randint(2, 3),
            "krylov": rng.choice([0, 4]), "delta": round(rng.uniform(0.5, 1.5), 3)}


def _options(bond, sweeps):
    return qa.DmrgOptions(convergence_criterion=0.0, maximum_bond=bond, maximum_iterations=sweeps)


def prepare(case, seed):
    ctx = _context(case.get("krylov", 0))
    if case["kind"] == "dmrg":
        mpo = [qa.BTensor.from_parts(ctx, **p) for p in _spins(case, seed)]
        mps = [qa.BTensor.from_parts(ctx, **p) for p in models.random_bmps_parts(case["sites"], 12, q=0, seed=seed)]
        return {"case": case, "mpo": mpo, "mps": qa.dmrg(mpo, qa.mps_prepare(mps), _options(12, 8))[1]}
    state = {k: qa.BTensor.from_parts(ctx, **p) for k, p in _inputs(case, seed).items()}
    if case["kind"] == "lanczos":
        state["w12"] = state.pop("w1").tensordot(state.pop("w2"), [2], [0]).permute([0, 1, 3, 4, 2, 5])
    state["case"] = case
    return state


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("theta", "gemms"):
        last = s["a"].rank - 1
        return Results(out=s["a"].tensordot(s["b"], [last], [0]))
    if kind == "env":
        return Results(out=s["a"].tensordot(s["b"], [1, 2], [0, 1]))
    if kind == "lanczos":
        h, a0, a1, b = qa.one_step_lanczos(s["theta"], s["w12"], s["left"], s["right"])
        return Results(vector=h, a0=a0, a1=a1, b=b)
    if kind == "split":
        u, d, v = qa.svd(s["theta"], 2, tol=CUTOFF, min_size=4, max_size=case["D"])
        right = v.mul(d).conj().permute([2, 0, 1])
        return Results(d=d, state=u.tensordot(right, [2], [0]), overlap=u.tensordot(u.conj(), [0, 1], [0, 1]))
    if kind == "svds":
        u, d, v = qa.svd(s["a"], 1)
        return Results(d=d, product=u.tensordot(v.mul(d).conj(), [1], [1]), overlap=u.tensordot(u.conj(), [0], [0]))
    if kind == "rho":
        d, u = qa.eigh(s["rho"], 1)
        return Results(d=d, product=u.mul(d).tensordot(u.conj(), [1], [1]), overlap=u.tensordot(u.conj(), [0], [0]))
    # the state that was prepared is kept: the solve replaces the handles it is given
    mps = [t.conj().conj() for t in s["mps"]]
    _, mps, log = qa.dmrg(s["mpo"], mps, _options(case["D"], case["sweeps"]))
    middle = case["sites"] // 2
    mps = qa.mps_move_oc(mps, 0, middle)
    values = _flat(qa.svd(mps[middle], 1)[1])
    spectrum = np.zeros(2 * case["D"])  # in the descending order of a plot, longer than a bond becomes
    spectrum[:len(values)] = np.sort(values)[::-1]
    return Results(energies=np.array(log["energies"]), spectrum=spectrum)


# ---- what a pass cannot do without ---------------------------------------------------------------

def _pairs(a, b, da, db):
    """Block pairs of a contraction by output block, in the output's order."""
    fa = [d for d in range(len(a["secs"])) if d not in da]
    fb = [d for d in range(len(b["secs"])) if d not in db]
    by = {}
    for j in sorted(b["blocks"]):
        by.setdefault(tuple(j[d] for d in db), []).append(j)
    out = {}
    for i in sorted(a["blocks"]):
        for j in by.get(tuple(i[d] for d in da), ()):
            out.setdefault(tuple(i[d] for d in fa) + tuple(j[d] for d in fb), []).append((i, j))
    return {k: out[k] for k in sorted(out)}


def _contract(a, b, da, db):
    """The contraction in plain numpy."""
    fa = [d for d in range(len(a["secs"])) if d not in da]
    fb = [d for d in range(len(b["secs"])) if d not in db]
    x = {i: v.transpose(fa + list(da)).reshape(math.prod(v.shape[d] for d in fa), -1) for i, v in a["blocks"].items()}
    y = {j: v.transpose(list(db) + fb).reshape(-1, math.prod(v.shape[d] for d in fb)) for j, v in b["blocks"].items()}
    blocks = {}
    for k, ij in _pairs(a, b, da, db).items():
        v = sum(x[i] @ y[j] for i, j in ij)
        i, j = ij[0]
        blocks[k] = v.reshape([a["blocks"][i].shape[d] for d in fa] + [b["blocks"][j].shape[d] for d in fb])
    pick = lambda name: [a[name][d] for d in fa] + [b[name][d] for d in fb]  # noqa: E731
    return dict(groups=U1, secs=pick("secs"), cvals=pick("cvals"), sel=(0,), blocks=blocks)


def _flops(a, b, da, db):
    """2 M N K over the block pairs."""
    dims = lambda t, i, which: math.prod(t["secs"][d][i[d]] for d in which)  # noqa: E731
    fa = [d for d in range(len(a["secs"])) if d not in da]
    fb = [d for d in range(len(b["secs"])) if d not in db]
    return sum(2.0 * dims(a, i, fa) * dims(a, i, da) * dims(b, j, fb)
               for ij in _pairs(a, b, da, db).values() for i, j in ij)


def _numel(t):
    return sum(math.prod(t["secs"][d][k] for d, k in enumerate(i)) for i in t["blocks"])


def _svd_flops(sizes):
    """14 m n^2 + 8 n^3, m >= n: the usual count of a singular value decomposition with vectors."""
    return sum(14.0 * max(s) * min(s) ** 2 + 8.0 * min(s) ** 3 for s in sizes)


def _w12(inputs):
    t = _contract(inputs["w1"], inputs["w2"], [2], [0])
    p = [0, 1, 3, 4, 2, 5]
    return dict(groups=U1, secs=[t["secs"][d] for d in p], cvals=[t["cvals"][d] for d in p], sel=(0,),
                blocks={tuple(i[d] for d in p): v.transpose(p) for i, v in t["blocks"].items()})


MATVEC = (([0], [0]), ([0, 2, 3], [0, 4, 5]), ([1, 4], [0, 1]))


def work(case):
    kind = case["kind"]
    if kind == "dmrg":
        # each update at the full bond: the state once through two Hamiltonians (one per Krylov
        # vector), one split; the first updates are smaller
        D, w = case["D"], 5.0
        state = _inputs({"kind": "split", "D": D, "decades": 6.0}, 0)["theta"]
        n = _numel(state)
        rows = [sum(r[2] for r in rc[0]) for rc in _sectors([_leg(state, d) for d in range(4)]).values()]
        updates = 2.0 * (case["sites"] - 2) * (case["sweeps"] - 0.5)
        applied = case["krylov"] or 2
        return {"bytes": updates * 8.0 * n * (2 * applied + 3),
                "flops": updates * (applied * 2.0 * n * (2.0 * w * max(rows) / 2) + _svd_flops((r, r) for r in rows))}
    t = _inputs(case, 0)
    if kind in ("theta", "gemms", "env"):
        da, db = ([1, 2], [0, 1]) if kind == "env" else ([len(t["a"]["secs"]) - 1], [0])
        out = sum(math.prod([t["a"]["secs"][d][i[d]] for d in range(len(i)) if d not in da]
                            + [t["b"]["secs"][d][j[d]] for d in range(len(j)) if d not in db])
                  for (i, j), *_ in _pairs(t["a"], t["b"], da, db).values())
        return {"bytes": 8.0 * (_numel(t["a"]) + _numel(t["b"]) + out), "flops": _flops(t["a"], t["b"], da, db)}
    if kind == "lanczos":
        x, flops = t["left"], 0.0
        for y, (da, db) in zip((t["theta"], _w12(t), t["right"]), MATVEC):
            flops += _flops(x, y, da, db)
            shape = _pairs(x, y, da, db)
            pick = lambda name: ([x[name][d] for d in range(len(x["secs"])) if d not in da]  # noqa: E731
                                 + [y[name][d] for d in range(len(y["secs"])) if d not in db])
            x = dict(groups=U1, secs=pick("secs"), cvals=pick("cvals"), sel=(0,), blocks=dict.fromkeys(shape))
        n = _numel(t["theta"])
        return {"bytes": 8.0 * (2 * n + _numel(t["left"]) + _numel(t["right"])), "flops": 2.0 * flops + 8.0 * n}
    name, a = next(iter(t.items()))
    if kind == "split":
        legs = [_leg(a, d) for d in range(4)]
        sizes = [(sum(r[2] for r in rows), sum(c[2] for c in cols)) for rows, cols in _sectors(legs).values()]
        return {"bytes": 8.0 * 3 * _numel(a), "flops": _svd_flops(sizes)}
    sizes = [b.shape for b in a["blocks"].values()]
    return {"bytes": 8.0 * 3 * _numel(a), "flops": _svd_flops(sizes) if kind == "svds" else
            sum(9.0 * n ** 3 for n, _ in sizes)}


# ---- the same results in plain numpy ---------------------------------------------------------------

def _all(blocks):
    return np.concatenate([np.ascontiguousarray(b).ravel() for b in blocks])


def exact(case, seed):
    kind = case["kind"]
    if kind == "dmrg":
        return None
    t = _inputs(case, seed)
    if kind in ("theta", "gemms", "env"):
        da, db = ([1, 2], [0, 1]) if kind == "env" else ([len(t["a"]["secs"]) - 1], [0])
        return {"out": _all(_contract(t["a"], t["b"], da, db)["blocks"].values())}
    if kind == "lanczos":
        w = _w12(t)

        def apply(v):
            x = t["left"]
            for y, (da, db) in zip((v, w, t["right"]), MATVEC):
                x = _contract(x, y, da, db)
            return x

        def dot(x, y):
            return sum(float(np.vdot(x["blocks"][k], y["blocks"][k])) for k in x["blocks"] if k in y["blocks"])

        theta = t["theta"]
        h = apply(theta)
        a0 = dot(h, theta)
        for k, b in theta["blocks"].items():
            h["blocks"][k] = h["blocks"][k] - a0 * b if k in h["blocks"] else -a0 * b
        b = math.sqrt(dot(h, h))
        h["blocks"] = {k: h["blocks"][k] / b for k in sorted(h["blocks"])}
        return {"vector": _all(h["blocks"].values()), "a0": a0, "a1": dot(apply(h), h), "b": b}
    if kind == "svds":
        f = [np.linalg.svd(b, full_matrices=False) for b in t["a"]["blocks"].values()]
        return {"d": _all(s for _, s, _ in f), "product": _all(t["a"]["blocks"].values()),
                "overlap": _all(np.eye(len(s)) for _, s, _ in f)}
    if kind == "rho":
        order = sorted(t["rho"]["blocks"], key=lambda k: t["rho"]["cvals"][0][k[0]])
        f = [np.linalg.eigvalsh(t["rho"]["blocks"][k]) for k in order]
        return {"d": _all(f), "product": _all(t["rho"]["blocks"].values()), "overlap": _all(np.eye(len(p)) for p in f)}
    # split: every sector's singular values, the largest D of them kept
    theta = t["theta"]
    legs = [_leg(theta, d) for d in range(4)]
    sectors = _sectors(legs)
    f = {}
    for q, (rows, cols) in sectors.items():
        a = np.zeros((sum(r[2] for r in rows), sum(c[2] for c in cols)))
        for (i, s), r0, r in rows:
            for (u, j), c0, c in cols:
                a[r0:r0 + r, c0:c0 + c] = theta["blocks"][(i, s, u, j)].reshape(r, c)
        f[q] = np.linalg.svd(a, full_matrices=False)
    values = np.sort(np.concatenate([s for _, s, _ in f.values()]))[::-1]
    weight = np.cumsum(values[::-1] ** 2)[::-1]  # of a value and all behind it
    keep = min(case["D"], int(np.sum(weight > CUTOFF ** 2)))
    least = values[keep - 1] * (1.0 - 2.0 * np.finfo(float).eps)
    blocks, d, overlap = {}, [], []
    for q, (rows, cols) in sectors.items():
        u, s, v = f[q]
        k = int(np.sum(s > least))
        if not k:
            continue
        a = (u[:, :k] * s[:k]) @ v[:k]
        d.append(s[:k])
        overlap.append(np.eye(k))
        for (i, s1), r0, r in rows:
            for (s2, j), c0, c in cols:
                blocks[(i, s1, s2, j)] = a[r0:r0 + r, c0:c0 + c]
    return {"d": _all(d), "state": _all(blocks[k] for k in sorted(blocks)), "overlap": _all(overlap)}
