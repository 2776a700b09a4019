"""The work that a program has this solver do, as measurable cases.

Six kinds, each through the public Python entry points:

  hv      one product y = H x of a sector Hamiltonian on device vectors
          (``qcm.Hamiltonian.apply_device``), the inner call of every Krylov
          method, from the 4 900 states of the 8-site chain to the
          165 636 900 of the periodic 4 x 4 cluster
  solve   one impurity: instance, ground state, Green function on a frequency
          grid (one CDMFT iteration)
  batch   a VCA sweep: many parameter points of one small cluster solved
          together (``qcm.solve_batch``), then G of both spins on one grid
  sef     the self-energy functional on a (frequency, k) grid
  cpt     the CPT Green function averaged over k
  mlp     the learned surrogate: a training run and the predictions after it

Models are Hubbard clusters with the sizes of this repository's workloads,
tests and benchmark; their parameters (U, mu, Weiss and bath values) and the
vectors are drawn from the seed.  ``exact`` builds every reference result
from the second-quantized definition with numpy / torch in 64 bits.
"""
import itertools
import math

import numpy as np
import torch

from pyqcm_amd import lattice, qcm, surrogate

_serial = itertools.count(1)


# --------------------------------------------------------------------------
# cases
# --------------------------------------------------------------------------
def listed():
    return [
        # the smallest product: a Lanczos step on a chain of 8, launch and wait
        {"name": "hv_chain8", "kind": "hv", "model": "chain", "L": 8, "nup": 4, "ndw": 4, "format": "G"},
        # an impurity's electron sector (792 x 924 states, distinct bath
        # values): the band-Lanczos product of a CDMFT iteration
        {"name": "hv_plaq8b_n13", "kind": "hv", "model": "plaq", "L": 12, "nup": 7, "ndw": 6, "format": "G"},
        # the stored-matrix format that the reference uses by default, on the
        # same impurity's ground-state sector
        {"name": "hv_csr_plaq8b", "kind": "hv", "model": "plaq", "L": 12, "nup": 6, "ndw": 6, "format": "S"},
        # the largest single sector: the half-filled periodic 4 x 4 cluster
        {"name": "hv_torus4x4", "kind": "hv", "model": "torus", "L": 16, "nup": 8, "ndw": 8, "format": "G"},
        # the smallest solve: the 4-site chain of the 1D examples, continued fractions
        {"name": "solve_chain4", "kind": "solve", "model": "chain", "L": 4, "method": "F", "nz": 64},
        # the 8-site chain on the Matsubara axis, the 36 orbital pairs' fractions
        {"name": "solve_chain8", "kind": "solve", "model": "chain", "L": 8, "method": "F", "nz": 512},
        # one CDMFT iteration on the plaquette with 8 bath orbitals: ground
        # state (853 776 states), band-Lanczos G on the Matsubara grid
        {"name": "solve_plaq8b", "kind": "solve", "model": "plaq", "L": 12, "method": "L", "nz": 1024},
        # VCA sweep over (U, M, mu) of the 2 x 3 cluster, sectors of 225-400 states
        {"name": "batch_2x3", "kind": "batch", "nx": 2, "ny": 3, "nb": 0, "points": 512, "nz": 256},
        # the upper end of the batched sectors: 2 x 3 with 6 bath orbitals
        # (48 400 states; fractions in sectors of 14 520 and 108 900)
        {"name": "batch_2x3_6b", "kind": "batch", "nx": 2, "ny": 3, "nb": 6, "points": 4, "nz": 256},
        # Potthoff functional of the Neel 2 x 2 cluster: 3 x 32 Legendre
        # frequencies, 128^2 wavevectors, both spins
        {"name": "sef_2x2", "kind": "sef", "nx": 2, "ny": 2, "nf": 32, "nk": 128},
        # spectral function of the CPT on 2 x 3 clusters: 256 real frequencies, 64^2 wavevectors
        {"name": "cpt_2x3", "kind": "cpt", "nx": 2, "ny": 3, "nz": 256, "nk": 64},
        # surrogate refit: 60 full-batch Adam steps on 2 048 rows, then 1 000 predictions
        {"name": "mlp_train", "kind": "mlp", "n_in": 12, "n_out": 641, "rows": 2048, "batch": 2048, "epochs": 60,
         "predict": 1000},
    ]


def draw(rng):
    kind = rng.choice(["hv", "hv", "hv", "solve", "batch", "batch", "sef", "cpt", "mlp"])
    if kind == "hv":
        model = rng.choice(["chain", "plaq", "torus"])
        fmt = "G"
        if model == "chain":
            L = rng.randint(8, 13)
            # fillings within two of half, odd and polarized ones among them
            nup, ndw = L // 2 + rng.randint(-2, 2), L // 2 + rng.randint(-2, 2)
            fmt = rng.choice(["G", "G", "S"])
        elif model == "plaq":
            L = 4 + rng.randint(4, 9)
            nup, ndw = L // 2 + rng.randint(-1, 1), L // 2 + rng.randint(-1, 1)
            fmt = rng.choice(["G", "G", "S"])
        else:
            L = rng.choice([12, 16])
            nup = rng.randint(4, 7 if L == 16 else 6)
            ndw = rng.randint(4, 8 if L == 16 else 6)
        if fmt == "S" and math.comb(L, nup) * math.comb(L, ndw) > 1000000:
            fmt = "G"
        return {"kind": "hv", "model": model, "L": L, "nup": nup, "ndw": ndw, "format": fmt}
    if kind == "solve":
        if rng.random() < 0.5:
            return {"kind": "solve", "model": "chain", "L": rng.randint(3, 9), "method": rng.choice(["F", "L"]),
                    "nz": int(round(math.exp(rng.uniform(math.log(33), math.log(1025)))))}
        return {"kind": "solve", "model": "plaq", "L": 4 + rng.randint(2, 8), "method": "L",
                "nz": int(round(math.exp(rng.uniform(math.log(33), math.log(1025)))))}
    if kind == "batch":
        nx, ny, nb = rng.choice([(2, 1, 0), (2, 2, 0), (2, 2, 0), (2, 3, 0), (2, 3, 0), (2, 2, 2), (2, 2, 4),
                                 (2, 3, 4)])
        top = 512 if nb == 0 else (64 if nx * ny + nb <= 8 else 16)
        return {"kind": "batch", "nx": nx, "ny": ny, "nb": nb,
                "points": int(round(math.exp(rng.uniform(math.log(3), math.log(top))))), "nz": rng.randint(65, 256)}
    if kind == "sef":
        nx, ny = rng.choice([(2, 1), (3, 1), (2, 2), (2, 3)])
        return {"kind": "sef", "nx": nx, "ny": ny, "nf": rng.randint(5, 32),
                "nk": int(round(math.exp(rng.uniform(math.log(9), math.log(96)))))}
    if kind == "cpt":
        nx, ny = rng.choice([(2, 1), (3, 1), (2, 2), (2, 3)])
        return {"kind": "cpt", "nx": nx, "ny": ny, "nz": rng.randint(33, 256),
                "nk": int(round(math.exp(rng.uniform(math.log(7), math.log(64)))))}
    batch = rng.choice([256, 512, 1000, 2048])
    return {"kind": "mlp", "n_in": rng.randint(4, 16), "n_out": rng.randint(33, 641), "rows": batch, "batch": batch,
            "epochs": rng.randint(10, 60), "predict": rng.randint(1, 2000)}


# --------------------------------------------------------------------------
# models: one-body matrix per unit of each operator, from plain bond lists
# --------------------------------------------------------------------------
def _grid_bonds(nx, ny, periodic=False):
    b = set()
    for y in range(ny):
        for x in range(nx):
            for dx, dy in ((1, 0), (0, 1)):
                x2, y2 = x + dx, y + dy
                if periodic:
                    x2, y2 = x2 % nx, y2 % ny
                if x2 < nx and y2 < ny and (x2, y2) != (x, y):
                    i, j = x + nx * y, x2 + nx * y2
                    b.add((min(i, j), max(i, j)))
    return sorted(b)


def _definition(case):
    """(n_sites, n_bath, {operator: (type, [(r, c, v)])}) with 0-based up-spin
    orbitals; 'stag' operators act with opposite sign on the down spin"""
    kind = case["kind"]
    if kind in ("hv", "solve"):
        L = case["L"]
        if case["model"] == "chain":
            ns, bonds = L, [(i, i + 1) for i in range(L - 1)]
        elif case["model"] == "torus":
            nx = 4
            ns, bonds = L, _grid_bonds(nx, L // nx, True)
        else:
            ns, bonds = 4, _grid_bonds(2, 2)
    else:
        ns, bonds = case["nx"] * case["ny"], _grid_bonds(case["nx"], case["ny"])
        L = ns + case.get("nb", 0)
    ops = {"t": ("hop", [(i, j, -1.0) for i, j in bonds]),
           "U": ("int", list(range(ns))),
           "mu": ("hop", [(i, i, -1.0) for i in range(ns)])}
    if kind in ("hv", "solve"):
        if case["model"] == "plaq":
            ops["tp"] = ("hop", [(0, 3, -1.0), (1, 2, -1.0)])
    else:
        nx = case["nx"]
        ops["M"] = ("stag", [(i, i, 1.0 if (i % nx + i // nx) % 2 == 0 else -1.0) for i in range(ns)])
    for b in range(L - ns):
        ops["eb%d" % (b + 1)] = ("hop", [(ns + b, ns + b, 1.0)])
        ops["tb%d" % (b + 1)] = ("hop", [(b % ns, ns + b, 1.0)])
    return ns, L - ns, ops


def _values(case, rng, k=None):
    """operator values of one instance (or of point k of a sweep)"""
    ns, nb, ops = _definition(case)
    v = {"t": 1.0}
    if case["kind"] in ("hv", "solve"):
        v["U"] = float(rng.uniform(4.0, 8.0))
        v["mu"] = 0.5 * v["U"]
        if "tp" in ops:
            v["tp"] = -0.3
    elif case["kind"] == "batch":
        v["U"] = float(rng.uniform(2.0, 10.0))
        v["M"] = float(rng.uniform(0.02, 0.3))
        v["mu"] = float(rng.uniform(-1.0, 1.0))
    else:
        v["U"] = float(rng.uniform(3.0, 8.0))
        v["M"] = float(rng.uniform(0.1, 0.3))
        v["mu"] = 0.5 * v["U"] + float(rng.uniform(-0.3, 0.3))
    bath = np.random.default_rng(7) if case["kind"] == "batch" else rng  # a sweep moves the cluster, not the bath
    eps, hyb = bath.uniform(-2.0, 2.0, nb), bath.uniform(0.2, 0.8, nb)
    for b in range(nb):
        v["eb%d" % (b + 1)] = float(eps[b])
        v["tb%d" % (b + 1)] = float(hyb[b])
    return v


def _sectors(case):
    """(nup, ndw) of the sectors searched for the ground state"""
    if case["kind"] == "hv":
        return [(case["nup"], case["ndw"])]
    ns, nb, _ = _definition(case)
    if case["kind"] == "solve":
        return [((ns + nb + 1) // 2, (ns + nb) // 2)]
    if nb:
        return [((ns + 1) // 2, ns // 2)]
    if case["kind"] in ("sef", "cpt"):
        return [((ns + 1) // 2, ns // 2)]
    if ns == 2:
        return [(1, 0), (0, 1), (1, 1), (2, 1), (1, 2)]
    h = ns // 2
    return [(h, h - 1), (h - 1, h), (h, h), (h + 1, h), (h, h + 1)]


def _sector_string(case):
    return "/".join("R0:N%d:S%d" % (u + d, u - d) for u, d in _sectors(case))


def _register(case):
    """the cluster model, as a program defines it once"""
    ns, nb, ops = _definition(case)
    L = ns + nb
    name = "case%d" % next(_serial)
    qcm.new_model(name, ns, nb)
    for op, (typ, el) in ops.items():
        if typ == "int":
            qcm.new_operator(name, op, "interaction", [(i + 1, i + L + 1, 1.0) for i in el])
        else:
            s = -1.0 if typ == "stag" else 1.0
            qcm.new_operator(name, op, "one-body", [(r + 1, c + 1, v) for r, c, v in el] +
                             [(r + L + 1, c + L + 1, s * v) for r, c, v in el])
    return name


class _Instance:
    """an instance label that goes when the state goes"""

    def __init__(self, name, values, sectors):
        self.label = 100000 + next(_serial)
        qcm.new_model_instanceC(name, values, sectors, self.label)

    def __del__(self):
        try:
            qcm.erase_model_instance(self.label)
        except Exception:
            pass


def _matsubara(nz, beta=50.0):
    return 1j * (2 * np.arange(nz) + 1) * np.pi / beta


def _superlattices(case, values):
    nx, ny = case["nx"], case["ny"]
    s = np.array([1.0 if (i % nx + i // nx) % 2 == 0 else -1.0 for i in range(nx * ny)])
    return tuple(lattice.square_superlattice(nx, ny, 1.0, weiss=sg * values["M"] * s) for sg in (1.0, -1.0))


def _mlp_data(case, seed):
    """cluster parameters and smooth targets with a little noise, as a corpus has them"""
    rng = np.random.default_rng(seed)
    n_in, n_out, n = case["n_in"], case["n_out"], case["rows"]
    x = rng.uniform(-1.0, 1.0, (n, n_in)) * 2.0 + 1.0
    A = rng.normal(size=(n_in, 24)) / math.sqrt(n_in)
    B = rng.normal(size=(24, n_out)) / math.sqrt(24)
    y = np.tanh(x @ A) @ B * 3.0 - 1.0 + 0.01 * rng.normal(size=(n, n_out))
    dims = [n_in] + [256] * 4 + [n_out]
    w = []
    for i, o in zip(dims[:-1], dims[1:]):
        w.append((rng.normal(size=(o, i)) * math.sqrt(2.0 / i)).reshape(-1))
        w.append(np.zeros(o))
    xp = rng.uniform(-1.0, 1.0, (case["predict"], n_in)) * 2.0 + 1.0
    # master weights are single precision: what the network starts from
    return x, y, np.concatenate(w).astype(np.float32).astype(np.float64), xp, dims


# --------------------------------------------------------------------------
# what a program holds before the call
# --------------------------------------------------------------------------
def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    qcm.set_global_parameterC("Hamiltonian_format", "G")
    st = {"kind": kind}
    if kind == "mlp":
        x, y, w, xp, dims = _mlp_data(case, seed)
        net = surrogate.MLP(case["n_in"], case["n_out"], 256, 4, seed=1)
        net.set_scaling(x.mean(0), x.std(0), y.mean(0), y.std(0), np.ones(case["n_out"]))
        st.update(net=net, x=x, y=y, w=w, xp=xp, epochs=case["epochs"], batch=case["batch"])
        return st
    name = _register(case)
    sectors = _sector_string(case)
    if kind == "hv":
        inst = _Instance(name, _values(case, rng), sectors)
        H = qcm.Hamiltonian(inst.label, sectors, case["format"])
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        x = torch.randn(H.dim, dtype=torch.float64, device="cuda", generator=g)
        x /= torch.linalg.vector_norm(x)
        y = torch.empty_like(x)
        torch.cuda.synchronize()
        st.update(inst=inst, H=H, x=x, y=y)
    elif kind == "solve":
        st.update(name=name, values=_values(case, rng), sectors=sectors, method=case["method"],
                  z=_matsubara(case["nz"]))
    elif kind == "batch":
        st.update(name=name, values=[_values(case, rng, k) for k in range(case["points"])], sectors=sectors,
                  z=np.linspace(-8.0, 8.0, case["nz"]) + 0.1j)
    else:
        v = _values(case, rng)
        inst = _Instance(name, v, sectors)
        qcm.set_global_parameterC("GF_method", "F")
        qcm.ground_state_solve(inst.label)
        qcm.Green_function_solveC(inst.label)
        up, dn = _superlattices(case, v)
        st.update(inst=inst, up=up, dn=dn)
        if kind == "sef":
            st["w"], st["p"] = lattice.legendre_frequency_grid(1.0, 20.0, case["nf"], case["nf"], case["nf"])
            st["kg"] = (2, (case["nk"], case["nk"]), 0.0)
        else:
            st["z"] = np.linspace(-6.0, 6.0, case["nz"]) + 0.1j
            st["kg"] = (2, (case["nk"], case["nk"]), 0.5)
    return st


def run(st):
    kind = st["kind"]
    if kind == "hv":
        st["H"].apply_device(st["x"].data_ptr(), st["y"].data_ptr())
        return st["y"]
    if kind == "solve":
        # the impurity of one iteration: instance, ground state, G on the grid
        qcm.set_global_parameterC("GF_method", st["method"])
        inst = _Instance(st["name"], st["values"], st["sectors"])
        E0, _ = qcm.ground_state_solve(inst.label)
        qcm.Green_function_solveC(inst.label)
        return {"E0": np.array([E0]), "G": qcm.Green_function_grid(st["z"], label=inst.label)}
    if kind == "batch":
        qcm.set_global_parameterC("GF_method", "F")
        insts = [_Instance(st["name"], v, st["sectors"]) for v in st["values"]]
        labels = [i.label for i in insts]
        qcm.solve_batch(labels)
        G = [np.stack(qcm.Green_function_batch(st["z"], labels, spin_down=s)) for s in (0, 1)]
        E0 = np.array([qcm.ground_state_solve(lab)[0] for lab in labels])
        return {"E0": E0, "Gup": G[0], "Gdn": G[1]}
    if kind == "sef":
        integral, per = qcm.SEF_grid(st["w"], st["p"], st["up"], st["kg"], st["dn"], st["inst"].label)
        return {"integral": np.array([integral]), "per_frequency": per}
    if kind == "cpt":
        return qcm.projected_Green_function(st["z"], st["up"], st["kg"], 0, st["inst"].label)
    net = st["net"]
    net.set_optimizer(lr=1e-3)
    net.set_weights(st["w"])
    hist, _ = net.train(st["x"], st["y"], st["epochs"], st["batch"], seed=5)
    return {"history": hist, "weights": net.get_weights(), "predictions": net.predict(st["xp"])}


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------
def _hops(case):
    """mean one-body neighbours of a state per spin, (up, down), for (nup, ndw)"""
    ns, nb, ops = _definition(case)
    L = ns + nb
    n = sum(len(el) for typ, el in ops.values() if typ == "hop" and el and el[0][0] != el[0][1])

    def per(k):
        return 2.0 * n * k * (L - k) / max(1, L * (L - 1))
    return L, per


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        dims = [case["n_in"]] + [256] * 4 + [case["n_out"]]
        mac = sum(i * o for i, o in zip(dims[:-1], dims[1:]))
        back = 2 * mac - dims[0] * dims[1]
        steps = case["epochs"] * (case["rows"] // case["batch"])
        flops = 2.0 * steps * case["batch"] * (mac + back) + 2.0 * case["predict"] * mac
        params = mac + sum(dims[1:])
        # per step: Adam reads and writes weights and both moments; rows once
        byts = steps * params * 4.0 * 6 + 8.0 * (case["rows"] + case["predict"]) * (case["n_in"] + case["n_out"])
        return {"bytes": byts, "flops": flops}
    L, per = _hops(case)
    if kind in ("sef", "cpt"):
        d = case["nx"] * case["ny"]
        nz = 3 * case["nf"] * 2 if kind == "sef" else case["nz"]
        pairs = nz * case["nk"] ** 2
        # V G and the factorization (for cpt the inverse too), complex
        flops = pairs * 8.0 * (d ** 3 + d ** 3 / 3.0 if kind == "sef" else d ** 3 + d ** 3 + d ** 3)
        return {"bytes": 16.0 * nz * d * d * 2, "flops": flops}
    if kind == "hv":
        u, d = case["nup"], case["ndw"]
        dim = math.comb(L, u) * math.comb(L, d)
        return {"bytes": 24.0 * dim, "flops": dim * (2.0 * (per(u) + per(d)) + 1.0)}
    if kind == "solve":
        (u, d), = _sectors(case)
        nz, ns = case["nz"], _definition(case)[0]
        dims = [math.comb(L, u) * math.comb(L, d), math.comb(L, u - 1) * math.comb(L, d),
                math.comb(L, min(u + 1, L)) * math.comb(L, d)]
        # Krylov steps that a ground state and the two parts of G take: each
        # one product (24 bytes a state) and one pass over three vectors
        if case["method"] == "L":
            steps = [min(200, dims[0])] + [min(48 * ns + 12, x) for x in dims[1:]]
        else:
            pairs = ns * (ns + 1) // 2
            steps = [min(60, dims[0])] + [pairs * min(400, x) for x in dims[1:]]
        byts = sum(s * x * (24.0 + 32.0) for s, x in zip(steps, dims))
        flops = sum(s * x * (2.0 * (per(u) + per(d)) + 9.0) for s, x in zip(steps, dims))
        return {"bytes": byts + 16.0 * nz * (1 + ns * ns), "flops": flops}
    # batch: every fraction of every point, max_iter_CF = 400 levels
    ns = case["nx"] * case["ny"]
    pairs = ns * (ns + 1) // 2
    P, nz = case["points"], case["nz"]
    flops = 0.0
    for u, d in _sectors(case):
        dim = math.comb(L, u) * math.comb(L, d)
        flops += P * min(60, dim) * dim * (2.0 * (per(u) + per(d)) + 9.0)
    u, d = _sectors(case)[len(_sectors(case)) // 2]
    for tu, td in ((u - 1, d), (u + 1, d), (u, d - 1), (u, d + 1)):
        if 0 <= tu <= L and 0 <= td <= L:
            dim = math.comb(L, tu) * math.comb(L, td)
            flops += P * pairs * min(400, dim) * dim * (2.0 * (per(tu) + per(td)) + 9.0)
    return {"bytes": 16.0 * P * nz * 2 * ns * ns, "flops": flops}


# --------------------------------------------------------------------------
# tolerances
# --------------------------------------------------------------------------
def tolerance(case):
    """About four times what a change of rounding was measured to do: start
    vectors of other seeds (solve, batch, sef, cpt), weights changed by 1e-7
    (mlp)."""
    kind = case["kind"]
    if kind == "hv":
        # sums of some twenty terms in another order
        return {"rel": 1e-15, "max": 4e-14}
    if kind == "solve":
        # band Lanczos: poles that merge or not; fractions: rounding
        return {"rel": 5e-10, "max": 5e-9} if case["method"] == "L" else {"rel": 1e-12, "max": 4e-11}
    if kind == "batch":
        # 400 Lanczos levels without reorthogonalization, eta = 0.1: rounding
        # grows with the size of the sector
        if case["nb"] == 0:
            return {"rel": 5e-8, "max": 1e-5}
        if case["nx"] * case["ny"] + case["nb"] <= 6:
            return {"rel": 5e-8, "max": 4e-6}
        if case["nx"] * case["ny"] + case["nb"] <= 8:
            return {"rel": 2e-5, "max": 5e-4}
        return {"rel": 6e-4, "max": 3e-2}
    if kind == "sef":
        # the tail's log|det| is near zero and weighted by w^2: against the
        # 64-bit reference the integral is off by 3e-12 to 1e-11
        return {"rel": 4e-11, "max": 4e-10}
    if kind == "cpt":
        return {"rel": 1e-12, "max": 2e-11}
    # bf16 activations and gradients through Adam's normalized steps
    return {"rel": 8e-3, "max": 0.1}


# --------------------------------------------------------------------------
# the same results from the definitions, in 64 bits
# --------------------------------------------------------------------------
def _half_states(L, n):
    return sorted(sum(1 << i for i in c) for c in itertools.combinations(range(L), n))


def _one_body(case, values, spin):
    ns, nb, ops = _definition(case)
    L = ns + nb
    h = np.zeros((L, L))
    for op, (typ, el) in ops.items():
        if typ == "int":
            continue
        s = -1.0 if typ == "stag" and spin else 1.0
        for r, c, v in el:
            h[r, c] += s * v * values[op]
            if r != c:
                h[c, r] += s * v * values[op]
    return h


def _half_matrix(h, L, n):
    """sum_ij h_ij c^dagger_i c_j on the half basis of n particles, dense"""
    st = np.array(_half_states(L, n), dtype=np.int64)
    K = np.zeros((len(st), len(st)))
    cols = np.arange(len(st))
    for i in range(L):
        occ_i = (st >> i) & 1
        K[cols, cols] += h[i, i] * occ_i
        for j in range(L):
            if i == j or h[i, j] == 0.0:
                continue
            ok = np.nonzero((occ_i == 0) & (((st >> j) & 1) == 1))[0]
            s = st[ok]
            new = s ^ (1 << i) ^ (1 << j)
            lo, hi = min(i, j), max(i, j)
            mid = (s >> (lo + 1)) & ((1 << (hi - lo - 1)) - 1)
            par = np.zeros(len(s), dtype=np.int64)
            for b in range(hi - lo - 1):
                par ^= (mid >> b) & 1
            K[np.searchsorted(st, new), ok] += h[i, j] * (1.0 - 2.0 * par)
    return K, st


def _double_occupancy(su, sd, ns):
    mask = (1 << ns) - 1
    both = (sd[:, None] & su[None, :]) & mask
    n = np.zeros(both.shape)
    for b in range(ns):
        n += (both >> b) & 1
    return n


def _dense(case, values, nup, ndw):
    """dense sector Hamiltonian, label i_up + dim_up * i_dn"""
    ns, nb, _ = _definition(case)
    L = ns + nb
    Ku, su = _half_matrix(_one_body(case, values, 0), L, nup)
    Kd, sd = _half_matrix(_one_body(case, values, 1), L, ndw)
    H = np.kron(np.eye(len(sd)), Ku) + np.kron(Kd, np.eye(len(su)))
    H[np.diag_indices_from(H)] += values["U"] * _double_occupancy(su, sd, ns).reshape(-1)
    return H, su, sd


def _remove(i, s_from, s_to, pm):
    """half-basis matrix of c_i (pm -1) or c^dagger_i (pm +1)"""
    pos = {int(v): k for k, v in enumerate(s_to)}
    C = np.zeros((len(s_to), len(s_from)))
    for k, s in enumerate(s_from):
        s = int(s)
        if ((s >> i) & 1) == (1 if pm < 0 else 0):
            sign = -1.0 if bin(s & ((1 << i) - 1)).count("1") & 1 else 1.0
            C[pos[s ^ (1 << i)], k] = sign
    return C


def _ground_states(case, values):
    best = []
    for nup, ndw in _sectors(case):
        H, su, sd = _dense(case, values, nup, ndw)
        w, V = np.linalg.eigh(H)
        best.append((w[0], nup, ndw, V[:, 0], su, sd))
    E0 = min(b[0] for b in best)
    return E0, [b for b in best if b[0] - E0 < 1e-5]


def _lehmann(case, values, states, z, spin):
    """G(z) (nz, ns, ns) of one spin, averaged over the ground states"""
    ns, nb, _ = _definition(case)
    L = ns + nb
    G = np.zeros((len(z), ns, ns), dtype=np.complex128)
    for E, nup, ndw, gs, su, sd in states:
        X = gs.reshape(len(sd), len(su))
        for pm in (-1, 1):
            tu, td = (nup + pm, ndw) if spin == 0 else (nup, ndw + pm)
            if not (0 <= tu <= L and 0 <= td <= L):
                continue
            H, tsu, tsd = _dense(case, values, tu, td)
            w, V = np.linalg.eigh(H)
            A = []
            for i in range(ns):
                if spin == 0:
                    A.append((X @ _remove(i, su, tsu, pm).T).reshape(-1))
                else:
                    A.append((_remove(i, sd, tsd, pm) @ X).reshape(-1))
            Q = V.T @ np.stack(A, 1)
            pole = (w - E) if pm > 0 else (E - w)
            G += np.einsum("zk,ka,kb->zab", 1.0 / (z[:, None] - pole[None, :]), Q, Q, optimize=True) / len(states)
    return G


def _vk(sl, k):
    d = sl["V0"].shape[0]
    V = np.repeat(np.asarray(sl["V0"], dtype=np.complex128)[None], len(k), 0)
    for r, c, n, v in sl["elements"]:
        V[:, r, c] += v * np.exp(2j * np.pi * (k @ np.asarray(sl["R"])[n][:2]))
    return V.reshape(len(k), d, d)


def _exact_mlp(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x, y, w, xp, dims = _mlp_data(case, seed)

    def t(a):
        return torch.tensor(a, dtype=torch.float64, device=dev)
    xm, xs, ym, ys = x.mean(0), x.std(0), y.mean(0), y.std(0)
    p = t(w)
    X, Y, XP = t((x - xm) / xs), t((y - ym) / ys), t((xp - xm) / xs)

    def forward(p, a):
        at = 0
        for l, (i, o) in enumerate(zip(dims[:-1], dims[1:])):
            W, b = p[at:at + i * o].view(o, i), p[at + i * o:at + i * o + o]
            at += i * o + o
            a = a @ W.T + b
            if l < len(dims) - 2:
                a = torch.nn.functional.gelu(a)
        return a
    m, v, hist = torch.zeros_like(p), torch.zeros_like(p), []
    for k in range(1, case["epochs"] + 1):
        q = p.detach().requires_grad_(True)
        loss = ((forward(q, X) - Y) ** 2).sum() / len(x)
        g, = torch.autograd.grad(loss, q)
        hist.append(float(loss.detach()))
        m = 0.9 * m + 0.1 * g
        v = 0.999 * v + 0.001 * g * g
        p = p - 1e-3 * (m / (1 - 0.9 ** k)) / (torch.sqrt(v / (1 - 0.999 ** k)) + 1e-8)
    with torch.no_grad():
        pred = forward(p, XP).cpu().numpy() * ys + ym
    return {"history": np.array(hist), "weights": p.cpu().numpy(), "predictions": pred}


def exact(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind == "mlp":
        return _exact_mlp(case, seed) if case["rows"] == case["batch"] else None
    if kind == "hv":
        v = _values(case, rng)
        ns, nb, _ = _definition(case)
        L = ns + nb
        Ku, su = _half_matrix(_one_body(case, v, 0), L, case["nup"])
        Kd, sd = _half_matrix(_one_body(case, v, 1), L, case["ndw"])
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        x = torch.randn(len(su) * len(sd), dtype=torch.float64, device="cuda", generator=g)
        x /= torch.linalg.vector_norm(x)
        X = x.view(len(sd), len(su))
        tu, td = torch.tensor(su, device="cuda"), torch.tensor(sd, device="cuda")
        both = td[:, None] & tu[None, :] & ((1 << ns) - 1)
        Y = torch.zeros_like(X)
        for b in range(ns):
            Y += (both >> b) & 1
        del both
        Y.mul_(v["U"]).mul_(X)
        Y.addmm_(X, torch.tensor(Ku, device="cuda"))
        Y.addmm_(torch.tensor(Kd, device="cuda"), X)
        return Y.view(-1)
    if kind == "solve":
        v = _values(case, rng)
        (u, d), = _sectors(case)
        L = case["L"]
        if max(math.comb(L, u) * math.comb(L, d), math.comb(L, u + 1) * math.comb(L, d)) > 1300:
            return None
        E0, states = _ground_states(case, v)
        return {"E0": np.array([E0]), "G": _lehmann(case, v, states, _matsubara(case["nz"]), 0)}
    if kind == "batch":
        L = case["nx"] * case["ny"] + case["nb"]
        big = max(math.comb(L, u) * math.comb(L, d) for u, d in _sectors(case))
        if big > 1000 or case["points"] * big ** 3 > 6e8:
            return None
        z = np.linspace(-8.0, 8.0, case["nz"]) + 0.1j
        E, G = [], [[], []]
        for k in range(case["points"]):
            v = _values(case, rng, k)
            E0, states = _ground_states(case, v)
            E.append(E0)
            for s in (0, 1):
                G[s].append(_lehmann(case, v, states, z, s))
        return {"E0": np.array(E), "Gup": np.stack(G[0]), "Gdn": np.stack(G[1])}
    v = _values(case, rng)
    _, states = _ground_states(case, v)
    nk = case["nk"]
    off = 0.0 if kind == "sef" else 0.5
    ax = (np.arange(nk) + off) / nk
    k = np.stack(np.meshgrid(ax, ax, indexing="ij"), -1).reshape(-1, 2)
    sls = _superlattices(case, v)
    if kind == "sef":
        w, p = lattice.legendre_frequency_grid(1.0, 20.0, case["nf"], case["nf"], case["nf"])
        per = np.zeros(len(w))
        eye = np.eye(case["nx"] * case["ny"])
        for s in (0, 1):
            G = _lehmann(case, v, states, 1j * w, s)
            V = _vk(sls[s], k)
            for n in range(len(w)):
                per[n] += np.log(np.abs(np.linalg.det(V @ G[n] - eye))).mean()
        return {"integral": np.array([p @ per]), "per_frequency": per}
    z = np.linspace(-6.0, 6.0, case["nz"]) + 0.1j
    G = _lehmann(case, v, states, z, 0)
    V = _vk(sls[0], k)
    eye = np.eye(case["nx"] * case["ny"])
    out = np.zeros_like(G)
    for n in range(len(z)):
        out[n] = (G[n] @ np.linalg.inv(eye - V @ G[n])).mean(0)
    return np.transpose(out, (0, 2, 1)).copy()
