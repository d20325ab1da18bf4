"""Performance cases of the RI-V J/K framework: what a user has it do, one pass at a time.

Kinds (each a call that a program of this framework makes in a loop):

  host    J and occupied-route K from host arrays, REST's vj/vk builders as a drop-in
  host_dm J and density-only K from host arrays, REST's RI-HF default with packed B
  jk      J and K on device pointers, the step of a device-resident SCF, at each precision and spin
  batch   J and K of many clusters in one grouped run, inputs and outputs on the host (batched SCF)
  build   the packed B = (mn|P) V^-1/2 of a molecule into device memory
  scf     a whole FP64 RI-HF from the SAD guess orbitals
  net     loss and gradients of the learned guess's network on one training batch

Sizes are (nbf, naux, nocc); water clusters in def2-SVP / def2-SVP-JKFIT have (24, 113, 5) a water.
B is uniform noise of variance 1/naux (the framework's synthetic fill), orbitals are orthonormal,
densities are occupation-weighted C C^T.
"""
import math

import numpy as np
import torch

from rest_amd import jk, learned, ri, scf, workload

PREC = {"fp64": jk.PREC_FP64, "fp32": jk.PREC_FP32, "bf16x2": jk.PREC_BF16X2, "bf16x3": jk.PREC_BF16X3}
DEV = "cuda"


def listed():
    return [
        # one water: the smallest molecule of the benchmark, every call is launches and copies
        {"name": "host_fp64_water1", "kind": "host", "nbf": 24, "naux": 113, "nocc": 5},
        # eight waters by the density-only K, as REST's RI-HF calls it with use_ri_symm
        {"name": "host_dm_fp64_water8", "kind": "host_dm", "nbf": 192, "naux": 904, "nocc": 40},
        # (H2O)16, the middle benchmark shape, one FP64 SCF step
        {"name": "jk_fp64_water16", "kind": "jk", "prec": "fp64", "spin": 1, "nbf": 384, "naux": 1808, "nocc": 80,
         "nocc_b": 0},
        # (H2O)64, the headline shape, one FP64 SCF step
        {"name": "jk_fp64_water64", "kind": "jk", "prec": "fp64", "spin": 1, "nbf": 1536, "naux": 7232, "nocc": 320,
         "nocc_b": 0},
        # an open-shell molecule: two spins, no size a multiple of a tile
        {"name": "jk_fp64_uhf_odd", "kind": "jk", "prec": "fp64", "spin": 2, "nbf": 333, "naux": 1571, "nocc": 71,
         "nocc_b": 67},
        # the FP32 rung of the precision ladder, 24 waters
        {"name": "jk_fp32_water24", "kind": "jk", "prec": "fp32", "spin": 1, "nbf": 576, "naux": 2712, "nocc": 120,
         "nocc_b": 0},
        # the first rung of the mixed ladder (two BF16 planes), 32 waters
        {"name": "jk_bf16x2_water32", "kind": "jk", "prec": "bf16x2", "spin": 1, "nbf": 768, "naux": 3616,
         "nocc": 160, "nocc_b": 0},
        # its second rung (three planes) at a size between tiles
        {"name": "jk_bf16x3_odd", "kind": "jk", "prec": "bf16x3", "spin": 1, "nbf": 645, "naux": 3037, "nocc": 133,
         "nocc_b": 0},
        # one iteration of the batched driver over uneven small clusters
        {"name": "batch_bf16x3_24", "kind": "batch", "prec": "bf16x3", "count": 24, "lo": 2, "hi": 16, "base": 24301},
        # the B producer for twelve waters
        {"name": "build_water12", "kind": "build", "waters": 12},
        # a whole SCF of eight waters
        {"name": "scf_fp64_water8", "kind": "scf", "waters": 8},
        # one training step's loss and gradients at the trainer's batch
        {"name": "net_grad_4096", "kind": "net", "batch": 4096},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sizes(rng, lo, hi):
    """A molecule's sizes: auxiliary functions 3.5 to 4.8 an orbital function, 15 to 28 % occupied."""
    nbf = _log(rng, lo, hi)
    return {"nbf": nbf, "naux": int(nbf * rng.uniform(3.5, 4.8)), "nocc": max(1, int(nbf * rng.uniform(0.15, 0.28)))}


def draw(rng):
    kind = rng.choice(["host", "host_dm", "jk", "jk", "jk", "jk", "batch", "build", "scf", "net"])
    if kind == "host":
        return {"kind": kind, **_sizes(rng, 20, 400)}
    if kind == "host_dm":
        return {"kind": kind, **_sizes(rng, 20, 400)}
    if kind == "jk":
        prec = rng.choice(["fp64", "fp64", "fp32", "bf16x2", "bf16x3"])
        spin = rng.choice([1, 1, 2])
        c = {"kind": kind, "prec": prec, "spin": spin, **_sizes(rng, 40, 1100 if prec == "fp64" else 900)}
        c["nocc_b"] = max(1, c["nocc"] - rng.randrange(0, 4)) if spin == 2 else 0
        return c
    if kind == "batch":
        lo = rng.randrange(1, 6)
        return {"kind": kind, "prec": rng.choice(["fp64", "fp32", "bf16x2", "bf16x3"]), "count": rng.randrange(2, 25),
                "lo": lo, "hi": lo + rng.randrange(1, 12), "base": rng.randrange(1 << 20)}
    if kind == "net":
        return {"kind": kind, "batch": _log(rng, 64, 8192)}
    return {"kind": kind, "waters": _log(rng, 1, 14)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _orbitals(seed, nbf, spin):
    """[spin][state][nbf] orthonormal orbitals (column-major eigenvectors, one a row)."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    out = []
    for _ in range(spin):
        a = torch.randn((nbf, nbf), generator=g, dtype=torch.float64, device=DEV)
        out.append(torch.linalg.qr(a)[0])
    return torch.stack(out)


def _occupations(case):
    spin = case.get("spin", 1)
    nw = [case["nocc"], case.get("nocc_b", 0)][:spin]
    occ = torch.zeros((spin, case["nbf"]), dtype=torch.float64, device=DEV)
    for s in range(spin):
        occ[s, :nw[s]] = 2.0 if spin == 1 else 1.0
    return nw, occ


def _density(c, occ):
    return torch.stack([(ci.T * oi) @ ci for ci, oi in zip(c, occ)])


def _clusters(case, seed):
    """Sizes of the batch's clusters, and their orbitals and densities on the host."""
    ns = workload.batched_cluster_sizes(case["count"], case["base"], case["lo"], case["hi"])
    out = []
    for i, n in enumerate(ns):
        c = _orbitals(seed * 1000 + i, 24 * n, 1)[0, :5 * n]
        out.append((n, (2.0 * (c.T @ c)).cpu().numpy(), np.ascontiguousarray(c.T.cpu().numpy()), np.full(5 * n, 2.0)))
    return out


def _molecule(case, seed):
    return ri.Molecule.water_cluster(workload.water_cluster(seed, case["waters"]))


def _net_data(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    b = case["batch"]
    x = torch.randn((b, learned.N_IN), generator=g, dtype=torch.float32, device=DEV)
    t = torch.randn((b, learned.N_OUT), generator=g, dtype=torch.float32, device=DEV)
    m = (torch.rand((b, learned.N_OUT), generator=g, device=DEV) < 0.6).float()
    return x, t, m


def prepare(case, seed):
    from rest_amd import guess
    kind = case["kind"]
    if kind in ("host", "host_dm", "jk"):
        r = jk.DeviceRI(case["nbf"], case["naux"])
        prec = case.get("prec", "fp64")
        store = jk.STORE_FP64 | (jk.STORE_FP32 if prec != "fp64" else 0) \
            | (jk.STORE_BF16 if prec.startswith("bf16") else 0)
        r.fill_synthetic(seed, store)
        c = _orbitals(seed, case["nbf"], case.get("spin", 1))
        nw, occ = _occupations(case)
        d = _density(c, occ)
        s = {"kind": kind, "ri": r, "spin": case.get("spin", 1), "homo": [n - 1 for n in nw], "prec": PREC[prec]}
        if kind == "jk":
            # J of the total density, as a Fock matrix takes it; K for each spin
            dt = d.sum(0).contiguous()
            s.update(c=c, occ=occ, d=dt, vj=torch.empty(r.npair, dtype=torch.float64, device=DEV),
                     vk=torch.empty((s["spin"], r.npair), dtype=torch.float64, device=DEV))
        else:
            s.update(c=c[0].T.cpu().numpy(), occ=occ[0].cpu().numpy(), d=d[0].cpu().numpy())
        return s
    if kind == "batch":
        cl = _clusters(case, seed)
        b = jk.Batch([24 * n for n, *_ in cl], [113 * n for n, *_ in cl], [5 * n for n, *_ in cl], PREC[case["prec"]])
        b.fill_synthetic(seed)
        return {"kind": kind, "batch": b, "inputs": [x[1:] for x in cl]}
    if kind == "build":
        mol = _molecule(case, seed)
        r = jk.DeviceRI(mol.nbf, mol.naux)
        return {"kind": kind, "mol": mol, "ri": r, "b": torch.empty((r.naux, r.ldb), dtype=torch.float64, device=DEV)}
    if kind == "scf":
        mol = _molecule(case, seed)
        S, T, V = mol.int1e()
        r = jk.DeviceRI(mol.nbf, mol.naux)
        mol.build_rimatr(r)
        g = guess.sad_guess(mol, r, S, T + V)
        return {"kind": kind, "ri": r, "S": S, "H": T + V, "enuc": mol.nuclear_repulsion(), "nel": mol.nelectron,
                "c": g.c1}
    x, t, m = _net_data(case, seed)
    return {"kind": kind, "net": learned.Net(max_batch=max(8192, case["batch"]), seed=seed), "x": x, "t": t, "m": m}


def run(s):
    kind = s["kind"]
    if kind == "host":
        vj = jk.vj_upper_with_rimatr_v_sync(s["ri"], [s["d"]], 1, 1.0)[0]
        vk = jk.vk_upper_with_ri_v_sync(s["ri"], [s["c"]], s["homo"], [s["occ"]], 1, -0.5)[0]
        return {"j": vj, "k": vk}
    if kind == "host_dm":
        vj = jk.vj_upper_with_rimatr_v_sync(s["ri"], [s["d"]], 1, 1.0)[0]
        vk = jk.vk_upper_with_rimatr_use_dm_only_sync(s["ri"], [s["d"]], 1, -0.5)[0]
        return {"j": vj, "k": vk}
    if kind == "jk":
        r = s["ri"]
        r.vj_dev(s["d"].data_ptr(), 1, 1.0, s["vj"].data_ptr(), s["prec"])
        r.vk_occ_dev(s["c"].data_ptr(), r.nbf, s["homo"], s["occ"].data_ptr(), s["spin"],
                     -0.5 if s["spin"] == 1 else -1.0, s["vk"].data_ptr(), s["prec"])
        return {"j": s["vj"], "k": s["vk"]}
    if kind == "batch":
        b = s["batch"]
        for i, (d, c, occ) in enumerate(s["inputs"]):
            b.set_inputs(i, d, c, occ)
        b.run(1.0, -0.5)
        b.synchronize()
        return [b.get_outputs(i) for i in range(len(s["inputs"]))]
    if kind == "build":
        r = s["ri"]
        s["mol"].build_rimatr(r)
        r.copy_dev(s["b"].data_ptr(), r.rimatr_dev_ptr(), 8 * r.naux * r.ldb)
        return s["b"][:, :r.npair]
    if kind == "scf":
        o = scf.rhf(s["ri"], s["S"], s["H"], s["enuc"], s["nel"], c_guess=s["c"])
        return {"energy": np.array([o.energy]), "iterations": o.iterations, "orbital_energies": o.mo_energy,
                "density": o.dm}
    loss, grad = s["net"].loss_grad_dev(s["x"], s["t"], s["m"], want_grad=True)
    return {"loss": loss, "grad": grad}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _jk_work(nbf, naux, nocc, size, spin=1):
    pairs = nbf * (nbf + 1) // 2
    flops = 4 * pairs * naux + (2 * nbf * nbf + nbf * (nbf + 1)) * nocc * naux
    return {"bytes": size * pairs * naux + 8 * (nbf * nbf + nbf * nocc + (1 + spin) * pairs), "flops": flops}


def work(case):
    kind = case["kind"]
    size = 8 if case.get("prec", "fp64") == "fp64" else 4
    if kind in ("host", "host_dm", "jk"):
        return _jk_work(case["nbf"], case["naux"], case["nocc"] + case.get("nocc_b", 0), size, case.get("spin", 1))
    if kind == "batch":
        ns = workload.batched_cluster_sizes(case["count"], case["base"], case["lo"], case["hi"])
        ws = [_jk_work(24 * n, 113 * n, 5 * n, size) for n in ns]
        return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}
    if kind == "net":
        dims = [learned.N_IN, 256, 256, 256, learned.N_OUT]
        p = sum(a * b + b for a, b in zip(dims[:-1], dims[1:]))
        mults = sum(a * b for a, b in zip(dims[:-1], dims[1:]))
        return {"bytes": 4 * (case["batch"] * (dims[0] + 2 * dims[-1]) + 2 * p),
                "flops": 2 * case["batch"] * (3 * mults - dims[0] * dims[1])}
    n = case["waters"]
    nbf, naux, pairs = 24 * n, 113 * n, 24 * n * (24 * n + 1) // 2
    if kind == "build":
        # the product with V^-1/2 and its eigenproblem (9 n^3), B written once
        return {"bytes": 8 * (pairs * naux + naux * naux), "flops": 2 * pairs * naux * naux + 9 * naux ** 3}
    # about ten iterations of J, K, the eigenproblem and the error vector's products
    w = _jk_work(nbf, naux, 5 * n, 8)
    return {"bytes": 10 * w["bytes"], "flops": 10 * (w["flops"] + 9 * nbf ** 3 + 10 * nbf ** 3)}


# ---------------------------------------------------------------------------
# the same in 64 bits, by plain torch
# ---------------------------------------------------------------------------
def _synthetic(seed, pairs, naux, p0, p1):
    """Columns [p0, p1) of the synthetic B: (2u - 1) sqrt(3 / naux), u the top 53 bits of splitmix64."""
    def wrap(v):
        v &= (1 << 64) - 1
        return v - (1 << 64) if v >> 63 else v

    def shr(z, k):
        return (z >> k) & ((1 << (64 - k)) - 1)
    z = torch.arange(p0 * pairs + 1, p1 * pairs + 1, dtype=torch.int64, device=DEV)
    z = z * wrap(0x9E3779B97F4A7C15) + wrap(seed)
    z = (z ^ shr(z, 30)) * wrap(0xBF58476D1CE4E5B9)
    z = (z ^ shr(z, 27)) * wrap(0x94D049BB133111EB)
    z = z ^ shr(z, 31)
    u = shr(z, 11).double() * 2.0 ** -53
    return ((2.0 * u - 1.0) * math.sqrt(3.0 / naux)).view(p1 - p0, pairs)


def _exact_jk(seed, nbf, naux, d, cols, weights, k_scale):
    """J of d, and for each spin K = k_scale * sum_P (B_P C) diag(w) (B_P C)^T, packed upper."""
    pairs = nbf * (nbf + 1) // 2
    tri = torch.tril_indices(nbf, nbf, device=DEV)       # row >= col: p = row(row+1)/2 + col
    j = torch.zeros(pairs, dtype=torch.float64, device=DEV)
    k = [torch.zeros((nbf, nbf), dtype=torch.float64, device=DEV) for _ in cols]
    w = d[tri[0], tri[1]] * torch.where(tri[0] == tri[1], 1.0, 2.0)
    step = max(1, (1 << 28) // (nbf * nbf))
    for p0 in range(0, naux, step):
        p1 = min(naux, p0 + step)
        b = _synthetic(seed, pairs, naux, p0, p1)
        j += (b @ w) @ b
        full = torch.zeros((p1 - p0, nbf, nbf), dtype=torch.float64, device=DEV)
        full[:, tri[0], tri[1]] = b
        full[:, tri[1], tri[0]] = b
        for s, (c, o) in enumerate(zip(cols, weights)):
            m = (full.view(-1, nbf) @ c).view(p1 - p0, nbf, -1).transpose(0, 1).reshape(nbf, -1)
            k[s] += (m * o.repeat(p1 - p0)) @ m.T
        del full, b
    return j, [k_scale * x[tri[0], tri[1]] for x in k]


def _exact_net(case, seed):
    net = learned.Net(max_batch=64, seed=seed)
    dims, p = net.dims, torch.from_numpy(net.init_params(seed)).double().to(DEV).requires_grad_(True)
    x, t, m = (v.double() for v in _net_data(case, seed))
    off = 0
    for n, (a, b) in enumerate(zip(dims[:-1], dims[1:])):
        x = x @ p[off:off + a * b].view(a, b) + p[off + a * b:off + a * b + b]
        off += a * b + b
        if n + 2 < len(dims):
            x = x * torch.sigmoid(x)
    loss = (m * (x - t) ** 2).sum() / m.sum()
    loss.backward()
    return {"loss": loss.item(), "grad": p.grad}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("host", "host_dm", "jk"):
        spin = case.get("spin", 1)
        c = _orbitals(seed, case["nbf"], spin)
        nw, occ = _occupations(case)
        j, k = _exact_jk(seed, case["nbf"], case["naux"], _density(c, occ).sum(0), [c[s, :nw[s]].T for s in range(spin)],
                         [occ[s, :nw[s]] for s in range(spin)], -0.5 if spin == 1 else -1.0)
        return {"j": j, "k": torch.stack(k) if kind == "jk" else k[0]}
    if kind == "batch":
        out = []
        for i, (n, d, c, occ) in enumerate(_clusters(case, seed)):
            j, k = _exact_jk(seed + i, 24 * n, 113 * n, torch.from_numpy(d).to(DEV), [torch.from_numpy(c).to(DEV)],
                             [torch.from_numpy(occ).to(DEV)], -0.5)
            out.append((j, k[0]))
        return out
    if kind == "net":
        return _exact_net(case, seed)
    return None
