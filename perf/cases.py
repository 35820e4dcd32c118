"""What a user of the framework has it do, as measurable cases.

Each case is one pass through the package's public entry points on states that stay in
device memory, as a program keeps them: gates, layers, canonical forms, contractions and
the MPO fit, from the smallest bonds to the widest.  A pass starts from a copy of the
prepared state (the entry points work in place), so it can be repeated.

What a pass returns does not depend on the gauge of the tensors (which a factorisation is
free to choose): kept dimensions, Schmidt coefficients, discarded weights, two-site wave
functions, expectation values and overlaps.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qrochet.jl_amd"))

import qrochet_hip as qh  # noqa: E402
from qrochet_hip import mpo as qmpo  # noqa: E402
from qrochet_hip import workloads as wl  # noqa: E402

Z = wl.Z


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # one two-site gate on a small chain, called by itself: the plain method's unit, all latency
        {"name": "gate-small", "kind": "gate", "n": 10, "chi": 12, "precision": "fp64"},
        # the plain method on a small circuit: n = 16, chi = 32, one call per gate, then <Z_i> and the
        # overlap with the initial state
        {"name": "circuit-32", "kind": "circuit", "n": 16, "chi": 32, "layers": 2},
        # Trotter evolution of a product state in Vidal form, a call per layer: bonds grow from 1, ragged and
        # rank-deficient
        {"name": "trotter", "kind": "trotter", "n": 25, "chi": 64, "steps": 3},
        # a brickwork layer of the saturated chain, n = 64, chi = 256: the headline workload's step
        {"name": "layer-256", "kind": "layer", "n": 64, "chi": 256},
        # the same at an odd size in the middle of the range
        {"name": "layer-90", "kind": "layer", "n": 31, "chi": 90},
        # many chains of uneven length and bond dimension, a call per layer, FP32 contraction
        {"name": "uneven-fp32", "kind": "uneven", "count": 16, "nmin": 8, "nmax": 32, "chimax": 128, "layers": 2},
        # Vidal-form update (simple update) of a layer, renormalised
        {"name": "vidal-96", "kind": "vidal", "n": 24, "chi": 96},
        # one update at the widest bond that serving admits: theta is 2048 x 2048
        {"name": "gate-1024", "kind": "gate", "n": 22, "chi": 1024, "precision": "fp64"},
        # Vidal form of a whole chain
        {"name": "canonize-128", "kind": "canonize", "n": 32, "chi": 128},
        # mixed canonical form around a site, normalised (QR sweeps from both ends)
        {"name": "mixed-200", "kind": "mixed", "n": 24, "chi": 200},
        # every <Z_i> and neighbouring <Z_i Z_j> of a saturated chain, its norm and an overlap
        {"name": "measure-256", "kind": "measure", "n": 64, "chi": 256, "chib": 181, "reach": 4},
        # H|psi> compressed back to psi's bonds: one fitting sweep there and back
        {"name": "mpo-fit", "kind": "mpo", "n": 20, "chi": 192, "bond": 8, "precision": "fp64"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gate", "gate", "circuit", "trotter", "layer", "layer", "uneven", "vidal", "canonize", "mixed",
                       "measure", "mpo"])
    if kind == "gate":
        chi = _log(rng, 4, 1024)
        need = 2 * math.ceil(math.log2(chi)) + 2
        return {"kind": kind, "n": need + rng.randint(0, 6), "chi": chi, "precision": rng.choice(["fp64", "fp64", "fp32"])}
    if kind == "circuit":
        return {"kind": kind, "n": rng.randint(6, 20), "chi": _log(rng, 4, 48), "layers": rng.randint(1, 3)}
    if kind == "trotter":
        return {"kind": kind, "n": rng.randint(8, 48), "chi": _log(rng, 16, 128), "steps": rng.randint(1, 3)}
    if kind == "layer":
        return {"kind": kind, "n": rng.randint(12, 64), "chi": _log(rng, 12, 256)}
    if kind == "uneven":
        return {"kind": kind, "count": rng.randint(3, 16), "nmin": 8, "nmax": rng.randint(16, 32),
                "chimax": _log(rng, 24, 128), "layers": rng.randint(1, 2)}
    if kind == "vidal":
        return {"kind": kind, "n": rng.randint(6, 32), "chi": _log(rng, 8, 128)}
    if kind == "canonize":
        return {"kind": kind, "n": rng.randint(6, 40), "chi": _log(rng, 8, 160)}
    if kind == "mixed":
        return {"kind": kind, "n": rng.randint(6, 32), "chi": _log(rng, 8, 256)}
    if kind == "measure":
        return {"kind": kind, "n": rng.randint(8, 64), "chi": _log(rng, 8, 256), "chib": _log(rng, 8, 256),
                "reach": rng.randint(1, 4)}
    return {"kind": "mpo", "n": rng.randint(6, 24), "chi": _log(rng, 16, 224), "bond": rng.randint(2, 8),
            "precision": rng.choice(["fp64", "fp64", "fp32", "bf16x3"])}


# ---------------------------------------------------------------------------
# inputs on the host, from the seed alone
# ---------------------------------------------------------------------------
def _gauss(rng, *shape):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)) / math.sqrt(2.0)


def _isometry(rng, rows, cols):
    """rows x cols with orthonormal columns (rows >= cols)."""
    return np.linalg.qr(_gauss(rng, rows, cols))[0]


def _dims(n, chi):
    return [1] + wl.max_profile(n, 2, chi) + [1]


def _left_chain(rng, n, chi, decay=0.0):
    """A random left-canonical chain of norm 1, arrays (chi_l, 2, chi_r); with `decay`, the weight of its bond
    states falls by that many decades (before the last site is normalised it is no longer canonical)."""
    dims, out = _dims(n, chi), []
    for i in range(n):
        l, r = dims[i], dims[i + 1]
        a = _isometry(rng, 2 * l, r) if 2 * l >= r else _gauss(rng, 2 * l, r) / math.sqrt(2 * l)
        if decay and r > 1:
            a = a * 10.0 ** (-decay * np.arange(r) / r)
        out.append(a.reshape(l, 2, r))
    out[-1] = out[-1] / np.linalg.norm(out[-1])
    return out


def _evolved_chain(rng, n, chi):
    """A chain as a long evolution leaves it before the next layer on bonds 1, 3, 5, ...: every bond has its
    spectrum, falling over eleven decades (five next to the ends), the left site of a bond to be updated has
    orthonormal rows and the right one orthonormal columns (they come from the previous layer's factors)."""
    dims, arrays, lambdas = _dims(n, chi), [], []
    for i in range(n):
        l, r = dims[i], dims[i + 1]
        if i % 2 == 0 and 2 * r >= l:
            a = _isometry(rng, 2 * r, l).T.reshape(l, 2, r)
        elif i % 2 == 1 and 2 * l >= r:
            a = _isometry(rng, 2 * l, r).reshape(l, 2, r)
        else:
            a = _gauss(rng, l, 2, r) / math.sqrt(2 * max(l, r))
        arrays.append(a)
        if r > 1:
            e = np.sort((11.0 if r == chi else 5.0) * rng.random(r))
            lambdas.append(3.0 * 10.0 ** -(e - e[0]))
        elif i < n - 1:
            lambdas.append(np.ones(1))
    return arrays, lambdas


def _vidal_chain(rng, n, chi):
    """Gammas and lambdas of a random state of norm 1 (QR sweep right to left, SVD sweep left to right)."""
    a = _left_chain(rng, n, chi, decay=3.0)
    for i in range(n - 1, 0, -1):
        l, d, r = a[i].shape
        q, t = np.linalg.qr(a[i].reshape(l, d * r).conj().T)
        a[i] = q.conj().T.reshape(-1, d, r)
        a[i - 1] = np.tensordot(a[i - 1], t.conj().T, axes=(2, 0))
    a[0] = a[0] / np.linalg.norm(a[0])
    gammas, lambdas, prev = [], [], np.ones(1)
    m = a[0]
    for i in range(n):
        l, d, r = m.shape
        if i == n - 1:
            gammas.append(m / prev[:, None, None])
            break
        u, s, vh = np.linalg.svd(m.reshape(l * d, r), full_matrices=False)
        gammas.append(u.reshape(l, d, -1) / prev[:, None, None])
        lambdas.append(s)
        m = np.tensordot(s[:, None] * vh, a[i + 1], axes=(1, 0))
        prev = s
    return gammas, lambdas


def _ising(rng, dt=0.05):
    return wl.ising_gate(rng.uniform(0.5, 1.5), rng.uniform(0.5, 1.5), dt)


def _inputs(case, seed):
    """The case's arrays, schedule and operators, as host arrays."""
    rng = np.random.default_rng([seed, len(case["kind"]), ord(case["kind"][0])])
    kind, n, chi = case["kind"], case.get("n"), case.get("chi")
    if kind == "gate":
        b = n // 2
        return {"chain": _left_chain(rng, n, chi), "bond": b, "gate": wl.haar_gate4(rng)}
    if kind == "circuit":
        return {"chain": _left_chain(rng, n, chi),
                "gates": [(b, wl.haar_gate4(rng)) for k in range(case["layers"]) for b in wl.brickwork_bonds(n, k)]}
    if kind == "trotter":
        chain = [v.reshape(1, 2, 1) / np.linalg.norm(v) for v in (_gauss(rng, 2) for _ in range(n))]
        J, h = rng.uniform(0.5, 1.5, n - 1), rng.uniform(0.5, 1.5, n - 1)
        layers = [[(b, wl.ising_gate(J[b - 1], h[b - 1], t)) for b in wl.brickwork_bonds(n, p)]
                  for _ in range(case["steps"]) for p, t in ((0, 0.025), (1, 0.05), (0, 0.025))]
        return {"chain": chain, "layers": layers}
    if kind == "layer":
        chain, lam = _evolved_chain(rng, n, chi)
        return {"chain": chain, "lambdas": lam, "layers": [[(b, _ising(rng)) for b in wl.brickwork_bonds(n, 0)]]}
    if kind == "uneven":
        r2 = np.random.default_rng([case["count"], case["nmax"], case["chimax"]])  # sizes: the case's own
        many = []
        for _ in range(case["count"]):
            m = int(r2.integers(case["nmin"], case["nmax"] + 1))
            x = int(round(math.exp(r2.uniform(math.log(16), math.log(case["chimax"])))))
            many.append({"chi": x, "chain": _left_chain(rng, m, x),
                         "layers": [[(b, wl.haar_gate4(rng)) for b in wl.brickwork_bonds(m, k)]
                                    for k in range(case["layers"])]})
        return {"many": many}
    if kind == "vidal":
        g, lam = _vidal_chain(rng, n, chi)
        return {"chain": g, "lambdas": lam, "layers": [[(b, _ising(rng)) for b in wl.brickwork_bonds(n, 1)]]}
    if kind in ("canonize", "mixed"):
        chain = _left_chain(rng, n, chi, decay=2.0)
        return {"chain": chain, "center": n // 2 + 1}
    if kind == "measure":
        return {"chain": _left_chain(rng, n, chi), "other": _left_chain(rng, n, case["chib"]),
                "pairs": [(i, j) for i in range(1, n + 1) for j in range(i + 1, min(n, i + case["reach"]) + 1)]}
    chain = _left_chain(rng, n, chi)
    return {"chain": chain, "mpo": wl.random_hermitian_mpo(rng, n, 2, case["bond"])}


# ---------------------------------------------------------------------------
# what a program has in hand, and a pass
# ---------------------------------------------------------------------------
def prepare(case, seed):
    x = _inputs(case, seed)
    s = {"case": case, "kind": case["kind"]}
    if "chain" in x:
        s["psi"] = qh.from_internal(x["chain"], lambdas=x.get("lambdas"))
    if "gate" in x:
        s["bond"], s["gate"] = x["bond"], qh.gate(x["gate"], x["bond"], x["bond"] + 1)
    if "gates" in x:
        s["gates"] = [qh.gate(g, b, b + 1) for b, g in x["gates"]]
    if "layers" in x:
        s["layers"] = [[qh.gate(g, b, b + 1) for b, g in layer] for layer in x["layers"]]
    if "many" in x:
        s["many"] = [{"chi": m["chi"], "psi": qh.from_internal(m["chain"]),
                      "layers": [[qh.gate(g, b, b + 1) for b, g in layer] for layer in m["layers"]]} for m in x["many"]]
    if case["kind"] in ("circuit", "trotter"):
        s["terms"] = [[qh.gate(Z, i)] for i in range(1, case["n"] + 1)]
    if "pairs" in x:
        s["other"] = qh.from_internal(x["other"])
        s["terms"] = [[qh.gate(Z, i)] for i in range(1, case["n"] + 1)]
        s["terms"] += [[qh.gate(Z, i), qh.gate(Z, j)] for i, j in x["pairs"]]
    if "center" in x:
        s["center"] = x["center"]
    if "mpo" in x:
        s["mpo"] = qmpo.MPO(x["mpo"])
    return s


def _spectra(psi):
    return np.concatenate([v for v in psi.lambdas() if v is not None])


def _table(lambdas, chi):
    """The spectra as rows of `chi` entries, zeros beyond each bond's own (a threshold decides their lengths)."""
    out = np.zeros((len(lambdas), chi))
    for row, v in zip(out, lambdas):
        if v is not None:
            row[:v.size] = v
    return out


def run(s):
    kind, case = s["kind"], s["case"]
    if kind == "uneven":
        live = [m["psi"].copy() for m in s["many"]]
        kept, disc = [], []
        for k in range(case["layers"]):
            updates = [(psi, g) for psi, m in zip(live, s["many"]) for g in m["layers"][k]]
            caps = [m["chi"] for m in s["many"] for _ in m["layers"][k]]
            a, b = qh.evolve_layer_(updates, maxdim=caps, precision="fp32")
            kept += a
            disc += b
        # the contraction is asked for in single precision, and so is the answer
        return {"kept": np.array(kept), "discarded": np.array(disc, np.float32),
                "schmidt": np.concatenate([_spectra(psi) for psi in live]).astype(np.float32)}
    if kind == "measure":
        return {"values": qh.expect_many(s["psi"], s["terms"]), "norm": qh.norm(s["psi"]),
                "overlap": np.array([qh.overlap(s["psi"], s["other"])])}
    if kind == "mpo":
        phi, ov = qmpo.compress(s["mpo"], s["psi"], sweeps=1, precision=case["precision"])
        out = np.array([ov, qh.overlap(phi, s["psi"])])
        return {"overlaps": out if case["precision"] == "fp64" else out.astype(np.complex64)}
    psi = s["psi"].copy()
    if kind == "gate":
        info, b = {}, s["bond"]
        qh.evolve_(psi, s["gate"], maxdim=case["chi"], precision=case["precision"], info=info)
        lam = psi.lambda_(b)
        out = {"kept": info["kept"], "discarded": np.array([info["discarded"]]), "schmidt": lam}
        if case["chi"] <= 64:  # the updated two-site wave function
            left, right = psi.site_array(b), psi.site_array(b + 1)
            out["theta"] = (left.reshape(-1, left.shape[-1]) * lam) @ right.transpose(1, 0, 2).reshape(lam.size, -1)
        else:
            out["overlap"] = np.array([qh.overlap(psi, s["psi"])])
        if case["precision"] != "fp64":
            out = {k: v if k == "kept" else v.astype(np.complex64 if v.dtype.kind == "c" else np.float32)
                   for k, v in out.items()}
        return out
    if kind == "circuit":
        for g in s["gates"]:
            qh.evolve_(psi, g, maxdim=case["chi"])
        return {"z": qh.expect_many(psi, s["terms"]), "overlap": np.array([qh.overlap(psi, s["psi"])]),
                "bonds": np.array(psi.bond_dims()), "schmidt": _spectra(psi)}
    if kind == "trotter":
        disc = []
        for layer in s["layers"]:
            _, d = qh.evolve_layer_([(psi, g) for g in layer], threshold=1e-7, maxdim=case["chi"], iscanonical=True)
            disc += d
        return {"z": qh.expect_many(psi, s["terms"]), "bonds": np.array(psi.bond_dims()),
                "schmidt": _table(psi.lambdas(), case["chi"]), "discarded": np.array(disc)}
    if kind in ("layer", "vidal"):
        kept, disc = qh.evolve_layer_([(psi, g) for g in s["layers"][0]],
                                      threshold=1e-9 if kind == "vidal" else 1e-12, maxdim=case["chi"],
                                      iscanonical=kind == "vidal", renormalize=kind == "vidal")
        return {"kept": np.array(kept), "discarded": np.array(disc), "schmidt": _table(psi.lambdas(), case["chi"]),
                "overlap": np.array([qh.overlap(psi, s["psi"])])}
    if kind == "canonize":
        qh.canonize_(psi)
        return {"schmidt": _spectra(psi), "overlap": np.array([qh.overlap(psi, s["psi"])])}
    qh.normalize_(psi, s["center"])
    return {"schmidt": psi.lambda_(s["center"] - 1), "overlap": np.array([qh.overlap(psi, s["psi"])])}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _update_work(l, m, r, cap):
    """One two-site update: theta and gate, an R-SVD (Golub and Van Loan's count, times four for complex numbers);
    the two sites read, the kept factors and spectrum written."""
    k = min(2 * l, 2 * r)
    keep = min(k, cap)
    gemm = 32.0 * l * m * r + 128.0 * l * r
    svd = 4.0 * (14.0 * max(2 * l, 2 * r) * k * k + 8.0 * k ** 3)
    return 16.0 * (2 * l * m + 2 * m * r + 16) + 32.0 * keep * (l + r) + 8.0 * keep, gemm + svd


def _sweep_work(da, db):
    """An overlap: both chains read, two products a site."""
    by = fl = 0.0
    for i in range(len(da) - 1):
        by += 32.0 * (da[i] * da[i + 1] + db[i] * db[i + 1])
        fl += 16.0 * db[i] * da[i] * da[i + 1] + 16.0 * db[i] * db[i + 1] * da[i + 1]
    return by, fl


def work(case):
    kind, n, chi = case["kind"], case.get("n"), case.get("chi")
    total = [0.0, 0.0]

    def add(w, times=1.0):
        total[0] += w[0] * times
        total[1] += w[1] * times

    def layer(dims, parity, cap):
        for b in wl.brickwork_bonds(len(dims) - 1, parity):
            add(_update_work(dims[b - 1], dims[b], dims[b + 1], cap))

    if kind == "gate":
        d, b = _dims(n, chi), n // 2
        add(_update_work(d[b - 1], d[b], d[b + 1], chi))
    elif kind == "circuit":
        for k in range(case["layers"]):
            layer(_dims(n, chi), k, chi)
        add(_sweep_work(_dims(n, chi), _dims(n, chi)), 3.0)
    elif kind == "trotter":  # (the bonds that the first layers grow to: at most twofold a layer, then the cap)
        grown = [1] * (n + 1)
        for _ in range(case["steps"]):
            for parity in (0, 1, 0):
                for b in wl.brickwork_bonds(n, parity):
                    add(_update_work(grown[b - 1], grown[b], grown[b + 1], chi))
                    grown[b] = min(chi, 16, 2 * grown[b - 1], 2 * grown[b + 1])
        add(_sweep_work(grown, grown), 2.0)
    elif kind in ("layer", "vidal"):
        layer(_dims(n, chi), 0 if kind == "layer" else 1, chi)
        add(_sweep_work(_dims(n, chi), _dims(n, chi)))
    elif kind == "uneven":
        r2 = np.random.default_rng([case["count"], case["nmax"], case["chimax"]])
        for _ in range(case["count"]):
            m = int(r2.integers(case["nmin"], case["nmax"] + 1))
            x = int(round(math.exp(r2.uniform(math.log(16), math.log(case["chimax"])))))
            for k in range(case["layers"]):
                layer(_dims(m, x), k, x)
    elif kind in ("canonize", "mixed"):
        d = _dims(n, chi)
        for i in range(n):
            l, r = d[i], d[i + 1]
            add((64.0 * l * r, 32.0 * l * r * min(l, r)))  # a QR (R and Q) and a product
            if kind == "canonize":
                add((32.0 * r * r, 4.0 * 22.0 * r ** 3))
        add(_sweep_work(d, d))
    elif kind == "measure":
        d, e = _dims(n, chi), _dims(n, case["chib"])
        add(_sweep_work(d, d), 2.0)
        add((0.0, _sweep_work(d, d)[1]), 1.0 + case["reach"])  # the segments between the operators
        add(_sweep_work(d, e))
    else:
        d, D = _dims(n, chi), [1] + [case["bond"]] * (n - 1) + [1]
        for i in range(n):
            l, r, w, v = d[i], d[i + 1], D[i], D[i + 1]
            step = 16.0 * l * r * r * v + 32.0 * l * r * w * v * 2 + 16.0 * l * l * r * w
            add((32.0 * l * r * 2 + 64.0 * w * v, 5.0 * step + 2 * 32.0 * l * r * min(l, r)))
        add(_sweep_work(d, d))
    return {"bytes": total[0], "flops": total[1]}


# ---------------------------------------------------------------------------
# the same in plain numpy / torch, 64 bits
# ---------------------------------------------------------------------------
def _t(a):
    a = torch.from_numpy(np.ascontiguousarray(a))
    return a.cuda() if torch.cuda.is_available() else a


def _exact_overlap(a, b, la=None, lb=None):
    """sum of a times conj(b); la, lb: the spectra on the bonds."""
    e = _t(np.ones((1, 1), complex))
    for i, (x, y) in enumerate(zip(a, b)):
        x, y = _t(x), _t(y)
        if i and la is not None and la[i - 1] is not None:
            x = _t(la[i - 1])[:, None, None] * x
        if i and lb is not None and lb[i - 1] is not None:
            y = _t(lb[i - 1])[:, None, None] * y
        t = (e @ x.reshape(x.shape[0], -1)).reshape(-1, x.shape[2])
        e = y.reshape(-1, y.shape[2]).conj().T @ t
    return complex(e.cpu()[0, 0])


def _exact_update(a, lam, b, g, threshold, maxdim, vidal=False, renormalize=True):
    """A two-site update of arrays `a` and spectra `lam` in place; kept dimension and discarded weight."""
    i = b - 1
    left, right = a[i], a[i + 1]
    if lam[i] is not None:
        right = lam[i][:, None, None] * right
    out_l = lam[i - 1] if vidal and i > 0 else None
    out_r = lam[i + 1] if vidal and i + 1 < len(lam) else None
    t = np.tensordot(left, right, axes=(2, 0))  # l o1 o2 r
    t = np.einsum("abxy,lxyr->labr", g, t)
    if out_l is not None:
        t = out_l[:, None, None, None] * t
    if out_r is not None:
        t = t * out_r
    l, _, _, r = t.shape
    u, s, vh = np.linalg.svd(t.reshape(2 * l, 2 * r), full_matrices=False)
    k = int(np.sum(s[:maxdim] > threshold))
    disc = math.sqrt(float(np.sum(s[k:] ** 2)))
    u, vh, s = u[:, :k].reshape(l, 2, k), vh[:k].reshape(k, 2, r), s[:k]
    if vidal:
        u = u / out_l[:, None, None] if out_l is not None else u
        vh = vh / out_r if out_r is not None else vh
        s = s / np.linalg.norm(s) if renormalize else s
    a[i], a[i + 1], lam[i] = u, vh, s
    return k, disc


def _exact_values(a, lam, terms):
    """<Z ... Z> of the chain for each tuple of sites in `terms` (unnormalised)."""
    n = len(a)
    z = _t(np.array([1.0, -1.0]))[None, :, None]
    x = [_t(v if i == 0 or lam is None or lam[i - 1] is None else lam[i - 1][:, None, None] * v)
         for i, v in enumerate(a)]
    one = _t(np.ones((1, 1), complex))

    def step(e, i, op):
        t = (e @ x[i].reshape(x[i].shape[0], -1)).reshape(-1, 2, x[i].shape[2])
        t = z * t if op else t
        return x[i].reshape(-1, x[i].shape[2]).conj().T @ t.reshape(-1, t.shape[2])

    left, right = [one], [one]
    for i in range(n):
        left.append(step(left[-1], i, False))
    for i in range(n - 1, -1, -1):  # right[k]: from the end, on bond n - k; rows bra, columns ket
        t = (x[i].reshape(-1, x[i].shape[2]) @ right[-1].T).reshape(x[i].shape[0], -1)
        right.append(x[i].reshape(x[i].shape[0], -1).conj() @ t.T)
    out = []
    for sites in terms:
        e = left[sites[0] - 1]
        for i in range(sites[0] - 1, sites[-1]):
            e = step(e, i, i + 1 in sites)
        out.append((e * right[n - sites[-1]]).sum())
    return torch.stack(out).cpu().numpy()


def _exact_fit(psi, mpo, sweeps=1):
    """One-site variational fit of H|psi>, started from psi: <phi|H psi> and <phi|psi>."""
    n = len(psi)
    A = [_t(a) for a in psi]
    W = []  # (w, o, i, v)
    for k, m in enumerate(mpo):
        m = m[:, :, None] if k == 0 else m
        m = m[..., None] if k == n - 1 else m
        W.append(_t(np.transpose(m, (2, 0, 1, 3))))

    def qr(m):  # (on the host: the factorisation there is LAPACK's)
        q, r = np.linalg.qr(m.cpu().numpy())
        return _t(q), _t(r)

    B = list(A)
    for i in range(n - 1, 0, -1):
        l, d, r = B[i].shape
        q, t = qr(B[i].reshape(l, d * r).conj().T)
        B[i] = q.conj().T.reshape(-1, d, r)
        B[i - 1] = torch.tensordot(B[i - 1], t.conj().T, dims=([2], [0]))
    one = _t(np.ones((1, 1, 1), complex))
    L, R = [one] + [None] * n, [None] * n + [one]

    def with_right(i):  # (b, o, w, x): psi and H contracted with R[i + 1] (c, x, v)
        t = torch.tensordot(A[i], R[i + 1], dims=([2], [0]))  # b i x v
        return torch.tensordot(t, W[i], dims=([1, 3], [2, 3])).permute(0, 3, 2, 1)

    def right(i):
        t = torch.tensordot(with_right(i), B[i].conj(), dims=([1, 3], [1, 2]))  # b w a
        R[i] = t.permute(0, 2, 1)

    def left(i):
        t = torch.tensordot(L[i], A[i], dims=([0], [0]))  # a w i c
        t = torch.tensordot(t, W[i], dims=([1, 2], [0, 2]))  # a c o v
        L[i + 1] = torch.tensordot(t, B[i].conj(), dims=([0, 2], [0, 1])).permute(0, 2, 1)  # c x v

    def local(i):  # (a, o, x)
        return torch.tensordot(L[i], with_right(i), dims=([0, 2], [0, 2]))

    for i in range(n - 1, 0, -1):
        right(i)
    for _ in range(sweeps):
        for i in range(n - 1):
            m = local(i)
            B[i] = qr(m.reshape(-1, m.shape[2]))[0].reshape(m.shape[0], 2, -1)
            left(i)
        for i in range(n - 1, 0, -1):
            m = local(i)
            B[i] = qr(m.reshape(m.shape[0], -1).conj().T)[0].conj().T.reshape(-1, 2, m.shape[2])
            right(i)
        B[0] = local(0)
    phi = [b.cpu().numpy() for b in B]
    return complex((B[0].abs() ** 2).sum().cpu()), _exact_overlap(phi, psi)


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "uneven":
        disc, spectra = [], []
        many = [(list(m["chain"]), [None] * (len(m["chain"]) - 1), m) for m in x["many"]]
        for k in range(case["layers"]):
            for a, lam, m in many:
                disc += [_exact_update(a, lam, b, g, 1e-16, m["chi"])[1] for b, g in m["layers"][k]]
        for _, lam, _ in many:
            spectra += [v for v in lam if v is not None]
        return {"kept": None, "discarded": np.array(disc, np.float64), "schmidt": np.concatenate(spectra)}
    a = list(x["chain"])
    lam = list(x["lambdas"]) if "lambdas" in x else [None] * (len(a) - 1)
    start, start_lam = list(a), list(lam)
    n = len(a)
    if kind == "gate":
        b = x["bond"]
        _, disc = _exact_update(a, lam, b, x["gate"], 1e-16, case["chi"])
        out = {"kept": None, "discarded": np.array([disc]), "schmidt": lam[b - 1]}
        if case["chi"] <= 64:
            u, v = a[b - 1].transpose(1, 0, 2), a[b]
            out["theta"] = (u.reshape(-1, u.shape[2]) * lam[b - 1]) @ v.reshape(v.shape[0], -1)
        else:
            out["overlap"] = np.array([_exact_overlap(a, start, lam, start_lam)])
        return out
    if kind == "circuit":
        for b, g in x["gates"]:
            _exact_update(a, lam, b, g, 1e-16, case["chi"])
        return {"z": _exact_values(a, lam, [(i,) for i in range(1, n + 1)]), "bonds": None,
                "overlap": np.array([_exact_overlap(a, start, lam, start_lam)]),
                "schmidt": np.concatenate([v for v in lam if v is not None])}
    if kind == "trotter":
        disc = [_exact_update(a, lam, b, g, 1e-7, case["chi"], vidal=True, renormalize=False)[1]
                for layer in x["layers"] for b, g in layer]
        return {"z": _exact_values(a, lam, [(i,) for i in range(1, n + 1)]), "bonds": None,
                "schmidt": _table(lam, case["chi"]), "discarded": np.array(disc)}
    if kind in ("layer", "vidal"):
        vidal = kind == "vidal"
        disc = [_exact_update(a, lam, b, g, 1e-9 if vidal else 1e-12, case["chi"], vidal=vidal)[1]
                for b, g in x["layers"][0]]
        return {"discarded": np.array(disc), "kept": None, "schmidt": _table(lam, case["chi"]),
                "overlap": np.array([_exact_overlap(a, start, lam, start_lam)])}
    if kind == "measure":
        terms = [(i,) for i in range(1, n + 1)] + x["pairs"]
        return {"values": _exact_values(a, None, terms), "norm": math.sqrt(abs(_exact_overlap(a, a))),
                "overlap": np.array([_exact_overlap(a, x["other"])])}
    if kind == "mpo":
        return {"overlaps": np.array(_exact_fit(a, x["mpo"]))}
    # canonize, mixed: the Schmidt coefficients of the state
    for i in range(n - 1, 0, -1):
        l, d, r = a[i].shape
        q, t = np.linalg.qr(a[i].reshape(l, d * r).conj().T)
        a[i] = q.conj().T.reshape(-1, d, r)
        a[i - 1] = np.tensordot(a[i - 1], t.conj().T, axes=(2, 0))
    spectra, m = [], a[0]
    for i in range(n - 1):
        l, d, r = m.shape
        q, t = np.linalg.qr(m.reshape(l * d, r))
        spectra.append(np.linalg.svd(t, compute_uv=False))
        m = np.tensordot(t, a[i + 1], axes=(1, 0))
    square = _exact_overlap(start, start)
    if kind == "canonize":
        return {"schmidt": np.concatenate(spectra), "overlap": np.array([square])}
    s = spectra[x["center"] - 2]
    return {"schmidt": s / np.linalg.norm(s), "overlap": np.array([math.sqrt(abs(square)) + 0j])}
