"""The work a user of this library has it do, as measurable cases.

A case is a dict of plain values; `kind` names the public entry point:

  solve  trlan() / ztrlan() on one device operator (solve_csr): plain FP64,
         mixed precision or complex, on the operators of
         nutrlan_amd/workloads.py with the solver parameters the benchmark
         and the tests use for them
  batch  trlan_batch() on many 2D lattices at once (solve_batch), from host
         start vectors or from the learned-start net's device outputs
  pass   one allocation-free classical Gram-Schmidt pass over caller device
         memory (trlhip_cgs_pass_noalloc), FP64, FP32 shadow or complex
  infer  learned start vectors for a set of lattices (start_vectors)
  train  loss and parameter gradients of the net on a batch of images
         (Net.loss_grad: forward and backward)

Eigenvectors and eigenvalues come back whole in the caller's buffers, the
pass's updated vector in the caller's device memory, gradients as one
vector.
"""
import ctypes

import numpy as np
import torch

from nutrlan_amd import learned as LN
from nutrlan_amd import trlan as T
from nutrlan_amd import workloads as W

TOL = 1e-8
MAXMV = 100000
# end of the spectrum, pairs, basis size: the benchmark's and the tests' own
# parameters for each operator family
SOLVER = {
    "diag": (1, 5, 40),
    "lattice2d": (-1, 8, 32),
    "laplace3d": (1, 16, 64),
    "anderson3d": (-1, 24, 80),
    "random": (1, 32, 128),
}
TILE = {"r64": (T.TRLHIP_R64, torch.float64), "r32": (T.TRLHIP_R32, torch.float32),
        "c128": (T.TRLHIP_C128, torch.complex128)}


def listed():
    return [
        # the smallest call: a quick solve whose time is launches and round trips
        {"name": "diag_1000", "kind": "solve", "op": "diag", "size": 1000, "path": "fp64"},
        # the drop-in trlan() call on one lattice
        {"name": "lattice_100", "kind": "solve", "op": "lattice2d", "size": 100, "W": 6.0, "path": "fp64"},
        # the same in mixed precision, an odd side: refinement at the end
        {"name": "lattice_181_mixed", "kind": "solve", "op": "lattice2d", "size": 181, "W": 4.0,
         "path": "mixed"},
        # the largest single solve: the 128^3 periodic Laplacian
        {"name": "laplace_128_mixed", "kind": "solve", "op": "laplace3d", "size": 128, "path": "mixed"},
        # ztrlan(): a Hermitian lattice with magnetic phases
        {"name": "anderson_48_complex", "kind": "solve", "op": "anderson3d", "size": 48, "path": "complex"},
        # rows of uneven length that gather from everywhere, many pairs, a wide basis
        {"name": "random_50001", "kind": "solve", "op": "random", "size": 50001, "path": "fp64"},
        # disorder averages: many lattices of mixed sizes, learned start vectors
        {"name": "batch_192_learned", "kind": "batch", "jobs": 192, "lo": 64, "hi": 256, "path": "mixed",
         "learned": True},
        # a smaller batch in plain FP64 from random starts
        {"name": "batch_40_fp64", "kind": "batch", "jobs": 40, "lo": 48, "hi": 160, "path": "fp64",
         "learned": False},
        # the start vectors of a batch alone, host to host
        {"name": "start_vectors_256", "kind": "infer", "images": 256, "lo": 64, "hi": 256},
        # one training batch of the net: forward and backward
        {"name": "train_64x64", "kind": "train", "images": 64, "size": 64},
        # a caller's own Gram-Schmidt pass, large and FP64
        {"name": "pass_fp64_large", "kind": "pass", "dtype": "r64", "n": 2097152, "m": 64},
        # and a small ragged one against an FP32 basis
        {"name": "pass_fp32_ragged", "kind": "pass", "dtype": "r32", "n": 28561, "m": 23},
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "solve", "batch", "batch", "pass", "pass", "infer", "train"])
    if kind == "solve":
        op = rng.choice(["diag", "lattice2d", "lattice2d", "laplace3d", "anderson3d", "random"])
        c = {"kind": kind, "op": op, "path": rng.choice(["fp64", "mixed"])}
        if op == "diag":
            c["size"], c["path"] = _log_int(rng, 500, 4000), "fp64"
        elif op == "lattice2d":
            c["size"], c["W"] = _log_int(rng, 40, 256), round(rng.uniform(1.0, 12.0), 2)
        elif op == "laplace3d":
            c["size"] = _log_int(rng, 12, 120)
        elif op == "anderson3d":
            c["size"], c["path"] = _log_int(rng, 12, 64), "complex"
        else:
            c["size"] = _log_int(rng, 3000, 200000)
        return c
    if kind == "batch":
        lo = rng.randint(40, 120)
        learned = rng.random() < 0.5
        return {"kind": kind, "jobs": _log_int(rng, 8, 192), "lo": lo, "hi": lo + rng.randint(10, 130),
                "path": "mixed" if learned else rng.choice(["fp64", "mixed"]), "learned": learned}
    if kind == "pass":
        dtype = rng.choice(["r64", "r32", "c128"])
        return {"kind": kind, "dtype": dtype, "n": _log_int(rng, 4000, 1048576 if dtype == "c128" else 2097152),
                "m": rng.randint(2, 96)}
    if kind == "infer":
        lo = rng.randint(32, 120)
        return {"kind": kind, "images": _log_int(rng, 4, 400), "lo": lo, "hi": lo + rng.randint(10, 136)}
    size = rng.randint(32, 200)
    return {"kind": kind, "images": max(1, int(_log_int(rng, 16384, 262144) // (size * size))), "size": size}


# ------------------------------------------------------------------ inputs

def _operator(case, seed):
    """CSR arrays of the case's operator and its row count."""
    op, size = case["op"], case["size"]
    if op == "diag":
        csr = W.diag_csr(size)
    elif op == "lattice2d":
        csr = W.anderson2d_csr(size, case["W"], seed=seed)[0]
    elif op == "laplace3d":
        csr = W.laplace3d_csr(size, seed=seed)
    elif op == "anderson3d":
        csr = W.anderson3d_csr(size, seed=seed)
    else:
        csr = W.random_sym_csr(size, seed=seed)
    return csr, len(csr[0]) - 1


def _lattices(count, lo, hi, seed):
    """(side, disorder, seed) of each lattice of a set: the sides are the
    case's own, the disorder is the seed's."""
    sides = np.random.default_rng(count * 1000 + lo).integers(lo, hi + 1, size=count)
    rng = np.random.default_rng(seed)
    return [(int(L), float(rng.uniform(1.0, 12.0)), int(rng.integers(1 << 30))) for L in sides]


def _prepare_solve(case, seed):
    csr, n = _operator(case, seed)
    cplx = case["path"] == "complex"
    nev = SOLVER[case["op"]][1]
    return {"A": T.Csr(*csr, complex_=cplx, mixed=case["path"] == "mixed"),
            "x0": W.start_vector(n, seed=seed + 1, complex_=cplx),
            "out": None if cplx else T.output_buffers(n, nev)}


def _prepare_batch(case, seed):
    nev, maxlan = LN.NEV, SOLVER["lattice2d"][2]
    probs, pots = [], []
    for L, Wd, s in _lattices(case["jobs"], case["lo"], case["hi"], seed):
        csr, pot = W.anderson2d_csr(L, Wd, seed=s)
        A = T.Csr(*csr, mixed=case["path"] == "mixed")
        start = None if case["learned"] else W.start_vector(L * L, seed=s + 1)
        probs.append((A, -1, nev, maxlan, TOL, 1, MAXMV, nev, start))
        pots.append(pot.reshape(L, L))
    # the caller's result arrays: the eigenvectors of all jobs back to back
    evals, resid = np.zeros((len(probs), nev)), np.zeros((len(probs), nev))
    evecs = np.ones(nev * sum(p.size for p in pots))
    out, o = [], 0
    for j, p in enumerate(pots):
        out.append((evals[j], evecs[o:o + nev * p.size].reshape(nev, p.size), resid[j]))
        o += nev * p.size
    return {"probs": probs, "pots": pots, "out": out, "evals": evals, "evecs": evecs,
            "net": LN.load_net() if case["learned"] else None}


def _prepare_pass(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    vt, dt = TILE[case["dtype"]]
    n, m = case["n"], case["m"]
    ld = (n + 63) & ~63
    wide = torch.complex128 if case["dtype"] == "c128" else torch.float64
    V = torch.zeros((m, ld), dtype=dt, device="cuda")
    V[:, :n] = torch.randn((m, n), dtype=dt, device="cuda", generator=g) / n ** 0.5
    r0 = torch.randn(n, dtype=wide, device="cuda", generator=g) / n ** 0.5 + 0.3 * V[0, :n]
    f = T.lib().trlhip_cgs_pass_noalloc
    P = ctypes.c_void_p
    f.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, P, ctypes.c_long, P, P, P, P, P]
    f.restype = ctypes.c_int
    h = np.zeros(m, dtype=np.complex128 if case["dtype"] == "c128" else np.float64)
    return {"f": f, "vt": vt, "n": n, "m": m, "ld": ld, "V": V, "r0": r0, "r": torch.empty_like(r0), "h": h}


def _prepare_infer(case, seed):
    pots = [(np.random.default_rng(s).random((L, L)) - 0.5) * Wd
            for L, Wd, s in _lattices(case["images"], case["lo"], case["hi"], seed)]
    return {"net": LN.load_net(), "pots": pots}


def _train_batch(case, seed):
    """Potentials and targets: localized positive amplitudes, as the density
    amplitude of a lattice's lowest states is."""
    rng = np.random.default_rng(seed)
    n, L = case["images"], case["size"]
    Wd = rng.uniform(1.0, 12.0, size=(n, 1, 1))
    x = ((rng.random((n, L, L)) - 0.5) * Wd * LN.SCALE).astype(np.float32)
    t = np.exp(-6.0 * (x + np.roll(x, 1, 1) + np.roll(x, 1, 2))).astype(np.float32)
    return x, t / np.sqrt((t * t).sum(axis=(1, 2), keepdims=True))


def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        x, t = _train_batch(case, seed)
        s = {"net": LN.load_net(), "x": x, "t": t}
    else:
        s = {"solve": _prepare_solve, "batch": _prepare_batch, "pass": _prepare_pass,
             "infer": _prepare_infer}[kind](case, seed)
    s["case"] = case
    return s


# --------------------------------------------------------------- the calls

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "solve":
        lohi, nev, maxlan = SOLVER[case["op"]]
        r = T.solve_csr(s["A"], lohi, nev, maxlan, TOL, 1, MAXMV, nev, s["x0"], out=s["out"])
        return {"eval": r["eval"], "evec": r["evec"], "nec": r["nec"]}
    if kind == "batch":
        starts = LN.start_vectors_device(s["net"], s["pots"]) if case["learned"] else None
        rc, res, _ = T.solve_batch(s["probs"], out=s["out"], dstarts=starts)
        if rc != 0:
            raise RuntimeError(f"trlan_batch failed ({rc})")
        return {"eval": s["evals"], "evec": s["evecs"], "nec": sum(r["nec"] for r in res)}
    if kind == "pass":
        s["r"].copy_(s["r0"])
        hh, rr2 = ctypes.c_double(), ctypes.c_double()
        rc = s["f"](s["n"], s["m"], s["vt"], s["V"].data_ptr(), s["ld"], s["r"].data_ptr(),
                    ctypes.byref(hh), ctypes.byref(rr2), s["h"].ctypes.data,
                    torch.cuda.current_stream().cuda_stream)
        if rc != 0:
            raise RuntimeError(f"trlhip_cgs_pass_noalloc failed ({rc})")
        return {"r": s["r"], "h": s["h"], "hh": hh.value, "rr2": rr2.value}
    if kind == "infer":
        y = LN.start_vectors(s["net"], s["pots"])
        # the vectors are views of one result array, images of equal size
        # together; a set has more of them than a caller lists one by one
        return y[0].base if y[0].base is not None else y[0]
    loss, grad = s["net"].loss_grad(s["x"], s["t"])
    return {"loss": loss, "grad": grad}


# ------------------------------------------------------ necessary work

def _sites(case):
    """Expected sites of a set of square lattices with sides lo..hi."""
    lo, hi = case["lo"], case["hi"]
    return sum(L * L for L in range(lo, hi + 1)) / (hi - lo + 1) * case.get("jobs", case.get("images", 1))


NET_FLOPS = 2.0 * (9 * 32 + 2 * 9 * 32 * 32 + 9 * 32)  # per pixel, forward


def work(case):
    """Each input read once, each output written once.  A solve's operator
    applications depend on the spectrum, so only one is counted."""
    kind = case["kind"]
    if kind == "solve":
        op, size = case["op"], case["size"]
        n = size if op in ("diag", "random") else size ** (2 if op == "lattice2d" else 3)
        per = {"diag": 1, "lattice2d": 5, "laplace3d": 7, "anderson3d": 7, "random": 17}[op]
        e = 16 if case["path"] == "complex" else 8
        nev = SOLVER[op][1]
        return {"bytes": n * (per * (e + 4) + 4 + e * (1 + nev)),
                "flops": (8.0 if e == 16 else 2.0) * n * per}
    if kind == "batch":
        n = _sites(case)
        return {"bytes": n * (5 * 12 + 4 + 8 * (1 + LN.NEV)),
                "flops": n * (10.0 + (NET_FLOPS if case["learned"] else 0.0))}
    if kind == "pass":
        n, m = case["n"], case["m"]
        v = {"r64": 8, "r32": 4, "c128": 16}[case["dtype"]]
        r = 16 if case["dtype"] == "c128" else 8
        return {"bytes": float(n) * (m * v + 2 * r), "flops": (16.0 if r == 16 else 4.0) * n * m}
    if kind == "infer":
        n = _sites(case)
        return {"bytes": n * 12.0, "flops": n * NET_FLOPS}
    n = float(case["images"]) * case["size"] ** 2
    return {"bytes": n * 8.0, "flops": 3.0 * n * NET_FLOPS}


# ------------------------------------------------- the same in 64 bits

def _dense(csr, n, dtype):
    rp, ci, v = csr
    rows = np.repeat(np.arange(n), np.diff(rp))
    M = torch.zeros((n, n), dtype=dtype, device="cuda")
    M.index_put_((torch.from_numpy(rows).cuda(), torch.from_numpy(ci.astype(np.int64)).cuda()),
                 torch.from_numpy(v).to(dtype).cuda(), accumulate=True)
    return M


def _conv(x, w, b):
    """3x3 periodic convolution, channels last: x (..., h, w, ci), w (co, 9,
    ci), taps (dy, dx) row by row."""
    y = b
    for t in range(9):
        y = y + torch.roll(x, (1 - t // 3, 1 - t % 3), (1, 2)) @ w[:, t].T
    return y


def _net64(params, x):
    C, o, layers = 32, 0, []
    for co, ci in ((C, 1), (C, C), (C, C), (1, C)):
        layers.append((params[o:o + co * 9 * ci].reshape(co, 9, ci), params[o + co * 9 * ci:o + co * (9 * ci + 1)]))
        o += co * (9 * ci + 1)
    a = x.unsqueeze(-1)
    for i, (w, b) in enumerate(layers):
        a = _conv(a, w, b)
        if i < 3:
            a = torch.relu(a)
    return a.squeeze(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "solve":
        lohi, nev, _ = SOLVER[case["op"]]
        if case["op"] == "diag":
            return {"eval": np.arange(case["size"] - nev + 1, case["size"] + 1, dtype=np.float64),
                    "evec": None, "nec": nev}
        csr, n = _operator(case, seed)
        if n > 4000:
            return None
        ev = torch.linalg.eigvalsh(_dense(csr, n, torch.complex128 if case["path"] == "complex"
                                          else torch.float64)).cpu().numpy()
        # an eigenvector's sign is the solver's own
        return {"eval": ev[:nev] if lohi < 0 else ev[-nev:], "evec": None, "nec": nev}
    if kind == "batch":
        return None
    if kind == "pass":
        s = _prepare_pass(case, seed)
        V = s["V"][:, :s["n"]].to(s["r0"].dtype)
        h = V.conj() @ s["r0"]
        r = s["r0"] - h @ V
        return {"r": r, "h": h.cpu().numpy(), "hh": float((h.abs() ** 2).sum()),
                "rr2": float((r.abs() ** 2).sum())}
    p = torch.from_numpy(np.load(LN.WEIGHTS, allow_pickle=False)).double().cuda()
    if kind == "infer":
        pots = _prepare_infer(case, seed)["pots"]
        sides, parts = [], []
        for d in pots:
            if len(d) not in sides:
                sides.append(len(d))
        for L in sides:  # images of equal size together, as start_vectors lays them out
            for d in pots:
                if len(d) == L:
                    x = torch.from_numpy((d * LN.SCALE).astype(np.float32)).double().cuda()
                    parts.append(_net64(p, x[None]).reshape(-1))
        return torch.cat(parts).cpu().numpy()
    x, t = _train_batch(case, seed)
    p.requires_grad_(True)
    o = _net64(p, torch.from_numpy(x).double().cuda()).flatten(1)
    t = torch.from_numpy(t).double().cuda().flatten(1)
    loss = (1 - (o * t).sum(1) ** 2 / ((o * o).sum(1) * (t * t).sum(1))).mean()
    loss.backward()
    return {"loss": float(loss.detach()), "grad": p.grad.cpu().numpy()}
