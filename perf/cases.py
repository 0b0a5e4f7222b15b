"""The work that users of this framework have it do, as measurable cases.

Each case is one pass through the public entry points on a pyrochlore
supercell diag(n0, n1, n2) (4 n0 n1 n2 spins, ice-rule sector n_spinon_pairs):

  apply         GpuOp.evaluate / evaluate_add, the matrix-free H.v that every
                Krylov solver calls; mode says what the program has prepared:
                "plain" nothing, "low" low keys built and verified, "cached"
                the connectivity kept on the device
  block         GpuOp.apply_block, R columns with their own (g, B) each: a
                parameter scan, or FTLM samples
  lanczos       GpuOp.lanczos_coeffs, M steps of the 3-term recurrence
  eigsh         GpuOp.eigsh, the lowest eigenvalues by thick-restart Lanczos
                (mfsparse over the search, sparse over the cached connectivity)
  ftlm          ftlm.lanczos_block over spinon sectors, then the thermodynamics
  served        serve.Engine, a batch of solve requests continuously batched
  correlations  observables.expectations and cross_correlations of the ring
                operators on eigenvector-like states
"""
import numpy as np
import torch

import qsi_subspace_ed_amd as q
from qsi_subspace_ed_amd import ftlm, latgen, observables, serve

# lattice -> (repeats, hexagon flips, {sector: (basis states, off-diagonal nonzeros)})
LATTICES = {
    "1x2x2": ((1, 2, 2), 32, {0: (114, 272), 1: (228, 496)}),
    "2x2x2": ((2, 2, 2), 64, {0: (2970, 15360), 1: (5940, 28548)}),
    "1x3x3": ((1, 3, 3), 72, {0: (13122, 81432), 1: (26244, 154512)}),
    "2x2x3": ((2, 2, 3), 96, {0: (87546, 703680), 1: (175092, 1338676)}),
    "1x3x4": ((1, 3, 4), 96, {0: (223650, 1858512), 1: (447300, 3566912)}),
    "1x2x6": ((1, 2, 6), 96, {0: (293394, 2543448), 1: (586788, 4834752)}),
    "2x2x4": ((2, 2, 4), 128, {0: (2756394, 30174720), 1: (5512788, 58090092)}),
    "1x3x5": ((1, 3, 5), 120, {0: (3897234, 40895820), 1: (7794468, 79080120)}),
    "2x3x3": ((2, 3, 3), 144, {0: (12846186, 156989808)}),
    "2x4x3": ((2, 4, 3), 192, {0: (2007260562, 33063045984)}),
}


def listed():
    return [
        # one H.v on a small cluster (32 spins): the time is launches and latency
        {"name": "apply_32_plain", "kind": "apply", "lattice": "2x2x2", "sector": 0, "mode": "plain",
         "add": False},
        # the H.v of a 64-spin matrix-free solve, low keys as mfsparse prepares them
        {"name": "apply_64_low", "kind": "apply", "lattice": "2x2x4", "sector": 0, "mode": "low",
         "add": False},
        # y += H x on two-word states (72 spins, an odd supercell) without any preparation
        {"name": "apply_72_add", "kind": "apply", "lattice": "2x3x3", "sector": 0, "mode": "plain",
         "add": True},
        # the largest H.v: 96 spins, 2.0e9 states, the benchmark's workload
        {"name": "apply_96_low", "kind": "apply", "lattice": "2x4x3", "sector": 0, "mode": "low",
         "add": False},
        # the H.v of a 64-spin sparse solve: the connectivity fits and is kept
        {"name": "apply_64_cached", "kind": "apply", "lattice": "2x2x4", "sector": 0,
         "mode": "cached", "add": False},
        # a parameter scan of seven (g, B) points over one search of the 64-spin basis
        {"name": "block_64_r7", "kind": "block", "lattice": "2x2x4", "sector": 0, "mode": "plain",
         "R": 7},
        # the density-of-states recurrence of a 64-spin run, matrix-free
        {"name": "lanczos_64_low", "kind": "lanczos", "lattice": "2x2x4", "sector": 0,
         "mode": "low", "M": 40},
        # five lowest levels of the 64-spin cluster, matrix-free (mfsparse)
        {"name": "eigsh_64_low", "kind": "eigsh", "lattice": "2x2x4", "sector": 0, "mode": "low",
         "nev": 5, "ncv": 15},
        # the default solve of a 48-spin cluster (sparse, one level): many short steps
        {"name": "eigsh_48_cached", "kind": "eigsh", "lattice": "2x2x3", "sector": 0,
         "mode": "cached", "nev": 1, "ncv": 15},
        # finite-temperature run over two spinon sectors: 64 samples each, 100 steps
        {"name": "ftlm_48_r64", "kind": "ftlm", "lattice": "2x2x3", "sectors": 2, "R": 64,
         "M": 100},
        # a queue of 24 parameter points on one 48-spin space, 16 solved side by side
        {"name": "served_48_c16", "kind": "served", "lattice": "2x2x3", "sector": 0, "cols": 16,
         "requests": 24, "nev": 5, "ncv": 15},
        # ring expectations and ring-ring correlations of two 48-spin eigenvectors
        {"name": "correlations_48", "kind": "correlations", "lattice": "2x2x3", "sector": 0,
         "nvec": 2},
    ]


def draw(rng):
    kind = rng.choice(["apply", "apply", "apply", "block", "block", "lanczos", "eigsh", "ftlm",
                       "served", "correlations"])
    # the lattices lie about evenly over the logarithm of the basis size
    small = ["1x2x2", "2x2x2", "1x3x3", "2x2x3", "1x3x4", "1x2x6"]
    sector = rng.randint(0, 1)
    if kind == "apply":
        name = rng.choice(small + ["2x2x4", "1x3x5", "2x3x3"])
        return {"kind": kind, "lattice": name, "sector": 0 if name == "2x3x3" else sector,
                "mode": rng.choice(["plain", "low", "cached"]), "add": rng.random() < 0.3}
    if kind == "block":
        return {"kind": kind, "lattice": rng.choice(small + ["2x2x4", "1x3x5"]), "sector": sector,
                "mode": rng.choice(["plain", "cached"]), "R": int(round(2.0 ** rng.uniform(0, 6)))}
    if kind == "lanczos":
        return {"kind": kind, "lattice": rng.choice(small[1:] + ["2x2x4"]), "sector": sector,
                "mode": rng.choice(["plain", "low", "cached"]), "M": rng.randint(10, 40)}
    if kind == "eigsh":
        return {"kind": kind, "lattice": rng.choice(small[1:] + ["2x2x4"]), "sector": 0,
                "mode": rng.choice(["low", "cached"]), "nev": rng.randint(1, 6),
                "ncv": rng.randint(14, 24)}
    if kind == "ftlm":
        return {"kind": kind, "lattice": rng.choice(small[1:4]), "sectors": rng.randint(1, 2),
                "R": int(round(2.0 ** rng.uniform(1, 6))), "M": rng.randint(40, 100)}
    if kind == "served":
        cols = rng.randint(3, 16)
        return {"kind": kind, "lattice": rng.choice(small[1:4]), "sector": sector, "cols": cols,
                "requests": rng.randint(cols, 24), "nev": rng.randint(1, 5), "ncv": 15}
    return {"kind": kind, "lattice": rng.choice(small[1:]), "sector": 0, "nvec": rng.randint(1, 3)}


def _lattice(case):
    return latgen.Supercell(LATTICES[case["lattice"]][0]).to_dict()


def _point(rng):
    """One parameter point: g_s ~ U[0.2, 1] with the workloads' sign
    H = -sum g_s (O + O^dagger), and a field of 0.1 in a random direction."""
    g = -rng.uniform(0.2, 1.0, size=4)
    B = rng.standard_normal(3)
    return g, 0.1 * B / np.linalg.norm(B)


def _hamiltonian(jdata, rng):
    g, B = _point(rng)
    H = q.build_hamiltonian_g(jdata, list(g))
    q.add_local_field(H, jdata, B)
    return H


def _coeffs(rng, R):
    """(8, R) slot coefficients of R parameter points of the slotted model."""
    out = np.empty((serve.N_SLOTS, R))
    for r in range(R):
        g, B = _point(rng)
        out[:, r] = serve.point_coeffs(g, q.get_loc_z() @ B)
    return out


def _operator(case, jdata, H):
    basis = q.enumerate_basis_device(jdata, case.get("sector", 0))
    op = q.GpuOp(basis, H)
    if case["mode"] == "low":
        basis.build_lowkeys()
        op.verify_lowkeys()
    elif case["mode"] == "cached":
        op.cache_connectivity()
        # the gather depth that the autotuner picks on these bases
        op.set_cached_pipe(32)
    return op


def _vectors(seed, *shape):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(*shape, dtype=torch.float64, device="cuda", generator=gen)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    jdata = _lattice(case)
    kind = case["kind"]
    s = {"case": case}
    if kind == "ftlm":
        H = _hamiltonian(jdata, rng)
        ops, starts = [], []
        for n in range(case["sectors"]):
            op = q.GpuOp(q.enumerate_basis_device(jdata, n), H)
            op.cache_connectivity()
            # the configuration that the autotuner picks for this recurrence
            op.set_block_cfg(9)
            ops.append(op)
            V = torch.sign(_vectors(seed + n, op.rows(), case["R"])) / np.sqrt(op.rows())
            starts.append(V.contiguous())
        s.update(ops=ops, starts=starts, temps=np.geomspace(0.1, 10.0, 48))
        return s
    if kind == "served":
        basis = q.enumerate_basis_device(jdata, case["sector"])
        op = q.GpuOp(basis, serve.slotted_hamiltonian(jdata))
        s["engine"] = serve.Engine(op, max_cols=case["cols"], nev=case["nev"], ncv=case["ncv"],
                                   tol=1e-10)
        s["points"] = _coeffs(rng, case["requests"])
        s["seeds"] = [int(v) for v in rng.integers(1, 1 << 30, size=case["requests"])]
        return s
    if kind == "correlations":
        basis = q.enumerate_basis_device(jdata, case["sector"])
        s["ops"] = observables.ring_operators(basis, jdata)
        psi = _vectors(seed, basis.dim(), case["nvec"])
        s["psi"] = torch.linalg.qr(psi)[0].contiguous()
        return s
    if kind == "block":
        op = _operator(case, jdata, serve.slotted_hamiltonian(jdata))
        s["coeffs"] = torch.from_numpy(_coeffs(rng, case["R"])).cuda()
        s["x"] = _vectors(seed, op.rows(), case["R"])
    else:
        op = _operator(case, jdata, _hamiltonian(jdata, rng))
        s["x"] = _vectors(seed, op.rows())
        s["x"] /= torch.linalg.norm(s["x"])
    s["op"] = op
    if kind in ("apply", "block"):
        s["y"] = torch.empty_like(s["x"])
    if case.get("add"):
        s["y0"] = _vectors(seed + 1, op.rows())
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "apply":
        x, y = state["x"], state["y"]
        if case["add"]:
            y.copy_(state["y0"])
            state["op"].evaluate_add(x, y)
        else:
            state["op"].evaluate(x, y)
        return y
    if kind == "block":
        state["op"].apply_block(state["x"], state["y"], coeffs=state["coeffs"])
        return state["y"]
    if kind == "lanczos":
        alpha, beta = state["op"].lanczos_coeffs(case["M"], v0=state["x"])
        return {"alpha": alpha, "beta": beta}
    if kind == "eigsh":
        return state["op"].eigsh(nev=case["nev"], ncv=case["ncv"], tol=1e-10, v0=state["x"])[0]
    if kind == "ftlm":
        alpha, beta, _ = ftlm.lanczos_block(state["ops"], state["starts"], case["M"])
        out = []
        for k, op in enumerate(state["ops"]):
            nodes = ftlm.quadrature(alpha[k], beta[k])
            t = ftlm.thermodynamics(nodes, op.rows(), state["temps"])
            out.append({"Z": t["Z_shifted"], "E": t["E"], "C": t["C"]})
        return out
    if kind == "served":
        ids = [state["engine"].submit(state["points"][:, k], seed)
               for k, seed in enumerate(state["seeds"])]
        done = {f.id: f.evals for f in state["engine"].run_all()}
        return np.stack([done[i] for i in ids])
    return {"ring": observables.expectations(state["ops"], state["psi"]),
            "ring_ring": observables.cross_correlations(state["ops"], state["psi"])}


def work(case):
    """Least work of a pass: for an apply every state, x and y once, two
    operations per nonzero; solvers as that many applies plus one read of what
    each step orthogonalises against."""
    repeats, flips, sizes = LATTICES[case["lattice"]]
    S = 8 if 4 * np.prod(repeats) <= 64 else 16
    D, nnz = sizes[case.get("sector", 0)]
    kind = case["kind"]
    if kind == "apply":
        return {"bytes": D * (S + 16 + (16 if case["add"] else 0)), "flops": 2 * nnz}
    if kind == "block":
        return {"bytes": D * (S + 16 * case["R"]), "flops": 2 * nnz * case["R"]}
    if kind == "lanczos":
        M = case["M"]
        return {"bytes": M * D * (S + 32), "flops": M * (2 * nnz + 8 * D)}
    if kind == "eigsh":
        # about 15 restarts of half a basis each
        steps = 15 * case["ncv"]
        return {"bytes": steps * D * (S + 16 + 8 * case["ncv"]),
                "flops": steps * (2 * nnz + 8 * case["ncv"] * D)}
    if kind == "ftlm":
        b = f = 0
        for n in range(case["sectors"]):
            D, nnz = sizes[n]
            b += case["M"] * D * (S + 32 * case["R"])
            f += case["M"] * case["R"] * (2 * nnz + 8 * D)
        return {"bytes": b, "flops": f}
    if kind == "served":
        steps = 15 * case["ncv"] * case["requests"]
        return {"bytes": steps * D * (16 + 8 * case["ncv"]),
                "flops": steps * (2 * nnz + 8 * case["ncv"] * D)}
    P = flips // 2 * case["nvec"]
    return {"bytes": 2 * D * (S + 8 * case["nvec"]), "flops": 2 * D * P * (P + case["nvec"])}


def _pull_lists(basis, H):
    """Per off-diagonal term (coefficient, slot, rows, columns, signs) of the
    pull form in plain torch, and the diagonal as [(c, slot, values)].  Ranks
    come from a search over the bit positions that tell the states apart."""
    st = torch.from_numpy(basis.states().view(np.int64)).cuda()
    D = st.shape[0]
    bits = []
    for p in range(127, -1, -1):
        b = (st[:, p >> 6] >> (p & 63)) & 1
        if D > 1 and bool((b[1:] != b[:-1]).any()):
            bits.append((p, b))
    # of the varying positions, those at which neighbours first differ
    key = torch.zeros(D, dtype=torch.int64, device="cuda")
    same = torch.ones(max(D - 1, 0), dtype=torch.bool, device="cuda")
    used = []
    for p, b in bits:
        diff = same & (b[1:] != b[:-1])
        if bool(diff.any()):
            used.append(p)
            key = (key << 1) | b
            same &= ~diff
    del bits
    words = lambda m: [torch.tensor(np.array([w], dtype=np.uint64).view(np.int64)[0],  # noqa: E731
                                    device="cuda") for w in (m & (2**64 - 1), m >> 64)]

    def parity(v):
        for s in (32, 16, 8, 4, 2, 1):
            v = v ^ (v >> s)
        return v & 1

    off, diag = [], []
    for c, o, slot in H.off_diag_terms:
        m = o.up | o.down
        mw, vw, xw, zw = words(m), words(o.up ^ (o.X & m)), words(o.X), words(o.Z)
        rows = torch.nonzero(((st[:, 0] & mw[0]) == vw[0]) & ((st[:, 1] & mw[1]) == vw[1]))[:, 0]
        s = st[rows]
        k = torch.zeros(rows.shape[0], dtype=torch.int64, device="cuda")
        for p in used:
            k = (k << 1) | (((s[:, p >> 6] ^ xw[p >> 6]) >> (p & 63)) & 1)
        cols = torch.searchsorted(key, k).clamp(max=D - 1)
        found = ((st[cols, 0] == (s[:, 0] ^ xw[0])) & (st[cols, 1] == (s[:, 1] ^ xw[1])))
        sign = 1.0 - 2.0 * parity((~s[:, 0] & zw[0]) ^ (~s[:, 1] & zw[1])).double()
        off.append((c, slot, rows[found], cols[found], (o.sign * sign)[found]))
    for c, o, slot in H.diagonal_terms:
        zw, uw, dw = words(o.Z), words(o.up), words(o.down)
        ok = ((st[:, 0] & (uw[0] | dw[0])) == uw[0]) & ((st[:, 1] & (uw[1] | dw[1])) == uw[1])
        sign = 1.0 - 2.0 * parity((~st[:, 0] & zw[0]) ^ (~st[:, 1] & zw[1])).double()
        diag.append((c, slot, o.sign * sign * ok))
    return D, off, diag


def _apply(lists, x, coeffs=None):
    D, off, diag = lists
    y = torch.zeros_like(x)
    col = (lambda v: v) if x.dim() == 1 else (lambda v: v[:, None])
    for c, slot, rows, cols, sign in off:
        w = c if coeffs is None or slot < 0 else coeffs[slot]
        y.index_add_(0, rows, w * col(sign) * x[cols])
    for c, slot, val in diag:
        w = c if coeffs is None or slot < 0 else coeffs[slot]
        y += w * col(val) * x
    return y


def exact(case, seed):
    kind = case["kind"]
    if LATTICES[case["lattice"]][2][0][0] > 5_000_000 or kind in ("ftlm", "served"):
        return None
    if kind == "eigsh" and case["lattice"] not in ("1x2x2", "2x2x2"):
        return None
    s = prepare(case, seed)
    rng = np.random.default_rng(seed)
    jdata = _lattice(case)
    if kind == "correlations":
        out = []
        for op, O in zip(s["ops"], q.get_ring_ops(jdata)[0]):
            H = q.SymbolicOpSum()
            H.add_term(1.0, O)
            out.append(_apply(_pull_lists(op.basis, H), s["psi"]))
        Y = torch.stack(out)  # operator, row, vector
        return {"ring": torch.stack([(Yl.t() @ s["psi"]) for Yl in Y]),
                "ring_ring": torch.stack([torch.stack([a.t() @ b for b in Y]) for a in Y])}
    if kind == "block":
        lists = _pull_lists(s["op"].basis, serve.slotted_hamiltonian(jdata))
        return _apply(lists, s["x"], s["coeffs"])
    lists = _pull_lists(s["op"].basis, _hamiltonian(jdata, rng))
    if kind == "apply":
        y = _apply(lists, s["x"])
        return y + s["y0"] if case["add"] else y
    if kind == "eigsh":
        full = _apply(lists, torch.eye(lists[0], dtype=torch.float64, device="cuda"))
        return torch.linalg.eigvalsh(full)[:case["nev"]].cpu().numpy()
    v, u, beta = s["x"] / torch.linalg.norm(s["x"]), None, 0.0
    alphas, betas = [], []
    for _ in range(case["M"]):
        w = _apply(lists, v)
        if u is not None:
            w = w - beta * u
        alpha = torch.dot(v, w)
        w = w - alpha * v
        beta = torch.linalg.norm(w)
        alphas.append(alpha)
        betas.append(beta)
        u, v = v, w / beta
    return {"alpha": torch.stack(alphas).cpu().numpy(), "beta": torch.stack(betas).cpu().numpy()}
