"""Timed cases of the plane-wave H.psi / S.psi and block-Davidson framework.

Each case is one call (or one short chain of calls) that a plane-wave program
makes on the device library, over the sizes that such programs have: the 8, 16,
32 and 64 atom silicon cells of the serving mix at 10 to 15 Ha, the two-species
32-atom slab at 20 Ha, Gamma and general k-points, blocks from the last few
unconverged bands of a small cell to the three-fold seed block of a large one.

Kinds of case:

* apply:   H x, S x or both on blocks resident in HBM (Operator.apply_device),
           the call an eigensolver of the user's own makes per expansion.
* accel:   the drop-in accelerator calls on host blocks (Context
           .local_hamiltonian and .paw_pair with resident operators), one H and
           S application of a host-side solver.
* kpoints: H x and S x of every k-point of a mesh in one batched call
           (Batch.apply on host blocks).
* solve:   a certified solve whose blocks stay in HBM (Operator.davidson with
           device_blocks; FP32 search with refinement, warm start), then the
           warm block projected on the occupied bands (the subspace alignment
           of a dynamics step, free of the bands' arbitrary phases).
* scf:     a certified FP64 solve on host blocks followed by the smooth density
           of the smeared occupations (Operator.davidson, Operator.density).
"""
import functools
import math
import os
import sys

import numpy as np
import torch

_PACKAGE = os.path.join(os.getcwd(), "sparse-dft_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from sdft_amd import native, synthetic  # noqa: E402

LATTICE = 10.26  # bohr, conventional silicon cell
HARTREE_EV = 27.211386245988
SMEARING = 0.004  # Ha, Gaussian width of the occupations


def listed():
    return [
        # the last unconverged bands of a small cell: launches and latency
        dict(name="apply_si8_pair_f64_4", kind="apply", cell="1x1x1", ecut=10.0, k="gamma", grid="32", columns=4,
             which="pair", precision=0),
        # search-precision H on a full small block at a general k-point
        dict(name="apply_si8_h_f32_20", kind="apply", cell="1x1x1", ecut=13.75, k="general", grid="rule", columns=20,
             which="h", precision=1),
        # an ordinary cell on the rule grid, odd block width
        dict(name="apply_si16_pair_f64_37", kind="apply", cell="2x1x1", ecut=12.5, k="general", grid="rule", columns=37,
             which="pair", precision=0),
        # two species (8 and 18 projectors an atom), anisotropic grid
        dict(name="apply_slab_pair_f64_96", kind="apply", cell="slab", ecut=20.0, k="general", grid="48x48x96", columns=96,
             which="pair", precision=0),
        # the 64-atom benchmark block in search and in certificate precision
        dict(name="apply_si64_pair_f32_160", kind="apply", cell="2x2x2", ecut=15.0, k="gamma", grid="72", columns=160,
             which="pair", precision=1),
        dict(name="apply_si64_pair_f64_160", kind="apply", cell="2x2x2", ecut=15.0, k="gamma", grid="72", columns=160,
             which="pair", precision=0),
        # S images of a warm start's seed block (three blocks of roots)
        dict(name="apply_si64_s_f64_480", kind="apply", cell="2x2x2", ecut=15.0, k="gamma", grid="72", columns=480,
             which="s", precision=0),
        # one application of a host-side solver through the drop-in calls
        dict(name="accel_si16_f64_40", kind="accel", cell="2x1x1", ecut=12.5, k="gamma", grid="rule", columns=40,
             precision=0),
        # every k-point of a 3x3x3 mesh in one call
        dict(name="kpoints_si8_mesh3_20", kind="kpoints", cell="1x1x1", ecut=10.0, mesh=3, grid="32", columns=20,
             precision=0),
        # one self-consistency step of a small cell, cold start, FP64 throughout
        dict(name="scf_si8_f64_20", kind="scf", cell="1x1x1", ecut=10.0, k="gamma", grid="32", roots=20),
        # a request of the serving mix
        dict(name="solve_si32_f32_80", kind="solve", cell="2x2x1", ecut=12.5, k="gamma", grid="rule", roots=80),
        # the 64-atom benchmark solve
        dict(name="solve_si64_f32_160", kind="solve", cell="2x2x2", ecut=15.0, k="gamma", grid="72", roots=160),
    ]


def _log_int(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["apply"] * 6 + ["accel", "kpoints", "scf", "solve", "solve"])
    ecut = round(rng.uniform(10.0, 15.0), 2)
    k = rng.choice(["gamma", "general"])
    if kind == "apply":
        cell = rng.choice(["1x1x1", "2x1x1", "2x2x1", "2x2x2", "slab"])
        return dict(kind=kind, cell=cell, ecut=20.0 if cell == "slab" else ecut, k=k,
                    grid="48x48x96" if cell == "slab" else "rule", columns=_log_int(rng, 2, 400),
                    which=rng.choice(["h", "s", "pair", "pair"]), precision=rng.choice([0, 1]))
    if kind == "accel":
        return dict(kind=kind, cell=rng.choice(["1x1x1", "2x1x1", "2x2x1"]), ecut=ecut, k=k, grid="rule",
                    columns=_log_int(rng, 4, 120), precision=rng.choice([0, 1]))
    if kind == "kpoints":
        return dict(kind=kind, cell="1x1x1", ecut=round(rng.uniform(9.0, 10.0), 2), mesh=rng.choice([2, 3]), grid="32",
                    columns=_log_int(rng, 4, 40), precision=rng.choice([0, 1]))
    if kind == "scf":
        cell = rng.choice(["1x1x1", "2x1x1"])
        return dict(kind=kind, cell=cell, ecut=ecut, k=k, grid="rule", roots=_atoms(cell) * 5 // 2 + rng.choice([0, 1, 3]))
    cell = rng.choice(["1x1x1", "2x1x1", "2x2x1"])
    return dict(kind=kind, cell=cell, ecut=ecut, k=k, grid="rule", roots=_atoms(cell) * 5 // 2 + rng.choice([0, 1, 3]))


# ---------------------------------------------------------------- structures
def _reps(cell):
    return tuple(int(v) for v in cell.split("x"))


def _atoms(cell):
    return 32 if cell == "slab" else 8 * int(np.prod(_reps(cell)))


def _kfrac(k):
    return {"gamma": (0.0, 0.0, 0.0), "general": (0.125, 0.25, 0.375)}[k]


def _shape(grid):
    """FFT grid; zeros ask for the library's smallest alias-free one."""
    if grid == "rule":
        return (0, 0, 0)
    sides = tuple(int(v) for v in grid.split("x"))
    return sides * 3 if len(sides) == 1 else sides


@functools.lru_cache(maxsize=64)
def _geometry(cell, ecut, kfrac, grid):
    """Sphere, projectors and on-site blocks of a structure: what stays the
    same from one potential to the next."""
    structure = synthetic.slab_cell() if cell == "slab" else synthetic.diamond_cell(LATTICE, _reps(cell))
    return synthetic.build_problem(structure, ecut, kfrac, _shape(grid), 3 if cell == "slab" else 1)


def _potential(cell, problem, seed):
    """The local potential of this seed: the atoms' wells plus a noise of its own."""
    return synthetic.lowpass_potential(problem.cell, 3 if cell == "slab" else 1, 0.02, seed % 4000 + 1)


def _problem(case, seed, kfrac=None):
    base = _geometry(case["cell"], case["ecut"], tuple(kfrac if kfrac is not None else _kfrac(case["k"])), case["grid"])
    hkl, values = _potential(case["cell"], base, seed)
    fields = dict(base.__dict__, v_hkl=hkl, v_values=values)
    return synthetic.Problem(**fields)


def _block(problem, columns, seed):
    """columns x n complex128 (rows are bands): complex normals / (1 + |G+k|^2)."""
    g = torch.Generator().manual_seed(int(seed) * 7919 + 17)
    z = torch.randn(columns, problem.n, 2, generator=g, dtype=torch.float64)
    q2 = torch.from_numpy(np.einsum("ij,ij->i", problem.qcart, problem.qcart))
    return torch.view_as_complex(z) / (1.0 + q2)


_CONTEXT = []


def _context():
    if not _CONTEXT:
        _CONTEXT.append(native.Context(0))
    return _CONTEXT[0]


def _mesh(case):
    return synthetic.mp_kpoints(case["mesh"])


# -------------------------------------------------------------------- passes
def prepare(case, seed):
    kind = case["kind"]
    if kind == "kpoints":
        problems = [_problem(case, seed, k) for k in _mesh(case)]
        ops = [native.Operator(_context(), p) for p in problems]
        blocks = [np.asfortranarray(_block(p, case["columns"], seed * 64 + i).numpy().T)
                  for i, p in enumerate(problems)]
        return dict(kind=kind, batch=native.Batch(_context(), ops, case["columns"], case["precision"]), blocks=blocks)
    problem = _problem(case, seed)
    if kind == "accel":
        context = native.Context(0)  # the calls' resident operators belong to the context
        op = native.Operator(context, problem)
        info = op.info()
        op.close()
        return dict(kind=kind, context=context, shape=op.shape, indices=info["indices"], kinetic=info["kinetic"],
                    potential=info["local_real"], b=np.asfortranarray(problem.all_b()),
                    d=np.asfortranarray(problem.block_d()), q=np.asfortranarray(problem.block_q()),
                    x=np.asfortranarray(_block(problem, case["columns"], seed).numpy().T), identity=int(seed) + 1,
                    precision=case["precision"])
    op = native.Operator(_context(), problem)
    if kind == "apply":
        x = _block(problem, case["columns"], seed).cuda()
        return dict(kind=kind, op=op, x=x, hy=torch.zeros_like(x), sy=torch.zeros_like(x), which=case["which"],
                    precision=case["precision"])
    if kind == "scf":
        return dict(kind=kind, op=op, roots=case["roots"], atoms=_atoms(case["cell"]),
                    volume=abs(float(np.linalg.det(problem.cell.lattice))), support=problem.v_hkl)
    x = _block(problem, case["roots"], seed).cuda()
    return dict(kind=kind, op=op, x=x, vectors=torch.zeros_like(x), roots=case["roots"], atoms=_atoms(case["cell"]))


def _occupations(energies, atoms):
    """Spin-summed Gaussian-smeared occupations of 4 electrons an atom."""
    def at(mu):
        return np.array([math.erfc((e - mu) / SMEARING) for e in energies])

    low, high = float(energies.min()) - 1.0, float(energies.max()) + 1.0
    for _ in range(80):
        mid = 0.5 * (low + high)
        low, high = (mid, high) if at(mid).sum() < 4 * atoms else (low, mid)
    return at(0.5 * (low + high))


def run(state):
    kind = state["kind"]
    if kind == "apply":
        x, which = state["x"], state["which"]
        state["op"].apply_device(x.data_ptr(), x.shape[0], state["hy"].data_ptr(), state["sy"].data_ptr(), which=which,
                                 precision=state["precision"])
        return {"pair": dict(h=state["hy"], s=state["sy"]), "h": dict(h=state["hy"]), "s": dict(s=state["sy"])}[which]
    if kind == "accel":
        ctx, i, x, precision = state["context"], state["identity"], state["x"], state["precision"]
        local = ctx.local_hamiltonian(state["shape"], state["indices"], state["kinetic"], state["potential"], x,
                                      operator_identity=i, precision=precision)
        h, s = ctx.paw_pair(i, state["b"], state["d"], state["q"], x, projector_identity=i, precision=precision)
        return dict(local=local, h=h, s=s)
    if kind == "kpoints":
        h, s = state["batch"].apply(state["blocks"])
        return dict(h=h, s=s)
    if kind == "scf":
        out = state["op"].davidson(state["roots"])
        f = _occupations(out["eigenvalues"], state["atoms"])
        rho = state["op"].density(out["eigenvectors"], f, state["volume"], state["support"])
        return dict(eigenvalues=out["eigenvalues"], converged=out["converged"], density=rho)
    x, v = state["x"], state["vectors"]
    out = state["op"].davidson(state["roots"], search_precision=1, search_handoff=1.0, stagnation_window=1,
                               subspace_factor=5, refinement=1, inner_iterations=6, bf16_projectors=1,
                               refinement_guards=max(1, state["roots"] * 3 // 8),
                               device_blocks=(x.data_ptr(), v.data_ptr()))
    f = torch.from_numpy(_occupations(out["eigenvalues"], state["atoms"])).to(x.device)
    # rows are bands: aligned = X0 (conj V)^T diag(f) V
    aligned = ((x @ v.conj().T) * f) @ v
    return dict(eigenvalues=out["eigenvalues"], converged=out["converged"], aligned=aligned)


# ---------------------------------------------------------------- what it takes
def _sizes(case, kfrac=None):
    p = _geometry(case["cell"], case["ecut"], tuple(kfrac if kfrac is not None else _kfrac(case["k"])), case["grid"])
    return p.n, p.np_total, p, _grid(p)


def _grid(problem):
    """The smallest alias-free 2,3,5,7-smooth grid, or the case's own."""
    out = []
    for a in range(3):
        if problem.shape[a] > 0:
            out.append(int(problem.shape[a]))
            continue
        m = max(3, 2 * int(problem.hkl[:, a].max() - problem.hkl[:, a].min()) + 1)
        while True:
            r = m
            for f in (2, 3, 5, 7):
                while r % f == 0:
                    r //= f
            if r == 1:
                break
            m += 1
        out.append(m)
    return tuple(out)


def _apply_work(n, projectors, grid, columns, which, real_bytes, products=1):
    """One application: the block in, the images out, the operator once; two
    transforms a column for H, B x and one back projection an image."""
    images = 2 if which == "pair" else 1
    count = float(np.prod(grid))
    flops = columns * 8.0 * n * projectors * (1 + images)
    size = 16.0 * n * columns * (1 + images) + 2 * real_bytes * n * projectors
    if which != "s":
        flops += columns * (10.0 * count * math.log2(count) + 2 * count)
        size += real_bytes * count + 8.0 * n
    return size * products, flops * products


def work(case):
    kind = case["kind"]
    if kind == "kpoints":
        total = [0.0, 0.0]
        for k in _mesh(case):
            n, projectors, _, grid = _sizes(case, k)
            b, f = _apply_work(n, projectors, grid, case["columns"], "pair", 8 if case["precision"] == 0 else 4)
            total[0] += b
            total[1] += f
        return dict(bytes=total[0], flops=total[1])
    n, projectors, _, grid = _sizes(case)
    if kind == "apply":
        b, f = _apply_work(n, projectors, grid, case["columns"], case["which"], 8 if case["precision"] == 0 else 4)
        return dict(bytes=b, flops=f)
    if kind == "accel":
        b, f = _apply_work(n, projectors, grid, case["columns"], "pair", 8 if case["precision"] == 0 else 4)
        return dict(bytes=b + 16.0 * n * case["columns"], flops=f)
    # a solve: ten pair applications of the block, each with the projection,
    # orthonormalisation and rotation of a block of twice as many columns
    r = case["roots"]
    b, f = _apply_work(n, projectors, grid, r, "pair", 8)
    return dict(bytes=10 * (b + 4 * 16.0 * n * r), flops=10 * (f + 4 * 8.0 * n * r * (2 * r)))


# ------------------------------------------------------- the same in plain torch
class _Plain:
    """The operator of a problem in complex128 torch."""

    def __init__(self, problem, device):
        self.p, self.device = problem, device
        self.grid = _grid(problem)
        n0, n1, n2 = self.grid
        wrap = problem.hkl.astype(np.int64) % np.array(self.grid)
        self.index = torch.from_numpy((wrap[:, 0] * n1 + wrap[:, 1]) * n2 + wrap[:, 2]).to(device)
        self.kinetic = torch.from_numpy(problem.kinetic_ev / HARTREE_EV).to(device)
        span = problem.hkl.max(axis=0) - problem.hkl.min(axis=0)
        keep = np.all(np.abs(problem.v_hkl) <= span, axis=1)
        vw = problem.v_hkl[keep].astype(np.int64) % np.array(self.grid)
        v = torch.zeros(n0 * n1 * n2, dtype=torch.complex128, device=device)
        v[torch.from_numpy((vw[:, 0] * n1 + vw[:, 1]) * n2 + vw[:, 2]).to(device)] = torch.from_numpy(
            problem.v_values[keep]).to(device)
        self.v = (torch.fft.ifftn(v.reshape(self.grid)) * float(np.prod(self.grid))).real
        self.b = torch.from_numpy(problem.all_b()).to(device)
        self.bt, self.bc = self.b.T.contiguous(), self.b.conj().resolve_conj().contiguous()
        self.d = torch.from_numpy(problem.block_d()).to(device)
        self.q = torch.from_numpy(problem.block_q()).to(device)

    def local(self, x):
        out = x * self.kinetic
        count = float(np.prod(self.grid))
        for c in range(0, x.shape[0], 16):
            g = torch.zeros((min(16, x.shape[0] - c), int(count)), dtype=torch.complex128, device=self.device)
            g[:, self.index] = x[c:c + 16]
            r = torch.fft.ifftn(g.reshape(-1, *self.grid), dim=(1, 2, 3)) * self.v
            out[c:c + 16] += torch.fft.fftn(r, dim=(1, 2, 3)).reshape(g.shape)[:, self.index]
        return out

    def nonlocal_pair(self, x):
        p = x @ self.bt  # columns x projectors
        return (p @ self.d.T.contiguous()) @ self.bc, (p @ self.q.T.contiguous()) @ self.bc

    def pair(self, x):
        h, s = self.nonlocal_pair(x)
        return self.local(x) + h, (1.0 + self.p.regularization) * x + s


def _plain_solve(problem, roots, device):
    """Lowest pairs of the dense pencil; bands are rows."""
    op = _Plain(problem, device)
    eye = torch.eye(problem.n, dtype=torch.complex128, device=device)
    h, s = op.pair(eye)
    h, s = h.T.cpu(), s.T.cpu()
    h, s = 0.5 * (h + h.conj().T), 0.5 * (s + s.conj().T)
    factor = torch.linalg.cholesky(s)
    c = torch.linalg.solve_triangular(factor, h, upper=False)
    c = torch.linalg.solve_triangular(factor, c.conj().T.resolve_conj(), upper=False)
    w, y = torch.linalg.eigh(0.5 * (c + c.conj().T))
    v = torch.linalg.solve_triangular(factor.conj().T.resolve_conj(), y[:, :roots].contiguous(), upper=True)
    return w[:roots].numpy(), v.T.contiguous()


def _plain_density(problem, bands, f, support):
    """FFT of sum_b f_b |psi_b(r)|^2 / volume on an alias-free grid."""
    span = problem.hkl.max(axis=0) - problem.hkl.min(axis=0)
    grid = tuple(int(2 * max(int(span[a]), int(np.abs(support[:, a]).max())) + 1) for a in range(3))
    wrap = problem.hkl.astype(np.int64) % np.array(grid)
    index = (wrap[:, 0] * grid[1] + wrap[:, 1]) * grid[2] + wrap[:, 2]
    count = int(np.prod(grid))
    rho = np.zeros(grid)
    for band, occupation in zip(bands.numpy(), f):
        g = np.zeros(count, dtype=np.complex128)
        g[index] = band
        rho += occupation * np.abs(np.fft.ifftn(g.reshape(grid)) * count) ** 2
    rho /= abs(float(np.linalg.det(problem.cell.lattice)))
    at = support.astype(np.int64) % np.array(grid)
    return (np.fft.fftn(rho) / count)[at[:, 0], at[:, 1], at[:, 2]]


def exact(case, seed):
    kind = case["kind"]
    device = "cuda" if torch.cuda.is_available() else "cpu"
    if kind == "kpoints":
        hs, ss = [], []
        for i, k in enumerate(_mesh(case)):
            p = _problem(case, seed, k)
            h, s = _Plain(p, device).pair(_block(p, case["columns"], seed * 64 + i).to(device))
            hs.append(h.T.cpu().numpy())
            ss.append(s.T.cpu().numpy())
        return dict(h=hs, s=ss)
    problem = _problem(case, seed)
    if kind in ("apply", "accel"):
        op = _Plain(problem, device)
        x = _block(problem, case["columns"], seed).to(device)
        if kind == "accel":
            h, s = op.nonlocal_pair(x)
            return dict(local=op.local(x).T.cpu().numpy(), h=h.T.cpu().numpy(), s=s.T.cpu().numpy())
        h, s = op.pair(x)
        return {"pair": dict(h=h, s=s), "h": dict(h=h), "s": dict(s=s)}[case["which"]]
    if problem.n > 2000:
        return None  # the dense pencil takes too long
    energies, bands = _plain_solve(problem, case["roots"], device)
    f = _occupations(energies, _atoms(case["cell"]))
    if kind == "scf":
        return dict(eigenvalues=energies, converged=None,
                    density=_plain_density(problem, bands, f, problem.v_hkl))
    x = _block(problem, case["roots"], seed)
    return dict(eigenvalues=energies, converged=None,
                aligned=((x @ bands.conj().T) * torch.from_numpy(f)) @ bands)
