"""Workloads of the SOAP + sparse-GAP path for timing: what a user of this
framework has it do, with inputs made from a seed and the same results in
plain 64-bit torch beside them.

Kinds of pass (case["kind"]):
  step       one molecular-dynamics step through the C ABI (as the benchmark
             and the MD driver do it): new positions, neighbour list,
             representation, energies, forces and stress of a GAP model
  batch      a model screened over a batch of new structures through the
             Python classes: AtomsList, transform, one prediction
  features   power spectra of a batch as a numpy matrix (transform, get_features)
  expansion  spherical expansion coefficients of a batch (the same, SphericalExpansion)
  soap       features as a device tensor behind autograd, for a network on
             top of them: forward only
  soap_grad  the same with the backward pass to the positions
  knm        training rows of a sparse GAP: K_NM per structure and its
             position gradients (compute_KNM), and K_MM

Structures: atoms on a jittered lattice with vacancies (a minimum separation
of about 1 A, the densities of the repository's benchmark workloads), cubic or
triclinic and periodic, or cube-shaped molecules without periodicity.  Sparse
points are environments of such structures, their features computed here in
64 bits.  The mixed path carries FP32 accuracy, so its callers take float32.
"""
import json
import math

import numpy as np
import torch

from librascal_amd import _capi
from librascal_amd.autograd import soap_features
from librascal_amd.models import KRR, Kernel, SparsePoints, compute_KNM
from librascal_amd.neighbourlist import AtomsList
from librascal_amd.representations import SphericalExpansion, SphericalInvariants

ELEMENTS = (1, 6, 7, 8, 14, 16)
DEV = torch.device("cuda")


def _case(kind, precision, shape, n_struct, n_min, n_max, density, n_species, rc, sigma, n_max_radial,
          l_max, sparse=0, zeta=2):
    return dict(kind=kind, precision=precision, shape=shape, n_struct=n_struct, n_min=n_min, n_max=n_max,
                density=density, n_species=n_species, rc=rc, sigma=sigma, N=n_max_radial, L=l_max,
                sparse=sparse, zeta=zeta)


def listed():
    c = []

    def add(name, *a, **k):
        c.append(dict(_case(*a, **k), name=name))

    # the smallest call: MD of a 64-atom single-species diamond-like cell with
    # a small model, in the library's default precision; latency counts
    add("step_64_fp64", "step", "fp64", "cubic", 1, 64, 64, 0.05, 1, 5.0, 0.5, 8, 6, 100, 2)
    # MD of an ordinary two-species cell in the default precision, 1000
    # sparse points per species (not a multiple of any tile)
    add("step_1024_fp64", "step", "fp64", "cubic", 1, 1024, 1024, 0.05, 2, 5.0, 0.5, 10, 8, 1000, 2)
    # the same model in mixed precision on a cell of an odd size
    add("step_1331_mixed", "step", "mixed", "cubic", 1, 1331, 1331, 0.05, 2, 5.0, 0.5, 10, 8, 1000, 2)
    # the headline workload: 8192 atoms, 4 species, 1024 sparse points each
    add("step_8192_mixed", "step", "mixed", "cubic", 1, 8192, 8192, 0.06, 4, 5.0, 0.5, 12, 9, 1024, 4)
    # its shape in FP64, the reference-accuracy path, half the box and points
    add("step_4096_fp64", "step", "fp64", "cubic", 1, 4096, 4096, 0.06, 4, 5.0, 0.5, 12, 9, 500, 4)
    # screening: a batch of uneven triclinic cells against a loaded model
    add("batch_cells_mixed", "batch", "mixed", "triclinic", 24, 32, 512, 0.06, 3, 6.0, 0.5, 12, 9, 300, 2)
    # plain featurisation of a few single-species cells, FP64, to numpy
    add("features_8x64_fp64", "features", "fp64", "cubic", 8, 64, 64, 0.05, 1, 5.0, 0.5, 8, 6)
    # expansion coefficients of two odd-sized cells, FP64, to numpy
    add("expansion_2x343_fp64", "expansion", "fp64", "cubic", 2, 343, 343, 0.05, 3, 5.0, 0.5, 9, 7)
    # features of a thousand uneven molecules on the device for a float32 network
    add("soap_molecules_mixed", "soap", "mixed", "molecule", 1024, 8, 64, 0.08, 4, 4.0, 0.4, 8, 6)
    # a training step's features and position gradients of molecules, FP64
    add("soap_grad_molecules_fp64", "soap_grad", "fp64", "molecule", 128, 8, 64, 0.08, 4, 4.0, 0.4, 8, 6)
    # GAP training rows with forces of uneven small cells, FP64
    add("knm_cells_fp64", "knm", "fp64", "triclinic", 24, 16, 64, 0.06, 3, 4.5, 0.5, 8, 6, 100, 2)
    return c


def draw(rng):
    def log(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["step", "step", "step", "batch", "features", "expansion", "soap", "soap_grad", "knm"])
    n, l = rng.choice([(6, 5), (8, 6), (9, 7), (10, 8), (12, 9)])
    rc = rng.choice([4.0, 4.5, 5.0])
    ns = rng.randint(1, 4)
    rho = rng.uniform(0.045, 0.065)
    precision = rng.choice(["fp64", "mixed"])
    zeta = rng.randint(1, 4)
    if kind == "step":
        a = log(40, 4000 if precision == "mixed" else 2000)
        return _case(kind, precision, rng.choice(["cubic", "triclinic"]), 1, a, a, rho, ns, rc, 0.5, n, l,
                     log(50, 700), zeta)
    if kind == "batch":
        return _case(kind, precision, "triclinic", log(4, 32), 24, log(48, 200), rho, min(ns, 3), rc, 0.5, n, l,
                     log(50, 250), zeta)
    if kind in ("features", "expansion"):
        return _case(kind, "fp64", rng.choice(["cubic", "triclinic"]), log(1, 12), 40, log(60, 160), rho,
                     min(ns, 2), rc, 0.5, n, l)
    if kind == "soap":
        return _case(kind, precision, "molecule", log(40, 700), 8, 64, 0.08, 4, 4.0, 0.4, 8, 6)
    if kind == "soap_grad":
        return _case(kind, precision, "molecule", log(16, 128), 8, 64, 0.08, rng.randint(2, 4), 4.0, 0.4,
                     rng.choice([6, 8]), rng.choice([5, 6]))
    return _case(kind, "fp64", "triclinic", log(4, 24), 16, 64, rho, min(ns, 3), 4.0, 0.5, rng.choice([6, 8]),
                 rng.choice([5, 6]), log(20, 40), zeta)


# --- structures -------------------------------------------------------------


def _structure(rng, shape, n, density, numbers):
    """One structure of n atoms: jittered lattice sites, some left empty."""
    k = max(1, math.ceil(n ** (1.0 / 3.0) - 1e-9))
    side = (n / density) ** (1.0 / 3.0)
    if shape == "triclinic":
        la, lb, lc = rng.uniform(11.0, 15.0, size=3)
        al, be, ga = np.radians(rng.uniform(75.0, 105.0, size=3))
        cx, cy = math.cos(be), (math.cos(al) - math.cos(be) * math.cos(ga)) / math.sin(ga)
        cell = np.array([[la, lb * math.cos(ga), lc * cx], [0.0, lb * math.sin(ga), lc * cy],
                         [0.0, 0.0, lc * math.sqrt(1.0 - cx * cx - cy * cy)]])
        cell *= (n / density / abs(np.linalg.det(cell))) ** (1.0 / 3.0)
    else:
        cell = np.eye(3) * side
    sites = rng.permutation(k ** 3)[:n]
    frac = (np.stack([sites // (k * k), sites // k % k, sites % k], axis=1) + 0.5) / k
    pos = frac @ cell.T + np.clip(rng.normal(0.0, 0.2, size=(n, 3)), -0.4, 0.4)
    frac = np.linalg.solve(cell, pos.T).T
    frac = np.clip(frac, 0.0, 1.0 - 1e-9) if shape == "molecule" else np.mod(frac, 1.0)
    return dict(positions=np.ascontiguousarray(frac @ cell.T), numbers=numbers.astype(np.int32), cell=cell,
                pbc=np.zeros(3, np.int32) if shape == "molecule" else np.ones(3, np.int32))


def _structures(case, seed, extra=0):
    rng = np.random.Generator(np.random.PCG64([int(seed) % (1 << 63), extra]))
    el = np.asarray(ELEMENTS[:case["n_species"]])
    # the sizes belong to the case, the coordinates and elements to the seed
    sizes = np.random.Generator(np.random.PCG64(extra)).integers(case["n_min"], case["n_max"] + 1,
                                                                 size=case["n_struct"])
    out = []
    for s, n in enumerate(sizes.tolist()):
        num = rng.permutation(el[(np.arange(n) + s) % len(el)])
        out.append(_structure(rng, case["shape"], n, case["density"], num))
    return out, rng


def _species(structures):
    return sorted(set(int(z) for s in structures for z in np.unique(s["numbers"])))


def _calculator(case):
    cls = SphericalExpansion if case["kind"] == "expansion" else SphericalInvariants
    return cls(interaction_cutoff=case["rc"], cutoff_smooth_width=0.5, max_radial=case["N"],
               max_angular=case["L"], gaussian_sigma_type="Constant", gaussian_sigma_constant=case["sigma"])


def _sparse(case, seed, species):
    """Sparse points (numbers, features [M][D]) and weights: environments of
    further structures of the same kind, the same number per species."""
    pool_case = dict(case, n_struct=max(2, math.ceil(1.25 * case["sparse"] * len(species) / case["n_max"])),
                     n_min=case["n_max"])
    pool, rng = _structures(pool_case, seed, extra=1)
    numbers = np.concatenate([s["numbers"] for s in pool])
    pick = [rng.permutation(np.where(numbers == z)[0])[:case["sparse"]] for z in species]
    pick = np.concatenate(pick)
    X = _features(case, pool, species, torch.from_numpy(pick).to(DEV))
    weights = rng.normal(size=len(pick))
    return numbers[pick].astype(np.int32), X, weights


# --- the same in plain 64-bit torch -----------------------------------------


class _Radial:
    """GTO radial functions (orthonormalised) and their derivative."""

    def __init__(self, case, dev):
        N, L, rc = case["N"], case["L"], case["rc"]
        n = torch.arange(N, dtype=torch.float64)
        lg = torch.lgamma
        sig = torch.clamp(n.sqrt(), min=1.0) * rc / N
        self.fa, fb = 0.5 / case["sigma"] ** 2, 0.5 / sig ** 2
        norm = 0.25 * torch.exp(0.5 * (math.log(2.0) - lg(1.5 + n) - (3 + 2 * n) * sig.log()))
        p = 0.5 * (3.0 + n[:, None] + n[None, :])
        S = torch.exp(-p * (fb[:, None] + fb[None, :]).log() - n[:, None] * sig.log()[:, None]
                      - n[None, :] * sig.log()[None, :] + lg(p)
                      - 1.5 * (sig.log()[:, None] + sig.log()[None, :])
                      - 0.5 * (lg(1.5 + n)[:, None] + lg(1.5 + n)[None, :]))
        w, V = torch.linalg.eigh(S)
        self.O = (norm[:, None] * (V @ torch.diag(w.rsqrt()) @ V.T)).to(dev)
        raw0 = torch.exp(lg(0.5 * (3.0 + n)) - lg(torch.tensor(1.5, dtype=torch.float64))
                         - 0.5 * (3.0 + n) * (self.fa + fb).log())
        self.centre = (self.O.T @ raw0.to(dev)) / math.sqrt(4.0 * math.pi)
        l = torch.arange(L + 1, dtype=torch.float64)
        self.a = (0.5 * (n[:, None] + l[None, :] + 3.0)).to(dev)
        self.b = (l + 1.5).to(dev).expand(N, L + 1)
        self.pre = torch.exp(lg(0.5 * (n[:, None] + l + 3.0)) - lg(l + 1.5)
                             - 0.5 * (3.0 + n[:, None] + l) * (self.fa + fb[:, None]).log()).to(dev)
        self.l = l.to(dev)
        self.zz = (self.fa ** 2 / (self.fa + fb)).to(dev)
        self.rc, self.sw = rc, 0.5
        self.terms = int(2.2 * float(self.zz.max()) * rc * rc) + 80

    def __call__(self, r):
        """fc R [P][N][L+1] and d(fc R)/dr."""
        z = (self.zz[None, :, None] * (r * r)[:, None, None]).expand(-1, -1, self.l.numel())
        f, df = torch.ones_like(z), torch.ones_like(z)
        t, dt = torch.ones_like(z), torch.ones_like(z)
        for k in range(self.terms):  # 1F1(a, b, z) and 1F1(a + 1, b + 1, z), all terms positive
            t = t * ((self.a + k) / ((self.b + k) * (k + 1))) * z
            dt = dt * ((self.a + 1 + k) / ((self.b + 1 + k) * (k + 1))) * z
            f, df = f + t, df + dt
        df = df * (self.a / self.b)
        e = torch.exp(-self.fa * r * r)[:, None, None]
        x = (self.fa * r)[:, None, None] ** self.l
        raw = self.pre * e * f * x
        draw = self.pre * e * x * (df * 2.0 * self.zz[:, None] * r[:, None, None] - 2.0 * self.fa * r[:, None, None] * f) \
            + raw * self.l / r[:, None, None]
        R, dR = torch.einsum("mn,pml->pnl", self.O, raw), torch.einsum("mn,pml->pnl", self.O, draw)
        u = (r - self.rc + self.sw) / self.sw
        inner = u <= 0
        fc = torch.where(inner, torch.ones_like(r), 0.5 * (1.0 + torch.cos(math.pi * u)))
        dfc = torch.where(inner, torch.zeros_like(r), -0.5 * math.pi / self.sw * torch.sin(math.pi * u))
        return R * fc[:, None, None], dR * fc[:, None, None] + R * dfc[:, None, None]


class _RadialFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, r, radial):
        R, dR = radial(r)
        ctx.save_for_backward(dR)
        return R

    @staticmethod
    def backward(ctx, g):
        return (ctx.saved_tensors[0] * g).sum(dim=(1, 2)), None


def _ylm(u, L):
    """Real spherical harmonics [P][(L+1)^2] of unit vectors."""
    x, y, z = u[:, 0], u[:, 1], u[:, 2]
    A, B = [torch.ones_like(x)], [torch.zeros_like(x)]
    for m in range(L):
        A, B = A + [x * A[m] - y * B[m]], B + [x * B[m] + y * A[m]]
    out = [None] * ((L + 1) ** 2)
    q = 1.0 / math.sqrt(2.0 * math.pi)
    for m in range(L + 1):
        if m:
            q *= -math.sqrt(1.0 + 0.5 / m)
        p2, p1 = torch.zeros_like(x), q * torch.ones_like(x)
        for l in range(m, L + 1):
            if l > m:
                c = math.sqrt((4.0 * l * l - 1.0) / (l * l - m * m))
                d = math.sqrt(((l - 1.0) ** 2 - m * m) / (4.0 * (l - 1.0) ** 2 - 1.0))
                p2, p1 = p1, c * (z * p1 - d * p2)
            b = l * l + l
            if m == 0:
                out[b] = p1 * math.sqrt(0.5)
            else:
                out[b + m], out[b - m] = p1 * A[m], p1 * B[m]
    return torch.stack(out, dim=1)


def _pairs(structures, rc, dev, centres=None):
    """(i, j, vector) of every pair within the cutoff, sorted by i, without the
    self pairs; atoms numbered over the batch.  centres: only these i."""
    I, J, V = [], [], []
    a0 = 0
    for s in structures:
        pos = torch.from_numpy(s["positions"]).to(dev)
        n = len(pos)
        idx = torch.arange(n, device=dev) if centres is None else centres[(centres >= a0) & (centres < a0 + n)] - a0
        cell = s["cell"]
        inv = np.linalg.inv(cell)
        rep = [int(math.ceil(rc * np.linalg.norm(inv[d]))) if s["pbc"][d] else 0 for d in range(3)]
        grid = np.array([[x, y, z] for x in range(-rep[0], rep[0] + 1) for y in range(-rep[1], rep[1] + 1)
                         for z in range(-rep[2], rep[2] + 1)], np.float64)
        shifts = torch.from_numpy(grid @ cell.T).to(dev)
        step = max(1, int(3e7 // max(1, len(idx) * n)))
        for k in range(0, len(shifts), step):
            sh = shifts[k:k + step]
            d = pos[None, None, :, :] + sh[:, None, None, :] - pos[idx][None, :, None, :]
            d2 = (d * d).sum(-1)
            w, p, q = torch.nonzero((d2 <= rc * rc) & (d2 > 1e-12), as_tuple=True)
            I.append(idx[p] + a0)
            J.append(q + a0)
            V.append(d[w, p, q])
        a0 += n
    i, j, v = torch.cat(I), torch.cat(J), torch.cat(V)
    order = torch.argsort(i, stable=True)
    return i[order], j[order], v[order]


def _expand(case, radial, rows, sp_rows, i, sj, v, S):
    """c [rows][S][N][(L+1)^2]; i: row of each pair, sj its species index."""
    N, L = case["N"], case["L"]
    r = v.norm(dim=1)
    R = _RadialFn.apply(r, radial)
    Y = _ylm(v / r[:, None], L)
    lof = torch.tensor([l for l in range(L + 1) for _ in range(2 * l + 1)], device=v.device)
    c = torch.zeros(rows * S, N, (L + 1) ** 2, dtype=torch.float64, device=v.device)
    c = c.index_add(0, i * S + sj, R[:, :, lof] * Y[:, None, :]).reshape(rows, S, N, -1)
    centre = torch.zeros_like(c)
    centre[torch.arange(rows, device=v.device), sp_rows, :, 0] = radial.centre
    return c + centre


def _power(case, c):
    """Normalised power spectrum [rows][K N^2 (L+1)]."""
    S, L = c.shape[1], case["L"]
    keys = [(a, b) for a in range(S) for b in range(a, S)]
    out = []
    for a, b in keys:
        w = math.sqrt(2.0) if a < b else 1.0
        out.append(torch.stack([torch.matmul(c[:, a, :, l * l:(l + 1) ** 2].contiguous(),
                                             c[:, b, :, l * l:(l + 1) ** 2].transpose(1, 2).contiguous())
                                * (w / math.sqrt(2 * l + 1)) for l in range(L + 1)], dim=-1).flatten(1))
    p = torch.cat(out, dim=1)
    return p / p.norm(dim=1, keepdim=True)


def _chunks(case, structures, species, centres=None):
    """Parts of the batch: (centre atoms, their species, pair row, pair j,
    species of j, pair vectors, radial)."""
    dev = DEV
    num = np.concatenate([s["numbers"] for s in structures])
    sp = torch.from_numpy(np.searchsorted(species, num)).to(dev)
    all_c = torch.arange(len(num), device=dev) if centres is None else torch.unique(centres)
    radial = _Radial(case, dev)
    i, j, v = _pairs(structures, case["rc"], dev, None if centres is None else all_c)
    per = max(1, int(2.5e9 / (8.0 * 60 * case["N"] * (case["L"] + 1) ** 2 * 2)))
    for k in range(0, len(all_c), per):
        part = all_c[k:k + per]
        lo = torch.searchsorted(i, part[0].unsqueeze(0))[0]
        hi = torch.searchsorted(i, part[-1].unsqueeze(0), right=True)[0]
        ii = torch.searchsorted(part, i[lo:hi].contiguous())
        yield part, sp[part], ii, j[lo:hi], sp[j[lo:hi]], v[lo:hi], radial


def _features(case, structures, species, centres):
    """Features of the given atoms of the batch, in their order (numpy)."""
    X = [_power(case, _expand(case, rad, len(part), sp, ii, sj, v, len(species))).cpu().numpy()
         for part, sp, ii, _, sj, v, rad in _chunks(case, structures, species, centres)]
    _, inverse = torch.unique(centres, return_inverse=True)
    return np.ascontiguousarray(np.concatenate(X)[inverse.cpu().numpy()])


def _segments(structures, dev):
    return torch.from_numpy(np.repeat(np.arange(len(structures)), [len(s["numbers"]) for s in structures])).to(dev)


def _volumes(structures, dev):
    return torch.tensor([abs(np.linalg.det(s["cell"])) for s in structures], dtype=torch.float64, device=dev)


VOIGT = ((0, 0), (1, 1), (2, 2), (1, 2), (2, 0), (0, 1))


def _exact_predict(case, structures, species, numbers, T, weights):
    """Energies, dE/dr and the negative stress of the GAP model."""
    dev = DEV
    seg, nat = _segments(structures, dev), sum(len(s["numbers"]) for s in structures)
    E = torch.zeros(len(structures), dtype=torch.float64, device=dev)
    g, vir = torch.zeros(nat, 3, dtype=torch.float64, device=dev), torch.zeros(len(structures), 6, dtype=torch.float64, device=dev)
    Td = [torch.from_numpy(T[numbers == z]).to(dev) for z in species]
    wd = [torch.from_numpy(weights[numbers == z]).to(dev) for z in species]
    for part, sp, ii, j, sj, v, rad in _chunks(case, structures, species):
        v = v.detach().requires_grad_(True)
        X = _power(case, _expand(case, rad, len(part), sp, ii, sj, v, len(species)))
        e = torch.zeros(len(part), dtype=torch.float64, device=dev)
        for s in range(len(species)):
            rows = torch.nonzero(sp == s)[:, 0]
            if len(rows) and len(Td[s]):
                e = e.index_add(0, rows, (X[rows] @ Td[s].T) ** case["zeta"] @ wd[s])
        d, = torch.autograd.grad(e.sum(), v)
        E.index_add_(0, seg[part], e.detach())
        i = part[ii]
        g.index_add_(0, j, d)
        g.index_add_(0, i, -d)
        v = v.detach()
        vir.index_add_(0, seg[i], torch.stack([-v[:, a] * d[:, b] for a, b in VOIGT], dim=1))
    return E.cpu().numpy(), g.cpu().numpy(), (vir / _volumes(structures, dev)[:, None]).cpu().numpy()


def _exact_knm(case, structures, species, numbers, T):
    """K_NM structure rows, then the 3 n_atoms gradient rows, and K_MM."""
    dev = DEV
    seg, nat, M = _segments(structures, dev), sum(len(s["numbers"]) for s in structures), len(numbers)
    K = torch.zeros(len(structures), M, dtype=torch.float64, device=dev)
    dK = torch.zeros(3 * nat, M, dtype=torch.float64, device=dev)
    Td = torch.from_numpy(T).to(dev)
    same = torch.from_numpy(numbers[:, None] == numbers[None, :]).to(dev)
    tsp = torch.from_numpy(np.searchsorted(species, numbers)).to(dev)
    for part, sp, ii, j, sj, v, rad in _chunks(case, structures, species):
        v = v.detach().requires_grad_(True)
        X = _power(case, _expand(case, rad, len(part), sp, ii, sj, v, len(species)))
        k = torch.where(sp[:, None] == tsp[None, :], (X @ Td.T) ** case["zeta"], torch.zeros((), dtype=torch.float64, device=dev))
        K.index_add_(0, seg[part], k.detach())
        i = part[ii]
        for m in range(M):
            d, = torch.autograd.grad(k[:, m].sum(), v, retain_graph=True)
            col = torch.zeros(nat, 3, dtype=torch.float64, device=dev).index_add_(0, j, d).index_add_(0, i, -d)
            dK[:, m] += col.reshape(-1)
    kmm = torch.where(same, (Td @ Td.T) ** case["zeta"], torch.zeros((), dtype=torch.float64, device=dev))
    return torch.cat([K, dK]).cpu().numpy(), kmm.cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    st, _ = _structures(case, seed)
    species = _species(st)
    if kind in ("step", "batch"):
        numbers, T, w = _sparse(case, seed, species)
        e, g, s = _exact_predict(case, st, species, numbers, T, w)
        return dict(energy=e, forces=-g, stress=-s) if kind == "batch" else dict(energy=e, gradient=g, neg_stress=s)
    if kind == "knm":
        numbers, T, _ = _sparse(case, seed, species)
        k, kmm = _exact_knm(case, st, species, numbers, T)
        return dict(knm=k, kmm=kmm)
    parts = list(_chunks(case, st, species))
    if kind == "expansion":
        return dict(c=np.concatenate([_expand(case, rad, len(part), sp, ii, sj, v, len(species)).flatten(1).cpu().numpy()
                                      for part, sp, ii, _, sj, v, rad in parts]))
    dX = _upstream(case, seed, sum(len(part) for part, *_ in parts), len(species)) if kind == "soap_grad" else None
    X, g = [], torch.zeros(sum(len(s["numbers"]) for s in st), 3, dtype=torch.float64, device=DEV)
    for part, sp, ii, j, sj, v, rad in parts:
        v = v.detach().requires_grad_(kind == "soap_grad")
        x = _power(case, _expand(case, rad, len(part), sp, ii, sj, v, len(species)))
        if kind == "soap_grad":
            d, = torch.autograd.grad(x, v, dX[part])
            g.index_add_(0, j, d)
            g.index_add_(0, part[ii], -d)
        X.append(x.detach())
    X = torch.cat(X)
    return dict(X=X, grad=g) if kind == "soap_grad" else dict(X=X)


# --- the framework's side ---------------------------------------------------


def _upstream(case, seed, n, S):
    """dL/dX of a training step: the gradient a network hands back."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(int(seed) % (1 << 62) + 7)
    D = S * (S + 1) // 2 * case["N"] ** 2 * (case["L"] + 1)
    return torch.randn(n, D, dtype=torch.float64, device=DEV, generator=gen)


def prepare(case, seed):
    kind = case["kind"]
    st, _ = _structures(case, seed)
    species = _species(st)
    mixed = case["precision"] == "mixed"
    state = dict(kind=kind, mixed=mixed)
    if kind == "step":
        # an MD program holds a context with the structure and the model loaded
        # and the neighbour-list pass and representation stage kept as graphs
        numbers, T, w = _sparse(case, seed, species)
        ctx = _capi.Context(json.dumps(_calculator(case).hypers))
        if mixed:
            ctx.set_precision(_capi.MIXED)
        ctx.enable_graphs(True)
        start = st[0]
        off = np.array([0, len(start["numbers"])], np.int64)
        ctx.set_structures(off, start["positions"], start["numbers"], start["cell"][None], start["pbc"][None], species)
        ctx.set_sparse_points(case["zeta"], numbers, T, w)
        ctx.update_positions(start["positions"])
        ctx.gap_predict()
        state.update(ctx=ctx, positions=start["positions"])
        return state
    rep = _calculator(case)
    rep.set_precision(case["precision"])
    state.update(rep=rep, frames=st)
    if kind in ("batch", "knm"):
        numbers, T, w = _sparse(case, seed, species)
        points = SparsePoints.from_arrays(rep, species, numbers, T)
        kernel = Kernel(rep, name="GAP", kernel_type="Sparse", target_type="Structure", zeta=case["zeta"])
        state.update(kernel=kernel, points=points)
        if kind == "batch":
            model = KRR(w, kernel, points, {z: 0.0 for z in species})
            # the model was last used on another batch of the same species
            model.predict_energy_forces_stress(rep.transform(_structures(case, seed, extra=2)[0]))
            state.update(model=model)
    elif kind in ("soap", "soap_grad"):
        atoms = rep.transform(AtomsList(st, rep.nl_options))
        pos = torch.from_numpy(atoms.positions.copy()).to(DEV)
        state.update(atoms=atoms, positions=pos.requires_grad_(kind == "soap_grad"))
        if kind == "soap_grad":
            state.update(dX=_upstream(case, seed, len(pos), len(species)))
    return state


def run(state):
    kind, mixed = state["kind"], state["mixed"]
    if kind == "step":
        ctx = state["ctx"]
        ctx.update_positions(state["positions"])
        out = ctx.gap_predict()
        if mixed:
            out = [x.astype(np.float32) for x in out]
        return dict(zip(("energy", "gradient", "neg_stress"), out))
    rep = state["rep"]
    if kind == "batch":
        out = state["model"].predict_energy_forces_stress(rep.transform(state["frames"]))
        if mixed:
            out = [x.astype(np.float32) for x in out]
        return dict(zip(("energy", "forces", "stress"), out))
    if kind == "features":
        return dict(X=rep.transform(state["frames"]).get_features(rep))
    if kind == "expansion":
        return dict(c=rep.transform(state["frames"]).get_features(rep))
    if kind == "knm":
        return dict(knm=compute_KNM(state["frames"], state["points"], state["kernel"], rep),
                    kmm=state["kernel"](state["points"]))
    X = soap_features(state["positions"], rep, state["atoms"])
    if kind == "soap":
        return dict(X=X.float() if mixed else X)
    g, = torch.autograd.grad(X, state["positions"], state["dX"])
    X = X.detach()
    return dict(X=X.float(), grad=g.float()) if mixed else dict(X=X, grad=g)


def work(case):
    """What a pass cannot do without: positions in, the model read once, the
    results out; the multiply-adds of the expansion over the pairs, of the
    power spectrum (symmetric blocks once), of the kernel and of their
    derivatives (as much again each)."""
    kind, N, L1, S = case["kind"], case["N"], case["L"] + 1, case["n_species"]
    n = case["n_struct"] * 0.5 * (case["n_min"] + case["n_max"])
    pairs = n * case["density"] * 4.0 / 3.0 * math.pi * case["rc"] ** 3 * (0.5 if case["shape"] == "molecule" else 1.0)
    size = 4.0 if case["precision"] == "mixed" else 8.0
    D = S * (S + 1) // 2 * N * N * L1
    Dp = S * N * (N + 1) // 2 * L1 + S * (S - 1) // 2 * N * N * L1
    expand, power = 2.0 * pairs * N * L1 * L1, 2.0 * n * Dp * L1
    M = case["sparse"] * S
    bytes_, flops = 24.0 * n, expand + power
    if kind == "expansion":
        return dict(bytes=bytes_ + 8.0 * n * S * N * L1 * L1, flops=expand)
    if kind == "features":
        return dict(bytes=bytes_ + 8.0 * n * D, flops=flops)
    if kind == "soap":
        return dict(bytes=bytes_ + size * n * D, flops=flops)
    if kind == "soap_grad":
        return dict(bytes=2 * bytes_ + (size + 8.0) * n * D, flops=flops + 2.0 * power + 4.0 * expand)
    bytes_ += size * M * Dp
    if kind == "knm":
        # each gradient row's column: its adjoint over the centres of its species
        cols = M / S
        return dict(bytes=bytes_ + 8.0 * M * (3.0 * n + case["n_struct"]) + 8.0 * M * M,
                    flops=flops + 2.0 * n * cols * Dp + 2.0 * M * cols * Dp + cols * (2.0 * power + 4.0 * expand))
    return dict(bytes=bytes_ + 24.0 * n, flops=flops + 4.0 * n * case["sparse"] * Dp + 2.0 * power + 4.0 * expand)
