"""Kernels at the sizes where their tiles, paddings and dispatch rules change.

The bounds are the repository's: mixed predictions within 1e-4 of the FP64
path (energy relative, forces relative RMS), FP64 results within 1e-10 of the
oracle or of the general path.
"""
import json

import numpy as np
import pytest
import torch

import oracle as O
from conftest import oracle_backward, ps_rel, soap_hypers
from librascal_amd import _capi
from librascal_amd.models import KRR, Kernel, SparsePoints
from librascal_amd.representations import SphericalInvariants
from librascal_amd.synthetic import pack, periodic_box

pytestmark = pytest.mark.gpu


def _context(hp, structures):
    ctx = _capi.Context(json.dumps(hp))
    off, pos, num, cells, pbc = pack(structures)
    ctx.set_structures(off, pos, num, cells, pbc, sorted(set(num.tolist())))
    return ctx, num


def _points(ctx, num, counts, rng):
    """counts[z] rows of the batch's features per species z, jittered."""
    X, _ = ctx.features()
    species = np.concatenate([np.full(m, z, np.int32) for z, m in counts.items()])
    values = np.concatenate([X[rng.choice(np.where(num == z)[0], m)] for z, m in counts.items()])
    values = values + 1e-3 * rng.normal(size=values.shape)
    perm = rng.permutation(len(species))
    return species[perm], values[perm], rng.normal(size=len(species))


@pytest.mark.parametrize("m1,m8", [(1, 33), (31, 32), (127, 129), (160, 1)])
def test_mixed_products_at_uneven_sparse_counts(m1, m8):
    """The force product pads each species' sparse points to whole K steps of
    32 with zeros: counts around a step, a column tile and one point."""
    sts = periodic_box(150, 0.05, (1, 8), d_min=1.0, seed=51)
    ctx, num = _context(soap_hypers(rc=4.0, sw=0.5, sigma=0.5, N=6, L=4, spline=1e-8), sts)
    # a point of a species outside the batch takes no column
    rng = np.random.default_rng(52)
    spec, vals, w = _points(ctx, num, {1: m1, 8: m8}, rng)
    spec, vals, w = np.append(spec, 9).astype(np.int32), np.vstack([vals, vals[:1]]), np.append(w, 1.0)
    ctx.set_sparse_points(3, spec, vals, w)
    e, g, _ = ctx.gap_predict()
    ctx.set_precision(_capi.MIXED)
    em, gm, _ = ctx.gap_predict()
    assert abs(em[0] - e[0]) <= 1e-4 * abs(e[0])
    assert np.sqrt(np.mean((gm - g) ** 2)) <= 1e-4 * np.sqrt(np.mean(g ** 2))


def test_model_kept_across_batches():
    """A loaded model stays in the context while batches share the species
    list, and is loaded again after a batch (or an empty layout batch) with
    another list or another model: every prediction equals a fresh
    calculator's bit for bit."""
    def calculator():
        return SphericalInvariants(interaction_cutoff=3.5, cutoff_smooth_width=0.5, max_radial=4,
                                   max_angular=3, gaussian_sigma_type="Constant")

    a = periodic_box(40, 0.05, (1, 8), d_min=1.0, seed=61)
    b = periodic_box(51, 0.05, (1, 8), d_min=1.0, seed=62)
    other = periodic_box(30, 0.05, (1, 6), d_min=1.0, seed=63)
    def model(rep, seed, species=(1, 8)):
        r = np.random.default_rng(seed)
        D = rep.get_num_coefficients(len(species))
        pts = SparsePoints.from_arrays(rep, species, np.repeat(species, 5), r.normal(size=(5 * len(species), D)))
        ker = Kernel(rep, name="GAP", kernel_type="Sparse", target_type="Structure", zeta=2)
        return KRR(r.normal(size=5 * len(species)), ker, pts, {z: 0.0 for z in (1, 6, 8)})

    rep = calculator()
    m1, m2, m3 = model(rep, 1), model(rep, 2), model(rep, 3, (1, 6))
    for m, seed, sp, frames in ((m1, 1, (1, 8), a), (m1, 1, (1, 8), b), (m3, 3, (1, 6), other),
                                (m1, 1, (1, 8), a), (m2, 2, (1, 8), b), (m1, 1, (1, 8), b)):
        got = m.predict_energy_forces_stress(rep.transform(frames))
        fresh = calculator()
        want = model(fresh, seed, sp).predict_energy_forces_stress(fresh.transform(frames))
        for x, y in zip(got, want):
            assert np.array_equal(x, y)
    # a batch of another list set in between without a prediction
    rep.transform(other)
    m1.predict(rep.transform(a))


@pytest.mark.parametrize("n_species,N,L,normalize", [
    (1, 1, 0, True), (3, 5, 4, True), (3, 5, 4, False), (2, 3, 11, True),
    (8, 8, 2, True), (9, 8, 2, True),    # 64 and 72 rows: one and two row blocks
    (12, 8, 1, True), (13, 8, 1, True),  # 96 and 104 rows: triangles in LDS or gathered
])
def test_fp64_rows_and_channels(n_species, N, L, normalize):
    """FP64 features, adjoint and prediction at the edges of the symmetric
    rows: lanes per row block, channel buffers, l_max past 9, one function."""
    el = list(range(1, n_species + 1))
    sts = periodic_box(3 * n_species + 5, 0.06, el, d_min=1.0, seed=70 + n_species)
    hp = soap_hypers(rc=3.5, sw=0.5, sigma=0.5, N=N, L=L, spline=1e-8, normalize=normalize)
    ctx, num = _context(hp, sts)
    calc, batch = O.Calculator(hp), O.BatchData(sts)
    X, _ = ctx.features()
    Xo, _ = calc.power_spectrum(batch)
    assert ps_rel(Xo, X, n_species, N, L) <= 1e-10
    rng = np.random.default_rng(71)
    G = rng.normal(size=X.shape)
    g, s = ctx.features_backward(G)
    g_ref, s_ref = oracle_backward(calc, batch, G)
    # (a single normalised function is 1 everywhere: the reference is exactly
    # zero there, and rounding of the O(1) terms that cancel is not)
    floor = 1e-14 * np.abs(G).max()
    assert np.abs(g - g_ref).max() <= 1e-10 * np.abs(g_ref).max() + floor
    assert np.abs(s - s_ref).max() <= 1e-10 * np.abs(s_ref).max() + floor
    spec, vals, w = _points(ctx, num, {z: 1 + 20 * (z % 2) for z in el}, rng)
    ctx.set_sparse_points(2, spec, vals, w)
    e, g, s = ctx.gap_predict()
    e_ref, g_ref, s_ref = O.gap_predict(calc, batch, O.SparseSet(spec, vals, 2), w)
    floor = 1e-14 * np.abs(w).sum()
    for a, b in ((e, e_ref), (g, g_ref), (s, s_ref)):
        assert np.abs(a - b).max() <= 1e-10 * np.abs(b).max() + floor
    k = ctx.gap_knm("Atom")
    assert np.abs(k - O.gap_knm(calc, batch, O.SparseSet(spec, vals, 2), "Atom")[:, np.argsort(np.argsort(
        spec, kind="stable"))]).max() <= 1e-10 * np.abs(k).max()


@pytest.mark.parametrize("atoms,points", [(3, 1), (40, 65), (700, 33), (1100, 330)])
def test_fp64_product_tiles(atoms, points):
    """The FP64 products in 16-, 32- and 64-row tiles, with remainders in
    every dimension: energies and forces against the oracle's K_NM and against
    the sum over halves of the model."""
    sts = periodic_box(atoms, 0.05, (1, 8), d_min=1.0, seed=81)
    ctx, num = _context(soap_hypers(rc=4.0, sw=0.5, sigma=0.5, N=9, L=6, spline=1e-8), sts)
    rng = np.random.default_rng(82)
    spec, vals, w = _points(ctx, num, {1: points, 8: points + 2}, rng)
    ctx.set_sparse_points(3, spec, vals, w)
    e, g, s = ctx.gap_predict()
    k = ctx.gap_knm("Structure")
    assert abs(k[0] @ w - e[0]) <= 1e-10 * (np.abs(k[0]) @ np.abs(w))
    X, _ = ctx.features()
    z = num[:, None] == spec[None, :]
    ref = np.where(z, (X @ vals.T) ** 3, 0.0)
    assert np.abs(ctx.gap_knm("Atom") - ref).max() <= 1e-10 * np.abs(ref).max()
    parts = []
    for sl in (slice(0, None, 2), slice(1, None, 2)):
        ctx.set_sparse_points(3, spec[sl], vals[sl], w[sl])
        parts.append(ctx.gap_predict())
    for a, b, c in zip((e, g, s), *parts):
        assert np.abs(a - b - c).max() <= 1e-10 * max(np.abs(b).max(), np.abs(c).max())


def _rows_backward(ctx, G, volume):
    """dL/dr and neg stress of one structure from its exported gradient rows."""
    off, j, vec = ctx.neighbours()[:3]
    f = np.einsum("pxd,pd->px", ctx.features_gradient().reshape(len(j), 3, -1),
                  np.repeat(G, np.diff(off), axis=0))
    g = np.zeros((len(off) - 1, 3))
    np.add.at(g, j, f)
    s = [-(vec[:, a] * f[:, b]).sum() / volume for a, b in ((0, 0), (1, 1), (2, 2), (1, 2), (2, 0), (0, 1))]
    return g, np.array([s])


@pytest.mark.parametrize("N,L", [(1, 0), (4, 4), (5, 5), (6, 6), (7, 7), (11, 9), (13, 4), (17, 9), (24, 2), (8, 10)])
def test_pair_forces_by_wavefronts(N, L):
    """The pair phase at the edges of its channel counts (4, 6, .. 24) and of
    the orders side by side (l_max 4, 6, 9; past 9 the general kernel), with
    more than 64 neighbours per centre: one structure, whose centres take four
    wavefronts each, against the oracle, and enough copies of it that centres
    take two or one against the one.  More functions than 16 use
    the DVR basis and the exported gradient rows: the overlap of so many GTOs
    is singular to rounding, and their orthonormal basis not determined."""
    sts = periodic_box(13, 0.08, (1, 8), d_min=1.0, seed=91)
    hp = soap_hypers(rc=6.0, sw=0.5, sigma=0.5, N=N, L=L, spline=1e-8, normalize=False)
    if N > 16:
        hp["radial_contribution"]["type"] = "DVR"
    ctx, _ = _context(hp, sts)
    X, _ = ctx.features()
    G = np.random.default_rng(92).normal(size=X.shape)
    g, s = ctx.features_backward(G)
    if N > 16:
        g_ref, s_ref = _rows_backward(ctx, G, 13 / 0.08)
    else:
        g_ref, s_ref = oracle_backward(O.Calculator(hp), O.BatchData(sts), G)
    assert np.abs(g - g_ref).max() <= 1e-10 * np.abs(g_ref).max()
    assert np.abs(s - s_ref).max() <= 1e-10 * np.abs(s_ref).max()
    for copies in (512 // 13 + 2, 2048 // 13 + 1):
        many, _ = _context(hp, sts * copies)
        gm, sm = many.features_backward(np.tile(G, (copies, 1)))
        assert np.abs(gm.reshape(copies, *g.shape) - g).max() <= 1e-10 * np.abs(g).max()
        assert np.abs(sm.reshape(copies, *s.shape) - s).max() <= 1e-10 * np.abs(s).max()
        assert len(set(map(bytes, gm.reshape(copies, *g.shape)))) == 1
    if L < 10 and N < 17:
        # the mixed path's key contraction before the same phase
        ctx.set_precision(_capi.MIXED)
        gm, _ = ctx.features_backward(G)
        assert np.sqrt(np.mean((gm - g) ** 2)) <= 1e-4 * np.sqrt(np.mean(g ** 2))



@pytest.mark.parametrize("N,L", [(1, 0), (4, 4), (5, 5), (7, 7), (11, 9), (13, 4), (24, 2), (8, 10)])
def test_expansion_by_wavefronts(N, L):
    """The expansion with a wavefront per centre (from 2048 centres on) against
    the per-entry kernel on one of its copies: centres with more than 64
    neighbours, an isolated atom, a species without neighbours, edges of the
    channel counts and orders; FP64 to rounding, FP32 as between the kernels
    elsewhere."""
    sts = periodic_box(12, 0.08, (1, 8), d_min=1.0, seed=93)
    sts = sts + [dict(sts[0], positions=np.zeros((1, 3)), numbers=np.array([6], np.int32),
                      cell=100 * np.eye(3))]
    hp = soap_hypers(rc=6.0, sw=0.5, sigma=0.5, N=N, L=L, spline=1e-8)
    if N > 16:
        hp["radial_contribution"]["type"] = "DVR"
    copies = 2048 // 13 + 1
    one, _ = _context(hp, sts)
    many, _ = _context(hp, sts * copies)
    for prec, tol in ((_capi.FP64, 1e-13), (_capi.MIXED, 1e-6)):
        one.set_precision(prec)
        many.set_precision(prec)
        one.compute()
        many.compute()
        c, km = one.expansion()
        cm, kmm = many.expansion()
        assert np.array_equal(kmm.reshape(copies, -1), np.tile(km, (copies, 1)))
        assert np.abs(cm.reshape(copies, *c.shape) - c).max() <= tol * np.abs(c).max()


@pytest.mark.parametrize("species,atoms,N,L,spline,normalize,zeta,points", [
    ((1, 8), 40, 8, 6, 1e-8, True, 2, {1: 3, 8: 2, 9: 1}),
    ((1, 8), 33, 5, 4, None, True, 3, {1: 2, 8: 3}),
    ((1, 8), 30, 4, 10, 1e-8, False, 1, {1: 2, 8: 1}),
    ((1, 8), 31, 6, 3, 1e-8, True, 2, {8: 4}),
    (tuple(range(1, 14)), 52, 8, 1, 1e-8, True, 2, {1: 2, 7: 1}),
    ((6,), 1500, 12, 9, 1e-8, True, 2, {6: 40}),
])
def test_knm_gradient_columns(species, atoms, N, L, spline, normalize, zeta, points):
    """K_NM gradient columns, formed several sparse points at a time, against
    the adjoint of each column's own dL/dX: columns of one species and of
    several, of a species outside the batch and of one without points, several
    workspaces full, triangles past the LDS, the general pair kernel."""
    sts = periodic_box(atoms, 0.05, species, d_min=1.0, seed=95)
    hp = soap_hypers(rc=3.5, sw=0.5, sigma=0.5, N=N, L=L, spline=spline, normalize=normalize)
    ctx, num = _context(hp, sts)
    rng = np.random.default_rng(96)
    spec, vals, w = _points(ctx, num, {z: m for z, m in points.items() if z in species}, rng)
    if 9 in points and 9 not in species:
        spec, vals, w = np.append(spec, 9).astype(np.int32), np.vstack([vals, vals[:1]]), np.append(w, 1.0)
    ctx.set_sparse_points(zeta, spec, vals, w)
    X, _ = ctx.features()
    out = ctx.gap_knm_gradient(True)
    for m in range(0, len(spec), max(1, len(spec) // 6)):
        scale = np.where(num == spec[m], zeta * (X @ vals[m]) ** (zeta - 1), 0.0)
        g, s = ctx.features_backward(scale[:, None] * vals[m])
        ref = np.concatenate([g.ravel(), s.ravel()])
        assert np.abs(out[:, m] - ref).max() <= 1e-10 * max(np.abs(out).max(), np.abs(ref).max())


@pytest.mark.parametrize("prec", [_capi.FP64, _capi.MIXED])
@pytest.mark.parametrize("n_species,N,L,normalize", [(1, 3, 0, True), (3, 5, 4, False), (4, 12, 9, True)])
def test_features_into_device_rows(prec, n_species, N, L, normalize):
    """Features written straight into a caller's device rows, with and without
    a centre mask, against the host copy: the same values; mixed rows within FP32 rounding of the FP64 ones."""
    sts = periodic_box(41, 0.05, tuple(range(1, n_species + 1)), d_min=1.0, seed=97)
    hp = soap_hypers(rc=3.5, sw=0.5, sigma=0.5, N=N, L=L, spline=1e-8, normalize=normalize)
    off, pos, num, cells, pbc = pack(sts)
    mask = np.random.default_rng(98).random(len(num)) < 0.4
    full = None
    for m in (None, mask):
        ctx = _capi.Context(json.dumps(hp))
        ctx.set_structures(off, pos, num, cells, pbc, sorted(set(num.tolist())), centre_mask=m)
        X64, _ = ctx.features()
        ctx.set_precision(prec)
        X, _ = ctx.features()
        rows = torch.full(X.shape, 7.0, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        ctx.features(out=rows)
        assert np.array_equal(rows.cpu().numpy(), X)
        assert np.abs(X - X64).max() <= (0 if prec == _capi.FP64 else 1e-5) * np.abs(X64).max()
        if m is None:
            full = X
        else:
            assert np.abs(X - full[mask]).max() <= 1e-6 * np.abs(full).max()


@pytest.mark.parametrize("atoms,points", [(66, 65), (520, 300), (2900, 1030)])
def test_mixed_product_tiles(atoms, points):
    """The mixed products in 64 x 64 tiles and, from three quarters of a
    128 x 128 tile per CU on, in those, with remainders of both: energies and
    forces against the FP64 path, and the energy against the K_NM of the same
    context."""
    sts = periodic_box(atoms, 0.05, (1, 8), d_min=1.0, seed=101)
    ctx, num = _context(soap_hypers(rc=4.0, sw=0.5, sigma=0.5, N=9, L=6, spline=1e-8), sts)
    rng = np.random.default_rng(102)
    counts = {z: min(points, int((num == z).sum())) for z in (1, 8)}
    spec, vals, w = _points(ctx, num, counts, rng)
    ctx.set_sparse_points(2, spec, vals, w)
    e, g, s = ctx.gap_predict()
    ctx.set_precision(_capi.MIXED)
    em, gm, sm = ctx.gap_predict()
    k = ctx.gap_knm("Structure")
    assert abs(em[0] - k[0] @ w) <= 1e-4 * (np.abs(k[0]) @ np.abs(w))
    assert abs(em[0] - e[0]) <= 1e-4 * (np.abs(k[0]) @ np.abs(w))
    assert np.sqrt(np.mean((gm - g) ** 2)) <= 1e-4 * np.sqrt(np.mean(g ** 2))


@pytest.mark.parametrize("pairs", [1, 1024, 1025, 32768, 32769])
def test_offsets_at_scan_tiles(pairs):
    """Neighbour lists of isolated pairs of atoms: offsets at one, two and
    many tiles of the one-launch prefix sum and past its largest length."""
    n = 2 * pairs
    pos = np.zeros((n, 3))
    pos[1::2, 0] = 1.0
    ctx = _capi.Context(json.dumps(soap_hypers(rc=2.0, sw=0.5, sigma=0.5, N=1, L=0, spline=1e-8)))
    ctx.set_structures(np.arange(0, n + 1, 2), pos, np.ones(n, np.int32),
                       np.tile((10 * np.eye(3)).ravel(), (pairs, 1)), np.zeros((pairs, 3), np.int32), [1])
    off, j, vec = ctx.neighbours()
    assert np.array_equal(off, 2 * np.arange(n + 1))
    assert np.array_equal(j[0::2], np.arange(n)) and np.array_equal(j[1::2], np.arange(n) ^ 1)
    c, _ = ctx.expansion()
    assert np.all(c == c[0])


@pytest.mark.parametrize("prec,tol", [(_capi.FP64, 1e-10), (_capi.MIXED, 1e-4)])
def test_masked_energies_after_other_predictions(prec, tol):
    """Energies of masked batches on a context that has predicted others
    before, with sparse points for every species: the atoms that the mask
    leaves out contribute nothing, whatever their energies were."""
    sts = periodic_box(60, 0.05, (1, 8), d_min=1.0, seed=12) + periodic_box(37, 0.05, (1, 8), d_min=1.0, seed=13)
    ctx, num = _context(soap_hypers(rc=4.0, sw=0.5, sigma=0.5, N=6, L=4, spline=1e-8), sts)
    off, pos, _, cells, pbc = pack(sts)
    rng = np.random.default_rng(11)
    spec, vals, _ = _points(ctx, num, {1: 7, 8: 9}, rng)
    w = rng.uniform(0.5, 1.5, len(spec))
    ctx.set_precision(prec)
    ctx.set_sparse_points(2, spec, vals, w)
    e_atom = ctx.gap_knm("Atom") @ w
    for mask in (rng.random(len(num)) < 0.5, num == 8, np.zeros(len(num), bool), np.arange(len(num)) < 60):
        ctx.set_structures(off, pos, num, cells, pbc, [1, 8])
        ctx.gap_predict()
        ctx.set_structures(off, pos, num, cells, pbc, [1, 8], centre_mask=mask)
        e = ctx.gap_predict(gradient=False, neg_stress=False)[0]
        ref = np.add.reduceat(np.where(mask, e_atom, 0.0), off[:-1])
        assert np.abs(e - ref).max() <= tol * np.abs(e_atom).sum()


@pytest.mark.parametrize("zeta,N,L,M,where", [
    (1, 4, 2, 2, "all"), (2, 5, 4, 33, "all"), (1, 8, 6, 70, "one entry"), (3, 6, 3, 65, "all"), (1, 1, 3, 4, "all"),
])
def test_kmm_of_points_that_are_not_symmetric(zeta, N, L, M, where):
    """K_MM of sparse points whose diagonal keys' blocks are not symmetric
    (random points, or one entry of one point), of symmetric ones after them
    and of the first again, with a species outside the batch, against the
    oracle."""
    sts = periodic_box(30, 0.05, (1, 8), d_min=1.0, seed=111)
    ctx, num = _context(soap_hypers(rc=3.5, sw=0.5, sigma=0.5, N=N, L=L, spline=1e-8), sts)
    X, _ = ctx.features()
    rng = np.random.default_rng(112)
    spec = np.concatenate([[1, 8, 9], rng.choice([1, 8, 9], M)]).astype(np.int32)
    symmetric = X[rng.choice(len(X), len(spec))]
    points = symmetric.copy()
    if where == "all":
        points = rng.normal(size=points.shape)
    else:
        points[2, 1 * (L + 1)] += 0.5  # key (1, 1), n1 = 0, n2 = 1, l = 0
    for vals in (points, symmetric, points):
        ctx.set_sparse_points(zeta, spec, vals, np.ones(len(spec)))
        ss = O.SparseSet(spec, vals, zeta)
        ref = np.zeros((len(spec), len(spec)))
        ref[np.ix_(ss.order, ss.order)] = O.gap_kmm(ss)
        assert np.abs(ctx.gap_kmm() - ref).max() <= 1e-10 * np.abs(ref).max()


@pytest.mark.parametrize("N,L", [(5, 3), (6, 6), (9, 2), (10, 8)])
def test_expansion_by_wavefronts_of_odd_pairs_of_channels(N, L):
    """The expansion by wavefronts built for 6 and 10 channels, whose rows are
    not whole 16-byte vectors in FP32, against the per-entry kernel; the bounds
    of the test of the other channel counts."""
    sts = periodic_box(12, 0.08, (1, 8), d_min=1.0, seed=121)
    hp = soap_hypers(rc=6.0, sw=0.5, sigma=0.5, N=N, L=L, spline=1e-8)
    copies = 2048 // 12 + 1
    one, _ = _context(hp, sts)
    many, _ = _context(hp, sts * copies)
    for prec, tol in ((_capi.FP64, 1e-13), (_capi.MIXED, 1e-6)):
        one.set_precision(prec)
        many.set_precision(prec)
        one.compute()
        many.compute()
        c, km = one.expansion()
        cm, kmm = many.expansion()
        assert np.array_equal(kmm.reshape(copies, -1), np.tile(km, (copies, 1)))
        assert np.abs(cm.reshape(copies, *c.shape) - c).max() <= tol * np.abs(c).max()


@pytest.mark.parametrize("shape", [(1, 1), (15, 1), (16, 63), (17, 64), (33, 65), (47, 3), (1001, 333)])
def test_gram_of_odd_and_even_columns(shape):
    """A^T A where the rows of A are padded to an even length (an odd number of
    columns) and where they are not, at the edges of the 64-wide tiles and of
    the K steps of 16."""
    A = np.random.default_rng(shape[0]).normal(size=shape)
    ref = A.T @ A
    assert np.abs(_capi.gram_f64(A) - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("spline,L", [(1e-8, 3), (1e-8, 10), (None, 3)])
def test_autotuned_fp64_pair_phase(spline, L):
    """The FP64 autotuner chooses pairs per batch for the general pair phase
    only: the one by wavefronts takes none, and the set reports none."""
    sts = periodic_box(60, 0.05, (1, 8), d_min=1.0, seed=131)
    ctx, _ = _context(soap_hypers(rc=3.5, sw=0.5, sigma=0.5, N=5, L=L, spline=spline), sts)
    X, _ = ctx.features()
    G = np.random.default_rng(132).normal(size=X.shape)
    g, s = ctx.features_backward(G)
    tiles = ctx.autotune()
    assert tiles["pairs_adj"] in ((0,) if spline and L <= 9 else (0, 2, 4, 6, 8, 12, 16, 24, 32))
    gt, st = ctx.features_backward(G)
    assert np.abs(gt - g).max() <= 1e-12 * np.abs(g).max()
    assert np.abs(st - s).max() <= 1e-12 * np.abs(s).max()


def _selection(S, N, L, seed, k=25, repeats=True):
    """k selected coefficients of species pairs a <= b, either order of the
    radial channels, and one of a species outside the batch: the hypers and the
    dense columns of all but that last one."""
    rng = np.random.default_rng(seed)
    a = rng.integers(1, S + 1, k)
    b = np.maximum(a, rng.integers(1, S + 1, k))
    rows = np.stack([a, b, rng.integers(0, N, k), rng.integers(0, N, k), rng.integers(0, L + 1, k)], axis=1)
    if not repeats:
        rows = rng.permutation(np.unique(rows, axis=0))
    a, b, n1, n2, l = rows.T
    key = (a - 1) * S - (a - 1) * (a - 2) // 2 + (b - a)
    sub = {q: v.tolist() + [e] for q, v, e in zip(("a", "b", "n1", "n2", "l"), rows.T, (1, 99, 0, 0, 0))}
    return sub, ((key * N + n1) * N + n2) * (L + 1) + l


@pytest.mark.parametrize("S,N,L,normalize", [(1, 2, 0, True), (2, 5, 3, True), (3, 4, 2, False), (2, 16, 4, True)])
def test_selected_invariants_from_packed_rows(S, N, L, normalize):
    """coefficient_subselection taken from the packed rows: the features, their
    adjoint (several times on one representation, and on the next positions
    through a graph replay) and K_NM gradient against the dense layout.
    (Repeated coefficients without normalisation.)"""
    sts = periodic_box(9 * S + 2, 0.05, tuple(range(1, S + 1)), d_min=1.0, seed=141)
    hp = soap_hypers(rc=3.5, sw=0.5, sigma=0.5, N=N, L=L, spline=1e-8, normalize=False)
    if N > 13:
        hp["radial_contribution"]["type"] = "DVR"
    rng = np.random.default_rng(142)
    sub, col = _selection(S, N, L, 143, repeats=not normalize)
    raw, num = _context(hp, sts)
    sel, _ = _context(dict(hp, normalize=normalize, coefficient_subselection=sub), sts)
    sel.enable_graphs()
    pos = pack(sts)[1]
    for step in range(2):
        for c in (raw, sel):
            c.update_positions(pos * (1 - 0.02 * step))
            c.compute()
        P, _ = raw.features()
        p = np.hstack([P[:, col], np.zeros((len(num), 1))])
        norm = np.linalg.norm(p, axis=1, keepdims=True) if normalize else np.ones((len(num), 1))
        X, _ = sel.features()
        assert np.abs(X - p / norm).max() <= 1e-12 * np.abs(p / norm).max()

        def backward(G):
            # dL/dp of the selection, summed into the dense columns
            g = (G - X * (X * G).sum(1, keepdims=True)) / norm if normalize else G
            dense = np.zeros(P.shape)
            np.add.at(dense.T, col, g[:, :-1].T)
            return raw.features_backward(dense)

        for _ in range(2):
            G = rng.normal(size=X.shape)
            for x, y in zip(backward(G), sel.features_backward(G)):
                assert np.abs(x - y).max() <= 1e-10 * np.abs(x).max()
        T = X[:3] + 0.01
        sel.set_sparse_points(2, num[:3], T, np.ones(3))
        out = sel.gap_knm_gradient()
        ref = np.stack([backward(np.where(num == num[m], 2 * (X @ T[m]), 0.0)[:, None] * T[m])[0].ravel()
                        for m in range(3)], axis=1)
        assert np.abs(out - ref).max() <= 1e-10 * np.abs(ref).max()


@pytest.mark.parametrize("S,N,L", [(1, 1, 0), (2, 3, 2)])
def test_adjoint_of_repeated_selections(S, N, L):
    """Normalised features whose selection repeats coefficients: the adjoint
    against the dense layout's (repeated entries of dL/dX add up; the
    normalisation's part is over the selection's own entries)."""
    sts = periodic_box(9 * S + 2, 0.05, tuple(range(1, S + 1)), d_min=1.0, seed=151)
    hp = soap_hypers(rc=3.5, sw=0.5, sigma=0.5, N=N, L=L, spline=1e-8, normalize=False)
    sub, col = _selection(S, N, L, 152, k=60)
    raw, num = _context(hp, sts)
    sel, _ = _context(dict(hp, normalize=True, coefficient_subselection=sub), sts)
    P, _ = raw.features()
    p = np.hstack([P[:, col], np.zeros((len(num), 1))])
    norm = np.linalg.norm(p, axis=1, keepdims=True)
    X, _ = sel.features()
    assert np.abs(X - p / norm).max() <= 1e-12
    G = np.random.default_rng(153).normal(size=X.shape)
    g = (G - X * (X * G).sum(1, keepdims=True)) / norm
    dense, scale = np.zeros(P.shape), np.zeros(P.shape)
    np.add.at(dense.T, col, g[:, :-1].T)
    np.add.at(scale.T, col, (np.abs(G) / norm)[:, :-1].T)
    # (a single function's reference is zero but for rounding)
    for x, y, s in zip(raw.features_backward(dense), sel.features_backward(G), raw.features_backward(scale)):
        assert np.abs(x - y).max() <= 1e-10 * np.abs(x).max() + 1e-13 * np.abs(s).max()


@pytest.mark.parametrize("S,N,L", [(6, 12, 9), (10, 6, 12), (8, 8, 8), (13, 2, 3)])
def test_mixed_power_spectrum_of_many_species(S, N, L):
    """Key blocks per pass of the mixed power spectrum on both sides of its
    rule (few large passes, many small ones, all keys in one): the features
    within FP32 rounding of the FP64 ones."""
    sts = periodic_box(3 * S + 1, 0.05, tuple(range(1, S + 1)), d_min=1.0, seed=161)
    ctx, _ = _context(soap_hypers(rc=3.5, sw=0.5, sigma=0.5, N=N, L=L, spline=1e-8), sts)
    X, _ = ctx.features()
    ctx.set_precision(_capi.MIXED)
    Xm, _ = ctx.features()
    assert np.abs(Xm - X).max() <= 1e-5 * np.abs(X).max()


@pytest.mark.parametrize("N,L", [(1, 0), (4, 4), (6, 6), (7, 7), (9, 2), (10, 8), (11, 9), (13, 4), (24, 2), (20, 7)])
def test_expansion_set_to_wavefronts(N, L):
    """The expansion by wavefronts where it is asked for, at every channel
    count it is built for, against the per-entry kernel on the same batch:
    centres with more than 64 neighbours, an isolated atom, a species without
    neighbours."""
    sts = periodic_box(12, 0.08, (1, 8), d_min=1.0, seed=171)
    sts = sts + [dict(sts[0], positions=np.zeros((1, 3)), numbers=np.array([6], np.int32), cell=100 * np.eye(3))]
    hp = soap_hypers(rc=6.0, sw=0.5, sigma=0.5, N=N, L=L, spline=1e-8)
    if N > 16:
        hp["radial_contribution"]["type"] = "DVR"
    ctx, _ = _context(hp, sts * 3)
    for prec, tol in ((_capi.FP64, 1e-13), (_capi.MIXED, 1e-6)):
        ctx.set_precision(prec)
        ctx.set_tiles(fused=0)
        c, km = ctx.expansion()
        ctx.set_tiles(fused=3)
        cw, kmw = ctx.expansion()
        assert np.array_equal(km, kmw)
        assert np.abs(cw - c).max() <= tol * np.abs(c).max()


@pytest.mark.parametrize("n,N,L", [(2047, 3, 9), (2048, 3, 9), (2048, 4, 6), (3072, 4, 6), (3072, 2, 0), (3072, 13, 4)])
def test_expansion_kernel_by_number_of_centres(n, N, L):
    """Both sides of the sizes at which the built-in expansion goes by
    wavefronts: the same coefficients as with either kernel set."""
    pos = np.zeros((n, 3))
    pos[1::2, 0] = 1.0
    pos[0::4, 1] = 0.3
    pos = pos + np.array([5.0, 5.0, 5.0])
    off = np.append(np.arange(0, n, 2), n)
    ctx = _capi.Context(json.dumps(soap_hypers(rc=2.0, sw=0.5, sigma=0.5, N=N, L=L, spline=1e-8)))
    ctx.set_structures(off, pos, np.ones(n, np.int32), np.tile((20 * np.eye(3)).ravel(), (len(off) - 1, 1)),
                       np.zeros((len(off) - 1, 3), np.int32), [1])
    for prec, tol in ((_capi.FP64, 1e-13), (_capi.MIXED, 1e-6)):
        ctx.set_precision(prec)
        c, _ = ctx.expansion()
        for fused in (0, 3):
            ctx.set_tiles(fused=fused)
            assert np.abs(ctx.expansion()[0] - c).max() <= tol * np.abs(c).max()
        ctx.set_tiles()


@pytest.mark.parametrize("S,N,L,normalize", [
    (5, 13, 1, True), (6, 11, 3, True), (3, 23, 10, False),  # 65, 66, 69 rows: own triangles, one shared by two row blocks
    (13, 10, 2, True), (12, 16, 1, True),                    # 130 and 192 rows: three row blocks
    (13, 16, 1, True), (13, 16, 0, False),                   # 208: entries from memory
    (4, 10, 8, True), (7, 8, 6, False),                      # 57 and 86 KB: formed whole in LDS, or packed first
    (2, 20, 12, True), (4, 12, 9, True),                     # past those, own triangles
])
def test_fp64_adjoint_of_wide_rows(S, N, L, normalize):
    """The FP64 adjoint from full rows at the edges of its forms (rows formed
    whole in LDS, a triangle per wavefront or per workgroup, entries from
    memory; the passes and channels of a row over several workgroups, for few
    centres, or one) and the prediction's on the same triangles."""
    sts = periodic_box(2 * S + 3, 0.06, tuple(range(1, S + 1)), d_min=1.0, seed=181)
    hp = soap_hypers(rc=3.5, sw=0.5, sigma=0.5, N=N, L=L, spline=1e-8, normalize=normalize)
    if N > 13:
        hp["radial_contribution"]["type"] = "DVR"
    ctx, num = _context(hp, sts)
    X, _ = ctx.features()
    rng = np.random.default_rng(182)
    G = rng.normal(size=X.shape)
    g, s = ctx.features_backward(G)
    ref = (oracle_backward(O.Calculator(hp), O.BatchData(sts), G) if N <= 13 else
           _rows_backward(ctx, G, (2 * S + 3) / 0.06))
    for x, y in zip((g, s), ref):
        assert np.abs(x - y).max() <= 1e-10 * np.abs(y).max()
    copies = 1024 // len(num) + 2
    many, _ = _context(hp, sts * copies)
    gm, sm = many.features_backward(np.tile(G, (copies, 1)))
    assert np.abs(gm.reshape(copies, *g.shape) - g).max() <= 1e-10 * np.abs(g).max()
    assert np.abs(sm.reshape(copies, *s.shape) - s).max() <= 1e-10 * np.abs(s).max()
    # a linear kernel's prediction is the adjoint of one dL/dX
    T = X[:4] + 0.1 * rng.normal(size=(4, X.shape[1]))
    w = rng.normal(size=4)
    ctx.set_sparse_points(1, num[:4], T, w)
    dX = (num[:, None] == num[None, :4]) @ (w[:, None] * T)
    for x, y in zip(ctx.gap_predict()[1:], ctx.features_backward(dX)):
        assert np.abs(x - y).max() <= 1e-10 * np.abs(y).max()


@pytest.mark.parametrize("S,N,L,spline", [(2, 20, 12, None), (2, 20, 12, 1e-8), (4, 12, 9, None), (10, 8, 10, 1e-8)])
def test_general_pair_phase_of_large_rows(S, N, L, spline):
    """The general pair phase of the FP64 adjoint where two workgroups per CU
    hold four pairs and more, and where one takes the whole LDS: against one
    pair at a time, and against the exported gradient rows."""
    sts = periodic_box(2 * S + 3, 0.06, tuple(range(1, S + 1)), d_min=1.0, seed=191)
    hp = soap_hypers(rc=3.5, sw=0.5, sigma=0.5, N=N, L=L, spline=spline, normalize=False)
    if N > 13:
        hp["radial_contribution"]["type"] = "DVR"
    ctx, _ = _context(hp, sts)
    X, _ = ctx.features()
    G = np.random.default_rng(192).normal(size=X.shape)
    got = ctx.features_backward(G)
    for x, y in zip(got, _rows_backward(ctx, G, (2 * S + 3) / 0.06)):
        assert np.abs(x - y).max() <= 1e-10 * np.abs(y).max()
    ctx.set_tiles(pairs_adj=1)
    for x, y in zip(got, ctx.features_backward(G)):
        assert np.abs(x - y).max() <= 1e-12 * np.abs(y).max()


@pytest.mark.parametrize("species,atoms,points,N,L", [((1, 6, 7, 8), 1003, 17, 12, 9), ((6,), 2890, 2885, 3, 2)])
def test_fp64_products_in_64_row_tiles(species, atoms, points, N, L):
    """The FP64 products past 2048 tiles of 64 x 64, with remainders of rows,
    columns and K steps: the force product (4 species: 184 column tiles of
    features) and the energy and K_NM products (2885 sparse points), against
    numpy and the adjoint of the model's dL/dX."""
    sts = periodic_box(atoms, 0.05, species, d_min=1.0, seed=201)
    ctx, num = _context(soap_hypers(rc=3.5, sw=0.5, sigma=0.5, N=N, L=L, spline=1e-8), sts)
    rng = np.random.default_rng(202)
    spec, vals, w = _points(ctx, num, {z: points for z in species}, rng)
    ctx.set_sparse_points(2, spec, vals, w)
    X, _ = ctx.features()
    dot = np.where(num[:, None] == spec[None, :], X @ vals.T, 0.0)
    assert np.abs(ctx.gap_knm("Atom") - dot ** 2).max() <= 1e-10 * np.abs(dot ** 2).max()
    e, g, s = ctx.gap_predict()
    assert abs(e[0] - (dot ** 2 @ w).sum()) <= 1e-10 * (np.abs(dot ** 2) @ np.abs(w)).sum()
    gr, sr = ctx.features_backward((2 * dot * w) @ vals)
    assert np.abs(g - gr).max() <= 1e-10 * np.abs(gr).max()
    assert np.abs(s - sr).max() <= 1e-10 * np.abs(sr).max()


def test_model_loaded_again_after_other_layouts():
    """Predictions after the context's model was dropped by a batch with another
    species list, or by a K_MM over one, equal a fresh calculator's."""
    def calculator():
        return SphericalInvariants(interaction_cutoff=3.5, cutoff_smooth_width=0.5, max_radial=4,
                                   max_angular=3, gaussian_sigma_type="Constant")

    frames = {sp: periodic_box(30, 0.05, sp, d_min=1.0, seed=210 + sp[-1]) for sp in ((1, 8), (1, 6))}

    def model(rep, sp):
        r = np.random.default_rng(sp[-1])
        pts = SparsePoints.from_arrays(rep, sp, np.repeat(sp, 5), r.normal(size=(10, rep.get_num_coefficients(2))))
        ker = Kernel(rep, name="GAP", kernel_type="Sparse", target_type="Structure", zeta=2)
        return ker, pts, KRR(r.normal(size=10), ker, pts, {z: 0.0 for z in (1, 6, 8)})

    fresh = calculator()
    want = model(fresh, (1, 8))[2].predict_energy_forces_stress(fresh.transform(frames[(1, 8)]))
    rep = calculator()
    _, _, m = model(rep, (1, 8))
    ker, pts, other = model(rep, (1, 6))
    between = (lambda: None, lambda: rep.transform(frames[(1, 6)]),
               lambda: other.predict(rep.transform(frames[(1, 6)])), lambda: ker(pts))
    for do in between:
        do()
        got = m.predict_energy_forces_stress(rep.transform(frames[(1, 8)]))
        for x, y in zip(got, want):
            assert np.array_equal(x, y)
