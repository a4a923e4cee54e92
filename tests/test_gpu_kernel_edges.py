"""Kernels at the sizes where their tiles, paddings and dispatch rules change.

The bounds are the repository's: mixed predictions within 1e-4 of the FP64
path (energy relative, forces relative RMS), FP64 results within 1e-10 of the
oracle or of the general path.
"""
import json

import numpy as np
import pytest

from conftest import soap_hypers
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
