"""Launch shapes chosen by size give the same bits on both sides of their line."""
from __future__ import annotations

import numpy as np
import pytest

from nuclearmpm_amd import MaterialModel, MPMBatch, MPMSimulation, Particles
from nuclearmpm_amd.sim import SceneSpec

pytestmark = pytest.mark.gpu


def _cloud(dim, n, seed, identity_mode=1):
    rng = np.random.default_rng(seed)
    p = Particles.from_positions((0.2 + 0.5 * rng.random((n, dim))).astype(np.float32), identity_mode=identity_mode)
    p.v = rng.normal(0, 2.0, p.v.shape).astype(np.float32)
    p.C = rng.normal(0, 5.0, p.C.shape).astype(np.float32)
    p.F = (p.F + rng.normal(0, 0.01, p.F.shape)).astype(np.float32)
    return p


@pytest.mark.parametrize("material,svd", [(MaterialModel.kJelly, "exact"), (MaterialModel.kSnow, "accurate")])
def test_3d_p2g_one_particle_per_thread_is_bitwise_the_same(material, svd):
    """3D P2G takes one particle per thread below 1024 full work items (524,288 particles at
    chunk 512) and 256 threads above: a scene below the line alone and in a batch above it."""
    opts = dict(identity_mode=1, svd=svd, p2g_chunk=512)
    line = 1024 * 512
    a, b = _cloud(3, 777, 1), _cloud(3, line - 500, 2)
    with MPMBatch([SceneSpec(a, material, 64), SceneSpec(b, material, 64)], **opts) as batch:
        batch.advance(2)
        got = batch.particles(1)
    with MPMSimulation(b, material, 64, **opts) as sim:
        sim.advance(2)
        ref = sim.particles()
    for k in ("x", "v", "F", "C", "Jp"):
        assert np.array_equal(getattr(got, k), getattr(ref, k)), k
