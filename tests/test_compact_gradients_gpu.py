"""Gradients of rollouts whose forward pass takes the compact step.

The compact step leaves its slots along a Hilbert curve; the backward pass recomputes with tiled steps, which order them
by tile.  Cotangents pass between the two in particle order."""
from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O

from nuclearmpm_amd import MaterialModel, MPMBatch, MPMSimulation, Particles, SceneSpec, autodiff
from nuclearmpm_amd._lib import check, lib

pytestmark = pytest.mark.gpu

FIELDS = ("x", "v", "F", "C")


def _cloud(dim, n, seed, lo=0.35, hi=0.65):
    rng = np.random.default_rng(seed)
    p = Particles.from_positions((lo + (hi - lo) * rng.random((n, dim))).astype(np.float32), identity_mode=1)
    p.v = rng.normal(0, 0.5, p.v.shape).astype(np.float32)
    p.F = (p.F + rng.normal(0, 0.02, p.F.shape)).astype(np.float32)
    return p


# res 64 / 15: the whole grid fits the compact step's box; res 100 / 40: it does not, and the launch's end is read back
@pytest.mark.parametrize("dim,n,res", [(2, 2000, 64), (2, 1500, 100), (3, 900, 15), (3, 700, 40)])
@pytest.mark.parametrize("plan", [(None, None, None), (1, None, 0), (None, 0, None)])
def test_gradients_through_compact_steps_match_the_fp64_adjoint(dim, n, res, plan, monkeypatch):
    """Checkpointed, recorded and mixed segments of 4, 4 and 1 steps: every field to 1e-3 of the FP64 chained adjoint,
    the multi-step bound of the tiled step's gradients."""
    p = _cloud(dim, n, seed=dim)
    rng = np.random.default_rng(5)
    cot = {k: rng.normal(size=getattr(p, k).shape).astype(np.float32) for k in FIELDS}
    monkeypatch.setattr(autodiff, "_record_plan", lambda *a: list(plan))
    with MPMSimulation(p, MaterialModel.kJelly, res, E=1e3, identity_mode=1, compact=1) as sim:
        s0 = sim.state_image().requires_grad_(True)
        E = torch.tensor([1e3], dtype=torch.float64, requires_grad=True)
        out = autodiff.rollout(sim, s0, E, steps=9, checkpoint_every=4)
        w = autodiff.pack(*(torch.from_numpy(cot[k]).cuda() for k in FIELDS), Jp=torch.zeros(n, device="cuda"))
        taken = sim.steps_taken
        g0, gE = torch.autograd.grad(out, (s0, E), w)
        assert sim.steps_taken == taken and torch.equal(sim.state_image(), s0)
        # a second pass over the same graph of another rollout: nothing of the first is left in the engine
        out = autodiff.rollout(sim, s0, E, steps=9, checkpoint_every=4)
        again = torch.autograd.grad(out, (s0, E), w)
    assert torch.equal(again[0], g0) and torch.equal(again[1], gE)
    st = O.State(x=p.x, v=p.v, F=p.F, C=p.C, Jp=p.Jp, mass=p.mass, volume=p.volume)
    ref = O.rollout_vjp(st, O.Grads(*(cot[k].astype(np.float64) for k in FIELDS)), 9, O.JELLY, res=res, E=1e3,
                        identity_mode=1)
    for k, g in zip(FIELDS, autodiff.unpack(g0, dim)):
        r = getattr(ref, k)
        e = float(np.abs(g.cpu().numpy().reshape(r.shape) - r).max() / np.abs(r).max())
        assert e < 1e-3, (k, e)
    assert abs(float(gE) - ref.E) <= 1e-3 * abs(ref.E) + 1e-6 * ref.E_abs, (float(gE), ref.E)


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("steps", [1, 2, 5])
def test_segment_in_particle_order_is_the_segment_in_slot_order(dim, steps):
    """mpm_backward_segment_particles is mpm_backward_segment between two re-indexings, bit for bit, in place too."""
    specs = [SceneSpec(_cloud(dim, 700 + 300 * s, 7 + s), MaterialModel.kSnow, 48, E=1e3) for s in range(2)]
    with MPMBatch(specs, identity_mode=1) as sim:
        L, h, n = lib(), sim._handle(), sim.n
        sim.advance(3)
        snap = torch.empty(int(L.mpm_state_bytes(h)), dtype=torch.uint8, device="cuda")
        cot = torch.randn(autodiff.channels(dim), n, generator=torch.Generator("cuda").manual_seed(3), device="cuda")
        slots, want, got = torch.empty_like(cot), torch.empty_like(cot), cot.clone()
        gE = torch.zeros(2, 2, dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        check(L.mpm_save_state(h, snap.data_ptr()))
        sim.advance(steps)
        check(L.mpm_grad_from_particle_order(h, cot.data_ptr(), slots.data_ptr()))
        check(L.mpm_load_state(h, snap.data_ptr()))
        check(L.mpm_backward_segment(h, steps, slots.data_ptr(), slots.data_ptr(), gE[0].data_ptr()))
        check(L.mpm_grad_to_particle_order(h, slots.data_ptr(), want.data_ptr()))
        check(L.mpm_load_state(h, snap.data_ptr()))
        check(L.mpm_backward_segment_particles(h, steps, got.data_ptr(), got.data_ptr(), gE[1].data_ptr()))
        sim.synchronize()
        assert torch.equal(got, want) and torch.equal(gE[0], gE[1])
        assert not torch.equal(got, cot)
