"""Slot order of the engine's state after it is set from a device image."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from nuclearmpm_amd import MaterialModel, MPMBatch, MPMSimulation, Particles, SceneSpec, autodiff
from nuclearmpm_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def _cloud(dim, n, seed):
    rng = np.random.default_rng(seed)
    p = Particles.from_positions((0.2 + 0.5 * rng.random((n, dim))).astype(np.float32), identity_mode=1)
    p.v = rng.normal(0, 1.0, p.v.shape).astype(np.float32)
    p.C = rng.normal(0, 1.0, p.C.shape).astype(np.float32)
    p.F = (p.F + rng.normal(0, 0.01, p.F.shape)).astype(np.float32)
    return p


@pytest.mark.parametrize("dim,n", [(2, 1001), (2, 262143), (2, 262144), (3, 262144), (3, 300007)])
def test_set_state_device_makes_the_slot_order_the_particle_order(dim, n):
    """At every size: a cotangent in slot order is one in particle order, and mpm_backward_step returns grad_in in
    particle order, bit for bit what a one-step rollout returns."""
    p = _cloud(dim, n, dim)
    ng = autodiff.channels(dim)
    with MPMSimulation(p, MaterialModel.kJelly, 64, E=1e3, identity_mode=1) as sim:
        L, h = lib(), sim._handle()
        image = sim.state_image()
        cot = torch.randn(ng, n, generator=torch.Generator("cuda").manual_seed(7), device="cuda")
        s0 = image.clone().requires_grad_(True)
        out = autodiff.rollout(sim, s0, torch.tensor([1e3]), steps=1, checkpoint_every=1)
        want = torch.autograd.grad(out, s0, cot)[0]
        sim.advance(2)  # slots in tile order
        snap = torch.empty(int(L.mpm_state_bytes(h)), dtype=torch.uint8, device="cuda")
        order = torch.empty(int(L.mpm_order_bytes(h)), dtype=torch.uint8, device="cuda")
        slots, gin = torch.empty_like(cot), torch.empty_like(cot)
        torch.cuda.synchronize()
        check(L.mpm_set_state_device(h, image.data_ptr()))
        check(L.mpm_save_order(h, order.data_ptr()))
        check(L.mpm_save_state(h, snap.data_ptr()))
        check(L.mpm_grad_from_particle_order(h, cot.data_ptr(), slots.data_ptr()))
        sim.synchronize()
        assert torch.equal(order.view(torch.int32)[:n], torch.arange(n, dtype=torch.int32, device="cuda"))
        assert torch.equal(slots, cot)
        sim.advance(1)
        check(L.mpm_grad_from_particle_order(h, cot.data_ptr(), slots.data_ptr()))
        check(L.mpm_load_state(h, snap.data_ptr()))
        check(L.mpm_backward_step(h, slots.data_ptr(), gin.data_ptr(), None))
        sim.synchronize()
        assert torch.equal(gin, want)


@pytest.mark.parametrize("dim,n", [(2, 300_000), (3, 200_000)])
def test_a_segment_takes_the_memory_that_tape_bytes_says(dim, n):
    """The first backward segment of an engine allocates what mpm_tape_bytes counts beyond a one-step segment, the
    dL/dE contributions of its steps among it (31 x 4 bytes per particle here)."""
    p, steps, taken = _cloud(dim, n, 5), 33, []
    for k in (1, steps):
        with MPMSimulation(p, MaterialModel.kJelly, 32, E=1.0, identity_mode=1) as sim:
            L, h = lib(), sim._handle()
            cot = torch.zeros(autodiff.channels(dim), n, device="cuda")
            gE = torch.zeros(1, dtype=torch.float64, device="cuda")
            torch.cuda.synchronize()
            bytes_k = int(L.mpm_tape_bytes(h, k))
            free = torch.cuda.mem_get_info()[0]
            check(L.mpm_backward_segment(h, k, cot.data_ptr(), cot.data_ptr(), gE.data_ptr()))
            sim.synchronize()
            taken.append(free - torch.cuda.mem_get_info()[0] - bytes_k)
    assert abs(taken[1] - taken[0]) < 20 << 20, taken  # some ten allocations, each rounded up to 2 MiB


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("recorded", [0, 1, 3])
def test_a_large_image_with_a_particle_off_one_scenes_grid(dim, recorded):
    """The image of a batch, stored in tile order: its first step (of mpm_advance, or of a recorded segment of 1 or 3
    steps, which sorts from that order) stops that scene alone.  The scene keeps its particles, grid and
    active nodes; the others step as they do alone, bit for bit."""
    sizes, res, steps = (100_001, 130_007, 40_003), 64, max(recorded, 1)
    before = [_cloud(dim, n, 40 + s) for s, n in enumerate(sizes)]
    for c in before:
        c.x = (c.x * np.float32(0.4) + np.float32(0.1)).astype(np.float32)
    after = [_cloud(dim, n, 50 + s) for s, n in enumerate(sizes)]
    for c in after:
        c.x = (c.x * np.float32(0.4) + np.float32(0.5)).astype(np.float32)  # no node tile in common
    after[1].x[777, 0] = 2.0
    rows = (torch.from_numpy(np.concatenate([getattr(c, k) for c in after])).cuda() for k in ("x", "v", "F", "C", "Jp"))
    image = autodiff.pack(*rows)
    with MPMBatch([SceneSpec(c, MaterialModel.kJelly, res, E=1.0) for c in before], identity_mode=1) as batch:
        L, h = lib(), batch._handle()
        batch.advance(2)
        grid, active = batch.grid(1), batch.active_nodes(1)
        tape = torch.empty(int(L.mpm_record_bytes(h, steps, 1)), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        batch.set_state_image(image)
        if recorded:
            check(L.mpm_advance_recorded(h, steps, tape.data_ptr(), 1))
        else:
            batch.advance(steps)
        assert batch.scene_status() == {1: {"flags": 1, "step": 3}}
        assert batch.active_nodes(1) == active > 0
        for a, b in zip(batch.grid(1), grid):
            assert np.array_equal(a, b)
        got = [batch.particles(s) for s in range(3)]
    for k in ("x", "v", "F", "C", "Jp"):
        assert np.array_equal(getattr(got[1], k), getattr(after[1], k)), k
    for s in (0, 2):
        with MPMSimulation(after[s], MaterialModel.kJelly, res, E=1.0, identity_mode=1) as sim:
            sim.advance(steps)
            alone = sim.particles()
        for k in ("x", "v", "F", "C", "Jp"):
            assert np.array_equal(getattr(got[s], k), getattr(alone, k)), (s, k)
