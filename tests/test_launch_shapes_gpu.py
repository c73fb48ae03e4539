"""Launch shapes chosen by size give the same bits on both sides of their line."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from parity import assert_parity

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


@pytest.mark.parametrize("dim,n,res,lo,hi,chunk", [
    (2, 70000, 128, 0.40, 0.50, 256),   # lists of a node tile longer than one round of 64 slots, four partial sums
    (3, 40000, 64, 0.40, 0.55, 256),    # the same in 3D, candidates on both sides of the tiles' faces
    (3, 12000, 200, 0.05, 0.95, 256),   # more node tiles in use than workgroups: each takes several
    (3, 513, 37, 0.10, 0.80, 512),      # a grid that does not fill its last node tiles
])
def test_grid_update_over_listed_node_tiles(dim, n, res, lo, hi, chunk):
    """One step against the oracle, particles and grid (the step's own bound), after a radix sort and
    after an incremental one."""
    rng = np.random.default_rng(n)
    p = Particles.from_positions((lo + (hi - lo) * rng.random((n, dim))).astype(np.float32), identity_mode=1)
    p.v = rng.normal(0, 1.0, p.v.shape).astype(np.float32)
    p.C = rng.normal(0, 2.0, p.C.shape).astype(np.float32)
    p.F = (p.F + rng.normal(0, 0.005, p.F.shape)).astype(np.float32)
    kw = dict(res=res, E=1e3, identity_mode=1)
    with MPMSimulation(p, MaterialModel.kJelly, res, E=1e3, identity_mode=1, p2g_chunk=chunk) as sim:
        before = p
        for kind in ("radix", "incremental"):
            sim.advance(1)
            got = sim.particles().copy()
            vel, mass = sim.grid()
            st = O.State(x=before.x, v=before.v, F=before.F, C=before.C, Jp=before.Jp, mass=before.mass,
                         volume=before.volume)
            assert_parity(got, O.run(st, O.JELLY, steps=1, **kw), inv_dx=float(res), label=f"{kind} sort")
            ref = O.p2g(st, O.JELLY, res=res, E=1e3)
            ref_vel, ref_mass = O.grid_op(ref[0], ref[1], dim, res)
            assert np.abs(mass.ravel() - ref_mass).max() <= 1e-5 * ref_mass.max()
            assert sim.active_nodes() == int((ref[1] > 0).sum())
            before = got


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), 1e37])
def test_a_cotangent_out_of_range_stays_with_its_neighbours(dim, bad):
    """The G2P adjoint deposits a particle whose bound is not finite with a check per contribution: its
    nodes' cotangents are lost (NaN), those of a far cluster are bit for bit what they are without it."""
    import torch

    from nuclearmpm_amd import autodiff

    rng = np.random.default_rng(dim)
    n = 300
    x = np.concatenate([0.2 + 0.1 * rng.random((n, dim)), 0.6 + 0.1 * rng.random((n, dim))]).astype(np.float32)
    p = Particles.from_positions(x, identity_mode=1)
    p.F = (p.F + rng.normal(0, 0.01, p.F.shape)).astype(np.float32)
    cot = torch.from_numpy(rng.normal(size=(autodiff.channels(dim), 2 * n)).astype(np.float32)).cuda()
    grads = []
    with MPMSimulation(p, MaterialModel.kJelly, 64, identity_mode=1) as sim:
        for value in (None, bad):
            c = cot.clone()
            if value is not None:
                c[2 * dim + dim * dim, 7] = value  # C_00 of particle 7
            s0 = sim.state_image().requires_grad_(True)
            out = autodiff.rollout(sim, s0, torch.tensor([1e4]), steps=1, checkpoint_every=1)
            grads.append(torch.autograd.grad(out, s0, c)[0].cpu().numpy())
    far = slice(n, 2 * n)
    assert np.isfinite(grads[0]).all()
    assert np.array_equal(grads[0][:, far], grads[1][:, far])
    assert np.isnan(grads[1][:, 7]).any()


@pytest.mark.parametrize("n", [1, 63, 65, 1024, 1025, 4097, 65536, 65537, 262144, 262145, 300001])
@pytest.mark.parametrize("bits", [0, 1, 7, 8, 9, 20, 32])
def test_radix_sort_at_the_edges_of_its_tiles(n, bits):
    """1024-key tiles up to 2^18 keys, 4096 above; digit offsets summed in the scatter up to 64 tiles;
    odd and even pass counts (the input buffer alternates)."""
    from nuclearmpm_amd._lib import sort_keys

    rng = np.random.default_rng(n + bits)
    for keys in (rng.integers(0, 1 << 32, n, dtype=np.uint32),                   # random order
                 np.sort(rng.integers(0, 1 << min(bits, 10), n).astype(np.uint32)),  # sorted, many equal
                 np.full(n, 0xA5A5A5A5, np.uint32)):                              # all equal
        low = keys if bits == 32 else keys & np.uint32((1 << bits) - 1)
        assert np.array_equal(sort_keys(keys, bits), np.argsort(low, kind="stable").astype(np.uint32))


@pytest.mark.parametrize("dim,scenes", [(2, 1), (3, 2)])
def test_segments_longer_than_one_sum_of_the_elasticity_gradient(dim, scenes):
    """dL/dE is summed up to 32 adjoint steps at a time, and a segment's last state is sorted from the
    step before's order: the same gradients, bit for bit, for segments of 1, 7 and 70 steps."""
    import torch

    from nuclearmpm_amd import autodiff

    specs = [SceneSpec(_cloud(dim, 900 + 700 * s, 5 + s), MaterialModel.kJelly, 48, E=1e3) for s in range(scenes)]
    cot = None
    grads = []
    with MPMBatch(specs, identity_mode=1) as sim:
        image = sim.state_image()
        for every in (1, 7, 70):
            s0 = image.clone().requires_grad_(True)
            E = torch.tensor([1e3 + 100.0 * s for s in range(scenes)], dtype=torch.float64, requires_grad=True)
            out = autodiff.rollout(sim, s0, E, steps=70, checkpoint_every=every)
            if cot is None:
                cot = torch.randn(out.shape, generator=torch.Generator("cuda").manual_seed(1), device="cuda")
            grads.append(torch.autograd.grad(out, (s0, E), cot))
    for g in grads[1:]:
        assert torch.equal(g[0], grads[0][0]) and torch.equal(g[1], grads[0][1])


@pytest.mark.parametrize("dim,n", [(2, 262144), (3, 300007)])
@pytest.mark.parametrize("mixed", [False, True])
def test_large_state_images_in_any_order(dim, n, mixed):
    """A state image of 2^18 particles or more is stored in tile order, and the channels go by rows where
    the order is incoherent (mixed): the image comes back as it was, the steps are bit for bit those
    of an engine built from the same particles, and cotangents survive both orders."""
    import torch

    from nuclearmpm_amd import autodiff
    from nuclearmpm_amd._lib import check, lib

    rng = np.random.default_rng(n)
    side = int(np.ceil(n ** (1.0 / dim)))
    idx = np.stack(np.unravel_index(np.arange(n), (side,) * dim), 1)
    x = (0.2 + 0.5 * idx / side + 0.001 * rng.random((n, dim))).astype(np.float32)
    p = Particles.from_positions(x[rng.permutation(n)] if mixed else x, identity_mode=1)
    p.v = rng.normal(0, 1.0, p.v.shape).astype(np.float32)
    p.C = rng.normal(0, 1.0, p.C.shape).astype(np.float32)
    p.mass = (1.0 + rng.random(n)).astype(np.float32)
    p.volume = (1.0 + rng.random(n)).astype(np.float32)
    image = autodiff.pack(*(torch.from_numpy(getattr(p, k)).cuda() for k in ("x", "v", "F", "C", "Jp")))
    cot = torch.randn(image.shape, generator=torch.Generator("cuda").manual_seed(3), device="cuda")
    with MPMSimulation(p, MaterialModel.kJelly, 64, E=1e3, identity_mode=1) as a, \
            MPMSimulation(p, MaterialModel.kJelly, 64, E=1e3, identity_mode=1) as b:
        b.advance(2)
        b.set_state_image(image)
        assert torch.equal(b.state_image(), image)
        a.advance(3)
        b.advance(3)
        pa, pb = a.particles(), b.particles()
        for k in ("x", "v", "F", "C", "Jp", "mass", "volume"):
            assert np.array_equal(getattr(pa, k), getattr(pb, k)), k
        s = torch.cat([torch.from_numpy(getattr(pb, k)).reshape(n, -1) for k in ("x", "v", "F", "C", "Jp")], 1).t()
        assert torch.equal(b.state_image().cpu(), s)
        torch.cuda.synchronize()
        slots, back = torch.empty_like(cot), torch.empty_like(cot)
        check(lib().mpm_grad_from_particle_order(b._handle(), cot.data_ptr(), slots.data_ptr()))
        check(lib().mpm_grad_to_particle_order(b._handle(), slots.data_ptr(), back.data_ptr()))
        b.synchronize()
        assert torch.equal(back, cot) and not torch.equal(slots, cot)
        b.advance(1)  # the other state buffer was scratch
        a.advance(1)
        assert np.array_equal(a.particles().x, b.particles().x)
        # a particle off its grid is found by the step, not by the call that sets the state
        bad = image.clone()
        bad[0, 12345] = 2.0
        b.set_state_image(bad)
        assert torch.equal(b.state_image(), bad)
        b.advance(1)
        with pytest.raises(IndexError):
            b.synchronize()
        b.set_state_image(image)
        b.advance(1)
        b.synchronize()


@pytest.mark.parametrize("n,res", [(0, 20), (1, 20), (777, 79), (77_672, 79), (77_673, 80)])
def test_host_reads_on_both_sides_of_the_pinned_size(n, res):
    """Particle arrays and grids up to 8 MiB are read through pinned memory (77,672 3D particles, res 79)."""
    import torch

    p = _cloud(3, n, 11)
    p.mass = np.linspace(1.0, 2.0, n, dtype=np.float32)
    p.volume = np.linspace(2.0, 3.0, n, dtype=np.float32)
    with MPMSimulation(p, MaterialModel.kJelly, res, E=1e3, identity_mode=1) as sim:
        sim.advance(2)
        for _ in range(2):  # a first read and one with the buffers kept
            sim._cache = None
            got, (vel, mass) = sim.particles(), sim.grid()
            image = sim.state_image().cpu() if n else torch.empty(25, 0)
            rows = [getattr(got, k).reshape(n, w) for k, w in (("x", 3), ("v", 3), ("F", 9), ("C", 9), ("Jp", 1))]
            assert np.array_equal(np.concatenate(rows, 1).T, image.numpy())
            assert np.array_equal(got.mass, p.mass) and np.array_equal(got.volume, p.volume)
            # mass on the nodes: n sums of 27 weights, each rounded; empty nodes carry neither mass nor velocity
            assert mass.shape == (res + 1,) * 3 and vel.shape == (res + 1,) * 3 + (3,)
            assert abs(float(mass.sum(dtype=np.float64)) - float(p.mass.sum(dtype=np.float64))) <= 1e-5 * n
            assert not vel[mass == 0].any()
        assert sim.active_nodes() == int((mass > 0).sum())


def test_queued_elasticity_and_saved_order():
    """set_elasticity between queued steps takes effect in their order, and a cotangent goes to a saved slot order as
    it did while that order was the current one."""
    import torch

    from nuclearmpm_amd._lib import check, lib

    a, b = _cloud(3, 5000, 3), _cloud(3, 3001, 4)
    specs = [SceneSpec(a, MaterialModel.kJelly, 40), SceneSpec(b, MaterialModel.kJelly, 40)]
    out = []
    for wait in (False, True):
        with MPMBatch(specs, identity_mode=1) as sim:
            for k in range(4):
                sim.advance(1)
                for s in range(2):
                    sim.set_elasticity(s, 1e3 * (1 + k + 5 * s))
                    if wait:
                        sim.synchronize()
            out.append(sim.state_image())
            if wait:
                L, h, n = lib(), sim._handle(), sim.n
                order = torch.empty(int(L.mpm_order_bytes(h)), dtype=torch.uint8, device="cuda")
                cot = torch.randn(25, n, device="cuda")
                now, later = torch.empty_like(cot), torch.empty_like(cot)
                torch.cuda.synchronize()
                check(L.mpm_save_order(h, order.data_ptr()))
                check(L.mpm_grad_from_particle_order(h, cot.data_ptr(), now.data_ptr()))
                sim.advance(3)
                check(L.mpm_grad_to_saved_order(h, order.data_ptr(), cot.data_ptr(), later.data_ptr()))
                sim.synchronize()
                assert torch.equal(now, later) and not torch.equal(now, cot)
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("dim,sizes", [(2, (129,)), (3, (129,)), (3, (129, 9)), (3, (9, 129, 129, 20)), (2, (20,) * 7)])
def test_sort_tables_at_the_edges_of_their_rounds(dim, sizes):
    """The sort's tables are built in rounds of 4096 tiles (16 per workgroup for the prefixes): 64, 4096, 4097 and 8202
    tiles, and 28; every scene of a batch as it is by itself, over steps in which particles change tiles."""
    clouds = [_cloud(dim, 1500 + 211 * i, 20 + i) for i in range(len(sizes))]
    for c, res in zip(clouds, sizes):
        c.v *= np.float32(0.1 * 1e4 / res)  # some tenths of a cell a step
    specs = [SceneSpec(c, MaterialModel.kJelly, res, E=1.0) for c, res in zip(clouds, sizes)]
    with MPMBatch(specs, identity_mode=1) as batch:
        batch.advance(6)
        got = [batch.particles(s) for s in range(len(sizes))]
    for c, res, g in zip(clouds, sizes, got):
        with MPMSimulation(c, MaterialModel.kJelly, res, E=1.0, identity_mode=1) as sim:
            for _ in range(6):  # the radix sort every step
                sim.advance(1)
                image = sim.state_image()
                sim.set_state_image(image)
            ref = sim.particles()
        for k in ("x", "v", "F", "C", "Jp"):
            # a tile's particles in another order: bitwise up to one work item per tile, else a few
            # roundings of a node's sum a step
            a, b = getattr(g, k), getattr(ref, k)
            assert np.array_equal(a, b) if dim == 3 and res == 129 else np.abs(a - b).max() <= 1e-5 * np.abs(b).max(), k


@pytest.mark.parametrize("d", [2, 3])
def test_jacobi_pairs_on_both_sides_of_the_plain_range_are_bitwise_the_oracle(d):
    """Quotients and roots of operands of ordinary size skip the IEEE range handling (2^-40 of the largest entry up):
    zeros of either sign, entries and differences around the line, equal diagonals, and matrices of any scale."""
    from nuclearmpm_amd._lib import check, lib, ptr

    rng = np.random.default_rng(17)
    n = 3000
    eye = np.eye(d)[None]
    tiny = lambda: np.exp2(rng.uniform(-52, -28, (n, d, d))) * rng.choice([-1.0, 1.0], (n, d, d))  # noqa: E731
    A = [rng.normal(size=(n, d, d)), eye + 0.01 * rng.normal(size=(n, d, d))]
    A.append(np.where(rng.random((n, d, d)) < 0.4, rng.choice([0.0, -0.0], (n, d, d)), rng.normal(size=(n, d, d))))
    A.append(eye + tiny())                              # off-diagonals around the line
    sym = rng.normal(size=(n, d, d))
    sym = (sym + sym.transpose(0, 2, 1)).astype(np.float32)
    A.append(sym)                                       # m10 - m01 = 0
    A.append(sym + 2.0 ** -22 * rng.normal(size=(n, d, d)))
    eq = rng.normal(size=(n, d, d))
    eq[:, range(d), range(d)] = rng.normal(size=(n, 1))  # equal diagonals
    A.append(eq)
    skew = rng.normal(size=(n, d, d))
    A.append(skew - skew.transpose(0, 2, 1) + tiny())   # m00 + m11 around the line
    A.append(rng.normal(size=(n, d, d)) * np.exp2(rng.integers(-148, 126, (n, 1, 1))))
    A.append(np.exp2(rng.integers(-60, 60, (n, d, d))) * rng.normal(size=(n, d, d)))
    A = np.ascontiguousarray(np.concatenate(A), np.float32)
    A = A[np.isfinite(A).all(axis=(1, 2))]
    U, V, S = np.empty_like(A), np.empty_like(A), np.empty(A.shape[:2], np.float32)
    check(lib().mpm_svd(d, len(A), ptr(A), ptr(U), ptr(S), ptr(V), 1, 0))
    Uo, So, Vo = O.svd(A)
    for a, b in ((U, Uo), (S, So), (V, Vo)):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("dim,n,record", [(2, 3000, "none"), (2, 66_000, "none"), (2, 66_000, "grid"), (3, 4001, "none"),
                                          (3, 4001, "grid"), (3, 4001, "nogrid")])
def test_backward_leaves_the_first_steps_grid(dim, n, record):
    """After a backward pass the grid and the active nodes are those of a step from the first state, though no step ran
    P2G for it again: 2D below and above the size from which node tiles are listed (256 items of 256), and 3D; particles
    cross tiles, so that later steps of the segment reach other node tiles."""
    import torch

    from nuclearmpm_amd import autodiff

    res = 128
    clouds = [_cloud(dim, n, 31), _cloud(dim, 500, 32)]
    for c in clouds:
        c.x = (c.x * np.float32(0.3)).astype(np.float32) + np.float32(0.1)
        c.v = c.v * 0 + np.float32(60.0)
    specs = [SceneSpec(c, MaterialModel.kJelly, res, E=1.0) for c in clouds]
    opts = dict(identity_mode=1, p2g_chunk=256)
    with MPMBatch(specs, **opts) as b, MPMBatch(specs, **opts) as fresh:
        fresh.advance(1)
        rows = [torch.cat([torch.from_numpy(getattr(c, k)) for c in clouds]).cuda() for k in ("x", "v", "F", "C", "Jp")]
        x0 = autodiff.pack(*rows).requires_grad_(True)
        E = torch.tensor([1.0, 1.0], requires_grad=True)
        for steps, every in ((12, 6), (3, 1)):
            autodiff.rollout(b, x0, E, steps, every, record=record).square().sum().backward()
            for s in range(2):
                for got, want in zip(b.grid(s), fresh.grid(s)):
                    assert np.array_equal(got, want)
                assert b.active_nodes(s) == fresh.active_nodes(s) > 0
        b.advance(2)
        fresh.advance(1)
        assert np.array_equal(b.particles(0).x, fresh.particles(0).x)


@pytest.mark.parametrize("dim,n,spread", [(3, 1, 0.0), (3, 63, 0.0), (3, 65, 0.0), (3, 449, 0.2), (3, 5003, 0.05),
                                          (3, 530_003, 8.0), (2, 140_003, 6.0), (2, 140_003, 40.0)])
def test_p2g_lane_order_of_particles_that_share_cells(dim, n, spread):
    """P2G orders a wave's particles by LDS bank (3D, and 2D with several particles per thread): waves with one particle,
    with all of them in one cell (spread 0: every rank up to 63), partly filled, and at large against the oracle."""
    res = 64
    rng = np.random.default_rng(n)
    x = (30.3 + spread * (rng.random((n, dim)) - 0.5)) / res
    p = Particles.from_positions(x.astype(np.float32), identity_mode=1)
    p.v = rng.normal(0, 1.0, p.v.shape).astype(np.float32)
    p.C = rng.normal(0, 2.0, p.C.shape).astype(np.float32)
    p.F = (p.F + rng.normal(0, 0.005, p.F.shape)).astype(np.float32)
    p.mass = (1.0 + rng.random(n)).astype(np.float32)
    with MPMSimulation(p, MaterialModel.kJelly, res, E=1e2, identity_mode=1, p2g_chunk=512) as sim:
        sim.advance(1)
        got, (vel, mass) = sim.particles(), sim.grid()
    st = O.State(x=p.x, v=p.v, F=p.F, C=p.C, Jp=p.Jp, mass=p.mass, volume=p.volume)
    assert_parity(got, O.run(st, O.JELLY, steps=1, res=res, E=1e2, identity_mode=1), inv_dx=float(res),
                  label=f"{dim}D n={n}")
    # up to 28,000 particles reach a node: masses against sums in 64 bits (the oracle's FP32 sums round more than the step)
    X = p.x.astype(np.float64) * res
    base = (X - 0.5).astype(np.int64)
    f = X - base
    w = [0.5 * (1.5 - f) ** 2, 0.75 - (f - 1.0) ** 2, 0.5 * (f - 0.5) ** 2]
    ref_mass = np.zeros((res + 1,) * dim)
    for o in np.ndindex(*(3,) * dim):
        np.add.at(ref_mass, tuple(base[:, a] + o[a] for a in range(dim)),
                  p.mass * np.prod([w[o[a]][:, a] for a in range(dim)], axis=0))
    assert np.abs(mass - ref_mass).max() <= 1e-5 * ref_mass.max()


@pytest.mark.parametrize("material,svd", [(MaterialModel.kJelly, "exact"), (MaterialModel.kSnow, "fast"),
                                          (MaterialModel.kLiquid, "exact")])
def test_3d_p2g_ends_the_waves_without_particles(material, svd):
    """One particle per thread (3D, chunk 512, below 1024 full work items: 524,288 particles): work items of 1 to 512
    particles, whose idle waves end before the barriers, in scenes alone and in a batch above the line."""
    opts = dict(identity_mode=1, svd=svd, p2g_chunk=512)
    res, tile, rng = 64, 8, np.random.default_rng(8)
    counts = (1, 64, 65, 128, 129, 255, 256, 257, 320, 321, 448, 449, 511, 512, 513, 769, 1024)
    x = []
    for k, c in enumerate(counts):  # a tile each, every second one along the axes; stencil bases inside the tile
        first = 0.5 + tile * (1 + 2 * np.array([k % 3, k // 3 % 3, k // 9]))
        x.append((first + 0.1 + (tile - 0.2) * rng.random((c, 3))) / res)
    a = Particles.from_positions(np.concatenate(x).astype(np.float32), identity_mode=1)
    a.v = rng.normal(0, 1.0, a.v.shape).astype(np.float32)
    a.F = (a.F + rng.normal(0, 0.01, a.F.shape)).astype(np.float32)
    b = _cloud(3, 1024 * 512, 9)
    with MPMBatch([SceneSpec(a, material, res), SceneSpec(b, material, res)], **opts) as batch:
        batch.advance(2)
        got = batch.particles(0)
    with MPMSimulation(a, material, res, **opts) as sim:
        sim.advance(2)
        ref = sim.particles()
    for k in ("x", "v", "F", "C", "Jp"):
        assert np.array_equal(getattr(got, k), getattr(ref, k)), k


@pytest.mark.parametrize("dim,sizes", [(2, (129,)), (3, (129,)), (3, (129, 9)), (3, (9, 129, 129, 20)), (2, (20,) * 7),
                                       (2, (8192,)), (2, (8192, 20)), (3, (512, 20))])
def test_incremental_sort_tables_are_bitwise_the_radix_sorts(dim, sizes):
    """Up to 64 rounds of 4096 tiles the sort's carries come from the tiles, above (65 rounds: res 8192 or 512 and a
    small scene) from the rounds' totals: bit for bit the steps of an engine that saves and loads its state
    before each one, which keeps the slot order and sorts from scratch."""
    import torch

    from nuclearmpm_amd._lib import check, lib

    clouds = [_cloud(dim, 1500 + 211 * i, 20 + i) for i in range(len(sizes))]
    for c, res in zip(clouds, sizes):
        c.v *= np.float32(0.1 * 1e4 / res)  # some tenths of a cell a step
    specs = [SceneSpec(c, MaterialModel.kJelly, res, E=1.0) for c, res in zip(clouds, sizes)]
    with MPMBatch(specs, identity_mode=1) as batch, MPMBatch(specs, identity_mode=1) as fresh:
        L, h = lib(), fresh._handle()
        snap = torch.empty(int(L.mpm_state_bytes(h)), dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        for _ in range(6):
            batch.advance(1)
            check(L.mpm_save_state(h, snap.data_ptr()))
            check(L.mpm_load_state(h, snap.data_ptr()))
            fresh.advance(1)
        assert torch.equal(batch.state_image(), fresh.state_image())
        assert not torch.equal(batch.state_image()[:dim], torch.from_numpy(np.concatenate([c.x for c in clouds]).T).cuda())
        for s in range(len(sizes)):
            assert batch.active_nodes(s) == fresh.active_nodes(s) > 0


@pytest.mark.parametrize("dim,n", [(3, 4001), (2, 66_000)])
@pytest.mark.parametrize("record", ["none", "grid", "nogrid"])
def test_backward_drops_the_node_counts_of_later_steps(dim, n, record):
    """As above, where the second step reaches node tiles that the first one does not list (the particles move down an
    axis, out of the lowest tile they are in): their counts must not stay."""
    import torch

    from nuclearmpm_amd import autodiff

    res, S = 128, 8 if dim == 3 else 16
    c = _cloud(dim, n, 33)
    base = 40 + c.x.astype(np.float64) * 20  # clear of the walls
    base[:, 0] += 4 * S + 0.05 - base[:, 0].min()  # the lowest stencil base is 4 S, a step later 4 S - 1
    c.x = ((base + 0.5) / res).astype(np.float32)
    c.v, c.C, c.F = c.v * 0, c.C * 0, c.F * 0 + np.eye(dim, dtype=np.float32)
    c.v[:, 0] = -60.0  # 0.77 cells a step
    tiles = ((c.x * np.float32(res) - np.float32(0.5)).astype(np.int64)) // S
    listed = {tuple(t + d) for t in np.unique(tiles, axis=0) for d in np.ndindex(*(2,) * dim)}
    opts = dict(identity_mode=1, E=1.0, p2g_chunk=256)
    with MPMSimulation(c, MaterialModel.kJelly, res, **opts) as b, MPMSimulation(c, MaterialModel.kJelly, res, **opts) as fresh:
        fresh.advance(2)
        assert not {tuple(t) for t in np.unique(np.argwhere(fresh.grid()[1] > 0) // S, axis=0)} <= listed
        x0 = autodiff.pack(*(torch.from_numpy(getattr(c, k)).cuda() for k in ("x", "v", "F", "C", "Jp"))).requires_grad_(True)
        out = autodiff.rollout(b, x0, torch.tensor([1.0], requires_grad=True), 2, 2, record=record)
        out.square().sum().backward()
        assert b.active_nodes() == int((b.grid()[1] > 0).sum()) > 0


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("material", [MaterialModel.kJelly, MaterialModel.kSnow])
def test_adjoint_of_particles_in_the_half_cell_at_the_lower_walls(dim, material):
    """Stencil base 0 with an offset below 0.5, where a node is up to 2.5 cells away: gradients against the FP64
    adjoint, and a cotangent whose bound is finite but whose bracket at the third node is not leaves that node
    NaN, as every contribution out of range does."""
    import torch

    from nuclearmpm_amd import autodiff

    res, n = 24, 64
    rng = np.random.default_rng(dim)
    s = 8.0 + 4.0 * rng.random((n, dim))
    s[:, 0] = rng.uniform(0.02, 0.98, n)  # in cells: base 0, offset as it is
    s[0] = [0.2] + [10.9] * (dim - 1)
    s[1] = [3.0] + [10.9] * (dim - 1)     # shares the third node with it, no other on that axis
    p = Particles.from_positions((s / res).astype(np.float32), identity_mode=1)
    p.F = (p.F + rng.normal(0, 0.01, p.F.shape)).astype(np.float32)
    p.v = rng.normal(0, 0.5, p.v.shape).astype(np.float32)
    cot = rng.normal(size=(autodiff.channels(dim), n)).astype(np.float32)
    with MPMSimulation(p, material, res, identity_mode=1) as sim:
        image = sim.state_image()

        def grad(c):
            s0 = image.clone().requires_grad_(True)
            out = autodiff.rollout(sim, s0, torch.tensor([1e4]), steps=1, checkpoint_every=1)
            return torch.autograd.grad(out, s0, torch.from_numpy(c).cuda())[0].cpu().numpy()

        got = grad(cot)
        huge = np.zeros_like(cot)
        huge[2 * dim + dim * dim, 0] = 1.95e38 / (4.0 * res)  # C_00: 1.5 of it in cells is in range, 1.8 is not
        lost = grad(huge)
    assert np.isnan(lost[dim, 1]), lost[dim, :4]
    if material != MaterialModel.kJelly:
        return
    parts, at = [], 0
    for shape in ((dim,), (dim,), (dim, dim), (dim, dim)):
        w = int(np.prod(shape))
        parts.append(np.ascontiguousarray(cot[at:at + w].T).reshape((n,) + shape).astype(np.float64))
        at += w
    ref = O.adjoint_jelly(O.State(x=p.x, v=p.v, F=p.F, C=p.C, Jp=p.Jp, mass=p.mass, volume=p.volume),
                          O.Grads(*parts, Jp=cot[at].astype(np.float64)), res=res, E=1e4, identity_mode=1)
    at = 0
    for k in ("x", "v", "F", "C"):
        r = getattr(ref, k).reshape(n, -1)
        g = got[at:at + r.shape[1]].T
        at += r.shape[1]
        assert np.abs(g - r).max() <= 1e-4 * np.abs(r).max(), k  # the bound of the one-step gradient tests
