"""GPU parity of the particle-mesh pieces (needs an MI355X) against the oracle.

Bars: the finite-difference acceleration, the grid kick and the CIC interpolation use the
oracle's operations in the oracle's order and must match it bit for bit; the CIC deposit
sums in exact fixed point (order-free), so it matches the oracle's sequential FP64 sums to
1e-13 per cell and is bit-identical under any permutation of the particles.
"""
import numpy as np
import pytest

import oracle
from torch_amd import LeafBlocks, ParticleMesh, TgravError
from torch_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def c2pm():
    """c2's 2,000 leaf blocks with 4 guard layers and the stars inside the 4 pc box."""
    w = W.c2(1002)
    st, ce = w["stars"], w["cells"]
    blk = W.containing_block(st["x"], st["y"], st["z"], ce["block_origin"], ce["block_size"])
    keep = blk >= 0
    B = LeafBlocks(ce["block_origin"], ce["block_size"], nb=8, ng=4)
    P = dict(x=st["x"][keep], y=st["y"][keep], z=st["z"][keep], m=st["m"][keep], blk=blk[keep])
    return B, P


def oblocks(B):
    return dict(origin=B.origin, size=B.size, nb=B.nb, ng=B.ng)


def plummer_phi(B, b=0.6, M=500.0):
    x, y, z = B.centres()
    return -M / np.sqrt(x * x + y * y + z * z + b * b)


@pytest.fixture()
def pm():
    f = ParticleMesh()
    yield f
    f.close()


def test_deposit_matches_oracle_and_is_order_free(pm, c2pm):
    B, P = c2pm
    got = pm.update_grid_var(P["x"], P["y"], P["z"], P["m"], P["blk"], B)
    ref = oracle.pm_deposit(P["x"], P["y"], P["z"], P["m"], P["blk"], oblocks(B))
    np.testing.assert_allclose(got, ref, rtol=1e-13, atol=1e-300)
    dv = np.repeat((B.size / B.nb) ** 3, B.nbg ** 3)
    np.testing.assert_allclose((got * dv).sum(), P["m"].sum(), rtol=1e-13)
    perm = W.rng_for(3).permutation(len(P["x"]))
    again = pm.update_grid_var(P["x"][perm], P["y"][perm], P["z"][perm], P["m"][perm], P["blk"][perm], B)
    np.testing.assert_array_equal(again, got)
    base = np.full(B.ncell, 0.25)
    acc = pm.update_grid_var(P["x"], P["y"], P["z"], P["m"], P["blk"], B, rho=base.copy(), accumulate=True)
    np.testing.assert_array_equal(acc, 0.25 + got)


def test_deposit_signed_and_tiny_masses(pm):
    """Mixed-sign masses spanning 30 decades still sum to the oracle's value per cell."""
    rng = W.rng_for(4)
    B = LeafBlocks(np.array([[0.0, 0.0, 0.0], [1.0, 0.0, 0.0]]), np.array([1.0, 1.0]), nb=8, ng=1)
    n = 4000
    blk = rng.integers(0, 2, n)
    pos = B.origin[blk] + rng.uniform(0, 1, (n, 3))
    m = rng.normal(0, 1, n) * 10.0 ** rng.uniform(-15, 15, n)
    got = pm.update_grid_var(pos[:, 0], pos[:, 1], pos[:, 2], m, blk, B)
    ref = oracle.pm_deposit(pos[:, 0], pos[:, 1], pos[:, 2], m, blk, oblocks(B))
    # the sequential FP64 sum itself carries ~n eps of the largest |term|
    scale = oracle.pm_deposit(pos[:, 0], pos[:, 1], pos[:, 2], np.abs(m), blk, oblocks(B))
    assert np.all(np.abs(got - ref) <= 1e-13 * scale + 1e-300)


def test_deposit_errors(pm, c2pm):
    B, P = c2pm
    bad = P["blk"].copy()
    bad[7] = (bad[7] + 1) % B.nblk if B.nblk > 1 else 5       # another block: cloud outside it
    with pytest.raises(TgravError):
        pm.update_grid_var(P["x"], P["y"], P["z"], P["m"], bad, B)
    bad[7] = B.nblk + 3
    with pytest.raises(TgravError):
        pm.update_grid_var(P["x"], P["y"], P["z"], P["m"], bad, B)
    assert pm.lib.tgrav_pm_deposit(pm.handle, 1, None, None, None, None, None, 1, 8, 0, None, None, None,
                                   None, None, 0, 0) == -1


def test_gradient_and_kick_bit_exact(pm, c2pm):
    B, _ = c2pm
    phi = plummer_phi(B)
    g = pm.accel_list_of_blocks(phi, B)
    ref = oracle.pm_gradient(phi, oblocks(B))
    for q in range(3):
        np.testing.assert_array_equal(g[q], ref[q])
    rng = W.rng_for(8)
    v = [rng.normal(0, 1, B.ncell) for _ in range(3)]
    v0 = [a.copy() for a in v]
    dt = 0.37
    g2 = pm.accel_list_of_blocks(phi, B, dt=dt, vel=v)
    for q in range(3):
        np.testing.assert_array_equal(g2[q], ref[q])
        np.testing.assert_array_equal(v[q], v0[q] + ref[q] * dt)
    # kick only
    v1 = [a.copy() for a in v0]
    assert pm.accel_list_of_blocks(phi, B, dt=dt, vel=v1, store=False) is None
    for q in range(3):
        np.testing.assert_array_equal(v1[q], v0[q] + ref[q] * dt)


def test_interpolation_and_long_range_force_bit_exact(pm, c2pm):
    B, P = c2pm
    phi = plummer_phi(B)
    g = oracle.pm_gradient(phi, oblocks(B))
    got = pm.map_mesh_to_particles(P["x"], P["y"], P["z"], P["blk"], B, *g)
    ref = oracle.pm_interpolate(P["x"], P["y"], P["z"], P["blk"], oblocks(B), *g)
    for q in range(3):
        np.testing.assert_array_equal(got[q], ref[q])
    lrf = pm.long_range_force(P["x"], P["y"], P["z"], P["blk"], B, phi)
    for q in range(3):
        np.testing.assert_array_equal(lrf[q], ref[q])
    # physical sanity: the FD + CIC field of the Plummer potential points inwards
    r = np.stack([P["x"], P["y"], P["z"]], 1)
    a = np.stack(lrf, 1)
    assert np.mean(np.sum(a * r, 1) < 0) > 0.99


def test_device_tensors_match_host(pm, c2pm):
    import torch
    B, P = c2pm
    d = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")  # noqa: E731
    BD = LeafBlocks(d(B.origin), d(B.size), nb=B.nb, ng=B.ng)
    rho_h = pm.update_grid_var(P["x"], P["y"], P["z"], P["m"], P["blk"], B)
    rho_d = pm.update_grid_var(d(P["x"]), d(P["y"]), d(P["z"]), d(P["m"]), d(P["blk"]), BD)
    phi = plummer_phi(B)
    g_h = pm.accel_list_of_blocks(phi, B)
    g_d = pm.accel_list_of_blocks(d(phi), BD)
    a_h = pm.map_mesh_to_particles(P["x"], P["y"], P["z"], P["blk"], B, *g_h)
    a_d = pm.map_mesh_to_particles(d(P["x"]), d(P["y"]), d(P["z"]), d(P["blk"]), BD, *g_d)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(rho_d.cpu().numpy(), rho_h)
    for q in range(3):
        np.testing.assert_array_equal(g_d[q].cpu().numpy(), g_h[q])
        np.testing.assert_array_equal(a_d[q].cpu().numpy(), a_h[q])


# guarded blocks of one slice of the LDS deposit, just over one, several, and too large for it; particles
# none, one, one per block and many in one block
@pytest.mark.parametrize("nb,ng,nblk", [(2, 1, 5), (8, 2, 300), (8, 4, 7), (11, 1, 3), (16, 2, 3), (18, 2, 2)])
@pytest.mark.parametrize("crowd", [0, 1, 700, 3000])
def test_deposit_and_long_range_at_block_sizes(pm, nb, ng, nblk, crowd):
    """The deposit against the oracle and under a permutation (bit for bit), clouds reaching into the
    guard layers, with accumulation; the long-range force equal to the gradient followed by the
    interpolation, bit for bit."""
    rng = W.rng_for(1000 * nb + 10 * ng + nblk + crowd)
    B = LeafBlocks(rng.uniform(-2, 2, (nblk, 3)), rng.uniform(0.1, 1.0, nblk), nb=nb, ng=ng)
    blk = np.concatenate([np.arange(nblk), np.full(crowd, nblk // 2)])[: crowd + nblk if crowd else 0]
    h = (B.size / nb)[blk]
    pos = B.origin[blk] + h[:, None] * rng.uniform(0.6 - ng, nb + ng - 0.6, (blk.size, 3))
    m = rng.uniform(0.1, 2.0, blk.size)
    a = [pos[:, 0], pos[:, 1], pos[:, 2], m, blk]
    got = pm.update_grid_var(*a, B)
    ref = oracle.pm_deposit(*a, oblocks(B)) if blk.size else np.zeros(B.ncell)
    np.testing.assert_allclose(got, ref, rtol=1e-13, atol=1e-300)
    p = rng.permutation(blk.size)
    np.testing.assert_array_equal(pm.update_grid_var(*[q[p] for q in a], B), got)
    base = rng.uniform(-1, 1, B.ncell)
    acc = pm.update_grid_var(*a, B, rho=base.copy(), accumulate=True)
    np.testing.assert_array_equal(acc, base + got)
    phi = rng.normal(size=B.ncell)
    one = pm.long_range_force(pos[:, 0], pos[:, 1], pos[:, 2], blk, B, phi)
    two = pm.map_mesh_to_particles(pos[:, 0], pos[:, 1], pos[:, 2], blk, B, *pm.accel_list_of_blocks(phi, B))
    for u, v in zip(one, two):
        np.testing.assert_array_equal(u, v)
    if blk.size:
        bad = blk.copy()
        bad[-1] = nblk
        with pytest.raises(TgravError):
            pm.long_range_force(pos[:, 0], pos[:, 1], pos[:, 2], bad, B, phi)
        keep = base.copy()
        with pytest.raises(TgravError):
            pm.update_grid_var(*a[:4], bad, B, rho=keep)
        np.testing.assert_array_equal(keep, base)


# the deposit in LDS (at most 8,192 cells a block) and through memory
@pytest.mark.parametrize("nb,ng", [(8, 2), (8, 4), (16, 4), (18, 2)])
@pytest.mark.parametrize("bad", ["block_low", "block_high", "cloud"])
def test_bad_particles_without_validation(nb, ng, bad):
    """A particle whose block index or cloud is outside: with validation an error (and rho untouched), without
    it the deposit is the other particles', and the forces are theirs with NaN for it."""
    rng = W.rng_for(nb + ng)
    nblk, n = 3, 200
    B = LeafBlocks(rng.uniform(-2, 2, (nblk, 3)), rng.uniform(0.1, 1.0, nblk), nb=nb, ng=ng)
    blk = rng.integers(0, nblk, n)
    pos = B.origin[blk] + B.size[blk][:, None] * rng.uniform(0.0, 1.0, (n, 3))
    m = rng.uniform(0.1, 2.0, n)
    phi = rng.normal(size=B.ncell)
    out = [0, 77, n - 1]
    good = np.setdiff1d(np.arange(n), out)
    b2, p2 = blk.copy(), pos.copy()
    if bad == "cloud":
        p2[out] = B.origin[blk[out]] - 1.5 * B.size[blk[out]][:, None] * ng
    else:
        b2[out] = -1 if bad == "block_low" else nblk
    base = rng.uniform(-1, 1, B.ncell)
    with ParticleMesh(validate=False) as f:
        ref = f.update_grid_var(*[np.ascontiguousarray(pos[good, q]) for q in range(3)], m[good], blk[good], B)
        got = f.update_grid_var(*[np.ascontiguousarray(p2[:, q]) for q in range(3)], m, b2, B)
        # each cell's fixed point is scaled by the number of particles, so the sums may round differently
        np.testing.assert_allclose(got, ref, rtol=1e-13, atol=0)
        g = f.accel_list_of_blocks(phi, B)
        want = f.map_mesh_to_particles(*[np.ascontiguousarray(pos[:, q]) for q in range(3)], blk, B, *g)
        for a in (f.long_range_force(*[np.ascontiguousarray(p2[:, q]) for q in range(3)], b2, B, phi),
                  f.map_mesh_to_particles(*[np.ascontiguousarray(p2[:, q]) for q in range(3)], b2, B, *g)):
            for u, v in zip(a, want):
                np.testing.assert_array_equal(u[good], v[good])
                assert np.isnan(u[out]).all()
    with ParticleMesh() as f:
        keep = base.copy()
        with pytest.raises(TgravError):
            f.update_grid_var(*[np.ascontiguousarray(p2[:, q]) for q in range(3)], m, b2, B, rho=keep)
        np.testing.assert_array_equal(keep, base)
        with pytest.raises(TgravError):
            f.long_range_force(*[np.ascontiguousarray(p2[:, q]) for q in range(3)], b2, B, phi)


# particles in the crowded blocks: around the line to several workgroups, and whole and part stretches of them
@pytest.mark.parametrize("counts", [(1023, 1024), (1025,), (1025, 2047, 2048, 2049), (5000, 1, 1024, 9000), (70000,)])
@pytest.mark.parametrize("nb,ng,nblk", [(8, 1, 40), (8, 4, 40), (16, 2, 9), (8, 1, 16385)])
def test_crowded_blocks(pm, counts, nb, ng, nblk):
    """Some blocks with many particles among others with few: the oracle's densities, the same bits under a
    permutation, without validation, and added to what is there."""
    rng = W.rng_for(sum(counts) + nb + nblk)
    B = LeafBlocks(rng.uniform(-2, 2, (nblk, 3)), rng.uniform(0.1, 1.0, nblk), nb=nb, ng=ng)
    where = rng.choice(nblk, len(counts), replace=False)
    blk = np.concatenate([np.full(n, b) for n, b in zip(counts, where)] + [rng.integers(0, nblk, 4100)])
    rng.shuffle(blk)
    h = (B.size / nb)[blk]
    pos = B.origin[blk] + h[:, None] * rng.uniform(0.6 - ng, nb + ng - 0.6, (blk.size, 3))
    m = rng.uniform(0.1, 2.0, blk.size) * 10.0 ** rng.uniform(-8, 8, blk.size)
    a = [np.ascontiguousarray(pos[:, q]) for q in range(3)] + [m, blk]
    got = pm.update_grid_var(*a, B)
    ref = oracle.pm_deposit(*a, oblocks(B))
    # the oracle's sequential sums of up to a few thousand positive terms a cell
    np.testing.assert_allclose(got, ref, rtol=1e-12, atol=1e-300)
    p = rng.permutation(blk.size)
    np.testing.assert_array_equal(pm.update_grid_var(*[q[p] for q in a], B), got)
    base = rng.uniform(-1, 1, B.ncell)
    np.testing.assert_array_equal(pm.update_grid_var(*a, B, rho=base.copy(), accumulate=True), base + got)
    with ParticleMesh(validate=False) as f:
        np.testing.assert_array_equal(f.update_grid_var(*a, B), got)
        few = [q[:37] for q in a]                      # nothing of the crowded call is left behind
        np.testing.assert_array_equal(f.update_grid_var(*few, B), pm.update_grid_var(*few, B))


@pytest.mark.parametrize("np_", [4095, 4096, 4097])
def test_deposit_routes_agree(pm, np_):
    """Few particles in very few cells go through memory, one more through LDS: the same densities."""
    rng = W.rng_for(np_)
    B = LeafBlocks(rng.uniform(-2, 2, (4, 3)), rng.uniform(0.1, 1.0, 4), nb=8, ng=4)
    blk = rng.integers(0, 4, np_)
    pos = B.origin[blk] + B.size[blk][:, None] * rng.uniform(0, 1, (np_, 3))
    a = [np.ascontiguousarray(pos[:, q]) for q in range(3)] + [rng.uniform(0.1, 2.0, np_), blk]
    np.testing.assert_allclose(pm.update_grid_var(*a, B), oracle.pm_deposit(*a, oblocks(B)), rtol=1e-13, atol=1e-300)


@pytest.mark.parametrize("nblk", [146, 147])              # 598,016 and 602,112 cells
@pytest.mark.parametrize("n", [600_000, 600_001])
def test_force_routes_agree(n, nblk):
    """Many particles in few cells take the gradient first: on either side of the line the same bits, phi and
    blocks as host arrays among the particles' tensors included."""
    import torch
    rng = W.rng_for(n + nblk)
    gen = torch.Generator(device="cuda").manual_seed(n)
    o, size = rng.uniform(-2, 2, (nblk, 3)), rng.uniform(0.1, 1.0, nblk)
    phi = rng.normal(size=nblk * 4096)
    B = LeafBlocks(*[torch.as_tensor(a, device="cuda") for a in (o, size)], nb=8, ng=4)
    blk = torch.randint(0, nblk, (n,), device="cuda", generator=gen)
    x, y, z = [B.origin[:, q][blk] + B.size[blk] * torch.rand(n, dtype=torch.float64, device="cuda", generator=gen)
               for q in range(3)]
    f_d = torch.as_tensor(phi, device="cuda")
    with ParticleMesh() as f:
        got = f.long_range_force(x, y, z, blk, B, f_d)
        mixed = f.long_range_force(x, y, z, blk, LeafBlocks(o, size, nb=8, ng=4), phi)
        few = f.long_range_force(x[:1000], y[:1000], z[:1000], blk[:1000], B, f_d)
        two = f.map_mesh_to_particles(x, y, z, blk, B, *f.accel_list_of_blocks(f_d, B))
        bad = blk.clone()
        bad[-1] = nblk
        with pytest.raises(TgravError):
            f.long_range_force(x, y, z, bad, B, f_d)
    for a, m_, b, c in zip(got, mixed, two, few):
        assert torch.equal(a, b) and torch.equal(m_, b) and torch.equal(a[:1000], c)
