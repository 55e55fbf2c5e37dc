"""Block kernels with several waves per workgroup (tgrav_set_column_waves).  Column kernel (block
targets): the W waves of a workgroup hold the same 8^3 leaf block, split its sources in rounds of
64 W, and add their partial sums in LDS in wave order.  Block-source kernel: the W waves hold the
same tile of targets (2 per lane mixed, 4 FP64) and split the source blocks (wave v takes every
W-th block).

For every W in (1, 2, 4): FP64 within 1e-12 of the FP64 oracle and mixed within the parity bar
(<= 1e-6 median, <= 1e-4 max relative acceleration error), with source counts below one round
(waves with nothing to do), ragged last rounds and source chunks split over workgroups.  For a
fixed W the block form, the explicit C-order form, the fused kick and the unsplit batch plan give
the same bits, and a repeated run is bit-identical."""
import numpy as np
import pytest

import oracle
from tests import _util
from tests.test_gpu_batch import cell_blocks, set_item, to_np
from torch_amd import GasGravityField, GravityField, StellarGravityField, TgravError
from torch_amd import workloads as W
from torch_amd.batch import BatchPlan, problems_from_workload

pytestmark = pytest.mark.gpu
G = W.G_PC_MSUN_KMS


@pytest.fixture(scope="module")
def c2():
    return W.c2(1002)


def check_bar(mode, s):
    if mode == "fp64":
        assert s["acc_max"] <= 1e-12 and s["pot_max"] <= 1e-12, s
    else:
        assert s["acc_median"] <= 1e-6 and s["acc_max"] <= 1e-4, s


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
@pytest.mark.parametrize("waves", [1, 2, 4])
def test_column_waves_match_oracle(mode, waves, c2):
    st, ce = c2["stars"], c2["cells"]
    o, dx = ce["block_origin"][:24], ce["block_size"][:24] / 8
    bx, by, bz = oracle.block_centres(o[:, 0], o[:, 1], o[:, 2], dx)
    te = np.repeat(dx, 512)
    with StellarGravityField(mode) as f:
        f.set_column_waves(waves)
        assert f.column_waves() == waves
        for ns in (1, 100, 257, 1000):          # below one round of 64 W sources, ragged rounds
            sl = slice(0, ns)
            S = [st[k][sl] for k in ("x", "y", "z", "m", "eps")]
            f.set_stars(*S)
            ref = oracle.eval_plummer(*S, bx, by, bz, te, G, mode=oracle.NEUMAIER, threads=16)
            for nsplit in (1, 3):
                f.set_config(nsplit=nsplit)
                got = f.evaluate_blocks(o, dx, eps=dx)
                s = _util.summary(got, ref)
                print(mode, "waves", waves, "ns", ns, "nsplit", nsplit, s, flush=True)
                check_bar(mode, s)
                again = f.evaluate_blocks(o, dx, eps=dx)
                explicit = f.evaluate(te, bx, by, bz)          # detected as columns
                for p, q, r in zip(got, again, explicit):
                    assert np.array_equal(p, q)
                    assert np.array_equal(p, r)
                v = [np.zeros(len(bx)) for _ in range(3)]
                f.evaluate_blocks(o, dx, eps=dx, dt=0.5, vel=v)
                for p, q in zip(v, got[:3]):
                    assert np.array_equal(p, 0.5 * q)
            f.set_config(nsplit=0)


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
def test_column_waves_batch_equals_eager(mode):
    """Four waves per column workgroup: block-target and explicit C-order problems in one plan,
    unsplit, equal the eager column kernels bit for bit; split (default item sizes), the plan meets
    the bar against the oracle and graph replays equal its eager run."""
    import torch
    rng = W.rng_for(73)
    o, dx, (cx, cy, cz), cm = cell_blocks(rng, 11)
    st = W.star_cluster(rng, 1500)
    seps = np.full(1500, 0.02)
    probs = [dict(sources=dict(x=st["x"], y=st["y"], z=st["z"], m=st["m"], eps=seps),
                  targets=dict(block_origin=o, block_dx=dx)),
             dict(sources=dict(x=st["x"][:150], y=st["y"][:150], z=st["z"][:150], m=st["m"][:150]),
                  targets=dict(x=cx, y=cy, z=cz))]
    dev = problems_from_workload(probs)
    with GravityField(mode) as f:
        f.set_column_waves(4)
        f.set_config(nsplit=1)
        f.set_sources(st["x"], st["y"], st["z"], st["m"], seps)
        e0 = f.evaluate_blocks(o, dx)
        f.set_sources(st["x"][:150], st["y"][:150], st["z"][:150], st["m"][:150])
        e1 = f.evaluate(None, cx, cy, cz)
        set_item(f, 1e30)                       # one chunk per problem, as the eager launches
        plan = BatchPlan(f, dev)
        got = to_np(plan.run(graph=True))
        torch.cuda.synchronize()
        for q in range(4):
            assert np.array_equal(got[0][q], e0[q]), q
            assert np.array_equal(got[1][q], e1[q]), q
        plan.close()
        set_item(f, 0)
        f.set_config(nsplit=0)
        plan = BatchPlan(f, dev)
        eager = to_np(plan.run(graph=False))
        torch.cuda.synchronize()
        for rep in range(2):
            again = to_np(plan.run(graph=True))
            torch.cuda.synchronize()
            for i in range(2):
                for q in range(4):
                    assert np.array_equal(again[i][q], eager[i][q]), (rep, i, q)
        plan.close()
    refs = [oracle.eval_plummer(st["x"], st["y"], st["z"], st["m"], seps, cx, cy, cz, None, G,
                                mode=oracle.NEUMAIER, threads=16),
            oracle.eval_plummer(st["x"][:150], st["y"][:150], st["z"][:150], st["m"][:150], None, cx, cy, cz,
                                None, G, mode=oracle.NEUMAIER, threads=16)]
    for i in range(2):
        s = _util.summary(tuple(eager[i]), refs[i])
        print(mode, "batch waves 4 problem", i, s, flush=True)
        check_bar(mode, s)


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
@pytest.mark.parametrize("waves", [1, 4])
def test_shared_and_per_lane_dz_agree(mode, waves, c2):
    """Explicit column targets whose 64 columns of a group hold the same 8 z take the shared dz (each
    source's 8 dz formed once, by the lane that stages the source); a group whose columns differ in z
    forms them per lane.  Reversing the 8 z of one column per group keeps every group's bounding box
    (the mixed anchor) and sends each group down the per-lane path: every other column gives the same
    bits as before, the reversed column the same values in reverse order, eagerly and in a batch plan
    (the persistent kernel), and both layouts meet the bar against the oracle."""
    import torch
    st, ce = c2["stars"], c2["cells"]
    o, dx = ce["block_origin"][:16], ce["block_size"][:16] / 8
    bx, by, bz = oracle.block_centres(o[:, 0], o[:, 1], o[:, 2], dx)
    te = np.repeat(dx, 512)
    rz = bz.reshape(-1, 64, 8).copy()
    rz[:, 37, :] = rz[:, 37, ::-1]                  # column 37 of every group, z reversed
    rz = rz.ravel()
    col = np.zeros(len(bz), dtype=bool)
    col.reshape(-1, 64, 8)[:, 37, :] = True
    perm = np.arange(len(bz)).reshape(-1, 64, 8)
    perm[:, 37, :] = perm[:, 37, ::-1]               # b[t] corresponds to a[perm[t]]
    perm = perm.ravel()
    S = [st[k][:2000] for k in ("x", "y", "z", "m", "eps")]
    with StellarGravityField(mode) as f:
        f.set_column_waves(waves)
        f.set_stars(*S)
        f.set_config(nsplit=1)
        a = f.evaluate(te, bx, by, bz)
        b = f.evaluate(te, bx, by, rz)
        for p, q in zip(a, b):
            assert np.array_equal(p[~col], q[~col])
            assert np.array_equal(p[perm[col]], q[col])
        ref = oracle.eval_plummer(*S, bx, by, rz, te, G, mode=oracle.NEUMAIER, threads=16)
        s = _util.summary(b, ref)
        print(mode, "waves", waves, "per-lane dz vs oracle", s, flush=True)
        check_bar(mode, s)
        if waves == 4:
            dev = problems_from_workload([dict(sources=dict(zip(("x", "y", "z", "m", "eps"), S)),
                                               targets=dict(x=bx, y=by, z=z, eps=te)) for z in (bz, rz)])
            set_item(f, 1e30)                       # one chunk per problem, as the eager launches
            plan = BatchPlan(f, dev)
            got = to_np(plan.run(graph=True))
            torch.cuda.synchronize()
            plan.close()
            set_item(f, 0)
            for q in range(4):
                assert np.array_equal(got[0][q], a[q]), q
                assert np.array_equal(got[1][q], b[q]), q
        f.set_config(nsplit=0)


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
@pytest.mark.parametrize("waves", [1, 2, 4])
def test_block_source_waves_match_oracle(mode, waves, c2):
    """13 source blocks (ragged rounds of W blocks, chunks of 1, 2 and 5 blocks) onto 700 stars
    (a partial last tile of 256): the oracle's field to the bar; repeated runs and explicit
    cells in the blocks' C order (detected as blocks) give the same bits."""
    st, ce = c2["stars"], c2["cells"]
    nb = 13
    sl = slice(0, nb * 512)
    o, dxb = ce["block_origin"][:nb], ce["block_size"][:nb] / 8
    tx, ty, tz = st["x"][:700], st["y"][:700], st["z"][:700]
    ref = oracle.eval_plummer(ce["x"][sl], ce["y"][sl], ce["z"][sl], ce["m"][sl], ce["eps"][sl], tx, ty, tz,
                              None, G, mode=oracle.NEUMAIER, threads=16)
    with GasGravityField(mode) as g:
        g.set_column_waves(waves)
        for nsplit in (13, 7, 3, 1):            # chunks of 1, 2, 5 and 13 blocks
            g.set_config(nsplit=nsplit)
            g.set_blocks(o, dxb, ce["m"][sl])
            got = g.evaluate(None, tx, ty, tz)
            s = _util.summary(got, ref)
            print(mode, "block sources waves", waves, "nsplit", nsplit, s, flush=True)
            check_bar(mode, s)
            again = g.evaluate(None, tx, ty, tz)
            g.set_sources(ce["x"][sl], ce["y"][sl], ce["z"][sl], ce["m"][sl], ce["eps"][sl])
            detected = g.evaluate(None, tx, ty, tz)
            for p, q, r in zip(got, again, detected):
                assert np.array_equal(p, q)
                assert np.array_equal(p, r)


def test_column_waves_argument_errors():
    with GravityField("fp64") as f:
        for bad in (0, 3, 8, -1):
            with pytest.raises(TgravError):
                f.set_column_waves(bad)
        assert f.column_waves() == 4           # the default


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
@pytest.mark.parametrize("ns", [1, 63, 64, 65, 255, 256, 257, 1000])
def test_thin_launches_give_the_column_kernels_bits(mode, ns):
    """Launches too small to fill the chip take one target per lane (k_eval_thin): block targets, the
    same targets as explicit centres and a plan (which keeps the column code) agree bit for bit, with
    softened and unsoftened sources (coincident pairs among them), and so do the potential and the
    acceleration asked for alone."""
    import torch
    from torch_amd.blocks import block_centres
    d = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")  # noqa: E731
    rng = W.rng_for(1300 + ns)
    nblk = 3
    o, w = rng.uniform(-1, 1, (nblk, 3)), rng.uniform(0.01, 0.1, nblk)
    cx, cy, cz, _ = block_centres(o, w)
    pos = rng.uniform(-1, 1, (3, ns))
    k = min(ns, 5)
    pos[:, :k] = np.stack([cx[:k * 100:100], cy[:k * 100:100], cz[:k * 100:100]])
    for eps in (None, np.full(ns, 0.01)):
        s = [d(a) for a in pos] + [d(rng.uniform(0.1, 1, ns)), None if eps is None else d(eps)]
        with StellarGravityField(mode) as f:
            f.set_config(nsplit=1)
            f.set_stars(*s)
            a = f.evaluate_blocks(d(o), d(w))
            b = f.evaluate(None, d(cx), d(cy), d(cz))
            src = dict(x=s[0], y=s[1], z=s[2], m=s[3])
            if eps is not None:
                src["eps"] = s[4]
            plan = BatchPlan(f, [dict(sources=src, targets=dict(block_origin=d(o), block_dx=d(w)))])
            c = plan.run()[0]
            phi = f.get_potential_at_point(None, d(cx), d(cy), d(cz))
            acc = f.get_gravity_at_point(None, d(cx), d(cy), d(cz))
            for q in range(4):
                assert torch.equal(a[q], b[q]) and torch.equal(a[q], c[q])
                assert torch.equal(a[q], phi if q == 3 else acc[q])
            assert torch.isfinite(a[3]).all()


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
@pytest.mark.parametrize("nblk,nt", [(1, 1), (3, 127), (4, 128), (5, 129), (37, 300), (130, 640)])
def test_block_source_chunks_match_oracle(mode, nblk, nt):
    """The automatic source split of the block-source kernel, in whole rounds of a block per wave: part
    rounds, part target tiles, and as many chunks as rounds; the unsplit evaluation gives the same sums
    of the same blocks."""
    rng = W.rng_for(nblk * 1000 + nt)
    o = rng.uniform(-2.0, 1.5, (nblk, 3))
    size = rng.choice([0.125, 0.25, 0.5], nblk)
    x, y, z, dx = W.block_cell_centres(o, size)
    m = 50.0 * np.exp(rng.normal(size=x.size)) * dx ** 3
    st = W.star_cluster(rng, max(nt, 2), binary_frac=0.0)
    T = [st[k][:nt] for k in "xyz"]
    ref = oracle.eval_plummer(x, y, z, m, dx, *T, np.zeros(nt), G, mode=oracle.NEUMAIER, threads=8)
    with GravityField(mode) as f:
        for waves in (1, 2, 4):
            f.set_column_waves(waves)
            f.set_sources(x, y, z, m, dx)              # recognised as 8^3 blocks
            for nsplit in (0, 1):
                f.set_config(nsplit=nsplit)
                s = _util.summary(f.evaluate(None, *T), ref)
                print(mode, nblk, nt, waves, nsplit, s, flush=True)
                check_bar(mode, s)


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
@pytest.mark.parametrize("nblk", [59, 60, 61, 64, 65, 95, 96, 97])
def test_line_between_thin_and_column_launches(mode, nblk):
    """4 chunks of 4 waves per block, on either side of 3.75, 4 and 6 column waves per CU: blocks, explicit
    centres and a plan (which keeps the column code) give the same bits."""
    import torch
    from torch_amd.blocks import block_centres
    d = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")  # noqa: E731
    rng = W.rng_for(nblk)
    o, w = rng.uniform(-1, 1, (nblk, 3)), rng.uniform(0.01, 0.1, nblk)
    cx, cy, cz, _ = block_centres(o, w)
    s = [d(a) for a in rng.uniform(-1, 1, (3, 1100))] + [d(rng.uniform(0.1, 1, 1100)), d(np.full(1100, 0.01))]
    with StellarGravityField(mode) as f:
        f.set_config(nsplit=4)
        f.set_stars(*s)
        a = f.evaluate_blocks(d(o), d(w))
        b = f.evaluate(None, d(cx), d(cy), d(cz))
        f.set_config(nsplit=1)
        one = f.evaluate_blocks(d(o), d(w))
        src = dict(x=s[0], y=s[1], z=s[2], m=s[3], eps=s[4])
        c = BatchPlan(f, [dict(sources=src, targets=dict(block_origin=d(o), block_dx=d(w)))]).run()[0]
        for q in range(4):
            assert torch.equal(a[q], b[q])
            assert torch.allclose(one[q], c[q], rtol=1e-5 if mode == "mixed" else 1e-12, atol=1e-12 * float(c[q].abs().max()))
            assert torch.allclose(one[q], a[q], rtol=1e-5 if mode == "mixed" else 1e-12, atol=(1e-6 if mode == "mixed" else 1e-12) * float(c[q].abs().max()))


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
@pytest.mark.parametrize("nblk,nt", [(7, 33000), (31, 5000), (32, 5000), (33, 5000), (61, 1500), (300, 3000), (29, 129)])
@pytest.mark.parametrize("waves", [1, 2, 4])
def test_block_source_chunks_by_xcd(mode, nblk, nt, waves):
    """The automatic source split at few chunks (shared by all places), at 8 and more (a chunk's tiles on one
    XCD) and with a part chunk at the end: the unsplit sums, to rounding."""
    import torch
    rng = W.rng_for(nblk * 7 + nt)
    d = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")  # noqa: E731
    o, w = d(rng.uniform(-2.0, 1.5, (nblk, 3))), d(rng.choice([0.125, 0.25, 0.5], nblk) / 8)
    m = d(rng.uniform(0.5, 1.0, nblk * 512))
    T = [d(a) for a in rng.uniform(-2, 2, (3, nt))]
    with GravityField(mode, tune_cache=None) as f:
        f.set_column_waves(waves)
        f.set_source_blocks(o, w, m)
        got = f.evaluate(None, *T)
        f.set_config(nsplit=1)
        one = f.evaluate(None, *T)
    size = m.sum() * W.G_PC_MSUN_KMS
    for q in range(4):
        tol = (1e-12 if mode == "fp64" else 1e-5) * (one[3].abs().max() if q == 3 else size / 0.01)
        assert bool(((got[q] - one[q]).abs() <= tol).all())


@pytest.mark.parametrize("mode", ["fp64", "mixed"])
@pytest.mark.parametrize("ns", [1, 64, 65, 128, 129])
@pytest.mark.parametrize("nblk", [200, 800, 1600])
def test_few_sources_on_many_blocks(mode, ns, nblk):
    """Chunks of one, two and more waves' sources, thin and column launches: blocks, explicit centres and a plan
    (whose workgroups keep their 4 waves) give the same bits."""
    import torch
    from torch_amd.blocks import block_centres
    d = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")  # noqa: E731
    rng = W.rng_for(nblk + ns)
    o, w = rng.uniform(-1, 1, (nblk, 3)), rng.uniform(0.01, 0.1, nblk)
    cx, cy, cz, _ = block_centres(o, w)
    s = [d(a) for a in rng.uniform(-1, 1, (3, ns))] + [d(rng.uniform(0.1, 1, ns)), d(np.full(ns, 0.01))]
    with StellarGravityField(mode) as f:
        f.set_config(nsplit=1)
        f.set_stars(*s)
        a = f.evaluate_blocks(d(o), d(w))
        b = f.evaluate(None, d(cx), d(cy), d(cz))
        src = dict(x=s[0], y=s[1], z=s[2], m=s[3], eps=s[4])
        c = BatchPlan(f, [dict(sources=src, targets=dict(block_origin=d(o), block_dx=d(w)))]).run()[0]
        for q in range(4):
            assert torch.equal(a[q], b[q]) and torch.equal(a[q], c[q])
