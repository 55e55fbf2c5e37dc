"""GPU tests of the one-pass input checks: statistics, NaN/Inf and structure found in a single launch
over one or many workgroups, and block sources expanded only where a kernel reads them cell by cell
(needs an MI355X)."""
import numpy as np
import pytest

from torch_amd import GasGravityField, StellarGravityField, TgravError, _lib
from torch_amd import workloads as W

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def dev(*arrs):
    return [torch.as_tensor(np.ascontiguousarray(a), device="cuda") for a in arrs]


# one lane, one workgroup, its edges, two workgroups, many, and past the most workgroups of a launch
@pytest.mark.parametrize("n", [1, 255, 256, 257, 512, 4097, 131072, 131073, 400000])
def test_bad_values_are_found_anywhere(n):
    """The first, the last and a middle element of every input array: refused as source and as target,
    and the next call on good inputs is accepted and equals the one before."""
    rng = W.rng_for(n)
    x, y, z, m, e = dev(*rng.uniform(-1, 1, (3, n)), rng.uniform(0.1, 1, n), np.full(n, 0.01))
    few = [a[:7].clone() for a in (e, x, y, z)]
    with StellarGravityField("fp64") as f:
        f.set_stars(x[:3].clone(), y[:3].clone(), z[:3].clone(), m[:3].clone(), e[:3].clone())
        ref = f.evaluate(e, x, y, z)
        for q in range(4):
            a = [e, x, y, z]
            for at in {0, n // 2, n - 1}:
                for v in (float("nan"), float("inf")):
                    a[q] = a[q].clone()
                    keep = float(a[q][at])
                    a[q][at] = v
                    with pytest.raises(TgravError) as err:
                        f.evaluate(*a)
                    assert err.value.code == _lib.ENONFINITE
                    a[q][at] = keep
        for r, g in zip(ref, f.evaluate(e, x, y, z)):
            assert torch.equal(r, g)
        src = [x, y, z, m, e]
        for q in range(5):
            for at in {0, n // 2, n - 1}:
                bad = list(src)
                bad[q] = src[q].clone()
                bad[q][at] = float("nan")
                with pytest.raises(TgravError) as err:
                    f.set_stars(*bad)
                assert err.value.code == _lib.ENONFINITE
                with pytest.raises(TgravError) as err:     # no source set is left behind
                    f.evaluate(*few)
                assert err.value.code == _lib.ENOSOURCES
        f.set_stars(*src)
        assert torch.isfinite(f.evaluate(*few)[3]).all()


@pytest.mark.parametrize("nblk", [1, 3, 300, 1025])
def test_structure_is_decided_by_every_element(nblk):
    """Explicit cells in block order take the column and block-source kernels, whose sums differ in
    rounding from the generic kernel's; one moved cell, anywhere, sends the call to the generic one.
    With and without validation (decided on the host, gated on the device) the bits are the same."""
    rng = W.rng_for(nblk)
    from torch_amd.blocks import block_centres
    o = rng.uniform(-1, 1, (nblk, 3))
    x, y, z, dx = block_centres(o, rng.uniform(0.01, 0.05, nblk))
    m = rng.uniform(0.5, 1, x.size)
    st = dev(*rng.uniform(-1, 1, (3, 700)), rng.uniform(0.1, 1, 700), np.full(700, 0.01))
    for move in (None, 0, x.size // 2, x.size - 1):
        cx = x.copy()
        if move is not None:
            cx[move] += 1e-3
        c = dev(cx, y, z, m, dx)
        got = []
        for validate in (True, False):
            with StellarGravityField("fp64", validate=validate) as f, GasGravityField("fp64", validate=validate) as g:
                f.set_stars(*st)
                a = f.evaluate(None, c[0], c[1], c[2])
                g.set_sources(*c)
                b = g.evaluate(None, st[0], st[1], st[2])
                f.set_block_kernel(False)
                g.set_block_kernel(False)
                got.append(a + b)
                if validate:
                    plain = f.evaluate(None, c[0], c[1], c[2]) + g.evaluate(None, st[0], st[1], st[2])
        for p, q in zip(*got):
            assert torch.equal(p, q)
        for p, q in zip(got[0], plain):
            assert torch.allclose(p, q, rtol=1e-11, atol=1e-11 * float(q.abs().max()))
        if move is not None:
            assert all(torch.equal(p, q) for p, q in zip(got[0], plain))


@pytest.mark.parametrize("nblk", [1, 5])
def test_block_sources_expand_where_needed(nblk):
    """Block sources under every kernel that reads them cell by cell equal the same cells given as
    points, also after the set is replaced (and through a graph captured before that)."""
    rng = W.rng_for(77 + nblk)
    from torch_amd.blocks import block_centres
    o, d = rng.uniform(-1, 1, (nblk, 3)), rng.uniform(0.02, 0.1, nblk)
    x, y, z, dx = block_centres(o, d)
    to, td = dev(rng.uniform(-1, 1, (2, 3)), np.full(2, 0.03))
    t = dev(*rng.uniform(-1, 1, (3, 300)))
    masses = [rng.uniform(0.5, 1, x.size) for _ in range(2)]
    with GasGravityField("fp64", validate=False) as g, GasGravityField("fp64") as p:
        g.set_block_kernel(False)
        p.set_block_kernel(False)
        outs = None
        graph = torch.cuda.CUDAGraph()
        for step, m in enumerate(masses):
            g.set_blocks(*dev(o, d, m))
            p.set_sources(*dev(x, y, z, m, dx))
            a = g.evaluate(None, *t) + g.evaluate_blocks(to, td)
            b = p.evaluate(None, *t) + p.evaluate_blocks(to, td)
            for q, r in zip(a, b):
                assert torch.equal(q, r)
            if step == 0:
                torch.cuda.synchronize()
                with torch.cuda.graph(graph):
                    outs = g.evaluate(None, *t)
            for _ in range(3):
                graph.replay()
                torch.cuda.synchronize()
                for q, r in zip(outs, b):
                    assert torch.equal(q, r)


def test_scalar_softening_and_origin_layouts():
    """Numbers for the softening (zero among them) and corners in any order or stride give the bits of
    whole vectors; a number that is not finite is still refused."""
    import torch
    rng = np.random.default_rng(12)
    st = [torch.as_tensor(rng.normal(size=200), device="cuda") for _ in range(3)]
    m = torch.ones(200, dtype=torch.float64, device="cuda")
    T = [torch.as_tensor(rng.normal(size=700), device="cuda") for _ in range(3)]
    o = torch.as_tensor(rng.uniform(-2, 2, (5, 3)), device="cuda")
    dx = torch.full((5,), 0.03, dtype=torch.float64, device="cuda")
    wide = torch.zeros(5, 7, dtype=torch.float64, device="cuda")
    wide[:, 1:4] = o
    layouts = [o, o.t().contiguous().t(), wide[:, 1:4], wide[:, 1:], o.cpu(), o.flip(0).flip(0)]
    with StellarGravityField("fp64") as f:
        for eps in (0.0, 0, -0.0, 0.02, np.float64(0.02), np.array(0.02), torch.tensor(0.02, dtype=torch.float64)):
            vec = torch.full((200,), float(eps), dtype=torch.float64, device="cuda")
            f.set_sources(*st, m, eps)
            got = f.evaluate(eps, *T)
            f.set_sources(*st, m, vec)
            ref = f.evaluate(torch.full((700,), float(eps), dtype=torch.float64, device="cuda"), *T)
            for a, b in zip(got, ref):
                assert torch.equal(a, b), eps
        with pytest.raises(TgravError):
            f.evaluate(float("nan"), *T)
        ref = None
        for q, lay in enumerate(layouts):
            got = f.evaluate_blocks(lay, dx)
            ref = ref or got
            for a, b in zip(got, ref):
                assert torch.equal(a, b), q
        with pytest.raises(TgravError):
            f.evaluate_blocks(o, dx[:4])


@pytest.mark.parametrize("nblk", [1, 40])
def test_captured_block_sets_are_whole(nblk):
    """A graph that sets block sources (and evaluates them block by block) sets them for every later call:
    after each replay, eager calls that read the set cell by cell see the masses of that replay."""
    rng = W.rng_for(nblk)
    from torch_amd.blocks import block_centres
    o, d = rng.uniform(-1, 1, (nblk, 3)), rng.uniform(0.02, 0.1, nblk)
    x, y, z, dx = block_centres(o, d)
    to, td = dev(rng.uniform(-1, 1, (2, 3)), np.full(2, 0.03))
    t = dev(*rng.uniform(-1, 1, (3, 300)))
    od, dd, m = dev(o, d, np.ones(x.size))
    with GasGravityField("fp64", validate=False) as g, GasGravityField("fp64") as p:
        g.set_blocks(od, dd, m)
        g.evaluate(None, *t)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            g.set_blocks(od, dd, m)
            outs = g.evaluate(None, *t)
        for step in range(4):
            m.copy_(dev(rng.uniform(0.5, 1, x.size))[0])
            graph.replay()
            torch.cuda.synchronize()
            p.set_blocks(od, dd, m)
            p.set_block_kernel(True)
            for a, b in zip(outs, p.evaluate(None, *t)):
                assert torch.equal(a, b)
            for on in (True, False):                  # block targets, then the generic kernel
                g.set_block_kernel(on)
                p.set_block_kernel(on)
                for a, b in zip(g.evaluate_blocks(to, td), p.evaluate_blocks(to, td)):
                    assert torch.equal(a, b), (step, on)


def test_block_set_read_on_two_streams():
    """Block sources set on one stream and read cell by cell on two others that wait for it."""
    rng = W.rng_for(5)
    from torch_amd.blocks import block_centres
    nblk = 600
    o, d, m = dev(rng.uniform(-1, 1, (nblk, 3)), rng.uniform(0.02, 0.1, nblk), rng.uniform(0.5, 1, nblk * 512))
    to, td = dev(rng.uniform(-1, 1, (1, 3)), np.full(1, 0.03))
    streams = [torch.cuda.Stream() for _ in range(3)]
    with GasGravityField("fp64", validate=False) as g, GasGravityField("fp64") as p:
        for f in (g, p):
            f.set_config(nsplit=1)                    # no partial sums, which calls of a context share
        p.set_blocks(o, d, m)
        ref = p.evaluate_blocks(to, td)
        torch.cuda.synchronize()
        with torch.cuda.stream(streams[0]):
            g.set_blocks(o, d, m)
            ready = streams[0].record_event()
        got = []
        for s in streams[1:]:
            s.wait_event(ready)
            with torch.cuda.stream(s):
                got.append(g.evaluate_blocks(to, td))
        torch.cuda.synchronize()
        for a in got:
            for u, v in zip(a, ref):
                assert torch.equal(u, v)


def test_contexts_made_while_the_null_stream_is_busy():
    """A context is ready for calls on its own stream when it is made, whatever the null stream still has to do."""
    rng = W.rng_for(3)
    st = [rng.uniform(-1, 1, 5000) for _ in range(3)] + [rng.uniform(0.1, 1, 5000), np.full(5000, 0.01)]
    t = [rng.uniform(-1, 1, 400) for _ in range(3)]
    ref = None
    a = torch.ones(4096, 4096, device="cuda")
    for step in range(4):
        with torch.cuda.stream(torch.cuda.default_stream()):
            for _ in range(200 if step else 0):
                a = a * 1.0001
        with StellarGravityField("fp64", validate=bool(step & 1)) as f:
            f.set_stars(*st)                      # host arrays: the context's own stream
            got = f.evaluate(None, *t)
        torch.cuda.synchronize()
        ref = ref or got
        for u, v in zip(got, ref):
            np.testing.assert_array_equal(u, v)


def test_set_and_fused_pass_on_two_streams():
    """A source set and the particles of a fused pass packed at once on two streams of one context: their
    results, and those of the calls after them, are the ones of calls in a row."""
    rng = W.rng_for(4)
    n = 120000
    S = dev(*rng.uniform(-1, 1, (3, n)), rng.uniform(0.1, 1, n), np.full(n, 0.01))
    o, d, m = dev(rng.uniform(-1, 1, (1, 3)), np.full(1, 0.03), rng.uniform(0.5, 1, 512))
    t = dev(*rng.uniform(-1, 1, (3, 40)))
    P = [a[: n - 777].clone() for a in S]
    with StellarGravityField("fp64", validate=False) as f:
        f.set_bidir_config(nsplit=1)               # no chunk sums, which calls of a context share
        f.set_sources(*S)
        want = f.evaluate(None, *t), f.bidirectional_blocks(o, d, m, d, *P)
        torch.cuda.synchronize()
        one, two = torch.cuda.Stream(), torch.cuda.Stream()
        for _ in range(20):
            with torch.cuda.stream(one):
                f.set_sources(*S)
            with torch.cuda.stream(two):
                fused = f.bidirectional_blocks(o, d, m, d, *P)
        torch.cuda.synchronize()
        got = f.evaluate(None, *t)
        for u, v in zip(got, want[0]):
            assert torch.equal(u, v)
        for side in range(2):
            for u, v in zip(fused[side], want[1][side]):
                assert torch.equal(u, v)
