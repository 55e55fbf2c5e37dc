"""tgrav_eval_static under capture: its replays need nothing of the context it was captured with and share
nothing with that context's other calls (needs an MI355X)."""
import ctypes

import numpy as np
import pytest

from torch_amd import _lib
from torch_amd import workloads as W

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def dev(a):
    return torch.as_tensor(np.ascontiguousarray(a), device="cuda")


def create(lib):
    ctx = ctypes.c_void_p()
    _lib.check(lib.tgrav_create(ctypes.byref(ctx), 0, None), "tgrav_create")
    return ctx


def bind(lib, ctx):
    s = torch.cuda.current_stream().cuda_stream
    _lib.check(lib.tgrav_set_stream(ctx, ctypes.c_void_p(s or None)), "tgrav_set_stream")


def make(ns, nt, seed):
    rng = W.rng_for(seed)
    S = [dev(a) for a in rng.uniform(-1, 1, (3, ns))] + [dev(rng.uniform(0.1, 1, ns)), dev(rng.uniform(0.01, 0.1, ns))]
    T = [dev(a) for a in rng.uniform(-1, 1, (3, nt))]
    return S, T, [torch.full((nt,), np.nan, dtype=torch.float64, device="cuda") for _ in range(4)]


def static(lib, ctx, S, T, out, mode):
    bind(lib, ctx)
    _lib.check(lib.tgrav_eval_static(ctx, S[0].numel(), *[_p(a) for a in S], T[0].numel(), None,
                                     *[_p(a) for a in T], *[_p(a) for a in out], mode), "tgrav_eval_static")


@pytest.mark.parametrize("mode", [_lib.PLAIN_FP64, _lib.MIXED])
@pytest.mark.parametrize("ns", [200, 5000, 200000])        # one, some and the most workgroups of the packing
def test_replays_outlive_the_context(mode, ns):
    lib = _lib.load()
    S, T, out = make(ns, 700, ns + mode)
    ref = [torch.empty_like(a) for a in out]
    ctx, other = create(lib), create(lib)
    try:
        static(lib, ctx, S, T, out, mode)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            static(lib, ctx, S, T, out, mode)
        lib.tgrav_destroy(ctx)
        ctx = None
        for step in range(3):
            S[3].mul_(1.5)
            S[4].mul_(0.5 if step < 2 else 0.0)           # at the end unsoftened: the statistics change
            for a in out:
                a.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            got = [a.clone() for a in out]
            static(lib, other, S, T, ref, mode)
            torch.cuda.synchronize()
            for a, b in zip(got, ref):
                assert torch.isfinite(a).all() and torch.equal(a, b)
    finally:
        for c in (ctx, other):
            if c:
                lib.tgrav_destroy(c)


def test_replay_beside_the_contexts_own_calls():
    """Replays on one stream while the context sets sources on another: both sides' results stay right, and
    so do the context's later calls."""
    lib = _lib.load()
    mode = _lib.PLAIN_FP64
    S, T, out = make(150000, 300, 1)
    P, Q, own = make(140000, 300, 2)
    ctx = create(lib)
    try:
        _lib.check(lib.tgrav_set_validation(ctx, 0), "tgrav_set_validation")
        side = torch.cuda.Stream()
        static(lib, ctx, S, T, out, mode)
        want = []
        for src, tgt in ((S, T), (P, Q)):
            _lib.check(lib.tgrav_set_sources(ctx, src[0].numel(), *[_p(a) for a in src], _lib.DEVICE), "set")
            res = [torch.empty_like(a) for a in own]
            _lib.check(lib.tgrav_eval(ctx, 300, None, *[_p(a) for a in tgt], *[_p(a) for a in res], mode,
                                      _lib.DEVICE), "tgrav_eval")
            torch.cuda.synchronize()
            want.append([a.clone() for a in res])
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            static(lib, ctx, S, T, out, mode)
        bind(lib, ctx)
        torch.cuda.synchronize()
        for _ in range(20):
            with torch.cuda.stream(side):
                graph.replay()
            for _ in range(3):
                _lib.check(lib.tgrav_set_sources(ctx, P[0].numel(), *[_p(a) for a in P], _lib.DEVICE), "set")
        _lib.check(lib.tgrav_eval(ctx, 300, None, *[_p(a) for a in Q], *[_p(a) for a in own], mode, _lib.DEVICE),
                   "tgrav_eval")
        torch.cuda.synchronize()
        for got, ref in ((out, want[0]), (own, want[1])):
            for a, b in zip(got, ref):
                assert torch.equal(a, b)
    finally:
        lib.tgrav_destroy(ctx)
