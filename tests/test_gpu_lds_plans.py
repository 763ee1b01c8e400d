"""The bitset search's contexts share a CU's LDS with node storage and with other
launches.  They give way where they do not fit: explicit workgroups keep their
nodes in LDS up to the sizes that fit without contexts (use_global_memory = 0
accepts what it accepted without them), on both sides of every limit; and a
solve beside a server of any size returns while the server runs.  Against the CPU
oracle, whole numbers only; the waits are bounded by the time limits."""
import time

import numpy as np
import pytest

import graphgen
import oracle as O
import vcgpu

pytestmark = pytest.mark.gpu


def _oracle(n, e):
    og = O.from_edges(n, e)
    want, stats, _ = O.mvc(og, max_nodes=2_000_000)
    assert stats["completed"]
    return og, want


def _check(og, r, want, u, where):
    assert r.solved and r.minimum == want, (where, r.minimum, want)
    if r.cover is not None:
        assert O.cover_is_valid(og, np.asarray(r.cover, np.uint8)) and int(np.sum(r.cover)) == want, where
    else:
        assert u == want, where


# threads; the largest n with 256-vertex contexts, with 128-vertex ones and without any
LIMITS = [(1024, (256, 960)), (512, (288, 1248, 2176)), (256, (2368, 3488, 4704)), (128, (7040, 7968, 9760)), (64, (17000, 18900, 19840))]


@pytest.mark.parametrize("block,n", [(b, n + d) for b, ns in LIMITS for n in ns for d in (0, 1) if n + d <= ns[-1]])
def test_explicit_workgroups_keep_nodes_in_lds(ctx, block, n):
    # m = 2: no leaves, and a tree that the oracle finishes
    e = graphgen.barabasi_albert(n, 2, 7)
    og, want = _oracle(n, e)
    g = vcgpu.csr_from_edges(n, e)
    u, _ = vcgpu.upper_bound(g, seed=1)
    gs = ctx.upload(g)
    for gm in (0, -1):
        (r,), info, st = ctx.solve(gs, vcgpu.Job(vcgpu.VC_MVC, 0, u, 0),
                                   vcgpu.Params(block_dim=block, use_global_memory=gm, time_limit_ms=60000), raise_on_error=False)
        assert st == vcgpu.VC_OK, (block, n, gm, st)
        if gm == 0:
            assert info.use_global_memory == 0
        _check(og, r, want, u, (block, n, gm))


def test_workgroups_beyond_lds_are_refused(ctx):
    for block, ns in LIMITS:
        n = ns[-1] + 64
        g = vcgpu.csr_from_edges(n, graphgen.barabasi_albert(n, 2, 7))
        (_,), _, st = ctx.solve(ctx.upload(g), vcgpu.Job(vcgpu.VC_MVC, 0, n - 1, 0),
                                vcgpu.Params(block_dim=block, use_global_memory=0), raise_on_error=False)
        assert st == vcgpu.VC_ENOTSUP, (block, n, st)


@pytest.mark.parametrize("n", [127, 128, 129, 160, 200, 256])
def test_small_contexts_match_oracle(ctx, n):
    """A 1,024-thread workgroup has room for 128-vertex contexts only."""
    for e in (graphgen.erdos_renyi(n, 5.0 / n, 31 + n), graphgen.erdos_renyi(n, 0.7, 32 + n)):
        og, want = _oracle(n, e)
        gs = ctx.upload([vcgpu.csr_from_edges(n, e)] * 3)
        jobs = [vcgpu.Job(vcgpu.VC_MVC, 0, n - 1, 0), vcgpu.Job(vcgpu.VC_PVC, want - 1, n - 1, 0), vcgpu.Job(vcgpu.VC_PVC, want, n - 1, 0)]
        (mvc, no, yes), info, st = ctx.solve(gs, jobs, vcgpu.Params(block_dim=1024, use_global_memory=0, time_limit_ms=60000))
        assert st == vcgpu.VC_OK and info.use_global_memory == 0
        _check(og, mvc, want, n - 1, n)
        assert no.solved and not no.k_found and yes.solved and yes.k_found and int(np.sum(yes.cover)) == want


@pytest.mark.parametrize("max_vertices", [400, 4000, 4700, 6000, 20000])
def test_solve_beside_a_server_returns(ctx, max_vertices):
    """Servers of up to about 4,700 vertices leave half the CUs free, larger ones
    some LDS on every CU."""
    def sparse(n, c, seed):
        p = np.random.default_rng(seed).integers(0, n, size=(int(n * c / 2), 2))
        return np.unique(np.sort(p[p[:, 0] != p[:, 1]], axis=1), axis=0).astype(np.uint32)

    sizes = [(120, graphgen.regular3_rewired(120, 3)), (400, sparse(400, 2.5, 4)), (24001, sparse(24001, 1.5, 5))]
    cases = [(n, e) + _oracle(n, e) for n, e in sizes]
    sets = [ctx.upload(vcgpu.csr_from_edges(n, e)) for n, e, _, _ in cases]
    srv = vcgpu.Server(ctx, max_vertices=max_vertices, slots=16, arena_bytes=16 << 20, stack_depth=300, time_limit_ms=20000)
    try:
        got = []
        for gs, (n, e, og, want) in zip(sets, cases):
            t = time.monotonic()
            (r,), _, _ = ctx.solve(gs, vcgpu.Job(vcgpu.VC_MVC, 0, n - 1, 0), vcgpu.Params(time_limit_ms=10000), raise_on_error=False)
            got.append((r, time.monotonic() - t))
        g0 = vcgpu.csr_from_edges(120, sizes[0][1])
        served, _ = srv.wait(srv.submit(g0, vcgpu.Job(vcgpu.VC_MVC, 0, 119, 0)), 20000)
    finally:
        srv.stop()
    for (r, t), (n, e, og, want) in zip(got, cases):
        _check(og, r, want, n - 1, (max_vertices, n))
        assert t < 5.0, (max_vertices, n, t)
    assert served.solved and served.minimum == cases[0][3]
