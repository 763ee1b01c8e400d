"""The root reduction of large sparse graphs over a workgroup (shrink_kernel)
around its limits: the smallest size that takes it (1,024 vertices), the
largest whose degrees are in LDS (36,864), graphs that it reduces to nothing
and graphs that it leaves a part of, one and several graphs in a set.  MVC,
PVC at k = MVC - 1, MVC and below the rules' own cover, and a bound that is
already optimal, against the CPU oracle; every cover is checked.  All answers
are whole numbers: no tolerance."""
import numpy as np
import pytest

import oracle as O
import vcgpu

pytestmark = pytest.mark.gpu


def _pairs(n, m, seed):
    rng = np.random.default_rng(seed)
    p = rng.integers(0, n, size=(2 * m + 64, 2))
    p = np.unique(np.sort(p[p[:, 0] != p[:, 1]], axis=1), axis=0)
    return rng.permutation(p)[:m].astype(np.uint32)


def _graph(kind, n, seed):
    if kind == "sparse":  # the rules leave nothing
        return _pairs(n, int(0.75 * n), seed)
    if kind == "core":  # a 3-regular-like core of 40 vertices inside a sparse graph
        e = _pairs(n - 40, int(0.7 * n), seed)
        core = _pairs(40, 70, seed + 1) + np.uint32(n - 40)
        return np.concatenate([e, core]).astype(np.uint32)
    # isolated edges, triangles and a star
    e = [(2 * i, 2 * i + 1) for i in range(100)]
    for t in range(200, 500, 3):
        e += [(t, t + 1), (t + 1, t + 2), (t, t + 2)]
    e += [(n - 1, v) for v in range(500, n - 1)]
    return np.asarray(e, np.uint32)


def _check(og, n, r, want, where):
    assert r.cover is not None, where
    assert O.cover_is_valid(og, np.asarray(r.cover, np.uint8)), where
    assert int(np.sum(r.cover)) == want, where


@pytest.mark.parametrize("kind", ["sparse", "core", "pieces"])
@pytest.mark.parametrize("n", [1023, 1024, 1025, 5000, 36864, 36865])
def test_shrunk_graphs_match_oracle(ctx, n, kind):
    e = _graph(kind, n, 70 + n)
    og = O.from_edges(n, e)
    want, stats, _ = O.mvc(og, max_nodes=200_000)
    assert stats["completed"]
    g = vcgpu.csr_from_edges(n, e)
    params = vcgpu.Params(time_limit_ms=60000)
    jobs = [vcgpu.Job(vcgpu.VC_MVC, 0, min(n, want + 3), 0), vcgpu.Job(vcgpu.VC_MVC, 0, want, 0),
            vcgpu.Job(vcgpu.VC_PVC, want - 1, want + 1, 0), vcgpu.Job(vcgpu.VC_PVC, want, want + 1, 0),
            vcgpu.Job(vcgpu.VC_PVC, 0, want + 1, 0)]
    one = ctx.upload(g)
    alone = [ctx.solve(one, j, params)[0][0] for j in jobs]
    together, _, st = ctx.solve(ctx.upload([g] * len(jobs)), jobs, params)
    assert st == vcgpu.VC_OK
    for mvc, tight, no, yes, zero in (alone, together):
        for r in (mvc, tight, no, yes, zero):
            assert r.solved and r.status == vcgpu.VC_OK, (n, kind)
        assert mvc.minimum == want, (n, kind, mvc.minimum, want)
        _check(og, n, mvc, want, (n, kind))
        assert tight.minimum == want and tight.cover is None, (n, kind)  # nothing below the bound
        assert not no.k_found and not zero.k_found, (n, kind)
        assert yes.k_found and yes.minimum == want, (n, kind)
        _check(og, n, yes, want, (n, kind))
