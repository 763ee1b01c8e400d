"""Sets in which some graphs have a node budget and others have not: solved in two
launches (one when the budgets are small), with the results, covers and limits
of one.  Against the CPU oracle, whole numbers only."""
import numpy as np
import pytest

import graphgen
import oracle as O
import vcgpu

pytestmark = pytest.mark.gpu


def _cases(count, seed):
    out = []
    for i in range(count):
        n = 30 + (7 * i) % 60
        e = graphgen.erdos_renyi(n, 0.12, seed + i) if i % 2 else graphgen.barabasi_albert(n, 2, seed + i)
        og = O.from_edges(n, e)
        want, stats, _ = O.mvc(og, max_nodes=2_000_000)
        assert stats["completed"]
        out.append((n, vcgpu.csr_from_edges(n, e), og, want))
    return out


@pytest.mark.parametrize("flags", [0, vcgpu.VC_FLAG_GRAPH])
@pytest.mark.parametrize("version", [vcgpu.VC_HYBRID, vcgpu.VC_STACK_ONLY])
@pytest.mark.parametrize("budget", [1 << 10, 1 << 20])
def test_mixed_sets_match_oracle(ctx, budget, version, flags):
    cases = _cases(21, 77)
    gs = ctx.upload([c[1] for c in cases])
    params = vcgpu.Params(version=version, start_depth=2, time_limit_ms=60000, flags=flags)
    for call, with_budget in enumerate([lambda i: i % 3 == 0, lambda i: i != 4, lambda i: i == 4, lambda i: i % 3 == 0, lambda i: True]):
        jobs, yes = [], []
        for i, (n, g, og, want) in enumerate(cases):
            k = want - (i + call) % 2
            pvc = i % 4 == 1
            yes.append(k >= want)
            jobs.append(vcgpu.Job(vcgpu.VC_PVC if pvc else vcgpu.VC_MVC, k if pvc else 0, n - 1, budget if with_budget(i) else 0))
        res, info, st = ctx.solve(gs, jobs, params)
        assert st == vcgpu.VC_OK
        assert info.tree_nodes == sum(r.tree_nodes for r in res)
        for i, (r, (n, g, og, want)) in enumerate(zip(res, cases)):
            if not r.solved:
                # only at the small budget, and only where it ran out
                assert jobs[i].max_nodes == 1 << 10 and r.tree_nodes >= 900 and r.status == vcgpu.VC_ETIMEOUT, (call, i)
                assert r.minimum >= want or jobs[i].instance == vcgpu.VC_PVC
            elif jobs[i].instance == vcgpu.VC_PVC:
                assert bool(r.k_found) == yes[i], (call, i)
            else:
                assert r.minimum == want, (call, i)
            if r.cover is not None:
                assert O.cover_is_valid(og, np.asarray(r.cover, np.uint8)) and int(np.sum(r.cover)) == r.minimum, (call, i)


def test_mixed_sets_refuse_what_they_refused(ctx):
    cases = _cases(3, 5)
    gs = ctx.upload([c[1] for c in cases])
    for bad in (vcgpu.Job(vcgpu.VC_MVC, 0, cases[2][0] + 1, 0), vcgpu.Job(7, 0, 5, 0)):
        jobs = [vcgpu.Job(vcgpu.VC_MVC, 0, cases[0][0], 1 << 20), vcgpu.Job(vcgpu.VC_MVC, 0, cases[1][0], 0), bad]
        _, _, st = ctx.solve(gs, jobs, vcgpu.Params(), raise_on_error=False)
        assert st == vcgpu.VC_EINVAL


def test_one_graph_without_a_budget_does_not_slow_the_others(ctx):
    """It once gave the whole launch the bitset search's grid, a seventh of the
    workers that the budgets' general search needs: five times the time."""
    graphs = [graphgen.batch_graph(i, 1000) for i in range(1024)]
    graphs = [vcgpu.csr_from_edges(n, e) for n, e, _ in graphs]
    small = min(range(1024), key=lambda i: graphs[i].n)
    gs = ctx.upload(graphs)
    jobs = [vcgpu.Job(vcgpu.VC_MVC, 0, vcgpu.upper_bound(g, seed=1)[0], 1 << 17) for g in graphs]
    params = vcgpu.Params(time_limit_ms=60000)
    ms = []
    for free in ([], [small]):
        jobs = [vcgpu.Job(vcgpu.VC_MVC, 0, j.upper_bound, 0 if i in free else 1 << 17) for i, j in enumerate(jobs)]
        runs = [ctx.solve(gs, jobs, params, want_covers=False, raise_on_error=False) for _ in range(2)]
        ms.append(min(info.kernel_ms for _, info, _ in runs))
        assert all(r.solved or j.max_nodes for r, j in zip(runs[-1][0], jobs))
    assert ms[1] < 2.0 * ms[0], ms
