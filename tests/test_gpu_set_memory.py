"""Graph sets take their memory from blocks of sets freed before: sets that
live at the same time and are freed in any order keep their own data, below and
above the size that is kept."""
import random

import numpy as np
import pytest

import graphgen
import oracle as O
import vcgpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 40, 400])
def test_sets_freed_in_any_order_keep_their_data(ctx, count):
    rng = random.Random(count)
    graphs = []
    for i in range(6):
        n = 30 + 5 * i
        e = graphgen.erdos_renyi(n, 0.2, 900 + i)
        og = O.from_edges(n, e)
        want, stats, _ = O.mvc(og, max_nodes=2_000_000)
        assert stats["completed"]
        graphs.append((n, vcgpu.csr_from_edges(n, e), og, want))
    alive = []
    for step in range(30):
        i = rng.randrange(len(graphs))
        alive.append((i, ctx.upload([graphs[i][1]] * count)))
        if len(alive) > 4:
            alive.pop(rng.randrange(len(alive)))
        i, gs = alive[rng.randrange(len(alive))]
        n, _, og, want = graphs[i]
        res, _, st = ctx.solve(gs, [vcgpu.Job(vcgpu.VC_MVC, 0, n - 1, 0)] * count, vcgpu.Params(time_limit_ms=60000))
        assert st == vcgpu.VC_OK
        assert all(r.solved and r.minimum == want for r in res)
        assert O.cover_is_valid(og, np.asarray(res[-1].cover, np.uint8))
