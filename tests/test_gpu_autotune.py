"""The autotuner keeps the automatic workgroup where the shapes differ by less
than two runs of one do (it once took the first that happened to be faster)."""
import pytest

import graphgen
import vcgpu

pytestmark = pytest.mark.gpu


def test_equal_shapes_leave_the_automatic_workgroup():
    # 64, 128 and 256 threads differ by less than 5% on these
    graphs = [graphgen.batch_graph(i, 1000) for i in range(512)]
    graphs = [vcgpu.csr_from_edges(n, e) for n, e, _ in graphs]
    jobs = [vcgpu.Job(vcgpu.VC_MVC, 0, vcgpu.upper_bound(g, seed=1)[0], 1 << 20) for g in graphs]
    with vcgpu.Context(0) as own:  # shapes are cached per context
        gs = own.upload(graphs)
        _, info, _ = own.solve(gs, jobs, vcgpu.Params(time_limit_ms=60000), want_covers=False, raise_on_error=False)
        best, ms = own.autotune(gs, jobs, vcgpu.Params(time_limit_ms=60000))
        gs.free()
    assert ms > 0 and best.block_dim == info.block_dim and best.use_global_memory == 0, (best, info.block_dim)
