"""A captured graph keeps the kernels chosen for the block counts at its capture; replayed while the
particles spread over several times as many blocks, it gives what eager substeps give, which choose anew
(bit-exact)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from zeno_amd import scenes  # noqa: E402
from zeno_amd.zmpm import MODEL_JFLUID, Context, StepParams  # noqa: E402

DEV = "cuda:0"


# side^3 cells of 8 particles: from 27 and 216 parts (nine waves a part) to more than 256 and 512
@pytest.mark.parametrize("side,parts", [(8, 128), (20, 513)])
def test_graph_replayed_over_growing_counts(side, parts):
    cells, steps, dt, grow = 128, 200, 2e-4, 2.2 if side == 8 else 1.7
    dx = 1.0 / cells
    x = scenes.jitter_cells(scenes.box_cells(((cells - side) // 2,) * 3, ((cells + side) // 2,) * 3), 8, dx, 3)
    n = x.shape[1]
    rate = (grow - 1.0) / (steps * dt)
    st = scenes._state(x, (0.0, 0.0, 0.0), np.zeros(n, np.int32), np.array([MODEL_JFLUID]))
    st["v"] = ((x - x.mean(axis=1, keepdims=True)) * rate).astype(np.float32)
    st["C"][[0, 4, 8]] = rate
    st = {k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for k, v in st.items()}
    p = StepParams(dt, (0.0, 0.0, 0.0), 1, 3)
    runs = []
    for graph in (False, True):
        ctx = Context(dx, cells, n)
        ctx.set_materials([dict(model=MODEL_JFLUID, rho=1000.0, vol=dx ** 3 / 8, bulk=1e-3)])
        ctx.import_state(st)
        first = ctx.num_block_parts()
        if graph:
            ctx.graph_capture(p, 10)
        for k in range(steps // 10):
            if graph:
                ctx.graph_launch()
            else:
                ctx.substeps(p, 10)
            if k % 5 == 0:
                ctx.sync()
        assert first <= 256 and ctx.num_block_parts() >= max(parts, 2 * first)
        runs.append(ctx.export_state(DEV))
        ctx.close()
    for k in runs[0]:
        assert torch.equal(runs[0][k], runs[1][k]), k
