"""Substeps beside kernels of other streams that take up the chip: the lattice scan's workgroups then start
late and apart.  The result is the one of the simulation alone, bit for bit, and no state error is raised;
lattices of two and of 63 tiles of 1,024 entries, and of 62 and 67 tiles of 4,096."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from zeno_amd import scenes  # noqa: E402
from zeno_amd.zmpm import MODEL_JFLUID, Context, StepParams  # noqa: E402

DEV = "cuda:0"


# entries: (ceil(cells / 4) + 3)^3 = 11^3 = 1,331; 40^3 = 64,000; 63^3 = 250,047; 65^3 = 274,625
@pytest.mark.parametrize("n_cells", [32, 148, 240, 248])
def test_scan_beside_other_streams(n_cells):
    n, dx = 4000, 1.0 / n_cells
    rng = np.random.default_rng(n_cells)
    x = (5 + (n_cells - 10) * rng.random((3, n))) * dx
    st = scenes._state(x.astype(np.float32), (0.0, 0.0, 0.0), np.zeros(n, np.int32), np.array([MODEL_JFLUID]))
    st["v"] = (0.5 * dx / 1e-3 * rng.uniform(-1, 1, (3, n))).astype(np.float32)
    st = {k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for k, v in st.items()}
    p = StepParams(1e-3, (0.0, 0.0, 0.0), 1, 3)

    def run(busy):
        ctx = Context(dx, n_cells, n)
        ctx.set_materials([dict(model=MODEL_JFLUID, rho=1000.0, vol=dx ** 3, bulk=1e-3)])
        ctx.import_state(st)
        s = torch.cuda.Stream()
        others = [torch.cuda.Stream() for _ in range(2)] if busy else []
        work = [torch.ones(1 << 24, device=DEV) for _ in others]
        torch.cuda.synchronize()
        for o, t in zip(others, work):
            with torch.cuda.stream(o):
                for _ in range(100):
                    t.mul_(1.0)
        ctx.set_stream(s.cuda_stream)
        ctx.substeps(p, 10)
        ctx.sync()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            out = ctx.export_state(DEV)
        torch.cuda.synchronize()
        ctx.close()
        return out

    alone, beside = run(False), run(True)
    for k in alone:
        assert torch.equal(alone[k], beside[k]), k
