"""The Morton reordering beside a simulation on another stream: it shares no buffer with the substeps and
the export, so either may run while the other waits on its stream, and both come out as they do alone
(bit-exact).  The waiting stream is held by a kernel that only lets time pass."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from zeno_amd import scenes  # noqa: E402
from zeno_amd.zmpm import LAYOUT_AOSOA32, MODEL_FCR, Context, StepParams  # noqa: E402

DEV = "cuda:0"
DX = 1.0 / 128
NCH = 20
HOLD = 20_000_000  # clock cycles


def simulation(n):
    x = scenes.jitter_cells(scenes.box_cells((10, 10, 10), (36, 36, 36)), 8, DX, 3)[:, :n]
    rng = np.random.default_rng(n)
    st = scenes._state(x, (0.3, -0.5, 0.2), np.zeros(n, np.int32), np.array([MODEL_FCR]))
    p = rng.permutation(n)
    st = {k: torch.from_numpy(np.ascontiguousarray(v[..., p])).to(DEV) for k, v in st.items()}
    ctx = Context(DX, 128, n)
    ctx.set_materials([dict(model=MODEL_FCR, E=2e4, nu=0.3, rho=1000.0, vol=DX ** 3 / 8)])
    ctx.import_state(st)
    return ctx


@pytest.mark.parametrize("reorder_waits", [True, False])
@pytest.mark.parametrize("n", [65536, 131071])
def test_reordering_beside_substeps(n, reorder_waits):
    p = StepParams(1e-4, (0.0, -9.8, 0.0), 1, 3)
    alone = simulation(n)
    alone.substeps(p, 3)
    want = alone.export_state(DEV)
    alone.close()

    g = torch.Generator(device=DEV).manual_seed(n)
    src = torch.rand(-(-n // 32), NCH, 32, generator=g, device=DEV)
    dst = torch.zeros_like(src)
    codes, order, inv = (torch.empty(n, dtype=torch.int32, device=DEV) for _ in range(3))
    ctx = simulation(n)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()

    def reorder():
        ctx.order_by_morton_code(LAYOUT_AOSOA32, NCH, n, src, dst, 1, (0.0, 0.0, 0.0), (1.0, 1.0, 1.0), codes, order,
                                 inv)

    def substeps():
        ctx.substeps(p, 3)  # an odd number: the state ends in the buffer that was free before

    first, second = (reorder, substeps) if reorder_waits else (substeps, reorder)
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        torch.cuda._sleep(HOLD)
    ctx.set_stream(a.cuda_stream)
    first()
    ctx.set_stream(b.cuda_stream)
    second()
    if not reorder_waits:
        torch.cuda.synchronize()
    with torch.cuda.stream(b):
        got = ctx.export_state(DEV)
    torch.cuda.synchronize()
    for k in want:
        assert torch.equal(got[k], want[k]), k
    assert torch.equal(torch.sort(order.long())[0], torch.arange(n, device=DEV))
    i = torch.arange(n, device=DEV)
    o = order.long()
    assert torch.equal(dst[i // 32, :, i % 32], src[o // 32, :, o % 32])
    ctx.close()
