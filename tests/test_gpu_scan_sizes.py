"""The lattice scan at the edges of its two forms: lattices just below and above 65,536 entries (64 tiles
of 1,024, every one visited; 4,096-entry tiles, empty ones skipped, above) and 262,144 (tiles by
workgroup number; by ticket), and batches whose scenes begin inside a tile.  Bars: the partition's
block ids equal the host's (NumPy) over several re-bins of moving particles; a batch equals its scenes
alone, bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from zeno_amd import scenes  # noqa: E402
from zeno_amd.zmpm import MODEL_JFLUID, Context, StepParams  # noqa: E402

DEV = "cuda:0"


def fluid(n_cells, n, seed):
    """n J-fluid particles anywhere inside the domain (far blocks, most entries empty), moving fast."""
    dx = 1.0 / n_cells
    rng = np.random.default_rng(seed)
    x = (5 + (n_cells - 10) * rng.random((3, n))) * dx
    st = scenes._state(x.astype(np.float32), (0.0, 0.0, 0.0), np.zeros(n, np.int32), np.array([MODEL_JFLUID]))
    st["v"] = (0.5 * dx / 1e-3 * rng.uniform(-1, 1, (3, n))).astype(np.float32)
    return dict(state=st, mats=[dict(model=MODEL_JFLUID, rho=1000.0, vol=dx ** 3, bulk=1e-3)], dx=dx,
                n_cells=n_cells, dt=1e-3, gravity=(0.0, 0.0, 0.0), pad=3)


# entries: (ceil(cells / 4) + 3)^3 = 40^3 = 64,000; 41^3 = 68,921; 63^3 = 250,047; 65^3 = 274,625
@pytest.mark.parametrize("n_cells", [8, 148, 152, 240, 248])
def test_block_count_follows_the_particles(n_cells):
    cfg = fluid(n_cells, 5000 if n_cells > 8 else 40, n_cells)
    n = cfg["state"]["x"].shape[1]
    ctx = Context(cfg["dx"], n_cells, n)
    ctx.set_materials(cfg["mats"])
    ctx.import_state({k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for k, v in cfg["state"].items()})
    p = StepParams(cfg["dt"], cfg["gravity"], 1, cfg["pad"])
    for steps in (0, 1, 1, 6):
        ctx.substeps(p, steps)
        x = ctx.export_state(DEV)["x"].cpu().numpy()
        b = (np.floor((x * np.float32(1.0 / np.float32(cfg["dx"]))).astype(np.float64) - 0.5).astype(np.int64)) >> 2
        want = np.unique((b[0] * 512 + b[1]) * 512 + b[2]).size
        assert ctx.num_particle_blocks() == want
    ctx.close()


@pytest.mark.parametrize("cells", [(8, 8, 12, 8, 30), (100, 8, 140, 9, 8)])
def test_batch_equals_scenes_alone(cells):
    cfgs = [fluid(c, 200 if c > 12 else 30, 7 * k + c) for k, c in enumerate(cells)]
    descs, mats, st, ranges = scenes.merge_scenes(cfgs)
    ctx = Context.scenes(descs, st["x"].shape[1])
    ctx.set_materials(mats)
    ctx.import_state({k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for k, v in st.items()})
    ctx.substeps(None, 5)
    both = {k: v.cpu().numpy() for k, v in ctx.export_state(DEV).items()}
    ctx.close()
    for cfg, (a, b) in zip(cfgs, ranges):
        ctx = Context(cfg["dx"], cfg["n_cells"], b - a)
        ctx.set_materials(cfg["mats"])
        ctx.import_state({k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for k, v in cfg["state"].items()})
        ctx.substeps(StepParams(cfg["dt"], cfg["gravity"], 1, cfg["pad"]), 5)
        alone = {k: v.cpu().numpy() for k, v in ctx.export_state(DEV).items()}
        ctx.close()
        for k in ("x", "v", "C", "F"):
            assert np.array_equal(both[k][:, a:b], alone[k]), k
