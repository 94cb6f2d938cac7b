"""P2G of few blocks (one nine-wave workgroup per block part, 576 particles a chunk) against P2G of
many blocks (three waves, chunks of 384): the two add the same numbers to a node in the same order,
so a scene alone (few blocks) and the same scene in a batch with 512 blocks of another are
bit-exact, in every transfer.  Sizes: one particle; around one wave, one chunk of either and one
part (1,024); a block of two parts and two chunks each.  With 1,728 blocks of few particles in the
batch the G2P kernels run with 64 threads a part in place of 512 (update) and 256.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from zeno_amd import scenes  # noqa: E402
from zeno_amd.zmpm import (MODEL_FCR, MODEL_JFLUID, TRANSFER_AFLIP, TRANSFER_APIC,  # noqa: E402
                           TRANSFER_FLIP, Context, StepParams)

DEV = "cuda:0"


def one_block(n, seed):
    """n particles of two materials in the 4^3 cells of one block, dx = 1/32."""
    dx = 1.0 / 32
    rng = np.random.default_rng(seed)
    x = ((12.5 + 4.0 * rng.random((3, n))) * dx).astype(np.float32)
    vol = dx ** 3 * 64 / max(n, 8)
    mats = [dict(model=MODEL_FCR, E=4e4, nu=0.3, rho=1000.0, vol=vol, flip_beta=0.5),
            dict(model=MODEL_JFLUID, rho=1000.0, vol=vol, bulk=4e3)]
    st = scenes._state(x, (0.4, -0.6, 0.2), (np.arange(n) % 3 == 2).astype(np.int32),
                       np.array([MODEL_FCR, MODEL_JFLUID]))
    st["v"] = (st["v"] + 0.3 * rng.standard_normal(st["x"].shape)).astype(np.float32)
    return dict(state=st, mats=mats, dx=dx, n_cells=32, dt=1e-4, gravity=(0.0, -9.8, 0.0), pad=3)


def filler(side=32, seed=5):
    """One particle in each of side^3 cells: at least (side / 4)^3 blocks, few particles to be quick."""
    dx = 1.0 / 64
    x = scenes.jitter_cells(scenes.box_cells((8, 8, 8), (8 + side,) * 3), 1, dx, seed)
    mats = [dict(model=MODEL_FCR, E=1e4, nu=0.3, rho=1000.0, vol=dx ** 3)]
    st = scenes._state(x, (0.0, 0.0, 0.0), np.zeros(x.shape[1], np.int32), np.array([MODEL_FCR]))
    return dict(state=st, mats=mats, dx=dx, n_cells=64, dt=1e-4, gravity=(0.0, -9.8, 0.0), pad=3)


def run(ctx, mats, state, params, transfer, steps):
    ctx.set_materials(mats)
    ctx.set_transfer(transfer)
    ctx.import_state({k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for k, v in state.items()})
    ctx.substeps(params, steps)
    nblocks = ctx.num_particle_blocks()
    out = {k: v.cpu().numpy() for k, v in ctx.export_state(DEV).items()}
    ctx.sync()
    ctx.close()
    return out, nblocks


@pytest.mark.parametrize("transfer", [TRANSFER_APIC, TRANSFER_AFLIP, TRANSFER_FLIP])
@pytest.mark.parametrize("n", [1, 63, 65, 383, 385, 575, 576, 577, 1024, 1025, 2300])
def test_few_blocks_equal_many(n, transfer):
    cfg = one_block(n, seed=n)
    steps = 4
    alone, nb = run(Context(cfg["dx"], cfg["n_cells"], n), cfg["mats"], cfg["state"],
                    StepParams(cfg["dt"], cfg["gravity"], 1, cfg["pad"]), transfer, steps)
    assert nb <= 8
    for side in (32, 48):
        descs, mats, st, ranges = scenes.merge_scenes([filler(side), cfg])
        both, nb = run(Context.scenes(descs, st["x"].shape[1]), mats, st, None, transfer, steps)
        assert nb >= (side // 4) ** 3
        a, b = ranges[1]
        for k in ("x", "v", "C", "F"):
            assert np.array_equal(both[k][:, a:b], alone[k], equal_nan=True), (k, side)
