"""What a 128-byte record of an import or export carries, beside x, v, C and F / J: the optional
attributes, in either direction, with one object and with several of which only some have or ask for an
attribute; and a loaded state that holds caller indices beyond the particle count.  All of it moves values,
so everything here is bit-exact."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from zeno_amd import scenes  # noqa: E402
from zeno_amd.zmpm import (LAYOUT_AOS, LAYOUT_AOSOA32, LAYOUT_SOA, MODEL_FCR, MODEL_JFLUID,  # noqa: E402
                           MODEL_STVK_HENCKY, PLASTIC_CAM_CLAY, TRANSFER_AFLIP, Context, particle_view)

DEV = "cuda:0"
DX = 1.0 / 128
VOL = DX ** 3 / 8
AUX = ("beta", "logJp", "mu", "lam", "m", "vol")
WIDTH = dict(x=3, v=3, C=9, F=9, J=1, beta=1, logJp=1, mu=1, lam=1, m=1, vol=1)
BETA = (0.25, 0.5)  # the materials' flip_beta


def particles(n, seed):
    """n particles in no spatial order, every attribute a different random value; two materials."""
    x = scenes.jitter_cells(scenes.box_cells((10, 10, 10), (37, 37, 37)), 8, DX, 3)[:, :n]
    rng = np.random.default_rng(seed)
    p = {k: rng.uniform(0.5, 2.0, (c, n)).astype(np.float32) for k, c in WIDTH.items()}
    p["x"] = x[:, rng.permutation(n)].astype(np.float32)
    out = {k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for k, v in p.items()}
    out["mat"] = torch.from_numpy((rng.random(n) < 0.4).astype(np.int32)).to(DEV)  # 1: fluid
    return out


def context(n):
    ctx = Context(DX, 128, n)
    ctx.set_materials([dict(model=MODEL_STVK_HENCKY, E=2e4, nu=0.3, rho=1000.0, vol=VOL, plasticity=PLASTIC_CAM_CLAY,
                            friction_angle=35.0, nacc_beta=0.5, nacc_xi=1.0, flip_beta=BETA[0]),
                       dict(model=MODEL_JFLUID, rho=800.0, vol=VOL, bulk=4e3, flip_beta=BETA[1])])
    ctx.set_transfer(TRANSFER_AFLIP)  # the particles' beta is kept
    return ctx


class Object:
    """Particles a .. b as a view of one layout that has the attributes `names`; fill: no values yet."""

    def __init__(self, p, a, b, layout, names, fill=None):
        self.n, self.layout, self.names = b - a, layout, names
        rows = {k: p[k][:, a:b] if fill is None else torch.full((WIDTH[k], b - a), fill, device=DEV) for k in names}
        kw = {}
        if layout == LAYOUT_AOSOA32:
            flat = torch.cat([rows[k] for k in names])
            chn, c = {}, 0
            for k in names:
                chn[k], c = c, c + WIDTH[k]
            tile = torch.zeros(-(-self.n // 32), c, 32, device=DEV)
            i = torch.arange(self.n, device=DEV)
            tile[i // 32, :, i % 32] = flat.t()
            self.buf = {k: tile for k in names}
            self.chn, kw = chn, dict(tile_channels=c, chn=chn)
        else:
            self.buf = {k: (r.t() if layout == LAYOUT_AOS else r).contiguous() for k, r in rows.items()}
        self.mat = p["mat"][a:b].contiguous()
        self.view = particle_view(self.n, *[self.buf.get(k) for k in ("x", "v", "C", "F", "J")], self.mat,
                                  layout=layout, **{k: self.buf.get(k) for k in AUX}, **kw)

    def rows(self, k):
        if self.layout == LAYOUT_AOSOA32:
            t = self.buf[k].permute(1, 0, 2).reshape(self.buf[k].shape[1], -1)
            return t[self.chn[k]:self.chn[k] + WIDTH[k], :self.n]
        return self.buf[k].t() if self.layout == LAYOUT_AOS else self.buf[k]


BASE = ("x", "v", "C", "F", "J")
ONE = [(LAYOUT_SOA, AUX, AUX), (LAYOUT_AOSOA32, AUX, ("logJp", "m", "vol")), (LAYOUT_AOS, (), AUX)]
MIXED = [(LAYOUT_AOSOA32, ("beta", "mu", "lam", "m", "vol"), AUX), (LAYOUT_SOA, ("logJp", "mu", "lam"), ("beta",)),
         (LAYOUT_AOS, AUX, ()), (LAYOUT_SOA, ("beta", "logJp", "mu", "lam", "m", "vol"), ("mu", "lam", "logJp"))]


def expected(p, n, objects, cuts):
    """What an export holds, by attribute: the imported value, or the material's where it was not given."""
    fluid = p["mat"] == 1
    want = {k: p[k].clone() for k in BASE}
    E, nu = 2e4, 0.3
    for k in AUX:
        group = dict(mu=("mu", "lam"), lam=("mu", "lam"), m=("m", "vol"), vol=("m", "vol")).get(k, (k,))
        whole = all(set(group) <= set(names) for _, names, _ in objects)  # per particle when every object has it
        w = torch.empty(1, n, device=DEV)
        for (_, names, _), a, b in zip(objects, cuts, cuts[1:]):
            f = fluid[a:b]
            if k in names and (whole or k in ("beta", "logJp")):
                w[:, a:b] = p[k][:, a:b]
            elif k == "beta":
                w[0, a:b] = torch.where(f, BETA[1], BETA[0])
            elif k == "logJp":
                w[:, a:b] = -0.04
            elif k in ("m", "vol"):
                w[0, a:b] = torch.where(f, *(np.float32(q * VOL).item() for q in (800.0, 1000.0))) if k == "m" else VOL
            else:
                w[:, a:b] = float("nan")  # the material's Lame parameters: not looked at
        want[k] = w
    return want


@pytest.mark.parametrize("n", [65536, 131071])
@pytest.mark.parametrize("objects", [ONE[0:1], ONE[1:2], ONE[2:3], MIXED], ids=["soa", "tiles", "defaults", "several"])
def test_every_attribute(n, objects):
    p = particles(n, n + len(objects))
    cuts = [0, n] if len(objects) == 1 else [0, 33, 30001, 50000, n]
    ctx = context(n)
    given = [Object(p, a, b, lay, BASE + tuple(names)) for (lay, names, _), a, b in zip(objects, cuts, cuts[1:])]
    ctx.import_objects([o.view for o in given])
    got = [Object(p, a, b, lay, BASE + tuple(ask), fill=-7.0) for (lay, _, ask), a, b in zip(objects, cuts, cuts[1:])]
    ctx.export_objects([o.view for o in got])
    want = expected(p, n, objects, cuts)
    for o, a, b in zip(got, cuts, cuts[1:]):
        fluid = p["mat"][a:b] == 1
        for k in o.names:
            r, w = o.rows(k), want[k][:, a:b]
            if k in ("F", "J"):  # F of solid and J of fluid particles; the others stay as they were
                own = fluid if k == "J" else ~fluid
                assert torch.equal(r[:, own], w[:, own]), k
                assert bool((r[:, ~own] == -7.0).all()), k
            elif not bool(w.isnan().any()):
                assert torch.equal(r, w.contiguous()), (o.layout, k)
    ctx.close()


def test_caller_index_beyond_the_count():
    """A state saved with more particles, loaded after an import of fewer: an export writes the particles
    whose caller index is below the count and leaves the other entries as they were."""
    many, n = 140001, 70001
    rng = np.random.default_rng(11)
    x = scenes.jitter_cells(scenes.box_cells((10, 10, 10), (37, 37, 37)), 8, DX, 3)[:, :many]
    st = scenes._state(x[:, rng.permutation(many)], (0.3, -0.5, 0.2), np.zeros(many, np.int32), np.array([MODEL_FCR]))
    st = {k: torch.from_numpy(np.ascontiguousarray(v)).to(DEV) for k, v in st.items()}
    ctx = Context(DX, 128, many)
    ctx.set_materials([dict(model=MODEL_FCR, E=2e4, nu=0.3, rho=1000.0, vol=VOL)])
    ctx.import_state(st)
    saved = ctx.new_state_buffer()
    ctx.state_save(saved)
    ctx.import_state({k: v[..., :n].contiguous() for k, v in st.items()})
    ctx.state_load(saved)
    pid = torch.from_numpy(ctx.order()).to(DEV).long()
    assert int((pid >= n).sum()) > 0 and int((pid < n).sum()) > 0
    out = {k: torch.full((c, n), -7.0, device=DEV) for k, c in (("x", 3), ("v", 3), ("C", 9), ("F", 9))}
    ctx.export_particles(particle_view(n, out["x"], out["v"], out["C"], out["F"], None, None))
    here = pid[pid < n]
    for k, t in out.items():
        want = torch.full_like(t, -7.0)
        want[:, here] = st[k][:, here]
        assert torch.equal(t, want), k
    ctx.close()


@pytest.mark.parametrize("first", ["cells", "shuffled"])
def test_way_follows_the_last_order_seen(first):
    """The way of an export goes by the order that the last import or export met, which a loaded state may
    not have: the exports after the load, one by each way, hold the same."""
    n = 66001
    x = scenes.jitter_cells(scenes.box_cells((10, 10, 10), (37, 37, 37)), 8, DX, 3)[:, :n]
    rng = np.random.default_rng(5)
    orders = dict(cells=np.arange(n), shuffled=rng.permutation(n))
    v = rng.standard_normal((3, n)).astype(np.float32)
    states = {}
    for k, o in orders.items():
        st = scenes._state(x[:, o], (0.0, 0.0, 0.0), np.zeros(n, np.int32), np.array([MODEL_FCR]))
        st["v"] = v[:, o]
        states[k] = {q: torch.from_numpy(np.ascontiguousarray(t)).to(DEV) for q, t in st.items()}
    second = "shuffled" if first == "cells" else "cells"
    ctx = Context(DX, 128, n)
    ctx.set_materials([dict(model=MODEL_FCR, E=2e4, nu=0.3, rho=1000.0, vol=VOL)])
    ctx.import_state(states[first])
    saved = ctx.new_state_buffer()
    ctx.state_save(saved)
    ctx.import_state(states[second])
    ctx.state_load(saved)
    for _ in range(2):
        out = ctx.export_state(DEV)
        for k in ("x", "v", "C", "F"):
            assert torch.equal(out[k], states[first][k]), k
    ctx.close()
