"""The radix sort on both sides of its rule of 64 tiles of 2,048 keys (the scatter sums the tiles' counts
itself, or a launch of one workgroup per digit does) and where that launch loops (more than 2,048
tiles): keys and permutation equal NumPy's stable argsort, for few and many distinct keys.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
if not torch.cuda.is_available():
    pytest.skip("no GPU", allow_module_level=True)

from zeno_amd.zmpm import Context  # noqa: E402

DEV = "cuda:0"


@pytest.mark.parametrize("n", [511, 64 * 2048 - 1, 64 * 2048, 64 * 2048 + 1, 2049 * 2048 + 5])
@pytest.mark.parametrize("bits,hi", [(16, 1 << 16), (17, 3), (32, 1 << 32)])
def test_sort_is_the_stable_argsort(n, bits, hi):
    rng = np.random.default_rng(n + bits)
    keys = rng.integers(0, hi, size=n, dtype=np.int64).astype(np.uint32)
    ctx = Context(1 / 64, 64, n)
    ko, po = ctx.sort_keys(torch.from_numpy(keys.view(np.int32)).to(DEV), bits)
    order = np.argsort(keys, kind="stable")
    assert np.array_equal(po.cpu().numpy(), order)
    assert np.array_equal(ko.cpu().numpy().view(np.uint32), keys[order])
    ctx.close()
