"""A tree whose lists do not fit into the GPU's memory is refused with an
error; the context then has no tree, and takes the next one that fits as if
nothing had happened."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fixes", [0, 0x7F])
def test_tree_after_a_failed_allocation(sph, orc, tables256, impact, fixes):
    ic = impact(5000, 3)
    prm = sph.default_params(max_unchecked_pointers=2_000_000_000, fixes=fixes)  # 10 GB for the root's list
    small = orc.build_octree(ic["pos"], prm.max_children_in_leaf, 1)
    large = orc.build_octree(ic["pos"], prm.max_children_in_leaf, 7)  # 20 TB for its levels'
    ctx = sph.Context(prm, ic, tables256)
    ctx.sort()
    acc = []
    for attempt in range(2):
        ctx.upload("gravnorm", np.ones(5000, np.float32))
        ctx.upload_tree(small)
        ctx.gravity()
        acc.append(ctx.download("acc"))
        with pytest.raises(sph.SphError):
            ctx.upload_tree(large)
        with pytest.raises(sph.SphError):
            ctx.gravity()
    ctx.close()
    assert np.any(acc[0]) and np.array_equal(acc[0].view(np.int32), acc[1].view(np.int32))
