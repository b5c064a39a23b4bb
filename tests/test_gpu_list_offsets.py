"""Gravity's unchecked lists where a level's lists together hold more than
2^32 entries (large max_unchecked_pointers times many nodes): the same field,
bit for bit, as with short lists that no node fills either.  As written with
one recursion (a group per node) and with two (a thread per node), and in the
near-field form, whose levels all keep their lists.  27 GB per buffer."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("over", [{}, {"gravity_max_recursion": 2}, {"fixes": 0x7F},
                                  {"fixes": 0x7F, "precision": 1, "expansion_order": 3}])
def test_lists_beyond_32_bits(sph, orc, tables256, impact, over):
    ic = impact(5000, 3)
    prm = sph.default_params()
    tree = orc.build_octree(ic["pos"], prm.max_children_in_leaf, prm.max_tree_depth)
    counts = tree["level_counts"]
    level = int(np.argmax(counts[:-1]))
    first = int(counts[:level].sum())
    long = int(1.3 * 2 ** 32 / counts[level])
    branches = np.flatnonzero(tree["octree"][tree["level_nodes"][first:first + counts[level]]] == 0)
    # branches on the far side, and lists that no node fills
    assert np.sum(branches * long >= 2 ** 32) > 5 and tree["node_count"] < 8192
    out = []
    for maxu in (8192, long):
        ctx = sph.Context(sph.default_params(max_unchecked_pointers=maxu, **over), ic, tables256)
        ctx.upload_tree(tree)
        ctx.sort()
        for _ in range(2):
            ctx.gravity()
        ctx.sync()
        out.append({f: ctx.download(f) for f in ("acc", "gravnorm")})
        ctx.close()
    for f in out[0]:
        assert np.array_equal(out[0][f].view(np.int32), out[1][f].view(np.int32)), f
