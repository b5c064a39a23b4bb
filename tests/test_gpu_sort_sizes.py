"""The cell sort at the edges of its tiles and of the rule that picks its
passes, against numpy's stable sort: whole numbers, so exactly equal."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _keys(pos, width, power):
    c = np.floor(pos[:, :3] / np.float32(width)).astype(np.int64) & ((1 << power) - 1)
    key = np.zeros(len(pos), np.int64)
    for b in range(power):
        for k in range(3):
            key |= ((c[:, k] >> b) & 1) << (3 * b + k)
    return key


@pytest.mark.parametrize("n", [1, 63, 64, 1023, 1024, 1025, 2047, 2049, 8193, 32767, 32768, 32769, 40961, 65537, 300000])
@pytest.mark.parametrize("power", [1, 3, 5, 8])
def test_sort_sizes(sph, n, power):
    g = np.random.default_rng(n + power)
    pos = (g.standard_normal((n, 4)) * 5).astype(np.float32)
    pos[: n // 2, :3] = 0.25  # half of them in one cell: their order is the index
    d_pos = torch.from_numpy(pos).cuda()
    pairs = torch.empty(n, 2, dtype=torch.int32, device="cuda")
    cells = torch.empty(1 << (3 * power), 2, dtype=torch.int32, device="cuda")
    for _ in range(2):
        cells.fill_(7)
        torch.cuda.synchronize()
        sph.sort_noalloc(d_pos.data_ptr(), n, 0.1, power, pairs.data_ptr(), cells.data_ptr())
        torch.cuda.synchronize()
        key = _keys(pos, 0.1, power)
        order = np.argsort(key, kind="stable")
        got = pairs.cpu().numpy()
        assert np.array_equal(got[:, 1], order) and np.array_equal(got[:, 0], key[order])
        first = np.full((1 << (3 * power), 2), (-1, 0), np.int64)
        used, at, count = np.unique(key[order], return_index=True, return_counts=True)
        first[used] = np.stack([at, at + count - 1], 1)
        assert np.array_equal(cells.cpu().numpy(), first)
