"""sort_noalloc with cell tables on both sides of the sizes up to which its
passes fill them, few pairs and many: every cell of the table and every pair,
equal to torch's stable sort of the keys."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("power", [8, 9, 10])
@pytest.mark.parametrize("n", [1, 5000, 32768, 32769, 70000])
def test_sort_tables(sph, n, power):
    g = torch.Generator().manual_seed(n + power)
    pos = (torch.randn(n, 4, generator=g) * 9).cuda()
    pos[: n // 2, :3] = 0.25
    pairs = torch.empty(n, 2, dtype=torch.int32, device="cuda")
    cells = torch.full((1 << (3 * power), 2), 7, dtype=torch.int32, device="cuda")
    sph.sort_noalloc(pos.data_ptr(), n, 0.1, power, pairs.data_ptr(), cells.data_ptr(),
                     torch.cuda.current_stream().cuda_stream)
    c = torch.floor(pos[:, :3].cpu() / 0.1).long().cuda() & ((1 << power) - 1)
    key = torch.zeros(n, dtype=torch.long, device="cuda")
    for b in range(power):
        for k in range(3):
            key |= ((c[:, k] >> b) & 1) << (3 * b + k)
    key, order = torch.sort(key, stable=True)
    assert torch.equal(pairs[:, 0].long(), key) and torch.equal(pairs[:, 1].long(), order)
    used, count = torch.unique_consecutive(key, return_counts=True)
    last = count.cumsum(0) - 1
    want = torch.empty_like(cells)
    want[:, 0], want[:, 1] = -1, 0
    want[used, 0], want[used, 1] = (last - count + 1).int(), last.int()
    assert torch.equal(cells, want)
