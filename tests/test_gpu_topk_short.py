"""Top-k of short rows (one workgroup per row) at the edges of its register tiles and dispatch: lengths around
4096, 8192 and 16384, few and many rows, ties, infinities, k equal to and next to the length."""
import numpy as np
import pytest
import torch

from tilert_amd.topk import topk_rows

pytestmark = pytest.mark.gpu


def _expect(row: np.ndarray, n: int, k: int) -> np.ndarray:
    """The k largest of row[:n], the lowest columns among equals, ascending; -1 padding."""
    out = np.full(k, -1, np.int64)
    if n <= k:
        out[:max(n, 0)] = np.arange(max(n, 0))
        return out
    order = np.lexsort((np.arange(n), -row[:n].astype(np.float64)))
    out[:] = np.sort(order[:k])
    return out


@pytest.mark.parametrize("rows,n,ld,k", [
    (1, 1, 4, 1), (3, 5, 8, 4), (4, 2049, 2052, 2048), (2, 4095, 4096, 512), (4, 4097, 4100, 2048),
    (2, 4096, 65536, 1024),      # a long buffer of which few columns are valid
    (4, 8192, 8192, 8191), (3, 8193, 8196, 2048), (1, 8190, 8192, 8192),
    (127, 9000, 9000, 512), (128, 9000, 9000, 512), (130, 16384, 16384, 2048), (128, 16385, 16388, 64),
])
@pytest.mark.parametrize("kind", ["normal", "ties", "special"])
def test_short_rows_exact(cuda, rows, n, ld, k, kind):
    g = torch.Generator().manual_seed(rows * n + k)
    x = torch.randn(rows, ld, generator=g)
    if kind == "ties":
        x = (x * 4).round() / 4
    elif kind == "special":
        x[:, ::7] = float("-inf")
        x[:, 3::11] = 0.0
        x[:, 5::13] = -0.0
        x[0, : min(n, 40)] = float("inf")
        x[-1] = 1.5  # every value equal
        x[:, 2::17] = -3.4028234663852886e38
    base = n - rows  # row i considers its first n - rows + 1 + i columns
    got = topk_rows(x.to(cuda), base, k).cpu().numpy()
    xs = x.numpy().copy()
    # the order is that of the bit patterns: -0 below +0
    key = xs.view(np.uint32).astype(np.int64)
    key = np.where(key & 0x80000000, 0xffffffff - key, key + 0x80000000).astype(np.float64)
    for i in sorted({0, rows // 2, rows - 1}):
        assert np.array_equal(got[i], _expect(key[i], min(max(base + 1 + i, 0), ld), k)), f"row {i}"


def test_short_and_chunked_rows_share_a_workspace(cuda):
    """Calls of both kinds in turn on one stream's workspace: the chunked kernel's counters stay as it left them."""
    g = torch.Generator().manual_seed(3)
    long, short = torch.randn(3, 40000, generator=g).to(cuda), torch.randn(3, 5000, generator=g).to(cuda)
    first = topk_rows(long, 40000 - 3, 2048), topk_rows(short, 5000 - 3, 2048)
    for _ in range(3):
        assert torch.equal(topk_rows(short, 5000 - 3, 2048), first[1])
        assert torch.equal(topk_rows(long, 40000 - 3, 2048), first[0])
