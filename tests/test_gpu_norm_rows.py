"""rmsnorm_quant's whole-row kernel against its row slices (a row alone, and the same row in a large batch, give
the same bytes), and act_quant of groups that hold infinities and NaN."""
import numpy as np
import pytest
import torch

from tilert_amd import kernel as K
from tilert_amd import synth
from tilert_amd.rmsnorm import rmsnorm_quant

pytestmark = pytest.mark.gpu

LOGS = torch.zeros(1)


def _run(x, w, scale_fmt):
    y = torch.empty_like(x)
    q = torch.empty(x.shape, dtype=torch.float8_e4m3fn, device=x.device)
    s = torch.empty(x.shape[0], x.shape[1] // 128, dtype=torch.float32, device=x.device)
    rmsnorm_quant(x, w, y, q, s, LOGS, model_arch="deepseek_v3_2", scale_fmt=scale_fmt)
    return y.view(torch.int16), q.view(torch.uint8), s.view(torch.int32)


@pytest.mark.parametrize("rows,dim,scale_fmt", [
    (255, 7168, None), (256, 7168, None), (257, 2176, "div"), (1025, 4096, "ue8m0"), (2049, 3072, None),
    (300, 8192, None), (1023, 10240, None), (1024, 10240, "div"), (1030, 16384, None)])
def test_rows_equal_single_rows(cuda, rows, dim, scale_fmt):
    g = synth.gen(rows + dim)
    x = (torch.randn(rows, dim, generator=g) * 3).to(torch.bfloat16).to(cuda)
    x[rows // 2] = 0
    w = (1 + 0.1 * torch.randn(dim, generator=g)).to(cuda)
    batch = _run(x, w, scale_fmt)
    for i in sorted({0, 1, rows // 2, rows - 2, rows - 1, min(1024, rows - 1)}):
        for a, b in zip(batch, _run(x[i:i + 1].contiguous(), w, scale_fmt)):
            assert torch.equal(a[i:i + 1], b), f"row {i}"


@pytest.mark.parametrize("rows,dim,scale_fmt", [
    (255, 8320, None), (256, 8320, "div"), (300, 10240, None), (1030, 10368, "ue8m0"), (257, 12288, None),
    (1023, 12416, None), (1024, 12416, None), (1100, 14336, "div"),
    (1700, 8320, None), (1400, 12288, None), (2048, 7168, "ue8m0"), (7000, 2048, None)])  # plain stores: outputs above 40 MB
def test_wide_rows_equal_single_rows(cuda, rows, dim, scale_fmt):
    """Rows of 5 to 8 slices, at the edges of the instances and of the dispatch."""
    test_rows_equal_single_rows(cuda, rows, dim, scale_fmt)


@pytest.mark.parametrize("dim", [128, 1536, 2048])
def test_one_slice_rows_vs_large_batch(cuda, dim):
    """dim <= 2048 takes whole rows at every batch: any batch gives a row the same bytes."""
    g = synth.gen(dim)
    x = torch.randn(3000, dim, generator=g).to(torch.bfloat16).to(cuda)
    w = torch.rand(dim, generator=g).to(cuda) + 0.5
    big, small = _run(x, w, None), _run(x[:5].contiguous(), w, None)
    for a, b in zip(big, small):
        assert torch.equal(a[:5], b)
    ref = x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + 1e-6) * w.double()
    assert (big[0].view(torch.bfloat16).double() - ref).abs().max() <= ref.abs().max() * 2.0 ** -8


@pytest.mark.parametrize("fmt", [None, "ue8m0", "div"])
def test_act_quant_non_finite_groups(cuda, fmt):
    """A group with an infinity has an infinite scale (finite values quantise to signed zeros, infinities, as
    inf / inf, to -448); NaN elements take no part in the amax and quantise to -448."""
    x = torch.linspace(-3, 3, 512).reshape(4, 128).to(torch.bfloat16)
    x[0, 3] = float("inf")
    x[1, 5], x[1, 9] = float("nan"), -0.0
    x[2, :] = float("nan")
    q, s = K.act_quant(x.to(cuda), scale_fmt=fmt)
    q, s, f = q.view(torch.uint8).cpu().numpy(), s.cpu().numpy(), x.float().numpy()
    if fmt != "ue8m0":  # (the power-of-two scale of an infinite amax is not a number the format holds)
        assert np.isinf(s[0, 0])
        want = np.where(np.signbit(f[0]), 0x80, 0)
        want[3] = 0xfe
        assert np.array_equal(q[0], want)
    assert q[1, 5] == 0xfe and q[1, 9] == 0x80 and np.all(q[2] == 0xfe)
    fin = f[1].copy()
    fin[5] = 0
    q1, _ = K.act_quant(torch.from_numpy(fin).reshape(1, 128).to(torch.bfloat16).to(cuda), scale_fmt=fmt)
    keep = np.arange(128) != 5
    assert np.array_equal(q[1][keep], q1.view(torch.uint8).cpu().numpy()[0][keep])
