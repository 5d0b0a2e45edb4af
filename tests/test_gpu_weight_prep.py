"""weight_quant / weight_dequant: the wide kernels against the element-wise ones (any K and alignment),
bit for bit, at ragged shapes and on special values.  A view that starts one element into its
storage is not aligned for the wide kernels, so the same values take the other path."""
import numpy as np
import pytest
import torch

from oracle import reference as ref
from tilert_amd import kernel as K

pytestmark = pytest.mark.gpu


def _shifted(t: torch.Tensor) -> torch.Tensor:
    """The same values, one element past an aligned address."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    buf[1:] = t.reshape(-1)
    return buf[1:].reshape(t.shape)


def _weights(N: int, Kd: int, special: bool) -> torch.Tensor:
    w = torch.randn(N, Kd, generator=torch.Generator().manual_seed(N * Kd)) * 0.02
    if special:
        f = w.reshape(-1)
        vals = torch.tensor([0.0, -0.0, float("nan"), float("inf"), -float("inf"), 1e-40, -1e-40, 3e38, -3e38, 1e-30])
        n = f.numel()
        for i, v in enumerate(vals):
            f[(i * 7919 + 13) % n] = v
    return w


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,Kd,special", [(1, 8, False), (127, 128, True), (129, 136, False), (300, 520, True),
                                          (16, 2048, True), (640, 7168, True)])
def test_weight_quant_wide_equals_any(cuda, dtype, N, Kd, special):
    w = _weights(N, Kd, special).to(dtype)
    if N == 300:
        w[:128, :128] = 0  # an all-zero block: scale 1
        w[128:256, :128] *= 1e-36  # a scale outside the range of the fast quotient
    g = w.to(cuda)
    q, s = K.weight_quant(g)
    q1, s1 = K.weight_quant(_shifted(g))
    assert torch.equal(s.view(torch.int32), s1.view(torch.int32))
    assert torch.equal(q.view(torch.uint8), q1.view(torch.uint8))
    if not special:
        rq, rs = ref.weight_quant(w.float())
        assert torch.equal(s.cpu(), rs) and torch.equal(q.cpu().view(torch.uint8), rq.view(torch.uint8))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,Kd", [(1, 8), (33, 256), (130, 520), (257, 4)])
def test_weight_dequant_wide_equals_any(cuda, dtype, N, Kd):
    """Every e4m3 code (both NaNs among them) under several scales."""
    s = torch.rand(-(-N // 128), -(-Kd // 128), generator=torch.Generator().manual_seed(1)) * 1e-3
    _dequant_both_ways(cuda, dtype, N, Kd, s)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("N,Kd", [(1023, 1024), (1024, 1024), (2017, 520), (130, 8072), (1 << 18, 4),
                                  (9363, 7168)])  # the fp32 result is just above the 256 MB of non-temporal stores
def test_weight_dequant_from_the_wide_kernels_size(cuda, dtype, N, Kd):
    """One row below the wide kernel's 1 M elements and at it, ragged rows and columns; the scales of every third block
    row give results that are subnormal."""
    s = torch.rand(-(-N // 128), -(-Kd // 128), generator=torch.Generator().manual_seed(2)) * 1e-3
    s[::3] *= 1e-35
    _dequant_both_ways(cuda, dtype, N, Kd, s)


def _dequant_both_ways(cuda, dtype, N, Kd, s):
    codes = torch.from_numpy(np.resize((np.arange(256) * 37 % 256).astype(np.uint8), N * Kd)).reshape(N, Kd)
    q = codes.view(torch.float8_e4m3fn).to(cuda)
    old = torch.get_default_dtype()
    torch.set_default_dtype(dtype)
    try:
        d = K.weight_dequant(q, s.to(cuda))
        d1 = K.weight_dequant(_shifted(q.view(torch.uint8)).view(torch.float8_e4m3fn), s.to(cuda))
    finally:
        torch.set_default_dtype(old)
    bits = torch.int16 if dtype == torch.bfloat16 else torch.int32
    nan = torch.isnan(d1)  # (a NaN's sign bit is not part of its value)
    assert torch.equal(torch.isnan(d), nan)
    assert torch.equal(d.view(bits)[~nan], d1.view(bits)[~nan])
