"""The wide FP8 GEMM at every row-tile count, with one and two token fragments a wave, unsplit and with K ranges, on
stored and packed weights (one call of each: _wide_plan.PLANS), against the same codes and scales in fp64."""
import pytest
import torch

from tests._tol import assert_gemm_close
from tests._wide_plan import PLANS
from tilert_amd import kernel as K

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,Kd", list(PLANS))
def test_every_plan_both_layouts(cuda, M, N, Kd):
    g = torch.Generator(device=cuda).manual_seed(M + N + Kd)
    x = torch.randn(M, Kd, generator=g, device=cuda).to(torch.bfloat16)
    xq, xs = K.act_quant(x)
    wq = (torch.randn(N, Kd, generator=g, device=cuda) * 112).clamp_(-448, 448).to(torch.float8_e4m3fn)
    ws = (torch.rand(-(-N // 128), Kd // 128, generator=g, device=cuda) + 0.5) * 2e-4
    a = xq.double() * xs.double().repeat_interleave(128, 1)
    want = torch.cat([a @ (wq[n:n + 2048].double() *
                           ws.double().repeat_interleave(128, 1).repeat_interleave(128, 0)[n:n + wq[n:n + 2048].shape[0]]).T
                      for n in range(0, N, 2048)], 1)
    out = K.fp8_gemm(xq, xs, wq, ws)
    assert_gemm_close(out, want, f"stored {PLANS[M, N, Kd]}")
    packed = K.pack_weight(wq, ws)
    for _ in range(3):
        assert torch.equal(K.fp8_gemm(xq, xs, packed), out)
        assert torch.equal(K.fp8_gemm(xq, xs, wq, ws), out)
