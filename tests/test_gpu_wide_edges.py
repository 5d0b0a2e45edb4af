"""The wide MFMA GEMM at the edges of its tiles, plans and layouts: row counts that are not a multiple of a
workgroup's row tiles (or of 128), token counts around the 64- and 128-token groups, K ranges of one block
and uneven ones, and the weight as stored against the packed one, bit for bit."""
import pytest
import torch

from oracle import reference as ref
from tests._tol import assert_gemm_close
from tilert_amd import _lib
from tilert_amd import kernel as K
from tilert_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,Kd", [
    (33, 16, 128),      # one row tile, one K block
    (17, 80, 2048),     # 5 row tiles, two-token-tile range
    (64, 208, 1408),    # 13 row tiles; K not a multiple of 512: stored layout only
    (65, 592, 640),     # 37 row tiles, 128-token groups
    (128, 48, 3584),    # 3 row tiles: many K ranges
    (129, 1040, 896),   # 65 row tiles, two token groups, a partial one
    (256, 576, 7168),   # wkv_a at the largest batch
    (100, 2112, 1024),  # wq_a + wkv_a's width
    (24, 3072, 1024),   # the GEMV's range at M = 17..32
    (32, 4096, 4096),
    (24, 4112, 1024),   # one row tile past it
    (24, 3072, 5120),   # the longest of the GEMV's range, and a block past it
    (24, 3072, 5248),
    (40, 18448, 512),   # more row tiles than one round of the smallest tile
])
def test_wide_edges_both_layouts(cuda, M, N, Kd):
    g = synth.gen(M * 7 + N + Kd)
    x = synth.activations(M, Kd, g)
    w = torch.randn(N, Kd, generator=g) * 0.02
    wq, ws = ref.weight_quant(w)
    xq, xs = ref.act_quant(x)
    # the same codes and scales in fp64: the kernel's fp32 sums of exact products stay inside the GEMM bar
    want = ((xq.double() * xs.double().repeat_interleave(128, 1)) @
            (wq.double() * ws.double().repeat_interleave(128, 0)[:N].repeat_interleave(128, 1)).T)
    d = [t.to(cuda) for t in (xq, xs, wq, ws)]
    out = K.fp8_gemm(*d)
    assert_gemm_close(out, want, "stored")
    for _ in range(3):
        assert torch.equal(K.fp8_gemm(*d), out)
    if Kd % 512 == 0:
        packed = K.pack_weight(d[2], d[3])
        for _ in range(3):
            assert torch.equal(K.fp8_gemm(d[0], d[1], packed), out)


@pytest.mark.parametrize("M,N,Kd", [(65, 16, 128), (100, 2112, 1536), (200, 4112, 1920), (129, 1040, 896)])
def test_wide_without_a_workspace(cuda, M, N, Kd):
    """The shapes that take no workspace run without one, stored and packed."""
    g = synth.gen(M + N + Kd)
    xq, xs = (t.to(cuda) for t in ref.act_quant(synth.activations(M, Kd, g)))
    wq, ws = (t.to(cuda) for t in ref.weight_quant(torch.randn(N, Kd, generator=g) * 0.02))
    want = ref.fp8_gemm(xq.cpu(), xs.cpu(), wq.cpu(), ws.cpu())
    lib, st = _lib.load(), torch.cuda.current_stream(cuda).cuda_stream
    out = torch.empty(M, N, dtype=torch.bfloat16, device=cuda)
    weights = [(lib.tl_fp8_gemm, wq)]
    if Kd % 512 == 0:
        weights.append((lib.tl_fp8_gemm_packed, K.pack_weight(wq, ws).data))
    for fn, w in weights:
        assert fn(xq.data_ptr(), xs.data_ptr(), w.data_ptr(), ws.data_ptr(), out.data_ptr(), M, N, Kd, None, 0, st) == 0, \
            lib.tl_last_error()
        assert_gemm_close(out, want, f"no workspace M={M} N={N} K={Kd}")
