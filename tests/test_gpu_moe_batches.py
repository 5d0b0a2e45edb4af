"""The MoE kernels beyond the small batches' LDS ones, and the edges between them: the ones that stream their
activations beside the weights with every group of 4 tokens, the register gate/up of small layers, K shorter than a
workgroup's waves and not a multiple of them, odd and even hit counts, one and many experts, more than 64 routed
pairs, repeated expert ids."""
import pytest
import torch

from oracle import reference as ref
from tests._tol import assert_gemm_close
from tests.test_gpu_moe import _experts, _run
from tilert_amd import moe, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,E,D,I,topk,n_exp,e0", [
    (6, 4, 128, 128, 2, 8, 0),      # one K block: 7 waves idle in gate/up, 3 of 4 in down
    (9, 3, 1152, 128, 3, 9, 3),     # 9 K blocks over 8 waves
    (13, 5, 640, 640, 4, 5, 0),     # 5 K blocks, all experts hit: an odd slot count
    (16, 64, 256, 128, 8, 64, 0),   # 64 local experts
    (16, 1, 896, 1408, 8, 32, 7),   # one local expert
    (12, 8, 512, 1152, 16, 64, 16),  # 192 routed pairs
    (10, 6, 7168, 256, 8, 48, 6),
])
def test_moe_batches_vs_oracle(cuda, M, E, D, I, topk, n_exp, e0):
    y, ry, hits = _run(M, E, D, I, topk, n_exp, e0, seed=M * 100 + E + D)
    if hits:
        assert_gemm_close(y, ry, "moe output")
    else:
        assert torch.equal(y, torch.zeros_like(y))


def test_moe_batch_equals_its_tokens(cuda):
    """A token's output does not depend on the batch it is in beyond the order of fp32 sums: batches of 16
    repeated are bit-identical, and agree with the oracle for each half."""
    M, E, D, I = 16, 8, 1024, 512
    W = _experts(E, D, I, 77)
    g = synth.gen(5)
    x = synth.activations(M, D, g)
    idx, w = synth.routing(M, 16, 8, g)
    ex = moe.LocalExperts(*(W[k][i].to(cuda) for k in ("gate", "up", "down") for i in (0, 1)))
    outs = [moe.moe_forward(x.to(cuda), ex, idx.to(cuda), w.to(cuda)) for _ in range(4)]
    for o in outs[1:]:
        assert torch.equal(o, outs[0])
    for lo in (0, 8):
        sl = slice(lo, lo + 8)
        rh, hits = ref.moe_gate_up(x[sl], W["gate"][0], W["gate"][1], W["up"][0], W["up"][1], idx[sl], 0)
        ry = ref.moe_down(rh, hits, W["down"][0], W["down"][1], idx[sl], w[sl], 0)
        assert_gemm_close(outs[0][sl], ry, f"tokens {lo}..")


def test_moe_batch_no_hits_and_repeated_ids(cuda):
    idx = torch.full((7, 12), 20, dtype=torch.int32)
    y, _, hits = _run(7, 4, 256, 256, 12, 32, 0, seed=3, idx=idx, w=torch.full((7, 12), 0.1))
    assert hits == [] and torch.equal(y, torch.zeros_like(y))
    # a token that names an expert twice: the last weight counts, as in the kernel for small batches
    ids = torch.tensor([[1, 2, 1]] * 6, dtype=torch.int32)
    w = torch.tensor([[0.5, 0.25, 0.75]] * 6)
    a, _, _ = _run(6, 4, 256, 256, 3, 32, 0, seed=4, idx=ids, w=w)
    b, _, _ = _run(6, 4, 256, 256, 3, 32, 0, seed=4, idx=torch.tensor([[30, 2, 1]] * 6, dtype=torch.int32), w=w)
    assert torch.equal(a, b)


def _coded(E, N, K, g):
    """Stacked e4m3fn weights [E, N, K] and scales, made as codes."""
    q = (torch.randn(E, N, K, generator=g, device="cuda", dtype=torch.bfloat16) * 112).clamp_(-448, 448)
    s = (torch.rand(E, N // 128, K // 128, generator=g, device="cuda") + 0.5) * 2e-4
    return q.to(torch.float8_e4m3fn), s


@pytest.mark.parametrize("M,E,D,I,topk,n_exp", [
    # gate/up: the streaming kernel's four groups of 4 tokens (M = 4 by its 68 pairs, and by x above 64 KB)
    (3, 32, 2176, 1792, 22, 96), (4, 32, 2176, 1408, 17, 96), (4, 16, 8320, 2688, 8, 128),
    (8, 32, 2176, 768, 9, 96), (12, 16, 2176, 896, 6, 64), (16, 16, 2176, 768, 5, 64),
    # its neighbours in the register kernel: D and the number of work items just inside its limits
    (16, 16, 1024, 1408, 5, 64), (13, 16, 2048, 1408, 5, 64), (16, 16, 2176, 640, 5, 64),
    # down at 6 to 8 tokens: h of 1, 2, 5 and 6 K blocks staged in LDS, of 3, 4 and 9 streamed
    (6, 8, 256, 128, 8, 32), (7, 8, 256, 256, 8, 32), (8, 8, 384, 640, 8, 32), (6, 8, 256, 768, 8, 32),
    (6, 8, 256, 384, 8, 32), (8, 8, 384, 512, 8, 32), (7, 8, 256, 1152, 8, 32), (9, 8, 256, 640, 7, 32),
])
def test_moe_dispatch_edges(cuda, M, E, D, I, topk, n_exp):
    g = torch.Generator(device=cuda).manual_seed(M * 1000 + E + D + I)
    gate, up, down = _coded(E, I, D, g), _coded(E, I, D, g), _coded(E, D, I, g)
    h_ = synth.gen(M + D)
    x, (idx, w) = synth.activations(M, D, h_), synth.routing(M, n_exp, topk, h_)
    ex = moe.LocalExperts(*gate, *up, *down)
    h = moe.ep_gate_up_swiglu(x.to(cuda), idx.to(cuda), ex)
    y = moe.ep_down_combine(h, ex, idx.to(cuda), w.to(cuda))
    hits = ref.hit_experts(idx, 0, E)
    cpu = [[t[hits].cpu() for t in pair] for pair in (gate, up, down)]
    slot = torch.full((n_exp,), -1, dtype=torch.int32)
    slot[torch.tensor(hits)] = torch.arange(len(hits), dtype=torch.int32)
    ids = slot[idx.long()]  # the hit experts renumbered 0, 1, ...
    rh, rhits = ref.moe_gate_up(x, *cpu[0], *cpu[1], ids, 0)
    assert rhits == list(range(len(hits)))
    assert_gemm_close(h[:len(hits)], rh, "gate/up")
    assert_gemm_close(y, ref.moe_down(h[:len(hits)].cpu(), rhits, *cpu[2], ids, w, 0), "down")
    for _ in range(2):
        assert torch.equal(moe.ep_gate_up_swiglu(x.to(cuda), idx.to(cuda), ex)[:len(hits)], h[:len(hits)])
        assert torch.equal(moe.ep_down_combine(h, ex, idx.to(cuda), w.to(cuda)), y)
