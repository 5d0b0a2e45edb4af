"""The wide FP8 GEMM's plan, on the CPU: the tests' restatement agrees with the library's workspace sizes, and the GPU
cases reach every row-tile count, both token-fragment counts, split and unsplit."""
import random

from tests._wide_plan import PLANS, wide_plan, workspace_bytes
from tilert_amd import _lib


def test_plan_restatement_matches_the_library():
    lib, r, split = _lib.load(), random.Random(11), 0
    for _ in range(4000):
        M, N, K = r.randint(33, 256), 16 * int(2 ** r.uniform(0, 12)), 128 * int(2 ** r.uniform(0, 7.5))
        want = workspace_bytes(M, N, K)
        split += want > 65536
        assert lib.tl_fp8_gemm_workspace_bytes(M, N, K) == want, (M, N, K)
    assert split > 1000  # (an unsplit plan's size does not tell its F)


def test_gpu_cases_reach_every_plan():
    for shape, plan in PLANS.items():
        assert wide_plan(*shape) == plan, shape
        assert workspace_bytes(*shape) == _lib.load().tl_fp8_gemm_workspace_bytes(*shape), shape
    reached = {(f, tj, s > 1) for f, tj, s in PLANS.values()}
    assert reached == {(f, tj, split) for f in range(4, 10) for tj in (1, 2) for split in (False, True)}
