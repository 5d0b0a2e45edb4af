"""The plan of the wide FP8 GEMM restated for the tests: which (F row tiles, TJ token fragments, S K ranges) a call of
more than 32 tokens runs.  test_wide_plan.py holds it against the library's workspace sizes, so the GPU cases that
target one plan notice when a plan moves."""
COUNTERS = 65536


def takes_no_workspace(M: int, N: int, K: int) -> bool:
    return M > 64 and (N % 128 != 0 or K % 512 != 0) and (K // 128 < 16 or N // 16 > 4088)


def wide_plan(M: int, N: int, K: int) -> tuple[int, int, int]:
    nt, kb = N // 16, K // 128
    tj = 1 if M <= 64 else 2
    tg = -(-M // (64 * tj))
    best, best_cost, floor = (4, tj, 1), None, N * K // 141312
    for f in range(4, 10):
        tiles = -(-nt // f)
        max_s = 1 if takes_no_workspace(M, N, K) else max(1, min(kb, 32, 256 // (tiles * tg)))
        for want in range(1, max_s + 1):
            per = -(-kb // want)
            s = -(-kb // per)
            if s != want:
                continue
            split = 60 * tj + s * (10 + 4 * f * tj) if s > 1 else 0
            if best_cost is not None and split >= best_cost:
                break
            cost = max(-(-tiles * tg * s // 256) * per * (2 * f + 8 * tj + 1), floor) + split
            if best_cost is None or cost < best_cost:
                best, best_cost = (f, tj, s), cost
    return best


def workspace_bytes(M: int, N: int, K: int) -> int:
    if takes_no_workspace(M, N, K):
        return 0
    f, tj, s = wide_plan(M, N, K)
    tiles, tg = -(-(N // 16) // f), -(-M // (64 * tj))
    return COUNTERS + (tiles * tg * s * f * 4 * tj * 1024 if s > 1 else 0)


# (M, N, K): (F, TJ, S), one call of every F, of one and two token fragments, unsplit and split, with the fewest weights;
# then layers of the models
PLANS = {
    (33, 16, 512): (4, 1, 1), (64, 16, 2048): (4, 1, 4),
    (64, 16400, 512): (5, 1, 1), (33, 5456, 3072): (5, 1, 3),
    (40, 20496, 512): (6, 1, 1), (64, 10256, 2560): (6, 1, 2),
    (33, 24640, 512): (7, 1, 1), (64, 8208, 4608): (7, 1, 3),
    (64, 28784, 512): (8, 1, 1), (50, 10256, 6144): (8, 1, 3),
    (64, 32816, 512): (9, 1, 1), (47, 16400, 5120): (9, 1, 2),
    (65, 16, 512): (4, 2, 1), (100, 16, 2048): (4, 2, 4),
    (129, 8208, 512): (5, 2, 1), (256, 2704, 3072): (5, 2, 3),
    (130, 10256, 512): (6, 2, 1), (255, 2704, 5120): (6, 2, 4),
    (200, 12304, 512): (7, 2, 1), (129, 3376, 5120): (7, 2, 4),
    (256, 14352, 512): (8, 2, 1), (200, 5136, 4608): (8, 2, 3),
    (145, 16400, 512): (9, 2, 1), (256, 5392, 6144): (9, 2, 3),
    (65, 18432, 7168): (9, 2, 2), (100, 18432, 7168): (9, 2, 2), (200, 2112, 7168): (5, 2, 4),
    (256, 18432, 7168): (9, 2, 1), (33, 7168, 18432): (7, 1, 4),
}
