"""Plans kept per thread (plan_sgemm, plan_bf16, plan_s8): a kept plan is the
one that a fresh thread makes, whatever else the slots held, and a tunable's
change is seen by the next plan."""
import random
import threading

import pytest


def shapes(count, seed=7):
    rng = random.Random(seed)
    size = lambda hi: int(2 ** rng.uniform(0, hi))
    return [(size(12), size(13), size(12)) for _ in range(count)]


def in_thread(fn):
    out = []
    t = threading.Thread(target=lambda: out.append(fn()))
    t.start()
    t.join()
    return out[0]


@pytest.mark.parametrize("kind", ["sgemm", "sgemm_nk", "sgemm_ta", "bf16", "bf16_nk", "bf16_f32", "s8", "s8_scale"])
def test_kept_plans_are_the_plans_made_anew(lib, kind):
    plan = {
        "sgemm": lambda m, n, k: lib.plan_sgemm(m, n, k),
        "sgemm_nk": lambda m, n, k: lib.plan_sgemm(m, n, k, transB=1),
        "sgemm_ta": lambda m, n, k: lib.plan_sgemm(m, n, k, transA=1),
        "bf16": lambda m, n, k: lib.plan_bf16(m, n, k),
        "bf16_nk": lambda m, n, k: lib.plan_bf16_ex(m, n, k, transB=1),
        "bf16_f32": lambda m, n, k: lib.plan_bf16(m, n, k, fp32_inputs=1),
        "s8": lambda m, n, k: lib.plan_s8(m, n, k),
        "s8_scale": lambda m, n, k: lib.plan_s8(m, n, k, with_scale=1),
    }[kind]
    work = shapes(300)  # several to a slot
    want = [in_thread(lambda s=s: plan(*s)) for s in work]  # each with empty slots
    order = [i for i in range(len(work)) for _ in range(2)]  # made, then kept
    random.Random(3).shuffle(order)
    for i in order + order[::-1]:
        assert plan(*work[i]) == want[i], work[i]


def test_a_tunable_is_seen_by_the_next_plan(lib):
    before = lib.plan_sgemm(384, 3072, 768, transB=1)
    assert lib.plan_sgemm(384, 3072, 768, transB=1) == before
    with lib.tunables(TILE_CFG=1, TILE_SPLITS=2):
        forced = lib.plan_sgemm(384, 3072, 768, transB=1)
        assert forced["splits"] == 2 and forced != before
        assert in_thread(lambda: lib.plan_sgemm(384, 3072, 768, transB=1)) == forced
    assert lib.plan_sgemm(384, 3072, 768, transB=1) == before


def test_plans_of_one_size_differ_by_layout(lib):
    """One size, the layouts in turn: no slot answers for another layout."""
    M, N, K = 200, 1000, 513
    made = [
        lambda: lib.plan_sgemm(M, N, K),
        lambda: lib.plan_sgemm(M, N, K, transB=1),
        lambda: lib.plan_sgemm(M, N, K, transA=1),
        lambda: lib.plan_bf16(M, N, K),
        lambda: lib.plan_bf16(M, N, K, fp32_inputs=1),
        lambda: lib.plan_s8(M, N, K),
    ]
    want = [in_thread(f) for f in made]
    for _ in range(3):
        assert [f() for f in made] == want
