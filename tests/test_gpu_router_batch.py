"""The router on calls of several thousand tokens (GPU), where a wave takes one token or two: the oracle's plan, at
token counts that leave waves and workgroups incomplete, with ties and thresholds that many experts share."""
import contextlib

import numpy as np
import pytest

import oracle_lib
from ncnn_moe_runtime_amd import hip_router

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")  # before the router library, so that both bind the same HIP runtime


@pytest.mark.parametrize("tokens,experts,top_k", [(8191, 64, 6), (8192, 8, 8), (8195, 100, 12), (4111, 256, 8), (1003, 512, 3), (515, 1024, 64)])
def test_batches_match_the_oracle(tokens, experts, top_k):
    rng = np.random.default_rng(tokens * 31 + experts)
    logits = (rng.standard_normal((tokens, experts)) * 2).astype(np.float32)
    logits[1::5] = np.round(logits[1::5] * 4) / 4   # ties all over the row
    logits[2::7] = np.float32(1.5)                  # every score equal
    logits[3::11, experts // 2:] *= np.float32(60)  # scores that saturate or vanish
    bias = (rng.standard_normal(experts) * 0.3).astype(np.float32)
    with contextlib.closing(hip_router.HipRouter(tokens, experts, top_k)) as router:
        for score in (hip_router.SOFTMAX, hip_router.SIGMOID, hip_router.SQRT_SOFTPLUS):
            for options in (dict(), dict(selection_bias=bias, renormalize=False, routed_scaling_factor=2.5),
                            dict(explicit_expert_ids=rng.integers(0, experts, (tokens, top_k)).astype(np.uint32), renormalize=False)):
                print("[case] %d tokens, %d experts, top %d, score %d, %s" % (tokens, experts, top_k, score, sorted(options)), flush=True)
                status, offsets, routes = router.dispatch(logits, top_k, score_function=score, **options)
                cpu_status, cpu_offsets, cpu_routes = oracle_lib.oracle_router_dispatch(logits, top_k, score_function=score, **options)
                assert status == cpu_status == 0
                assert np.array_equal(offsets, cpu_offsets)
                for field in ("token_index", "rank"):
                    assert np.array_equal(routes[field], cpu_routes[field]), field
                assert np.array_equal(routes["weight"].view(np.uint32), cpu_routes["weight"].view(np.uint32))
        logits[tokens - 1, experts - 1] = np.inf
        assert router.dispatch(logits, top_k)[0] == hip_router.STATUS_NON_FINITE_LOGIT


@pytest.mark.parametrize("tokens", [1, 3, 257, 4095, 4096])
@pytest.mark.parametrize("experts,top_k", [(1, 1), (2, 1), (7, 3), (8, 2), (8, 8), (9, 9)])
def test_few_experts_match_the_oracle(tokens, experts, top_k):
    """Up to eight experts are ranked against each other, more go through a threshold: ties, equal rows, scores that vanish."""
    rng = np.random.default_rng(tokens * 31 + experts)
    logits = (rng.standard_normal((tokens, experts)) * 2).astype(np.float32)
    logits[1::5] = np.round(logits[1::5])
    logits[2::7] = np.float32(1.5)
    logits[3::11, (experts + 1) // 2:] *= np.float32(6)
    bias = (rng.standard_normal(experts) * 0.3).astype(np.float32)
    print("[case] %d tokens, %d experts, top %d" % (tokens, experts, top_k), flush=True)
    with contextlib.closing(hip_router.HipRouter(tokens, experts, top_k)) as router:
        for score in (hip_router.SOFTMAX, hip_router.SIGMOID, hip_router.SQRT_SOFTPLUS):
            for options in (dict(), dict(selection_bias=bias, routed_scaling_factor=2.5)):
                status, offsets, routes = router.dispatch(logits, top_k, score_function=score, **options)
                cpu_status, cpu_offsets, cpu_routes = oracle_lib.oracle_router_dispatch(logits, top_k, score_function=score, **options)
                assert status == cpu_status == 0
                assert np.array_equal(offsets, cpu_offsets)
                for field in ("token_index", "rank"):
                    assert np.array_equal(routes[field], cpu_routes[field]), field
                assert np.array_equal(routes["weight"].view(np.uint32), cpu_routes["weight"].view(np.uint32))


def _thresholds(logits, top_k):
    """Where the kernels find each row's threshold: "quads", or by the search, since the rule asks for that ("searched"), two quads' largest are
    the same ("tied") or too many experts lie above it ("many")."""
    experts = logits.shape[1]
    with_experts = min((experts + 3) // 4, 16)
    if 4 * top_k > 3 * with_experts:
        return ["searched"] * len(logits)
    of_quad = np.arange(experts) % 64 // 4
    largest = np.full((len(logits), 16), -np.inf, dtype=np.float32)
    for quad in range(with_experts):
        largest[:, quad] = logits[:, of_quad == quad].max(axis=1)
    ways = []
    for row, above in enumerate((largest[:, None, :] > largest[:, :, None]).sum(axis=2)):
        kth = np.nonzero(above == top_k - 1)[0]
        most = min(64, top_k + top_k // 2 + 8)
        ways.append("tied" if kth.size == 0 else "many" if (logits[row] >= largest[row, kth[0]]).sum() > most else "quads")
    return ways


@pytest.mark.parametrize("tokens", [5, 263, 1030, 2111])
@pytest.mark.parametrize("experts,top_k", [(17, 16), (64, 15), (130, 16), (256, 17), (512, 1), (1024, 16), (17, 3), (17, 4), (33, 6), (64, 12), (64, 13),
                                           (65, 12), (130, 12), (256, 8), (256, 12), (512, 5), (1024, 2), (1024, 12)])
def test_thresholds_of_quads_match_the_oracle(tokens, experts, top_k):
    """The threshold is the top_k-th of the sixteen quads' largest (up to three quarters as many routes as there are quads with experts) or searched for:
    the best experts spread over the quads, all in one quad, equal in two of them, and too many above the threshold; then a call with rejected rows, and one
    more.  Above 2,048 tokens the softmax's sums of a workgroup's rows go side by side."""
    rng = np.random.default_rng(tokens * 31 + experts)
    logits = rng.standard_normal((tokens, experts)).astype(np.float32)
    lanes = np.arange(experts) % 64
    for row in range(tokens):
        quad = rng.integers(0, 16)
        if row % 4 == 1:
            logits[row, lanes // 4 == quad] += np.float32(8)      # one quad holds the best
        elif row % 4 == 2:
            logits[row, lanes // 4 != quad] += np.float32(8)      # ... or all but the best
        elif row % 4 == 3:
            logits[row] = np.round(logits[row] * 2) / 2           # quads with the same largest
    print("[case] quads, %d tokens, %d experts, top %d" % (tokens, experts, top_k), flush=True)
    if tokens >= 263:
        ways = _thresholds(logits, top_k)
        if 4 * top_k > 3 * min((experts + 3) // 4, 16):
            assert set(ways) == {"searched"}
        else:
            assert ways[::4].count("quads") > ways[::4].count("many") and (top_k == 1 or "tied" in ways[3::4])
            assert experts < 256 or top_k == 1 or set(ways[1::4]) == {"many"}
    bad = logits.copy()
    bad[tokens // 2, experts // 2] = np.nan
    with contextlib.closing(hip_router.HipRouter(tokens, experts, top_k)) as router:
        for score in (hip_router.SOFTMAX, hip_router.SIGMOID):
            cpu_status, cpu_offsets, cpu_routes = oracle_lib.oracle_router_dispatch(logits, top_k, score_function=score)
            for _ in range(2):
                status, offsets, routes = router.dispatch(logits, top_k, score_function=score)
                assert status == cpu_status == 0
                assert np.array_equal(offsets, cpu_offsets)
                for field in ("token_index", "rank"):
                    assert np.array_equal(routes[field], cpu_routes[field]), field
                assert np.array_equal(routes["weight"].view(np.uint32), cpu_routes["weight"].view(np.uint32))
                assert router.dispatch(bad, top_k, score_function=score)[0] == hip_router.STATUS_NON_FINITE_LOGIT
